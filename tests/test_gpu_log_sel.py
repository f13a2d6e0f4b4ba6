"""The branch-free logarithm equals the branching one bit for bit, over normal
and subnormal arguments and at the special ones."""
import ctypes
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
SO = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "liblog_sel_dev.so")


def _eval(x):
    lib = ctypes.CDLL(SO)
    lib.log_sel_eval.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p, ctypes.c_void_p]
    xd = torch.from_numpy(x).to("cuda:0")
    sel, ref = torch.empty_like(xd), torch.empty_like(xd)
    torch.cuda.synchronize()
    assert lib.log_sel_eval(xd.data_ptr(), xd.numel(), sel.data_ptr(), ref.data_ptr()) == 0
    return sel.cpu().numpy(), ref.cpu().numpy()


@pytest.mark.parametrize("values", ["normal", "near_one", "subnormal", "special"])
def test_log_sel(values):
    rng = np.random.default_rng(3)
    x = {"normal": 10 ** rng.uniform(-307, 308, 1 << 18),
         "near_one": 1 + np.concatenate([rng.uniform(-1e-6, 1e-6, 1 << 16), rng.uniform(-0.5, 1.0, 1 << 16)]),
         "subnormal": rng.integers(1, 1 << 52, 1 << 16).view(np.float64),
         "special": np.array([0.0, -0.0, 1.0, -1.0, -1e300, -1e-310, np.inf, -np.inf, np.nan, 5e-324, 1e-310,
                              2.2250738585072014e-308, 1.7976931348623157e308])}[values]
    np.testing.assert_array_equal(*_eval(x))
