"""PUMAS tables of more elements than one launch holds, 30 in the table's and 48 in the envelope's, against the oracle
within the bounds of the other table tests: even and uneven splits, launches whose first element is not the table's
first (which alone takes the model everywhere), and the envelope's kernels on either side of 8000 rows per launch."""
import numpy as np
import pytest
import torch

import oracle
from noa_amd import pumas
from tests.test_gpu_pumas import MUON, _check_envmax, _check_table, _ulps32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_el, n_K, cutoff, mass", [(30, 4, 0.05, MUON), (31, 5, 0.05, MUON), (48, 7, 0.2, MUON),
                                                     (49, 6, 0.05, 1.77682), (61, 3, 1e-4, MUON), (97, 4, 0.05, MUON),
                                                     (49, 110, 0.05, MUON)])
def test_table_of_several_launches(device, n_el, n_K, cutoff, mass):
    rng = np.random.default_rng(1000 * n_el + n_K)
    Z = rng.permutation(1.0 + np.arange(n_el) * 91 // max(1, n_el - 1))
    A = np.where(Z == 1.0, 1.00794, Z * rng.uniform(2.0, 2.6, n_el))
    K = np.sort(10.0 ** rng.uniform(-2, 8, n_K))
    print(f"pumas table {n_el} x {n_K}, cutoff {cutoff}", flush=True)
    table, x, env = (t.cpu().numpy() for t in pumas.dcs_table(Z, A, mass, cutoff, torch.from_numpy(K).to(device)))
    dcs, xf, _, oenv = oracle.pumas_dcs_table(Z, A, mass, cutoff, K, threads=0)
    assert np.array_equal(x, xf)
    _check_table(table, dcs, "table")
    assert np.array_equal(env[..., 0] == 0, oenv[..., 0] == 0) and _ulps32(env[..., 0], oenv[..., 0]).max() <= 1
    _check_envmax(env[..., 1], oenv[..., 1], "envelope maximum", dcs)
