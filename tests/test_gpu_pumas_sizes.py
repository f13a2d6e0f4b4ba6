"""PUMAS tables at the sizes where the envelope launch changes: more elements
than one launch holds (24), more rows than two waves per SIMD (2048), one
element and one energy; energies up to the scan next to the upper end (1e7)
and a step beyond the table's. The bounds are those of the other table tests."""
import numpy as np
import pytest
import torch

import oracle
from noa_amd import pumas
from tests.test_gpu_pumas import MUON, _check_envmax, _check_table, _ulps32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_el, n_K, cutoff, mass", [(1, 1, 0.05, MUON), (1, 2, 0.3, MUON), (25, 3, 0.05, MUON),
                                                     (26, 30, 0.05, MUON), (24, 29, 0.01, 1.77682),
                                                     (3, 40, 1e-6, MUON)])
def test_table_sizes(device, n_el, n_K, cutoff, mass):
    rng = np.random.default_rng(100 * n_el + n_K)
    Z = np.arange(1, n_el + 1) * 3.0 - 2.0
    A = np.where(Z == 1.0, 1.00794, Z * rng.uniform(2.0, 2.6, n_el))
    K = np.sort(10.0 ** rng.uniform(-3 if n_K > 3 else 1, 9, n_K))
    table, x, env = (t.cpu().numpy() for t in pumas.dcs_table(Z, A, mass, cutoff, torch.from_numpy(K).to(device)))
    dcs, xf, _, oenv = oracle.pumas_dcs_table(Z, A, mass, cutoff, K, threads=0)
    assert np.array_equal(x, xf)
    _check_table(table, dcs, "table")
    assert np.array_equal(env[..., 0] == 0, oenv[..., 0] == 0) and _ulps32(env[..., 0], oenv[..., 0]).max() <= 1
    _check_envmax(env[..., 1], oenv[..., 1], "envelope maximum", dcs)
