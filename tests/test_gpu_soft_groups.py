"""Soft scattering at the sizes where its kernel changes (open integrals spread
over lanes by node up to 2048 energies, whole integrals per lane above), at
odd counts and for special energies, against the oracle within 1e-10, the
bound of the other soft-scattering test: the skipped nodes' terms are exact
zeros and the terms are non-negative, so only the nodes' own error counts."""
import numpy as np
import pytest
import torch

import oracle
from noa_amd import dcs
from noa_amd.physics import MUON_MASS, STANDARD_ROCK, TAU_MASS, AtomicElement
from tests.parity import assert_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("el, mass", [(STANDARD_ROCK, MUON_MASS), (AtomicElement(1.00794, 19.2e-9, 1), TAU_MASS)],
                         ids=["rock-muon", "H-tau"])
@pytest.mark.parametrize("n", [1, 2, 3, 1023, 1025, 2047, 2048, 2049, 22529, 65537])
def test_soft_sizes(device, el, mass, n):
    Kh = 10.0 ** np.random.default_rng(n).uniform(-3, 6, n)
    K = torch.from_numpy(Kh).to(device)
    out = torch.full((n + 8,), -3.0, dtype=torch.float64, device=device)
    dcs.soft_scattering(out[:n], K, el, mass)
    at = np.unique(np.concatenate([np.arange(min(n, 400)), np.arange(max(0, n - 400), n)]))
    assert_parity(out.cpu().numpy()[:n][at], oracle.soft_scattering(Kh[at], el, mass, threads=0), 1e-10, str(n))
    assert bool((out[n:] == -3.0).all()) and not bool(out[:n].isnan().any())


@pytest.mark.parametrize("n", [1500, 3000])
def test_soft_special_energies(device, n):
    special = np.array([np.nan, np.inf, -np.inf, 0., -1., 1e-310, 1e-25, 1e-19, 1e-9, 19.9, 20.0, 20.1, 500.0,
                        1e12, 1e29, 1e31, 1e150, 1e300])
    Kh = np.concatenate([special, 10.0 ** np.random.default_rng(n).uniform(-3, 6, n - special.size)])
    out = torch.empty(n, dtype=torch.float64, device=device)
    dcs.soft_scattering(out, torch.from_numpy(Kh).to(device), STANDARD_ROCK, MUON_MASS)
    exp = oracle.soft_scattering(Kh[:200], STANDARD_ROCK, MUON_MASS, threads=0)
    assert_parity(out.cpu().numpy()[:200], exp, 1e-10, str(n))
