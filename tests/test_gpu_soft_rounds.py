"""Soft scattering where the K values per workgroup change: the largest call of
one round of 1024 workgroups of 66 K values, one more, and the same of two
rounds. First and last values against the oracle, within the bound of the other
soft-scattering tests, and every value against the calls of a few thousand."""
import numpy as np
import pytest
import torch

import oracle
from noa_amd import dcs
from noa_amd.physics import MUON_MASS, STANDARD_ROCK
from tests.parity import assert_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [67583, 67584, 67585, 135168, 135169])
def test_soft_rounds(device, n):
    Kh = 10.0 ** np.random.default_rng(n).uniform(-3, 6, n)
    K = torch.from_numpy(Kh).to(device)
    out = torch.full((n + 8,), -3.0, dtype=torch.float64, device=device)
    dcs.soft_scattering(out[:n], K, STANDARD_ROCK, MUON_MASS)
    parts = torch.empty(n, dtype=torch.float64, device=device)
    for a in range(0, n, 4000):
        b = min(n, a + 4000)
        dcs.soft_scattering(parts[a:b], K[a:b].contiguous(), STANDARD_ROCK, MUON_MASS)
    assert bool((out[n:] == -3.0).all())
    assert_parity(out.cpu().numpy()[:n], parts.cpu().numpy(), 1e-10, str(n))
    at = np.concatenate([np.arange(200), np.arange(n - 200, n)])
    assert_parity(out.cpu().numpy()[:n][at], oracle.soft_scattering(Kh[at], STANDARD_ROCK, MUON_MASS, threads=0), 1e-10,
                  str(n))
