"""Soft scattering of particles so light or heavy that a node's transport ratio overflows: its NaN reaches the sum
through the nodes whose DCS is zero, as in the oracle. Otherwise within the bound of the other soft-scattering
tests."""
import numpy as np
import pytest
import torch

import oracle
from noa_amd import dcs
from noa_amd.physics import STANDARD_ROCK
from tests.parity import assert_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [300, 2500])
@pytest.mark.parametrize("mass", [1e-200, 1e-170, 1e-100, 1e-20, 1e30, 1e100, 1e154, 1e160, 1e200, 1e300])
def test_soft_masses(device, mass, n):
    Kh = np.concatenate([[1e-3, 1., 10., 100., 1e4], 10.0 ** np.random.default_rng(n).uniform(-3, 7, n - 5)])
    out = torch.empty(n, dtype=torch.float64, device=device)
    dcs.soft_scattering(out, torch.from_numpy(Kh).to(device), STANDARD_ROCK, mass)
    exp = oracle.soft_scattering(Kh[:300], STANDARD_ROCK, mass, threads=0)
    assert_parity(out.cpu().numpy()[:300], exp, 1e-10, f"mass {mass}")
