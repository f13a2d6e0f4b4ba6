"""Calls whose workgroups make 2^32 work items and more, the most that HIP takes in one launch, so that they go in
several: against the same rows or energies in calls that one launch holds, bit for bit (a value does not depend on
its place in a call). Most of the work is kept out of them: one closed-form process, or rows without a cross section."""
import numpy as np
import pytest
import torch

from noa_amd import dcs, pumas
from noa_amd.physics import MUON_MASS, STANDARD_ROCK

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, min_points", [(2 ** 25 + 9, 180), (2 ** 24 + 9, 516)])
def test_recoil(device, n, min_points):
    """2^24 workgroups and more, of two energies and of one."""
    K = torch.logspace(-3, 6, n, dtype=torch.float64, device=device)
    out = torch.full_like(K, np.nan)
    dcs.recoil_integrals(K, 0.05, STANDARD_ROCK, MUON_MASS, min_points, dels=(out, None, None, None))
    per = 2 if min_points == 180 else 1
    for a in (0, per * (2 ** 24 - 1) - 70000, n - 70000):
        part = torch.full_like(K[a:a + 70000], np.nan)
        dcs.recoil_integrals(K[a:a + 70000].contiguous(), 0.05, STANDARD_ROCK, MUON_MASS, min_points,
                             dels=(part, None, None, None))
        assert torch.equal(out[a:a + 70000], part), a
    assert not bool(out.isnan().any())
