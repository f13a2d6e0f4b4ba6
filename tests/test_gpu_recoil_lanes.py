"""Recoil integrals where the lanes per workgroup change with the number of
workgroups: a K's sums are taken in the same order whatever the workgroup, so
its values are the same bit for bit, and the first and last are within 1e-10 of
the oracle (the bound of the other recoil tests)."""
import numpy as np
import pytest
import torch

import oracle
from noa_amd import dcs
from noa_amd.physics import MUON_MASS, STANDARD_ROCK
from tests.parity import assert_parity

pytestmark = pytest.mark.gpu


def _run(K, min_points):
    outs = [tuple(torch.full_like(K, np.nan) for _ in range(4)) for _ in range(2)]
    dcs.recoil_integrals(K, 0.05, STANDARD_ROCK, MUON_MASS, min_points, dels=outs[0], cels=outs[1])
    return outs


@pytest.mark.parametrize("min_points", [6, 180, 186, 512, 1021])
def test_lanes(device, min_points):
    n = 700
    Kh = 10.0 ** np.random.default_rng(min_points).uniform(-3, 6, n)
    Kh[:4] = [1e-9, 1e9, 1e30, 3e12]  # (beyond the integrals' fast path)
    K = torch.from_numpy(Kh).to(device)
    full = _run(K, min_points)
    for m in (1, 33, 256, 257, 512, 513):
        part = _run(K[:m].contiguous(), min_points)
        for a, b in zip(full[0] + full[1], part[0] + part[1]):
            assert torch.equal(a[:m].nan_to_num(nan=-7.0), b.nan_to_num(nan=-7.0)), m
    at = np.concatenate([np.arange(4, 24), np.arange(n - 20, n)])
    for cel in (0, 1):
        for p in range(4):
            exp = oracle.recoil(p, cel, Kh[at], 0.05, STANDARD_ROCK, MUON_MASS, min_points, threads=0)
            assert_parity(full[cel][p].cpu().numpy()[at], exp, 1e-10, f"process {p}, cel {cel}")
