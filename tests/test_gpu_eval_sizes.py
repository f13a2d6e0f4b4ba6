"""The map at the sizes where its kernels change: one workgroup per 64 pairs
with the integrals spread by node for small maps, tiles of 256 to 2048 pairs
above. FP64 results of a pair do not depend on the size of the map it is in
(every kernel rounds alike), so each size is compared bit for bit with the
same pairs inside a large map, which itself is held to the oracle."""
import numpy as np
import pytest
import torch

import oracle
from noa_amd import dcs, workload
from noa_amd.physics import MUON_MASS, STANDARD_ROCK, TAU_MASS, AtomicElement
from tests.parity import assert_parity

pytestmark = pytest.mark.gpu

BIG = 7_000_003  # tiles of 2048, shortening
SIZES = [1, 63, 64, 65, 127, 10007, 200000, 200001, 300000, 300001, 700001, 1500000, 1500001, 2500001]
HYDROGEN = AtomicElement(A=1.00794, I=19.2e-9, Z=1)


def _special():
    """NaN, infinities, zeros, negatives, subnormals and energies above 1e30."""
    v = np.array([np.nan, np.inf, -np.inf, 0., -1., 5e-324, 1e-310, 1e-3, 2.5, 1e6, 1e29, 1e31, 1e150, 1e300])
    return [a.ravel().copy() for a in np.meshgrid(v, v)]


@pytest.fixture(scope="module")
def big(device):
    K = torch.empty(BIG, dtype=torch.float64, device=device)
    q = torch.empty_like(K)
    workload.fill_device(K, q, seed=11)
    sk, sq = (torch.from_numpy(a).to(device) for a in _special())
    for at in (0, 64 * 700 + 5, 200001, BIG - sk.numel()):  # inside the small kernel's, in a tile's middle, at the end
        K[at:at + sk.numel()], q[at:at + sk.numel()] = sk, sq
    return K, q, {}


def _full(big, el, mass):
    K, q, seen = big
    key = (el.Z, mass)
    if key not in seen:
        seen[key] = dcs.hip.map_all(K, q, el, mass)
    return seen[key]


def _same(a, b):
    return torch.equal(a.view(torch.int64), b.view(torch.int64)) or \
        torch.equal(torch.nan_to_num(a, nan=-7.), torch.nan_to_num(b, nan=-7.))


@pytest.mark.parametrize("el, mass", [(STANDARD_ROCK, MUON_MASS), (HYDROGEN, TAU_MASS)], ids=["rock-muon", "H-tau"])
def test_large_map_against_the_oracle(big, el, mass):
    K, q, _ = big
    full = _full(big, el, mass)
    for a, b in ((0, 4096), (199000, 203000), (BIG - 4096, BIG)):
        exp = oracle.dcs_map_all(K[a:b].cpu().numpy(), q[a:b].cpu().numpy(), el, mass, threads=0)
        for p in range(4):
            assert_parity(full[p][a:b].cpu().numpy(), exp[p], 1e-10, f"process {p} at {a}")


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("el, mass", [(STANDARD_ROCK, MUON_MASS), (HYDROGEN, TAU_MASS)], ids=["rock-muon", "H-tau"])
def test_f64_result_does_not_depend_on_the_size(big, el, mass, n):
    K, q, _ = big
    full = _full(big, el, mass)
    guard = torch.full((n + 64,), -3.0, dtype=torch.float64, device=K.device)
    outs = [guard.clone() for _ in range(4)]
    dcs.hip.vmap_all([o[:n] for o in outs], K[:n], q[:n], el, mass)
    for p in range(4):
        assert _same(outs[p][:n], full[p][:n]), (n, p)
        assert bool((outs[p][n:] == -3.0).all()), (n, p, "written past the end")


@pytest.mark.parametrize("n", [65, 10007, 300001])
@pytest.mark.parametrize("p", range(4))
def test_one_output_requested(big, n, p):
    K, q, _ = big
    full = _full(big, STANDARD_ROCK, MUON_MASS)
    got = dcs.map(dcs.PROCESSES[p])(K[:n].contiguous(), q[:n].contiguous(), STANDARD_ROCK, MUON_MASS)
    assert _same(got, full[p][:n])


@pytest.mark.parametrize("n", [1, 257, 262145, 5_000_001])
def test_closed_forms_only(big, n):
    """Bremsstrahlung and ionisation without the integrals, together and alone,
    as in the full map; the mixed form within its 1e-5 of FP64 there (these two
    have no branch on an FP32 value)."""
    K, q, _ = big
    full = _full(big, STANDARD_ROCK, MUON_MASS)
    K, q = K[:n].contiguous(), q[:n].contiguous()
    b, i = (torch.full((n,), -3.0, dtype=torch.float64, device=K.device) for _ in range(2))
    dcs.eval_f64(K, q, STANDARD_ROCK, MUON_MASS, brems=b, ion=i)
    assert _same(b, full[0][:n]) and _same(i, full[3][:n])
    for p in (0, 3):
        alone = [None] * 4
        alone[p] = torch.full((n,), -3.0, dtype=torch.float32, device=K.device)
        dcs.eval_f32mixed(K, q, STANDARD_ROCK, MUON_MASS, *alone)
        assert_parity(alone[p].cpu().numpy(), full[p][:n].float().cpu().numpy(), 1e-5, f"process {p}")


@pytest.fixture(scope="module")
def mixed_full(big):
    K, q, _ = big
    return dcs.hip.map_all_f32mixed(K, q, STANDARD_ROCK, MUON_MASS)


@pytest.mark.parametrize("n", [1, 65, 10007, 200000, 200001, 300001, 700001, 1500001, 2500000])
def test_mixed_at_the_same_sizes(big, mixed_full, n):
    """The small-map kernel's mixed results are the rounded FP64 ones, every
    tile's the same as in tiles of 2048."""
    K, q, _ = big
    got = dcs.hip.map_all_f32mixed(K[:n].contiguous(), q[:n].contiguous(), STANDARD_ROCK, MUON_MASS)
    for p in range(4):
        exp = _full(big, STANDARD_ROCK, MUON_MASS)[p][:n].float() if n <= 200000 else mixed_full[p][:n]
        same = (got[p] == exp) | (got[p].isnan() & exp.isnan())
        assert bool(same.all()), (n, p, int((~same).sum()))
