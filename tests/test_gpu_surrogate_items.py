"""The surrogate's work items: a call is cut into items of 256 to 4096 queries
by its size, whole items first and the elements' remainders after them, and a
query's result is the same in whichever item it falls."""
import numpy as np
import pytest
import torch

from noa_amd import surrogate as S
from noa_amd.physics import AtomicElement

pytestmark = pytest.mark.gpu


def _elements(n):
    return [AtomicElement(1. + 2.3 * (e + 1), 1.2e-8 * (e + 1), e + 1) for e in range(n)]


@pytest.mark.parametrize("counts", [
    (1,), (0, 257, 0), (255, 512, 513), (4095, 4097), (0,) * 7, (1365,) * 48, (5461, 1, 0) * 16,
    (300000, 17, 65536), (1,) * 700, (1,) * 1500])
def test_items_hold_every_query_once(device, counts):
    """Against one call per element, cut from the same queries (bitwise: the
    same operations on the same operands), with the counts of exact
    evaluations equal to the sum; the recheck sample goes by the query's
    index in the call and stays off."""
    els = _elements(len(counts)) if len(counts) <= 60 else _elements(60) * 25
    els = els[:len(counts)]
    off = np.concatenate([[0], np.cumsum(counts)])
    K, q = S.make_pairs(off, seed=9, device=device)
    stats = {"mean": np.linspace(-3, -1, 4), "std": np.ones(4), "trend": np.zeros((4, S.NTREND))}
    net = S.Network(seed=4, device=device)
    flags = np.random.default_rng(1).integers(0, 16, (len(els), S.MAP_BINS, S.MAP_BINS)).astype(np.uint8)
    got, cnt = S.Surrogate(net, els, stats, flags, 1e-3).evaluate(K, q, off, recheck_per_mille=0)
    n_exact = S.Surrogate.read_counters(cnt)[0]
    want, n_want = [], 0
    step = max(1, len(els) // 60)  # many one-query elements: in groups of `step`
    for e in range(0, len(els), step):
        a, b = int(off[e]), int(off[min(e + step, len(els))])
        if a == b:
            continue
        part = S.Surrogate(net, els[e:e + step], stats, flags[e:e + step], 1e-3)
        out, c = part.evaluate(K[a:b].contiguous(), q[a:b].contiguous(), off[e:e + step + 1] - a,
                               recheck_per_mille=0)
        want.append([o.clone() for o in out])
        n_want += S.Surrogate.read_counters(c)[0]
    assert n_exact == n_want
    for p in range(4):
        w = torch.cat([o[p] for o in want]) if want else got[p][:0]
        assert torch.equal(got[p], w), p
    net.close()
