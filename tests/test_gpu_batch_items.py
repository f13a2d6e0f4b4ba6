"""The batch's work items: at most 64 pairs each in small batches, elsewhere
tiles that shorten towards the end of the list. A pair's result is the same
in whichever item and kernel it falls, so a batch whose ranges belong to one
element is compared bit for bit with one map over all its pairs, which
itself is held to the oracle elsewhere."""
import numpy as np
import pytest
import torch

from noa_amd import dcs, workload
from noa_amd.batch import BatchPlan
from noa_amd.physics import MUON_MASS, STANDARD_ROCK, AtomicElement

pytestmark = pytest.mark.gpu


def _map(K, q, el, precision):
    if precision == "f64":
        return dcs.hip.map_all(K, q, el, MUON_MASS)
    return dcs.hip.map_all_f32mixed(K, q, el, MUON_MASS)


@pytest.mark.parametrize("precision", ["f64", "f32mixed"])
@pytest.mark.parametrize("counts,config", [
    ((1,), {}), ((0, 64, 65, 63, 0, 1), {}), ((0, 0), {}), ((1,) * 3000, {}), ((200000,), {}),
    ((100000, 100001), {}), ((511, 513, 0, 299000), {}), ((70001,) * 11, {}), ((2500001, 2048, 17), {}),
    ((5000, 64, 3), {"tile": 1024}), ((5000, 64, 3), {"waves_per_cu": 1}), ((300001, 7), {"waves_per_cu": 32}),
    ((300001, 7), {"tile": 4096, "waves_per_cu": 2, "use_graph": False})])
def test_batch_of_one_element_is_its_map(device, counts, config, precision):
    off = np.concatenate([[0], np.cumsum(counts)])
    n = int(off[-1])
    K = torch.empty(max(n, 1), dtype=torch.float64, device=device)
    q = torch.empty_like(K)
    workload.fill_device(K, q, seed=3)
    plan = BatchPlan([STANDARD_ROCK] * len(counts), off, K, q, MUON_MASS, precision=precision, **config)
    info = plan.info()
    for key in ("tile", "waves_per_cu"):
        assert info[key] == config.get(key, info[key]), info
    for o in plan.outputs:
        o.fill_(-1.)
    for _ in range(2):
        plan.launch()
    if n:
        # a mixed map of up to 200,000 pairs holds rounded FP64 values, a pinned plan mixed ones
        if config and n <= 200000 and precision == "f32mixed":
            big = torch.cat([K] * (200000 // n + 1)), torch.cat([q] * (200000 // n + 1))
            want = [w[:n] for w in _map(*big, STANDARD_ROCK, precision)]
        else:
            want = _map(K, q, STANDARD_ROCK, precision)
        for g, w in zip(plan.outputs, want):
            assert torch.equal(g, w)
    plan.close()


def test_items_read_their_own_element(device):
    """Elements of very different Z, every second one empty or a single pair, against the element's own map."""
    els = [AtomicElement(2.2 * Z, 16e-9 * Z ** 0.9, Z) for Z in (1, 92, 11, 47, 6, 82)]
    for counts in ((700, 0, 1300, 1, 64, 65), (150000, 0, 130001, 1, 64, 90000)):  # small items, tiles
        off = np.concatenate([[0], np.cumsum(counts)])
        K = torch.empty(int(off[-1]), dtype=torch.float64, device=device)
        q = torch.empty_like(K)
        workload.fill_device(K, q, seed=5)
        plan = BatchPlan(els, off, K, q, MUON_MASS)
        plan.launch()
        for e, el in enumerate(els):
            a, b = int(off[e]), int(off[e + 1])
            if a < b:
                for g, w in zip(plan.outputs, _map(K[a:b].contiguous(), q[a:b].contiguous(), el, "f64")):
                    assert torch.equal(g[a:b], w), e
        plan.close()
