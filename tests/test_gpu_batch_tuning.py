"""The batch's autotuner and its cache file: which plans are timed, and which lines of the file they take. A timed
plan leaves its results in the outputs before it is launched, which is how these tests see it. Batches of up to
200,000 pairs with nothing pinned run in groups of 64 and have nothing to time."""
import threading
import time

import numpy as np
import pytest
import torch

import oracle
from noa_amd import workload
from noa_amd.batch import BatchPlan
from noa_amd.physics import MUON_MASS, STANDARD_ROCK, AtomicElement
from tests.parity import compare

pytestmark = pytest.mark.gpu

ELS = [STANDARD_ROCK, AtomicElement(207.2, 823e-9, 82)]


def _batch(n, device, els=ELS, seed=1):
    off = np.linspace(0, n, len(els) + 1).astype(np.int64)
    K = torch.empty(n, dtype=torch.float64, device=device)
    q = torch.empty_like(K)
    workload.fill_device(K, q, seed=seed)
    return els, off, K, q, MUON_MASS


def _plan(batch, cache=None, precision="f64", **config):
    """The plan, and whether its creation evaluated the batch."""
    n = batch[2].numel()
    dtype = torch.float64 if precision == "f64" else torch.float32
    outs = tuple(torch.full((n,), -1., dtype=dtype, device=batch[2].device) for _ in range(4))
    plan = BatchPlan(*batch, precision=precision, outputs=outs, tune_cache=None if cache is None else str(cache),
                     **config)
    return plan, not bool((outs[0] == -1.).any())


def test_small_plans_and_larger_ones_keep_their_own_lines(device, tmp_path):
    """150,000 and 250,000 pairs fall into one bucket of the key's size (2^17 to 2^18): the first runs in groups and is
    not timed, so the second must not take its line."""
    cache = tmp_path / "tune.txt"
    small, timed = _plan(_batch(150_000, device), cache)
    assert not timed and small.info()["n_items"] == 2 * -(-75_000 // 64)
    large, timed = _plan(_batch(250_000, device), cache)
    assert timed
    keys = [line.split()[0] for line in cache.read_text().splitlines()]
    assert len(keys) == 2 and keys[0] != keys[1]
    for n, want in ((150_000, small), (250_000, large)):  # and each finds its own again
        again, timed = _plan(_batch(n, device), cache)
        assert not timed and again.info() == want.info()
    assert len(cache.read_text().splitlines()) == 2


def test_cache_line_is_taken(device, tmp_path):
    """A valid line decides tile and unroll without timing, an invalid one is passed over."""
    cache = tmp_path / "tune.txt"
    batch = _batch(700_001, device)
    first, timed = _plan(batch, cache)
    info = first.info()
    key, *values = cache.read_text().split()
    assert timed and [int(v) for v in values] == [info["tile"], info["waves_per_cu"], info["unroll"]]
    first.launch()
    for tile in (1024, 2048, 4096):
        cache.write_text(f"{key} {tile} 4 1\n")
        plan, timed = _plan(batch, cache)
        pinned, _ = _plan(batch, tile=tile, unroll=1)
        assert not timed and plan.info() == pinned.info() and plan.info()["tile"] == tile
        plan.launch()
        for a, b in zip(plan.outputs, first.outputs):
            assert torch.equal(a, b)
    for bad in (f"{key} 999 4 1\n", f"{key} 2048 0 1\n", f"{key} 2048 4 3\n", "other 1024 4 1\n"):
        cache.write_text(bad)
        plan, timed = _plan(batch, cache)
        assert timed and len(cache.read_text().splitlines()) == 2


@pytest.mark.parametrize("precision, tol", [("f64", 1e-10), ("f32mixed", 1e-5)])
def test_tuned_plan_parity(device, precision, tol):
    """A tuned plan above the line, replayed from its graph, against the oracle (the bounds of the other batch
    tests)."""
    els, off, K, q, mass = batch = _batch(260_000, device)
    plan, timed = _plan(batch, precision=precision)
    assert timed
    for _ in range(3):
        for o in plan.outputs:
            o.fill_(-1.)
        plan.launch()
        torch.cuda.synchronize()
        for e, el in enumerate(els):
            a, b = int(off[e]), int(off[e + 1])
            exp = oracle.dcs_map_all(K[a:b].cpu().numpy(), q[a:b].cpu().numpy(), el, mass, threads=0)
            for p in range(4):
                r = compare(plan.outputs[p][a:b].double().cpu().numpy(), exp[p])
                assert r["finite"] and r["zero_mismatch"] == 0 and r["max_rel"] <= tol, (e, p, r)


@pytest.mark.parametrize("config, timed", [({"tile": 2048}, True), ({"tile": 4096, "waves_per_cu": 3}, True),
                                           ({"waves_per_cu": 4}, True), ({"unroll": 2}, True),
                                           ({"tile": 2048, "unroll": 1}, False)])
@pytest.mark.parametrize("precision", ["f64", "f32mixed"])
def test_what_is_not_given_is_timed(device, precision, config, timed):
    """A given tile leaves the unroll open, which has a choice in the mixed form only."""
    if precision == "f64" and "tile" in config:
        timed = False
    batch = _batch(70_001, device)
    plan, was_timed = _plan(batch, precision=precision, **config)
    assert was_timed == timed
    info = plan.info()
    assert {k: info[k] for k in config} == config and info["unroll"] in (1, 2)
    if precision == "f64":
        assert info["unroll"] == config.get("unroll", 1)
    plan.launch()
    both = [_plan(batch, precision=precision, tile=2048, unroll=u)[0] for u in (1, 2)]
    for p in both:
        p.launch()
        for a, b in zip(plan.outputs, p.outputs):
            assert torch.equal(a, b)


def test_given_plans_do_not_wait_for_timing(device):
    """A plan with nothing to choose is created while another thread's is being timed (on a stream of its own). Each
    creation takes a fraction of a millisecond, the timing ten passes over 2^26 pairs."""
    big, small = _batch(1 << 26, device), _batch(5000, device)
    given = dict(tile=2048, waves_per_cu=4, unroll=1, use_graph=False)
    _plan(small, **given)[0].close()
    torch.cuda.synchronize()
    span = []

    def timed():
        with torch.cuda.stream(torch.cuda.Stream(device)):
            t = time.perf_counter()
            plan, _ = _plan(big, use_graph=False)
            span.append(time.perf_counter() - t)
            torch.cuda.synchronize()
            plan.close()

    outs = tuple(torch.empty(5000, dtype=torch.float64, device=device) for _ in range(4))
    torch.cuda.synchronize()
    thread = threading.Thread(target=timed)
    thread.start()
    waits, plans = [], []
    while not span and len(plans) < 4000:
        t = time.perf_counter()
        plans.append(BatchPlan(*small, outputs=outs, **given))
        waits.append(time.perf_counter() - t)
    thread.join()
    for p in plans:
        p.close()
    print(f"timing {span[0] * 1e3:.1f} ms; {len(waits)} creations beside it, the longest {max(waits) * 1e3:.2f} ms")
    assert max(waits) < 0.5 * span[0]
