"""Calls whose workgroups make 2^32 work items and more, the most that HIP takes in one launch, so that they go in
several: against the same rows or energies in calls that one launch holds, bit for bit (a value does not depend on
its place in a call). Most of the work is kept out of them: one closed-form process, or rows without a cross section."""
import ctypes

import numpy as np
import pytest
import torch

from noa_amd import _lib, dcs, pumas, workload
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


def _csn(n_el, n_K, at, device):
    csn = torch.zeros(3, n_el, n_K, dtype=torch.float64, device=device)
    csn[:, :, at] = 1.
    return csn


@pytest.mark.parametrize("n_el, n_K, cutoff", [(48, 466_100, 0.05), (30, 186_500, 3e-8)])
def test_pumas_table(device, n_el, n_K, cutoff):
    """2^26 rows and more of the envelope's 64-lane workgroups, and 2^24 and more of the table's of 256 lanes (one row
    each where the grid has more than 128 nodes). A row depends on its own element's only, but for the first
    element, whose envelope search takes the model everywhere."""
    print(f"pumas table {n_el} x {n_K}, {pumas.n_table_dcs(cutoff)} nodes", flush=True)
    Z = np.arange(1., n_el + 1.)
    A = np.where(Z == 1., 1.008, 2.1 * Z)
    K = torch.logspace(-2, 8, n_K, dtype=torch.float64, device=device)
    at = torch.tensor([0, 1, n_K // 3, n_K // 2, n_K - 240, n_K - 204, n_K - 203, n_K - 202, n_K - 90, n_K - 2, n_K - 1],
                      device=device)
    table, x, env = pumas.dcs_table(Z, A, MUON_MASS, cutoff, K, csn=_csn(n_el, n_K, at, device))
    some = [0, 1, n_el // 2, n_el - 1]
    part, x_p, env_p = pumas.dcs_table(Z[some], A[some], MUON_MASS, cutoff, K, csn=_csn(4, n_K, at, device))
    assert torch.equal(x, x_p)
    for i, e in enumerate(some):
        for a, b in ((table, part), (env, env_p)):
            assert torch.equal(a[:, e].nan_to_num(nan=-7.0), b[:, i].nan_to_num(nan=-7.0)), e
    assert bool((table[:, :, -1] != 0).any()) and bool((env[:, :, -1, 1] != 0).any())


def test_batch(device):
    """2^24 work items and more, of one pair each: a captured graph of two launches, replayed, against the map."""
    n = 2 ** 24 + 5
    els = np.zeros(n, dtype=np.dtype([("A", "f8"), ("I", "f8"), ("Z", "i4")], align=True))
    assert els.itemsize == ctypes.sizeof(_lib.Element)
    els["A"], els["I"], els["Z"] = STANDARD_ROCK.A, STANDARD_ROCK.I, STANDARD_ROCK.Z
    off = np.arange(n + 1, dtype=np.int64)
    K = torch.empty(n, dtype=torch.float64, device=device)
    q = torch.empty_like(K)
    workload.fill_device(K, q, seed=1)
    outs = [torch.empty_like(K) for _ in range(4)]
    want = dcs.hip.map_all(K, q, STANDARD_ROCK, MUON_MASS)
    config = _lib.BatchConfig(_lib.PREC_F64, 2048, 0, 1, None, 1)
    plan = ctypes.c_void_p()
    print("batch of 2^24 + 5 elements", flush=True)
    _lib.check(_lib.lib().noa_dcs_batch_create(
        els.ctypes.data_as(ctypes.POINTER(_lib.Element)), off.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), n,
        MUON_MASS, K.data_ptr(), q.data_ptr(), *[o.data_ptr() for o in outs], ctypes.byref(config),
        _lib.raw_stream(0), ctypes.byref(plan)))
    for _ in range(3):
        for o in outs:
            o.fill_(-1.)
        _lib.launch(_lib.lib().noa_dcs_batch_launch, 0, plan)
        for g, w in zip(outs, want):
            assert torch.equal(g, w)
    _lib.check(_lib.lib().noa_dcs_batch_destroy(plan))
