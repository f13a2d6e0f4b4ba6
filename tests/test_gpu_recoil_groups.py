"""Recoil integrals at the edges of a workgroup's group of kinetic energies and
of its node tile (512): one node block or several, one K value per workgroup
or as many as a tile holds, odd counts, and the workspace and no-allocation
entry points alike. Held to the oracle within 1e-10, the bound of the other
recoil tests: each node value is within it, the terms are non-negative, and
the sums' own rounding is below 6000 ulps."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from noa_amd import _lib, dcs
from noa_amd.physics import MUON_MASS, STANDARD_ROCK
from tests.parity import assert_parity

pytestmark = pytest.mark.gpu


def _run(K, min_points):
    dels = tuple(torch.full_like(K, np.nan) for _ in range(4))
    cels = tuple(torch.full_like(K, np.nan) for _ in range(4))
    dcs.recoil_integrals(K, 0.05, STANDARD_ROCK, MUON_MASS, min_points, dels=dels, cels=cels)
    return dels, cels


@pytest.mark.parametrize("n, min_points", [(1, 1), (1, 180), (3, 6000), (5, 512), (5, 511), (7, 1021), (129, 7),
                                           (1024, 30), (1025, 30), (2049, 180), (5000, 6), (100003, 6)])
def test_group_and_tile_edges(device, n, min_points):
    Kh = 10.0 ** np.random.default_rng(n + min_points).uniform(-3, 6, n)
    K = torch.from_numpy(Kh).to(device)
    dels, cels = _run(K, min_points)
    at = np.unique(np.concatenate([np.arange(min(n, 40)), np.arange(max(0, n - 40), n)]))
    for cel, outs in ((0, dels), (1, cels)):
        for p in range(4):
            exp = oracle.recoil(p, cel, Kh[at], 0.05, STANDARD_ROCK, MUON_MASS, min_points, threads=0)
            assert_parity(outs[p].cpu().numpy()[at], exp, 1e-10, f"process {p}, cel {cel}")
            assert not bool(outs[p].isnan().any())


def test_one_output_and_special_energies(device):
    """One integral at a time gives the same bits as all eight; NaN, zero,
    negative and infinite energies give the oracle's values or its NaN."""
    Kh = np.concatenate([10.0 ** np.linspace(-3, 6, 97), [0.0, -1.0, np.nan, np.inf, 1e31, 1e-25]])
    K = torch.from_numpy(Kh).to(device)
    dels, cels = _run(K, 60)
    for p, f in enumerate(dcs.PROCESSES):
        for cel, integrand, outs in ((0, dcs.del_integrand, dels), (1, dcs.cel_integrand, cels)):
            one = torch.full_like(K, -3.0)
            dcs.vmap_integral(dcs.recoil_integral(f, integrand))(one, K, 0.05, STANDARD_ROCK, MUON_MASS, 60)
            assert torch.equal(one.nan_to_num(nan=-7.0), outs[p].nan_to_num(nan=-7.0)), (p, cel)
            exp = oracle.recoil(p, cel, Kh, 0.05, STANDARD_ROCK, MUON_MASS, 60, threads=0)
            assert_parity(outs[p].cpu().numpy(), exp, 1e-10, f"process {p}, cel {cel}")


def test_in_place_and_workspace_entry(device):
    """result may be the energies themselves, and the entry point that asks for
    a workspace gives the same bits."""
    lib = _lib.lib()
    K = torch.from_numpy(10.0 ** np.random.default_rng(9).uniform(-3, 6, 3001)).to(device)
    dels, _ = _run(K, 180)
    e = _lib.Element(STANDARD_ROCK.A, STANDARD_ROCK.I, STANDARD_ROCK.Z)
    out = torch.full_like(K, np.nan)
    o = _lib.OutputsF64(None, ctypes.c_void_p(out.data_ptr()), None, None)
    nbytes = lib.noa_dcs_recoil_workspace_bytes(K.numel(), 180)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=device)
    stream = ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)
    _lib.check(lib.noa_dcs_recoil_integrals_f64(ctypes.c_void_p(K.data_ptr()), K.numel(), 0.05, ctypes.byref(e),
                                                MUON_MASS, 180, ctypes.byref(o), None,
                                                ctypes.c_void_p(ws.data_ptr()), nbytes, stream))
    assert torch.equal(out, dels[1])
    same = K.clone()
    dcs.vmap_integral(dcs.recoil_integral(dcs.pair_production, dcs.del_integrand))(
        same, same, 0.05, STANDARD_ROCK, MUON_MASS, 180)
    assert torch.equal(same, dels[1])
