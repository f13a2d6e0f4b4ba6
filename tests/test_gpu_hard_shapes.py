"""Hard scattering for every way its kernel spreads a mixture over lanes and
registers: 1 to 14 elements, a few energies (one element per lane) and many
(several per lane). The sums keep the element order in all of them, so a K's
result is the same bit for bit whatever the call's size; the small calls are
held to the oracle within the bounds of the other hard-scattering test (1e-8 at
most, 1e-11 on average: the root's last step amplifies an ulp)."""
import numpy as np
import pytest
import torch

import oracle
from noa_amd import dcs
from noa_amd.physics import MUON_MASS, AtomicElement

pytestmark = pytest.mark.gpu


def _elements(nel):
    return [AtomicElement(A=(1.00794 if Z == 1 else 2.2 * Z), I=16e-9 * Z ** 0.9, Z=Z) for Z in range(1, 6 * nel, 6)]


def _chain(K, els):
    n, nel, dev = K.numel(), len(els), K.device
    new = lambda *s: torch.full(s, -3.0, dtype=torch.float64, device=dev)  # noqa: E731
    fCM, scr, fs, il, G, mu0, lb = new(nel, n, 2), new(nel, n, 9), new(nel, n), new(nel, n), new(nel, n, 2), new(n), new(n)
    for e, el in enumerate(els):
        dcs.coulomb_data(fCM[e], scr[e], fs[e], il[e], K, el, MUON_MASS)
        dcs.coulomb_transport(G[e], scr[e], fs[e], torch.ones(1, dtype=torch.float64, device=dev))
    dcs.hard_scattering(mu0, lb, G, fCM, scr, il, fs)
    return [t.cpu().numpy() for t in (G, fCM, scr, il, fs)], mu0, lb


@pytest.mark.parametrize("nel", [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 14])
def test_mixture_shapes(device, nel):
    els = _elements(nel)
    big = 140_001  # more than two waves per SIMD at any spread
    Kh = 10.0 ** np.random.default_rng(nel).uniform(-9, 7, big)
    Kh[:6] = [1e-12, 1e-3, 1e30, 1e60, 1e-30, 5e-324]
    K = torch.from_numpy(Kh).to(device)
    _, mu0, lb = _chain(K, els)
    arrays, mu0_s, lb_s = _chain(K[:501].contiguous(), els)
    for a, b in ((mu0_s, mu0[:501]), (lb_s, lb[:501])):
        assert torch.equal(a.nan_to_num(nan=-7.0), b.nan_to_num(nan=-7.0))
    exp_mu, exp_lb = oracle.hard_scattering(*arrays)
    for got, exp in ((mu0_s.cpu().numpy(), exp_mu), (lb_s.cpu().numpy(), exp_lb)):
        assert np.array_equal(np.isnan(got), np.isnan(exp))
        ok = ~np.isnan(exp) & (exp != 0) & np.isfinite(exp)
        assert np.array_equal(got == 0, exp == 0)
        rel = np.abs(got[ok] / exp[ok] - 1)
        assert rel.max() <= 1e-8 and rel.mean() <= 1e-11, (nel, rel.max(), rel.mean())
