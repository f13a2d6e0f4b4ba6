"""The training step's gradients over the numbers of rows at which its tiles,
row splits and their places change, against the bf16-emulating FP64 network."""
import numpy as np
import pytest
import torch

from noa_amd import surrogate as S
from tests import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 31, 64, 65, 960, 1024, 2048, 2049, 3072, 8192])
def test_gradients_at_tile_and_split_edges(device, rows):
    """As the gradient test at one size holds them (2e-3 in relative L2 norm per parameter block)."""
    rng = np.random.default_rng(rows)
    X = rng.uniform(-1, 1, (rows, 3)).astype(np.float32)
    T = rng.normal(0, 1, (rows, 4)).astype(np.float32)
    M = (rng.uniform(0, 1, (rows, 4)) < 0.7).astype(np.float32)
    M[0] = 1.
    net = S.Network(seed=3, max_rows=8192, device=device)
    loss, g = net.forward_backward(*(torch.from_numpy(a).to(device) for a in (X, T, M)))
    want_loss, want = mlp_ref.loss_and_grad(net.get_params(), X, T, M, round_bf16=True)
    assert abs(loss / want_loss - 1) < 1e-4, (loss, want_loss)
    for name, (o, s) in mlp_ref.OFF.items():
        a, b = g[o:o + s].astype(np.float64), want[o:o + s]
        assert np.linalg.norm(a - b) <= 2e-3 * np.linalg.norm(b), name
    net.close()


def test_epoch_losses_are_the_call_s_own(device):
    """A call's losses start from zero, whatever an earlier, longer call left."""
    rng = np.random.default_rng(0)
    X, T = (torch.from_numpy(rng.normal(0, 1, (4096, k)).astype(np.float32)).to(device) for k in (3, 4))
    M = torch.ones_like(T)
    runs = []
    for before in (0, 5):
        net = S.Network(seed=1, max_rows=1024, device=device)
        p = net.get_params()
        if before:
            net.train(X, T, M, epochs=before, batch=1024)
            net.set_params(p)
        # without a step size the parameters stay: every epoch has the same mean loss
        runs.append(net.train(X, T, M, epochs=2, batch=1024, lr_max=0., lr_min=0.))
        net.close()
    assert np.allclose(runs[0], runs[1], rtol=1e-6, atol=0) and np.allclose(runs[0][0], runs[0][1], rtol=1e-6, atol=0)
