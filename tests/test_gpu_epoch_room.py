"""The epochs' losses of a training call where their buffer changes (the
network's own up to 511 epochs, one that grows beyond): every epoch's loss is
the same without a step size, and a shorter call afterwards is unaffected."""
import numpy as np
import pytest
import torch

from noa_amd import surrogate as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("epochs", [511, 512, 600])
def test_epoch_room(device, epochs):
    rng = np.random.default_rng(0)
    X, T = (torch.from_numpy(rng.normal(0, 1, (256, k)).astype(np.float32)).to(device) for k in (3, 4))
    net = S.Network(seed=1, max_rows=256, device=device)
    want = net.train(X, T, torch.ones_like(T), epochs=1, batch=256, lr_max=0., lr_min=0.)
    for n in (epochs, 3, 640):
        got = net.train(X, T, torch.ones_like(T), epochs=n, batch=256, lr_max=0., lr_min=0.)
        # each epoch sums the same rows in an order of its own, in FP32
        assert len(got) == n and np.allclose(got, want[0], rtol=1e-5, atol=0)
    net.close()
