"""The network's gradient and forward kernels take tiles of 16 samples over the
waves of a launch: sample counts around a tile, a workgroup's four tiles, the
largest launch's first pass (32,768 samples) and beyond it, with and without a
permutation, against a float64 restatement.  Tolerance: FP32 sums of n terms
and the tanh's 1e-7, held to 1e-5 of the largest gradient entry (and of the
loss); a wrong or dropped sample moves them by 1 / n of themselves or more, so
the counts around the tiles are small."""
import numpy as np
import pytest
import torch

import trixiatmo_hip as T

pytestmark = pytest.mark.gpu

SIZES = [1, 15, 16, 17, 63, 64, 65, 257, 32768, 32769, 70000]


def reference(p, x, y):
    p = torch.tensor(p, dtype=torch.float64, requires_grad=True)
    h = torch.tanh(x @ p[:96].view(32, 3).T + p[96:128])
    h = torch.tanh(h @ p[128:1152].view(32, 32).T + p[1152:1184])
    out = h @ p[1184:1248].view(2, 32).T + p[1248:1250]
    loss = ((out - y) ** 2).sum(1).mean()
    g, = torch.autograd.grad(loss, p)
    return out.detach().numpy(), float(loss.detach()), g.numpy()


@pytest.mark.parametrize("n", SIZES)
def test_gradient_and_forward_at_tile_edges(n):
    print(f"case: {n} samples", flush=True)
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, 3)).astype(np.float32)
    y = rng.standard_normal((n, 2)).astype(np.float32)
    mlp = T.SaturationMLP(seed=3)
    xd, yd = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    loss, g = mlp.loss_grad(xd, yd)
    out = torch.full((n + 4, 2), 7.0, device="cuda")  # rows past n stay as they are
    mlp.forward(xd, out[:n])
    ref_out, ref_loss, ref_g = reference(mlp.params(), torch.from_numpy(x).double(),
                                         torch.from_numpy(y).double())
    assert abs(loss - ref_loss) <= 1e-5 * ref_loss
    assert np.abs(g - ref_g).max() <= 1e-5 * np.abs(ref_g).max()
    assert np.abs(out[:n].cpu().numpy() - ref_out).max() <= 1e-5
    assert (out[n:] == 7.0).all()


def test_training_step_takes_the_permuted_samples():
    """one Adam step on a batch in the middle of a permutation: its loss is the
    loss of exactly those samples, and the step moves every parameter by the
    learning rate in the direction of its gradient"""
    n, batch = 300, 100
    rng = np.random.default_rng(8)
    x = rng.standard_normal((n, 3)).astype(np.float32)
    y = rng.standard_normal((n, 2)).astype(np.float32)
    perm = rng.permutation(n).astype(np.int32)
    mlp = T.SaturationMLP(seed=5)
    p0 = mlp.params()
    d = [torch.from_numpy(a).cuda() for a in (x, y, perm)]
    loss = mlp.train(d[0], d[1], d[2], batch, 1, 1e-3)
    _, ref_loss, ref_g = reference(p0, torch.from_numpy(x[perm[:batch]]).double(),
                                   torch.from_numpy(y[perm[:batch]]).double())
    assert abs(loss - ref_loss) <= 1e-5 * ref_loss
    big = np.abs(ref_g) > 1e-3 * np.abs(ref_g).max()
    # Adam's first step is lr g / (|g| + eps), on parameters stored in FP32
    step = mlp.params().astype(np.float64) - p0
    assert np.abs(step + 1e-3 * np.sign(ref_g))[big].max() <= 1e-6
