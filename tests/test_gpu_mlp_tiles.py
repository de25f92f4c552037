"""The warm-start network's kernels at the edges of their tiles (64 samples a wave, 256 a block,
131072 a full grid of the evaluation), on rows whose address is not a multiple of 16 bytes, and
the operand copies that the Adam step writes."""
import numpy as np
import pytest

import mlp_ref as R
from test_gpu_mlp import _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 8192 + 33])
def test_gradient_at_tile_edges(n):
    net, p, x, xm, xs, t, xd, td = _setup(20, 8192 + 33)
    g, loss = net.gradient(xd[:n], td[:n])
    gr, lr_ = R.gradient(p.astype(np.float64), R.features_in(x[:n], xm, xs), t[:n].astype(np.float64))
    # a factor that FP32 accumulation puts on the other side of a bf16 rounding differs by 2^-8;
    # an entry of the gradient is a product with at most three such factors
    for a, b in ((R.OW1, R.OB1), (R.OB1, R.OW2), (R.OW2, R.OB2), (R.OB2, R.OW3), (R.OW3, R.OB3), (R.OB3, R.NPARAM)):
        assert np.linalg.norm(g[a:b] - gr[a:b]) <= 3 * 2.0**-8 * np.linalg.norm(gr[a:b])
    assert abs(loss - lr_) <= 3 * 2.0**-8 * lr_
    net.close()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257, 131071, 131072 + 1, 3 * 131072 + 100])
@pytest.mark.parametrize("shift", [0, 1, 2])
def test_predict_at_tile_edges_and_alignments(n, shift):
    import torch

    net, p, x, xm, xs, t, xd, td = _setup(21, 512)
    rows = xd.repeat((n + 511) // 512, 1)[:n].contiguous()
    y0 = net.predict(xd, torch.empty(512, dtype=torch.float32, device="cuda")).cpu()
    flat = torch.empty(8 * n + shift, dtype=torch.float32, device="cuda")
    flat[shift:] = rows.reshape(-1)
    out = torch.full((n + 64,), 7.0, dtype=torch.float32, device="cuda")
    y = net.predict(flat[shift:].view(n, 8), out[:n]).cpu()
    assert torch.equal(y, y0.repeat((n + 511) // 512)[:n])
    assert bool((out[n:] == 7.0).all())
    net.close()


@pytest.mark.parametrize("n,batch", [(1000, 64), (1000, 448), (5000, 4096)])
def test_training_keeps_the_operand_copies_current(n, batch):
    import torch

    from wflowhip import Mlp

    net, p, x, xm, xs, t, xd, td = _setup(22, n)
    net.train_epoch(xd, td, batch=batch, lr=2e-3)
    other = Mlp(device=0, seed=1)
    other.set_normalization(xm, xs, 0.0, 1.0)
    other.set_params(net.params())
    assert not np.array_equal(net.params(), p)
    ya, yb = (m.predict(xd, torch.empty(n, dtype=torch.float32, device="cuda")).cpu() for m in (net, other))
    assert torch.equal(ya, yb)
    ga, gb = (m.gradient(xd, td)[0] for m in (net, other))  # the transposed copies
    assert np.array_equal(ga, gb)
    net.close()
    other.close()
