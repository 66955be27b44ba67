"""The weight-gradient kernel where its strips of 32 pixels by some rows do not
fit the levels evenly: level widths of one and a half strips and of half a
strip, heights that are no multiple of three or of a strip's rows, and batches
whose strips are longer.  Reference and tolerance as in test_gpu_nn: the CPU
FP64 network with the same BF16 roundings, to within three times the distance
its own FP32 sums move it."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_nn import _batch, _rel, _to_dev  # noqa: E402

pytestmark = pytest.mark.gpu


def _gradient(H, W, nb, w, x, t, m):
    from simcoflow_amd.learned import Trainer
    tr = Trainer(H, W, nb, weights=w)
    try:
        g, loss = tr.gradient(*_to_dev(x, t, m), nb)
    finally:
        tr.close()
    return g, loss


@pytest.mark.parametrize("H,W,nb", [(8, 128, 1), (24, 384, 3), (40, 128, 2)])
def test_weight_gradient_on_uneven_strips(H, W, nb):
    from oracle import nn_reference as R
    from simcoflow_amd.learned import SPEC, init_weights, kpad, split_weights
    print(f"[nn] weight gradient H={H} W={W} nb={nb}", flush=True)
    w = init_weights(5)
    x, t, m = _batch(H, W, nb, 9)
    g, loss = _gradient(H, W, nb, w, x, t, m)

    def ref(dt):
        Ws = [torch.from_numpy(R.bf16_round(a)).to(dt) for a in split_weights(w)]
        xr = torch.from_numpy(x[:, 1:-1, 1:-1, :].transpose(0, 3, 1, 2).copy()).to(dt)
        lo, _, gr = R.loss_and_grads(xr, torch.from_numpy(t).to(dt), torch.from_numpy(m).to(dt), Ws)
        return lo, [a.numpy().astype(np.float64) for a in gr]
    lo64, g64 = ref(torch.float64)
    _, g32 = ref(torch.float32)
    assert abs(loss - lo64) <= 1e-2 * abs(lo64)
    got = split_weights(g)
    at = 0
    for l, (cin, cout, _) in enumerate(SPEC):
        own = _rel(g32[l], g64[l])
        err = _rel(got[l], g64[l])
        assert err <= min(5e-2, 3 * own + 1e-3), (l, err, own)
        # the padding columns of a layer stay zero
        kp = kpad(cin)
        assert not g[at:at + cout * kp].reshape(cout, kp)[:, 9 * cin:].any()
        at += cout * kp


def test_weight_gradient_of_long_strips():
    """A batch of 16 x 256 x 256 takes strips of 16 rows, its halves of 8: the
    loss is a mean over the points, so the batch's gradient is the mean of its
    halves'.  They differ by the order of FP32 sums of 1e6 terms, whose error
    grows like the square root of their number: 1e3 * 6e-8 = 6e-5."""
    from simcoflow_amd.learned import init_weights
    w = init_weights(3)
    x, t, m = _batch(256, 256, 16, 2)
    whole, _ = _gradient(256, 256, 16, w, x, t, m)
    parts = [_gradient(256, 256, 8, w, x[k:k + 8], t[k:k + 8], m[k:k + 8])[0] for k in (0, 8)]
    mean = 0.5 * (parts[0].astype(np.float64) + parts[1])
    # the output gradient is rounded to BF16 after the division by the number
    # of points, a power of two here, so the halves round alike
    assert _rel(whole.astype(np.float64), mean) <= 6e-5


@pytest.mark.parametrize("H,W,copies", [(8, 128, 128), (16, 128, 64), (64, 128, 16), (24, 384, 16), (72, 256, 8)])
def test_weight_gradient_of_an_image_and_of_its_copies(H, W, copies):
    """An image alone has so few strips that a wave takes one row of taps, in strips
    of one row and a few; a batch of its copies has 4096 of a row or more on the
    finest level, whose waves take all nine taps, and longer ones below.  The loss is
    a mean, so the gradients are equal: the copies' number is a power of two, so the
    output gradient rounds alike, and both take the same convolutions.  What is left
    is the order of FP32 sums of at most 1.5e5 terms: 4e2 * 6e-8 = 2.4e-5 (the loss,
    added up by workgroups of other sizes, likewise)."""
    from simcoflow_amd.learned import init_weights
    print(f"[nn] weight gradient H={H} W={W}, {copies} copies", flush=True)
    w = init_weights(4)
    x, t, m = _batch(H, W, 1, 5)
    one, loss = _gradient(H, W, 1, w, x, t, m)
    many, loss_many = _gradient(H, W, copies, w, *(np.repeat(a, copies, axis=0) for a in (x, t, m)))
    assert _rel(many.astype(np.float64), one.astype(np.float64)) <= 2.4e-5
    assert abs(float(loss_many) - float(loss)) <= 2.4e-5 * float(loss)
