"""The network on batches large enough for the convolutions that take strips of
rows, against the same images one at a time, which take the other kernel: whole
and broken strips, 64- and 32-pixel ones, levels that stay with the other kernel.

The two sum in different orders in FP32 (differences of about 1e-6), which flips
the rounding of an activation to BF16 (2^-9) now and then: far less than one
rounding a value in each of the 15 layers, whose norm is sqrt(15) 2^-9 = 7.6e-3 of
the output's; the gradient passes through as many again.  A tap, row or channel
out of place changes either by its own size."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_nn import _batch, _rel, _to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,nb", [(256, 256, 16), (248, 384, 13)])
def test_batch_equals_its_images(H, W, nb):
    from simcoflow_amd.learned import Trainer, init_weights
    x, t, m = _batch(H, W, nb, 7)
    print(f"[nn strips] H={H} W={W} nb={nb}", flush=True)
    tr = Trainer(H, W, nb, weights=init_weights(3))
    try:
        xd, td, md = _to_dev(x, t, m)
        y = torch.zeros((nb, H, W), device="cuda", dtype=torch.float32)
        y1 = torch.zeros((nb, H, W), device="cuda", dtype=torch.float32)
        torch.cuda.synchronize()
        tr.forward(xd, y, nb)
        g, loss = tr.gradient(xd, td, md, nb)
        g1, loss1 = 0.0, 0.0
        for b in range(nb):
            tr.forward(xd[b:b + 1].contiguous(), y1[b:b + 1], 1)
            gb, lb = tr.gradient(xd[b:b + 1].contiguous(), td[b:b + 1].contiguous(), md[b:b + 1].contiguous(), 1)
            g1, loss1 = g1 + np.asarray(gb, np.float64) / nb, loss1 + float(lb) / nb
        y, y1 = (a.cpu().numpy().astype(np.float64) for a in (y, y1))
    finally:
        tr.close()
    bound = 15 ** 0.5 * 2.0 ** -9
    assert _rel(y, y1) <= bound
    assert abs(float(loss) - loss1) <= bound * loss1
    assert _rel(np.asarray(g, np.float64), g1) <= 2 * bound
