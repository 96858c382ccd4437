"""Training gradients at batch sizes off and on the kernels' 16-row blocks and
row splits, with contigs that hold no valid window, against the FP64 oracle;
and the same bits from every call."""
import numpy as np
import pytest

import mdet_amd as M
from mdet_amd import learned as L
from mdet_amd import workload
from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 7, 8, 9, 63, 65, 129, 1000])
def test_gradient_by_batch_size(ctx, batch):
    w = workload.make(ctx, "c1_2k", n=300, seed=batch)
    tnf = w.tnf.numpy()
    mean, istd = L.input_norm(tnf)
    tnf[::37] = np.nan
    rng = np.random.default_rng(batch)
    mlp = M.Mlp(ctx, seed=5)
    p = mlp.params()
    p += (0.01 * rng.standard_normal(len(p))).astype(np.float32)
    mlp.set_params(p)
    mlp.set_input_norm(mean, istd)
    pi, pj = (rng.integers(0, 300, batch).astype(np.uint32) for _ in range(2))
    y = (rng.random(batch) < 0.5).astype(np.float32)
    margin = 1e3  # every negative inside the margin: no kinks near the data
    dev = [ctx.to_device(a) for a in (tnf, pi, pj, y)]
    loss, g = mlp.grad(*dev, batch, margin)
    again, g2 = mlp.grad(*dev, batch, margin)
    want_loss, want = MO.loss_and_grad(p.astype(np.float64), mean, istd, np.nan_to_num(tnf, nan=0.0), pi, pj, y, margin,
                                       round_weights=True)
    for a in dev:
        a.free()
    mlp.close()
    assert loss == again and np.array_equal(g, g2)
    assert abs(loss - want_loss) <= 1e-4 * abs(want_loss)
    off = 0
    for name, shp in MO.SHAPES:
        k = int(np.prod(shp))
        a, b = g[off:off + k].astype(np.float64), want[off:off + k]
        # FP32 products and sums and the 1.5e-7 error function; the last bias's
        # gradient is a difference of equal sums
        scale = max(np.linalg.norm(b), 1e-6 * np.linalg.norm(want))
        print(f"batch {batch} {name}: rel err {np.linalg.norm(a - b) / scale:.2e}", flush=True)
        assert np.linalg.norm(a - b) < 1e-4 * scale, name
        off += k
