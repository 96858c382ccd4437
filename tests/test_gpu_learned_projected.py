"""The learned filter on either side of the sizes from which its probed pairs and
its fallback scan projected rows: with every row completed the edges equal the exhaustive mode's,
with rows that hold no valid window, rows far from unit norm and duplicates."""
import numpy as np
import pytest

import mdet_amd as M
from mdet_amd import learned as L
from mdet_amd import workload

pytestmark = pytest.mark.gpu

LINE = 38_730  # n x n pairs of full rows and contigs reach PROJ_PAIRS


# 32 probes of 40 clusters: 36,000 contigs stay below the line in the probed
# pairs, 44,000 pass it
@pytest.mark.parametrize("n,n_clusters,n_probe", [(LINE - 500, 0, 1), (LINE + 401, 0, 1), (36_000, 40, 32),
                                                  (44_000, 40, 32)])
def test_completed_rows_equal_the_exhaustive_mode(ctx, n, n_clusters, n_probe):
    w = workload.make(ctx, "c2_50k", n=n, seed=n)
    t, ls = w.tnf.numpy(), w.logsize.numpy()
    mean, istd = L.input_norm(t)
    rng = np.random.default_rng(n)
    t[rng.choice(n, 60, replace=False)] = np.nan
    good = np.flatnonzero(~np.isnan(t[:, 0]))
    t[good[:40]] = t[good[40:80]]
    t[good[100:110]] *= 1.02
    dt, dl = ctx.to_device(t), ctx.to_device(ls)
    mlp = M.Mlp(ctx, seed=4)
    mlp.set_input_norm(mean, istd)
    try:
        f0, t0, s0, _ = ctx.tnf_edges(dt, dl, n, 0.95, 50, M.BF16_REFINE)
        ctx.set_learned_fallback_margin(1)
        f, to, s, st = ctx.tnf_edges(dt, dl, n, 0.95, 50, M.LEARNED, mlp=mlp, radius2=0.0, n_clusters=n_clusters,
                                     n_probe=n_probe)
    finally:
        ctx.set_learned_fallback_margin(32)
        mlp.close()
        for a in (dt, dl, w.tnf, w.logsize, w.counts):
            a.free()
    print(f"n {n}: {len(f)} edges, {st.fallback_rows} full rows, {st.pairs_evaluated} pairs", flush=True)
    assert st.fallback_rows == n and len(f0) > 100_000
    assert np.array_equal(f, f0) and np.array_equal(to, t0) and np.array_equal(s, s0)
