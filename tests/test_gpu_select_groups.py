"""Selection of rows whose bucket of 64 fits the kernel's LDS, just does, just
does not and does not by far: rows selected in place, rows staged from memory,
and rows of either kind handed to the block-wide path (a near-tie zone wider
than a wave: all partners of the sets of small spread lie in one)."""
import numpy as np
import pytest

import mdet_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu

LENGTH = 20000


def _group(n, spread):
    """n rows around one random composition; spread .03: every pair is a candidate"""
    rng = np.random.default_rng(n)
    p = rng.dirichlet(np.full(136, 4.0)) * np.abs(1 + spread * rng.standard_normal((n, 136)))
    counts = np.rint(p / p.sum(1, keepdims=True) * LENGTH).astype(np.uint32)
    return O.normalize_f32(counts), M.logsize_host(np.full(n, LENGTH, np.uint64) + np.arange(n, dtype=np.uint64))


# 64 rows of 103 partners are 6592 entries, of 104 they are 6656
@pytest.mark.parametrize("n,spread", [(64, 0.03), (65, 0.03), (104, 0.03), (105, 0.03), (200, 0.1), (513, 0.03),
                                      (514, 0.03), (513, 0.1), (1000, 0.1)])
@pytest.mark.parametrize("K", [0, 20, 200])
def test_rows_in_lds_and_beyond(ctx, n, spread, K):
    tnf, ls = _group(n, spread)
    f0, t0, s0 = O.edges(tnf, ls, 0.95, K)
    want = f0.astype(np.uint64) * np.uint64(n) + t0.astype(np.uint64)
    order = np.argsort(want)
    dt, dl = ctx.to_device(tnf), ctx.to_device(ls)
    try:
        for mode in (M.EXACT_F32, M.BF16_REFINE):
            f, t, s, st = ctx.tnf_edges(dt, dl, n, 0.95, K, mode)
            print(f"  n={n} K={K} mode {mode}: {len(f)} edges, capped {st.rows_capped}, block rows {st.rows_block}",
                  flush=True)
            assert np.array_equal(f.astype(np.uint64) * np.uint64(n) + t.astype(np.uint64), want[order])
            assert np.max(np.abs(s.astype(np.float64) - s0[order])) < 2e-6
    finally:
        dt.free()
        dl.free()
