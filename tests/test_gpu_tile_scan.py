"""The two routes of the exhaustive edge-list modes against the oracle: every
32 x 32 tile straight to the pair pass (small inputs), and the projected tile
scan ahead of it, at sizes around the line between them and off the tile and
block sizes, over cutoffs with and without the second logistic model, with rows
that hold no valid window, duplicate rows, rows of a norm far from one, rows
without 16-byte alignment, and inputs whose survivors overflow the buffers'
first size."""
import numpy as np
import pytest

import mdet_amd as M
from mdet_amd import workload
from oracle import oracle as O

pytestmark = pytest.mark.gpu

MODES = [M.EXACT_F32, M.BF16_REFINE, M.F16_REFINE]
LINE = 6144  # contigs from which on the scan runs (DIRECT_MAX)


def _rows(ctx, n, seed):
    w = workload.make(ctx, "c2_50k", n=n, seed=seed)
    t, ls = w.tnf.numpy(), w.logsize.numpy()
    for a in (w.tnf, w.logsize, w.counts):
        a.free()
    return t, ls


def _check(ctx, t, ls, cutoff, max_edges, modes=MODES):
    n = len(ls)
    f0, t0, s0 = O.edges(t, ls, cutoff, max_edges)
    order = np.lexsort((t0, f0))
    dt, dl = ctx.to_device(t), ctx.to_device(ls)
    try:
        for mode in modes:
            f, to, s, st = ctx.tnf_edges(dt, dl, n, cutoff, max_edges, mode)
            print(f"n {n} cutoff {cutoff} mode {mode}: {len(f)} edges, {st.survivors} survivors", flush=True)
            assert np.array_equal(f, f0[order]) and np.array_equal(to, t0[order]), f"mode {mode}"
            assert len(s) == 0 or np.max(np.abs(s - s0[order])) < 2e-6
    finally:
        dt.free()
        dl.free()
    return len(f0)


@pytest.mark.parametrize("n,cutoff,max_edges", [(2, 0.95, 200), (33, 0.8, 200), (LINE, 0.95, 200), (LINE + 1, 0.95, 200),
                                                (LINE + 1, 0.8, 20), (6687, 0.98, 0), (7171, 0.8, 200)])
def test_both_routes_equal_the_oracle(ctx, n, cutoff, max_edges):
    t, ls = _rows(ctx, n, seed=n)
    k = _check(ctx, t, ls, cutoff, max_edges)
    assert n < 1000 or k > 1000


@pytest.mark.parametrize("n", [2500, LINE + 300])
def test_rows_without_windows_and_duplicates(ctx, n):
    t, ls = _rows(ctx, n, seed=3)
    rng = np.random.default_rng(n)
    bad = rng.choice(n, 40, replace=False)
    t[bad] = np.nan
    good = np.setdiff1d(np.arange(n), bad)
    a, b = rng.choice(good, (2, 30), replace=False)
    t[a] = t[b]  # pairs at distance 0 (no ties at a cut: max_edges 0)
    # the oracle compares NaN as not above the threshold, as the device does
    _check(ctx, t, ls, 0.95, 0)


@pytest.mark.parametrize("n", [1000, LINE + 300])
def test_exact_mode_takes_rows_of_any_norm(ctx, n):
    """Distances between long rows are far above every threshold; only equal
    rows are within it.  (The Gram modes are defined for unit rows.)"""
    t, ls = _rows(ctx, n, seed=9)
    for scale in (500.0, 1e6):
        x = t.copy()
        x[::2] *= np.float32(scale)
        x[1:200:2] = x[0:199:2]
        k = _check(ctx, x, ls, 0.95, 0, modes=[M.EXACT_F32])
        assert k >= 100


@pytest.mark.parametrize("n", [700, LINE + 300])
def test_rows_without_16_byte_alignment(ctx, n):
    t, ls = _rows(ctx, n, seed=5)
    pad = ctx.to_device(np.concatenate([np.zeros(1, np.float32), t.ravel()]))
    dt, dl = ctx.to_device(t), ctx.to_device(ls)

    class Shifted:
        ptr = pad.ptr + 4

    try:
        for mode in MODES:
            a = ctx.tnf_edges(dt, dl, n, 0.95, 200, mode)
            b = ctx.tnf_edges(Shifted, dl, n, 0.95, 200, mode)
            assert all(np.array_equal(x, y) for x, y in zip(a[:3], b[:3]))
    finally:
        for d in (pad, dt, dl):
            d.free()


@pytest.mark.parametrize("n", [3000, LINE + 800])
def test_survivors_past_the_first_capacity(n):
    """Nearly equal rows: every pair survives, far more than the 128 a contig
    that a new context reserves; the pass runs again with larger buffers."""
    rng = np.random.default_rng(n)
    base = rng.random(136)
    t = base / np.linalg.norm(base) + rng.normal(0, 2e-3, (n, 136))
    t = (t / np.linalg.norm(t, axis=1, keepdims=True)).astype(np.float32)
    ls = np.log10(rng.uniform(3e3, 2e5, n).round())
    with M.Ctx(0) as ctx:
        dt, dl = ctx.to_device(t), ctx.to_device(ls)
        got = [ctx.tnf_edges(dt, dl, n, 0.95, 30, mode) for mode in MODES]
        assert got[0][3].survivors > 200 * n
        for g in got[1:]:
            assert all(np.array_equal(x, y) for x, y in zip(g[:3], got[0][:3]))
        rows = (0, 40)
        f0, t0, _ = O.edges(t, ls, 0.95, 30, rows=rows)
        want = set(zip(f0.tolist(), t0.tolist()))
        f, to = got[0][0], got[0][1]
        k = f < rows[1]
        assert set(zip(f[k].tolist(), to[k].tolist())) == want
