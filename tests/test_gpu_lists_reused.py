"""Inputs whose tiles with survivors outgrow their list, on a context that a
larger, different input has filled: the pass over them is repeated, and nothing
of the larger input's candidate records, whose contigs this input does not have,
may be read meanwhile.  Edges as from a new context, and as the oracle's on a
row sample."""
import numpy as np
import pytest

import mdet_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu

BIG, N, K = 50_000, 20_000, 50


def _unit(x):
    return (x / np.linalg.norm(x, axis=1, keepdims=True)).astype(np.float32)


def _populations(n, size, seed):
    """n rows in tight populations of `size`: about n * size / 2 survivors."""
    rng = np.random.default_rng(seed)
    centre = rng.random((n // size, 136), np.float32)
    x = centre[np.arange(n) % len(centre)] / np.float32(6.7)
    return _unit(x + rng.normal(0, 2e-3, (n, 136)).astype(np.float32))


def _diffuse(n, radius, seed):
    """One cloud whose pair distances concentrate where under 1% of them lie below
    the radius: no order of the rows helps, nearly every tile keeps a few pairs."""
    rng = np.random.default_rng(seed)
    base = rng.random(136)
    sigma = radius / 0.85 / np.sqrt(2 * 135)
    return _unit(base / np.linalg.norm(base) + rng.normal(0, sigma, (n, 136)))


@pytest.fixture(scope="module")
def inputs():
    size = float(np.log10(20_000.0))
    t = _diffuse(N, M.model_radius(size, size, 0.95), 2)
    ls = np.full(N, size)
    big = _populations(BIG, 250, 1)
    return big, np.full(BIG, size), t, ls


def _run(ctx, dt, dl, mode):
    if mode != M.LEARNED:
        return ctx.tnf_edges(dt, dl, N, 0.95, K, mode)
    net = M.Mlp(ctx, seed=1)
    try:  # every pair of clusters probed
        return ctx.tnf_edges(dt, dl, N, 0.95, K, M.LEARNED, mlp=net, radius2=0.0, n_clusters=8, n_probe=8)
    finally:
        net.close()


@pytest.mark.parametrize("mode", [M.EXACT_F32, M.BF16_REFINE, M.F16_REFINE, M.LEARNED])
def test_a_smaller_input_after_a_larger_one(inputs, mode):
    big, big_ls, t, ls = inputs
    got = []
    for warm in (True, False):
        with M.Ctx(0) as ctx:
            if warm:
                db, dbl = ctx.to_device(big), ctx.to_device(big_ls)
                st = ctx.tnf_edges(db, dbl, BIG, 0.95, K, M.BF16_REFINE)[3]
                print(f"larger input: {st.survivors} survivors", flush=True)
                assert 6_000_000 < st.survivors < 128 * BIG  # within the first capacity
                db.free()
                dbl.free()
            dt, dl = ctx.to_device(t), ctx.to_device(ls)
            got.append(_run(ctx, dt, dl, mode))
            dt.free()
            dl.free()
    (f, to, s, st), (f1, to1, s1, _) = got
    tiles = (N // 32) * (N // 32 + 1) // 2
    print(f"mode {mode}: {len(f)} edges, {st.survivors} survivors, {tiles} tiles", flush=True)
    # several a tile, so past the 2.25 x BIG tiles with survivors that the first
    # capacity holds, and fewer than the larger input's
    assert 5 * tiles < st.survivors < 6_000_000
    assert np.array_equal(f, f1) and np.array_equal(to, to1) and np.array_equal(s, s1)
    f0, t0, _ = O.edges(t, ls, 0.95, K, rows=(0, 40))
    k = f < 40
    assert set(zip(f[k].tolist(), to[k].tolist())) == set(zip(f0.tolist(), t0.tolist()))
    assert len(f) > 100_000
