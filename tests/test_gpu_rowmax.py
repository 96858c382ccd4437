"""Sampled row maxima on the MFMA scans and on the direct kernel, against the
oracle: sizes around the line between the two and off the tile and block sizes,
samples of part of the rows, repeated positions, contigs all of one size, rows
without a valid window, rows whose maximum lies below the floor of the second
logistic model or exactly on it, rows of a norm the bounds do not cover, and so
many equal pairs that the list of the scan overflows."""
import numpy as np
import pytest

import mdet_amd as M
from mdet_amd import workload
from oracle import oracle as O

pytestmark = pytest.mark.gpu

LINE = 64  # contigs up to which the direct kernel runs alone (RM_DIRECT_MAX)


def _rows(ctx, n, seed):
    w = workload.make(ctx, "c2_50k", n=n, seed=seed)
    t, ls = w.tnf.numpy(), w.logsize.numpy()
    for a in (w.tnf, w.logsize, w.counts):
        a.free()
    return t, ls


def _check(ctx, t, ls, idx, sample):
    dt, dl = ctx.to_device(t), ctx.to_device(ls)
    try:
        got = ctx.tnf_rowmax(dt, dl, len(ls), idx.astype(np.uint64), sample)
    finally:
        dt.free()
        dl.free()
    want = O.rowmax(t, ls, idx.astype(np.uint64), sample)
    print(f"n {len(ls)} sample {sample}: {np.min(want)} .. {np.max(want)}, off by {np.max(np.abs(got - want))}", flush=True)
    # the same FP64 maximum; exp() may differ in the last bit
    assert np.max(np.abs(got - want)) <= 4e-16
    return want


def _unit(x):
    return (x / np.sqrt((x.astype(np.float64) ** 2).sum(1, keepdims=True))).astype(np.float32)


@pytest.mark.parametrize("n,sample", [(1, 1), (2, 2), (LINE, LINE), (LINE + 1, LINE), (129, 129), (1025, 1025),
                                      (1999, 1999), (2600, 500), (33_000, 32)])
def test_rowmax_sizes(ctx, n, sample):
    t, ls = _rows(ctx, n, seed=n)
    _check(ctx, t, ls, np.random.default_rng(n).permutation(n), sample)


@pytest.mark.parametrize("case", ["repeated", "one_size", "two_sizes", "nonfinite", "all_nan_but_one"])
def test_rowmax_special_rows(ctx, case):
    n = 1300
    t, ls = _rows(ctx, n, seed=7)
    rng = np.random.default_rng(1)
    idx = rng.permutation(n)
    if case == "repeated":
        idx[700:720] = idx[3]
        idx[5] = idx[4]
    elif case == "one_size":
        ls[:] = ls[0]
    elif case == "two_sizes":
        ls[:] = np.where(rng.random(n) < 0.5, ls.min(), ls.max())
    elif case == "nonfinite":
        t[rng.choice(n, 50, replace=False)] = np.nan
        t[rng.choice(n, 5, replace=False), 7] = np.inf
    else:
        t[np.arange(n) != 11] = np.nan
    with np.errstate(invalid="ignore"):
        _check(ctx, t, ls, idx, n)


def floor_rows(seed=5):
    # 22 groups of 60 unit rows, all pairs of a group at one distance from 0.2 to
    # 0.28; at this size model 1 passes ln 9 at 0.2368 and model 2 at 0.2410
    rng = np.random.default_rng(seed)
    rows = []
    for r in np.concatenate([np.linspace(0.2, 0.236, 6), np.linspace(0.2375, 0.2405, 10), np.linspace(0.242, 0.28, 6)]):
        q, _ = np.linalg.qr(rng.standard_normal((136, 61)))
        rows.append(np.sqrt(1 - r * r / 2) * q[:, 0] + r / np.sqrt(2) * q[:, 1:].T)
    lo, hi = M.model_cheb()[2]
    t = np.concatenate(rows).astype(np.float32)
    return t, np.full(len(t), lo + (hi - lo) * (1 - 0.825) / 2)


def test_rowmax_below_and_on_the_floor(ctx):
    t, ls = floor_rows()
    n = len(ls)
    want = _check(ctx, t, ls, np.random.default_rng(6).permutation(n), n)
    floor = 1 - 1 / (1 + np.exp(2.1972245773362196))
    assert (want < floor - 1e-9).sum() == 360 and (want > floor + 1e-9).sum() == 360
    assert (np.abs(want - floor) < 1e-12).sum() == 600


@pytest.mark.parametrize("case", ["norm", "ties"])
def test_rowmax_outside_the_bounds(ctx, case):
    n = 1300
    t, ls = _rows(ctx, n, seed=9)
    if case == "norm":
        t[17] *= 1.5
    else:
        t[:] = t[0]
        ls[:] = ls[0]
    _check(ctx, t, ls, np.random.default_rng(2).permutation(n), n)


def test_similarity_runs_of_equal_rows(ctx):
    # runs of one i of every length from the same lanes on, contig 0 among them
    t, ls = _rows(ctx, 400, seed=11)
    rng = np.random.default_rng(3)
    pi = np.concatenate([[5], np.zeros(3, int), [7], np.repeat(rng.integers(0, 400, 300), rng.integers(1, 70, 300)),
                         np.tile([9, 0], 64)])
    pi = np.concatenate([pi, pi[::-1], [3]])
    pj = rng.integers(0, 400, len(pi))
    dt, dl = ctx.to_device(t), ctx.to_device(ls)
    got = ctx.tnf_similarity64(dt, dl, 400, pi, pj)
    _, pre = ctx.tnf_preprob(dt, dl, 400, pi, pj)
    dt.free()
    dl.free()
    want = 1 - 1 / (1 + np.exp(pre))  # one thread a pair, the same order of the sums
    assert np.max(np.abs(got - want)) <= 4e-16
