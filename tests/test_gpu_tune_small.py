"""Tuning on an input that skips the scan: there is nothing to time, and the
shape set for larger inputs stays."""
import numpy as np
import pytest

import mdet_amd as M
from mdet_amd import workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [M.BF16_REFINE, M.F16_REFINE, M.EXACT_F32])
def test_a_small_input_leaves_the_scan_shape(mode):
    with M.Ctx(0) as ctx:
        w = workload.make(ctx, "c1_2k", seed=5)
        base = ctx.tnf_edges(w.tnf, w.logsize, w.n, 0.95, 200, mode)
        shape = dict(seg_cols=2048, persistent=0, item_order=0)
        ctx.tune_set(mode, refine_blocks=2, **shape)
        t = ctx.autotune(w.tnf, w.logsize, w.n, 0.95, 200, mode, reps=2)
        print(f"mode {mode}: {t}", flush=True)
        assert {k: t[k] for k in shape} == shape and t["ms_prefilter"] == 0
        assert t["refine_blocks"] == 64 and t["ms_refine"] > 0
        got = ctx.tnf_edges(w.tnf, w.logsize, w.n, 0.95, 200, mode)
        assert all(np.array_equal(x, y) for x, y in zip(got[:3], base[:3]))
        for a in (w.tnf, w.logsize, w.counts):
            a.free()
