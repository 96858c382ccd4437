"""Offsets that do not fit the stream: the call is refused, counts and rows stay
as they were, and the next call counts as if nothing had been."""
import ctypes as C

import numpy as np
import pytest

import mdet_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _count(ctx, packed, total, off, n, cnt, tnf):
    return M.lib().mdet_tnf_count(ctx.h, C.c_void_p(packed.ptr), total, None, 0, C.c_void_p(off.ptr), n,
                                  C.c_void_p(cnt.ptr), C.c_void_p(tnf.ptr))


@pytest.mark.parametrize("n", [1, 3, 400])
def test_refused_offsets_leave_the_outputs(ctx, n):
    rng = np.random.default_rng(n)
    seqs = [rng.choice(np.frombuffer(b"ACGT", np.uint8), int(k)).tobytes() for k in rng.integers(70, 3000, n)]
    packed_h, _, off_h = M.pack_ascii(seqs)
    total = int(off_h[-1])
    beyond, backwards = off_h.copy(), off_h.copy()
    beyond[-1] = total + 1
    backwards[0], backwards[-1] = 5, 4
    packed = ctx.to_device(packed_h)
    good, bad1, bad2 = (ctx.to_device(np.ascontiguousarray(o, np.uint64)) for o in (off_h, beyond, backwards))
    mark_c, mark_t = np.full((n, 136), 77, np.uint32), np.full((n, 136), -3.0, np.float32)
    want = np.stack([O.count_seq(s) for s in seqs])
    for bad in (bad1, bad2):
        cnt, tnf = ctx.to_device(mark_c), ctx.to_device(mark_t)
        assert _count(ctx, packed, total, bad, n, cnt, tnf) == -1
        assert np.array_equal(cnt.numpy(), mark_c) and np.array_equal(tnf.numpy(), mark_t)
        assert _count(ctx, packed, total, good, n, cnt, tnf) == 0
        assert np.array_equal(cnt.numpy(), want)
        assert np.array_equal(tnf.numpy(), O.normalize_f32(want))
        cnt.free()
        tnf.free()
    for a in (packed, good, bad1, bad2):
        a.free()
