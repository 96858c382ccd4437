"""The device packer around the edges of its chunks (1,024 bases) and blocks
(65,536 bases): lengths off and on them, N runs that end, start, stay open or
fill the text across them, chunks without an N behind an open run, and every
byte value; bit for bit against the host packer, at unaligned starts too."""
import numpy as np
import pytest

import mdet_amd as M

pytestmark = pytest.mark.gpu

CHUNK, BLOCK = 1024, 65536


def _check(ctx, text, offset=0):
    packed_h, runs_h, _ = M.pack_ascii([text.tobytes()])
    n = len(text)
    raw = ctx.to_device(np.concatenate([np.zeros(offset, np.uint8), text, np.zeros(16, np.uint8)]))
    packed, runs, nr = ctx.pack_ascii(raw, n, offset=offset)
    got_p, got_r = packed.numpy()[:(n + 15) // 16], runs.numpy()[:2 * nr]
    for a in (raw, packed, runs):
        a.free()
    assert np.array_equal(got_p, packed_h[:(n + 15) // 16])
    assert np.array_equal(got_r, runs_h)


@pytest.mark.parametrize("n", [1, 16, CHUNK - 1, CHUNK, CHUNK + 1, 4 * CHUNK + 5, BLOCK - 1, BLOCK, BLOCK + 1, 3 * BLOCK + 77])
def test_lengths_and_runs_across_edges(ctx, n):
    rng = np.random.default_rng(n)
    base = rng.choice(np.frombuffer(b"ACGTacgt", np.uint8), n)
    _check(ctx, base)
    for edge in (CHUNK, 2 * CHUNK, 16 * CHUNK, BLOCK, n):
        for a, b in ((edge - 1, edge), (edge, edge + 1), (edge - 1, edge + 1), (edge - 40, edge + 3 * CHUNK + 9), (edge - CHUNK, edge)):
            t = base.copy()
            t[max(a, 0):b] = ord("N")
            _check(ctx, t, offset=(a + b) % 4)
    _check(ctx, np.full(n, ord("n"), np.uint8))


def test_every_byte_value(ctx):
    t = np.tile(np.arange(256, dtype=np.uint8), 41)
    _check(ctx, t)
    _check(ctx, np.repeat(np.arange(256, dtype=np.uint8), 37), offset=1)
