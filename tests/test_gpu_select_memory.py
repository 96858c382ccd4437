"""Above 2^20 contigs the selection's memory goes by the candidates found, not by
the 128 a contig that the first capacity allows for: an input with hardly a pair
in range takes less than 7 KB a contig, and its edges are the oracle's."""
import numpy as np
import pytest

import mdet_amd as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu

N = (1 << 20) + 40


def test_memory_of_an_input_with_few_survivors():
    rng = np.random.default_rng(4)
    t = np.empty((N, 136), np.float32)
    t[:] = rng.random((N // 4, 136), np.float32)[np.arange(N) % (N // 4)]  # four contigs a population
    for i in range(0, N, 1 << 18):
        t[i:i + (1 << 18)] += 0.01 * rng.random((min(1 << 18, N - i), 136), np.float32)
    t /= np.linalg.norm(t, axis=1, keepdims=True)
    ls = np.full(N, np.log10(20_000.0))
    with M.Ctx(0) as ctx:
        dt, dl = ctx.to_device(t), ctx.to_device(ls)
        ctx.sync()
        free = ctx.mem_info()[0]
        f, to, s, st = ctx.tnf_edges(dt, dl, N, 0.95, 200, M.BF16_REFINE)
        used = (free - ctx.mem_info()[0]) / N
        print(f"{len(f)} edges, {st.survivors} survivors, {used:.0f} bytes a contig", flush=True)
        dt.free()
        dl.free()
    assert used < 7000
    assert len(f) == 6 * (N // 4) and st.survivors >= len(f)
    f0, t0, s0 = O.edges(t, ls, 0.95, 200, rows=(0, 8))
    k = f < 8
    assert set(zip(f[k].tolist(), to[k].tolist())) == set(zip(f0.tolist(), t0.tolist()))
