"""GPU: the lockstep rows' attention (one workgroup per row and kv head).

Sessions of very different lengths stepped together -- an empty one, lengths
around the edges of a chunk and of the positions where the chunk grows -- must
each get the bits of stepping alone, however many teams share a workgroup
(which follows from the rows and the longest row's chunks), at every head
size and group.
"""
import numpy as np
import pytest

from defer_amd import gpu as G
from defer_amd import synthetic

pytestmark = pytest.mark.gpu

# (heads, kv heads, head_dim, hidden, intermediate)
SHAPES = [(6, 2, 64, 128, 128), (4, 1, 128, 128, 200), (8, 2, 32, 96, 160), (2, 2, 16, 64, 96)]
LENGTHS = [0, 1, 16, 127, 128, 129, 255, 300, 600, 1100, 2046, 2047, 2048, 2049, 2600, 4090, 4096]


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_rows_of_distinct_caches_equal_single_steps(shape):
    nh, nkv, hd, h, ff = shape
    cfg = synthetic._cfg(80, h, ff, 2, nh, nkv, hd, 10000.0, True, max_seq=4200)
    m = G.GpuModel(G.Config.from_dict(cfg), synthetic.make_weights(cfg, 7, std=0.12))
    toks = synthetic.make_prompt(80, 4200, seed=hd)
    long = m.new_cache(4200)
    m.prompt(long, toks[:4100])
    for rows in (LENGTHS[:1], LENGTHS[2:4], LENGTHS[:7], LENGTHS[3:], LENGTHS * 3):
        print(f"{shape} rows={rows}", flush=True)
        A, B = [], []
        for n in rows:
            for side in (A, B):
                c = long.clone()
                c.truncate(n)
                side.append(c)
        feed = toks[: len(rows)]
        got = m.forward_batch(A, feed, logits=True)
        for i, (b, t) in enumerate(zip(B, feed)):
            assert np.array_equal(bits(got[i]), bits(m.forward(int(t), b))), (i, rows[i])
        # a second step reads the rows the first one wrote
        got = m.forward_batch(A, feed[::-1].copy(), logits=True)
        for i, (a, b, t) in enumerate(zip(A, B, feed[::-1])):
            assert np.array_equal(bits(got[i]), bits(m.forward(int(t), b))), (i, rows[i])
            if i % 5 == 0:
                for l in range(2):
                    for x, y in zip(a.read(l), b.read(l)):
                        assert np.array_equal(bits(x), bits(y)), (i, l)
        for c in A + B:
            c.close()
