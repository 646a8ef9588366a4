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


@pytest.mark.parametrize("shape", SHAPES + [(4, 1, 256, 128, 128)], ids=lambda s: "x".join(map(str, s)))
def test_few_rows_with_long_histories_equal_single_steps(shape):
    """Few rows of many chunks: a group's chunks go to several workgroups (as
    many as the longest row's, fewer for a shorter one), past 8192 positions
    too; enough rows to fill the CUs without bring one workgroup each back."""
    nh, nkv, hd, h, ff = shape
    cfg = synthetic._cfg(200, h, ff, 2, nh, nkv, hd, 10000.0, True, max_seq=10400)
    m = G.GpuModel(G.Config.from_dict(cfg), synthetic.make_weights(cfg, 8, std=0.12))
    toks = synthetic.make_prompt(200, 10400, seed=hd)
    long = m.new_cache(10400)
    m.prompt(long, toks[:10300])
    for rows in ([10300, 3], [700, 640], [9000, 0, 10300, 2100, 130], [1000] * 24):
        print(f"{shape} rows={rows}", flush=True)
        A, B = [], []
        for n in rows:
            for side in (A, B):
                c = long.clone()
                c.truncate(n)
                side.append(c)
        for step in range(2):
            feed = toks[step:step + len(rows)]
            got = m.forward_batch(A, feed, logits=True)
            for i, (b, t) in enumerate(zip(B, feed)):
                assert np.array_equal(bits(got[i]), bits(m.forward(int(t), b))), (step, i, rows[i])
        for x, y in zip(A[0].read(1), B[0].read(1)):
            assert np.array_equal(bits(x), bits(y))
        for c in A + B:
            c.close()


def test_few_rows_with_long_histories_use_the_idle_compute_units():
    """Two rows of 16 chunks: each chunk has CUs of its own, so the attention
    takes about as long as over one chunk (1.05 times, measured) and not four
    rounds of it (3.5 times with a workgroup per row and kv head)."""
    cfg = synthetic._cfg(2000, 576, 1536, 12, 9, 3, 64, 10000.0, True, max_seq=2100)
    m = G.GpuModel(G.Config.from_dict(cfg), synthetic.make_weights(cfg, 8))
    toks = synthetic.make_prompt(2000, 2040, seed=1)
    ms = {}
    for n in (100, 2030):
        cs = [m.new_cache(2100), m.new_cache(2100)]
        for c in cs:
            m.prompt(c, toks[:n])
        m.set_profiling(True)
        best = []
        for _ in range(8):
            for c in cs:
                c.truncate(n)
            m.batch_stats()
            m.forward_batch(cs, [1, 2])
            best.append(m.batch_stats()["attn_ms"])
        m.set_profiling(False)
        ms[n] = min(best)
        for c in cs:
            c.close()
    print(ms, ms[2030] / ms[100], flush=True)
    assert ms[2030] < 2.5 * ms[100], ms


@pytest.mark.parametrize("rows", [1, 2, 5, 7, 40, 130])
def test_sampled_steps_equal_single_steps(rows):
    """A step's sampling ops share the CUs (several workgroups per op for few
    rows, one for many): the tokens are those of stepping each session alone."""
    cfg = synthetic._cfg(20000, 64, 96, 1, 2, 1, 32, 10000.0, True, max_seq=64)
    m = G.GpuModel(G.Config.from_dict(cfg), synthetic.make_weights(cfg, 9, std=0.3))
    rng = np.random.Generator(np.random.PCG64(rows))
    A, B = [], []
    for i in range(rows):
        a = m.new_cache(16)
        m.prompt(a, synthetic.make_prompt(20000, 1 + i % 3, seed=i))
        A.append(a)
        B.append(a.clone())
    for T in (0.05, 0.7, 1.0, 0.0, 8.0):
        print(f"rows={rows} T={T}", flush=True)
        words = rng.integers(0, 1 << 32, size=rows, dtype=np.uint32)
        words[0] = [0, 0xFFFFFFFF][rows % 2]
        got = m.step_batch(A, T, words)
        assert got == [m.step(b, T, int(w)) for b, w in zip(B, words)], T
