"""GPU: the tiled attention of consecutive rows against the one-token path.

Windows of consecutive positions that begin and end inside tiles of 16, cross
chunk boundaries and the positions where the chunk size grows (every 2048), at
both head sizes of the tiled kernel and every group size: each window's keys,
values and last logits must be the bits of feeding its tokens one at a time.
"""
import numpy as np
import pytest

from defer_amd import gpu as G
from defer_amd import synthetic

pytestmark = pytest.mark.gpu

# (heads, kv heads, head_dim): groups of 3, 1, 4 and 2
SHAPES = [(6, 2, 64), (2, 2, 64), (4, 1, 128), (2, 1, 128)]
WINDOWS = [(0, 16), (0, 17), (0, 300), (5, 130), (120, 20), (127, 2), (128, 1), (1000, 1100), (2040, 24),
           (2048, 16), (2047, 33), (4090, 300), (4096, 17), (6100, 90), (6143, 18), (7000, 1100)]


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
def test_windows_equal_token_by_token(shape):
    nh, nkv, hd = shape
    cfg = synthetic._cfg(64, 128, 128, 2, nh, nkv, hd, 10000.0, False, max_seq=8192)
    m = G.GpuModel(G.Config.from_dict(cfg), synthetic.make_weights(cfg, 3, std=0.15))
    toks = synthetic.make_prompt(64, 8192, seed=nh)
    ref = m.new_cache(8192)
    m.set_batching(0)
    m.prompt(ref, toks[:8190])
    want = [ref.read(l) for l in range(2)]
    m.set_batching(1)
    for start, n in WINDOWS:
        print(f"{shape} positions {start}..{start + n - 1}", flush=True)
        c = ref.clone()
        c.truncate(start)
        m.prompt(c, toks[start:start + n])
        for l in range(2):
            for got, exp in zip(c.read(l), want[l]):
                assert np.array_equal(bits(got[start:]), bits(exp[start:start + n])), (start, n, l)
        got = c.last_logits()
        c.truncate(start + n - 1)
        assert np.array_equal(bits(got), bits(m.forward(int(toks[start + n - 1]), c))), (start, n)
        c.close()
