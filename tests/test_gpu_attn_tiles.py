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
    # a vocabulary of four 64-row chunks: the one-token path runs on four workgroups
    cfg = synthetic._cfg(250, 128, 128, 2, nh, nkv, hd, 10000.0, False, max_seq=8192)
    m = G.GpuModel(G.Config.from_dict(cfg), synthetic.make_weights(cfg, 3, std=0.15))
    toks = synthetic.make_prompt(250, 8192, seed=nh)
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


# first position, rows, the row with the odd token: in the first and in later
# tiles, in the tile's first, last and middle row, in chunks of 128 to 512
ODD = [(0, 40, 7), (0, 16, 15), (120, 30, 8), (120, 30, 16), (1000, 20, 2), (2040, 40, 12), (4090, 40, 10), (6150, 20, 9)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}x{s[2]}")
@pytest.mark.parametrize("value", ["nan", "inf"])
def test_rows_before_an_infinite_or_nan_value_row_are_untouched(shape, value):
    """A token whose value row holds NaNs, or one infinity beside finite keys:
    the rows before it in its tile do not see it. Every row's logits must be
    those of feeding the tokens one at a time (NaN where those are NaN)."""
    nh, nkv, hd = shape
    V, h, odd = 200, 128, 199
    cfg = synthetic._cfg(V, h, 128, 2, nh, nkv, hd, 10000.0, False, max_seq=8192)
    w = synthetic.make_weights(cfg, 3, std=0.15)
    embed, wv = w[0], w[4]  # layer 0: norm, q, k, v
    if value == "nan":
        embed[odd, 3] = np.nan
    else:  # element 5 of the hidden row is this token's alone, and reaches one value of each head
        embed[:, 5] = 0.0
        embed[odd, 5] = 10.0
        for t in w[2:4]:
            t[:, 5] = 0.0
        wv[:, 5] = 0.0
        wv[hd - 3::hd, 5] = 3e38
    m = G.GpuModel(G.Config.from_dict(cfg), w)
    toks = synthetic.make_prompt(odd, 8192, seed=nh)
    ref = m.new_cache(8192)
    m.prompt(ref, toks[:6200])
    for start, n, at in ODD:
        print(f"{shape} {value} positions {start}..{start + n - 1}, odd row {at}", flush=True)
        feed = toks[start:start + n].copy()
        feed[at] = odd
        a, b = ref.clone(), ref.clone()
        a.truncate(start)
        b.truncate(start)
        got = m.forward_batch([a] * n, feed, logits=True)
        for i, t in enumerate(feed):
            want = m.forward(int(t), b)
            assert np.all(np.isfinite(want)) == (i < at), (start, i)
            same = (bits(got[i]) == bits(want)) | (np.isnan(got[i]) & np.isnan(want))
            assert np.all(same), (start, i)
        a.close()
        b.close()
