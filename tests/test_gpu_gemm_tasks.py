"""GPU: the batched matrix products' task shapes against the one-token path.

The task shape of a product (4x2, 2x2, 2x1 or 1x1 tiles of 16) follows from the
rows, the columns and the compute units the launch is shaped for; every shape
must give each output the one-token order's bits, whatever the product writes
(plain rows, the residual, logits, rotated queries and cache rows, activations). The compute-unit count is
forced so that each shape is chosen, at row counts on both sides of the tile
edges, with dimensions that are not whole tiles or whole 64-element chunks.
"""
import numpy as np
import pytest

from defer_amd import gpu as G
from defer_amd import synthetic

pytestmark = pytest.mark.gpu

SHAPES = {
    # hidden, intermediate, heads, kv heads, head_dim, vocabulary, activation, biases
    "whole-chunks": (128, 192, 4, 2, 32, 250, 0, 0),
    "odd-tiles": (192, 320, 3, 1, 64, 331, 0, 0),
    "biases-gelu": (128, 144, 2, 1, 128, 90, 1, 1),
    "partial-chunks": (96, 200, 6, 2, 16, 77, 0, 1),
    "partial-chunks-tiled": (96, 208, 3, 1, 64, 77, 0, 1),
}


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("cus", [1, 3, 16, 0])
def test_rows_equal_single_forwards_for_every_task_shape(shape, cus):
    h, ff, nh, nkv, hd, V, act, bias = SHAPES[shape]
    cfg = synthetic._cfg(V, h, ff, 2, nh, nkv, hd, 10000.0, False, max_seq=256,
                         act=act, bias=bias)
    m = G.GpuModel(G.Config.from_dict(cfg), synthetic.make_weights(cfg, 11, std=0.08))
    m.set_grid(0, cus)
    rng = np.random.Generator(np.random.PCG64(cus))
    toks = rng.integers(0, V, size=131, dtype=np.uint32)
    ref = m.new_cache(256)
    want = np.stack([m.forward(int(t), ref) for t in toks])
    for n in (1, 7, 15, 16, 17, 31, 33, 64, 65, 131):
        print(f"{shape} cus={cus} rows={n}", flush=True)
        c = m.new_cache(256)
        got = m.forward_batch([c] * n, toks[:n], logits=True)
        assert np.array_equal(got.view(np.uint32), want[:n].view(np.uint32)), n
        c.close()
