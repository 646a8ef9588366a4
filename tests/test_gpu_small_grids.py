"""GPU: grids so small that a workgroup owns more rows than it has threads.

A vocabulary of one or two 64-row chunks, or a grid set by hand, leaves the
one-token path with one or two workgroups. Their logits must be the batched
path's bits and the oracle's to rounding, in every execution mode, with hidden
sizes on both sides of one row per thread.
"""
import numpy as np
import pytest

import oracle_py as O
from defer_amd import gpu as G
from defer_amd import synthetic

pytestmark = pytest.mark.gpu

# vocabulary, hidden, grid set by hand (0: as the model has it)
GRIDS = [(64, 380, 0), (64, 384, 0), (64, 388, 0), (64, 512, 0), (64, 516, 0), (64, 576, 0), (64, 1024, 0),
         (128, 2048, 0), (250, 576, 1), (250, 1160, 2)]


@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "V%d-h%d-G%d" % g)
def test_one_token_path_equals_the_batched_path_and_the_oracle(grid):
    V, h, g = grid
    cfg = synthetic._cfg(V, h, 96, 2, 2, 1, 16, 10000.0, True, max_seq=64)
    w = synthetic.make_weights(cfg, V + h, std=0.1)
    m, om = G.GpuModel(G.Config.from_dict(cfg), w), O.OracleModel(cfg, w)
    if g:
        m.set_grid(g, 0)
    toks = synthetic.make_prompt(V, 20, seed=h)
    c, oc = m.new_cache(), om.new_cache()
    want = m.forward_batch([c] * len(toks), toks, logits=True)
    for t, row in zip(toks, want):
        ref = om.forward(int(t), oc)
        # The oracle adds a product's h terms one after another: up to h
        # roundings of 2^-24 each (measured 1.6e-5 of the largest logit at
        # h = 2048, where this allows 1.2e-4).
        assert np.max(np.abs(row - ref)) <= h * 2.0 ** -24 * np.max(np.abs(ref)), "batched against the oracle"
    for mode in (G.EXEC_PERSISTENT, G.EXEC_GRAPH, G.EXEC_EAGER):
        print(f"{grid} mode={mode}", flush=True)
        m.set_exec(mode)
        x = m.new_cache()
        for i, t in enumerate(toks):
            got = m.forward(int(t), x)
            assert np.array_equal(got.view(np.uint32), want[i].view(np.uint32)), (mode, i)
        x.close()
