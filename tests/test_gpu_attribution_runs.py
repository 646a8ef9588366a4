"""GPU: traced and masked forwards, and value norms, however they run.

A traced or masked forward runs as one persistent kernel; per-phase kernels
(eager mode) must give the same logits, cache rows and probabilities, bit for
bit. Value norms share W_o's reads among up to eight positions of a workgroup;
asking for them one position at a time must give the same bits.
"""
import numpy as np
import pytest

from defer_amd import gpu as G
from defer_amd import synthetic

pytestmark = pytest.mark.gpu

# heads, kv heads, head_dim, hidden, intermediate, biases
SHAPES = [(4, 2, 16, 64, 160, 0), (6, 2, 64, 192, 256, 1), (4, 1, 128, 320, 224, 0)]


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def model(shape):
    nh, nkv, hd, h, ff, bias = shape
    cfg = synthetic._cfg(90, h, ff, 3, nh, nkv, hd, 10000.0, True, max_seq=2200, bias=bias)
    return cfg, G.GpuModel(G.Config.from_dict(cfg), synthetic.make_weights(cfg, 21, std=0.1))


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_traced_and_masked_forwards_equal_the_phase_kernels(shape):
    cfg, m = model(shape)
    toks = synthetic.make_prompt(90, 2200, seed=5)
    ref = m.new_cache(2200)
    m.prompt(ref, toks[:2120])
    for ctx, mask in ((1, ()), (1, (0,)), (130, (0, 3, 127, 128)), (256, ()), (2050, tuple(range(40, 1900, 7)))):
        got = {}
        for mode in (G.EXEC_PERSISTENT, G.EXEC_EAGER, G.EXEC_GRAPH):
            print(f"{shape} ctx={ctx} mask={len(mask)} mode={mode}", flush=True)
            m.set_exec(mode)
            c = ref.clone()
            c.truncate(ctx)
            lg, tr = m.forward(7, c, masked=mask, trace=True)
            c.truncate(ctx)
            plain = m.forward(7, c, masked=mask)
            k, v = c.read(cfg["num_layers"] - 1)
            assert np.array_equal(bits(lg), bits(plain))
            assert np.all(tr[:, :, list(mask)] == 0.0)
            assert np.allclose(tr.sum(-1), 1.0, atol=(ctx + 1) * 2.0 ** -24)
            got[mode] = (bits(lg), bits(tr), bits(k), bits(v))
            c.close()
        m.set_exec(G.EXEC_PERSISTENT)
        for mode in (G.EXEC_EAGER, G.EXEC_GRAPH):
            for x, y in zip(got[G.EXEC_PERSISTENT], got[mode]):
                assert np.array_equal(x, y), (ctx, mode)


@pytest.mark.parametrize("name", ["smollm2-135m", "smollm2-360m", "llama-3.2-1b", "llama-3-8b"])
def test_traced_and_masked_forwards_at_the_specialised_shapes(name):
    """The shapes with a persistent kernel of their own, on the whole grid, one
    chunk and several: as the phase kernels, which are not specialised."""
    cfg = synthetic.CONFIGS[name]
    m = G.GpuModel(G.Config.from_dict(cfg), synthetic.make_weights(cfg, 5, threads=16))
    toks = synthetic.make_prompt(cfg["vocab_size"], 601, seed=2)
    c = m.new_cache(610)
    m.prompt(c, toks[:600])
    for ctx, mask in ((600, tuple(range(40, 500, 7))), (100, (0, 3, 99))):
        got = {}
        for mode in (G.EXEC_PERSISTENT, G.EXEC_EAGER):
            print(f"{name} ctx={ctx} mode={mode}", flush=True)
            m.set_exec(mode)
            out = []
            for kw in ({"trace": True}, {"trace": True, "masked": mask}, {"masked": mask}):
                c.truncate(ctx)
                r = m.forward(int(toks[600]), c, **kw)
                out += list(r) if isinstance(r, tuple) else [r]
                out += [x[ctx] for x in c.read(cfg["num_layers"] - 1)]
            got[mode] = [bits(x) for x in out]
            assert np.array_equal(got[mode][4], got[mode][8])  # tracing leaves the logits alone
        for x, y in zip(got[G.EXEC_PERSISTENT], got[G.EXEC_EAGER]):
            assert np.array_equal(x, y), ctx


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_value_norms_do_not_depend_on_how_many_are_asked_for(shape):
    cfg, m = model(shape)
    c = m.new_cache(64)
    m.prompt(c, synthetic.make_prompt(90, 40, seed=6))
    one = np.concatenate([c.value_norms(t, t + 1) for t in range(40)], axis=1)
    for t0, n in ((0, 2), (3, 3), (0, 7), (1, 8), (5, 9), (0, 40)):
        print(f"{shape} norms [{t0}, {t0 + n})", flush=True)
        assert np.array_equal(bits(c.value_norms(t0, t0 + n)), bits(one[:, t0:t0 + n]))
