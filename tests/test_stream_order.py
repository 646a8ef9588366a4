"""Host path: what the library queues, on which stream, and what it waits for.

The library is loaded over a stand-in for the HIP runtime (tests/probe/fake_hip.c:
device memory is host memory, kernels do nothing) that keeps which stream still
has unfinished work, in a child process, so that no GPU is needed and the real
runtime is not in the way. The model's stream does not block on the null stream:
work queued on one while the other's is unfinished is in no order.
"""
import ctypes
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["gcc", "-O1", "-Wall", "-shared", "-fPIC", "-I/opt/rocm/include", "-o", out,
                    os.path.join(ROOT, "tests", "probe", "fake_hip.c")], check=True)
    return out


def child(fake, check):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), fake, check], cwd=ROOT,
                       env=dict(os.environ, PYTHONPATH=ROOT), capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip().endswith("ok"), r.stdout + r.stderr


def test_a_clone_is_ordered_before_the_next_call(fake):
    """... and so is what a call itself hands over: a mask, a stop list, a new
    cache's or model's memory."""
    child(fake, "clone")


def check_clone(hip, G, m, cfg, w):
    c = m.new_cache(64)
    m.prompt(c, list(range(20)))  # batched: the cache's length is the host's
    calls = {
        "forward": lambda x: m.forward(1, x),
        "truncate + forward": lambda x: (x.truncate(10), m.forward(1, x)),
        "masked, traced forward": lambda x: m.forward(1, x, masked=[2], trace=True),
        "prompt": lambda x: m.prompt(x, [3] * 20),
        "forward_batch": lambda x: m.forward_batch([x, m.new_cache(64)], [1, 2]),
        "step_batch": lambda x: m.step_batch([x, c], 0.7, [1, 2]),
        "generate": lambda x: m.generate(x, 2, 0.7, [1, 2], stop=[4]),
        "value_norms": lambda x: x.value_norms(0, 5),
        "read": lambda x: x.read(0),
        "set_logits": lambda x: x.set_logits([0.0] * cfg["vocab_size"]),
        "the source": lambda x: m.forward_batch([c], [1]),
        "a new cache": lambda x: m.forward(1, m.new_cache(8)),
        "a new model": lambda x: G.GpuModel(m.cfg, w).new_cache(8).clone(),
    }
    bad = []
    for name, call in calls.items():
        before = hip.fake_unordered()
        x = c.clone()
        if hip.fake_pending():
            bad.append("clone, unfinished on return, before " + name)
        try:
            call(x)
        except G.DeferGpuError as e:  # no kernel ran: nothing was sampled
            print(name, e)
        if hip.fake_unordered() != before:
            bad.append(name)
        x.close()
    assert not bad, bad


def test_a_failed_call_leaves_nothing_running(fake):
    """A copy that fails ends the call with an error and the stream idle, so
    that nothing writes the caller's arrays afterwards; the cache keeps its
    length, and its logits unless they may be overwritten."""
    child(fake, "failure")


def check_failure(hip, G, m, cfg, w):
    # per call the copies it makes on the stream, in order: whether the cache
    # still has its logits when that copy fails
    calls = {
        # the run's state, the probabilities, the logits: the run has written its own
        "forward": ([False, False, False], lambda a, b: m.forward(1, a, trace=True)),
        # the rows, the run's state, the logits, the list of caches to commit
        "forward_batch": ([True, True, True, False], lambda a, b: m.forward_batch([a, b], [1, 2], logits=True)),
    }
    bad = []
    for name, (keeps, call) in calls.items():
        for k, keep in enumerate(keeps):
            a, b = m.new_cache(64), m.new_cache(64)
            for c in (a, b):
                m.prompt(c, list(range(20)))
            hip.fake_fail_in(k + 1)
            try:
                call(a, b)
                bad.append((name, k, "no error"))
            except G.DeferGpuError:
                pass
            hip.fake_fail_in(0)
            if hip.fake_pending():
                bad.append((name, k, "still running"))
            assert len(a) == 20
            try:
                a.last_logits()
                kept = True
            except G.DeferGpuError:
                kept = False
            if kept != keep:
                bad.append((name, k, "logits kept" if kept else "logits lost"))
            a.close()
            b.close()
    assert not bad, bad


if __name__ == "__main__":
    hip = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # found before the real runtime
    hip.fake_unordered.restype = ctypes.c_long
    from defer_amd import gpu as G
    from defer_amd import synthetic

    cfg = synthetic.CONFIGS["tiny"]
    weights = synthetic.make_weights(cfg, 1)
    model = G.GpuModel(G.Config.from_dict(cfg), weights)
    {"clone": check_clone, "failure": check_failure}[sys.argv[2]](hip, G, model, cfg, weights)
    print("ok")
