"""Captures in a process whose workspace only one call has set up.

What a call finds in the workspace depends on every call before it, so these
cases need a fresh process: the parent test (test_gpu_capture.py) runs
``python capture_child.py CASE``.  Each case makes one eager call, captures
others (never called before) and compares every replay, with eager work and a
synchronisation in between, with the eager call of the same arguments made after
the capture: the same bits.  Exit status 0 means every check passed.
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import mtlqwen_amd as q4k  # noqa: E402
from q4k_ref import TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, make_weight, make_x  # noqa: E402

dev = torch.device("cuda:0")
rng = np.random.default_rng(9500)


def _x(m, k):
    return torch.from_numpy(make_x(rng, m, k, 0.25)).to(dev)


def _weight(t, n, k):
    return q4k.Weight(make_weight(rng, n, k, t), n, k, ggml_type=t)


def linear(t, m, n, k):
    W, x = _weight(t, n, k), _x(m, k)
    return f"linear {t} {m}x{k}->{n}", (m, n), lambda y: q4k.linear(x, W, m, y, query_counts=[1] * m if m <= 8 else [m])


def pair(t, m, n, k):
    G, U, x = _weight(t, n, k), _weight(t, n, k), _x(m, k)
    return f"pair {t} {m}x{k}->{n}", (m, n), lambda y: q4k.mlp_gate_up(x, G, U, m, y, query_counts=[1] * m if m <= 8 else [m])


def capture(call):
    name, shape, fn = call
    print("capture", name, flush=True)
    y = torch.empty(shape, device=dev)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.Stream()):
        fn(y)
    return g, y


def check(call):
    g, y = capture(call)
    ref = torch.empty_like(y)
    call[2](ref)
    torch.cuda.synchronize()
    assert torch.isfinite(ref).all()
    for _ in range(3):
        y.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref), call[0]
        call[2](torch.empty_like(y))


def eager(call):
    print("eager", call[0], flush=True)
    call[2](torch.empty(call[1], device=dev))
    torch.cuda.synchronize()


case = sys.argv[1]
if case == "prefill":
    # 512 rows of 4096 -> 4096 sum no K-slices, fewer rows do.
    eager(linear(TYPE_Q4_K, 512, 4096, 4096))
    for c in (linear(TYPE_Q4_K, 64, 4096, 4096), linear(TYPE_Q6_K, 100, 1024, 4096), pair(TYPE_Q4_K, 64, 1024, 4096),
              linear(TYPE_Q4_K, 40, 65552, 512), linear(TYPE_Q5_K, 63, 1024, 4096)):
        check(c)
elif case == "decode":
    # 8 rows of K = 4096 stage nothing; more rows and other K do.
    eager(linear(TYPE_Q6_K, 8, 1024, 4096))
    for c in (linear(TYPE_Q6_K, 40, 1024, 4096), pair(TYPE_Q5_K, 19, 1024, 4096), linear(TYPE_Q4_K, 40, 65552, 512), linear(TYPE_Q4_K, 8, 4096, 12288),
              linear(TYPE_Q6_K, 8, 1024, 12288), linear(TYPE_Q4_K, 64, 4096, 4096)):
        check(c)
else:
    # Nothing called yet: what needs a workspace is refused, what needs none is not.
    for c in (linear(TYPE_Q4_K, 64, 1024, 4096), linear(TYPE_Q6_K, 40, 1024, 4096), pair(TYPE_Q5_K, 19, 1024, 4096), linear(TYPE_Q4_K, 40, 65552, 512)):
        try:
            capture(c)
            raise SystemExit(f"{c[0]}: captured without a workspace")
        except q4k.Q4KError as e:
            assert e.code == q4k.ECAPTURE, (c[0], e.code, e.message)
    check(linear(TYPE_Q4_K, 8, 1024, 4096))
print("ok", flush=True)
