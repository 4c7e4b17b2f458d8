"""Prefill GEMMs of the middle row counts (mid_gemm_kernel: 64-column tiles,
K in slices over the idle CUs) against the CPU oracle, at the edges of their
tiles: one row above and below the 64- and 128-row blocks, a last column block
of one live tile, K of one to three blocks (one slice; slices of unequal
length), every weight type, epilogue and activation type; the gated form
against the two calls; a capture after the same call (test_gpu_capture.py has
those after other calls).  Bar: max row-relative error 1e-3, the one fp16
rounding of the activations and of the tile weights (2^-11 each) over at least
256 outputs of a row."""
import numpy as np
import pytest
import torch

from q4k_ref import TYPE_IQ4_XS, TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, make_q4k, make_weight, make_x, row_rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-3
TYPES = [TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, TYPE_IQ4_XS]

# (m, n, k, post, dtype)
SHAPES = [(64, 1024, 256, 0, torch.float32), (65, 272, 512, 1, torch.float32), (127, 1040, 768, 2, torch.float32), (128, 512, 4096, 0, torch.float16),
          (129, 1296, 1280, 1, torch.float16), (511, 272, 2816, 0, torch.float32)]


@pytest.mark.parametrize("m,n,k,post,dtype", SHAPES)
@pytest.mark.parametrize("t", TYPES)
def test_mid_gemm(q4k, oracle, gpu, t, m, n, k, post, dtype):
    rng = np.random.default_rng(7100 + m + n + t)
    npdt = np.float16 if dtype == torch.float16 else np.float32
    w = make_weight(rng, n, k, t)
    x = make_x(rng, m, k, 0.25).astype(npdt)
    aux = make_x(rng, m, n, 2.0).astype(npdt) if post else None
    W = q4k.Weight(w, n, k, ggml_type=t)
    y = torch.from_numpy(aux).to(gpu) if post else torch.full((m, n), float("nan"), device=gpu, dtype=dtype)
    q4k.linear(torch.from_numpy(x).to(gpu), W, m, y, auxiliary=y if post else None, gated=post == 2, query_counts=[m])
    torch.cuda.synchronize()
    got = y.float().cpu().numpy()
    assert np.all(np.isfinite(got))
    ref = oracle.linear(x, w, n, k, aux=aux, post=post, ggml_type=t).astype(np.float32)
    assert row_rel_err(got, ref) <= TOL


@pytest.mark.parametrize("m,n,k", [(49, 256, 256), (64, 1040, 4096), (128, 12288, 512)])
def test_gated_matches_two_calls(q4k, gpu, m, n, k):
    rng = np.random.default_rng(7200 + m)
    G, U = q4k.Weight(make_q4k(rng, n, k), n, k), q4k.Weight(make_q4k(rng, n, k), n, k)
    x = torch.from_numpy(make_x(rng, m, k, 0.1)).to(gpu)
    y1, y2 = (torch.full((m, n), float("nan"), device=gpu) for _ in range(2))
    q4k.linear(x, G, m, y1, query_counts=[m])
    q4k.linear(x, U, m, y1, auxiliary=y1, gated=True, query_counts=[m])
    q4k.mlp_gate_up(x, G, U, m, y2, query_counts=[m])
    torch.cuda.synchronize()
    assert torch.isfinite(y2).all() and torch.equal(y1, y2)


def test_capture_replays(q4k, gpu):
    """K-slices inside a HIP graph: every replay, with eager work between,
    gives the eager call's output."""
    m, n, k = 96, 1024, 4096
    rng = np.random.default_rng(7300)
    W = q4k.Weight(make_q4k(rng, n, k), n, k)
    x = torch.from_numpy(make_x(rng, m, k)).to(gpu)
    y_ref, y = torch.empty((m, n), device=gpu), torch.empty((m, n), device=gpu)
    q4k.linear(x, W, m, y_ref, query_counts=[m])
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.Stream()):
        q4k.linear(x, W, m, y, query_counts=[m])
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, y_ref)
        q4k.linear(x * 0.5, W, m, torch.empty_like(y), query_counts=[m])
