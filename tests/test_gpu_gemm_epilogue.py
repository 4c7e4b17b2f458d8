"""Epilogues of the prefill GEMMs (outputs and aux four columns to a lane)
against the CPU oracle: every weight type, epilogue and activation type, a
last row block of one row, a last column block with few live tiles, and
outputs and aux whose address is aligned to one element only.  Bar: max
row-relative error 1e-3, the one fp16 rounding of the activations and of the
tile weights (2^-11 each) over at least 256 outputs of a row."""
import numpy as np
import pytest
import torch

from q4k_ref import TYPE_IQ4_XS, TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, make_q4k, make_weight, make_x, row_rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-3


def _buffer(m, n, dtype, gpu, shift):
    """A contiguous [m, n] tensor `shift` elements into its allocation."""
    return torch.full((m * n + shift,), float("nan"), device=gpu, dtype=dtype)[shift:].view(m, n)


@pytest.mark.parametrize("post,dtype,shift", [(0, torch.float32, 0), (1, torch.float32, 1), (2, torch.float32, 0), (0, torch.float16, 1),
                                              (1, torch.float16, 0), (2, torch.float16, 3)])
@pytest.mark.parametrize("t", [TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, TYPE_IQ4_XS])
def test_epilogue(q4k, oracle, gpu, t, post, dtype, shift):
    m, n, k = 1025, 2064, 256  # 9 row blocks x 33 blocks of 64 columns: past the middle row counts' form
    rng = np.random.default_rng(7800 + t + post)
    npdt = np.float16 if dtype == torch.float16 else np.float32
    w = make_weight(rng, n, k, t)
    x = make_x(rng, m, k, 0.25).astype(npdt)
    aux = make_x(rng, m, n, 2.0).astype(npdt)
    W = q4k.Weight(w, n, k, ggml_type=t)
    y, a = _buffer(m, n, dtype, gpu, shift), _buffer(m, n, dtype, gpu, shift)
    a.copy_(torch.from_numpy(aux))
    q4k.linear(torch.from_numpy(x).to(gpu), W, m, y, auxiliary=a if post else None, gated=post == 2, query_counts=[m])
    torch.cuda.synchronize()
    got = y.float().cpu().numpy()
    assert np.all(np.isfinite(got))
    ref = oracle.linear(x, w, n, k, aux=aux if post else None, post=post, ggml_type=t).astype(np.float32)
    assert row_rel_err(got, ref) <= TOL


@pytest.mark.parametrize("shift", [0, 1])
def test_gated_epilogue(q4k, gpu, shift):
    m, n, k = 1025, 2064, 256
    rng = np.random.default_rng(7900)
    G, U = q4k.Weight(make_q4k(rng, n, k), n, k), q4k.Weight(make_q4k(rng, n, k), n, k)
    x = torch.from_numpy(make_x(rng, m, k, 0.05)).to(gpu).half()
    y1, y2 = _buffer(m, n, torch.float16, gpu, 0), _buffer(m, n, torch.float16, gpu, shift)
    q4k.linear(x, G, m, y1, query_counts=[m])
    q4k.linear(x, U, m, y1, auxiliary=y1, gated=True, query_counts=[m])
    q4k.mlp_gate_up(x, G, U, m, y2, query_counts=[m])
    torch.cuda.synchronize()
    assert torch.isfinite(y2).all() and torch.equal(y1, y2)


@pytest.mark.parametrize("m,n,k,post", [(1500, 4096, 8192, 1), (1536, 4080, 8448, 0), (1408, 4096, 8192, 2)])
def test_narrowing_projection_in_segments(q4k, oracle, gpu, m, n, k, post):
    """Long K in two K-segments of unequal length, the short ones three to a
    workgroup (192 tiles on 256 CUs; 176 tiles stay whole): sampled rows against
    the oracle, the same bits from one call to the next (the segments' exchange),
    and the pair's one launch against the two calls."""
    rng = np.random.default_rng(7950 + m)
    w = make_q4k(rng, n, k)
    x, aux = make_x(rng, m, k, 0.1), make_x(rng, m, n, 2.0)
    W, U = q4k.Weight(w, n, k), q4k.Weight(make_q4k(rng, n, k), n, k)
    xt, at = torch.from_numpy(x).to(gpu), torch.from_numpy(aux).to(gpu)
    ys = [torch.full((m, n), float("nan"), device=gpu) for _ in range(3)]
    for y in ys:
        q4k.linear(xt, W, m, y, auxiliary=at if post else None, gated=post == 2, query_counts=[m])
    torch.cuda.synchronize()
    assert torch.equal(ys[0], ys[1]) and torch.equal(ys[0], ys[2])
    rows = np.r_[0:m:149, m - 1]
    ref = oracle.linear(x[rows], w, n, k, aux=aux[rows] if post else None, post=post)
    assert row_rel_err(ys[0].cpu().numpy()[rows], ref) <= TOL
    q4k.linear(xt, W, m, ys[0], query_counts=[m])
    q4k.linear(xt, U, m, ys[0], auxiliary=ys[0], gated=True, query_counts=[m])
    q4k.mlp_gate_up(xt, W, U, m, ys[1], query_counts=[m])
    torch.cuda.synchronize()
    assert torch.equal(ys[0], ys[1])
