"""The pipelined prefill GEMMs (q4k_gemm2_kernel, typed_gemm_kernel) over
several blocks of K, at row counts past the middle GEMM's: every weight type at
the widths where each of its tilings is taken on 256 CUs (128, 192, 256 and 384
columns per workgroup), with a ragged last column block.  The identity as x
reads every dequantised weight out, bit for bit; random x, with and without the
norm in its staging, meets the oracle within 1e-3 (one fp16 rounding of the
activations and of the tile weights, 2^-11 each, over 1024 outputs of a row and
more)."""
import numpy as np
import pytest
import torch

from q4k_ref import TYPE_IQ4_XS, TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, make_weight, make_x, row_rel_err

pytestmark = pytest.mark.gpu
TYPES = [TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, TYPE_IQ4_XS]
WIDTHS = [1040, 3056, 4080, 6128]


def _past_middle(m, n):
    """Whether the 128 x 64 tiles of the middle GEMM would take more than one round."""
    return (n + 63) // 64 * ((m + 127) // 128) > torch.cuda.get_device_properties(0).multi_processor_count


@pytest.mark.parametrize("n", WIDTHS)
@pytest.mark.parametrize("t", TYPES)
def test_dequant_bit_exact(q4k, oracle, gpu, t, n):
    """y of the identity is the transposed weight: each element the oracle's
    fp32 value rounded once to fp16 (times 1, plus zeros)."""
    k = m = 2048
    assert _past_middle(m, n)
    w = make_weight(np.random.default_rng(8100 + t), n, k, t)
    W = q4k.Weight(w, n, k, ggml_type=t)
    y = torch.full((m, n), float("nan"), device=gpu)
    q4k.linear(torch.eye(m, device=gpu), W, m, y, query_counts=[m])
    torch.cuda.synchronize()
    blocks = w.reshape(n * (k // 256), -1)
    expect = np.stack([oracle.dequant_block(b, t) for b in blocks]).reshape(n, k).astype(np.float16).astype(np.float32)
    got = y.cpu().numpy().T
    assert np.all(np.isfinite(got))
    bad = np.argwhere(got != expect)  # exact (a zero weight may carry either sign)
    assert bad.size == 0, f"type={t}: {len(bad)} weights differ, first (column, k) {bad[:4].tolist()}"


@pytest.mark.parametrize("m,n,k,post,norm,dtype", [(2047, 1040, 768, 1, False, torch.float32), (2047, 1040, 2816, 0, True, torch.float16),
                                                   (1921, 4080, 512, 2, False, torch.float16), (1921, 4080, 1280, 0, True, torch.float32)])
@pytest.mark.parametrize("t", TYPES)
def test_against_oracle(q4k, oracle, gpu, t, m, n, k, post, norm, dtype):
    assert _past_middle(m, n)
    rng = np.random.default_rng(8200 + t + k)
    npdt = np.float16 if dtype == torch.float16 else np.float32
    w = make_weight(rng, n, k, t)
    x = make_x(rng, m, k, 0.25).astype(npdt)
    aux = make_x(rng, m, n, 2.0).astype(npdt)
    nw = (0.2 * (1.0 + 0.2 * rng.standard_normal(k))).astype(np.float32)
    W = q4k.Weight(w, n, k, ggml_type=t)
    y = torch.from_numpy(aux).to(gpu) if post else torch.full((m, n), float("nan"), device=gpu, dtype=dtype)
    xt, kw = torch.from_numpy(x).to(gpu), dict(auxiliary=y if post else None, gated=post == 2, query_counts=[m])
    if norm:
        q4k.linear_norm(xt, W, torch.from_numpy(nw).to(gpu), m, y, **kw)
    else:
        q4k.linear(xt, W, m, y, **kw)
    torch.cuda.synchronize()
    got = y.float().cpu().numpy()
    assert np.all(np.isfinite(got))
    rows = np.r_[0:m:97, m - 128 : m]  # some of every row block, all of the ragged last one
    xr = oracle.rms_norm(x[rows].astype(np.float32), nw) if norm else x[rows]
    ref = oracle.linear(xr, w, n, k, aux=aux[rows] if post else None, post=post, ggml_type=t).astype(np.float32)
    assert row_rel_err(got[rows], ref) <= 1e-3


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_two_halves_of_k(q4k, oracle, gpu, dtype):
    """Long K on few tiles: two K-halves to a tile (81 tiles of 256 columns), the
    pair's one launch with the bits of the two calls."""
    m, n, k = 1025, 2064, 8192
    assert _past_middle(m, n)
    rng = np.random.default_rng(8300)
    npdt = np.float16 if dtype == torch.float16 else np.float32
    w = make_weight(rng, n, k, TYPE_Q4_K)
    x = make_x(rng, m, k, 0.02).astype(npdt)
    G, U = q4k.Weight(w, n, k), q4k.Weight(make_weight(rng, n, k, TYPE_Q4_K), n, k)
    xt = torch.from_numpy(x).to(gpu)
    y1, y2 = (torch.full((m, n), float("nan"), device=gpu, dtype=dtype) for _ in range(2))
    q4k.linear(xt, G, m, y1, query_counts=[m])
    torch.cuda.synchronize()
    rows = np.r_[0:m:97, m - 1]
    got = y1.float().cpu().numpy()[rows]
    assert row_rel_err(got, oracle.linear(x[rows], w, n, k).astype(np.float32)) <= 1e-3
    q4k.linear(xt, U, m, y1, auxiliary=y1, gated=True, query_counts=[m])
    q4k.mlp_gate_up(xt, G, U, m, y2, query_counts=[m])
    torch.cuda.synchronize()
    assert torch.isfinite(y2).all() and torch.equal(y1, y2)
