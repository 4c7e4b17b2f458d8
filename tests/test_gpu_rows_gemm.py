"""9 to 63 rows of the other weight types in one GEMM with hi/lo activations
(rows_gemm_kernel) against the CPU oracle at the edges of its row tiles (16
rows), column blocks (128 columns, 64 gated) and K-slices (one block; an odd
count of blocks), with more column blocks than CUs (several items per
workgroup), every type, epilogue and activation type.
Bars: Q5_K products are exact and the activations keep 22 bits, so fp32
outputs stay within 1e-5 (fp32 sums in another order); the other types round
each product once to fp16 (2^-11 = 4.9e-4 at most for a whole row); fp16
outputs add their own rounding, 1e-3 in all."""
import numpy as np
import pytest
import torch

from q4k_ref import TYPE_IQ4_XS, TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, dequant_numpy, make_q4k, make_weight, make_x, row_rel_err

pytestmark = pytest.mark.gpu
TYPES = [TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, TYPE_IQ4_XS]


def _bar(t, dtype):
    return 1e-3 if dtype == torch.float16 else 1e-5 if t == TYPE_Q5_K else 4.9e-4


# (m, n, k, post, dtype)
SHAPES = [(9, 16, 256, 0, torch.float32), (16, 144, 768, 1, torch.float32), (17, 1040, 4096, 2, torch.float32), (32, 512, 1280, 0, torch.float16),
          (33, 272, 2816, 1, torch.float16), (48, 256, 512, 0, torch.float32), (49, 34816, 256, 0, torch.float32), (63, 1024, 4096, 1, torch.float32)]


@pytest.mark.parametrize("m,n,k,post,dtype", SHAPES)
@pytest.mark.parametrize("t", TYPES)
def test_rows_gemm(q4k, oracle, gpu, t, m, n, k, post, dtype):
    rng = np.random.default_rng(7500 + m + n + t)
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
    assert row_rel_err(got, ref) <= _bar(t, dtype)


@pytest.mark.parametrize("m,n,k,counts", [(9, 80, 512, [9]), (40, 1040, 4096, [5] * 8), (63, 17408, 256, [63])])
@pytest.mark.parametrize("t", TYPES)
def test_rows_gemm_gated(q4k, oracle, gpu, t, m, n, k, counts):
    rng = np.random.default_rng(7600 + m + n + t)
    wg, wu = make_weight(rng, n, k, t), make_weight(rng, n, k, t)
    x = make_x(rng, m, k, 0.05)
    G, U = q4k.Weight(wg, n, k, ggml_type=t), q4k.Weight(wu, n, k, ggml_type=t)
    y = torch.full((m, n), float("nan"), device=gpu)
    nw = torch.ones(k, device=gpu)
    q4k.mlp_gate_up(torch.from_numpy(x).to(gpu), G, U, m, y, query_counts=counts)
    torch.cuda.synchronize()
    # Two projections' errors meet in each output.
    assert row_rel_err(y.cpu().numpy(), oracle.mlp_gate_up(x, wg, wu, n, k, ggml_type=t)) <= 2 * _bar(t, torch.float32)
    # The norm folded into the staging (all-ones weight) against the same norm done first.
    y1, y2, h = torch.empty_like(y), torch.empty_like(y), torch.from_numpy(x * 30.0).to(gpu)
    hn = torch.empty_like(h)
    q4k.rms_norm(h, nw, hn)
    q4k.linear(hn, G, m, y1, query_counts=counts)
    q4k.linear_norm(h, G, nw, m, y2, query_counts=counts)
    torch.cuda.synchronize()
    assert row_rel_err(y2.cpu().numpy(), y1.cpu().numpy()) <= 1e-5


def test_rows_gemm_capture(q4k, gpu):
    """The rows GEMM inside a HIP graph: every replay, with eager work between,
    gives the eager call's output."""
    m, n, k = 24, 512, 1024
    rng = np.random.default_rng(7700)
    W = q4k.Weight(make_weight(rng, n, k, TYPE_Q6_K), n, k, ggml_type=TYPE_Q6_K)
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


@pytest.mark.parametrize("t,m,n,k,launches", [(TYPE_Q6_K, 16, 1024, 1024, 2), (TYPE_IQ4_XS, 9, 4096, 2048, 2), (TYPE_Q6_K, 12, 256, 768, 2),
                                              (TYPE_Q6_K, 17, 1024, 1024, 1), (TYPE_IQ4_XS, 16, 256, 512, 1), (TYPE_IQ4_XS, 9, 144, 2304, 2), (TYPE_Q6_K, 16, 144, 2560, 1),
                                              (TYPE_IQ4_XS, 16, 4112, 2048, 1), (TYPE_Q5_K, 16, 1024, 1024, 1), (TYPE_Q8_0, 16, 512, 2048, 1)])
def test_few_rows_of_short_k(q4k, oracle, gpu, t, m, n, k, launches):
    """9 to 16 rows at the edges of the sizes that keep one GEMV per 8 rows:
    `launches` of the GEMV family."""
    rng = np.random.default_rng(7800 + m + n + k)
    w = make_weight(rng, n, k, t)
    W = q4k.Weight(w, n, k, ggml_type=t)
    x = make_x(rng, m, k, 0.25)
    y, xt = torch.full((m, n), float("nan"), device=gpu), torch.from_numpy(x).to(gpu)
    torch.cuda.synchronize()
    q4k.profile_enable(True)
    q4k.linear(xt, W, m, y, query_counts=[m])
    torch.cuda.synchronize()
    got = q4k.profile_query(q4k.KERNEL_GEMV)[0]
    q4k.profile_enable(False)
    assert got == launches
    assert row_rel_err(y.cpu().numpy(), oracle.linear(x, w, n, k, ggml_type=t)) <= _bar(t, torch.float32)


def _first_wide():
    """The fewest Q4_K outputs that take the rows GEMM (16 column tiles per CU), and a tile."""
    return 16 * (16 * torch.cuda.get_device_properties(0).multi_processor_count + 1)


@pytest.mark.parametrize("m,k,post,dtype", [(9, 512, 0, torch.float32), (17, 256, 1, torch.float32), (32, 768, 2, torch.float16), (33, 1280, 2, torch.float32),
                                            (48, 512, 1, torch.float16), (48, 512, 0, torch.float32), (49, 512, 0, torch.float32)])
def test_wide_q4k(q4k, oracle, gpu, m, k, post, dtype):
    """Wide Q4_K outputs, several items to a workgroup and a last column block
    of one tile: 9 to 48 rows on the rows GEMM (beyond 24 rows only it keeps 22
    bits of the activations), 49 on the prefill GEMM."""
    n = _first_wide()
    rng = np.random.default_rng(7900 + m + k)
    npdt = np.float16 if dtype == torch.float16 else np.float32
    w = make_q4k(rng, n, k)
    x = make_x(rng, m, k, 0.05).astype(npdt)
    aux = make_x(rng, m, n, 2.0).astype(npdt) if post else None
    W = q4k.Weight(w, n, k)
    y = torch.from_numpy(aux).to(gpu) if post else torch.full((m, n), float("nan"), device=gpu, dtype=dtype)
    xt = torch.from_numpy(x).to(gpu)
    torch.cuda.synchronize()
    q4k.profile_enable(True)
    q4k.linear(xt, W, m, y, auxiliary=y if post else None, gated=post == 2, query_counts=[m])
    torch.cuda.synchronize()
    launches = [q4k.profile_query(f)[0] for f in (q4k.KERNEL_STAGE, q4k.KERNEL_GEMV, q4k.KERNEL_GEMM)]
    q4k.profile_enable(False)
    assert launches == ([1, 1, 0] if m <= 48 else [1, 0, 1])
    got = y.float().cpu().numpy()
    assert np.all(np.isfinite(got))
    ref = oracle.linear(x, w, n, k, aux=aux, post=post).astype(np.float32)
    assert row_rel_err(got, ref) <= (1e-3 if dtype == torch.float16 or m > 48 else 1e-5)


@pytest.mark.parametrize("m", [9, 24])
def test_wide_q4k_sums(q4k, gpu, m):
    """The error against 64 bits of a wide Q4_K projection's first outputs is
    that of the same rows of a narrow one (the staged GEMV, whose waves sum one
    or two blocks each), within 5 %: both keep hi/lo activations, and the sums
    over all of K in one workgroup are made as short.  Weights about zero, as
    trained ones: the unsigned quants' part and the min part of a sum are each
    larger than the result."""
    n, narrow, k = _first_wide(), 2048, 4096
    rng = np.random.default_rng(7950)
    w = rng.integers(0, 256, (n, k // 256, 144), dtype=np.uint8)
    d = ((0.5 + rng.random((n, k // 256, 1))) / 21760.0).astype(np.float16)
    w[:, :, :4] = np.concatenate([d, (7.5 * d.astype(np.float32)).astype(np.float16)], axis=2).view(np.uint8)
    w = w.reshape(n, -1)
    x = make_x(rng, m, k)
    ref = x.astype(np.float64) @ dequant_numpy(w[:narrow], narrow, k).astype(np.float64).T
    err = []
    for rows in (n, narrow):
        W = q4k.Weight(np.ascontiguousarray(w[:rows]), rows, k)
        y = torch.empty((m, rows), device=gpu)
        q4k.linear(torch.from_numpy(x).to(gpu), W, m, y, query_counts=[m])
        torch.cuda.synchronize()
        err.append(np.linalg.norm(y[:, :narrow].double().cpu().numpy() - ref) / np.linalg.norm(ref))
    print("wide, narrow", err)
    assert err[0] <= 1.05 * err[1], err
