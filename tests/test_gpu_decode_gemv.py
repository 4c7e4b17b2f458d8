"""The one-launch decode GEMV with K = 4096 (decode_gemv_kernel) against the CPU
oracle: 1 to 8 rows, every count of column tiles per workgroup with a partial
last workgroup, every weight type, epilogue and activation type, with and
without the RMS norm, plain and gate/up pairs; no staging and no norm launch
precedes it.  Bars: activations keep 22 bits and Q4_K / Q5_K
products are exact, 1e-5 with fp32 outputs; the other types round each product
once to fp16 (2^-11 = 4.9e-4 at most for a whole row); fp16 outputs 1e-3."""
import numpy as np
import pytest
import torch

from q4k_ref import TYPE_IQ4_XS, TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, make_weight, make_x, row_rel_err

pytestmark = pytest.mark.gpu
K = 4096

# (m, n, post, dtype, norm): one column tile past a round of 256 workgroups of one, two, three and four tiles; two rounds of six
SHAPES = [(1, 16, 0, torch.float32, False), (1, 4096, 1, torch.float32, False), (5, 1024, 0, torch.float16, True), (8, 4112, 2, torch.float32, True),
          (3, 8208, 1, torch.float16, False), (8, 12304, 0, torch.float32, False), (2, 16400, 2, torch.float16, False),
          (7, 32784, 0, torch.float32, True)]


@pytest.mark.parametrize("m,n,post,dtype,norm", SHAPES)
@pytest.mark.parametrize("t", [TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, TYPE_IQ4_XS])
def test_decode_gemv(q4k, oracle, gpu, t, m, n, post, dtype, norm):
    rng = np.random.default_rng(8000 + m + n + t)
    npdt = np.float16 if dtype == torch.float16 else np.float32
    w = make_weight(rng, n, K, t)
    x = make_x(rng, m, K, 0.05).astype(npdt)
    aux = make_x(rng, m, n, 2.0).astype(npdt) if post else None
    nw = (1.0 + 0.2 * rng.standard_normal(K)).astype(np.float32) * 0.05
    W = q4k.Weight(w, n, K, ggml_type=t)
    y = torch.from_numpy(aux).to(gpu) if post else torch.full((m, n), float("nan"), device=gpu, dtype=dtype)
    xt = torch.from_numpy(x).to(gpu)
    kw = dict(auxiliary=y if post else None, gated=post == 2, query_counts=[1] * m)
    torch.cuda.synchronize()
    q4k.profile_enable(True)
    if norm:
        q4k.linear_norm(xt, W, torch.from_numpy(nw).to(gpu), m, y, **kw)
    else:
        q4k.linear(xt, W, m, y, **kw)
    torch.cuda.synchronize()
    launches = [q4k.profile_query(kind)[0] for kind in (q4k.KERNEL_STAGE, q4k.KERNEL_GEMV, q4k.KERNEL_AUX)]
    q4k.profile_enable(False)
    assert launches == [0, 1, 0], launches
    got = y.float().cpu().numpy()
    assert np.all(np.isfinite(got))
    xn = oracle.rms_norm(x, nw).astype(np.float32) if norm else x
    ref = oracle.linear(xn, w, n, K, aux=aux, post=post, ggml_type=t).astype(np.float32)
    bar = 1e-3 if dtype == torch.float16 else 1e-5 if t in (TYPE_Q4_K, TYPE_Q5_K) else 4.9e-4
    assert row_rel_err(got, ref) <= bar


@pytest.mark.parametrize("m,n,dtype", [(1, 16, torch.float32), (8, 4112, torch.float16), (5, 8208, torch.float32), (3, 12304, torch.float16)])
@pytest.mark.parametrize("t", [TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, TYPE_IQ4_XS])
def test_decode_gemv_gate_up(q4k, oracle, gpu, t, m, n, dtype):
    rng = np.random.default_rng(8200 + m + n + t)
    wg, wu = make_weight(rng, n, K, t), make_weight(rng, n, K, t)
    x = make_x(rng, m, K, 0.05).astype(np.float16 if dtype == torch.float16 else np.float32)
    G, U = q4k.Weight(wg, n, K, ggml_type=t), q4k.Weight(wu, n, K, ggml_type=t)
    y = torch.full((m, n), float("nan"), device=gpu, dtype=dtype)
    xt = torch.from_numpy(x).to(gpu)
    torch.cuda.synchronize()
    q4k.profile_enable(True)
    q4k.mlp_gate_up(xt, G, U, m, y, query_counts=[1] * m)
    torch.cuda.synchronize()
    launches = [q4k.profile_query(kind)[0] for kind in (q4k.KERNEL_STAGE, q4k.KERNEL_GEMV, q4k.KERNEL_GEMV_GATED, q4k.KERNEL_AUX)]
    q4k.profile_enable(False)
    assert launches == [0, 0, 1, 0], launches
    got = y.float().cpu().numpy()
    assert np.all(np.isfinite(got))
    # Two projections' errors meet in each output; fp16 rounds gate, up and output.
    bar = 2e-5 if t in (TYPE_Q4_K, TYPE_Q5_K) else 1e-3
    assert row_rel_err(got, oracle.mlp_gate_up(x, wg, wu, n, K, ggml_type=t).astype(np.float32)) <= (2e-3 if dtype == torch.float16 else bar)


def _picking_q4k(n, k):
    """Q4_K bytes of the n x k matrix that has a single 1 per row (row r picks
    element pick[r]) and zeros elsewhere: d = 1, scales 1, mins 0."""
    pick = (np.arange(n, dtype=np.int64) * (k // n if k >= n else 1)) % k
    w = np.zeros((n, k // 256, 144), dtype=np.uint8)
    w[:, :, 0:2] = np.frombuffer(np.float16(1.0).tobytes(), dtype=np.uint8)
    w[:, :, 4:8] = 1
    w[:, :, 12:16] = 1
    e = pick % 256
    w[np.arange(n), pick // 256, 16 + 32 * (e // 64) + e % 32] = np.where(e % 64 < 32, 1, 16)
    return w.reshape(-1), pick


@pytest.mark.parametrize("m,n,k", [(1, 4096, K), (8, 1024, K), (5, 12288, K), (8, 4096, 12288)])
def test_activations_keep_23_bits(q4k, gpu, m, n, k):
    """Rows of x picked one element per output: hi + lo, both rounded to
    nearest, hold any value of 23 significant bits exactly, and no other term of
    the sum is non-zero, so the outputs equal the activations bit for bit."""
    rng = np.random.default_rng(8400 + m + n)
    x = (rng.uniform(0.125, 1.0, (m, k)) * rng.choice([-1.0, 1.0], (m, k))).astype(np.float32)
    x = (x.view(np.uint32) & np.uint32(0xFFFFFFFE)).view(np.float32)
    w, pick = _picking_q4k(n, k)
    W = q4k.Weight(w, n, k)
    y = torch.full((m, n), float("nan"), device=gpu)
    q4k.linear(torch.from_numpy(x).to(gpu), W, m, y, query_counts=[1] * m)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), x[:, pick])
