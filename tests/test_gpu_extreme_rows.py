"""Extreme activations on the one-launch decode GEMV, the rows GEMM and the
middle GEMM: a row with an infinity and one with a NaN have no finite output
and leave the other rows' bits alone; fp16 rows of the largest finite values
and of subnormals match the CPU oracle (row-relative 1e-3: fp16 outputs, and
the single fp16 rounding of the weights' products)."""
import numpy as np
import pytest
import torch

from q4k_ref import TYPE_IQ4_XS, TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, make_weight, make_x, row_rel_err

pytestmark = pytest.mark.gpu
SHAPES = [(8, 272, 4096), (40, 272, 512), (70, 512, 1024)]  # one of each kernel (Q4_K at 40 rows: the staged GEMV)
TYPES = [TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, TYPE_IQ4_XS]


def _run(q4k, gpu, W, x, m, n, dtype):
    y = torch.zeros((m, n), device=gpu, dtype=dtype)
    q4k.linear(torch.from_numpy(x).to(gpu), W, m, y, query_counts=[1] * m if m <= 8 else [m])
    torch.cuda.synchronize()
    return y.float().cpu().numpy()


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("t", TYPES)
def test_non_finite_rows_stay_apart(q4k, gpu, t, m, n, k):
    rng = np.random.default_rng(9700 + m + t)
    W = q4k.Weight(make_weight(rng, n, k, t), n, k, ggml_type=t)
    x = make_x(rng, m, k, 0.25)
    clean = _run(q4k, gpu, W, x, m, n, torch.float32)
    x[1, 5], x[m - 2, k - 3] = np.inf, np.nan
    got = _run(q4k, gpu, W, x, m, n, torch.float32)
    bad = np.zeros(m, bool)
    bad[[1, m - 2]] = True
    assert not np.isfinite(got[bad]).any()
    assert np.array_equal(got[~bad], clean[~bad])


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("t", TYPES)
def test_largest_and_smallest_halves(q4k, oracle, gpu, t, m, n, k):
    rng = np.random.default_rng(9800 + m + t)
    w = make_weight(rng, n, k, t)
    x = make_x(rng, m, k, 0.25).astype(np.float16)
    x[0] = rng.choice([-65504.0, 65504.0, 1.0], k)
    x[m - 1] = (rng.integers(-1023, 1024, k) * 2.0**-24).astype(np.float16)
    W = q4k.Weight(w, n, k, ggml_type=t)
    # fp32 outputs of the same rows (an fp16 output of 65504s would overflow), and fp16 ones of the rest.
    got = _run(q4k, gpu, W, x.astype(np.float32), m, n, torch.float32)
    ref = oracle.linear(x.astype(np.float32), w, n, k, ggml_type=t)
    assert row_rel_err(got, ref) <= 1e-3
    x[0] = x[2]
    half = _run(q4k, gpu, W, x, m, n, torch.float16)[:m - 1]
    assert row_rel_err(half, oracle.linear(x.astype(np.float32), w, n, k, ggml_type=t)[:m - 1]) <= 1e-3
