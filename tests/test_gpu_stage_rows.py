"""Hi/lo activation staging of the decode and short-prompt kernels
(stage_x_kernel) through calls that read it, against the CPU oracle: rows of
one block, rows that fill the workgroup's registers exactly and the first past
them, with and without the RMS norm.  Bar: Q4_K products are exact and hi + lo
keep 22 bits of each activation (at up to 24 rows; beyond, these kernels hold one
fp16 value, a coarser bar), with a norm too (its scale is no power of
two), so fp32 outputs stay within 1e-5."""
import numpy as np
import pytest
import torch

from q4k_ref import make_q4k, make_x, row_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k", [(1, 256), (8, 3840), (9, 4096), (23, 4352), (24, 12288), (13, 12544)])
@pytest.mark.parametrize("norm", [False, True])
def test_staged_rows(q4k, oracle, gpu, norm, m, k):
    n = 1024
    rng = np.random.default_rng(9200 + m + k)
    w = make_q4k(rng, n, k)
    x = make_x(rng, m, k, 0.05)
    nw = (1.0 + 0.2 * rng.standard_normal(k)).astype(np.float32) * 0.05
    W = q4k.Weight(w, n, k)
    y = torch.full((m, n), float("nan"), device=gpu)
    xt = torch.from_numpy(x).to(gpu)
    if norm:
        q4k.linear_norm(xt, W, torch.from_numpy(nw).to(gpu), m, y, query_counts=[m])
    else:
        q4k.linear(xt, W, m, y, query_counts=[m])
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    assert np.all(np.isfinite(got))
    ref = oracle.linear(oracle.rms_norm(x, nw) if norm else x, w, n, k)
    assert row_rel_err(got, ref) <= 1e-5
