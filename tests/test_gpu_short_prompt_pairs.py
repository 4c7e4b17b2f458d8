"""Gate/up pairs of short prompts (prefill phase, up to 48 rows, K = 4096) on
the fused decode kernels of the same row counts, against the CPU oracle: one
fused launch at the edges of those kernels' ranges.  Bars: hi/lo activations
up to 24 rows and exact products leave fp32 sums in another order, 1e-5 per
projection, two of which meet in an output; beyond 24 rows single fp16
activations, the projections' own 1e-3."""
import numpy as np
import pytest
import torch

from q4k_ref import TYPE_IQ4_XS, TYPE_Q4_K, TYPE_Q6_K, make_weight, make_x, row_rel_err

pytestmark = pytest.mark.gpu
K = 4096


@pytest.mark.parametrize("t,m,n,fused", [(TYPE_Q4_K, 6, 1024, True), (TYPE_Q4_K, 8, 8208, True), (TYPE_Q6_K, 7, 512, True), (TYPE_IQ4_XS, 8, 1040, True),
                                         (TYPE_Q4_K, 9, 12288, True), (TYPE_Q4_K, 24, 12288, True), (TYPE_Q4_K, 25, 12288, True),
                                         (TYPE_Q4_K, 48, 12288, True), (TYPE_Q4_K, 16, 1024, False)])
def test_short_prompt_pair(q4k, oracle, gpu, t, m, n, fused):
    rng = np.random.default_rng(9300 + m + n + t)
    wg, wu = make_weight(rng, n, K, t), make_weight(rng, n, K, t)
    x = make_x(rng, m, K, 0.05)
    G, U = q4k.Weight(wg, n, K, ggml_type=t), q4k.Weight(wu, n, K, ggml_type=t)
    y = torch.full((m, n), float("nan"), device=gpu)
    xt = torch.from_numpy(x).to(gpu)
    torch.cuda.synchronize()
    q4k.profile_enable(True)
    q4k.mlp_gate_up(xt, G, U, m, y, query_counts=[m])
    torch.cuda.synchronize()
    gated = q4k.profile_query(q4k.KERNEL_GEMV_GATED)[0]
    q4k.profile_enable(False)
    assert gated == (1 if fused else 0)
    got = y.cpu().numpy()
    assert np.all(np.isfinite(got))
    bar = 2e-5 if t == TYPE_Q4_K and m <= 24 else 1e-3
    assert row_rel_err(got, oracle.mlp_gate_up(x, wg, wu, n, K, ggml_type=t)) <= bar
