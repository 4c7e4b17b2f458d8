"""Activations, norm weights, outputs and aux at addresses aligned to one
element only, on the kernels that load them several elements at a time (the
one-launch decode GEMV, the row staging of the rows and middle GEMMs): the bits
of the same call on aligned buffers."""
import numpy as np
import pytest
import torch

from q4k_ref import TYPE_IQ4_XS, TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K, TYPE_Q8_0, make_weight, make_x

pytestmark = pytest.mark.gpu


def _shifted(a, shift, gpu, dtype):
    """The array on the GPU, `shift` elements into its allocation."""
    t = torch.empty(a.size + shift, device=gpu, dtype=dtype)[shift:].view(a.shape)
    return t.copy_(torch.from_numpy(a))


@pytest.mark.parametrize("dtype,shift", [(torch.float32, 1), (torch.float32, 3), (torch.float16, 1), (torch.float16, 6)])
@pytest.mark.parametrize("t,m,n,k", [(TYPE_Q4_K, 1, 1040, 4096), (TYPE_Q6_K, 8, 4112, 4096), (TYPE_Q8_0, 5, 8208, 4096), (TYPE_IQ4_XS, 19, 272, 512),
                                     (TYPE_Q5_K, 63, 144, 4352), (TYPE_Q6_K, 65, 272, 512), (TYPE_Q4_K, 130, 528, 12544)])
def test_shifted_buffers(q4k, gpu, t, m, n, k, dtype, shift):
    rng = np.random.default_rng(9600 + m + t)
    W = q4k.Weight(make_weight(rng, n, k, t), n, k, ggml_type=t)
    x, aux = make_x(rng, m, k, 0.05), make_x(rng, m, n, 2.0)
    nw = (1.0 + 0.2 * rng.standard_normal(k)).astype(np.float32) * 0.05
    out = []
    for s in (0, shift):
        xs, ys = _shifted(x, s, gpu, dtype), _shifted(aux, s, gpu, dtype)
        ws = _shifted(nw, s, gpu, torch.float32)
        assert s == 0 or xs.data_ptr() % 16 != 0
        counts = [1] * m if m <= 8 else [m]
        y1 = _shifted(np.full((m, n), np.nan, np.float32), s, gpu, dtype)
        q4k.linear(xs, W, m, y1, auxiliary=ys, gated=True, query_counts=counts)
        y2 = q4k.linear_norm(xs, W, ws, m, _shifted(np.zeros((m, n), np.float32), s, gpu, dtype), query_counts=counts)
        q4k.linear(xs, W, m, ys, auxiliary=ys, query_counts=counts)
        torch.cuda.synchronize()
        out.append([v.float().cpu().numpy() for v in (y1, y2, ys)])
    for a, b in zip(*out):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
