"""RMS norm rows taken 8 elements at a time (rms_norm8_kernel) and the general
form beside it, against the CPU oracle at the edges of the rule between them:
the shortest rows, rows of one chunk per thread and the first past it, the
longest rows of three chunks and the first past them, lengths that are no
multiple of 8, and rows that do not start on 16 bytes.  Bars: 1e-5 of the
element in fp32 (the sum of squares is taken in another order), one fp16 ulp
in fp16."""
import numpy as np
import pytest
import torch

from q4k_ref import make_x

pytestmark = pytest.mark.gpu


def _close(got, ref):
    if got.dtype == np.float16:
        ulp = np.spacing(np.abs(ref).astype(np.float16)).astype(np.float32)
        return np.all(np.abs(got.astype(np.float32) - ref.astype(np.float32)) <= ulp)
    return np.all(np.abs(got - ref) <= 1e-5 * np.abs(ref) + 1e-30)


@pytest.mark.parametrize("m,k", [(1, 8), (3, 4096), (5, 4104), (2, 12288), (2, 12296), (7, 100), (300, 512)])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_rms_norm_forms(q4k, oracle, gpu, dtype, offset, m, k):
    rng = np.random.default_rng(9100 + m + k)
    npdt = np.float16 if dtype == torch.float16 else np.float32
    x = make_x(rng, m, k, 2.0).astype(npdt)
    w = (1.0 + 0.2 * rng.standard_normal(k)).astype(np.float32)
    ref = oracle.rms_norm(x, w)
    for buf in ("x", "y", "w"):  # the one that starts off 16 bytes
        xs = torch.empty(m * k + 1, device=gpu, dtype=dtype)
        ys = torch.full((m * k + 1,), float("nan"), device=gpu, dtype=dtype)
        wsb = torch.empty(k + 1, device=gpu)
        xt, yt, wt = (t[offset if name == buf else 0:][:size] for name, t, size in (("x", xs, m * k), ("y", ys, m * k), ("w", wsb, k)))
        xt.copy_(torch.from_numpy(x).reshape(-1))
        wt.copy_(torch.from_numpy(w))
        q4k.rms_norm(xt.view(m, k), wt, yt.view(m, k))
        torch.cuda.synchronize()
        assert _close(yt.view(m, k).cpu().numpy(), ref), buf
    y = torch.from_numpy(x).to(gpu)
    q4k.rms_norm(y, torch.from_numpy(w).to(gpu), y)  # in place
    torch.cuda.synchronize()
    assert _close(y.cpu().numpy(), ref)


@pytest.mark.parametrize("k", [4096, 5120, 12288])
def test_rms_norm_sum_order(q4k, gpu, k):
    """A row's scale, read out of an element of x that is 1 under a weight of 1,
    against 64 bits, beside that of the fp32 sum of squares rounded once (both
    with the division and square root in fp32).  With the eight waves' sums added
    in pairs the root mean square over the rows is 1.06 to 1.075 times as large
    (numpy, the kernel's order of sums), in turn 1.12 to 1.16; 16384 rows hold
    each to 0.01.  K = 4096 is one chunk per thread, 5120 one or two, 12288 three."""
    m, eps = 16384, 1e-6
    g = torch.Generator(device=gpu)
    g.manual_seed(9300 + k)
    x = torch.randn(m, k, device=gpu, generator=g) * torch.exp(2 * torch.rand(m, 1, device=gpu, generator=g) - 1)
    x[:, 0] = 1.0
    y = torch.empty_like(x)
    q4k.rms_norm(x, torch.ones(k, device=gpu), y, eps=eps)
    torch.cuda.synchronize()
    total = torch.cat([(c.double() ** 2).sum(1) for c in x.split(2048)]).cpu().numpy()
    exact = 1.0 / np.sqrt(total / k + eps)
    once = np.float32(1) / np.sqrt(total.astype(np.float32) / np.float32(k) + np.float32(eps))
    got = y[:, 0].cpu().numpy()

    def rms(s):
        return np.sqrt(np.mean((s / exact - 1) ** 2))

    print("scale error", k, rms(got), "sum rounded once", rms(once))
    assert rms(got) <= 1.095 * rms(once)
