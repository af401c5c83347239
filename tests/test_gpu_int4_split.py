"""INT4 products with their K split among blocks, from one row up: both ways round, with residual,
beta and fp32 output.  Against float64 products with the dequantized weight: fp32 results within
the rounding of their sums, bf16 results within one rounding."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from autonomousaicore_amd import _lib  # noqa: E402
from tests.gpu_util import bf16_round, call, dev, host, ptr, rel, stream  # noqa: E402

F32, BF16, F16 = _lib.AIC_F32, _lib.AIC_BF16, _lib.AIC_F16


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


def weight(rng, rows, cols, G):
    w = dev(rng.standard_normal((rows, cols)).astype(np.float32))
    q = torch.empty(rows * cols // 2, dtype=torch.uint8, device="cuda")
    s = torch.empty(rows * cols // G, dtype=torch.float16, device="cuda")
    call("aic_hip_int4_quantize", ptr(w), rows * cols, G, ptr(q), ptr(s), F16, stream())
    d = torch.empty((rows, cols), dtype=torch.bfloat16, device="cuda")
    call("aic_hip_int4_dequantize", ptr(q), ptr(s), F16, rows * cols, G, ptr(d), BF16, stream())
    return q, s, host(d).astype(np.float64)


# K split in 2 (128 tiles over a long K), up to 16 parts, an odd number of K tiles, no split
@pytest.mark.parametrize("tw", [1, 0])
@pytest.mark.parametrize("M,N,K,G", [(1, 2112, 2048, 64), (7, 192, 1088, 64), (65, 256, 5632, 128), (200, 2048, 1024, 128),
                                     (1000, 2048, 4096, 128), (130, 320, 1216, 64), (100, 128, 512, 128)])
def test_split_products(tw, M, N, K, G):
    rng = np.random.default_rng(M + N + K)
    q, s, w = weight(rng, *((N, K) if tw else (K, N)), G)
    x = bf16_round(rng.standard_normal((M, K)).astype(np.float32))
    r = bf16_round(rng.standard_normal((M, N)).astype(np.float32))
    ref = x.astype(np.float64) @ (w.T if tw else w)
    xd, rd = dev(x, torch.bfloat16), dev(r, torch.bfloat16)
    out = torch.full((M, N), 2.0, device="cuda")
    call("aic_hip_int4_dequant_gemm", tw, M, N, K, 1.0, ptr(xd), K, ptr(q), ptr(s), F16, G, 0.5, ptr(out), N, None, 0, BF16, F32,
         stream())
    assert rel(host(out), ref + 1.0) < 2e-6
    low = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    call("aic_hip_int4_dequant_gemm", tw, M, N, K, -2.0, ptr(xd), K, ptr(q), ptr(s), F16, G, 0.0, ptr(low), N, ptr(rd), N, BF16,
         BF16, stream())
    assert rel(host(low), r - 2.0 * ref) < 4e-3


@pytest.mark.parametrize("T", [1, 7, 70, 300])
@pytest.mark.parametrize("rank", [8, 16])
def test_projection_with_adapter(T, rank):
    """A whole QLoRA projection on few tokens: the low-rank term joins one K part only."""
    import ctypes
    rng = np.random.default_rng(T + rank)
    i, o, G, alpha = 1024, 2048, 128, 24.0
    q, s, w = weight(rng, o, i, G)
    x, dy, A, B = (bf16_round(rng.standard_normal(n).astype(np.float32) * c) for n, c in
                   (((T, i), 1.0), ((T, o), 1.0), ((rank, i), 0.05), ((o, rank), 0.05)))
    xd, dyd, Ad, Bd = (dev(t, torch.bfloat16) for t in (x, dy, A, B))
    y, dx = torch.empty((T, o), dtype=torch.bfloat16, device="cuda"), torch.empty((T, i), dtype=torch.bfloat16, device="cuda")
    dA, dB = torch.full((rank, i), 1.0, device="cuda"), torch.full((o, rank), 1.0, device="cuda")
    h = ctypes.c_void_p()
    call("aic_qlora_linear_create", i, o, rank, alpha, G, F16, BF16, ctypes.byref(h))
    call("aic_qlora_linear_forward", h, ptr(xd), T, ptr(q), ptr(s), ptr(Ad), ptr(Bd), None, ptr(y), stream())
    call("aic_qlora_linear_backward", h, ptr(dyd), ptr(dx), ptr(dA), ptr(dB), 1, stream())
    torch.cuda.synchronize()
    call("aic_qlora_linear_destroy", h)
    X, DY, A, B = (t.astype(np.float64) for t in (x, dy, A, B))
    sc = alpha / rank
    assert rel(host(y), X @ w.T + sc * (X @ A.T) @ B.T) < 5e-3
    assert rel(host(dx), DY @ w + sc * (DY @ B) @ A) < 5e-3
    assert rel(host(dA) - 1.0, sc * (DY @ B).T @ X) < 5e-3
    assert rel(host(dB) - 1.0, sc * DY.T @ (X @ A.T)) < 5e-3
