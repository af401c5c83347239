"""Products of few rows (csrc/kernels/gemm_skinny.hip) at the edges of their tiles: 1 to 64 rows,
columns that are no multiple of 16, K around the 32-, 16- and 128-deep steps and the eight waves,
every epilogue, and the INT4 weight.  Against float64 products of the same operands: fp32 results
within the rounding of their sums, bf16 results within one rounding (2^-9 of the largest term, so
4e-3 in the 2-norm)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from autonomousaicore_amd import _lib  # noqa: E402
from tests.gpu_util import bf16_round, call, dev, host, ptr, rel, stream  # noqa: E402

F32, BF16, F16 = _lib.AIC_F32, _lib.AIC_BF16, _lib.AIC_F16
T = {F32: torch.float32, BF16: torch.bfloat16}
TOL = {F32: 2e-6, BF16: 4e-3}


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


def mk(rng, dt, *shape):
    a = rng.standard_normal(shape).astype(np.float32)
    return a if dt == F32 else bf16_round(a)


@pytest.mark.parametrize("ab,c", [(BF16, BF16), (BF16, F32), (F32, F32)])
@pytest.mark.parametrize("M,N,K", [(1, 16, 8), (1, 100, 768), (3, 33, 40), (15, 24, 264), (16, 2304, 768), (17, 48, 2048),
                                   (32, 90, 1000), (33, 130, 72), (64, 512, 320), (2, 32768, 64), (65, 64, 128)])
def test_product_with_alpha_beta_residual(ab, c, M, N, K):
    rng = np.random.default_rng(M * 31 + N + K)
    A, B, C0, R = mk(rng, ab, M, K), mk(rng, ab, N, K), mk(rng, c, M, N), mk(rng, c, M, N + 3)
    ref = A.astype(np.float64) @ B.astype(np.float64).T
    a, b, r = dev(A, T[ab]), dev(B, T[ab]), dev(R, T[c])
    for alpha, beta, res, ldc in ((1.0, 0.0, None, N), (0.5, -1.5, r, N + 5)):
        out = torch.full((M, ldc), 9.0, dtype=T[c], device="cuda")
        out[:, :N] = dev(C0, T[c])
        call("aic_hip_gemm", 0, 1, M, N, K, alpha, ptr(a), K, ptr(b), K, beta, ptr(out), ldc, ptr(res), N + 3 if res is not None else 0,
             ab, c, stream())
        want = alpha * ref + (beta * C0 + R[:, :N] if res is not None else 0.0)
        got = host(out)
        assert rel(got[:, :N], want) < TOL[c]
        assert np.all(got[:, N:] == 9.0)


def _small_ints(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    return [torch.randint(-2, 3, s, generator=g, device="cuda").bfloat16() for s in ((M, K), (N, K), (M, N))]


def _product(A, B, R, out):
    (M, K), N = A.shape, B.shape[0]
    call("aic_hip_gemm", 0, 1, M, N, K, 1.0, ptr(A), K, ptr(B), K, 0.0, ptr(out), N, ptr(R), N, BF16, BF16, stream())


@pytest.mark.parametrize("M,N,K", [(1, 16, 16384), (8, 16, 5632), (16, 16, 5632), (16, 24, 8192), (32, 40, 5632), (64, 264, 5632),
                                   (64, 264, 2048), (1, 16400, 2048), (16, 16400, 2048), (64, 16, 33344), (64, 16, 5640)])
def test_long_rows(M, N, K):
    """Either side of the lengths and weight sizes from which a few-row product is cut among tile
    blocks, a K that no part count divides and one outside the tiles' layouts.  The operands are
    small integers: exact sums in any order, rounded once."""
    A, B, R = _small_ints(M, N, K)
    out, plain = torch.empty_like(R), torch.empty_like(R)
    _product(A, B, R, out)
    _product(A, B, None, plain)
    ref = A.cpu().double() @ B.cpu().double().T
    assert torch.equal(plain.cpu(), ref.to(torch.bfloat16))
    assert torch.equal(out.cpu(), (ref + R.cpu().double()).to(torch.bfloat16))


@pytest.mark.parametrize("N,K", [(16, 32768), (8, 65536), (256, 8192)])
def test_few_long_rows_cost_no_more_than_more_rows(N, K):
    """64 rows against 65, which never run the few-row kernel: 7 times the time there once."""
    def us(M):
        A, B, R = _small_ints(M, N, K)
        out, a, b = torch.empty_like(R), torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        best = 1e9
        for _ in range(6):
            a.record()
            for _ in range(30):
                _product(A, B, R, out)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 1e3 / 30)
        return best

    assert us(64) < 2.0 * us(65)


@pytest.mark.parametrize("M,seg", [(1, 0), (5, 96), (33, 32)])
@pytest.mark.parametrize("r2", [8, 16, 40])
@pytest.mark.parametrize("ab", [BF16, F32])
def test_low_rank_term(ab, r2, M, seg):
    rng = np.random.default_rng(r2 + M)
    N, K = 192, 128
    A, B, Y2 = mk(rng, ab, M, K), mk(rng, ab, N, K), mk(rng, ab, N, r2)
    X2 = mk(rng, ab, M, r2 * (N // seg if seg else 1))
    ref = A.astype(np.float64) @ B.astype(np.float64).T
    for n in range(N):
        g = n // seg if seg else 0
        ref[:, n] += X2[:, g * r2:(g + 1) * r2].astype(np.float64) @ Y2[n].astype(np.float64)
    a, b, x2, y2 = (dev(x, T[ab]) for x in (A, B, X2, Y2))
    out = torch.empty((M, N), dtype=T[ab], device="cuda")
    call("aic_hip_gemm_lowrank", 0, 1, M, N, K, 1.0, ptr(a), K, ptr(b), K, ptr(x2), X2.shape[1], ptr(y2), r2, r2, seg, 0, 0.0,
         ptr(out), N, None, 0, ab, ab, stream())
    assert rel(host(out), ref) < TOL[ab]


def test_low_rank_segments_past_the_last_tile():
    """16464 columns in blocks of 32: the last block's second tile starts past the end, and its
    low-rank columns with it.  X2 is the head of a larger buffer."""
    rng = np.random.default_rng(9)
    M, N, K, seg, r2 = 4, 16464, 64, 5488, 16
    A, B, Y2, X2 = (mk(rng, BF16, *s) for s in ((M, K), (N, K), (N, r2), (M, r2 * N // seg)))
    ref = A.astype(np.float64) @ B.astype(np.float64).T
    for g in range(N // seg):
        c = slice(g * seg, (g + 1) * seg)
        ref[:, c] += X2[:, g * r2:(g + 1) * r2].astype(np.float64) @ Y2[c].astype(np.float64).T
    a, b, y2 = (dev(x, T[BF16]) for x in (A, B, Y2))
    buf = torch.full((X2.size + 1024,), float("nan"), dtype=T[BF16], device="cuda")
    buf[:X2.size] = dev(X2, T[BF16]).reshape(-1)
    out = torch.empty((M, N), dtype=T[BF16], device="cuda")
    call("aic_hip_gemm_lowrank", 0, 1, M, N, K, 1.0, ptr(a), K, ptr(b), K, ptr(buf), X2.shape[1], ptr(y2), r2, r2, seg, 0, 0.0,
         ptr(out), N, None, 0, BF16, BF16, stream())
    assert rel(host(out), ref) < TOL[BF16]


@pytest.mark.parametrize("B,S,H,hd,start", [(1, 1, 2, 64, 7), (3, 5, 4, 32, 0), (2, 32, 2, 128, 11)])
def test_rotary_columns(B, S, H, hd, start):
    """The rotated q/k/v product equals the product followed by the rotary pass, to a bf16 unit."""
    rng = np.random.default_rng(hd + S)
    M, d, K = B * S, H * hd, 96
    a, w = dev(mk(rng, BF16, M, K), T[BF16]), dev(mk(rng, BF16, 3 * d, K), T[BF16])
    cos, sin = (np.empty((start + S, hd // 2), np.float32) for _ in range(2))
    call("aic_hip_rope_tables", cos.ctypes.data, sin.ctypes.data, start + S, hd, 10000.0)
    cd, sd = dev(cos), dev(sin)
    out, ref = (torch.empty((M, 3 * d), dtype=T[BF16], device="cuda") for _ in range(2))
    call("aic_hip_gemm_rope", M, 3 * d, K, ptr(a), K, ptr(w), K, ptr(out), 3 * d, 2 * d, hd, S, start, ptr(cd), ptr(sd), stream())
    call("aic_hip_gemm", 0, 1, M, 3 * d, K, 1.0, ptr(a), K, ptr(w), K, 0.0, ptr(ref), 3 * d, None, 0, BF16, BF16, stream())
    call("aic_hip_rope", ptr(ref), 3 * d, B, S, 2 * H, hd, start, ptr(cd), ptr(sd), 0, BF16, stream())
    assert rel(host(out), host(ref)) < 1e-3


@pytest.mark.parametrize("M,f", [(1, 16), (7, 352), (40, 208)])
def test_swiglu_pairs(M, f):
    rng = np.random.default_rng(M + f)
    K = 136
    a, w = dev(mk(rng, BF16, M, K), T[BF16]), dev(mk(rng, BF16, 2 * f, K) * 0.1, T[BF16])
    gu, h = torch.empty((M, 2 * f), dtype=T[BF16], device="cuda"), torch.empty((M, f), dtype=T[BF16], device="cuda")
    call("aic_hip_gemm_swiglu", M, f, K, ptr(a), K, ptr(w), K, ptr(gu), 2 * f, ptr(h), f, stream())
    ref = host(a).astype(np.float64) @ host(w).astype(np.float64).T
    g, u = ref[:, :f], ref[:, f:]
    assert rel(host(gu), ref) < 4e-3
    assert rel(host(h), g / (1 + np.exp(-g)) * u) < 1e-2  # two rounded factors and the result


@pytest.mark.parametrize("M,N,K,G", [(1, 64, 64, 64), (3, 40, 192, 128), (16, 256, 2048, 128), (7, 48, 320, 320), (50, 96, 448, 64)])
def test_int4_weight(orc, M, N, K, G):
    rng = np.random.default_rng(M + N + K)
    W, x = rng.standard_normal((N, K)).astype(np.float32), mk(rng, BF16, M, K)
    wd = dev(W)
    q = torch.empty(N * K // 2, dtype=torch.uint8, device="cuda")
    sc = torch.empty((N * K + G - 1) // G, dtype=torch.float16, device="cuda")
    call("aic_hip_int4_quantize", ptr(wd), N * K, G, ptr(q), ptr(sc), F16, stream())
    deq = torch.empty((N, K), dtype=T[BF16], device="cuda")
    call("aic_hip_int4_dequantize", ptr(q), ptr(sc), F16, N * K, G, ptr(deq), BF16, stream())
    xd, out = dev(x, T[BF16]), torch.empty((M, N), dtype=torch.float32, device="cuda")
    call("aic_hip_int4_dequant_gemm", 1, M, N, K, 1.0, ptr(xd), K, ptr(q), ptr(sc), F16, G, 0.0, ptr(out), N, None, 0, BF16, F32,
         stream())
    assert rel(host(out), x.astype(np.float64) @ host(deq).astype(np.float64).T) < 2e-6
