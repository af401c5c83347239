"""Row counts that end inside a 256-row tile, in every epilogue form of the large tiles: each row
equals, bit for bit, the same row of the product over whole tiles (the same tile kernel, so the
same sums in the same order), and nothing past the last row is written."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from autonomousaicore_amd import _lib  # noqa: E402
from tests.gpu_util import call, stream  # noqa: E402

F32, BF16 = _lib.AIC_F32, _lib.AIC_BF16
FULL, N, K = 512, 16384, 256  # two row tiles by 64 column tiles: enough for the fused forms


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


@pytest.fixture(scope="module")
def ops():
    g = torch.Generator(device="cuda").manual_seed(11)
    mk = lambda *s: torch.randn(s, generator=g, device="cuda").bfloat16()  # noqa: E731
    cos, sin = (np.empty((FULL, 64), np.float32) for _ in range(2))
    call("aic_hip_rope_tables", cos.ctypes.data, sin.ctypes.data, FULL, 128, 10000.0)
    cos6, sin6 = (np.empty((FULL, 32), np.float32) for _ in range(2))
    call("aic_hip_rope_tables", cos6.ctypes.data, sin6.ctypes.data, FULL, 64, 10000.0)
    d = dict(A=mk(FULL, K), W=mk(N, K), Wt=mk(K, N), R=mk(FULL, N), GU=mk(FULL, 2 * N))
    d.update({n: torch.from_numpy(a).cuda() for n, a in dict(c128=cos, s128=sin, c64=cos6, s64=sin6).items()})
    return d


def run(o, form, M):
    """The outputs of `form` over M rows, each with 8 rows more than M that must stay at 5."""
    p = lambda t: t.data_ptr()  # noqa: E731
    out = lambda c, dt=torch.bfloat16: torch.full((M + 8, c), 5.0, dtype=dt, device="cuda")  # noqa: E731
    st = stream()
    if form in ("plain", "residual", "float", "dgrad"):
        C = out(N, torch.float32 if form == "float" else torch.bfloat16)
        tb = 0 if form == "dgrad" else 1
        R = o["R"] if form == "residual" else None
        call("aic_hip_gemm", 0, tb, M, N, K, 1.0, p(o["A"]), K, p(o["W"] if tb else o["Wt"]), K if tb else N, 0.0, p(C), N,
             None if R is None else p(R), N if R is not None else 0, BF16, F32 if form == "float" else BF16, st)
        return [C]
    if form.startswith("rope"):
        hd = int(form[4:])
        C = out(N)
        call("aic_hip_gemm_rope", M, N, K, p(o["A"]), K, p(o["W"]), K, p(C), N, N // 2, hd, M, 0, p(o[f"c{hd}"]), p(o[f"s{hd}"]), st)
        return [C]
    if form == "glu":
        C, H = out(N), out(N // 2)
        call("aic_hip_gemm_swiglu", M, N // 2, K, p(o["A"]), K, p(o["W"]), K, p(C), N, p(H), N // 2, st)
        return [C, H]
    D, G = out(N), out(2 * N)
    call("aic_hip_gemm_swiglu_bwd", M, N, K, p(o["A"]), K, p(o["Wt"]), N, p(o["GU"]), 2 * N, p(D), N, p(G), st)
    return [G]


@pytest.mark.parametrize("form", ["plain", "residual", "float", "dgrad", "rope128", "rope64", "glu", "dglu"])
@pytest.mark.parametrize("M", [257, 300, 383, 384, 385, 511])
def test_rows_of_a_partial_tile(ops, form, M):
    for got, want in zip(run(ops, form, M), run(ops, form, FULL)):
        assert torch.equal(got[:M], want[:M])
        assert bool((got[M:] == 5.0).all())


def test_the_whole_product_is_right(ops):
    ref = ops["A"].double() @ ops["W"].double().T
    (C,) = run(ops, "plain", 300)
    assert float((C[:300].double() - ref[:300]).norm() / ref[:300].norm()) < 4e-3


def test_swiglu_backward_keeps_the_product_of_a_partial_tile(ops):
    M, p = 300, lambda t: t.data_ptr()  # noqa: E731
    D, G, want = (torch.zeros((M, n), dtype=torch.bfloat16, device="cuda") for n in (N, 2 * N, N))
    call("aic_hip_gemm_swiglu_bwd", M, N, K, p(ops["A"]), K, p(ops["Wt"]), N, p(ops["GU"]), 2 * N, p(D), N, p(G),
         stream())
    call("aic_hip_gemm", 0, 0, M, N, K, 1.0, p(ops["A"]), K, p(ops["Wt"]), N, 0.0, p(want), N, None, 0, BF16, BF16,
         stream())
    assert torch.equal(D, want)
