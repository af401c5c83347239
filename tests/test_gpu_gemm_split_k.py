"""Dense products whose K is cut into parts, around the limits of the reduction: tiles that end
inside a stripe, rows whose width or leading dimension rules out four-element loads, 131072 results
and fewer (reduced in row order) and more, beta and a residual, each output type, and inside a graph
capture on a stream without scratch memory (one part).  The operands are small integers, so the float32 sums are exact in any order."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from autonomousaicore_amd import _lib  # noqa: E402
from tests.gpu_util import call, stream  # noqa: E402

F32, BF16 = _lib.AIC_F32, _lib.AIC_BF16


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


def _run(M, N, K, pad, ct, beta, residual, ta=0, st=None, capture=None):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    mk = lambda *s: torch.randint(-2, 3, s, generator=g, device="cuda").float()  # noqa: E731
    A, B = (mk(K, M) if ta else mk(M, K)).bfloat16(), (mk(K, N) if ta else mk(N, K)).bfloat16()
    t = torch.float32 if ct == F32 else torch.bfloat16
    C, R = mk(M, N + pad).to(t), mk(M, N + pad).to(t)
    ref = (A.float().T @ B.float() if ta else A.float() @ B.float().T) + beta * C[:, :N].float()
    ref = (ref + R[:, :N].float() if residual else ref).to(t)
    keep = C.clone()

    def product():
        call("aic_hip_gemm", ta, 1 - ta, M, N, K, 1.0, A.data_ptr(), A.shape[1], B.data_ptr(), B.shape[1], beta,
             C.data_ptr(), N + pad, R.data_ptr() if residual else None, N + pad, BF16, ct, st or stream())

    (capture or (lambda f: f()))(product)
    torch.cuda.synchronize()
    assert torch.equal(C[:, :N], ref) and torch.equal(C[:, N:], keep[:, N:])


@pytest.mark.parametrize("ct", [F32, BF16])
@pytest.mark.parametrize("M,N,K,pad,beta,residual", [(128, 512, 4096, 0, 0.0, False), (129, 516, 4096, 4, 1.0, True),
                                                     (70, 130, 8192, 1, 0.0, True), (1000, 768, 2560, 0, 1.0, False),
                                                     (1000, 2304, 4096, 8, 0.0, True), (256, 512, 4096, 0, 1.0, True),
                                                     (257, 512, 4096, 0, 1.0, True), (40, 24, 16384, 1, 1.0, True)])
def test_split_k_reduction(ct, M, N, K, pad, beta, residual):
    _run(M, N, K, pad, ct, beta, residual)


@pytest.mark.parametrize("M,N,K", [(768, 768, 8192), (768, 768, 1024), (256, 264, 3001)])
def test_split_k_weight_gradient(M, N, K):
    _run(M, N, K, 0, F32, 0.0, False, ta=1)


def test_split_k_captured_without_scratch():
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()

    def capture(product):
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=s):
            product()
        for _ in range(3):
            graph.replay()

    _run(250, 512, 4096, 0, BF16, 0.0, False, st=s.cuda_stream, capture=capture)
