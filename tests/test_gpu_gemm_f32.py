"""fp32 products (csrc/kernels/gemm_f32.hip): every layout at the edges of the 16-row tiles and
16-deep steps, rows without 16-byte alignment, waves sharing a tile's K, K in parts, both tile
sizes.  Against float64: within the rounding of fp32 sums of K terms in a tree of chains."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from autonomousaicore_amd import _lib  # noqa: E402
from tests.gpu_util import call, host, rel, stream  # noqa: E402

F32 = _lib.AIC_F32


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
# one element; ragged everything; K below, at and past a step; waves sharing K; eight K parts, the
# last one shorter; 64x64 tiles
@pytest.mark.parametrize("M,N,K,pad", [(65, 1, 1, 0), (70, 33, 7, 0), (66, 31, 17, 1), (96, 64, 16, 0), (512, 128, 352, 0),
                                       (129, 100, 515, 3), (384, 128, 8192, 0), (72, 40, 2050, 2), (2050, 2111, 36, 0),
                                       (2113, 2049, 50, 1)])
def test_product(ta, tb, M, N, K, pad):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    mk = lambda r, c: torch.randn((r, c + pad), generator=g, device="cuda")[:, :c]  # noqa: E731
    A, B, R = mk(K, M) if ta else mk(M, K), mk(N, K) if tb else mk(K, N), mk(M, N)
    ref = ((A.T if ta else A).double() @ (B.T if tb else B).double()).cpu().numpy()
    for alpha, beta, res in ((1.0, 0.0, None), (-0.5, 2.0, R)):
        out = torch.full((M, N + pad), 3.0, device="cuda")
        call("aic_hip_gemm", ta, tb, M, N, K, alpha, A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), beta, out.data_ptr(),
             N + pad, None if res is None else res.data_ptr(), 0 if res is None else res.stride(0), F32, F32, stream())
        want = alpha * ref + (beta * 3.0 + host(R.contiguous()) if res is not None else 0.0)
        got = host(out)
        assert rel(got[:, :N], want) < 2e-6
        assert np.all(got[:, N:] == 3.0)


def test_no_terms():
    """K 0: beta C + R."""
    out = torch.full((100, 70), 3.0, device="cuda")
    a = torch.empty(1, device="cuda")
    call("aic_hip_gemm", 0, 1, 100, 70, 0, 1.0, a.data_ptr(), 1, a.data_ptr(), 1, 2.0, out.data_ptr(), 70, None, 0, F32, F32, stream())
    assert np.all(host(out) == 6.0)


def test_fused_norm_of_an_fp32_step():
    """An untied fp32 model's gradient norm comes from the products' epilogues."""
    import autonomousaicore_amd as aic
    m = aic.TransformerLM(aic.TransformerLMConfig(vocab_size=320, hidden_dim=128, num_layers=2, num_heads=4,
                                                  intermediate_dim=384, max_seq_len=300), aic.TrainingConfig(max_grad_norm=1.0))
    m.init_normal(3, 0.02)
    for S in (40, 300):  # K 320, and 2400 in parts
        ids, tgt = aic.batch(5, 8, S, 320)
        st = m.train_step(ids, tgt, 8, S)
        g = m.get_grads().astype(np.float64)
        assert m.fused_grad_norm(True)
        assert abs(st.grad_norm - np.linalg.norm(g)) < 1e-6 * st.grad_norm
    m.close()
