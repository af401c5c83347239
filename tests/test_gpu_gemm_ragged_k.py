"""Weight gradients dW = dY^T X whose token count is no multiple of the 64-deep K tiles: the tile
kernels' last partial tile (plain, K split and grouped launches).  Against float64 products of the
same bf16 operands, within the rounding of fp32 sums; the rows after the last token hold NaN."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from autonomousaicore_amd import _lib  # noqa: E402
from tests.gpu_util import call, host, ptr, rel, stream  # noqa: E402

F32, BF16 = _lib.AIC_F32, _lib.AIC_BF16


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


def rows(T, n, g):
    """[T, n] bf16 in the middle of a larger matrix whose other rows are NaN."""
    buf = torch.full((T + 80, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    buf[8:8 + T] = torch.randn((T, n), generator=g, device="cuda").bfloat16()
    return buf[8:8 + T]


def product(a, b):
    return (a.double().T @ b.double()).cpu().numpy()


# (dW rows, dW columns): one 128x128 tile and a ragged one, 128x256 tiles, 256x256 tiles, K split
@pytest.mark.parametrize("M,N", [(128, 128), (200, 72), (4096, 768), (8192, 1024), (768, 768)])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 63, 65, 130, 999, 1000, 2111, 8191])
def test_weight_gradient(M, N, T):
    g = torch.Generator(device="cuda").manual_seed(M + T)
    dy, x = rows(T, M, g), rows(T, N, g)
    ref = product(dy, x)
    out = torch.full((M, N), 3.0, device="cuda")
    for beta in (0.0, 1.0):
        call("aic_hip_gemm", 1, 0, M, N, T, 1.0, ptr(dy), M, ptr(x), N, beta, ptr(out), N, None, 0, BF16, F32, stream())
        assert rel(host(out), ref * (1.0 + beta)) < 3e-6
    low = torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    call("aic_hip_gemm", 1, 0, M, N, T, 1.0, ptr(dy), M, ptr(x), N, 0.0, ptr(low), N, None, 0, BF16, BF16, stream())
    assert rel(host(low), ref) < 4e-3


@pytest.mark.parametrize("T", [7, 333, 1000])
@pytest.mark.parametrize("shapes", [((384, 128), (128, 128)), ((2304, 768), (768, 768), (4096, 768), (768, 2048)),
                                    ((6144, 2048), (2048, 2048))])
def test_grouped_weight_gradients(shapes, T):
    g = torch.Generator(device="cuda").manual_seed(T)
    ops = [(rows(T, m, g), rows(T, n, g), torch.full((m, n), 5.0, device="cuda")) for m, n in shapes]
    d = (_lib.GemmDesc * len(ops))(*[_lib.GemmDesc(1, 0, a.shape[1], b.shape[1], T, a.data_ptr(), a.shape[1], b.data_ptr(),
                                                   b.shape[1], c.data_ptr(), b.shape[1]) for a, b, c in ops])
    call("aic_hip_gemm_grouped", len(ops), d, 1.0, 0.0, BF16, F32, stream())
    for a, b, c in ops:
        assert rel(host(c), product(a, b)) < 3e-6


def test_step_gradients_at_a_ragged_token_count(orc):
    """The fused gradient norm (partial sums from the weight gradients' epilogues) on 3 x 333
    tokens equals the norm of the gradients read back."""
    import autonomousaicore_amd as aic
    m = aic.TransformerLM(aic.TransformerLMConfig(vocab_size=512, hidden_dim=128, num_layers=2, num_heads=2,
                                                  intermediate_dim=384, max_seq_len=333, compute="bfloat16"),
                          aic.TrainingConfig(max_grad_norm=1.0))
    m.init_normal(3, 0.02)
    ids, tgt = aic.batch(5, 3, 333, 512)
    st = m.train_step(ids, tgt, 3, 333)
    grads = m.get_grads().astype(np.float64)
    assert m.fused_grad_norm(True)
    assert abs(st.grad_norm - np.linalg.norm(grads)) < 1e-5 * st.grad_norm
    m.close()
