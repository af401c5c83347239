"""The embedding backward around the limits of its sorting by counting: blocks of 32 tokens, the
16384 tokens up to which it is used, and runs of equal ids around the 16 that one wave sums and the
64 positions that one look covers.  The gradients are small integers, so every order of adding
them is exact and the result has to be equal."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from autonomousaicore_amd import _lib  # noqa: E402
from tests.gpu_util import call, ptr, stream  # noqa: E402

F32, BF16 = _lib.AIC_F32, _lib.AIC_BF16


def _ids(kind, N, V, rng):
    if kind == "one":
        return np.full(N, V - 1, np.int64)
    if kind == "outside":
        return np.where(rng.random(N) < 0.5, V + 3, -1).astype(np.int64)
    if kind == "runs":  # runs of 1, 15, 16, 17, 62, 63, 64, 65 and the rest, in shuffled order
        n = np.array([1, 15, 16, 17, 62, 63, 64, 65])
        n = n[np.cumsum(n) <= N]
        i = np.repeat(np.arange(len(n) + 1), np.append(n, N - n.sum()))
        return rng.permutation(i * 7 % V).astype(np.int64)
    i = rng.integers(0, V, N)
    i[:: 11] = -5
    return i.astype(np.int64)


@pytest.mark.parametrize("dt,D", [(BF16, 512), (F32, 64), (BF16, 40)])
@pytest.mark.parametrize("kind", ["one", "outside", "runs", "mixed"])
@pytest.mark.parametrize("N", [1, 31, 32, 33, 1000, 16384, 16385])
def test_embed_bwd_by_counting(kind, N, dt, D):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    V = 300
    rng = np.random.default_rng(N + D)
    ids = _ids(kind, N, V, rng)
    dout = rng.integers(-3, 4, (N, D)).astype(np.float32)
    ref = np.zeros((V, D), np.float32)
    ok = (ids >= 0) & (ids < V)
    np.add.at(ref, ids[ok], dout[ok])
    dd = torch.from_numpy(dout).cuda().to(torch.float32 if dt == F32 else torch.bfloat16)
    idd = torch.from_numpy(ids).cuda()
    dW = torch.full((V, D), 5.0, dtype=torch.float32, device="cuda")
    for acc in (0, 1):
        call("aic_hip_embed_bwd", ptr(idd), N, ptr(dd), V, D, ptr(dW), acc, dt, stream())
        np.testing.assert_array_equal(dW.cpu().numpy(), ref * (1 + acc))
