"""The RMSNorm backward on either side of the row counts at which a wave takes one row more: a
row's dx does not depend on how many rows there are, and dw stays within the float32 sum's bound."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from autonomousaicore_amd import _lib  # noqa: E402
from tests.gpu_util import call, ptr, stream  # noqa: E402

F32, BF16 = _lib.AIC_F32, _lib.AIC_BF16


@pytest.mark.parametrize("dt,dim", [(BF16, 768), (F32, 100)])
@pytest.mark.parametrize("rows", [1, 1024, 1025, 2049, 7168, 7169, 8193])
def test_rmsnorm_bwd_rows(rows, dt, dim):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    tdt = torch.float32 if dt == F32 else torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(3)
    x, dy = (torch.randn(8200, dim, generator=g, device="cuda").to(tdt) for _ in range(2))
    w = 1 + 0.1 * torch.randn(dim, generator=g, device="cuda")
    y, rms = torch.empty_like(x), torch.empty(8200, device="cuda")
    call("aic_hip_rmsnorm_fwd", ptr(x), dim, ptr(w), ptr(y), dim, ptr(rms), 8200, dim, 1e-6, dt, stream())

    def bwd(n):
        dx, dw = torch.full((8200, dim), 9.0, device="cuda").to(tdt), torch.full((dim,), 7.0, device="cuda")
        call("aic_hip_rmsnorm_bwd", ptr(dy), dim, ptr(x), dim, ptr(w), ptr(rms), None, 0, ptr(dx), dim, ptr(dw), 0, n,
             dim, dt, stream())
        return dx, dw

    dx, dw = bwd(rows)
    full, _ = bwd(8200)
    assert torch.equal(dx[:rows], full[:rows]) and bool((dx[rows:] == 9).all())
    # a term dy x / rms has at most 3 roundings and goes through at most `rows` additions
    term = dy[:rows].double() * x[:rows].double() / rms[:rows, None].double()
    err = (dw.double() - term.sum(0)).abs()
    assert bool((err <= (rows + 3) * 2.0 ** -24 * term.abs().sum(0)).all())
