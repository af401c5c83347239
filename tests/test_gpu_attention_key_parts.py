"""The general attention forward with the keys of a few queries shared by several blocks: where a
head's row times the blocks of 32 keys passes 2816 bytes, so past 704 keys of 128 bytes (bf16 heads of
64) and 352 of 256 (bf16 heads of 128, fp32 heads of 64), with uneven shares, a causal offset, an
infinity that one block sees, and inside a graph capture, where one block keeps all keys.  Bounds as for
the same entry at its tile edges: fp32 sums, and one bf16 rounding of the outputs."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from autonomousaicore_amd import _lib  # noqa: E402
from tests.gpu_util import call, host, rel, stream  # noqa: E402

F32, BF16 = _lib.AIC_F32, _lib.AIC_BF16


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


def _ops(B, H, Sq, Sk, D, dt, seed=5):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = torch.float32 if dt == F32 else torch.bfloat16
    return [torch.randn((B * n, H * D), generator=g, device="cuda").to(t) for n in (Sq, Sk, Sk)]


def _fwd(q, k, v, B, H, Sq, Sk, D, causal, dt, out=None, st=None):
    o, lse = out or (torch.empty_like(q), torch.empty((B, H, Sq), device="cuda"))
    call("aic_hip_attn_fwd_qk", q.data_ptr(), H * D, k.data_ptr(), v.data_ptr(), H * D, o.data_ptr(), H * D,
         lse.data_ptr(), B, H, Sq, Sk, D, int(causal), 1.0 / np.sqrt(D), dt, stream() if st is None else st)
    return o, lse


def _heads(x, B, S, H, D):
    return np.ascontiguousarray(host(x).reshape(B, S, H, D).transpose(0, 2, 1, 3).reshape(B * H, S, D))


@pytest.mark.parametrize("dt", [F32, BF16])
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal", [(1, 2, 1, 768, 64, False), (1, 2, 1, 769, 64, False),
                                                (2, 3, 1, 801, 128, False), (1, 2, 16, 1100, 32, True),
                                                (1, 1, 7, 4100, 16, True), (8, 16, 1, 1500, 64, False),
                                                (1, 2, 1, 704, 64, False), (1, 2, 1, 705, 64, False),
                                                (1, 2, 3, 352, 128, False), (1, 2, 3, 353, 128, False),
                                                (1, 2, 1, 352, 64, False), (1, 2, 1, 353, 64, False)])
def test_attention_key_parts(orc, dt, B, H, Sq, Sk, D, causal):
    q, k, v = _ops(B, H, Sq, Sk, D, dt)
    o, lse = _fwd(q, k, v, B, H, Sq, Sk, D, causal, dt)
    o_ref, lse_ref = orc.flash_fwd(_heads(q, B, Sq, H, D), _heads(k, B, Sk, H, D), _heads(v, B, Sk, H, D), causal)
    assert np.max(np.abs(host(lse).reshape(B * H, Sq) - lse_ref)) < (2e-5 if dt == F32 else 1e-3)
    assert rel(_heads(o, B, Sq, H, D), o_ref) < (2e-6 if dt == F32 else 4e-3)


@pytest.mark.parametrize("dt", [F32, BF16])
def test_attention_key_parts_infinity(dt):
    shape = (1, 1, 2, 2000, 64)
    q, k, v = _ops(*shape, dt)
    clean, _ = _fwd(q, k, v, *shape, False, dt)
    v[1500, 5] = float("inf")
    dirty, _ = _fwd(q, k, v, *shape, False, dt)
    a, b = host(clean), host(dirty)
    assert np.all(np.isposinf(b[:, 5]))
    # formed row by row there: equal up to the order of the sums
    assert rel(np.delete(b, 5, 1), np.delete(a, 5, 1)) < (1e-5 if dt == F32 else 8e-3)


def test_attention_key_parts_captured_without_scratch():
    shape = (1, 3, 1, 1777, 64)
    q, k, v = _ops(*shape, BF16)
    want, _ = _fwd(q, k, v, *shape, False, BF16)
    out = torch.empty_like(q), torch.empty((1, 3, 1), device="cuda")
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=s):
        _fwd(q, k, v, *shape, False, BF16, out, s.cuda_stream)
    for _ in range(3):
        out[0].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert rel(host(out[0]), host(want)) < 8e-3
        _fwd(q, k, v, *shape, False, BF16)
