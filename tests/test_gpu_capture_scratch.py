"""Captured calls whose eager form keeps partial sums in the stream's scratch memory: the stream has a
scratch buffer when they are captured, a larger eager call on it then replaces that buffer, and
another owner takes the memory.  Replays must neither write there nor read from it."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from autonomousaicore_amd import _lib  # noqa: E402
from tests.gpu_util import call, host, ptr, rel  # noqa: E402

F32, BF16, F16 = _lib.AIC_F32, _lib.AIC_BF16, _lib.AIC_F16


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


def _ints(dt, *s):
    g = torch.Generator(device="cuda").manual_seed(sum(s))
    return torch.randint(-2, 3, s, generator=g, device="cuda").to(torch.float32 if dt == F32 else torch.bfloat16)


def _product(dt):
    """out = A^T B over 4096 tokens: eight K parts in fp32, K splits in bf16.  Whole numbers: exact."""
    def make(scale):
        M, N, K = 256 * scale, 128, 4096
        A, B, out = _ints(dt, K, M), _ints(dt, K, N), torch.empty((M, N), device="cuda")
        return out, lambda st: call("aic_hip_gemm", 1, 0, M, N, K, 1.0, ptr(A), M, ptr(B), N, 0.0, ptr(out), N, None, 0, dt, F32, st)
    return make


def _int4(scale):
    M, N, K, G = 100 * scale, 256, 4096, 128
    w, x = _ints(F32, N, K), _ints(BF16, M, K)
    q, s = torch.empty(N * K // 2, dtype=torch.uint8, device="cuda"), torch.empty(N * K // G, dtype=torch.float16, device="cuda")
    call("aic_hip_int4_quantize", ptr(w), N * K, G, ptr(q), ptr(s), F16, torch.cuda.current_stream().cuda_stream)
    out = torch.empty((M, N), device="cuda")
    return out, lambda st: call("aic_hip_int4_dequant_gemm", 1, M, N, K, 1.0, ptr(x), K, ptr(q), ptr(s), F16, G, 0.0, ptr(out), N, None, 0,
                                BF16, F32, st)


def _attention(scale):
    H, Sk, D = 3 * scale, 1777, 64
    q, k, v = (torch.randn((n, H * D), device="cuda").bfloat16() for n in (1, Sk, Sk))
    out = torch.empty_like(q)
    return out, lambda st: call("aic_hip_attn_fwd_qk", ptr(q), H * D, ptr(k), ptr(v), H * D, ptr(out), H * D, None, 1, H, 1, Sk, D, 0,
                                1.0 / np.sqrt(D), BF16, st)


@pytest.mark.parametrize("make,tol", [(_product(F32), 0.0), (_product(BF16), 0.0), (_int4, 2e-6), (_attention, 8e-3)],
                         ids=["fp32", "bf16", "int4", "attention"])
def test_replays_leave_the_streams_scratch_alone(make, tol):
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    out, run = make(1)
    _, larger = make(8)
    torch.cuda.synchronize()
    run(s.cuda_stream)  # the stream's scratch buffer exists from here on
    torch.cuda.synchronize()
    want = host(out)
    with torch.cuda.graph(graph, stream=s):
        run(s.cuda_stream)
    larger(s.cuda_stream)
    n = 8 << 20  # the memory given back, under another owner
    mine, theirs = np.full(n, 0x5a, np.uint8), np.empty(n, np.uint8)
    p = ctypes.c_void_p()
    call("aic_hip_mem_alloc_async", ctypes.byref(p), n, s.cuda_stream)
    call("aic_hip_memcpy_sync", p, mine.ctypes.data, n, s.cuda_stream)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            graph.replay()
        torch.cuda.synchronize()
        assert rel(host(out), want) <= tol
        call("aic_hip_memcpy_sync", theirs.ctypes.data, p, n, s.cuda_stream)
        assert np.array_equal(mine, theirs)
        larger(s.cuda_stream)
    call("aic_hip_mem_free_async", p, s.cuda_stream)
    torch.cuda.synchronize()
    call("aic_hip_mem_release_stream", s.cuda_stream)
