"""Calls of several threads on one stream whose kernels pass partial sums through the stream's scratch
memory: each call's launches stay together and no call's buffer is given back before its launches.
Sizes differ between the threads, so that the buffer grows while others use it."""
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from autonomousaicore_amd import _lib  # noqa: E402
from tests.gpu_util import call, host, ptr, rel  # noqa: E402

F32, BF16 = _lib.AIC_F32, _lib.AIC_BF16


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


def _product(dt, M, N, K, st):
    """out = A^T B in K parts; small integers, exact in float32."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A, B = (torch.randint(-2, 3, (K, n), generator=g, device="cuda").to(torch.float32 if dt == F32 else torch.bfloat16) for n in (M, N))
    out = torch.empty((M, N), device="cuda")
    want = A.cpu().double().T @ B.cpu().double()
    return out, want, lambda: call("aic_hip_gemm", 1, 0, M, N, K, 1.0, ptr(A), M, ptr(B), N, 0.0, ptr(out), N, None, 0, dt, F32, st)


def _attention(H, Sk, st):
    D = 64
    q, k, v = (torch.randn((n, H * D), device="cuda") for n in (1, Sk, Sk))
    out = torch.empty_like(q)
    Q, K, V = (x.cpu().double().view(-1, H, D) for x in (q, k, v))
    p = torch.softmax(torch.einsum("qhd,khd->hqk", Q, K) / np.sqrt(D), -1)
    want = torch.einsum("hqk,khd->qhd", p, V).reshape(1, H * D)
    return out, want, lambda: call("aic_hip_attn_fwd_qk", ptr(q), H * D, ptr(k), ptr(v), H * D, ptr(out), H * D, None, 1, H, 1, Sk, D, 0,
                                   1.0 / np.sqrt(D), F32, st)


def test_threads_share_a_stream():
    s = torch.cuda.Stream()
    st = s.cuda_stream
    jobs = [_product(F32, 128, 352, 4096, st), _product(F32, 320, 128, 8192, st), _product(BF16, 256, 264, 4096, st),
            _attention(3, 1777, st), _attention(12, 2048, st)]
    torch.cuda.synchronize()
    wrong, start = [], threading.Barrier(len(jobs))

    def work(i):
        out, want, run = jobs[i]
        start.wait()
        for rep in range(12):
            for _ in range(25):
                run()
            with torch.cuda.stream(s):
                got = out.clone()
            s.synchronize()
            if not rel(host(got), want.numpy()) <= 5e-6:
                wrong.append((i, rep))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    call("aic_hip_mem_release_stream", st)
