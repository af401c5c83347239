"""The general attention kernels (csrc/kernels/attention_general.hip) where their tiling can go
wrong: lengths around the 16-row tiles and 32-row blocks, one query, groups shared by several
waves, head_dim 16 to 128, and rows whose leading dimension or base rules out 16-byte loads.
Each head against the oracle's restatement of the CPU path (src/ops/flash_attention.cpp:32-260)
within the bounds that the launcher tests use for the same entries: fp32 sums over up to 2000
keys, and one bf16 rounding of the outputs."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from autonomousaicore_amd import _lib  # noqa: E402
from tests.gpu_util import bf16_round, call, host, rel, stream  # noqa: E402

F32, BF16 = _lib.AIC_F32, _lib.AIC_BF16


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


# (B, H, Sq, Sk, D, causal, pad, shift): rows of H * D + pad elements from an address shifted by
# `shift` elements
CASES = [(1, 1, 1, 1, 64, False, 0, 0), (1, 2, 1, 2000, 128, False, 0, 0), (2, 3, 16, 32, 32, True, 0, 0),
         (1, 2, 17, 33, 16, False, 0, 0), (2, 2, 33, 31, 128, True, 8, 0), (1, 3, 47, 65, 64, False, 3, 0),
         (1, 2, 31, 97, 128, True, 0, 1), (3, 4, 200, 130, 64, True, 8, 0), (1, 1, 5, 700, 16, False, 1, 3)]


@pytest.mark.parametrize("dt", [F32, BF16])
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,pad,shift", CASES)
def test_attention_tile_edges(orc, dt, B, H, Sq, Sk, D, causal, pad, shift):
    rng = np.random.default_rng(Sq * 7 + Sk * 3 + D + pad)
    t, ld = torch.float32 if dt == F32 else torch.bfloat16, H * D + pad

    def rows(n, fill=None):
        """A [n, ld] matrix of its own, `shift` elements into its storage, between guard values."""
        buf = torch.full((n * ld + shift + 16,), 7.0, dtype=t, device="cuda")
        x = buf[shift:shift + n * ld].view(n, ld)
        if fill is not None:
            a = fill.standard_normal((n, ld)).astype(np.float32)
            x.copy_(torch.from_numpy(a if dt == F32 else bf16_round(a)).to(t))
        return buf, x

    (_, q), (_, k), (_, v), (_, do) = rows(B * Sq, rng), rows(B * Sk, rng), rows(B * Sk, rng), rows(B * Sq, rng)
    (bo, o), (bdq, dq), (bdk, dk), (bdv, dv) = rows(B * Sq), rows(B * Sq), rows(B * Sk), rows(B * Sk)
    lse = torch.empty((B, H, Sq), dtype=torch.float32, device="cuda")
    shape = (B, H, Sq, Sk, D, int(causal), 1.0 / np.sqrt(D), dt, stream())
    p = lambda x: x.data_ptr()  # noqa: E731
    call("aic_hip_attn_fwd_qk", p(q), ld, p(k), p(v), ld, p(o), ld, p(lse), *shape)
    call("aic_hip_attn_bwd_qk", p(q), ld, p(k), p(v), ld, p(o), p(do), ld, p(lse), p(dq), ld, p(dk), p(dv), ld, *shape)

    def heads(x, S):
        return np.ascontiguousarray(host(x)[:, :H * D].reshape(B, S, H, D).transpose(0, 2, 1, 3).reshape(B * H, S, D))

    Q, K, V, O, DO = heads(q, Sq), heads(k, Sk), heads(v, Sk), heads(o, Sq), heads(do, Sq)
    o_ref, lse_ref = orc.flash_fwd(Q, K, V, causal)
    L = host(lse).reshape(B * H, Sq)
    assert np.max(np.abs(L - lse_ref)) < (2e-5 if dt == F32 else 1e-3)
    assert rel(O, o_ref) < (2e-6 if dt == F32 else 4e-3)
    tol = 2e-5 if dt == F32 else 8e-3
    for name, got, ref in zip("q k v".split(), (heads(dq, Sq), heads(dk, Sk), heads(dv, Sk)),
                              orc.flash_bwd(Q, K, V, O, DO, L, causal)):
        # one key: dS = P (dP - D) cancels exactly in the reference; then the bound is absolute
        assert np.max(np.abs(got - ref)) < tol if Sk == 1 else rel(got, ref) < tol, name
    for buf, x in ((bo, o), (bdq, dq), (bdk, dk), (bdv, dv)):  # nothing outside the heads was written
        inside = np.zeros(buf.numel(), bool)
        inside[shift:shift + x.numel()].reshape(x.shape)[:, :H * D] = True
        assert np.all(host(buf)[~inside] == 7.0)


@pytest.mark.parametrize("dt", [F32, BF16])
def test_attention_infinities_stay_where_they_are_seen(dt):
    """Causal attention over 37 tokens whose last value row holds an infinity and whose last query
    and key rows are NaN: only the last query's output, and no other row's gradient of the keys
    and queries before it, may show them (the tiles give hidden rows weight zero, and zero times
    an infinity is NaN)."""
    t = torch.float32 if dt == F32 else torch.bfloat16
    S, D = 37, 64
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v, do = (torch.randn((S, D), generator=g, device="cuda").to(t) for _ in range(4))

    def run(q, k, v, do):
        o, lse = torch.empty_like(q), torch.empty((1, 1, S), device="cuda")
        dq, dk, dv = (torch.empty_like(q) for _ in range(3))
        shape = (1, 1, S, S, D, 1, 0.125, dt, stream())
        p = [x.data_ptr() for x in (q, k, v, o, lse, do, dq, dk, dv)]
        call("aic_hip_attn_fwd_qk", p[0], D, p[1], p[2], D, p[3], D, p[4], *shape)
        call("aic_hip_attn_bwd_qk", p[0], D, p[1], p[2], D, p[3], p[5], D, p[4], p[6], D, p[7], p[8], D, *shape)
        return [host(x) for x in (o, dq)]

    clean = run(q, k, v, do)
    v[S - 1, 5] = float("inf")
    dirty = run(q, k, v, do)
    assert np.isinf(dirty[0][S - 1, 5]) and np.all(np.isfinite(np.delete(dirty[0][S - 1], 5)))
    k[S - 1], q[S - 1] = float("nan"), float("nan")
    worse = run(q, k, v, do)
    # the last 16-row tile's sums are formed row by row there: equal up to the order of the sums
    tol = 1e-5 if dt == F32 else 8e-3
    for got in (dirty, worse):
        for a, b in zip(got, clean):
            assert rel(a[:S - 1], b[:S - 1]) < tol


def _visible_only(q, k, v, do, scale):
    """Causal attention and its gradients in float64, each sum over exactly the rows that are seen."""
    S, D = q.shape
    o, dq, dk, dv = (np.zeros((S, D)) for _ in range(4))
    lse = np.zeros(S)
    P, dS = np.zeros((S, S)), np.zeros((S, S))
    for i in range(S):
        s = k[:i + 1] @ q[i] * scale
        m = np.fmax.reduce(s)
        lse[i] = m + np.log(np.sum(np.exp(s - m)))
        P[i, :i + 1] = np.exp(s - lse[i])
        o[i] = np.sum(P[i, :i + 1, None] * v[:i + 1], 0)
    for i in range(S):
        dS[i, :i + 1] = P[i, :i + 1] * (v[:i + 1] @ do[i] - do[i] @ o[i])
        dq[i] = np.sum(dS[i, :i + 1, None] * k[:i + 1], 0) * scale
    for j in range(S):
        dk[j] = np.sum(dS[j:, j, None] * q[j:], 0) * scale
        dv[j] = np.sum(P[j:, j, None] * do[j:], 0)
    return dict(o=o, dq=dq, dk=dk, dv=dv)


INF, NAN = float("inf"), float("nan")
POISON = {"value": [("v", 36, 5, INF)], "first output gradient": [("do", 0, 5, INF)], "first query": [("q", 0, slice(None), NAN)],
          "first rows": [("q", 0, slice(None), NAN), ("do", 0, slice(None), NAN)], "key": [("k", 20, 3, INF)],
          "two values": [("v", 3, 7, -INF), ("v", 3, 9, NAN)], "all": [(n, slice(None), slice(None), NAN) for n in "q k v do".split()]}


@pytest.mark.parametrize("dt", [F32, BF16])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("poison", POISON)
def test_non_finite_rows_as_in_float64(dt, D, poison):
    """Every output and gradient of 70 causal tokens with infinities or NaN in some rows: the same
    entries infinite and NaN as in float64 over the visible rows alone, and the rest within the bounds
    of finite inputs (rows next to a non-finite one are formed row by row, in fp32)."""
    t, S = torch.float32 if dt == F32 else torch.bfloat16, 70
    g = torch.Generator(device="cuda").manual_seed(D)
    x = {n: torch.randn((S, D), generator=g, device="cuda").to(t) for n in ("q", "k", "v", "do")}
    for n, r, c, val in POISON[poison]:
        x[n][r, c] = val
    o, lse = torch.empty_like(x["q"]), torch.empty((1, 1, S), device="cuda")
    dq, dk, dv = (torch.empty_like(o) for _ in range(3))
    scale = 1.0 / np.sqrt(D)
    shape = (1, 1, S, S, D, 1, scale, dt, stream())
    q, k, v, do = (x[n].data_ptr() for n in ("q", "k", "v", "do"))
    call("aic_hip_attn_fwd_qk", q, D, k, v, D, o.data_ptr(), D, lse.data_ptr(), *shape)
    call("aic_hip_attn_bwd_qk", q, D, k, v, D, o.data_ptr(), do, D, lse.data_ptr(), dq.data_ptr(), D, dk.data_ptr(), dv.data_ptr(), D,
         *shape)
    with np.errstate(all="ignore"):
        want = _visible_only(*(host(x[n]).astype(np.float64) for n in ("q", "k", "v", "do")), scale)
    for n, got in dict(o=host(o), dq=host(dq), dk=host(dk), dv=host(dv)).items():
        ref = want[n]
        assert np.array_equal(np.isfinite(got), np.isfinite(ref)) and np.array_equal(np.isnan(got), np.isnan(ref)), n
        assert np.array_equal(got[np.isinf(got)], ref[np.isinf(ref)]), n
        ok = np.isfinite(ref)
        assert rel(got[ok], ref[ok]) < (2e-5 if dt == F32 else 8e-3), n


@pytest.mark.parametrize("dt", [F32, BF16])
def test_non_finite_batches_cost_little_more(dt):
    """16 heads of 64 over 512 causal tokens, NaN throughout and an infinity in every value row, against
    finite rows: about 1 and 10 times their time; formed row by row it was 200 times."""
    t, B, H, S, D = torch.float32 if dt == F32 else torch.bfloat16, 4, 16, 512, 64
    q, k, v, do = (torch.randn((B * S, H * D), device="cuda").to(t) for _ in range(4))
    o, lse = torch.empty_like(q), torch.empty((B, H, S), device="cuda")
    dq, dk, dv = (torch.empty_like(q) for _ in range(3))
    shape = (B, H, S, S, D, 1, 0.125, dt, stream())
    ld = H * D

    def us():
        a, b, best = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True), 1e9
        for _ in range(5):
            a.record()
            for _ in range(4):
                call("aic_hip_attn_fwd_qk", q.data_ptr(), ld, k.data_ptr(), v.data_ptr(), ld, o.data_ptr(), ld, lse.data_ptr(), *shape)
                call("aic_hip_attn_bwd_qk", q.data_ptr(), ld, k.data_ptr(), v.data_ptr(), ld, o.data_ptr(), do.data_ptr(), ld,
                     lse.data_ptr(), dq.data_ptr(), ld, dk.data_ptr(), dv.data_ptr(), ld, *shape)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    finite = us()
    v[:, 1::D] = INF
    assert us() < 30 * finite
    q.fill_(NAN)
    assert us() < 3 * finite
