"""The work that the library's speed is measured on.

Each case is one pass of something that a program using the library runs: the blocks of a training
step at the widths of the bench configurations (forward and backward), the vocabulary end of the
step with its optimizer update, a whole fp32 training step, prompt processing and single-token
decoding with the KV cache, and attention over keys and queries of different lengths.  `listed`
names the sizes that are followed one by one; `draw` gives others of the same ranges.

Widths (bench.py's configurations): 125M d 768, 12 heads, SwiGLU 2048, 12 layers; MoE d 1024,
16 heads, 8 experts of 2816, top-2; 1B d 2048, 16 heads, SwiGLU 5632; tiny d 128, 4 heads, SwiGLU
352, vocabulary 512; vocabulary 32000 otherwise.  Whole models of the 1B widths have two layers.
"""
import ctypes
import math

import numpy as np
import torch

import autonomousaicore_amd as aic
from autonomousaicore_amd import _lib
from autonomousaicore_amd._lib import AIC_BF16, AIC_F16, AIC_F32

WIDTHS = {
    "tiny": dict(V=512, d=128, H=4, f=352, L=2, tied=True),
    "125m": dict(V=32000, d=768, H=12, f=2048, L=12, tied=False),
    "moe": dict(V=32000, d=1024, H=16, f=2816, L=2, tied=False),
    "1b": dict(V=32000, d=2048, H=16, f=5632, L=2, tied=False),
}
MAX_SEQ = 2048
EPS = 1e-6
GROUP = 128       # INT4 group of the QLoRA base
LORA_RANK, LORA_ALPHA = 16, 32.0


def listed():
    return [
        # one token of one sequence through the 125M model with 512 positions cached: chat-style
        # generation, where launches and the weights' read time count
        dict(name="decode_125m_b1", kind="decode", widths="125m", dtype="bf16", lora=False, B=1, pos=512),
        # one token of four sequences on the QLoRA model (INT4 base, rank-16 adapters), 1000 cached
        dict(name="decode_qlora_1b_b4", kind="decode", widths="1b", dtype="bf16", lora=True, B=4, pos=1000),
        # a prompt of 1000 tokens at the 1B widths, every position's logits
        dict(name="prefill_1b_s1000", kind="prefill", widths="1b", dtype="bf16", lora=False, B=1, S=1000),
        # the fp32 reference configuration's training step, gradients read back
        dict(name="train_tiny_fp32", kind="train", d=128, H=4, f=352, L=2, V=512, tied=True, B=8, S=64),
        # the attention half of a 1B layer, forward and backward, at the bench shape
        dict(name="attn_block_1b", kind="attn_block", widths="1b", B=4, S=2048),
        # the same at the 125M widths on a batch that is no multiple of any tile
        dict(name="attn_block_125m_s1000", kind="attn_block", widths="125m", B=3, S=1000),
        # the SwiGLU half of a 1B layer, forward and backward, at the bench shape
        dict(name="ffn_block_1b", kind="ffn_block", widths="1b", T=8192),
        # the same at the 125M widths on a small ragged batch (3 x 333 tokens)
        dict(name="ffn_block_125m_t999", kind="ffn_block", widths="125m", T=999),
        # a chunk of 128 queries against 2048 keys (cross attention, chunked prefill), both directions
        dict(name="attn_qk_128_2048", kind="attn_qk", dtype="bf16", B=4, H=16, hd=128, Sq=128, Sk=2048, causal=False),
        # head product, loss, their gradients, the embedding's, clipping and AdamW of both tables
        dict(name="vocab_end_125m", kind="vocab_end", V=32000, d=768, T=8192),
        # the MoE layer of the MoE configuration, forward and backward
        dict(name="moe_ffn", kind="moe_ffn", d=1024, f=2816, E=8, k=2, T=8192),
        # a QLoRA gate projection at the 1B widths, forward and backward
        dict(name="qlora_linear_1b", kind="qlora_linear", n_in=2048, n_out=5632, rank=16, T=8192),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "train", "attn_block", "attn_block", "ffn_block", "ffn_block",
                       "attn_qk", "vocab_end", "moe_ffn", "qlora_linear"])
    if kind == "decode":
        w, dtype, lora = rng.choice([("125m", "bf16", False), ("1b", "bf16", False), ("1b", "bf16", True),
                                     ("tiny", "f32", False)])
        B = _log(rng, 1, 16)
        return dict(kind=kind, widths=w, dtype=dtype, lora=lora, B=B, pos=_log(rng, 16, min(MAX_SEQ - 8, 16384 // B)))
    if kind == "prefill":
        w, lora = rng.choice([("125m", False), ("1b", False), ("1b", True)])
        B = rng.choice([1, 1, 2, 4])
        return dict(kind=kind, widths=w, dtype="bf16", lora=lora, B=B, S=_log(rng, 8, MAX_SEQ // B))
    if kind == "train":
        d, H, f = rng.choice([(128, 4, 352), (128, 4, 384), (256, 4, 704)])
        return dict(kind=kind, d=d, H=H, f=f, L=rng.choice([2, 4]), V=rng.choice([320, 512]), tied=rng.random() < 0.5,
                    B=_log(rng, 1, 16), S=_log(rng, 16, 512))
    if kind == "attn_block":
        w, B = rng.choice(["125m", "moe", "1b"]), rng.choice([1, 2, 3, 4])
        return dict(kind=kind, widths=w, B=B, S=_log(rng, 32, MAX_SEQ))
    if kind == "ffn_block":
        return dict(kind=kind, widths=rng.choice(["125m", "moe", "1b"]), T=_log(rng, 32, 8192))
    if kind == "attn_qk":
        hd = rng.choice([64, 128])
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "f32"]), B=rng.choice([1, 2, 4]), H=rng.choice([4, 12, 16]),
                    hd=hd, Sq=_log(rng, 1, 512), Sk=_log(rng, 16, 2048), causal=rng.random() < 0.25)
    if kind == "vocab_end":
        V, d = rng.choice([(32000, 768), (32000, 1024), (512, 768)])
        return dict(kind=kind, V=V, d=d, T=_log(rng, 64, 8192))
    if kind == "moe_ffn":
        d, f, E, k = rng.choice([(1024, 2816, 8, 2), (768, 2048, 4, 1)])
        return dict(kind=kind, d=d, f=f, E=E, k=k, T=_log(rng, 16, 8192))
    n_in, n_out = rng.choice([(2048, 2048), (2048, 5632), (5632, 2048), (768, 768)])
    return dict(kind=kind, n_in=n_in, n_out=n_out, rank=rng.choice([8, 16, 32]), T=_log(rng, 1, 8192))


# ------------------------------------------------------------------------------- inputs
# Made from the seed on the GPU; fp64 references (exact) and the library get the same tensors.
class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
        return (torch.randn(*shape, generator=self.g, device="cuda") * std + mean).to(dtype)

    def zipf(self, n, V):
        """Token ids with P(k) ~ 1 / (k + 1)."""
        w = 1.0 / torch.arange(1, V + 1, device="cuda", dtype=torch.float32)
        return torch.multinomial(w, n, replacement=True, generator=self.g)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _call(name, *args):
    _lib.call(name, *[a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args])


def _bf(*shape):
    return torch.empty(*shape, dtype=torch.bfloat16, device="cuda")


def _f32(*shape):
    return torch.empty(*shape, dtype=torch.float32, device="cuda")


def _rope_tables(n, hd):
    """cos, sin [n, hd / 2] in float, as a rotary cache is built."""
    half = hd // 2
    freq = np.float32(1.0) / np.power(np.float32(10000.0), np.arange(half, dtype=np.float32) * 2 / np.float32(hd))
    angle = np.arange(n, dtype=np.float32)[:, None] * freq[None].astype(np.float32)
    return torch.from_numpy(np.cos(angle)).cuda(), torch.from_numpy(np.sin(angle)).cuda()


def _attn_inputs(case, seed):
    w, g = WIDTHS[case["widths"]], _Gen(seed)
    T, d = case["B"] * case["S"], w["d"]
    return dict(x=g.normal(T, d), dy=g.normal(T, d, std=1e-2), wqkv=g.normal(3 * d, d, std=1.5 / math.sqrt(d)),
                wo=g.normal(d, d, std=1 / math.sqrt(d)), nw=g.normal(d, std=0.1, mean=1.0, dtype=torch.float32))


def _ffn_inputs(case, seed):
    w, g = WIDTHS[case["widths"]], _Gen(seed)
    T, d, f = case["T"], w["d"], w["f"]
    return dict(x=g.normal(T, d), dy=g.normal(T, d, std=1e-2), wgu=g.normal(2 * f, d, std=1 / math.sqrt(d)),
                wd=g.normal(d, f, std=1 / math.sqrt(f)), nw=g.normal(d, std=0.1, mean=1.0, dtype=torch.float32))


def _qk_inputs(case, seed):
    g, dt = _Gen(seed), torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    d, nq, nk = case["H"] * case["hd"], case["B"] * case["Sq"], case["B"] * case["Sk"]
    return dict(q=g.normal(nq, d, dtype=dt), k=g.normal(nk, d, dtype=dt), v=g.normal(nk, d, dtype=dt),
                do=g.normal(nq, d, std=1e-2, dtype=dt))


def _vocab_inputs(case, seed):
    g, V, d, T = _Gen(seed), case["V"], case["d"], case["T"]
    ids = g.zipf(T + 1, V)
    return dict(h=g.normal(T, d), ids=ids[:-1].contiguous(), targets=ids[1:].contiguous(),
                head=g.normal(V, d, std=0.02, dtype=torch.float32), emb=g.normal(V, d, std=0.02, dtype=torch.float32))


def _moe_inputs(case, seed):
    g, d, f, E, T = _Gen(seed), case["d"], case["f"], case["E"], case["T"]
    ex = [t for _ in range(E) for t in (g.normal(f * d, std=1 / math.sqrt(d)), g.normal(f * d, std=1 / math.sqrt(d)),
                                        g.normal(d * f, std=1 / math.sqrt(f)))]
    return dict(h=g.normal(T, d), res=g.normal(T, d), dy=g.normal(T, d, std=1e-2),
                router=g.normal(E, d, std=2 / math.sqrt(d)), experts=torch.cat(ex))


def _qlora_inputs(case, seed):
    g, i, o, r, T = _Gen(seed), case["n_in"], case["n_out"], case["rank"], case["T"]
    return dict(x=g.normal(T, i), dy=g.normal(T, o, std=1e-2), w=g.normal(o, i, std=1 / math.sqrt(i), dtype=torch.float32),
                A=g.normal(r, i, std=1 / math.sqrt(i)), Bm=g.normal(o, r, std=0.02))


def _lm_shapes(w):
    d, f, V = w["d"], w["f"], w["V"]
    out = [("tok_embeddings.weight", (V, d))]
    for l in range(w["L"]):
        p = f"layers.{l}."
        out += [(p + f"attn.{n}_proj.weight", (d, d)) for n in ("q", "k", "v", "out")]
        out += [(p + "ffn.gate_proj.weight", (f, d)), (p + "ffn.up_proj.weight", (f, d)),
                (p + "ffn.down_proj.weight", (d, f)), (p + "norm1.weight", (d,)), (p + "norm2.weight", (d,))]
    out.append(("norm.weight", (d,)))
    return out if w["tied"] else out + [("lm_head.weight", (V, d))]


def _lora_shapes(w, r):
    d, f, out = w["d"], w["f"], []
    for l in range(w["L"]):
        p = f"layers.{l}."
        out += [(p + f"attn.{n}_proj.lora_A", (r, d)) for n in "qkv"] + [(p + f"attn.{n}_proj.lora_B", (d, r)) for n in "qkv"]
        out += [(p + "attn.out_proj.lora_A", (r, d)), (p + "attn.out_proj.lora_B", (d, r)),
                (p + "ffn.gate_proj.lora_A", (r, d)), (p + "ffn.up_proj.lora_A", (r, d)),
                (p + "ffn.gate_proj.lora_B", (f, r)), (p + "ffn.up_proj.lora_B", (f, r)),
                (p + "ffn.down_proj.lora_A", (r, f)), (p + "ffn.down_proj.lora_B", (d, r))]
    return out


def _lm_weights(w, g, lora):
    """{name: fp32 tensor} in the arena's order, and the adapters'."""
    def mk(shapes):
        return {n: g.normal(*s, std=0.1, mean=1.0, dtype=torch.float32) if len(s) == 1 else
                g.normal(*s, std=0.02 if "emb" in n or "head" in n else 1 / math.sqrt(s[-1] if "lora" not in n else w["d"]),
                         dtype=torch.float32) for n, s in shapes}
    return mk(_lm_shapes(w)), mk(_lora_shapes(w, LORA_RANK)) if lora else {}


def _lm_case(case):
    if case["kind"] == "train":
        return dict(V=case["V"], d=case["d"], H=case["H"], f=case["f"], L=case["L"], tied=case["tied"]), "f32", False
    return WIDTHS[case["widths"]], case["dtype"], case["lora"]


def _pack(named):
    return torch.cat([t.reshape(-1) for t in named.values()]).cpu().numpy()


def _model(case, g):
    w, dtype, lora = _lm_case(case)
    base, ad = _lm_weights(w, g, lora)
    m = aic.TransformerLM(
        aic.TransformerLMConfig(vocab_size=w["V"], hidden_dim=w["d"], num_layers=w["L"], num_heads=w["H"],
                                intermediate_dim=w["f"], max_seq_len=MAX_SEQ, rms_norm_eps=EPS,
                                tie_word_embeddings=w["tied"], compute="bfloat16" if dtype == "bf16" else "float32",
                                lora_rank=LORA_RANK if lora else 0, lora_alpha=LORA_ALPHA, quant_group=GROUP),
        aic.TrainingConfig(adamw=aic.AdamWOptions(lr=3e-4, beta1=0.9, beta2=0.95, eps=1e-8, weight_decay=0.1)))
    if lora:
        m.set_base_params(_pack(base))
        m.set_params(_pack(ad))
    else:
        m.set_params(_pack(base))
    return m


def _lm_ids(case, g):
    w, _, _ = _lm_case(case)
    if case["kind"] == "decode":
        return g.zipf(case["B"] * (case["pos"] + 1), w["V"]).reshape(case["B"], -1)
    if case["kind"] == "prefill":
        return g.zipf(case["B"] * case["S"], w["V"]).reshape(case["B"], case["S"])
    return g.zipf(case["B"] * (case["S"] + 1), w["V"]).reshape(case["B"], -1)


class _Handle:
    """A native layer that is destroyed with the state that holds it."""

    def __init__(self, make, destroy, *args):
        self.h, self._destroy = ctypes.c_void_p(), destroy
        _lib.call(make, *args, ctypes.byref(self.h))

    def __del__(self):
        _lib.call(self._destroy, self.h)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill", "train"):
        g = _Gen(seed)
        s = dict(case=case, model=_model(case, g))
        ids = _lm_ids(case, g)
        if kind == "decode":   # the prompt is in the cache; the next token comes from the host's sampling
            prompt, logits = ids[:, :-1].contiguous(), _f32(case["B"], case["pos"], _lm_case(case)[0]["V"])
            torch.cuda.synchronize()
            _call("aic_lm_forward_step", s["model"]._h, prompt, case["B"], case["pos"], 0, 1, logits)
            s["model"].synchronize()
            s["next"] = np.ascontiguousarray(ids[:, -1:].cpu().numpy())
        elif kind == "prefill":
            s["ids"] = ids.contiguous()
            s["logits"] = _f32(case["B"], case["S"], _lm_case(case)[0]["V"])
        else:
            s["ids"], s["targets"] = ids[:, :-1].contiguous(), ids[:, 1:].contiguous()
        return s
    if kind == "attn_block":
        w, T, d = WIDTHS[case["widths"]], case["B"] * case["S"], WIDTHS[case["widths"]]["d"]
        s = _attn_inputs(case, seed)
        s["cos"], s["sin"] = _rope_tables(case["S"], d // w["H"])
        s.update(case=case, h=_bf(T, d), rms=_f32(T), qkv=_bf(T, 3 * d), o=_bf(T, d), lse=_f32(T * w["H"]), y=_bf(T, d),
                 do=_bf(T, d), dqkv=_bf(T, 3 * d), dh=_bf(T, d), dx=_bf(T, d), dwqkv=_f32(3 * d, d), dwo=_f32(d, d),
                 dnw=_f32(d))
        return s
    if kind == "ffn_block":
        T, d, f = case["T"], WIDTHS[case["widths"]]["d"], WIDTHS[case["widths"]]["f"]
        s = _ffn_inputs(case, seed)
        s.update(case=case, h=_bf(T, d), rms=_f32(T), gu=_bf(T, 2 * f), act=_bf(T, f), y=_bf(T, d), da=_bf(T, f),
                 dgu=_bf(T, 2 * f), dh=_bf(T, d), dx=_bf(T, d), dwgu=_f32(2 * f, d), dwd=_f32(d, f), dnw=_f32(d))
        return s
    if kind == "attn_qk":
        s = _qk_inputs(case, seed)
        s.update(case=case, o=torch.empty_like(s["q"]), lse=_f32(case["B"], case["H"], case["Sq"]),
                 dq=torch.empty_like(s["q"]), dk=torch.empty_like(s["k"]), dv=torch.empty_like(s["v"]))
        return s
    if kind == "vocab_end":
        V, d, T = case["V"], case["d"], case["T"]
        s = _vocab_inputs(case, seed)
        ctl = _lib.OptimCtl(scale=1024.0, use_scaler=1, growth_factor=2.0, backoff_factor=0.5, growth_interval=1 << 30,
                            min_scale=1.0, max_scale=65536.0, max_grad_norm=1.0)
        s.update(case=case, ctl=torch.frombuffer(bytearray(bytes(ctl)), dtype=torch.uint8).cuda(),
                 head16=s["head"].bfloat16(), emb16=s["emb"].bfloat16(), logits=_bf(T, V), lse=_f32(T), losses=_f32(T),
                 loss=_f32(1), valid=torch.empty(1, dtype=torch.int64, device="cuda"), dh=_bf(T, d), dhead=_f32(V, d),
                 demb=_f32(V, d), sq=torch.empty(1, dtype=torch.float64, device="cuda"),
                 nf=torch.empty(1, dtype=torch.int32, device="cuda"))
        for n in ("head", "emb"):
            s["m_" + n], s["v_" + n] = torch.zeros_like(s[n]), torch.zeros_like(s[n])
        ptrs = ctypes.c_void_p * 2
        s["ptrs"] = {k: ptrs(*[s[n].data_ptr() for n in names]) for k, names in dict(
            p=("head", "emb"), g=("dhead", "demb"), m=("m_head", "m_emb"), v=("v_head", "v_emb"),
            low=("head16", "emb16")).items()}
        s["sizes"] = (ctypes.c_int64 * 2)(V * d, V * d)
        return s
    if kind == "moe_ffn":
        s = _moe_inputs(case, seed)
        s["layer"] = _Handle("aic_moe_ffn_create", "aic_moe_ffn_destroy", case["d"], case["f"], case["E"], case["k"], 0.01,
                             AIC_BF16)
        s.update(case=case, y=torch.empty_like(s["h"]), aux=_f32(1), dh=torch.empty_like(s["h"]),
                 drouter=_f32(case["E"], case["d"]), dexperts=_f32(s["experts"].numel()))
        return s
    s = _qlora_inputs(case, seed)
    n = s["w"].numel()
    s["wq"] = torch.empty(n // 2, dtype=torch.uint8, device="cuda")
    s["scales"] = torch.empty(n // GROUP, dtype=torch.float16, device="cuda")
    _call("aic_hip_int4_quantize", s["w"], n, GROUP, s["wq"], s["scales"], AIC_F16, _stream())
    s["layer"] = _Handle("aic_qlora_linear_create", "aic_qlora_linear_destroy", case["n_in"], case["n_out"], case["rank"],
                         LORA_ALPHA, GROUP, AIC_F16, AIC_BF16)
    s.update(case=case, y=_bf(case["T"], case["n_out"]), dx=_bf(case["T"], case["n_in"]), dA=_f32(case["rank"], case["n_in"]),
             dB=_f32(case["n_out"], case["rank"]))
    del s["w"]
    return s


# ------------------------------------------------------------------------------- one pass
def run(s):
    return RUN[s["case"]["kind"]](s, s["case"])


def _run_decode(s, c):
    return s["model"].forward_step(s["next"], c["pos"])


def _run_prefill(s, c):
    _call("aic_lm_forward_step", s["model"]._h, s["ids"], c["B"], c["S"], 0, 1, s["logits"])
    return s["logits"]


def _run_train(s, c):
    st = s["model"].train_step(s["ids"].data_ptr(), s["targets"].data_ptr(), c["B"], c["S"])
    return dict(loss=st.loss, grad_norm=st.grad_norm, grads=s["model"].get_grads())


def _gemm(ta, tb, M, N, K, A, B, C, R=None, c_type=AIC_BF16):
    """C = op(A) op(B) (+ R), all contiguous."""
    _call("aic_hip_gemm", ta, tb, M, N, K, 1.0, A, M if ta else K, B, K if tb else N, 0.0, C, N, R, N if R is not None else 0,
          AIC_BF16, c_type, _stream())


def _wgrads(T, *ops):
    """dW = dY^T X of each (dY, X, dW) in one launch."""
    d = (_lib.GemmDesc * len(ops))(*[
        _lib.GemmDesc(1, 0, dy.shape[1], x.shape[1], T, dy.data_ptr(), dy.shape[1], x.data_ptr(), x.shape[1], dw.data_ptr(),
                      x.shape[1]) for dy, x, dw in ops])
    _call("aic_hip_gemm_grouped", len(ops), d, 1.0, 0.0, AIC_BF16, AIC_F32, _stream())


def _run_attn_block(s, c):
    w, st = WIDTHS[c["widths"]], _stream()
    B, S, H, d, T = c["B"], c["S"], w["H"], w["d"], c["B"] * c["S"]
    hd, scale = d // H, 1.0 / math.sqrt(d // H)
    _call("aic_hip_rmsnorm_fwd", s["x"], d, s["nw"], s["h"], d, s["rms"], T, d, EPS, AIC_BF16, st)
    _call("aic_hip_gemm_rope", T, 3 * d, d, s["h"], d, s["wqkv"], d, s["qkv"], 3 * d, 2 * d, hd, S, 0, s["cos"], s["sin"], st)
    q = s["qkv"].data_ptr()
    _call("aic_hip_attn_fwd", q, q + 2 * d, q + 4 * d, 3 * d, s["o"], d, s["lse"], B, H, S, hd, 1, scale, AIC_BF16, st)
    _gemm(0, 1, T, d, d, s["o"], s["wo"], s["y"], s["x"])
    # backward of y = x + out_proj(attention(norm(x))) from dy
    _gemm(0, 0, T, d, d, s["dy"], s["wo"], s["do"])
    g = s["dqkv"].data_ptr()
    _call("aic_hip_attn_bwd_rope", q, q + 2 * d, q + 4 * d, 3 * d, s["o"], s["do"], d, s["lse"], g, g + 2 * d, g + 4 * d, 3 * d,
          B, H, S, hd, 1, scale, s["cos"], s["sin"], AIC_BF16, st)
    _wgrads(T, (s["dqkv"], s["h"], s["dwqkv"]), (s["dy"], s["o"], s["dwo"]))
    _gemm(0, 0, T, d, 3 * d, s["dqkv"], s["wqkv"], s["dh"])
    _call("aic_hip_rmsnorm_bwd", s["dh"], d, s["x"], d, s["nw"], s["rms"], s["dy"], d, s["dx"], d, s["dnw"], 0, T, d, AIC_BF16, st)
    return dict(y=s["y"], dx=s["dx"], dwqkv=s["dwqkv"], dwo=s["dwo"], dnw=s["dnw"])


def _run_ffn_block(s, c):
    w, st = WIDTHS[c["widths"]], _stream()
    T, d, f = c["T"], w["d"], w["f"]
    _call("aic_hip_rmsnorm_fwd", s["x"], d, s["nw"], s["h"], d, s["rms"], T, d, EPS, AIC_BF16, st)
    _call("aic_hip_gemm_swiglu", T, f, d, s["h"], d, s["wgu"], d, s["gu"], 2 * f, s["act"], f, st)
    _gemm(0, 1, T, d, f, s["act"], s["wd"], s["y"], s["x"])
    # backward of y = x + down(silu(gate) * up) from dy
    _call("aic_hip_gemm_swiglu_bwd", T, f, d, s["dy"], d, s["wd"], f, s["gu"], 2 * f, s["da"], f, s["dgu"], st)
    _wgrads(T, (s["dgu"], s["h"], s["dwgu"]), (s["dy"], s["act"], s["dwd"]))
    _gemm(0, 0, T, d, 2 * f, s["dgu"], s["wgu"], s["dh"])
    _call("aic_hip_rmsnorm_bwd", s["dh"], d, s["x"], d, s["nw"], s["rms"], s["dy"], d, s["dx"], d, s["dnw"], 0, T, d, AIC_BF16, st)
    return dict(y=s["y"], dx=s["dx"], dwgu=s["dwgu"], dwd=s["dwd"], dnw=s["dnw"])


def _run_attn_qk(s, c):
    d, st, dt = c["H"] * c["hd"], _stream(), AIC_BF16 if c["dtype"] == "bf16" else AIC_F32
    shape = (c["B"], c["H"], c["Sq"], c["Sk"], c["hd"], int(c["causal"]), 1.0 / math.sqrt(c["hd"]), dt, st)
    _call("aic_hip_attn_fwd_qk", s["q"], d, s["k"], s["v"], d, s["o"], d, s["lse"], *shape)
    _call("aic_hip_attn_bwd_qk", s["q"], d, s["k"], s["v"], d, s["o"], s["do"], d, s["lse"], s["dq"], d, s["dk"], s["dv"], d,
          *shape)
    return dict(o=s["o"], lse=s["lse"], dq=s["dq"], dk=s["dk"], dv=s["dv"])


def _run_vocab_end(s, c):
    V, d, T, st, p = c["V"], c["d"], c["T"], _stream(), s["ptrs"]
    _gemm(0, 1, T, V, d, s["h"], s["head16"], s["logits"])
    # the loss scale is the control block's first field
    _call("aic_hip_ce_fwd_bwd", s["logits"], V, s["targets"], T, V, -100, s["losses"], s["lse"], s["loss"], s["valid"], s["ctl"],
          AIC_BF16, st)
    _gemm(1, 0, V, d, T, s["logits"], s["h"], s["dhead"], c_type=AIC_F32)
    _gemm(0, 0, T, d, V, s["logits"], s["head16"], s["dh"])
    _call("aic_hip_embed_bwd", s["ids"], T, s["dh"], V, d, s["demb"], 0, AIC_BF16, st)
    _call("aic_hip_grad_sqnorm_multi", p["g"], s["sizes"], 2, s["sq"], s["nf"], st)
    _call("aic_hip_optim_finalize", s["sq"], s["nf"], s["ctl"], st)
    _call("aic_hip_adamw_multi", p["p"], p["g"], p["m"], p["v"], p["low"], s["sizes"], 2, 3e-4, 0.9, 0.95, 1e-8, 0.1, 0, s["ctl"],
          st)
    return {n: s[n] for n in ("loss", "losses", "dh", "dhead", "demb", "sq", "head", "emb", "m_head", "v_head", "m_emb", "v_emb")}


def _run_moe_ffn(s, c):
    st = _stream()
    _call("aic_moe_ffn_forward", s["layer"].h, s["h"], c["T"], s["router"], s["experts"], s["res"], s["y"], s["aux"], st)
    _call("aic_moe_ffn_backward", s["layer"].h, s["dy"], 1.0, s["dh"], s["drouter"], s["dexperts"], st)
    return dict(y=s["y"], aux=s["aux"], dh=s["dh"], drouter=s["drouter"], dexperts=s["dexperts"])


def _run_qlora_linear(s, c):
    st = _stream()
    _call("aic_qlora_linear_forward", s["layer"].h, s["x"], c["T"], s["wq"], s["scales"], s["A"], s["Bm"], None, s["y"], st)
    _call("aic_qlora_linear_backward", s["layer"].h, s["dy"], s["dx"], s["dA"], s["dB"], 0, st)
    return dict(y=s["y"], dx=s["dx"], dA=s["dA"], dB=s["dB"])


RUN = dict(decode=_run_decode, prefill=_run_prefill, train=_run_train, attn_block=_run_attn_block, ffn_block=_run_ffn_block,
           attn_qk=_run_attn_qk, vocab_end=_run_vocab_end, moe_ffn=_run_moe_ffn, qlora_linear=_run_qlora_linear)


# ------------------------------------------------------------------------------- the least work
def work(c):
    """Inputs and weights read once and results written once; the products' multiply-adds."""
    kind = c["kind"]
    if kind in ("decode", "prefill", "train"):
        w, dtype, lora = _lm_case(c)
        es, d, f, L, V = 2 if dtype == "bf16" else 4, w["d"], w["f"], w["L"], w["V"]
        layer = 4 * d * d + 3 * d * f
        if kind == "train":
            T, P = c["B"] * c["S"], L * layer + V * d
            n = P + (2 * L + 1) * d + (0 if w["tied"] else V * d)
            # weights, gradients and both moments: 28 bytes a parameter; gradients to the host
            return dict(bytes=32.0 * n, flops=6.0 * T * P + 6.0 * L * T * c["S"] * d)
        S, keys = (1, c["pos"] + 1) if kind == "decode" else (c["S"], c["S"])
        T = c["B"] * S
        lr = LORA_RANK * (4 * 2 * d + 3 * (d + f)) if lora else 0
        per_weight = 0.5 + 2.0 / GROUP if lora else es
        kv = 2 * es * c["B"] * keys * d * L
        attn = 4.0 * L * c["B"] * d * (keys if kind == "decode" else S * (S + 1) / 2)
        return dict(bytes=L * (layer * per_weight + lr * es) + V * d * es + kv + 4.0 * T * V,
                    flops=2.0 * T * (L * (layer + lr) + V * d) + attn)
    if kind == "attn_block":
        w = WIDTHS[c["widths"]]
        d, S, T = w["d"], c["S"], c["B"] * c["S"]
        return dict(bytes=2.0 * 4 * T * d + (2 + 4) * 4.0 * d * d, flops=6.0 * T * 4 * d * d + 6.0 * c["B"] * S * (S + 1) * d)
    if kind == "ffn_block":
        w = WIDTHS[c["widths"]]
        d, f, T = w["d"], w["f"], c["T"]
        return dict(bytes=2.0 * 4 * T * d + (2 + 4) * 3.0 * d * f, flops=6.0 * T * 3 * d * f)
    if kind == "attn_qk":
        es, d = 2 if c["dtype"] == "bf16" else 4, c["H"] * c["hd"]
        Sq, Sk = c["Sq"], c["Sk"]
        pairs = Sq * Sk if not c["causal"] else sum(min(i + 1, Sk) for i in range(Sq))
        return dict(bytes=float(es * d * c["B"] * (4 * Sq + 4 * Sk)), flops=14.0 * c["B"] * pairs * d)
    if kind == "vocab_end":
        n = c["V"] * c["d"]
        return dict(bytes=2.0 * 28 * n + 2.0 * 2 * n + 4.0 * c["T"] * c["d"], flops=6.0 * c["T"] * n)
    if kind == "moe_ffn":
        d, f, E, k, T = c["d"], c["f"], c["E"], c["k"], c["T"]
        return dict(bytes=(2 + 4) * 3.0 * E * d * f + 2.0 * 5 * T * d, flops=6.0 * T * k * 3 * d * f + 6.0 * T * E * d)
    i, o, r, T = c["n_in"], c["n_out"], c["rank"], c["T"]
    return dict(bytes=(0.5 + 2.0 / GROUP) * i * o + 2.0 * 2 * T * (i + o) + (2 + 4) * r * (i + o),
                flops=4.0 * T * i * o + 6.0 * T * r * (i + o))


def tolerance(c):
    """About four times the distance from the 64-bit result that the listed and drawn cases show."""
    kind = c["kind"]
    if c.get("dtype") == "f32":
        return {"rel": 1e-5}    # 32-bit sums: 1e-6 seen
    if kind == "train":
        return {"rel": 2e-5}    # the same, and AdamW's first steps carry signs of small gradients on
    # bf16 operands and results, one rounding per stored intermediate: attention with fp32 weights
    # 1.7e-3, the vocabulary end and a QLoRA projection 3e-3, the FFN 4e-3, the attention block 9e-3;
    # whole models add up their layers' roundings (1.4e-2)
    return {"rel": dict(attn_qk=6e-3, vocab_end=1e-2, qlora_linear=1e-2, ffn_block=1.5e-2, moe_ffn=1.5e-2, attn_block=3e-2,
                        decode=4e-2, prefill=4e-2)[kind]}


# ------------------------------------------------------------------------------- in 64 bits
def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rope(x, cos, sin):
    """x [B, S, H, hd], rotated by halves."""
    h = x.shape[-1] // 2
    a, b, cos, sin = x[..., :h], x[..., h:], cos[None, :, None], sin[None, :, None]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _attention(q, k, v, causal):
    """q [B, Sq, H, hd], k and v [B, Sk, H, hd]; query r sees the keys c <= r when causal."""
    out, lse = [], []
    for b in range(q.shape[0]):
        s = torch.matmul(q[b].transpose(0, 1), k[b].permute(1, 2, 0)) / math.sqrt(q.shape[-1])
        if causal:
            hide = torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).triu(1)
            s = s.masked_fill(hide, float("-inf"))
        l = torch.logsumexp(s, -1)
        out.append(torch.matmul(torch.exp(s - l[..., None]), v[b].transpose(0, 1)).transpose(0, 1))
        lse.append(l)
    return torch.stack(out), torch.stack(lse)


def _attn_block64(x, nw, wqkv, wo, B, S, H, cos, sin):
    d = x.shape[-1]
    q, k, v = (_rms(x, nw) @ wqkv.T).reshape(B, S, 3, H, d // H).unbind(2)
    o, _ = _attention(_rope(q, cos, sin), _rope(k, cos, sin), v, True)
    return x + o.reshape(B * S, d) @ wo.T


def _ffn_block64(x, nw, wgu, wd):
    g, u = (_rms(x, nw) @ wgu.T).chunk(2, -1)
    return x + (torch.nn.functional.silu(g) * u) @ wd.T


def _int4_64(w):
    """The weight that the INT4 format holds: groups of GROUP, absmax / 7 scales kept in fp16."""
    x = w.reshape(-1, GROUP)
    s = (x.abs().amax(-1, keepdim=True) / 7.0).clamp_min(1e-8)
    q = x / s
    q = (torch.sign(q) * torch.floor(q.abs() + 0.5)).clamp(-7, 7)
    return (q.double() * s.half().double()).reshape(w.shape)


def _lm64(w, P, ids, lora_scale=None, ad=None, last=False):
    """Logits [B, S, V] of the whole model (last: of the last position, [B, 1, V])."""
    B, S = ids.shape
    d, H = w["d"], w["H"]
    cos, sin = (t.double() for t in _rope_tables(S, d // H))

    def W(n):
        if ad:
            return P[n] + lora_scale * ad[n[:-6] + "lora_B"] @ ad[n[:-6] + "lora_A"]
        return P[n]

    x = P["tok_embeddings.weight"][ids.reshape(-1)]
    for l in range(w["L"]):
        p = f"layers.{l}."
        wqkv = torch.cat([W(p + f"attn.{n}_proj.weight") for n in "qkv"])
        x = _attn_block64(x, P[p + "norm1.weight"], wqkv, W(p + "attn.out_proj.weight"), B, S, H, cos, sin)
        wgu = torch.cat([W(p + "ffn.gate_proj.weight"), W(p + "ffn.up_proj.weight")])
        x = _ffn_block64(x, P[p + "norm2.weight"], wgu, W(p + "ffn.down_proj.weight"))
    head = P["tok_embeddings.weight" if w["tied"] else "lm_head.weight"]
    if last:
        x, S = x.reshape(B, S, d)[:, -1], 1
    return (_rms(x, P["norm.weight"]) @ head.T).reshape(B, S, -1)


def exact(c, seed):
    kind = c["kind"]
    if kind in ("decode", "prefill", "train"):
        w, _, lora = _lm_case(c)
        g = _Gen(seed)
        base, ad = _lm_weights(w, g, lora)
        ids = _lm_ids(c, g)
        if lora:
            base = {n: _int4_64(t) if n.startswith("layers") and t.dim() == 2 else t for n, t in base.items()}
        P = {n: t.double() for n, t in base.items()}
        ad = {n: t.double() for n, t in ad.items()}
        if kind != "train":
            with torch.no_grad():
                return _lm64(w, P, ids, LORA_ALPHA / LORA_RANK, ad, last=kind == "decode")
        for t in P.values():
            t.requires_grad_(True)
        logits = _lm64(w, P, ids[:, :-1])
        loss = torch.nn.functional.cross_entropy(logits.reshape(-1, w["V"]), ids[:, 1:].reshape(-1))
        grads = torch.cat([t.reshape(-1) for t in torch.autograd.grad(loss, list(P.values()))])
        return dict(loss=float(loss), grad_norm=float(grads.norm()), grads=grads)
    if kind in ("attn_block", "ffn_block"):
        s = _attn_inputs(c, seed) if kind == "attn_block" else _ffn_inputs(c, seed)
        t = {n: v.double().requires_grad_(n != "dy") for n, v in s.items()}
        w = WIDTHS[c["widths"]]
        if kind == "attn_block":
            cos, sin = (v.double() for v in _rope_tables(c["S"], w["d"] // w["H"]))
            y = _attn_block64(t["x"], t["nw"], t["wqkv"], t["wo"], c["B"], c["S"], w["H"], cos, sin)
            dx, a, b, dnw = torch.autograd.grad(y, [t["x"], t["wqkv"], t["wo"], t["nw"]], t["dy"])
            return dict(y=y.detach(), dx=dx, dwqkv=a, dwo=b, dnw=dnw)
        y = _ffn_block64(t["x"], t["nw"], t["wgu"], t["wd"])
        dx, a, b, dnw = torch.autograd.grad(y, [t["x"], t["wgu"], t["wd"], t["nw"]], t["dy"])
        return dict(y=y.detach(), dx=dx, dwgu=a, dwd=b, dnw=dnw)
    if kind == "attn_qk":
        t = {n: v.double().reshape(c["B"], -1, c["H"], c["hd"]).requires_grad_(n != "do") for n, v in _qk_inputs(c, seed).items()}
        o, lse = _attention(t["q"], t["k"], t["v"], c["causal"])
        dq, dk, dv = torch.autograd.grad(o, [t["q"], t["k"], t["v"]], t["do"])
        d = c["H"] * c["hd"]
        return dict(o=o.detach().reshape(-1, d), lse=lse.detach(), dq=dq.reshape(-1, d), dk=dk.reshape(-1, d), dv=dv.reshape(-1, d))
    if kind == "vocab_end":
        return _vocab64(c, seed)
    if kind == "moe_ffn":
        return _moe64(c, seed)
    s = _qlora_inputs(c, seed)
    x, dy, A, B = (s[n].double() for n in ("x", "dy", "A", "Bm"))
    W, sc = _int4_64(s["w"]), LORA_ALPHA / c["rank"]
    dxa = sc * dy @ B
    return dict(y=x @ W.T + sc * (x @ A.T) @ B.T, dx=dy @ W + dxa @ A, dA=dxa.T @ x, dB=dy.T @ (sc * x @ A.T))


def _vocab64(c, seed):
    s = _vocab_inputs(c, seed)
    T, V = c["T"], c["V"]
    scale = 1024.0
    h, W = s["h"].double(), s["head"].bfloat16().double()
    z = h @ W.T
    lse = torch.logsumexp(z, -1)
    losses = lse - z.gather(1, s["targets"][:, None])[:, 0]
    g = torch.exp(z - lse[:, None])
    del z
    g[torch.arange(T, device="cuda"), s["targets"]] -= 1.0
    g *= scale / T
    dhead, dh = g.T @ h, g @ W
    del g
    demb = torch.zeros(V, c["d"], dtype=torch.float64, device="cuda").index_add_(0, s["ids"], dh)
    sq = dhead.square().sum() + demb.square().sum()
    norm = sq.sqrt() / scale
    mult = min(1.0, 1.0 / (float(norm) + 1e-6)) / scale
    out = dict(loss=losses.mean().reshape(1), losses=losses, dh=dh, dhead=dhead, demb=demb, sq=sq.reshape(1))
    for n, gr in (("head", dhead), ("emb", demb)):
        gm = gr * mult
        m, v = 0.1 * gm, 0.05 * gm * gm
        p = s[n].double() * (1.0 - 3e-4 * 0.1)
        out[n] = p - 3e-4 * (m / 0.1) / (torch.sqrt(v / 0.05) + 1e-8)
        out["m_" + n], out["v_" + n] = m, v
    return out


def _moe64(c, seed):
    d, f, E, k, T = c["d"], c["f"], c["E"], c["k"], c["T"]
    t = {n: v.double().requires_grad_(n not in ("dy", "res")) for n, v in _moe_inputs(c, seed).items()}
    p = torch.softmax(t["h"] @ t["router"].T, -1)
    top, idx = p.topk(k, -1)
    gate = top / (top.sum(-1, keepdim=True) + 1e-9)
    y = t["res"]
    for e, w in enumerate(t["experts"].reshape(E, 3, f * d)):
        tok, slot = (idx == e).nonzero(as_tuple=True)
        x = t["h"][tok]
        a = torch.nn.functional.silu(x @ w[0].reshape(f, d).T) * (x @ w[1].reshape(f, d).T)
        y = y.index_add(0, tok, gate[tok, slot][:, None] * (a @ w[2].reshape(d, f).T))
    counts = torch.bincount(idx.reshape(-1), minlength=E).double()
    aux = (p.mean(0) * counts).sum() * E * 0.01 / (T * k)
    dh, dr, de = torch.autograd.grad((y * t["dy"]).sum() + aux, [t["h"], t["router"], t["experts"]])
    return dict(y=y.detach(), aux=aux.detach().reshape(1), dh=dh, drouter=dr, dexperts=de)
