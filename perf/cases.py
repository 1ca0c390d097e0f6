"""The layer-kernel library's work as a program that serves a language model has it
do, one case per kind of call, through the Python entry points (mi_kernels,
mi_chain).

A case is a dict with a "kind":

  step     one decoder layer's non-GEMM launches and the sampling step, issued by
           one mi_chain call over a packed batch of decode and prefill tokens
  norm     the residual add + RMSNorm, or the RMSNorm alone, of a block of tokens
  act      the gated activation between the MLP's products
  softmax  attention probabilities: one row per (head, query), as long as the keys
  sample   the sampling step over a batch's logits
  rope     rotary embedding of Q and K, in each of the forms the models need
  embed    the embedding gather, alone or with the first norm

Model shapes are in MODELS; everything is fp16, as the library takes it.  The
GEMM outputs that a step starts from are random tensors of the activations'
scale.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "mini-infer_amd"))

import mi_chain  # noqa: E402
import mi_kernels as mk  # noqa: E402

F16 = torch.float16

MODELS = {
    # Qwen2.5-7B: projection bias, no Q/K norm
    "qwen2.5-7b": dict(use_qk_norm=0, qkv_bias=1),
    # the same widths with the per-head Q/K norm
    "qk-norm-7b": dict(use_qk_norm=1, qkv_bias=0),
    # eight KV heads, neither bias nor Q/K norm
    "gqa8-8b": dict(hidden_size=4096, intermediate_size=14336, num_heads=32, num_kv_heads=8,
                    vocab=128256, rope_theta=5e5, use_qk_norm=0, qkv_bias=0),
    # a small model: 64-wide heads, two KV heads, projection bias
    "small-64": dict(hidden_size=896, intermediate_size=4864, num_heads=14, num_kv_heads=2,
                     head_dim=64, vocab=151936, use_qk_norm=0, qkv_bias=1),
    # Gemma 3's form: (1 + w) norms, scaled embedding, norms around both blocks, GeGLU
    "gemma-256": dict(hidden_size=2560, intermediate_size=10240, num_heads=8, num_kv_heads=4,
                      head_dim=256, vocab=262144, use_qk_norm=1, qkv_bias=0, norm_add_one=1,
                      embed_scale=1, double_norm=1, act=1),
}

HIDDEN = (896, 1152, 1536, 2048, 2560, 3072, 3584, 4096, 5120, 6144, 8192)
INTER = (4864, 8960, 10240, 11008, 13824, 14336, 18944)
HEADS = ((28, 4, 128), (32, 8, 128), (14, 2, 64), (8, 4, 256), (16, 16, 64), (32, 32, 80),
         (64, 8, 128))
# padded vocabularies, and ones their tokenizer left as they are
VOCABS = (32000, 32001, 49153, 50257, 128256, 151643, 151936, 152064)
MAX_START = 28000


def listed():
    return [
        # one user's next token: the latency of seven small launches
        dict(name="step_decode_1", kind="step", model="qwen2.5-7b", n_decode=1, prefills=0,
             prefill_len=0),
        # a decode batch of the Gemma form, every option on
        dict(name="step_decode_24_gemma", kind="step", model="gemma-256", n_decode=24, prefills=0,
             prefill_len=0),
        # a decode batch with one chunk of a prompt, grouped-query heads
        dict(name="step_chunk_1048_gqa8", kind="step", model="gqa8-8b", n_decode=37, prefills=1,
             prefill_len=1011),
        # continuous batching at full load: 64 decodes beside two long prompts
        dict(name="step_mixed_6064", kind="step", model="qwen2.5-7b", n_decode=64, prefills=2,
             prefill_len=3000),
        # the headline: residual add + norm of a large prefill
        dict(name="norm_8192", kind="norm", T=8192, D=3584, fused=True, add_one=False),
        # the same of a short prompt, a wider model and (1 + w) weights
        dict(name="norm_333_wide", kind="norm", T=333, D=5120, fused=True, add_one=True),
        # a prompt through GeGLU
        dict(name="act_geglu_2047", kind="act", T=2047, I=10240, gelu=True),
        # attention probabilities, a batch of four at 512 keys (28 heads)
        dict(name="softmax_512", kind="softmax", N=57344, D=512),
        # and of one prompt chunk against a cache of a length as it comes
        dict(name="softmax_1203", kind="softmax", N=28 * 611, D=1203),
        # the sampling step over a vocabulary that is no multiple of anything
        dict(name="sample_48x50257", kind="sample", N=48, V=50257, form="softmax_argmax"),
        # RoPE of a prefill
        dict(name="rope_4096", kind="rope", T=4096, Hq=28, Hkv=4, hd=128, form="plain"),
        # the first layer's gather + norm of a prefill, wide rows
        dict(name="embed_2048_wide", kind="embed", T=2048, D=8192, V=128256, norm=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("step", "step", "norm", "act", "softmax", "sample", "rope", "embed"))
    if kind == "step":
        prefills = rng.choice((0, 0, 1, 2))
        return dict(kind=kind, model=rng.choice(sorted(MODELS)), n_decode=_log_int(rng, 2, 64),
                    prefills=prefills, prefill_len=_log_int(rng, 16, 2800) if prefills else 0)
    if kind == "norm":
        return dict(kind=kind, T=_log_int(rng, 1, 8192), D=rng.choice(HIDDEN),
                    fused=rng.random() < 0.7, add_one=rng.random() < 0.4)
    if kind == "act":
        return dict(kind=kind, T=_log_int(rng, 1, 4096), I=rng.choice(INTER),
                    gelu=rng.random() < 0.4)
    if kind == "softmax":
        D = _log_int(rng, 16, 4096)
        return dict(kind=kind, N=_log_int(rng, 28, min(57344, 100_000_000 // D)), D=D)
    if kind == "sample":
        form = rng.choice(("softmax_argmax", "argmax", "softmax", "top_p"))
        V = _log_int(rng, 2000, 30000) if form == "top_p" else rng.choice(VOCABS)
        return dict(kind=kind, N=_log_int(rng, 1, 256), V=V, form=form)
    if kind == "rope":
        Hq, Hkv, hd = rng.choice(HEADS)
        form = rng.choice(("plain", "bias", "tables", "norm"))
        if form == "norm" and hd == 80:  # the norm form takes 16 * 2^k wide heads
            form = "plain"
        return dict(kind=kind, T=_log_int(rng, 1, 6064), Hq=Hq, Hkv=Hkv, hd=hd, form=form)
    return dict(kind="embed", T=_log_int(rng, 1, 6064), D=rng.choice(HIDDEN),
                V=rng.choice((32000, 50257, 128256)), norm=rng.random() < 0.6)


# --- the step ---------------------------------------------------------------

def _model(case):
    return dict(mi_chain.QWEN25_7B, **MODELS[case["model"]])


def _step_shape(case):
    m = _model(case)
    T = case["n_decode"] + case["prefills"] * case["prefill_len"]
    N = case["n_decode"] + case["prefills"]  # one row of logits per sequence
    return m, T, N


STEP_OUT = ("hidden", "normed", "q", "k", "k_cache", "v_cache", "post_normed", "act_out",
            "final_normed", "probs", "next_tokens")


def _prepare_step(case, seed):
    m, T, N = _step_shape(case)
    w = mi_chain.Workload(torch.device("cuda:0"), seed=seed, n_decode=case["n_decode"],
                          prefills=(case["prefill_len"],) * case["prefills"], logit_rows=N,
                          num_layers=2, layer=1, host=False, **MODELS[case["model"]])
    # a KV pool of the engine's own size, the same whatever blocks the batch falls on
    blocks = case["n_decode"] + case["prefills"] * (case["prefill_len"] // 16 + 2) + 64
    for name in ("k_cache", "v_cache"):
        w.t[name] = torch.zeros((2, blocks, m["num_kv_heads"], 16, m["head_dim"]), dtype=F16,
                                device="cuda:0")
    w.shapes["num_blocks"] = blocks
    w.desc, w.keep = mi_chain.make_desc(w.shapes, w.t, w.segments)
    return w


def _run_step(w):
    w.run()
    return {n: w.t[n] for n in STEP_OUT}


def _exact_step(case, seed):
    w = _prepare_step(case, seed)
    m, T, N = _step_shape(case)
    t = {n: v for n, v in w.t.items() if v is not None}
    Hq, Hkv, hd = m["num_heads"], m["num_kv_heads"], m["head_dim"]
    one = m["norm_add_one"]

    def norm(x, name):
        return _norm64(x, t[name], m["rms_eps"], one)

    out = {}
    h = t["embed"][t["ids"]].double()
    if m["embed_scale"]:
        h = h * math.sqrt(m["hidden_size"])
    out["normed"] = norm(h, "input_norm")
    q, k, v = (t[n].double() for n in "qkv")
    if m["qkv_bias"]:
        q = q + t["q_bias"].double().view(1, Hq, hd)
        k = k + t["k_bias"].double().view(1, Hkv, hd)
        v = v + t["v_bias"].double().view(1, Hkv, hd)
    if m["use_qk_norm"]:
        q = _norm64(q, t["q_norm"], m["qk_norm_eps"], 0)
        k = _norm64(k, t["k_norm"], m["qk_norm_eps"], 0)
    q, k = (_rope64(x, t["positions"], m["rope_theta"]) for x in (q, k))
    out["q"], out["k"] = q, k
    for name, rows in (("k_cache", k), ("v_cache", v)):
        cache = t[name].double()
        for g in w.segments:
            bs = cache.shape[3]
            s = torch.arange(g["S"], device=cache.device)
            pos = g["start_pos"].long()[:, None] + s[None, :]
            phys = torch.gather(g["block_table"].long(), 1, pos // bs)
            part = rows[g["token_offset"]:g["token_offset"] + g["B"] * g["S"]]
            cache[1][phys.reshape(-1), :, (pos % bs).reshape(-1)] = part
        out[name] = cache
    x = t["attn_out"].double()
    if m["double_norm"]:
        h = h + norm(x, "post_attn_norm")
        out["post_normed"] = norm(h, "pre_ff_norm")
    else:
        h = h + x
        out["post_normed"] = norm(h, "post_attn_norm")
    out["act_out"] = _act64(t["gate"], t["up"], bool(m["act"]))
    x = t["mlp_out"].double()
    h = h + (norm(x, "post_ff_norm") if m["double_norm"] else x)
    out["hidden"], out["final_normed"] = h, norm(h, "final_norm")
    out["probs"] = torch.softmax(t["logits"].double(), -1)
    out["next_tokens"] = None
    return {n: out[n] for n in STEP_OUT}


# --- the same in 64 bits ----------------------------------------------------

def _norm64(x, w, eps, add_one):
    x = x.double()
    w = w.double() + (1.0 if add_one else 0.0)
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _rope64(x, positions, theta):
    """NeoX rotation of x [T, H, hd]; the angle is the fp32 product of the position and
    the fp32 inverse frequency, as the library defines it."""
    hd = x.shape[-1]
    inv = torch.from_numpy(mk.rope_inv_freq(hd, theta)).to(x.device)
    ang = (positions.float()[:, None] * inv[None, :]).double()[:, None, :]
    c, s = torch.cos(ang), torch.sin(ang)
    a, b = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _act64(gate, up, gelu):
    g, u = gate.double(), up.double()
    return (torch.nn.functional.gelu(g, approximate="tanh") if gelu
            else torch.nn.functional.silu(g)) * u


# --- every kind -------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        return "step", None, _prepare_step(case, seed)
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(seed)

    def r(shape, mean=0.0, std=1.0):
        return torch.randn(shape, generator=gen, device=dev).mul_(std).add_(mean).to(F16)

    def e(shape, dtype=F16):
        return torch.empty(shape, dtype=dtype, device=dev)

    s = {}
    if kind == "norm":
        T, D = case["T"], case["D"]
        s.update(x=r((T, D)), y=e((T, D)))
        s["w"] = r((D,), 0.0 if case["add_one"] else 1.0, 0.1)
        if case["fused"]:
            s["res"] = r((T, D))
    elif kind == "act":
        T, I = case["T"], case["I"]
        s.update(gate=r((T, I)), up=r((T, I)), out=e((T, I)))
    elif kind == "softmax":
        s.update(x=r((case["N"], case["D"]), 0.0, 2.0), y=e((case["N"], case["D"])))
    elif kind == "sample":
        N, V, form = case["N"], case["V"], case["form"]
        s.update(x=r((N, V), 0.0, 4.0), out=e((N,), torch.int32))
        nbytes = {"softmax_argmax": mk.softmax_argmax_workspace_bytes,
                  "argmax": mk.greedy_argmax_workspace_bytes,
                  "softmax": mk.softmax_workspace_bytes}.get(form, lambda n, v: 0)(N, V)
        s["ws"] = torch.zeros(max(16, nbytes), dtype=torch.uint8, device=dev)
        if form.startswith("softmax"):
            s["y"] = e((N, V))
    elif kind == "rope":
        T, Hq, Hkv, hd = case["T"], case["Hq"], case["Hkv"], case["hd"]
        start = int(torch.randint(0, MAX_START, (1,), generator=gen, device=dev))
        s.update(q=r((T, Hq, hd)), k=r((T, Hkv, hd)),
                 pos=torch.arange(start, start + T, device=dev), inv=mk.rope_inv_freq(hd))
        if case["form"] == "bias":
            s.update(bq=r((Hq * hd,), 0.0, 0.5), bk=r((Hkv * hd,), 0.0, 0.5))
        elif case["form"] == "norm":
            s.update(wq=r((hd,), 1.0, 0.1), wk=r((hd,), 1.0, 0.1))
        elif case["form"] == "tables":
            s.update(cos=e((T, hd // 2)), sin=e((T, hd // 2)), yq=e((1, T, Hq, hd)),
                     yk=e((1, T, Hkv, hd)))
    else:
        T, D, V = case["T"], case["D"], case["V"]
        s.update(table=r((V, D), 0.0, 0.02), h=e((T, D)),
                 ids=torch.randint(0, V, (T,), generator=gen, device=dev))
        if case["norm"]:
            s.update(w=r((D,), 1.0, 0.1), y=e((T, D)))
    return kind, case, s


def run(state):
    kind, case, s = state
    if kind == "step":
        return _run_step(s)
    if kind == "norm":
        if case["fused"]:
            mk.fused_add_rmsnorm(s["x"], s["res"], s["w"], y=s["y"], add_one=case["add_one"])
            return s["res"], s["y"]
        return mk.rmsnorm(s["x"], s["w"], y=s["y"], add_one=case["add_one"])
    if kind == "act":
        return (mk.geglu if case["gelu"] else mk.swiglu)(s["gate"], s["up"], out=s["out"])
    if kind == "softmax":
        return mk.softmax(s["x"], y=s["y"])
    if kind == "sample":
        form = case["form"]
        if form == "softmax_argmax":
            return mk.softmax_argmax(s["x"], s["ws"], probs=s["y"], out=s["out"])
        if form == "softmax":
            return mk.softmax(s["x"], y=s["y"], workspace=s["ws"])
        if form == "argmax":
            return mk.greedy_argmax(s["x"], out=s["out"], workspace=s["ws"])
        return mk.top_p_sample(s["x"], 0.9, 0.8, 1234, out=s["out"])
    if kind == "rope":
        form = case["form"]
        if form == "bias":
            return mk.bias_rope_neox_qk(s["q"], s["k"], s["bq"], s["bk"], s["pos"], s["inv"])
        if form == "norm":
            return mk.qk_norm_rope(s["q"], s["k"], s["wq"], s["wk"], s["pos"], s["inv"])
        if form == "plain":
            return mk.rope_neox_qk(s["q"], s["k"], s["pos"], s["inv"])
        mk.rope_tables(s["inv"], s["pos"], s["cos"], s["sin"])
        return (mk.rope_neox(s["q"][None], s["cos"], s["sin"], y=s["yq"]),
                mk.rope_neox(s["k"][None], s["cos"], s["sin"], y=s["yk"]))
    if case["norm"]:
        return mk.embedding_rmsnorm(s["ids"], s["table"], s["w"], hidden=s["h"], y=s["y"])
    return mk.embedding_gather(s["ids"], s["table"], out=s["h"])


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "sample" and case["form"] in ("argmax", "top_p"):
        return None  # token indices
    s = prepare(case, seed)[2]
    if kind == "norm":
        x = s["x"].double()
        if case["fused"]:
            x = x + s["res"].double()
            return x, _norm64(x, s["w"], 1e-6, case["add_one"])
        return _norm64(x, s["w"], 1e-6, case["add_one"])
    if kind == "act":
        return _act64(s["gate"], s["up"], case["gelu"])
    if kind in ("softmax", "sample"):
        y = torch.softmax(s["x"].double(), -1)
        return (y, None) if kind == "sample" and case["form"] == "softmax_argmax" else y
    if kind == "rope":
        q, k = s["q"].double(), s["k"].double()
        if case["form"] == "bias":
            q = q + s["bq"].double().view(1, *q.shape[1:])
            k = k + s["bk"].double().view(1, *k.shape[1:])
        elif case["form"] == "norm":
            q, k = _norm64(q, s["wq"], 1e-6, 0), _norm64(k, s["wk"], 1e-6, 0)
        q, k = _rope64(q, s["pos"], 1e6), _rope64(k, s["pos"], 1e6)
        return (q[None], k[None]) if case["form"] == "tables" else (q, k)
    h = s["table"][s["ids"]].double()
    return (h, _norm64(h, s["w"], 1e-6, 0)) if case["norm"] else h


def work(case):
    """Bytes: each input read once, each output written once.  Operations: a few per
    element, far below any rate that could bound a pass."""
    kind = case["kind"]
    if kind == "step":
        m, T, N = _step_shape(case)
        D, I, V = m["hidden_size"], m["intermediate_size"], m["vocab"]
        Hq, Hkv, hd = m["num_heads"], m["num_kv_heads"], m["head_dim"]
        # tokens: the embedding row, attn_out and mlp_out read; hidden and three norms written
        # (the step's residual stream, one layer deep); q, k rotated in place, v read, both
        # cached; gate, up read, act written
        per = 2 * (7 * D + 2 * (Hq + Hkv) * hd + 3 * Hkv * hd + 3 * I) + 16
        if m["double_norm"]:
            per += 2 * 2 * D  # both blocks' outputs normalised in place
        elems = T * (7 * D + 2 * (Hq + Hkv) * hd + I) + N * V
        return {"bytes": T * per + N * (4 * V + 4) + 2 * 5 * D, "flops": 8 * elems}
    if kind == "norm":
        n = case["T"] * case["D"]
        return {"bytes": (8 if case["fused"] else 4) * n + 2 * case["D"], "flops": 5 * n}
    if kind == "act":
        n = case["T"] * case["I"]
        return {"bytes": 6 * n, "flops": 12 * n}
    if kind == "softmax":
        n = case["N"] * case["D"]
        return {"bytes": 4 * n, "flops": 5 * n}
    if kind == "sample":
        n = case["N"] * case["V"]
        probs = case["form"].startswith("softmax")
        return {"bytes": (4 if probs else 2) * n + 4 * case["N"], "flops": 5 * n}
    if kind == "rope":
        T, hd = case["T"], case["hd"]
        n = T * (case["Hq"] + case["Hkv"]) * hd
        tables = T * hd * 2 if case["form"] == "tables" else 0
        return {"bytes": 4 * n + 8 * T + tables, "flops": 6 * n}
    n = case["T"] * case["D"]
    return {"bytes": (6 if case["norm"] else 4) * n + 8 * case["T"], "flops": 5 * n}


def tolerance(case):
    """Results are fp16, rounded once from fp32: a correct implementation differs from
    another where its fp32 value falls on the other side of a rounding boundary, by one
    fp16 ulp (2^-10 of the value).  Against torch's fp32 forms, rounded at the same
    places, over these ranges: at most 1.7e-5 in the 2-norm, 9.8e-4 at one value."""
    kind = case["kind"]
    if kind == "embed" and not case["norm"]:
        return "exact"
    if kind == "rope" and case["form"] != "norm":
        return "exact"  # both products of the rotation are exact in fp32
    return {"rel": 7e-5, "max": 4e-3}
