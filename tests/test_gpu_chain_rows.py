"""GPU parity of the chain's stages in shared launches, against the same stages as
separate calls through the C ABI (mk.*), which the other tests hold against the
oracle.  Every output has the separate kernels' bits, with two exceptions: normed
where the rows' lanes are not the gather's 256 (it sums the squares of a row in
another order: at most 30 fp32 roundings, 2^-19 relative, so one fp16 ulp), and the
probabilities where the sampling cuts the rows in chunks of another size (one fp16
ulp).  How many launches a run took is counted from a capture, so that each case is
known to have taken the form that it is there for.  A caller that reuses one scratch
buffer for several stages gets the sequential result."""
import ctypes

import numpy as np
import pytest

import mi_chain

pytestmark = pytest.mark.gpu
Stage = mi_chain.Stage


def _launches(w, last):
    """Kernels that a run enqueues: the nodes of its capture (nothing runs)."""
    import torch
    with open("/proc/self/maps") as f:
        path = next(ln.split()[-1] for ln in f if "libamdhip64.so" in ln)
    hip = ctypes.CDLL(path)
    vp = ctypes.c_void_p
    side = torch.cuda.Stream()
    graph, n = vp(), ctypes.c_size_t()
    assert hip.hipStreamBeginCapture(vp(side.cuda_stream), 2) == 0  # relaxed mode
    try:
        w.run(last, stream=side)
    finally:
        assert hip.hipStreamEndCapture(vp(side.cuda_stream), ctypes.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    return n.value


def _work(dev, D, double, seed=3, n_decode=5, **kw):
    return mi_chain.Workload(dev, seed=seed, n_decode=n_decode, prefills=(3,), logit_rows=2,
                             hidden_size=D, intermediate_size=64, num_heads=2, num_kv_heads=1,
                             head_dim=16, vocab=200, double_norm=int(double),
                             norm_add_one=int(double), embed_scale=int(double), **kw)


def _one_by_one(mk, w):
    """The row-wise stages as separate calls; the tensors by the chain's names."""
    t, c = w.t, w.cfg
    add1, eps = bool(c["norm_add_one"]), c["rms_eps"]
    scale = float(np.sqrt(np.float32(c["hidden_size"]))) if c["embed_scale"] else 1.0
    attn, mlp = t["attn_out"].clone(), t["mlp_out"].clone()
    hidden, normed = mk.embedding_rmsnorm(t["ids"], t["embed"], t["input_norm"], scale=scale,
                                          eps=eps, add_one=add1)
    if c["double_norm"]:
        mk.rmsnorm(attn, t["post_attn_norm"], y=attn, eps=eps, add_one=add1)
        mk.rmsnorm(mlp, t["post_ff_norm"], y=mlp, eps=eps, add_one=add1)
    post = mk.fused_add_rmsnorm(attn, hidden, t["pre_ff_norm" if c["double_norm"] else
                                                "post_attn_norm"], eps=eps, add_one=add1)
    fin = mk.fused_add_rmsnorm(mlp, hidden, t["final_norm"], eps=eps, add_one=add1)
    return dict(hidden=hidden, normed=normed, post_normed=post, final_normed=fin, attn_out=attn,
                mlp_out=mlp)


def _rope_and_cache(mk, w):
    """Rotation and cache writes as separate calls; the tensors by the chain's names."""
    t, c, s = w.t, w.cfg, w.shapes
    Hkv, hd = c["num_kv_heads"], c["head_dim"]
    q, k, v = (t[n].clone() for n in "qkv")
    kc, vc = t["k_cache"].clone(), t["v_cache"].clone()
    inv = mk.rope_inv_freq(hd, c["rope_theta"])
    if c["use_qk_norm"]:
        mk.qk_norm_rope(q, k, t["q_norm"], t["k_norm"], t["positions"], inv, eps=c["qk_norm_eps"])
    elif c["qkv_bias"]:
        mk.bias_rope_neox_qk(q, k, t["q_bias"], t["k_bias"], t["positions"], inv)
    else:
        mk.rope_neox_qk(q, k, t["positions"], inv)
    for g in w.segments:
        B, S, at = g["B"], g["S"], g["token_offset"]
        part = slice(at, at + B * S)
        mk.paged_kv_scatter(k[part].view(B, S, Hkv, hd), kc, g["block_table"], g["seq_len"],
                            g["start_pos"], s["layer"], s["block_size"],
                            v_src=v[part].view(B, S, Hkv, hd), v_cache=vc,
                            v_bias=t["v_bias"] if c["qkv_bias"] else None)
    return dict(q=q, k=k, v=v, k_cache=kc, v_cache=vc)


def _ulps(a, b):
    """Largest distance in fp16 values between a and b."""
    def order(x):
        i = x.cpu().numpy().view(np.int16).astype(np.int32)
        return np.where(i < 0, -32768 - i, i)
    return int(np.abs(order(a) - order(b)).max())


def _assert_rows(w, want):
    """Bits, but for normed where a token's lanes hold several vectors each and are
    fewer than 256 (chain_step.hip: the fewest wavefronts, as the row norms')."""
    import torch
    D = w.cfg["hidden_size"]
    vectors = D // 8
    per_lane = -(-vectors // 256)
    lanes = -(-(-(-vectors // per_lane)) // 64) * 64
    shared = D % 8 == 0 and D <= 8192  # rows that one launch takes
    for n, ref in want.items():
        if n == "normed" and shared and per_lane > 1 and lanes < 256:
            assert _ulps(w.t[n], ref) <= 1, n
        else:
            assert torch.equal(w.t[n], ref), n


# one vector, the edges of the vectors per lane, fewer lanes than 256, the longest
# row, and rows the single launch does not take
@pytest.mark.parametrize("D", [8, 520, 2040, 2048, 2056, 2560, 4104, 6152, 8192, 8200, 100])
@pytest.mark.parametrize("double", [False, True])
def test_rows_in_one_launch(mk, dev, D, double):
    import torch
    print(f"[case] chain rows D={D} double={double}", flush=True)
    w = _work(dev, D, double)
    w.t["ids"][2] = -1    # zero rows
    w.t["ids"][3] = 200
    want = _one_by_one(mk, w)
    # rows, RoPE + cache, activation; or the rows' stages apart
    shared = D % 8 == 0 and D <= 8192
    assert _launches(w, Stage.FINAL_NORM) == (3 if shared else 7 if double else 5)
    w.run(Stage.FINAL_NORM)
    torch.cuda.synchronize()
    _assert_rows(w, want)


@pytest.mark.parametrize("double", [False, True])
def test_shared_scratch_keeps_the_order(mk, dev, double):
    """normed, post_normed and final_normed one buffer; mlp_out normalised into it."""
    import torch
    print(f"[case] chain rows, one scratch buffer, double={double}", flush=True)
    w = _work(dev, 256, double)
    want = _one_by_one(mk, w)
    w.t["post_normed"] = w.t["final_normed"] = w.t["normed"]
    w.desc, w.keep = mi_chain.make_desc(w.shapes, w.t, w.segments)
    w.run(Stage.FINAL_NORM)
    torch.cuda.synchronize()
    assert torch.equal(w.t["hidden"], want["hidden"])
    assert torch.equal(w.t["final_normed"], want["final_normed"])


# one slot per lane exactly, one unit more, two and three slots, and past them
@pytest.mark.parametrize("Hq,Hkv,hd", [(28, 4, 128), (32, 1, 128), (32, 8, 128), (24, 24, 128),
                                       (64, 8, 128), (80, 16, 128), (96, 8, 128), (32, 32, 80),
                                       (40, 1, 256), (5, 60, 64)])
@pytest.mark.parametrize("kind", ["plain", "bias", "norm"])
def test_wide_tokens_into_the_cache(mk, dev, Hq, Hkv, hd, kind):
    """RoPE and the cache writes in the chain's one launch against the RoPE entry
    point and the scatters, bit for bit."""
    import torch
    if kind == "norm" and hd == 80:
        pytest.skip("the norm takes heads of 16 * 2^k")
    print(f"[case] chain rope + scatter {Hq}|{Hkv}x{hd} {kind}", flush=True)
    w = mi_chain.Workload(dev, seed=Hq * hd + Hkv, n_decode=7, prefills=(37, 37), logit_rows=2,
                          hidden_size=64, intermediate_size=64, num_heads=Hq, num_kv_heads=Hkv,
                          head_dim=hd, vocab=200, use_qk_norm=int(kind == "norm"),
                          qkv_bias=int(kind == "bias"))
    want = _rope_and_cache(mk, w)
    # gather + norm, RoPE + cache; past three units per lane RoPE and a scatter for
    # each of the two segments
    slots = max((Hq + Hkv) * hd // 16, Hkv * hd // 8)
    assert _launches(w, Stage.KV_SCATTER) == (2 if slots <= 768 else 4)
    w.run(Stage.KV_SCATTER)
    torch.cuda.synchronize()
    for n, ref in want.items():
        assert torch.equal(w.t[n], ref), n


SMALL = dict(hidden_size=64, intermediate_size=72, num_heads=2, num_kv_heads=1, head_dim=64,
             vocab=9000, use_qk_norm=0)


# one token; the tiles' and vectors' edges; every rotation and head width; chunks of
# either size, ragged vocabularies; more chunks than one launch keeps resident (the
# sampling apart), rows that softmax takes whole (its two halves apart); and steps that
# the launch does not take: rows, rotation, activation (7 columns: with a launch for
# the remainder) and sampling apart
@pytest.mark.parametrize("n_decode,prefill,rows,kw,launches", [
    (1, 0, 1, {}, 1),
    (3, 0, 2, dict(vocab=8192, hidden_size=2048, intermediate_size=2048), 1),
    (5, 6, 3, dict(vocab=8201, hidden_size=2056, head_dim=128, qkv_bias=1), 1),
    (2, 40, 9, dict(vocab=16391, hidden_size=4096, num_heads=28, num_kv_heads=5, head_dim=128,
                    use_qk_norm=1), 1),
    (7, 33, 5, dict(head_dim=256, num_heads=8, num_kv_heads=4, use_qk_norm=1, double_norm=1,
                    norm_add_one=1, embed_scale=1, act=1), 1),
    (4, 0, 60, dict(vocab=152064, num_heads=4, qkv_bias=1), 1),
    (4, 0, 24, dict(vocab=262144, double_norm=1), 1),
    (4, 0, 128, dict(vocab=152064), 2),
    (4, 0, 500, dict(vocab=32001), 3),
    (4, 0, 3, dict(hidden_size=4104), 4),
    (4, 0, 3, dict(intermediate_size=7), 5),
    (4, 0, 3, dict(head_dim=80), 4),
])
@pytest.mark.parametrize("polls", [True, False])
def test_step_in_one_launch(mk, dev, n_decode, prefill, rows, kw, launches, polls):
    """A whole step against its stages as separate calls."""
    import torch
    print(f"[case] step T={n_decode + 2 * prefill} rows={rows} {kw} polls={polls}", flush=True)
    w = mi_chain.Workload(dev, seed=11, n_decode=n_decode, prefills=(prefill,) * 2 if prefill else (),
                          logit_rows=rows, **dict(SMALL, **kw))
    t = w.t
    norms, same = _one_by_one(mk, w), _rope_and_cache(mk, w)
    same["act_out"] = (mk.geglu if w.cfg["act"] else mk.swiglu)(t["gate"], t["up"])
    for n in ("gate", "up", "logits"):
        same[n] = t[n].clone()
    probs, tokens = mk.softmax_argmax(t["logits"], torch.zeros_like(t["sample_ws"]))
    assert set(norms) | set(same) | {"probs", "next_tokens"} == set(mi_chain._BUFS)
    assert _launches(w, Stage.SAMPLE) == launches
    prev = mk.softmax_test_poll_limit(1 << 16 if polls else 0)
    try:
        for i in range(2):  # the records serve the next call
            if i:
                w.reload("q", "k", "attn_out", "mlp_out")
                for n in ("k_cache", "v_cache", "probs", "act_out", "hidden", *list(norms)[1:4]):
                    t[n].zero_()
            w.run()
            torch.cuda.synchronize()
            _assert_rows(w, norms)
            for n, ref in same.items():
                assert torch.equal(t[n], ref), n
            assert torch.equal(t["next_tokens"], tokens)
            assert _ulps(t["probs"], probs) <= 1
    finally:
        mk.softmax_test_poll_limit(prev)
