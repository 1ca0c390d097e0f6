"""GPU parity of the chain's stages in shared launches.  The row-wise stages (hookless
chains that run to the final norm) against the same stages issued one by one
through the C ABI: the residual stream bit for bit without the blocks' output norms, and every
norm within one fp16 ulp of the separate kernel's (the two may sum the squares
of a row in another order).  A caller that reuses one scratch buffer for several
stages gets the sequential result."""
import numpy as np
import pytest

import mi_chain

pytestmark = pytest.mark.gpu
Stage = mi_chain.Stage


def _work(dev, D, double, seed=3, n_decode=5, **kw):
    return mi_chain.Workload(dev, seed=seed, n_decode=n_decode, prefills=(3,), logit_rows=2,
                             hidden_size=D, intermediate_size=64, num_heads=2, num_kv_heads=1,
                             head_dim=16, vocab=200, double_norm=int(double),
                             norm_add_one=int(double), embed_scale=int(double), **kw)


def _one_by_one(mk, w):
    """The stages as separate calls; returns the tensors by the chain's names."""
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


def _ulps(a, b):
    """Largest distance in fp16 values between a and b."""
    def order(x):
        i = x.cpu().numpy().view(np.int16).astype(np.int32)
        return np.where(i < 0, -32768 - i, i)
    return int(np.abs(order(a) - order(b)).max())


# one vector, the edges of the vectors per lane, the longest row, and rows the
# single launch does not take
@pytest.mark.parametrize("D", [8, 2040, 2048, 2056, 4104, 6152, 8192, 8200, 100])
@pytest.mark.parametrize("double", [False, True])
def test_rows_in_one_launch(mk, dev, D, double):
    import torch
    print(f"[case] chain rows D={D} double={double}", flush=True)
    w = _work(dev, D, double)
    w.t["ids"][2] = -1    # zero rows
    w.t["ids"][3] = 200
    want = _one_by_one(mk, w)
    w.run(Stage.FINAL_NORM)
    torch.cuda.synchronize()
    for n, ref in want.items():
        exact = not double and n in ("hidden", "attn_out", "mlp_out")
        # DOUBLE: a norm one ulp off moves the residual, and the norm of that
        far = 0 if exact else 1 if not double else 3
        got = w.t[n]
        if double and n == "hidden":  # cancelling sums: an absolute bound, an ulp of the addends
            assert (got.float() - ref.float()).abs().max() <= 2 ** -10 * 2 * max(
                w.t["attn_out"].abs().max().item(), w.t["mlp_out"].abs().max().item(), 1.0), n
        elif double and n in ("post_normed", "final_normed"):
            d = (got.float() - ref.float()).abs()
            assert (d <= 2 ** -9 * (ref.float().abs() + 1)).all(), n
        else:
            assert _ulps(got, ref) <= far, n


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
    t, c = w.t, w.cfg
    q, k, v = (t[n].clone() for n in "qkv")
    kc, vc = t["k_cache"].clone(), t["v_cache"].clone()
    inv = mk.rope_inv_freq(hd, c["rope_theta"])
    if kind == "norm":
        mk.qk_norm_rope(q, k, t["q_norm"], t["k_norm"], t["positions"], inv, eps=c["qk_norm_eps"])
    elif kind == "bias":
        mk.bias_rope_neox_qk(q, k, t["q_bias"], t["k_bias"], t["positions"], inv)
    else:
        mk.rope_neox_qk(q, k, t["positions"], inv)
    for g in w.segments:
        B, S, at = g["B"], g["S"], g["token_offset"]
        part = slice(at, at + B * S)
        mk.paged_kv_scatter(k[part].view(B, S, Hkv, hd), kc, g["block_table"], g["seq_len"],
                            g["start_pos"], 1, 16, v_src=v[part].view(B, S, Hkv, hd), v_cache=vc,
                            v_bias=t["v_bias"] if kind == "bias" else None)
    w.run(Stage.KV_SCATTER)
    torch.cuda.synchronize()
    assert torch.equal(t["q"], q) and torch.equal(t["k"], k) and torch.equal(t["v"], v)
    assert torch.equal(t["k_cache"], kc) and torch.equal(t["v_cache"], vc)


SMALL = dict(hidden_size=64, intermediate_size=72, num_heads=2, num_kv_heads=1, head_dim=64,
             vocab=9000, use_qk_norm=0)


# one token; the tiles' and vectors' edges; every rotation and head width; chunks of
# either size, ragged vocabularies, and more logit rows than one launch keeps resident
@pytest.mark.parametrize("n_decode,prefill,rows,kw", [
    (1, 0, 1, {}),
    (3, 0, 2, dict(vocab=8192, hidden_size=2048, intermediate_size=2048)),
    (5, 6, 3, dict(vocab=8201, hidden_size=2056, head_dim=128, qkv_bias=1)),
    (2, 40, 9, dict(vocab=16391, hidden_size=4096, num_heads=28, num_kv_heads=5, head_dim=128,
                    use_qk_norm=1)),
    (7, 33, 5, dict(head_dim=256, num_heads=8, num_kv_heads=4, use_qk_norm=1, double_norm=1,
                    norm_add_one=1, embed_scale=1, act=1)),
    (4, 0, 60, dict(vocab=152064, num_heads=4, qkv_bias=1)),
    (4, 0, 24, dict(vocab=262144, double_norm=1)),
    (4, 0, 500, dict(vocab=32001)),
    (4, 0, 3, dict(hidden_size=4104)),
    (4, 0, 3, dict(intermediate_size=7)),
    (4, 0, 3, dict(head_dim=80)),
])
@pytest.mark.parametrize("polls", [True, False])
def test_step_in_one_launch(mk, dev, n_decode, prefill, rows, kw, polls):
    """A whole step against the rows, rotation and activation as launches of their
    own and the sampling entry point: the same bits but for the probabilities,
    whose row sums may be taken in chunks of another size (one fp16 ulp)."""
    import torch
    print(f"[case] step T={n_decode + 2 * prefill} rows={rows} {kw} polls={polls}", flush=True)
    args = dict(seed=11, n_decode=n_decode, prefills=(prefill,) * 2 if prefill else (),
                logit_rows=rows, **dict(SMALL, **kw))
    ref, w = mi_chain.Workload(dev, **args), mi_chain.Workload(dev, **args)
    ref.run(Stage.FINAL_NORM)
    probs, tokens = mk.softmax_argmax(ref.t["logits"], ref.t["sample_ws"])
    names = [n for n in mi_chain._BUFS if n not in ("probs", "next_tokens")]
    prev = mk.softmax_test_poll_limit(1 << 16 if polls else 0)
    try:
        for i in range(2):  # the records serve the next call
            if i:
                w.reload("q", "k", "attn_out", "mlp_out")
            w.run()
            torch.cuda.synchronize()
            for n in names:
                assert torch.equal(w.t[n], ref.t[n]), n
            assert torch.equal(w.t["next_tokens"], tokens)
            assert _ulps(w.t["probs"], probs) <= 1
    finally:
        mk.softmax_test_poll_limit(prev)
