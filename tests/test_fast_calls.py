"""The wrappers' native calls (host/python/fast_calls.cpp): what they take gives the
wrapper's result, and what they leave -- wrong types, shapes, devices, layouts,
tensor subclasses, sequences for the inverse frequencies -- is checked, converted
and refused by the wrapper as before."""
import numpy as np
import pytest

from helpers import assert_bits_equal, normal_f16, to_dev, to_host


def test_cpu_tensors_are_refused(monkeypatch):
    torch = pytest.importorskip("torch")
    import mi_kernels as mk
    x = torch.zeros(4, 8, dtype=torch.float16)
    w = torch.zeros(8, dtype=torch.float16)
    for call in (lambda: mk.rmsnorm(x, w, y=x), lambda: mk.swiglu(x, x), lambda: mk.softmax(x),
                 lambda: mk.greedy_argmax(x), lambda: mk.fused_add_rmsnorm(x, x, w)):
        with pytest.raises(ValueError, match="GPU"):
            call()
    with pytest.raises(TypeError):
        mk.softmax(np.zeros((4, 8), np.float16))


@pytest.mark.gpu
def test_taken_and_left(mk, orc, dev):
    import torch
    print("[case] native calls, taken and left", flush=True)
    rng = np.random.default_rng(9)
    x, w = normal_f16(rng, (6, 64)), normal_f16(rng, (64,), 1.0, 0.1)
    xd, wd = to_dev(x, dev), to_dev(w, dev)
    want = to_host(mk.rmsnorm(xd, wd))
    y = torch.empty_like(xd)
    assert mk.rmsnorm(xd, wd, y=y, eps=1e-6) is y
    assert_bits_equal(to_host(y), want, what="y given")
    assert_bits_equal(to_host(mk.rmsnorm(torch.nn.Parameter(xd, requires_grad=False), wd,
                                         eps=np.float32(1e-6))), want, what="a Parameter, numpy eps")

    class Own(torch.Tensor):
        pass

    assert_bits_equal(to_host(mk.rmsnorm(xd.as_subclass(Own), wd).as_subclass(torch.Tensor)), want,
                      what="a subclass")
    for call, err in ((lambda: mk.rmsnorm(xd.t(), wd), ValueError),
                      (lambda: mk.rmsnorm(xd.float(), wd), TypeError),
                      (lambda: mk.rmsnorm(xd, wd[:8]), ValueError),
                      (lambda: mk.rmsnorm(xd, wd, y=y[:3]), ValueError),
                      (lambda: mk.rmsnorm(xd, wd.cpu()), ValueError),
                      (lambda: mk.swiglu(xd, xd[:2]), ValueError),
                      (lambda: mk.greedy_argmax(xd, out=y), TypeError),
                      (lambda: mk.softmax(xd, y=xd.view(-1)[1:65].view(1, 64)), ValueError),
                      (lambda: mk.fused_add_rmsnorm(xd, xd, wd), RuntimeError)):  # aliasing
        with pytest.raises(err):
            call()
    # the current stream, and a given one
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        a = mk.rmsnorm(xd, wd)
        assert (mk._fast or mk._load_fast()).current_stream() == side.cuda_stream
    b = mk.rmsnorm(xd, wd, stream=side)
    side.synchronize()
    assert_bits_equal(to_host(a), want, what="current stream")
    assert_bits_equal(to_host(b), want, what="given stream")
    # inverse frequencies: float32, or anything numpy makes float32 of
    q = normal_f16(rng, (5, 3, 16))
    inv = mk.rope_inv_freq(16)
    pos = torch.arange(5, device=dev)
    outs = []
    for f in (inv, inv.astype(np.float64), list(map(float, inv)), np.repeat(inv, 2)[::2]):
        qd = to_dev(q, dev)
        r = mk.rope_neox_qk(qd, None, pos, f)
        assert r[0] is qd and r[1] is None
        outs.append(to_host(qd))
    for o in outs[1:]:
        assert_bits_equal(o, outs[0], what="inverse frequencies")
    # outputs that the call makes
    table = to_dev(normal_f16(rng, (50, 64)), dev)
    ids = torch.arange(6, device=dev).view(2, 3)
    h, n = mk.embedding_rmsnorm(ids, table, wd)
    assert h.shape == n.shape == (2, 3, 64) and torch.equal(h, table[ids])
    assert torch.equal(mk.embedding_gather(ids, table), table[ids])
    assert torch.equal(n.view(6, 64), mk.rmsnorm(h.view(6, 64), wd))
    np.testing.assert_array_equal(to_host(mk.greedy_argmax(xd[0])), orc.greedy_argmax(x[:1]))
    np.testing.assert_array_equal(to_host(mk.greedy_argmax(xd)), orc.greedy_argmax(x))
