"""GPU parity of the sampling kernels over vocabularies that are no whole number
of 16-byte vectors (each row walked through its aligned window): softmax, greedy
argmax and the fused pass, in one launch, with the polling fallback forced, and
in the two-launch forms.

Probabilities: an output is RN16 of an fp32 value whose exponent argument
(|x - m| < 64) is off by at most 2^-18 and whose sum by less, so |y - ref| <=
2^-11 (1 + 2^-5) ref + 2^-25.  Indices are exact (the reference's tie order).
"""
import numpy as np
import pytest

from helpers import assert_bits_equal, normal_f16, to_dev, to_host

pytestmark = pytest.mark.gpu
GUARD = 64


def _buffer(dev, off, N, V):
    import torch
    b = torch.full((GUARD + off + N * V + GUARD,), 7.0, dtype=torch.float16, device=dev)
    return b, b[GUARD + off:GUARD + off + N * V].view(N, V)


def _guards_intact(b, off, N, V):
    h = to_host(b)
    return (h[:GUARD + off] == 7).all() and (h[GUARD + off + N * V:] == 7).all()


def _close(y, x):
    x = x.astype(np.float64)
    e = np.exp(x - x.max(-1, keepdims=True))
    ref = e / e.sum(-1, keepdims=True)
    assert (np.abs(y.astype(np.float64) - ref) <= 2.0 ** -11 * (1 + 2.0 ** -5) * ref + 2.0 ** -25).all()


# chunk edges (8192 and 4096 elements, up to 7 past them in the window), one
# row, rows in rounds (more than the grid holds), more rows than split at all
@pytest.mark.parametrize("N,V", [(1, 8193), (3, 8185), (9, 16378), (16, 16391), (48, 50257),
                                 (64, 151643), (200, 32001), (7, 262138), (600, 40001),
                                 (520, 8209)])
@pytest.mark.parametrize("off", [0, 5])
def test_ragged_vocab(mk, orc, dev, N, V, off):
    import torch
    print(f"[case] ragged vocabulary [{N},{V}] offset {off}", flush=True)
    rng = np.random.default_rng(N * 7 + V + off)
    x = normal_f16(rng, (N, V), 0, 4)
    x[::2] = np.rint(x[::2])  # ties at the maximum
    if N > 2:
        x[1, 5:] = -np.inf
        x[2, : V // 2] = 0.0
        x[2, V // 2:] = -0.0
    want = orc.greedy_argmax(x)
    xb, xd = _buffer(dev, off, N, V)
    xd.copy_(to_dev(x, dev))
    side = torch.cuda.Stream()

    def run(what, fn, probs=True, idx=True):
        yb, y = _buffer(dev, off, N, V)
        out = torch.full((N,), -7, dtype=torch.int32, device=dev)
        fn(y, out)
        torch.cuda.synchronize()
        if probs:
            _close(to_host(y), x)
            assert _guards_intact(yb, off, N, V), what
        if idx:
            np.testing.assert_array_equal(to_host(out), want, err_msg=what)

    ws = torch.zeros(max(16, mk.softmax_workspace_bytes(N, V)), dtype=torch.uint8, device=dev)
    aw = torch.zeros(max(16, mk.greedy_argmax_workspace_bytes(N, V)), dtype=torch.uint8, device=dev)
    fw = torch.zeros(mk.softmax_argmax_workspace_bytes(N, V), dtype=torch.uint8, device=dev)
    fused = lambda y, o: mk.softmax_argmax(xd, fw, probs=y, out=o)  # noqa: E731
    soft = lambda y, o: mk.softmax(xd, y=y, workspace=ws)  # noqa: E731
    amax = lambda y, o: mk.greedy_argmax(xd, out=o, workspace=aw)  # noqa: E731
    for _ in range(2):  # the records serve the next call
        run("fused", fused)
        run("softmax", soft, idx=False)
        run("argmax", amax, probs=False)
    prev = mk.softmax_test_poll_limit(0), mk.greedy_argmax_test_poll_limit(0)
    try:
        run("fused, no polls", fused)
        run("softmax, no polls", soft, idx=False)
        run("argmax, no polls", amax, probs=False)
    finally:
        mk.softmax_test_poll_limit(prev[0])
        mk.greedy_argmax_test_poll_limit(prev[1])
    run("fused, after", fused)

    def on_side(y, o):  # no records there: the two-launch forms
        side.wait_stream(torch.cuda.current_stream())
        mk.softmax(xd, y=y, stream=side)
        mk.greedy_argmax(xd, out=o, stream=side)

    run("two launches", on_side)
    assert_bits_equal(to_host(xd), x, what="logits")
    mk.softmax(xd, y=xd, workspace=ws)  # in place
    _close(to_host(xd), x)
    assert _guards_intact(xb, off, N, V)


# an odd number of softmax chunks (N * splits): the argmax's part of the workspace
# comes after them
@pytest.mark.parametrize("N,V", [(1, 8193), (5, 50257), (1, 151643), (7, 262138)])
@pytest.mark.parametrize("in_place", [True, False])
def test_softmax_and_argmax_apart(mk, orc, dev, N, V, in_place):
    """The fused entry point where its one-launch form does not apply: probs on the
    logits, or at another offset from a 16-byte boundary."""
    import torch
    print(f"[case] softmax + argmax apart [{N},{V}] in place={in_place}", flush=True)
    x = np.rint(normal_f16(np.random.default_rng(N + V), (N, V), 0, 4))
    xb, xd = _buffer(dev, 0, N, V)
    yb, y = (xb, xd) if in_place else _buffer(dev, 3, N, V)
    ws = torch.zeros(mk.softmax_argmax_workspace_bytes(N, V), dtype=torch.uint8, device=dev)
    for _ in range(2):
        xd.copy_(to_dev(x, dev))
        out = torch.full((N,), -7, dtype=torch.int32, device=dev)
        mk.softmax_argmax(xd, ws, probs=y, out=out)
        torch.cuda.synchronize()
        _close(to_host(y), x)
        np.testing.assert_array_equal(to_host(out), orc.greedy_argmax(x))
        assert _guards_intact(yb, 0 if in_place else 3, N, V)


# rows in registers, in one launch in one round and in rounds, as many short rows
@pytest.mark.parametrize("N,V", [(64, 1203), (12, 8193), (9, 16391), (48, 50257), (600, 40001)])
@pytest.mark.parametrize("off", [0, 5])
def test_ragged_special_values(mk, orc, dev, N, V, off):
    """NaN and infinities at the ends of a row share 16-byte granules with its
    neighbours' elements; inside it they reach the element-by-element tie search."""
    import torch
    print(f"[case] ragged special values [{N},{V}] offset {off}", flush=True)
    x = normal_f16(np.random.default_rng(N + V + off), (N, V), 0, 4)
    bits = x.view(np.uint16)
    x[1, 0], x[1, -1] = np.inf, np.nan
    x[3, V // 2] = np.nan                       # never chosen
    x[4, [7, V // 3, V - 1]] = np.inf           # ties, in the reference's order
    bits[6, :] = 0x7e00                         # only NaN: -1
    bits[7, :] = 0x7e00
    x[7, V - 2] = -65504.0                      # the one finite value
    bits[8, ::2] = 0x7d01                       # signalling NaNs
    want = orc.greedy_argmax(x)
    assert want[1] == 0 and want[6] == -1 and want[7] == V - 2
    plain = [r for r in range(N) if r not in (1, 3, 4, 6, 7, 8)]
    xb, xd = _buffer(dev, off, N, V)
    xd.copy_(to_dev(x, dev))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    ws = torch.zeros(max(16, mk.softmax_workspace_bytes(N, V)), dtype=torch.uint8, device=dev)
    aw = torch.zeros(max(16, mk.greedy_argmax_workspace_bytes(N, V)), dtype=torch.uint8, device=dev)
    fw = torch.zeros(mk.softmax_argmax_workspace_bytes(N, V), dtype=torch.uint8, device=dev)

    def check(what, fn):
        yb, y = _buffer(dev, off, N, V)
        out = torch.full((N,), -7, dtype=torch.int32, device=dev)
        fn(y, out)
        torch.cuda.synchronize()
        h = to_host(y)
        _close(h[plain], x[plain])
        assert np.isnan(h[[1, 3, 4]]).all(), what  # the sum is NaN
        assert _guards_intact(yb, off, N, V), what
        np.testing.assert_array_equal(to_host(out), want, err_msg=what)

    def apart(y, o):
        mk.softmax(xd, y=y, workspace=ws)
        mk.greedy_argmax(xd, out=o, workspace=aw)

    def on_side(y, o):
        mk.softmax(xd, y=y, stream=side)
        mk.greedy_argmax(xd, out=o, stream=side)

    check("fused", lambda y, o: mk.softmax_argmax(xd, fw, probs=y, out=o))
    check("apart", apart)
    check("two launches", on_side)
    prev = mk.softmax_test_poll_limit(0), mk.greedy_argmax_test_poll_limit(0)
    try:
        check("fused, no polls", lambda y, o: mk.softmax_argmax(xd, fw, probs=y, out=o))
        check("apart, no polls", apart)
    finally:
        mk.softmax_test_poll_limit(prev[0])
        mk.greedy_argmax_test_poll_limit(prev[1])
