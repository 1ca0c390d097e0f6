"""The wrappers' native calls (host/python/fast_calls.cpp): what they take gives the
wrapper's result, and what they leave -- wrong types, shapes, devices, layouts,
tensor subclasses, sequences for the inverse frequencies -- is checked, converted
and refused by the wrapper as before."""
import importlib.util
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

import numpy as np
import pytest

from helpers import assert_bits_equal, normal_f16, to_dev, to_host

PKG = Path(__file__).resolve().parent.parent / "mini-infer_amd"


def _child(code, *args):
    """Runs code in a process of its own (a native fault ends only that); its output."""
    r = subprocess.run([sys.executable, "-c", code, *map(str, args)], capture_output=True, text=True,
                       timeout=110)
    assert r.returncode == 0, f"exit status {r.returncode}\n{r.stdout}\n{r.stderr[-2000:]}"
    return r.stdout


VMAP = """
import sys
sys.path.insert(0, sys.argv[1])
import numpy as np
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
import mi_kernels as mk


class Stream:
    cuda_stream = 0


s, n = Stream(), 0


def refused(call, *args):
    def body(*a):
        t = next(x for x in a if x is not None)
        assert type(t) is torch.Tensor and t.is_cuda and t.is_contiguous()
        return call(*a)
    try:
        torch.vmap(body)(*args)
    except RuntimeError as e:
        assert "data pointer" in str(e), e
        global n
        n += 1
    else:
        raise AssertionError("not refused")


def h(*shape, dtype=torch.float16):
    return torch.empty((3, *shape), dtype=dtype, device="cuda")


with FakeTensorMode():
    x, w, q, k = h(4, 8), h(8), h(4, 2, 16), h(4, 1, 16)
    hd, b, i32 = h(16), h(1024, dtype=torch.uint8), h(4, dtype=torch.int32)
    pos, inv = h(4, dtype=torch.int64), np.ones(8, np.float32)
    refused(lambda x, w, y: mk.rmsnorm(x, w, y=y, stream=s), x, w, x)
    refused(lambda x, w: mk.rmsnorm(x, w, stream=s), x, w)
    refused(lambda x, r, w: mk.fused_add_rmsnorm(x, r, w, stream=s), x, x, w)
    refused(lambda x, y: mk.swiglu(x, y, stream=s), x, x)
    refused(lambda x, y: mk.geglu(x, y, stream=s), x, x)
    refused(lambda x: mk.softmax(x, stream=s), x)
    refused(lambda x, b: mk.softmax(x, workspace=b, stream=s), x, b)
    refused(lambda x, b, o: mk.softmax_argmax(x, b, out=o, stream=s), x, b, i32)
    refused(lambda x, o: mk.greedy_argmax(x, out=o, stream=s), x, i32)
    refused(lambda x, o, b: mk.greedy_argmax(x, out=o, workspace=b, stream=s), x, i32, b)
    refused(lambda x, o: mk.top_p_sample(x, 0.9, 1.0, 7, out=o, stream=s), x, i32)
    refused(lambda q, k, p: mk.rope_neox_qk(q, k, p, inv, stream=s), q, k, pos)
    refused(lambda q, k, b, c, p: mk.bias_rope_neox_qk(q, k, b, c, p, inv, stream=s), q, k, h(32), hd,
            pos)
    refused(lambda q, k, w, p: mk.qk_norm_rope(q, k, w, w, p, inv, stream=s), q, k, hd, pos)
    refused(lambda x, c: mk.rope_neox(x, c, c, stream=s), h(1, 4, 2, 16), h(4, 8))
    refused(lambda p, c, d: mk.rope_tables(inv, p, c, d, stream=s), pos, h(4, 8), h(4, 8))
    refused(lambda i, t: mk.embedding_gather(i, t, stream=s), pos, h(50, 8))
    refused(lambda i, t, w: mk.embedding_rmsnorm(i, t, w, stream=s), pos, h(50, 8), w)
print("refused", n)
"""


def test_tensors_without_memory_are_refused():
    """torch.vmap hands in tensors of exact type and layout whose data_ptr() throws."""
    pytest.importorskip("torch")
    assert "refused 18" in _child(VMAP, PKG)


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


ONCE = """
import ctypes
import sys
sys.path.insert(0, sys.argv[1])
import numpy as np
import torch
import mi_kernels as mk

mk._need = lambda *a: None  # the wrapper too would take these tensors
stub = ctypes.CDLL(sys.argv[1] + "/libmi_kernels.so")
calls = ctypes.c_int.in_dll(stub, "calls")
status = ctypes.c_int.in_dll(stub, "status")


class Stream:
    cuda_stream = 0


s = Stream()


def h(*shape, dtype=torch.float16):
    return torch.zeros(shape, dtype=dtype)


x, w, q, k, hd, ws = h(4, 8), h(8), h(4, 2, 16), h(4, 1, 16), h(16), h(64, dtype=torch.uint8)
pos, inv = h(4, dtype=torch.int64), np.ones(8, np.float32)
each = {
    "mi_rmsnorm_f16": lambda: mk.rmsnorm(x, w, stream=s),
    "mi_fused_add_rmsnorm_f16": lambda: mk.fused_add_rmsnorm(x, x, w, stream=s),
    "mi_swiglu_f16": lambda: mk.swiglu(x, x, stream=s),
    "mi_geglu_f16": lambda: mk.geglu(x, x, stream=s),
    "mi_softmax_f16": lambda: mk.softmax(x, stream=s),
    "mi_softmax_ws_f16": lambda: mk.softmax(x, workspace=ws, stream=s),
    "mi_softmax_argmax_ws_f16": lambda: mk.softmax_argmax(x, ws, stream=s),
    "mi_greedy_argmax_f16": lambda: mk.greedy_argmax(x, stream=s),
    "mi_greedy_argmax_ws_f16": lambda: mk.greedy_argmax(x, workspace=ws, stream=s),
    "mi_top_p_sample_batched_f16": lambda: mk.top_p_sample(x, 0.9, 1.0, 7, stream=s),
    "mi_rope_neox_qk_f16": lambda: mk.rope_neox_qk(q, k, pos, inv, stream=s),
    "mi_bias_rope_neox_qk_f16": lambda: mk.bias_rope_neox_qk(q, k, h(32), hd, pos, inv, stream=s),
    "mi_qk_norm_rope_f16": lambda: mk.qk_norm_rope(q, k, hd, hd, pos, inv, stream=s),
    "mi_rope_neox_f16": lambda: mk.rope_neox(h(1, 4, 2, 16), h(4, 8), h(4, 8), stream=s),
    "mi_rope_tables_f16": lambda: mk.rope_tables(inv, pos, stream=s),
    "mi_embedding_gather_f16": lambda: mk.embedding_gather(pos, x, stream=s),
    "mi_embedding_rmsnorm_f16": lambda: mk.embedding_rmsnorm(pos, x, w, stream=s),
}
if sys.argv[2] != "built":
    del each["mi_softmax_ws_f16"]  # its wrapper has a check of the workspace's device
for name, call in each.items():
    calls.value = status.value = 0
    assert call() is not None and calls.value == 1, name
    for st in (100, -1, -2):  # a HIP error, refusals
        calls.value, status.value = 0, st
        try:
            call()
        except RuntimeError as e:
            assert str(e) == f"{name} failed: status {st} (why)", e
        else:
            raise AssertionError(name + ": status lost")
        assert calls.value == 1, (name, st, calls.value)
print("once", len(each))
"""


@pytest.mark.parametrize("native", ["built", "missing", "unloadable"])
def test_a_failed_call_is_made_once(tmp_path, native):
    """The binding over a library whose calls only count themselves and return a
    status: whatever it is, there is one call, and the status is raised.  The native
    part is built to take CPU tensors for it; without one that loads, the wrappers
    make the calls."""
    pytest.importorskip("torch")
    import mi_kernels as mk
    names = [*mk.SIGNATURES, "mi_greedy_argmax_workspace_bytes", "mi_softmax_workspace_bytes",
             "mi_softmax_argmax_workspace_bytes", "mi_decoder_chain_run"]
    stub = tmp_path / "stub.c"
    stub.write_text("int calls, status;\nconst char* mi_status_string(int s) { return \"why\"; }\n" +
                    "".join(f"int {n}() {{ ++calls; return status; }}\n" for n in names))
    lib = tmp_path / "libmi_kernels.so"
    subprocess.run(["gcc", "-shared", "-fPIC", str(stub), "-o", str(lib)], check=True)
    shutil.copy(PKG / "mi_kernels.py", tmp_path)
    if native == "unloadable":
        (tmp_path / "_mi_fast.so").write_bytes(b"")
    if native != "built":
        assert "once 16" in _child(ONCE, tmp_path, native)
        return
    src = (PKG / "host/python/fast_calls.cpp").read_text()
    assert src.count("t.is_cuda()") == 2
    cpu = tmp_path / "fast_calls_cpu.cpp"
    cpu.write_text(src.replace("t.is_cuda()", "t.is_cpu()"))
    at = Path(importlib.util.find_spec("torch").submodule_search_locations[0])
    subprocess.run(["g++", "-O0", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1",
                    "-DUSE_ROCM=1", f"-I{PKG.parent / 'include'}", f"-I{sysconfig.get_paths()['include']}",
                    "-isystem", str(at / "include"), "-isystem", "/opt/rocm/include", "-o",
                    str(tmp_path / "_mi_fast.so"), str(cpu), str(lib), f"-L{at / 'lib'}", "-ltorch_python",
                    "-ltorch_cpu", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"], check=True)
    assert "once 17" in _child(ONCE, tmp_path, native)


def test_all_is_built_without_torch():
    for without in ("TORCH=", "PYINC="):
        out = subprocess.run(["make", "-n", "-B", "-C", str(PKG), "all", without], check=True,
                             capture_output=True, text=True).stdout
        assert "libmini_infer.so" in out and "_mi_fast.so" not in out


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
