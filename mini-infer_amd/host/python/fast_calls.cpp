// fast_calls.cpp -- the Python binding's calls made natively: the checks of
// mi_kernels.py's wrappers on the tensors themselves, torch's current stream, and
// the C ABI call, without a ctypes object per argument.
//
// A small call is bound by the host.  Of the 9.8 us that mi_kernels.rmsnorm took
// for [16, 3584] through ctypes, the launch is 3; torch.cuda.current_stream()
// took 2.8, the attribute checks and pointer objects of three tensors most of
// the rest.  Here: 4.1; swiglu 9.3 -> 3.4, rope_neox_qk 11.7 -> 4.7 us.
//
// Every function returns the wrapper's result when the call was launched (an
// output that is None is allocated, as the wrapper does), and otherwise None,
// having launched nothing: an argument is not what the call needs (a tensor on
// another device, of another type or shape, not contiguous, a subclass with its
// own ways, one without memory of its own, as under torch.vmap).  The Python
// wrapper then makes the call itself and raises what there is to raise, so its
// errors and conversions stay where they were.  A library call that was made is
// never made again: its status, if not 0, is raised here.  (A status does not say
// that nothing ran: an error that an earlier HIP call left behind is reported by
// the next launch, and a second call would add a residual or rotate twice.)
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "mi_chain.h"
#include "mi_kernels.h"

namespace {

// Thrown where a call is left to the Python wrapper.
struct Leave {};

// Thrown where the library call was made and gave a status other than 0.
struct Failed {
    const char* what;
    int status;
};

void need(bool ok) {
    if (!ok) throw Leave{};
}

const at::Tensor& tensor(PyObject* o, at::ScalarType type) {
    need(THPVariable_CheckExact(o));
    const at::Tensor& t = THPVariable_Unpack(o);
    need(t.is_cuda() && t.scalar_type() == type && t.is_contiguous());
    return t;
}
const at::Tensor& half(PyObject* o) { return tensor(o, at::kHalf); }

void* ptr(const at::Tensor& t) { return t.data_ptr(); }

void* stream_of(PyObject* o) {
    if (o == Py_None) return c10::hip::getCurrentHIPStream().stream();
    PyObject* v = PyObject_GetAttrString(o, "cuda_stream");
    if (!v) {
        PyErr_Clear();
        throw Leave{};
    }
    void* s = PyLong_Check(v) ? PyLong_AsVoidPtr(v) : nullptr;
    const bool ok = PyLong_Check(v) && !PyErr_Occurred();
    Py_DECREF(v);
    if (!ok) {
        PyErr_Clear();
        throw Leave{};
    }
    return s;
}

double number(PyObject* o) {
    need(PyFloat_CheckExact(o) || PyLong_CheckExact(o));
    const double v = PyFloat_AsDouble(o);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        throw Leave{};
    }
    return v;
}
int64_t whole(PyObject* o) {
    need(PyLong_CheckExact(o));
    const int64_t v = PyLong_AsLongLong(o);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        throw Leave{};
    }
    return v;
}
int truth(PyObject* o) {
    need(PyBool_Check(o) || PyLong_CheckExact(o));
    return PyObject_IsTrue(o);
}

// The host's fp32 inverse frequencies, in a contiguous float32 buffer.
struct Floats {
    Py_buffer view{};
    explicit Floats(PyObject* o) {
        if (!PyObject_CheckBuffer(o)) throw Leave{};
        if (PyObject_GetBuffer(o, &view, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) != 0) {
            PyErr_Clear();
            throw Leave{};
        }
        if (view.itemsize != 4 || !view.format || view.format[0] != 'f' || view.format[1]) {
            PyBuffer_Release(&view);
            throw Leave{};
        }
    }
    ~Floats() { PyBuffer_Release(&view); }
    Floats(const Floats&) = delete;
    int64_t size() const { return view.len / 4; }
    const float* data() const { return static_cast<const float*>(view.buf); }
};

// Without the GIL for its lifetime, also where that ends in an exception.
struct NoGil {
    PyThreadState* thread = PyEval_SaveThread();
    NoGil() = default;
    NoGil(const NoGil&) = delete;
    ~NoGil() { PyEval_RestoreThread(thread); }
};

// The library call f(args...) without the GIL (it may wait for room in the
// stream's queue).  The arguments are values, so that what makes them runs with
// the GIL held: ptr() throws for a tensor without memory of its own, and the
// handlers below are Python calls.
template <typename F, typename... A>
void launch(const char* what, F f, A... args) {
    int st;
    {
        const NoGil released;
        st = f(args...);
    }
    if (st != 0) throw Failed{what, st};
}
#define MI_CALL(f, ...) launch(#f, f, __VA_ARGS__)

// An output: the caller's tensor, or where it is None a new one of x's shape or
// of `sizes`.
struct Out {
    at::Tensor made;
    const at::Tensor* t;
    PyObject* given;
    Out(PyObject* o, const at::Tensor& x) : given(o == Py_None ? nullptr : o) {
        if (!given) made = at::empty_like(x);
        t = given ? &half(o) : &made;
    }
    Out(PyObject* o, const at::Tensor& on, at::ScalarType type, at::IntArrayRef sizes)
        : given(o == Py_None ? nullptr : o) {
        if (!given) made = at::empty(sizes, on.options().dtype(type));
        t = given ? &tensor(o, type) : &made;
    }
    PyObject* result() const {  // a new reference
        if (!given) return THPVariable_Wrap(made);
        Py_INCREF(given);
        return given;
    }
};
PyObject* pair(PyObject* a, PyObject* b) {
    PyObject* r = a && b ? PyTuple_Pack(2, a, b) : nullptr;
    Py_XDECREF(a);
    Py_XDECREF(b);
    return r;
}

// Runs body() for exactly n arguments: its result, None where it is left, or the
// error of a library call that failed.
template <typename F>
PyObject* guarded(Py_ssize_t got, Py_ssize_t n, F body) {
    if (got != n) {
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
        return nullptr;
    }
    try {
        return body();
    } catch (const Leave&) {
        Py_RETURN_NONE;
    } catch (const Failed& e) {  // the wrapper's message
        PyErr_Format(PyExc_RuntimeError, "%s failed: status %d (%s)", e.what, e.status,
                     mi_status_string(e.status));
        return nullptr;
    } catch (const std::exception&) {  // torch: a tensor without memory of its own
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

#define MI_FAST(name) PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n)

// (x, weight, y, eps, add_one, stream)
MI_FAST(rmsnorm) {
    return guarded(n, 6, [&] {
        const auto &x = half(a[0]), &w = half(a[1]);
        need(x.dim() == 2 && w.numel() == x.size(1));
        const Out out(a[2], x);
        const at::Tensor& y = *out.t;
        need(y.sizes() == x.sizes());
        const float eps = static_cast<float>(number(a[3]));
        const int one = truth(a[4]);
        void* s = stream_of(a[5]);
        MI_CALL(mi_rmsnorm_f16, ptr(x), ptr(w), ptr(y), x.size(0), x.size(1), eps, one, s);
        return out.result();
    });
}

// (x, residual, weight, y, eps, add_one, stream)
MI_FAST(fused_add_rmsnorm) {
    return guarded(n, 7, [&] {
        const auto &x = half(a[0]), &r = half(a[1]), &w = half(a[2]);
        need(x.dim() == 2 && r.sizes() == x.sizes() && w.numel() == x.size(1));
        const Out out(a[3], x);
        const at::Tensor& y = *out.t;
        need(y.sizes() == x.sizes());
        const float eps = static_cast<float>(number(a[4]));
        const int one = truth(a[5]);
        void* s = stream_of(a[6]);
        MI_CALL(mi_fused_add_rmsnorm_f16, ptr(x), ptr(r), ptr(w), ptr(y), x.size(0), x.size(1), eps,
                one, s);
        return out.result();
    });
}

// (a, b, out, stream)
template <typename F>
PyObject* binary(PyObject* const* a, Py_ssize_t n, const char* what, F f) {
    return guarded(n, 4, [&] {
        const auto &x = half(a[0]), &y = half(a[1]);
        need(y.numel() == x.numel());
        const Out out(a[2], x);
        need(out.t->numel() == x.numel());
        void* s = stream_of(a[3]);
        launch(what, f, ptr(x), ptr(y), ptr(*out.t), x.numel(), s);
        return out.result();
    });
}
MI_FAST(swiglu) { return binary(a, n, "mi_swiglu_f16", mi_swiglu_f16); }
MI_FAST(geglu) { return binary(a, n, "mi_geglu_f16", mi_geglu_f16); }

const at::Tensor& bytes_on_gpu(PyObject* o) {  // a workspace of any type
    need(THPVariable_CheckExact(o));
    const at::Tensor& t = THPVariable_Unpack(o);
    need(t.is_cuda() && t.is_contiguous());
    return t;
}

// (x, y, workspace or None, stream)
MI_FAST(softmax) {
    return guarded(n, 4, [&] {
        const auto& x = half(a[0]);
        need(x.dim() == 2);
        const Out out(a[1], x);
        const at::Tensor& y = *out.t;
        need(y.sizes() == x.sizes());
        void* s = stream_of(a[3]);
        if (a[2] == Py_None) {
            MI_CALL(mi_softmax_f16, ptr(x), ptr(y), x.size(0), x.size(1), s);
        } else {
            const auto& w = bytes_on_gpu(a[2]);
            MI_CALL(mi_softmax_ws_f16, ptr(x), ptr(y), x.size(0), x.size(1), ptr(w),
                    static_cast<int64_t>(w.nbytes()), s);
        }
        return out.result();
    });
}

// (logits, workspace, probs, out, stream)
MI_FAST(softmax_argmax) {
    return guarded(n, 5, [&] {
        const auto& x = half(a[0]);
        const auto& w = bytes_on_gpu(a[1]);
        need(x.dim() == 2);
        const Out probs(a[2], x), next(a[3], x, at::kInt, {x.size(0)});
        const at::Tensor &y = *probs.t, &o = *next.t;
        need(y.sizes() == x.sizes() && o.numel() == x.size(0));
        void* s = stream_of(a[4]);
        MI_CALL(mi_softmax_argmax_ws_f16, ptr(x), ptr(y), static_cast<int32_t*>(ptr(o)), x.size(0),
                x.size(1), ptr(w), static_cast<int64_t>(w.nbytes()), s);
        return pair(probs.result(), next.result());
    });
}

// (logits [B, V], out, workspace or None, stream)
MI_FAST(greedy_argmax) {
    return guarded(n, 4, [&] {
        const auto& x = half(a[0]);
        need(x.dim() == 2);
        const Out next(a[1], x, at::kInt, {x.size(0)});
        need(next.t->numel() == x.size(0));
        auto* out = static_cast<int32_t*>(ptr(*next.t));
        void* s = stream_of(a[3]);
        if (a[2] == Py_None) {
            MI_CALL(mi_greedy_argmax_f16, ptr(x), x.size(0), x.size(1), out, s);
        } else {
            const auto& w = bytes_on_gpu(a[2]);
            MI_CALL(mi_greedy_argmax_ws_f16, ptr(x), x.size(0), x.size(1), out, ptr(w),
                    static_cast<int64_t>(w.nbytes()), s);
        }
        return next.result();
    });
}

// (logits [B, V], p, temperature, seed, out, stream)
MI_FAST(top_p_sample) {
    return guarded(n, 6, [&] {
        const auto& x = half(a[0]);
        need(x.dim() == 2);
        const Out next(a[4], x, at::kInt, {x.size(0)});
        need(next.t->numel() == x.size(0));
        const float p = static_cast<float>(number(a[1])), temp = static_cast<float>(number(a[2]));
        const int64_t seed = whole(a[3]);
        void* s = stream_of(a[5]);
        MI_CALL(mi_top_p_sample_batched_f16, ptr(x), x.size(0), x.size(1), p, temp,
                static_cast<uint64_t>(seed), static_cast<int32_t*>(ptr(*next.t)), s);
        return next.result();
    });
}

// q [T, Hq, hd], k [T, Hkv, hd] or None, positions [T], inv_freq [hd / 2]
struct QkRope {
    const at::Tensor& q;
    const at::Tensor* k;
    const at::Tensor& pos;
    int64_t T, Hq, Hkv, hd;
    QkRope(PyObject* q_, PyObject* k_, PyObject* pos_)
        : q(half(q_)), k(k_ == Py_None ? nullptr : &half(k_)), pos(tensor(pos_, at::kLong)) {
        need(q.dim() == 3);
        T = q.size(0);
        Hq = q.size(1);
        hd = q.size(2);
        need(!k || (k->dim() == 3 && k->size(0) == T && k->size(2) == hd));
        Hkv = k ? k->size(1) : 0;
        need(pos.numel() == T);
    }
    void* kp() const { return k ? ptr(*k) : nullptr; }
    const int64_t* pp() const { return static_cast<const int64_t*>(ptr(pos)); }
};

// (q, k or None, positions, inv_freq, stream)
MI_FAST(rope_neox_qk) {
    return guarded(n, 5, [&] {
        const QkRope r(a[0], a[1], a[2]);
        const Floats inv(a[3]);
        need(inv.size() == r.hd / 2);
        void* s = stream_of(a[4]);
        MI_CALL(mi_rope_neox_qk_f16, ptr(r.q), r.kp(), r.pp(), inv.data(), r.T, r.Hq, r.Hkv, r.hd, s);
        return PyTuple_Pack(2, a[0], a[1]);
    });
}

// (q, k or None, q_bias, k_bias, positions, inv_freq, stream)
MI_FAST(bias_rope_neox_qk) {
    return guarded(n, 7, [&] {
        const QkRope r(a[0], a[1], a[4]);
        const auto& bq = half(a[2]);
        const at::Tensor* bk = r.k ? &half(a[3]) : nullptr;
        need(bq.numel() == r.Hq * r.hd && (!bk || bk->numel() == r.Hkv * r.hd));
        const Floats inv(a[5]);
        need(inv.size() == r.hd / 2);
        void* s = stream_of(a[6]);
        MI_CALL(mi_bias_rope_neox_qk_f16, ptr(r.q), r.kp(), ptr(bq), bk ? ptr(*bk) : nullptr, r.pp(),
                inv.data(), r.T, r.Hq, r.Hkv, r.hd, s);
        return PyTuple_Pack(2, a[0], a[1]);
    });
}

// (q, k or None, q_weight, k_weight, positions, inv_freq, eps, add_one, stream)
MI_FAST(qk_norm_rope) {
    return guarded(n, 9, [&] {
        const QkRope r(a[0], a[1], a[4]);
        const auto& wq = half(a[2]);
        const at::Tensor* wk = r.k ? &half(a[3]) : nullptr;
        need(wq.numel() == r.hd && (!wk || wk->numel() == r.hd));
        const Floats inv(a[5]);
        need(inv.size() == r.hd / 2);
        const float eps = static_cast<float>(number(a[6]));
        const int one = truth(a[7]);
        void* s = stream_of(a[8]);
        MI_CALL(mi_qk_norm_rope_f16, ptr(r.q), r.kp(), ptr(wq), wk ? ptr(*wk) : nullptr, r.pp(),
                inv.data(), r.T, r.Hq, r.Hkv, r.hd, eps, one, s);
        return PyTuple_Pack(2, a[0], a[1]);
    });
}

// (x [B, S, H, D], cos_t, sin_t, y, stream)
MI_FAST(rope_neox) {
    return guarded(n, 5, [&] {
        const auto &x = half(a[0]), &c = half(a[1]), &sn = half(a[2]);
        need(x.dim() == 4);
        const Out out(a[3], x);
        const at::Tensor& y = *out.t;
        need(y.sizes() == x.sizes());
        const int64_t B = x.size(0), S = x.size(1), H = x.size(2), D = x.size(3);
        need(c.numel() == B * S * (D / 2) && sn.numel() == B * S * (D / 2));
        void* s = stream_of(a[4]);
        MI_CALL(mi_rope_neox_f16, ptr(x), ptr(c), ptr(sn), ptr(y), B, S, H, D, s);
        return out.result();
    });
}

// (inv_freq, positions, cos_t, sin_t, stream)
MI_FAST(rope_tables) {
    return guarded(n, 5, [&] {
        const Floats inv(a[0]);
        const auto& pos = tensor(a[1], at::kLong);
        const int64_t N = pos.numel(), hf = inv.size();
        const Out oc(a[2], pos, at::kHalf, {N, hf}), os(a[3], pos, at::kHalf, {N, hf});
        const at::Tensor &c = *oc.t, &sn = *os.t;
        need(c.numel() == N * hf && sn.numel() == N * hf);
        void* s = stream_of(a[4]);
        MI_CALL(mi_rope_tables_f16, inv.data(), static_cast<const int64_t*>(ptr(pos)), ptr(c),
                ptr(sn), N, hf, s);
        return pair(oc.result(), os.result());
    });
}

// ids' shape with one more dimension of `width`
std::vector<int64_t> rows_of(const at::Tensor& ids, int64_t width) {
    std::vector<int64_t> v(ids.sizes().begin(), ids.sizes().end());
    v.push_back(width);
    return v;
}

// (ids, table, out, check_range, stream)
MI_FAST(embedding_gather) {
    return guarded(n, 5, [&] {
        const auto& ids = tensor(a[0], at::kLong);
        const auto& tb = half(a[1]);
        need(tb.dim() == 2);
        const int64_t V = tb.size(0), H = tb.size(1), T = ids.numel();
        const Out out(a[2], tb, at::kHalf, rows_of(ids, H));
        const at::Tensor& o = *out.t;
        need(o.numel() == T * H);
        const int check = truth(a[3]);
        void* s = stream_of(a[4]);
        MI_CALL(mi_embedding_gather_f16, static_cast<const int64_t*>(ptr(ids)), ptr(tb), ptr(o), T,
                H, check ? V : 0, s);
        return out.result();
    });
}

// (ids, table, weight, hidden, y, scale, eps, add_one, check_range, stream)
MI_FAST(embedding_rmsnorm) {
    return guarded(n, 10, [&] {
        const auto& ids = tensor(a[0], at::kLong);
        const auto &tb = half(a[1]), &w = half(a[2]);
        need(tb.dim() == 2);
        const int64_t V = tb.size(0), D = tb.size(1), T = ids.numel();
        const auto sizes = rows_of(ids, D);
        const Out oh(a[3], tb, at::kHalf, sizes), oy(a[4], tb, at::kHalf, sizes);
        const at::Tensor &h = *oh.t, &y = *oy.t;
        need(w.numel() == D && h.numel() == T * D && y.numel() == T * D);
        const float scale = static_cast<float>(number(a[5])), eps = static_cast<float>(number(a[6]));
        const int one = truth(a[7]), check = truth(a[8]);
        void* s = stream_of(a[9]);
        MI_CALL(mi_embedding_rmsnorm_f16, static_cast<const int64_t*>(ptr(ids)), ptr(tb), ptr(h),
                ptr(w), ptr(y), T, D, check ? V : 0, scale, eps, one, s);
        return pair(oh.result(), oy.result());
    });
}

// (address of an mi_chain_desc, last_stage, stream): the call's status.
MI_FAST(chain_run) {
    if (n != 3) {
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
        return nullptr;
    }
    int st;
    try {
        const auto* d = reinterpret_cast<const mi_chain_desc*>(static_cast<intptr_t>(whole(a[0])));
        const int last = static_cast<int>(whole(a[1]));
        void* s = stream_of(a[2]);
        const NoGil released;
        st = mi_decoder_chain_run(d, last, s);
    } catch (const Leave&) {
        Py_RETURN_NONE;
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
    return PyLong_FromLong(st);
}

// The handle of torch's current stream.
PyObject* current_stream(PyObject*, PyObject*) {
    try {
        return PyLong_FromVoidPtr(c10::hip::getCurrentHIPStream().stream());
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

#define MI_METHOD(name) \
    {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {MI_METHOD(rmsnorm),
                         MI_METHOD(fused_add_rmsnorm),
                         MI_METHOD(swiglu),
                         MI_METHOD(geglu),
                         MI_METHOD(softmax),
                         MI_METHOD(softmax_argmax),
                         MI_METHOD(greedy_argmax),
                         MI_METHOD(top_p_sample),
                         MI_METHOD(rope_neox_qk),
                         MI_METHOD(bias_rope_neox_qk),
                         MI_METHOD(qk_norm_rope),
                         MI_METHOD(rope_neox),
                         MI_METHOD(rope_tables),
                         MI_METHOD(embedding_gather),
                         MI_METHOD(embedding_rmsnorm),
                         MI_METHOD(chain_run),
                         {"current_stream", current_stream, METH_NOARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_mi_fast", nullptr, -1, methods,
                      nullptr,               nullptr,    nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__mi_fast() { return PyModule_Create(&module); }
