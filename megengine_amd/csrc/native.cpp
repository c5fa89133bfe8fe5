// The Python operators of megengine_amd.ops over the C ABI, as a CPython extension: an operator call from Python costs
// the host little more than its kernel launch.  PyTorch is plumbing only here, as it is in ops.py: it owns device memory
// and the streams.
//
// Through ctypes and torch's Python API one bound call took 6.3 us of host time against 2.7 us for the launch itself:
// 2.7 us in torch.cuda.current_stream() (which builds a Stream object), the rest in argument conversion and in the
// validation that exec repeats.  Here the stream handle is read from c10 directly, tensors are unpacked in place, and a
// bound call replays the launches it was bound to (mi355_convbias_s8_bind): networks of one image are bound by exactly
// this time (58 launches, 20 to 200 us of it).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/Context.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty.h>
#include <ATen/record_function.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mi355_convbias.h"

namespace {

PyObject* g_check = nullptr;       // megengine_amd.lib.check: raises Mi355Error for a non-zero status
PyObject* g_ew_modes = nullptr;    // _abi.EW_MODES, _abi.EW_ARITY
PyObject* g_ew_arity = nullptr;
PyObject* g_error = nullptr;       // megengine_amd.lib.Mi355Error

PyObject* raise_status(int st) {
    PyObject* r = PyObject_CallFunction(g_check, "i", st);
    Py_XDECREF(r);
    if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "mi355 status %d", st);
    return nullptr;
}

void* current_stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

// A ctypes structure's bytes; held while the call runs.
template <class T>
class Struct {
public:
    ~Struct() {
        if (held_) PyBuffer_Release(&view_);
    }
    bool get(PyObject* o, const char* what) {
        if (PyObject_GetBuffer(o, &view_, PyBUF_SIMPLE) != 0) return false;
        held_ = true;
        if (view_.len != (Py_ssize_t)sizeof(T)) {
            PyErr_Format(PyExc_TypeError, "%s has %zd bytes, expected %zu", what, view_.len, sizeof(T));
            return false;
        }
        return true;
    }
    const T* ptr() const { return static_cast<const T*>(view_.buf); }
    const T* operator->() const { return ptr(); }

private:
    Py_buffer view_;
    bool held_ = false;
};

// A tensor argument: null for None, else a contiguous tensor in device memory.
struct Arg {
    const at::Tensor* t = nullptr;
    void* p = nullptr;
    bool get(PyObject* o) {
        if (!o || o == Py_None) return true;
        if (!THPVariable_Check(o)) {
            PyErr_Format(PyExc_TypeError, "expected a torch tensor, got %s", Py_TYPE(o)->tp_name);
            return false;
        }
        const at::Tensor& x = THPVariable_Unpack(o);
        if (!x.is_cuda()) {
            PyErr_Format(PyExc_RuntimeError, "mi355 operators take GPU tensors only (got %s)", x.device().str().c_str());
            return false;
        }
        if (!x.is_contiguous()) {
            PyErr_SetString(PyExc_RuntimeError, "tensor must be contiguous");
            return false;
        }
        t = &x;
        p = x.data_ptr();
        return true;
    }
    bool required(PyObject* o) {
        if (!get(o)) return false;
        if (!t) PyErr_SetString(PyExc_TypeError, "expected a torch tensor, got None");
        return t != nullptr;
    }
};

// Positional and keyword arguments of a fast call into named slots.
bool parse(const char* fn, const char* const* names, int count, int required, PyObject* const* args, Py_ssize_t nargs,
           PyObject* kwnames, PyObject** out) {
    if (nargs > count) {
        PyErr_Format(PyExc_TypeError, "%s() takes at most %d arguments (%zd given)", fn, count, nargs);
        return false;
    }
    for (int i = 0; i < count; ++i) out[i] = i < nargs ? args[i] : nullptr;
    const Py_ssize_t nk = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
    for (Py_ssize_t k = 0; k < nk; ++k) {
        PyObject* name = PyTuple_GET_ITEM(kwnames, k);
        int at = -1;
        for (int i = 0; i < count && at < 0; ++i)
            if (PyUnicode_CompareWithASCIIString(name, names[i]) == 0) at = i;
        if (at < 0 || out[at]) {
            PyErr_Format(PyExc_TypeError, at < 0 ? "%s() got an unexpected keyword argument '%U'" : "%s() got multiple values for argument '%U'",
                         fn, name);
            return false;
        }
        out[at] = args[nargs + k];
    }
    for (int i = 0; i < required; ++i)
        if (!out[i]) {
            PyErr_Format(PyExc_TypeError, "%s() missing required argument '%s'", fn, names[i]);
            return false;
        }
    return true;
}

bool given(PyObject* o) { return o && o != Py_None; }

// the exceptions of c10 as Python exceptions
template <class F>
PyObject* guarded(F f) {
    try {
        return f();
    } catch (const std::exception& e) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// Whether nothing stands between at::empty and the allocator that has to see the call: keys that somebody has included for this thread
// (dispatch modes, functorch, functionalization, tracing), a profiler's callbacks, and the fill of new memory in deterministic runs, which
// shows between the images of an output with a batch stride.
bool straight_to_allocator() {
    const at::Context& context = at::globalContext();
    return (c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty() && !at::hasCallbacks() &&
           !(context.deterministicAlgorithms() && context.deterministicFillUninitializedMemory());
}

// Straight from the allocator where that is so (0.93 us of a call through the dispatcher, 0.73 here)
at::Tensor empty_like_device(at::IntArrayRef shape, at::ScalarType dt, const at::Tensor& like) {
    if (straight_to_allocator()) return at::Tensor(at::detail::empty_cuda(shape, dt, like.device(), std::nullopt));
    return at::empty(shape, at::TensorOptions().dtype(dt).device(like.device()));
}

// Runs a C-ABI call without the GIL (a full queue blocks it).  Taken back also when the call ends in an exception (the host
// caches behind it allocate), which guarded() then turns into a Python one.
template <class F>
int without_gil(F f) {
    struct Released {
        PyThreadState* s = PyEval_SaveThread();
        ~Released() { PyEval_RestoreThread(s); }
    };
    const Released released;
    return f();
}

// dst as given, or a new tensor
struct Out {
    Arg arg;
    at::Tensor fresh;
    PyObject* given_obj = nullptr;
    PyObject* result() {
        if (given_obj) return Py_NewRef(given_obj);
        return THPVariable_Wrap(fresh);
    }
    bool take(PyObject* o) {
        if (!given(o)) return true;
        given_obj = o;
        return arg.get(o);
    }
    void make(at::IntArrayRef shape, at::ScalarType dt, const at::Tensor& like) {
        fresh = empty_like_device(shape, dt, like);
        arg.p = fresh.data_ptr();
        arg.t = &fresh;
    }
};

int out_pack(uint32_t fmt) {
    switch (fmt) {
        case MI355_FMT_NCHW: case MI355_FMT_NCHW4_NCHW: return 1;
        case MI355_FMT_NCHW4: case MI355_FMT_NCHW44: case MI355_FMT_NCHW32_NCHW4: return 4;
        default: return 32;
    }
}

// the output of a ConvBias descriptor; false with a Python error set
bool make_conv_dst(const mi355_conv_desc* d, const at::Tensor& src, Out* out) {
    uint32_t oh, ow;
    const int st = mi355_convbias_deduce_out(d, &oh, &ow);
    if (st) {
        raise_status(st);
        return false;
    }
    const at::ScalarType dt = d->dst_dtype == MI355_DT_QS8 ? at::kChar : d->dst_dtype == MI355_DT_QS32 ? at::kInt : at::kFloat;
    const int64_t po = out_pack(d->format), n = d->n, oc = d->oc;
    if (d->dst_stride_n)
        out->make({n, d->dst_stride_n}, dt, src);
    else if (po == 1)
        out->make({n, oc, (int64_t)oh, (int64_t)ow}, dt, src);
    else
        out->make({n, oc / po, (int64_t)oh, (int64_t)ow, po}, dt, src);
    return true;
}

PyObject* conv_bias_exec(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    static const char* const names[] = {"desc", "src", "flt", "bias", "z", "dst", "algo", "workspace"};
    PyObject* a[8];
    if (!parse("conv_bias_exec", names, 8, 3, args, nargs, kwnames, a)) return nullptr;
    return guarded([&]() -> PyObject* {
        Struct<mi355_conv_desc> d;
        Arg src, flt, bias, z, ws;
        Out dst;
        if (!d.get(a[0], "desc")) return nullptr;
        // the algorithm: the heuristic's, the one of an id, or the caller's own choice
        mi355_algo algo;
        size_t need = 0;
        int st = MI355_OK;
        if (!given(a[6])) {
            st = mi355_convbias_s8_query(d.ptr(), MI355_ALGO_HEURISTIC, &algo, &need);
        } else if (PyLong_Check(a[6])) {
            const int id = (int)PyLong_AsLong(a[6]);
            if (PyErr_Occurred()) return nullptr;
            st = mi355_convbias_s8_query(d.ptr(), id, &algo, &need);
        } else {
            Struct<mi355_algo> given_algo;
            if (!given_algo.get(a[6], "algo")) return nullptr;
            algo = *given_algo.ptr();
            if (!given(a[7]) && algo.id >= 0) st = mi355_convbias_s8_query(d.ptr(), algo.id, nullptr, &need);
        }
        if (st) return raise_status(st);
        if (!src.required(a[1]) || !flt.get(a[2]) || !bias.get(a[3]) || !z.get(a[4]) || !ws.get(a[7]) || !dst.take(a[5])) return nullptr;
        if (!dst.arg.t && !make_conv_dst(d.ptr(), *src.t, &dst)) return nullptr;
        at::Tensor own_ws;
        size_t ws_bytes = ws.t ? (size_t)ws.t->numel() : 0;
        if (!ws.t && need) {
            own_ws = empty_like_device({(int64_t)need}, at::kByte, *src.t);
            ws.p = own_ws.data_ptr();
            ws_bytes = need;
        }
        void* stream = current_stream();
        st = without_gil([&] {
            return mi355_convbias_s8_exec(stream, d.ptr(), &algo, (const int8_t*)src.p, (const int8_t*)flt.p, (const int32_t*)bias.p,
                                          (const int8_t*)z.p, dst.arg.p, ws.p, ws_bytes);
        });
        return st ? raise_status(st) : dst.result();
    });
}

PyObject* conv_bias_exec_preprocessed(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    static const char* const names[] = {"desc", "src", "pre", "bias", "z", "dst", "algo"};
    PyObject* a[7];
    if (!parse("conv_bias_exec_preprocessed", names, 7, 3, args, nargs, kwnames, a)) return nullptr;
    return guarded([&]() -> PyObject* {
        Struct<mi355_conv_desc> d;
        Struct<mi355_algo> algo;
        Arg src, pre, bias, z;
        Out dst;
        if (!d.get(a[0], "desc") || !algo.get(a[6] ? a[6] : Py_None, "algo")) return nullptr;
        if (!src.required(a[1]) || !pre.required(a[2]) || !bias.get(a[3]) || !z.get(a[4]) || !dst.take(a[5])) return nullptr;
        if (!dst.arg.t && !make_conv_dst(d.ptr(), *src.t, &dst)) return nullptr;
        void* stream = current_stream();
        const int st = without_gil([&] {
            return mi355_convbias_s8_exec_preprocessed(stream, d.ptr(), algo.ptr(), (const int8_t*)src.p, pre.p,
                                                       (size_t)pre.t->numel(), (const int32_t*)bias.p, (const int8_t*)z.p, dst.arg.p,
                                                       nullptr, 0);
        });
        return st ? raise_status(st) : dst.result();
    });
}

PyObject* relayout_exec(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    static const char* const names[] = {"d", "src", "dst"};
    PyObject* a[3];
    if (!parse("relayout_exec", names, 3, 2, args, nargs, kwnames, a)) return nullptr;
    return guarded([&]() -> PyObject* {
        Struct<mi355_relayout_desc> d;
        Arg src;
        Out dst;
        if (!d.get(a[0], "d") || !src.required(a[1]) || !dst.take(a[2])) return nullptr;
        if (!dst.arg.t) {
            uint32_t nd, shape[7];
            const int st = mi355_relayout_deduce(d.ptr(), &nd, shape);
            if (st) return raise_status(st);
            int64_t s[7];
            for (uint32_t i = 0; i < nd; ++i) s[i] = shape[i];
            dst.make(at::IntArrayRef(s, nd), src.t->scalar_type(), *src.t);
        }
        void* stream = current_stream();
        const int st = without_gil([&] { return mi355_relayout_exec(stream, d.ptr(), src.p, dst.arg.p); });
        return st ? raise_status(st) : dst.result();
    });
}

bool as_float(PyObject* o, float* out) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) return false;
    *out = (float)v;
    return true;
}

PyObject* requant_exec(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    static const char* const names[] = {"src", "scale_src", "scale_dst", "nonline", "z", "scale_z", "dst"};
    PyObject* a[7];
    if (!parse("requant_exec", names, 7, 3, args, nargs, kwnames, a)) return nullptr;
    return guarded([&]() -> PyObject* {
        mi355_requant_desc d;
        memset(&d, 0, sizeof(d));
        d.nonline = MI355_NL_IDENTITY;
        d.scale_z = 1.f;
        if (given(a[3])) {
            if (PyLong_Check(a[3])) {
                d.nonline = (uint32_t)PyLong_AsLong(a[3]);
                if (PyErr_Occurred()) return nullptr;
            } else {
                static const char* const nl[] = {"IDENTITY", "RELU", "SIGMOID", "H_SWISH"};
                int at = -1;
                for (int i = 0; i < 4 && at < 0; ++i)
                    if (PyUnicode_Check(a[3]) && PyUnicode_CompareWithASCIIString(a[3], nl[i]) == 0) at = i;
                if (at < 0) {
                    PyErr_SetObject(PyExc_KeyError, a[3]);
                    return nullptr;
                }
                d.nonline = (uint32_t)at;
            }
        }
        Arg src, z;
        Out dst;
        if (!src.required(a[0])) return nullptr;
        const at::ScalarType dt = src.t->scalar_type();
        if (dt != at::kInt && dt != at::kChar) {
            PyErr_SetString(PyExc_RuntimeError, "requant_exec takes an int32 or int8 tensor");
            return nullptr;
        }
        if (!as_float(a[1], &d.scale_src) || !as_float(a[2], &d.scale_dst) || (a[5] && !as_float(a[5], &d.scale_z))) return nullptr;
        if (!z.get(a[4]) || !dst.take(a[6])) return nullptr;
        if (!dst.arg.t) dst.make(src.t->sizes(), at::kChar, *src.t);
        d.has_z = z.t ? 1 : 0;
        d.count = (uint64_t)src.t->numel();
        void* stream = current_stream();
        const int st = without_gil([&] {
            return dt == at::kInt ? mi355_requant_s32_s8_exec(stream, &d, (const int32_t*)src.p, (const int8_t*)z.p, (int8_t*)dst.arg.p)
                                  : mi355_requant_s8_s8_exec(stream, &d, (const int8_t*)src.p, (const int8_t*)z.p, (int8_t*)dst.arg.p);
        });
        return st ? raise_status(st) : dst.result();
    });
}

PyObject* elemwise_q_exec(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    static const char* const names[] = {"mode", "srcs", "scales_src", "scale_dst", "dst_dtype", "dst"};
    PyObject* a[6];
    if (!parse("elemwise_q_exec", names, 6, 4, args, nargs, kwnames, a)) return nullptr;
    return guarded([&]() -> PyObject* {
        PyObject* arity = PyDict_GetItemWithError(g_ew_arity, a[0]);
        PyObject* mode = arity ? PyDict_GetItemWithError(g_ew_modes, a[0]) : nullptr;
        if (!arity || !mode) {
            if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, a[0]);
            return nullptr;
        }
        mi355_elemwise_desc d;
        memset(&d, 0, sizeof(d));
        d.mode = (uint32_t)PyLong_AsLong(mode);
        d.arity = (uint32_t)PyLong_AsLong(arity);
        PyObject* srcs = PySequence_Fast(a[1], "srcs must be a sequence");
        if (!srcs) return nullptr;
        PyObject* scales = PySequence_Fast(a[2], "scales_src must be a sequence");
        struct Release {
            PyObject *x, *y;
            ~Release() { Py_XDECREF(x); Py_XDECREF(y); }
        } release{srcs, scales};
        if (!scales) return nullptr;
        if (PySequence_Fast_GET_SIZE(srcs) != (Py_ssize_t)d.arity || PySequence_Fast_GET_SIZE(scales) != (Py_ssize_t)d.arity) {
            PyErr_Format(PyExc_RuntimeError, "%S takes %u inputs", a[0], d.arity);
            return nullptr;
        }
        Arg s[3];
        for (uint32_t i = 0; i < d.arity; ++i) {
            if (!s[i].required(PySequence_Fast_GET_ITEM(srcs, i)) || !as_float(PySequence_Fast_GET_ITEM(scales, i), &d.scale_src[i]))
                return nullptr;
        }
        const at::ScalarType dt = s[0].t->scalar_type();
        bool same = dt == at::kChar || dt == at::kInt;
        for (uint32_t i = 1; i < d.arity; ++i) same = same && s[i].t->scalar_type() == dt && s[i].t->sizes() == s[0].t->sizes();
        if (!same) {
            PyErr_SetString(PyExc_RuntimeError, "elemwise_q_exec takes int8 or int32 tensors of one dtype and shape");
            return nullptr;
        }
        if (!as_float(a[3], &d.scale_dst)) return nullptr;
        Out dst;
        if (!dst.take(a[5])) return nullptr;
        if (!dst.arg.t) {
            at::ScalarType ddt = at::kChar;
            if (given(a[4])) {
                if (!THPDtype_Check(a[4])) {
                    PyErr_SetString(PyExc_TypeError, "dst_dtype must be a torch dtype");
                    return nullptr;
                }
                ddt = reinterpret_cast<THPDtype*>(a[4])->scalar_type;
            }
            dst.make(s[0].t->sizes(), ddt, *s[0].t);
        }
        const at::ScalarType ddt = dst.arg.t->scalar_type();
        if (ddt != at::kChar && ddt != at::kInt) {
            PyErr_SetString(PyExc_KeyError, "dst must be an int8 or int32 tensor");
            return nullptr;
        }
        d.src_dtype = dt == at::kChar ? MI355_DT_QS8 : MI355_DT_QS32;
        d.dst_dtype = ddt == at::kChar ? MI355_DT_QS8 : MI355_DT_QS32;
        d.count = (uint64_t)s[0].t->numel();
        void* stream = current_stream();
        const int st = without_gil([&] { return mi355_elemwise_q_exec(stream, &d, s[0].p, s[1].p, s[2].p, dst.arg.p); });
        return st ? raise_status(st) : dst.result();
    });
}

PyObject* pooling_exec(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    static const char* const names[] = {"d", "src", "dst"};
    PyObject* a[3];
    if (!parse("pooling_exec", names, 3, 2, args, nargs, kwnames, a)) return nullptr;
    return guarded([&]() -> PyObject* {
        Struct<mi355_pooling_desc> d;
        Arg src;
        Out dst;
        if (!d.get(a[0], "d")) return nullptr;
        if (!THPVariable_Check(a[1]) || THPVariable_Unpack(a[1]).scalar_type() != at::kChar) {
            PyErr_SetString(PyExc_RuntimeError, "pooling_exec takes an int8 tensor");
            return nullptr;
        }
        const int64_t pack = d->format == MI355_FMT_NCHW ? 1 : d->format == MI355_FMT_NCHW32 ? 32 : 4;
        const int64_t want[5] = {d->n, d->c / pack, d->ih, d->iw, pack};
        const at::Tensor& x = THPVariable_Unpack(a[1]);
        if (x.sizes() != at::IntArrayRef(want, pack == 1 ? 4 : 5)) {
            PyErr_SetString(PyExc_RuntimeError, "the shape of src does not match the descriptor");
            return nullptr;
        }
        if (!src.required(a[1]) || !dst.take(a[2])) return nullptr;
        if (!dst.arg.t) {
            uint32_t oh, ow;
            const int st = mi355_pooling_deduce_out(d.ptr(), &oh, &ow);
            if (st) return raise_status(st);
            const int64_t shape[5] = {d->n, d->c / pack, oh, ow, pack};
            dst.make(at::IntArrayRef(shape, pack == 1 ? 4 : 5), at::kChar, *src.t);
        }
        void* stream = current_stream();
        const int st = without_gil([&] { return mi355_pooling_s8_exec(stream, d.ptr(), (const int8_t*)src.p, (int8_t*)dst.arg.p); });
        return st ? raise_status(st) : dst.result();
    });
}

PyObject* typecvt_exec(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    static const char* const names[] = {"src", "scale", "dst"};
    PyObject* a[3];
    if (!parse("typecvt_exec", names, 3, 2, args, nargs, kwnames, a)) return nullptr;
    return guarded([&]() -> PyObject* {
        float scale;
        Arg src;
        Out dst;
        if (!as_float(a[1], &scale)) return nullptr;
        if (!THPVariable_Check(a[0]) ||
            (THPVariable_Unpack(a[0]).scalar_type() != at::kFloat && THPVariable_Unpack(a[0]).scalar_type() != at::kChar)) {
            PyErr_SetString(PyExc_RuntimeError, "typecvt_exec takes a float32 or an int8 tensor");
            return nullptr;
        }
        if (!src.required(a[0]) || !dst.take(a[2])) return nullptr;
        const bool quantize = src.t->scalar_type() == at::kFloat;
        if (!dst.arg.t) dst.make(src.t->sizes(), quantize ? at::kChar : at::kFloat, *src.t);
        const uint64_t n = (uint64_t)src.t->numel();
        void* stream = current_stream();
        const int st = without_gil([&] {
            return quantize ? mi355_typecvt_f32_s8_exec(stream, n, scale, (const float*)src.p, (int8_t*)dst.arg.p)
                            : mi355_typecvt_s8_f32_exec(stream, n, scale, (const int8_t*)src.p, (float*)dst.arg.p);
        });
        return st ? raise_status(st) : dst.result();
    });
}

// ---- bound calls ----
struct BoundCall {
    PyObject_HEAD
    vectorcallfunc vectorcall;
    mi355_bound_call* call;
    void* stream;       // a fixed stream, when has_stream
    int has_stream;
    PyObject* error;    // what exec would raise, for a call that could not be bound: raised when it is called
    PyObject* keep;     // the tensors and the descriptor
};

PyObject* bound_run(PyObject* self, PyObject* const*, size_t nargsf, PyObject* kwnames) {
    BoundCall* b = reinterpret_cast<BoundCall*>(self);
    if (PyVectorcall_NARGS(nargsf) || (kwnames && PyTuple_GET_SIZE(kwnames))) {
        PyErr_SetString(PyExc_TypeError, "a bound call takes no arguments");
        return nullptr;
    }
    if (b->error) {
        PyErr_SetObject(g_error, b->error);
        return nullptr;
    }
    return guarded([&]() -> PyObject* {
        void* stream = b->has_stream ? b->stream : current_stream();
        const int st = without_gil([&] { return mi355_bound_call_launch(stream, b->call); });
        if (st) return raise_status(st);
        Py_RETURN_NONE;
    });
}

void bound_dealloc(PyObject* self) {
    BoundCall* b = reinterpret_cast<BoundCall*>(self);
    mi355_bound_call_destroy(b->call);
    Py_XDECREF(b->error);
    Py_XDECREF(b->keep);
    Py_TYPE(self)->tp_free(self);
}

PyTypeObject BoundCallType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* conv_bias_bind(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
    static const char* const names[] = {"desc", "src", "flt", "bias", "z", "dst", "algo", "workspace", "stream", "preprocessed"};
    PyObject* a[10];
    if (!parse("conv_bias_bind", names, 10, 7, args, nargs, kwnames, a)) return nullptr;
    return guarded([&]() -> PyObject* {
        Struct<mi355_conv_desc> d;
        Struct<mi355_algo> algo;
        Arg src, flt, bias, z, dst, ws, pre;
        if (!d.get(a[0], "desc") || !algo.get(a[6], "algo")) return nullptr;
        if (!src.get(a[1]) || !flt.get(a[2]) || !bias.get(a[3]) || !z.get(a[4]) || !dst.get(a[5]) || !ws.get(a[7]) || !pre.get(a[9]))
            return nullptr;
        void* stream = nullptr;
        if (given(a[8])) {
            stream = PyLong_AsVoidPtr(a[8]);
            if (PyErr_Occurred()) return nullptr;
        }
        mi355_bound_call* call = nullptr;
        const int st = mi355_convbias_s8_bind(d.ptr(), algo.ptr(), (const int8_t*)src.p, pre.t ? pre.p : flt.p,
                                              pre.t ? (size_t)pre.t->numel() : 0, (const int32_t*)bias.p, (const int8_t*)z.p, dst.p,
                                              ws.p, ws.t ? (size_t)ws.t->numel() : 0, &call);
        PyObject* error = nullptr;
        if (st && !(error = Py_BuildValue("(is)", st, mi355_last_error()))) return nullptr;
        BoundCall* b = PyObject_New(BoundCall, &BoundCallType);
        if (!b) {
            mi355_bound_call_destroy(call);
            Py_XDECREF(error);
            return nullptr;
        }
        b->vectorcall = bound_run;
        b->call = call;
        b->stream = stream;
        b->has_stream = given(a[8]);
        b->error = error;
        b->keep = PyTuple_New(10);
        if (!b->keep) {
            Py_DECREF(b);
            return nullptr;
        }
        for (int i = 0; i < 10; ++i) PyTuple_SET_ITEM(b->keep, i, Py_NewRef(a[i] ? a[i] : Py_None));
        return reinterpret_cast<PyObject*>(b);
    });
}

#define FAST(name, sig, doc) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL | METH_KEYWORDS, #name sig "\n--\n\n" doc}
PyMethodDef methods[] = {
        FAST(conv_bias_exec, "($module, desc, src, flt, bias=None, z=None, dst=None, algo=None, workspace=None)",
             "megdnn::ConvBiasForward::exec on the current stream; algo: None (the heuristic's), an algorithm id or an Algo."),
        FAST(conv_bias_exec_preprocessed, "($module, desc, src, pre, bias=None, z=None, dst=None, algo=None)",
             "exec with a PreprocessedFilter (the result of conv_bias_preprocess for the same algorithm)."),
        FAST(conv_bias_bind, "($module, desc, src, flt, bias, z, dst, algo, workspace=None, stream=None, preprocessed=None)",
             "Fixes one exec call; the returned callable launches it on the CURRENT torch stream when `stream` is None, else on\n"
             "that raw stream handle, and raises on a non-zero status.  Keeps the tensors alive.  For callers that replay the\n"
             "same launch many times.  With `preprocessed` (the result of conv_bias_preprocess for the same algo) the call is\n"
             "exec with a PreprocessedFilter."),
        FAST(relayout_exec, "($module, d, src, dst=None)", "megdnn::RelayoutFormat::exec."),
        FAST(requant_exec, "($module, src, scale_src, scale_dst, nonline='IDENTITY', z=None, scale_z=1.0, dst=None)",
             "QuantizedS32 or QuantizedS8 (+ QuantizedS8 z) -> QuantizedS8 with the ConvBias epilogue arithmetic."),
        FAST(elemwise_q_exec, "($module, mode, srcs, scales_src, scale_dst, dst_dtype=None, dst=None)",
             "ElemwiseMultiType quantized mode `mode` (name of the Elemwise::Mode, e.g. \"FUSE_MUL_ADD3\") on one to three int8 or\n"
             "int32 tensors of one shape with their scales; dst is QuantizedS8 unless dst_dtype says torch.int32."),
        FAST(pooling_exec, "($module, d, src, dst=None)",
             "megdnn::PoolingForward::exec on a QuantizedS8 tensor (dst carries the scale of src)."),
        FAST(typecvt_exec, "($module, src, scale, dst=None)",
             "megdnn::TypeCvt between Float32 and QuantizedS8: a float32 tensor is quantized with `scale`, an int8 tensor is\n"
             "dequantized with it."),
        {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "Operators over the C ABI (see megengine_amd.ops).", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
    BoundCallType.tp_name = "megengine_amd._native.BoundCall";
    BoundCallType.tp_basicsize = sizeof(BoundCall);
    BoundCallType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
    BoundCallType.tp_vectorcall_offset = offsetof(BoundCall, vectorcall);
    BoundCallType.tp_call = PyVectorcall_Call;
    BoundCallType.tp_dealloc = bound_dealloc;
    BoundCallType.tp_doc = "one ConvBias exec call with its arguments fixed";
    if (PyType_Ready(&BoundCallType) < 0) return nullptr;
    PyObject* lib = PyImport_ImportModule("megengine_amd.lib");
    PyObject* abi = PyImport_ImportModule("megengine_amd._abi");
    if (!lib || !abi) return nullptr;
    g_check = PyObject_GetAttrString(lib, "check");
    g_error = PyObject_GetAttrString(lib, "Mi355Error");
    g_ew_modes = PyObject_GetAttrString(abi, "EW_MODES");
    g_ew_arity = PyObject_GetAttrString(abi, "EW_ARITY");
    if (!g_check || !g_error || !g_ew_modes || !g_ew_arity) return nullptr;
    return PyModule_Create(&module);
}
