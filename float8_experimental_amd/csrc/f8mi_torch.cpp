// The host path of the fused linear (training forward, backward; inference) over libf8mi's C ABI, as a CPython module on
// torch tensors: one call allocates what the kernels write and queues all launches of a direction.  Host code only.
//
// Why: a layer of 512 tokens, 1024 -> 1024, is 59 us of kernels; issued launch by launch from Python (allocation, checks,
// pointer and stream look-ups and a ctypes call each) the same step was bound by the host at 172 - 218 us.
//
// Every function returns None, without having queued or allocated anything, for arguments that it does not take (subclasses,
// other devices, layouts that need a copy, odd scales): the caller then goes through the checked Python functions of
// _native.py, which raise what there is to raise.  Workspaces are temporaries of torch's caching allocator: it hands their
// memory out again in stream order, so calls on any number of threads, streams and captures share nothing but the delayed
// cast's words, which the library guards.
//
// The Python arguments are read first, tensors by value; allocations and launches then run without the GIL, as under ctypes and
// torch's own bindings: a launch may block on a full queue, an allocation on hipMalloc, and other Python threads go on.
#include <dlfcn.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/f8mi.h"

namespace {

struct Lib {
    decltype(&f8mi_cast_dynamic) cast_dynamic;
    decltype(&f8mi_cast_layout) cast_layout;
    decltype(&f8mi_cast_delayed) cast_delayed;
    decltype(&f8mi_cast_dynamic_pair) cast_dynamic_pair;
    decltype(&f8mi_cast_delayed_pair) cast_delayed_pair;
    decltype(&f8mi_gemm_nt_ws) gemm_nt_ws;
    decltype(&f8mi_gemm_nt_kb_ws) gemm_nt_kb_ws;
    decltype(&f8mi_gemm_kb_ex) gemm_kb_ex;
    decltype(&f8mi_gemm_pair) gemm_pair;
    decltype(&f8mi_gemm_kb_bias) gemm_kb_bias;
    decltype(&f8mi_column_sum) column_sum;
    decltype(&f8mi_column_sum_workspace_bytes) column_sum_workspace_bytes;
    decltype(&f8mi_gemm_plan) gemm_plan;
    decltype(&f8mi_linear_few_rows) linear_few_rows;
    decltype(&f8mi_last_error) last_error;
    size_t workspace_bytes;
} L;
PyObject* native_error = nullptr;  // float8_experimental_amd._native.Float8NativeError

struct NativeFailure {
    const char* what;
    int rc;
};
void check(int rc, const char* what) {
    if (rc != 0) throw NativeFailure{what, rc};
}

int dtype_code(at::ScalarType t) {
    return t == at::kBFloat16 ? F8MI_BF16 : t == at::kHalf ? F8MI_FP16 : t == at::kFloat ? F8MI_FP32 : -1;
}
int fp8_code(at::ScalarType t) { return t == at::kFloat8_e4m3fn ? F8MI_E4M3FN : t == at::kFloat8_e5m2 ? F8MI_E5M2 : -1; }
at::ScalarType fp8_type(int fmt) { return fmt == F8MI_E4M3FN ? at::kFloat8_e4m3fn : at::kFloat8_e5m2; }
int64_t padded(int64_t k, int layout) { return layout == F8MI_LAYOUT_KBLOCK64_PAD128 ? (k + 127) / 128 * 128 : k; }

// sizes of the fp8 copy of `rows` rows that contracts over kc, in the layout
std::vector<int64_t> copy_sizes(int64_t rows, int64_t kc, int layout) {
    if (layout == F8MI_LAYOUT_ROWMAJOR) return {rows, kc};
    return {padded(kc, layout) / 64, rows, 64};
}

// Undefined: not taken.  A plain tensor (or Parameter) on the current device: nothing of a subclass, no other layout, no lazy negation ...
at::Tensor plain(PyObject* o, int device) {
    if (!THPVariable_CheckExact(o)) return {};
    const at::Tensor& t = THPVariable_Unpack(o);
    constexpr c10::DispatchKeySet lazy({c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(lazy) && t.get_device() == device ? t : at::Tensor();
}
// ... that the cast kernels read as it is: 2-D, not empty, unit column stride
at::Tensor matrix(PyObject* o, int device) {
    const at::Tensor t = plain(o, device);
    return t.defined() && t.dim() == 2 && dtype_code(t.scalar_type()) >= 0 && t.size(0) > 0 && t.size(1) > 0 && t.stride(1) == 1 && t.stride(0) >= t.size(1) ? t : at::Tensor();
}
// ... one fp32 element: a scale or an amax
at::Tensor one_float(PyObject* o, int device) {
    const at::Tensor t = plain(o, device);
    return t.defined() && t.scalar_type() == at::kFloat && t.numel() == 1 ? t : at::Tensor();
}

// How one tensor is scaled: dynamically, with a scale known beforehand, or delayed (with its amax buffer).
struct Scaling {
    at::Tensor scale, amax;
    // `known`: a scale or None; `delayed`: (amax, scale) or None.  False: not taken.
    bool parse(PyObject* known, PyObject* delayed, int device) {
        if (delayed != Py_None) {
            if (!PyTuple_Check(delayed) || PyTuple_GET_SIZE(delayed) != 2) return false;
            amax = one_float(PyTuple_GET_ITEM(delayed, 0), device);
            scale = one_float(PyTuple_GET_ITEM(delayed, 1), device);
            return amax.defined() && scale.defined();
        }
        if (known == Py_None) return true;
        scale = one_float(known, device);
        return scale.defined();
    }
};

struct Call {
    void* stream;
    int device;
    void* delayed_ws;

    at::Tensor make(at::IntArrayRef sizes, at::ScalarType t) const {
        return at::empty(sizes, at::TensorOptions().dtype(t).device(at::Device(at::kCUDA, (c10::DeviceIndex)device)));
    }
    at::Tensor copy(int64_t rows, int64_t kc, int layout, int fmt) const {
        return make(copy_sizes(rows, kc, layout), fp8_type(fmt));
    }

    // The fp8 copies of x: `row` contracts over the columns, `tr` (the transpose) over the rows.
    void cast(const at::Tensor& x, const Scaling& s, int fmt, bool want_row, int row_layout, bool want_tr, int tr_layout, at::Tensor& row,
              at::Tensor& tr, at::Tensor& scale, int product_dtype = -1) const {
        const int64_t m = x.size(0), k = x.size(1), ld = x.stride(0);
        const int dt = dtype_code(x.scalar_type());
        if (want_row) row = copy(m, k, row_layout, fmt);
        if (want_tr) tr = copy(k, m, tr_layout, fmt);
        uint8_t* pr = want_row ? (uint8_t*)row.data_ptr() : nullptr;
        uint8_t* pt = want_tr ? (uint8_t*)tr.data_ptr() : nullptr;
        if (!s.scale.defined()) {
            scale = make({}, at::kFloat);
            const at::Tensor ws = make({(int64_t)L.workspace_bytes / 4}, at::kInt);
            check(L.cast_dynamic(x.data_ptr(), m, k, ld, dt, fmt, (float*)scale.data_ptr(), pr, row_layout, pt, tr_layout, ws.data_ptr(), stream),
                  "f8mi_cast_dynamic");
            return;
        }
        scale = s.scale;
        if (s.amax.defined())
            check(L.cast_delayed(x.data_ptr(), m, k, ld, dt, (const float*)scale.data_ptr(), fmt, pr, row_layout, pt, tr_layout,
                                 (float*)s.amax.data_ptr(), delayed_ws, stream), "f8mi_cast_delayed");
        else
            check(L.cast_layout(x.data_ptr(), m, k, ld, dt, (const float*)scale.data_ptr(), product_dtype < 0 ? dt : product_dtype, fmt, pr, row_layout,
                                pt, tr_layout, nullptr, stream), "f8mi_cast_layout");
    }

    // The e4m3 copies of two tensors, both scaled dynamically or both delayed, as one library call.
    struct Cast {
        const at::Tensor& x;
        const Scaling& s;
        bool want_tr;
        int row_layout, tr_layout;
        at::Tensor &row, &tr, &scale;
    };
    void cast_two(const Cast& a, const Cast& b) const {
        const bool delayed = a.s.amax.defined() && b.s.amax.defined(), dynamic = !a.s.scale.defined() && !b.s.scale.defined();
        if (!delayed && !dynamic) {
            for (const Cast* c : {&a, &b}) cast(c->x, c->s, F8MI_E4M3FN, true, c->row_layout, c->want_tr, c->tr_layout, c->row, c->tr, c->scale);
            return;
        }
        f8mi_cast_job jobs[2];
        int i = 0;
        for (const Cast* c : {&a, &b}) {
            const int64_t m = c->x.size(0), k = c->x.size(1);
            c->row = copy(m, k, c->row_layout, F8MI_E4M3FN);
            if (c->want_tr) c->tr = copy(k, m, c->tr_layout, F8MI_E4M3FN);
            c->scale = delayed ? c->s.scale : make({}, at::kFloat);
            jobs[i++] = {c->x.data_ptr(), m, k, c->x.stride(0), (float*)c->scale.data_ptr(), (uint8_t*)c->row.data_ptr(), c->want_tr ? (uint8_t*)c->tr.data_ptr() : nullptr,
                         delayed ? (float*)c->s.amax.data_ptr() : nullptr, dtype_code(c->x.scalar_type()), c->row_layout, c->tr_layout};
        }
        if (delayed) {
            check(L.cast_delayed_pair(&jobs[0], &jobs[1], delayed_ws, stream), "f8mi_cast_delayed_pair");
        } else {
            const at::Tensor ws = make({(int64_t)L.workspace_bytes / 4}, at::kInt);
            check(L.cast_dynamic_pair(&jobs[0], &jobs[1], ws.data_ptr(), stream), "f8mi_cast_dynamic_pair");
        }
    }

    // scratch for a product that is split over k
    at::Tensor split_workspace(int64_t m, int64_t n, int64_t k, int layout, int64_t& bytes) const {
        bytes = 0;
        if (m < 17 || k < 2048 || (layout == F8MI_LAYOUT_ROWMAJOR && k % 16 != 0)) return {};  // below these none is
        const int plan = L.gemm_plan(m, n, k, 1, F8MI_GEMM_WORKSPACE_BYTES);
        if ((plan & 0xff) != F8MI_PLAN_TILES128_SPLIT_K) return {};
        bytes = (int64_t)((plan >> 8) & 0xff) * m * n * 4;
        return make({bytes / 4}, at::kFloat);
    }

    // a [m][k] times bt [n][k] in the layout, both contracting over kc (before padding)
    at::Tensor gemm(const at::Tensor& a, const at::Tensor& sa, const at::Tensor& bt, const at::Tensor& sb, int layout, int64_t m, int64_t n,
                    int64_t kc, at::ScalarType out, const at::Tensor& bias = {}) const {
        const at::Tensor c = make({m, n}, out);
        const int64_t k = padded(kc, layout);
        int64_t ws_bytes = 0;
        const at::Tensor ws = split_workspace(m, n, k, layout, ws_bytes);
        void* pws = ws_bytes ? ws.data_ptr() : nullptr;
        const float *pa = (const float*)sa.data_ptr(), *pb = (const float*)sb.data_ptr();
        const int fa = fp8_code(a.scalar_type()), fb = fp8_code(bt.scalar_type()), dt = dtype_code(out);
        const void* pbias = bias.defined() ? bias.data_ptr() : nullptr;
        if (layout == F8MI_LAYOUT_ROWMAJOR)
            check(L.gemm_nt_ws(a.data_ptr(), fa, k, bt.data_ptr(), fb, k, m, n, k, pa, pb, c.data_ptr(), dt, n, pbias, pws, ws_bytes, stream), "f8mi_gemm_nt_ws");
        else
            check(L.gemm_nt_kb_ws(a.data_ptr(), fa, bt.data_ptr(), fb, m, n, k, pa, pb, c.data_ptr(), dt, n, pbias, pws, ws_bytes, stream), "f8mi_gemm_nt_kb_ws");
        return c;
    }
    // y = x8 w8^T (in the type of x), plus the bias added to the rounded product
    at::Tensor gemm_biased(const at::Tensor& a, const at::Tensor& sa, const at::Tensor& bt, const at::Tensor& sb, int layout, int64_t m, int64_t n,
                           int64_t kc, at::ScalarType out, const at::Tensor& bias) const {
        const int64_t k = padded(kc, layout);
        if (layout != F8MI_LAYOUT_ROWMAJOR && (bias.scalar_type() == out || bias.scalar_type() == at::kFloat)) {
            const at::Tensor c = make({m, n}, out);
            const int rc = L.gemm_kb_bias(a.data_ptr(), bt.data_ptr(), m, n, k, (const float*)sa.data_ptr(), (const float*)sb.data_ptr(), c.data_ptr(),
                                          dtype_code(out), n, bias.data_ptr(), dtype_code(bias.scalar_type()), F8MI_GEMM_WORKSPACE_BYTES, stream);
            if (rc != F8MI_ERR_UNSUPPORTED) {
                check(rc, "f8mi_gemm_kb_bias");
                return c;
            }
        }
        return gemm(a, sa, bt, sb, layout, m, n, kc, out).add_(bias.to(out));
    }

    at::Tensor gemm_tr(const at::Tensor& a, bool a_tr, const at::Tensor& sa, const at::Tensor& bt, const at::Tensor& sb, int64_t m, int64_t n,
                       int64_t k, at::ScalarType out) const {
        at::Tensor c = make({m, n}, out);
        check(L.gemm_kb_ex(a.data_ptr(), fp8_code(a.scalar_type()), a_tr, bt.data_ptr(), fp8_code(bt.scalar_type()), 1, m, n, k, (const float*)sa.data_ptr(),
                           (const float*)sb.data_ptr(), c.data_ptr(), dtype_code(out), n, nullptr, stream), "f8mi_gemm_kb_ex");
        return c;
    }

    // One product of a library call that computes two, of k-blocked operands.
    struct Product {
        const at::Tensor &a, &sa, &bt, &sb;
        bool a_tr, b_tr;
        int layout;
        int64_t m, n, kc;
        at::Tensor& c;
    };
    // wide: the second result in fp32, rounded to `out` as the first
    void gemm_two(const Product& p, const Product& q, at::ScalarType out, bool wide) const {
        f8mi_gemm_job jobs[2];
        at::Tensor ws[2];
        int i = 0;
        for (const Product* g : {&p, &q}) {
            const int64_t k = padded(g->kc, g->layout);
            int64_t bytes = 0;
            if (!g->b_tr) ws[i] = split_workspace(g->m, g->n, k, g->layout, bytes);
            const bool fp32 = wide && g == &q;
            g->c = make({g->m, g->n}, fp32 ? at::kFloat : out);
            jobs[i] = {g->a.data_ptr(), g->bt.data_ptr(), fp8_code(g->a.scalar_type()), fp8_code(g->bt.scalar_type()), g->a_tr, g->b_tr, g->m, g->n, k,
                       (const float*)g->sa.data_ptr(), (const float*)g->sb.data_ptr(), g->c.data_ptr(), g->n, !fp32 ? dtype_code(out) : out == at::kHalf ? F8MI_FP16_IN_FP32 : F8MI_BF16_IN_FP32, bytes ? ws[i].data_ptr() : nullptr, bytes};
            i++;
        }
        const int rc = L.gemm_pair(&jobs[0], &jobs[1], F8MI_PAIR_BY_SIZE, stream);
        if (wide && rc == F8MI_ERR_UNSUPPORTED) return gemm_two(p, q, out, false);  // the caller converts it
        check(rc, "f8mi_gemm_pair");
    }
};

PyObject* wrap(const at::Tensor& t) {
    if (!t.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(t);
}
template <typename... T>
PyObject* wrap_all(const T&... t) {
    PyObject* r = PyTuple_New(sizeof...(t));
    if (!r) return nullptr;
    Py_ssize_t i = 0;
    for (PyObject* o : {wrap(t)...}) PyTuple_SET_ITEM(r, i++, o);
    return r;
}
struct WithoutGil {
    PyThreadState* state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};
template <typename F>
PyObject* guarded(F body) {
    HANDLE_TH_ERRORS
    try {
        return body();
    } catch (const NativeFailure& f) {
        PyErr_Format(native_error, "%s failed with code %d: %s", f.what, f.rc, L.last_error());
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}
bool expect(Py_ssize_t got, Py_ssize_t want, const char* name, int optional = 0) {
    if (!L.gemm_plan) PyErr_SetString(PyExc_RuntimeError, "f8mi_torch: load() has not been called");
    else if (got < want || got > want + optional) PyErr_Format(PyExc_TypeError, "%s takes %zd arguments, got %zd", name, want, got);
    else return true;
    return false;
}
int as_int(PyObject* o) { return (int)PyLong_AsLong(o); }
void* as_ptr(PyObject* o) { return o == Py_None ? nullptr : PyLong_AsVoidPtr(o); }

// linear_forward(x [m, k], weight [n, k], one_copy, kb_fwd, kb_dx, kb_dw, need_dx, need_dw, delayed_x, delayed_w, weight_scale,
//                delayed_workspace, device, stream, bias = None) -> (y, saved of x, saved of weight, scale of x, scale of weight) or None
PyObject* linear_forward(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    if (!expect(n_args, 14, "linear_forward", 1)) return nullptr;
    return guarded([&]() -> PyObject* {
        const Call c{as_ptr(a[13]), as_int(a[12]), as_ptr(a[11])};
        const at::Tensor x = matrix(a[0], c.device), w = matrix(a[1], c.device);
        Scaling in, we;
        if (!x.defined() || !w.defined() || x.size(1) != w.size(1) || !in.parse(Py_None, a[8], c.device) || !we.parse(a[10], a[9], c.device)) Py_RETURN_NONE;
        if ((in.amax.defined() || we.amax.defined()) && !c.delayed_ws) Py_RETURN_NONE;
        const bool with_bias = n_args > 14 && a[14] != Py_None;
        const at::Tensor bias = with_bias ? plain(a[14], c.device) : at::Tensor();
        if (with_bias && (!bias.defined() || dtype_code(bias.scalar_type()) < 0 || bias.dim() != 1 || bias.size(0) != w.size(0) || !bias.is_contiguous())) Py_RETURN_NONE;
        const bool one_copy = as_int(a[2]), need_dx = as_int(a[6]), need_dw = as_int(a[7]);
        const int kb_fwd = as_int(a[3]), kb_dx = as_int(a[4]), kb_dw = as_int(a[5]);
        at::Tensor y, x8, x8t, sx, w8, w8t, sw;
        {
            const WithoutGil no_gil;
            c.cast_two({x, in, !one_copy && need_dw, kb_fwd, kb_dw, x8, x8t, sx}, {w, we, !one_copy && need_dx, kb_fwd, kb_dx, w8, w8t, sw});
            if (with_bias) y = c.gemm_biased(x8, sx, w8, sw, kb_fwd, x.size(0), w.size(0), x.size(1), x.scalar_type(), bias);
            else y = c.gemm(x8, sx, w8, sw, kb_fwd, x.size(0), w.size(0), x.size(1), x.scalar_type());
        }
        if (one_copy) return wrap_all(y, x8, w8, sx, sw);
        return wrap_all(y, x8t, w8t, sx, sw);
    });
}

// linear_backward(dy [m, n], saved of x, saved of weight, scale of x, scale of weight, k, one_copy, kb_dx, kb_dw, need_dx, need_dw,
//                 delayed_dy, delayed_workspace, device, stream, fp32 weight = False) -> (grad of x [m, k], grad of weight [n, k]) or None.
//                 The gradient of an fp32 weight comes in fp32 where a kernel stores it so (both gradients wanted, products on tiles), with the
//                 values of dy's type; else in that type.
PyObject* linear_backward(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    if (!expect(n_args, 15, "linear_backward", 1)) return nullptr;
    return guarded([&]() -> PyObject* {
        const Call c{as_ptr(a[14]), as_int(a[13]), as_ptr(a[12])};
        const at::Tensor dy = matrix(a[0], c.device);
        const bool one_copy = as_int(a[6]), need_dx = as_int(a[9]), need_dw = as_int(a[10]);
        const at::Tensor xs = need_dw ? plain(a[1], c.device) : at::Tensor(), ws = need_dx ? plain(a[2], c.device) : at::Tensor();
        const at::Tensor sx = one_float(a[3], c.device), sw = one_float(a[4], c.device);
        Scaling go;
        if (!dy.defined() || !sx.defined() || !sw.defined() || xs.defined() != need_dw || ws.defined() != need_dx || !(need_dx || need_dw) ||
            !go.parse(Py_None, a[11], c.device))
            Py_RETURN_NONE;
        if (go.amax.defined() && !c.delayed_ws) Py_RETURN_NONE;
        const int kb_dx = as_int(a[7]), kb_dw = as_int(a[8]);
        const int64_t m = dy.size(0), n = dy.size(1), k = PyLong_AsLongLong(a[5]);
        // what saved-tensor hooks hand back has to be what was saved: dense fp8 copies of the sizes the products assume
        for (const at::Tensor* t : {&xs, &ws}) {
            if (!t->defined()) continue;
            const int64_t rows = one_copy ? (t == &xs ? m : n) : k, kc = one_copy ? k : (t == &xs ? m : n);
            const int layout = one_copy ? F8MI_LAYOUT_KBLOCK64 : t == &xs ? kb_dw : kb_dx;
            if (fp8_code(t->scalar_type()) < 0 || !t->is_contiguous() || t->sizes() != copy_sizes(rows, kc, layout)) Py_RETURN_NONE;
        }
        const bool wide = n_args > 15 && as_int(a[15]) && dy.scalar_type() != at::kFloat;
        at::Tensor g8, g8t, sg, dx, dw;
        const auto compute = [&] {
            if (one_copy) {
                c.cast(dy, go, F8MI_E5M2, true, F8MI_LAYOUT_KBLOCK64, false, 0, g8, g8t, sg);
                if (need_dx && need_dw) {
                    c.gemm_two({g8, sg, ws, sw, false, true, F8MI_LAYOUT_KBLOCK64, m, k, n, dx}, {g8, sg, xs, sx, true, true, F8MI_LAYOUT_KBLOCK64, n, k, m, dw}, dy.scalar_type(), wide);
                    return;
                }
                if (need_dx) dx = c.gemm_tr(g8, false, sg, ws, sw, m, k, n, dy.scalar_type());
                if (need_dw) dw = c.gemm_tr(g8, true, sg, xs, sx, n, k, m, dy.scalar_type());
            } else {
                c.cast(dy, go, F8MI_E5M2, need_dx, kb_dx, need_dw, kb_dw, g8, g8t, sg);
                if (need_dx && need_dw && kb_dx != F8MI_LAYOUT_ROWMAJOR && kb_dw != F8MI_LAYOUT_ROWMAJOR) {
                    c.gemm_two({g8, sg, ws, sw, false, false, kb_dx, m, k, n, dx}, {g8t, sg, xs, sx, false, false, kb_dw, n, k, m, dw}, dy.scalar_type(), wide);
                    return;
                }
                if (need_dx) dx = c.gemm(g8, sg, ws, sw, kb_dx, m, k, n, dy.scalar_type());
                if (need_dw) dw = c.gemm(g8t, sg, xs, sx, kb_dw, n, k, m, dy.scalar_type());
            }
        };
        {
            const WithoutGil no_gil;
            compute();
        }
        return wrap_all(dx, dw);
    });
}

// Whether a kernel may take t's memory for its values, and nobody has to see the operators: no subclass, functional transform, dispatch mode
// or lazy negation.
bool memory_holds_values(const at::Tensor& t) {
    using K = c10::DispatchKey;
    constexpr c10::DispatchKeySet others({K::Python, K::FuncTorchBatched, K::FuncTorchGradWrapper, K::Batched, K::Functionalize, K::Negative, K::Conjugate, K::ZeroTensor});
    return t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(others) && !c10::impl::TorchDispatchModeTLS::any_modes_set();
}

// The gradient of a bias: the columns of dy summed in fp32, rounded to dy's type, in the type of the bias.
at::Tensor bias_gradient(const at::Tensor& dy, at::ScalarType type) {
    const at::Tensor d = dy.reshape({-1, dy.size(-1)});
    if (at::GradMode::is_enabled() || !memory_holds_values(d) || dtype_code(d.scalar_type()) < 0 || d.numel() == 0 || d.stride(1) != 1 || d.stride(0) < d.size(1))
        return d.sum(0).to(type);  // with create_graph a sum that has a gradient itself
    const c10::DeviceGuard guard(d.device());
    const int64_t rows = d.size(0), cols = d.size(1);
    const int dt = dtype_code(d.scalar_type());
    const int64_t bytes = L.column_sum_workspace_bytes(rows, cols, dt);
    const at::Tensor out = at::empty({cols}, d.options().dtype(type)), ws = bytes ? at::empty({bytes / 4}, d.options().dtype(at::kFloat)) : at::Tensor();
    const int rc = L.column_sum(d.data_ptr(), rows, cols, d.stride(0), dt, out.data_ptr(), dtype_code(type), bytes ? ws.data_ptr() : nullptr, bytes,
                                c10::hip::getCurrentHIPStream(d.get_device()).stream());
    TORCH_CHECK(rc == 0, "f8mi_column_sum failed with code ", rc, ": ", L.last_error());
    return out;
}

// y + bias as a node of its own behind the product's, as an addition is one: asked for the gradient of the bias alone, autograd leaves the
// product's node, its saved tensors and the maxima of a delayed dy alone.  added: y holds the sum already, and nobody else has it: its memory
// is the result, neither a view (which a caller could not change in place) nor marked as changed (which compiled autograd does not take).
struct AddBias : torch::autograd::Function<AddBias> {
    static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& y, const at::Tensor& bias, bool added) {
        ctx->saved_data["type"] = (int64_t)bias.scalar_type();
        return added ? at::_unsafe_view(y, y.sizes()) : y + bias.to(y.scalar_type());
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, const torch::autograd::variable_list& grads) {
        at::Tensor db;
        if (ctx->needs_input_grad(1)) db = bias_gradient(grads[0], (at::ScalarType)ctx->saved_data["type"].toInt());
        return {grads[0], db, at::Tensor()};
    }
};

// add_bias(y, bias, added) -> y + bias with a history.  For a bias of one of the kernels' types.
PyObject* add_bias(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    if (!expect(n_args, 3, "add_bias")) return nullptr;
    return guarded([&]() -> PyObject* {
        if (!THPVariable_Check(a[0]) || !THPVariable_Check(a[1])) return PyErr_Format(PyExc_TypeError, "add_bias takes two tensors");
        const at::Tensor y = THPVariable_Unpack(a[0]), bias = THPVariable_Unpack(a[1]);
        const bool added = PyObject_IsTrue(a[2]);
        at::Tensor out;
        {
            const WithoutGil no_gil;
            out = AddBias::apply(y, bias, added);
        }
        return wrap(out);
    });
}

// Cast and product of a few rows in one kernel: every workgroup of 16 or 32 columns converts all of the activations for itself, which
// costs more than the launch it saves once there are many of them and many rows.  us, two launches / one kernel, bf16: 1 row, 65536 x
// 4096: 67.4 / 64.3; 8 rows, 24576 x 4096: 26.2 / 25.4, 98304 x 4096: 81.2 / 86.9; 16 rows, 14336 x 2048: 15.0 / 12.9, 24576 x 2048: 18.3 /
// 19.2, 131072 x 2048: 67.3 / 84.0.  fp32 holds twice the registers and reaches the line earlier: 4 rows, 14336 x 8192: 29.9 / 24.9, 24576
// x 8192: 44.5 / 46.1; 8 rows, 24576 x 4096: 28.8 / 29.3, 98304 x 4096: 88.9 / 107.8.
bool one_kernel_pays(int64_t m, int64_t n, int64_t k, int dt) {
    if (m > 16 || m * k > F8MI_FEW_ROWS_ELEMS) return false;
    return dt == F8MI_FP32 ? n <= 16384 || m * n <= 65536 : m * n <= 262144;
}

// inference_linear(x [m, k], weight (fp8, [n, k] or k-blocked), n, layout, weight_scale, static_scale, bias, device, stream) -> y or None
PyObject* inference_linear(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    if (!expect(n_args, 9, "inference_linear")) return nullptr;
    return guarded([&]() -> PyObject* {
        const Call c{as_ptr(a[8]), as_int(a[7]), nullptr};
        const at::Tensor x = matrix(a[0], c.device), w = plain(a[1], c.device), sw = one_float(a[4], c.device);
        const at::Tensor bias = a[6] == Py_None ? at::Tensor() : plain(a[6], c.device);
        const int64_t n = PyLong_AsLongLong(a[2]);
        const int layout = as_int(a[3]);
        Scaling in;
        if (!x.defined() || !w.defined() || !sw.defined() || (a[6] != Py_None && !bias.defined()) || !in.parse(a[5], Py_None, c.device)) Py_RETURN_NONE;
        const int64_t m = x.size(0), k = x.size(1);
        if (n <= 0 || fp8_code(w.scalar_type()) < 0 || !w.is_contiguous() || w.numel() != n * padded(k, layout)) Py_RETURN_NONE;
        if (bias.defined() && (bias.scalar_type() != x.scalar_type() || bias.numel() != n || !bias.is_contiguous())) Py_RETURN_NONE;
        // a 0-dim scale leaves the product in x's dtype, a scale with a dimension promotes it to fp32
        const int dt = dtype_code(x.scalar_type()), product = in.scale.defined() && in.scale.dim() > 0 ? F8MI_FP32 : dt;
        const auto compute = [&]() -> at::Tensor {
            if (one_kernel_pays(m, n, k, dt) && layout != F8MI_LAYOUT_KBLOCK64_PAD128) {  // cast and product in one kernel
                const at::Tensor y = c.make({m, n}, x.scalar_type());
                const int rc = L.linear_few_rows(x.data_ptr(), x.stride(0), dt, in.scale.defined() ? (const float*)in.scale.data_ptr() : nullptr, product,
                                                 w.data_ptr(), fp8_code(w.scalar_type()), layout, (const float*)sw.data_ptr(), m, n, k, y.data_ptr(), n,
                                                 bias.defined() ? bias.data_ptr() : nullptr, c.stream);
                if (rc != F8MI_ERR_UNSUPPORTED) {
                    check(rc, "f8mi_linear_few_rows");
                    return y;
                }
            }
            at::Tensor x8, none, sx;
            c.cast(x, in, F8MI_E4M3FN, true, layout, false, 0, x8, none, sx, product);
            return c.gemm(x8, sx, w, sw, layout, m, n, k, x.scalar_type(), bias);
        };
        at::Tensor y;
        {
            const WithoutGil no_gil;
            y = compute();
        }
        return wrap(y);
    });
}

// load(path of libf8mi.so, error class): resolves the entry points
PyObject* load(PyObject*, PyObject* args) {
    const char* path;
    PyObject* error;
    if (!PyArg_ParseTuple(args, "sO", &path, &error)) return nullptr;
    void* h = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    if (!h) return PyErr_Format(PyExc_ImportError, "%s", dlerror());
    const char* missing = nullptr;
    auto get = [&](auto& f, const char* name) {
        f = reinterpret_cast<std::decay_t<decltype(f)>>(dlsym(h, name));
        if (!f) missing = name;
    };
    decltype(&f8mi_workspace_bytes) workspace_bytes;
    get(workspace_bytes, "f8mi_workspace_bytes");
    get(L.cast_dynamic, "f8mi_cast_dynamic");
    get(L.cast_layout, "f8mi_cast_layout");
    get(L.cast_delayed, "f8mi_cast_delayed");
    get(L.gemm_nt_ws, "f8mi_gemm_nt_ws");
    get(L.gemm_nt_kb_ws, "f8mi_gemm_nt_kb_ws");
    get(L.gemm_kb_ex, "f8mi_gemm_kb_ex");
    get(L.linear_few_rows, "f8mi_linear_few_rows");
    get(L.last_error, "f8mi_last_error");
    get(L.gemm_plan, "f8mi_gemm_plan");
    get(L.cast_dynamic_pair, "f8mi_cast_dynamic_pair");
    get(L.cast_delayed_pair, "f8mi_cast_delayed_pair");
    get(L.gemm_pair, "f8mi_gemm_pair");
    get(L.gemm_kb_bias, "f8mi_gemm_kb_bias");
    get(L.column_sum, "f8mi_column_sum");
    get(L.column_sum_workspace_bytes, "f8mi_column_sum_workspace_bytes");
    if (missing) {
        L.gemm_plan = nullptr;
        return PyErr_Format(PyExc_ImportError, "%s does not export %s", path, missing);
    }
    L.workspace_bytes = workspace_bytes();
    Py_INCREF(error);
    native_error = error;
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"load", load, METH_VARARGS, nullptr},
    {"linear_forward", (PyCFunction)(void (*)(void))linear_forward, METH_FASTCALL, nullptr},
    {"linear_backward", (PyCFunction)(void (*)(void))linear_backward, METH_FASTCALL, nullptr},
    {"add_bias", (PyCFunction)(void (*)(void))add_bias, METH_FASTCALL, nullptr},
    {"inference_linear", (PyCFunction)(void (*)(void))inference_linear, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_f8mi_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__f8mi_torch(void) { return PyModule_Create(&module); }
