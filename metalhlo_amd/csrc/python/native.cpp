// The host path of metalhlo_amd.kernels in C++ (CPython extension `_native`): argument checks, the
// result tensor, the current stream and the call of one C-ABI entry point per operator.  A small operator
// runs for 3 to 6 us on the device; in Python these steps took 8 to 14 us (attribute look-ups, torch.empty,
// torch.cuda.current_stream, ctypes conversions), here about 1 us plus the launch itself.
// Each function takes positional arguments only; metalhlo_amd/kernels.py holds the signatures.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <string>

#include "../../../include/mhip.h"

namespace {

PyObject* g_error = nullptr;      // metalhlo_amd._lib.MhipError(code, message)

struct Failed {};                  // a Python exception is set

[[noreturn]] void raise(PyObject* type, const char* msg) {
    PyErr_SetString(type, msg);
    throw Failed();
}

// Runs the library call `f` without the interpreter lock (a launch waits when the device's queue is full).
template <typename F>
void check(F&& f) {
    PyThreadState* state = PyEval_SaveThread();
    const int code = f();
    PyEval_RestoreThread(state);
    if (code == MHIP_OK) return;
    if (PyObject* args = Py_BuildValue("(is)", code, mhip_last_error())) {
        PyErr_SetObject(g_error, args);
        Py_DECREF(args);
    }
    throw Failed();
}

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kHalf: return MHIP_F16;
        case at::kFloat: return MHIP_F32;
        case at::kDouble: return MHIP_F64;
        case at::kBFloat16: return MHIP_BF16;
        case at::kBool: return MHIP_I1;
        case at::kChar: return MHIP_I8;
        case at::kShort: return MHIP_I16;
        case at::kInt: return MHIP_I32;
        case at::kLong: return MHIP_I64;
        case at::kByte: return MHIP_UI8;
        default: raise(PyExc_TypeError, "unsupported dtype");
    }
}

const at::Tensor& tensor(PyObject* o) {
    if (!THPVariable_Check(o)) raise(PyExc_TypeError, "expected a torch.Tensor");
    return THPVariable_Unpack(o);
}
// a dense device tensor
const at::Tensor& dense(PyObject* o) {
    const at::Tensor& t = tensor(o);
    if (!t.is_cuda()) raise(PyExc_RuntimeError, "metalhlo_amd kernels need device tensors (no CPU path exists)");
    if (!t.is_contiguous()) raise(PyExc_ValueError, "tensors must be dense row-major (contiguous)");
    return t;
}
const at::Tensor* optional_dense(PyObject* o) { return o == Py_None ? nullptr : &dense(o); }
void* ptr(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }

void* stream_of(const at::Tensor&) { return c10::hip::getCurrentHIPStream().stream(); }

at::Tensor empty(at::IntArrayRef shape, at::ScalarType dtype, const at::Tensor& like) {
    return at::detail::empty_cuda(shape, dtype, like.device(), std::nullopt);
}
// Memory that only makes a call faster, from the current stream's pool or a capturing graph's own: none where the device has no more, the
// call then takes its form without it.
at::Tensor workspace(int64_t bytes, const at::Tensor& like) {
    if (bytes <= 0) return {};
    try {
        return empty({bytes}, at::kByte, like);
    } catch (const c10::OutOfMemoryError&) {
        return {};
    }
}
at::Tensor result_like(const at::Tensor& t) { return empty(t.sizes(), t.scalar_type(), t); }

bool truth(PyObject* o) {
    const int r = PyObject_IsTrue(o);
    if (r < 0) throw Failed();
    return r != 0;
}
double number(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw Failed();
    return v;
}
int64_t integer(PyObject* o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw Failed();
    return v;
}

// Runs `f`, turning C++ exceptions into Python ones; checks the number of arguments.
template <typename F>
PyObject* guarded(Py_ssize_t got, Py_ssize_t want, F&& f) {
    if (got != want) {
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
        return nullptr;
    }
    try {
        return f();
    } catch (const Failed&) {
        return nullptr;
    } catch (const std::exception& e) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

#define FUNCTION(name) PyObject* name(PyObject*, PyObject* const* arg, Py_ssize_t n)

// softmax(x, axis)
FUNCTION(softmax) {
    return guarded(n, 2, [&] {
        const at::Tensor& x = dense(arg[0]);
        int64_t axis = integer(arg[1]);
        if (axis < 0) axis += x.dim();
        if (axis < 0 || axis >= x.dim()) raise(PyExc_ValueError, "softmax axis out of range");
        const int dt = dtype_code(x.scalar_type());
        at::Tensor y = result_like(x);
        int64_t outer = 1, inner = 1;
        for (int64_t d = 0; d < axis; d++) outer *= x.size(d);
        for (int64_t d = axis + 1; d < x.dim(); d++) inner *= x.size(d);
        if (inner == 1) check([&] { return mhip_softmax(stream_of(x), x.data_ptr(), y.data_ptr(), outer, x.size(axis), dt); });
        else check([&] { return mhip_softmax_strided(stream_of(x), x.data_ptr(), y.data_ptr(), outer, x.size(axis), inner, dt); });
        return THPVariable_Wrap(std::move(y));
    });
}

void row_parameter(const at::Tensor* p, const at::Tensor& x, int64_t cols, const char* msg) {
    if (p && (p->numel() != cols || p->scalar_type() != x.scalar_type())) raise(PyExc_ValueError, msg);
}

int64_t last_size(const at::Tensor& x) {
    if (x.dim() == 0) raise(PyExc_IndexError, "tuple index out of range");
    return x.size(-1);
}

// layer_norm(x, gamma, beta, eps)
FUNCTION(layer_norm) {
    return guarded(n, 4, [&] {
        const at::Tensor& x = dense(arg[0]);
        const at::Tensor *g = optional_dense(arg[1]), *b = optional_dense(arg[2]);
        const int64_t cols = last_size(x);
        row_parameter(g, x, cols, "gamma/beta must have the row length and dtype of x");
        row_parameter(b, x, cols, "gamma/beta must have the row length and dtype of x");
        const float eps = (float)number(arg[3]);
        const int dt = dtype_code(x.scalar_type());
        at::Tensor y = result_like(x);
        check([&] { return mhip_layer_norm(stream_of(x), x.data_ptr(), ptr(g), ptr(b), y.data_ptr(), x.numel() / (cols > 0 ? cols : 1), cols,
                              eps, dt); });
        return THPVariable_Wrap(std::move(y));
    });
}

// rms_norm(x, gamma, eps)
FUNCTION(rms_norm) {
    return guarded(n, 3, [&] {
        const at::Tensor& x = dense(arg[0]);
        const at::Tensor* g = optional_dense(arg[1]);
        const int64_t cols = last_size(x);
        row_parameter(g, x, cols, "gamma must have the row length and dtype of x");
        const float eps = (float)number(arg[2]);
        const int dt = dtype_code(x.scalar_type());
        at::Tensor y = result_like(x);
        check([&] { return mhip_rms_norm(stream_of(x), x.data_ptr(), ptr(g), y.data_ptr(), x.numel() / (cols > 0 ? cols : 1), cols,
                            eps, dt); });
        return THPVariable_Wrap(std::move(y));
    });
}

// bias_gelu(x, bias, exact)
FUNCTION(bias_gelu) {
    return guarded(n, 3, [&] {
        const at::Tensor& x = dense(arg[0]);
        const at::Tensor* b = optional_dense(arg[1]);
        const int64_t cols = x.dim() ? x.size(-1) : 1;
        row_parameter(b, x, cols, "bias must have the row length and dtype of x");
        const auto entry = truth(arg[2]) ? mhip_bias_gelu_erf : mhip_bias_gelu;
        const int dt = dtype_code(x.scalar_type());
        at::Tensor y = result_like(x);
        check([&] { return entry(stream_of(x), x.data_ptr(), ptr(b), y.data_ptr(),
                                                                   x.numel() / (cols > 0 ? cols : 1), cols, dt); });
        return THPVariable_Wrap(std::move(y));
    });
}

// matmul(a, b, bias, activation code, trans_a, trans_b, out, residual)
FUNCTION(matmul) {
    return guarded(n, 8, [&] {
        const at::Tensor &a = dense(arg[0]), &b = dense(arg[1]);
        const at::Tensor *bias = optional_dense(arg[2]), *out = optional_dense(arg[6]), *res = optional_dense(arg[7]);
        const bool ta = truth(arg[4]), tb = truth(arg[5]);
        if (a.scalar_type() != b.scalar_type()) raise(PyExc_TypeError, "operand dtypes differ");
        const int64_t ad = a.dim(), bd = b.dim();
        if (ad < 1 || bd < 2) raise(PyExc_ValueError, "matmul needs matrices");
        int64_t batch = 1, sa = 0, sb = 0, rows, M, K;
        c10::SmallVector<int64_t, 8> shape;
        if (bd == 2) {
            if (ta && ad != 2) raise(PyExc_ValueError, "trans_a needs a 2-D lhs when rhs is 2-D");
            const int64_t last = a.size(-1);
            // (as `a.reshape(-1, 0)` says: no number of rows follows from the element count)
            if (ad != 2 && last == 0) raise(PyExc_RuntimeError, "matmul cannot fold the leading dims of an lhs whose last axis is empty");
            rows = ad == 2 ? a.size(0) : a.numel() / last;
            M = ta ? last : rows;
            K = ta ? rows : last;
            if (ta) shape.push_back(last);
            else for (int64_t d = 0; d + 1 < ad; d++) shape.push_back(a.size(d));
        } else {
            bool same = ad == bd;
            for (int64_t d = 0; same && d + 2 < ad; d++) same = a.size(d) == b.size(d);
            if (!same) raise(PyExc_ValueError, "batched matmul needs equal batch dims");
            for (int64_t d = 0; d + 2 < ad; d++) { batch *= a.size(d); shape.push_back(a.size(d)); }
            M = a.size(ta ? -1 : -2);
            K = a.size(ta ? -2 : -1);
            sa = M * K;
            sb = b.size(-1) * b.size(-2);
            shape.push_back(M);
        }
        const int64_t Kb = b.size(tb ? -1 : -2), N = b.size(tb ? -2 : -1);
        if (K != Kb) raise(PyExc_ValueError, ("contracting sizes differ: " + std::to_string(K) + " vs " + std::to_string(Kb)).c_str());
        if (bias && (bias->numel() != N || bias->scalar_type() != a.scalar_type())) raise(PyExc_ValueError, "bias must be [N] of the operand dtype");
        shape.push_back(N);
        at::Tensor c = out ? *out : empty(shape, a.scalar_type(), a);
        if (res && (res->numel() != c.numel() || res->scalar_type() != c.scalar_type()))
            raise(PyExc_ValueError, "residual must have the result's size and dtype");
        const int dt = dtype_code(a.scalar_type()), act = (int)integer(arg[3]);
        const at::Tensor work = workspace(mhip_gemm_workspace(M, N, K, batch, ta, tb, dt), a);
        check([&] { return mhip_gemm_ws(stream_of(a), a.data_ptr(), b.data_ptr(), ptr(bias), ptr(res), c.data_ptr(), M, N, K, batch, sa, sb, M * N, ta, tb,
                           act, dt, work.defined() ? work.data_ptr() : nullptr, work.defined() ? work.numel() : 0); });
        return THPVariable_Wrap(std::move(c));
    });
}

const float* f32(const at::Tensor* t) { return t ? t->data_ptr<float>() : nullptr; }

// A tuple of up to two matrices that the next calls read.
int weights_ahead(PyObject* o, mhip_weights (&ahead)[2]) {
    int n = 0;
    if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) > 2) raise(PyExc_ValueError, "ahead must be a tuple of up to two matrices");
    for (; n < PyTuple_GET_SIZE(o); n++) {
        const at::Tensor* t = &dense(PyTuple_GET_ITEM(o, n));
        if (t->dim() != 2 || t->scalar_type() != at::kFloat) raise(PyExc_TypeError, "weights ahead must be fp32 matrices");
        ahead[n] = {t->data_ptr<float>(), t->size(1), t->size(0)};
    }
    return n;
}

// linear(x, weight, bias, residual, activation code, trans_b, parts, (weights ahead)): parameters in fp32;
// parts > 0: the fp32 sums of so many shares of K instead
FUNCTION(linear) {
    return guarded(n, 8, [&] {
        const at::Tensor &x = dense(arg[0]), &w = dense(arg[1]);
        const at::Tensor *bias = optional_dense(arg[2]), *res = optional_dense(arg[3]);
        const bool tb = truth(arg[5]);
        const int parts = (int)integer(arg[6]);
        if (x.dim() != 2 || w.dim() != 2) raise(PyExc_ValueError, "linear needs matrices");
        const int64_t M = x.size(0), K = x.size(1), N = w.size(tb ? 0 : 1);
        if (w.size(tb ? 1 : 0) != K) raise(PyExc_ValueError, "contracting sizes differ");
        for (const at::Tensor* p : {&w, bias})
            if (p && p->scalar_type() != at::kFloat) raise(PyExc_TypeError, "parameters must be fp32");
        if (bias && bias->numel() != N) raise(PyExc_ValueError, "bias must be [N]");
        if (res && (res->numel() != M * N || res->scalar_type() != x.scalar_type())) raise(PyExc_ValueError, "residual must have the result's size and dtype");
        const int dt = dtype_code(x.scalar_type()), act = (int)integer(arg[4]);
        at::Tensor c = parts > 0 ? empty({parts, M, N}, at::kFloat, x) : empty({M, N}, x.scalar_type(), x);
        mhip_weights ahead[2] = {};
        const int n_ahead = weights_ahead(arg[7], ahead);
        check([&] { return mhip_linear_w32(stream_of(x), x.data_ptr(), f32(&w), f32(bias), ptr(res),
                                           parts > 0 ? nullptr : c.data_ptr(), M, N, K, tb, act, dt, parts > 0 ? c.data_ptr<float>() : nullptr,
                                           parts > 0 ? parts : 1, n_ahead, ahead); });
        return THPVariable_Wrap(std::move(c));
    });
}

// tied_head(x, weight fp32 [N, K])
FUNCTION(tied_head) {
    return guarded(n, 2, [&] {
        const at::Tensor &x = dense(arg[0]), &w = dense(arg[1]);
        if (x.dim() != 2 || w.dim() != 2 || x.size(1) != w.size(1)) raise(PyExc_ValueError, "tied_head needs [M, K] and [N, K]");
        if (w.scalar_type() != at::kFloat) raise(PyExc_TypeError, "parameters must be fp32");
        const int dt = dtype_code(x.scalar_type());
        at::Tensor c = empty({x.size(0), w.size(0)}, x.scalar_type(), x);
        check([&] { return mhip_tied_head(stream_of(x), x.data_ptr(), w.data_ptr<float>(), c.data_ptr(), x.size(0), w.size(0), x.size(1), dt); });
        return THPVariable_Wrap(std::move(c));
    });
}

// matmul_sums(a, b, parts) -> [parts, M, N] fp32
FUNCTION(matmul_sums) {
    return guarded(n, 3, [&] {
        const at::Tensor &a = dense(arg[0]), &b = dense(arg[1]);
        const int64_t parts = integer(arg[2]);
        if (a.dim() != 2 || b.dim() != 2 || a.size(1) != b.size(0)) raise(PyExc_ValueError, "matmul_sums needs [M, K] and [K, N]");
        if (a.scalar_type() != b.scalar_type()) raise(PyExc_TypeError, "operand dtypes differ");
        if (parts < 1 || parts > 8) raise(PyExc_ValueError, "1 to 8 parts");
        const int dt = dtype_code(a.scalar_type());
        at::Tensor c = empty({parts, a.size(0), b.size(1)}, at::kFloat, a);
        check([&] { return mhip_gemm_sums(stream_of(a), a.data_ptr(), b.data_ptr(), c.data_ptr<float>(), a.size(0), b.size(1), a.size(1), dt, (int)parts); });
        return THPVariable_Wrap(std::move(c));
    });
}

// linear_layer(x, norm or None = (gamma, beta, eps), weight, bias, residual, activation code, (weights ahead))
FUNCTION(linear_layer) {
    return guarded(n, 7, [&] {
        const at::Tensor &x = dense(arg[0]), &w = dense(arg[2]);
        const at::Tensor *bias = optional_dense(arg[3]), *res = optional_dense(arg[4]), *gamma = nullptr, *beta = nullptr;
        float eps = 0.f;
        if (arg[1] != Py_None) {
            if (!PyTuple_Check(arg[1]) || PyTuple_GET_SIZE(arg[1]) != 3) raise(PyExc_ValueError, "norm must be (gamma, beta, eps)");
            gamma = &dense(PyTuple_GET_ITEM(arg[1], 0));
            beta = optional_dense(PyTuple_GET_ITEM(arg[1], 1));
            eps = (float)number(PyTuple_GET_ITEM(arg[1], 2));
        }
        if (x.dim() != 2 || w.dim() != 2 || w.size(0) != x.size(1)) raise(PyExc_ValueError, "linear_layer needs matrices [M, K] and [K, N]");
        const int64_t M = x.size(0), K = x.size(1), N = w.size(1);
        for (const at::Tensor* p : {&w, bias, gamma, beta})
            if (p && p->scalar_type() != at::kFloat) raise(PyExc_TypeError, "parameters must be fp32");
        if (bias && bias->numel() != N) raise(PyExc_ValueError, "bias must be [N]");
        if ((gamma && gamma->numel() != K) || (beta && beta->numel() != K)) raise(PyExc_ValueError, "gamma and beta must be [K]");
        if (res && (res->numel() != M * N || res->scalar_type() != x.scalar_type())) raise(PyExc_ValueError, "residual must have the result's size and dtype");
        const int dt = dtype_code(x.scalar_type()), act = (int)integer(arg[5]);
        at::Tensor c = empty({M, N}, x.scalar_type(), x), work;
        const int64_t bytes = gamma ? 0 : mhip_linear_w32_workspace(M, N, K);
        if (bytes > 0) work = empty({bytes}, at::kByte, x);
        mhip_weights ahead[2] = {};
        const int n_ahead = weights_ahead(arg[6], ahead);
        check([&] { return mhip_linear_w32_layer(stream_of(x), x.data_ptr(), f32(gamma), f32(beta), eps, f32(&w), f32(bias), ptr(res), c.data_ptr(), M, N, K, act, dt,
                                                 bytes > 0 ? work.data_ptr() : nullptr, bytes, n_ahead, ahead); });
        return THPVariable_Wrap(std::move(c));
    });
}

// finish_norm(sums or None, bias, residual, gamma, beta, eps) -> (c, LayerNorm(c)); without sums c is the residual
FUNCTION(finish_norm) {
    return guarded(n, 6, [&]() -> PyObject* {
        const at::Tensor *sums = optional_dense(arg[0]), *bias = optional_dense(arg[1]), *beta = optional_dense(arg[4]);
        const at::Tensor &res = dense(arg[2]), &gamma = dense(arg[3]);
        const int64_t N = last_size(res), M = N ? res.numel() / N : 0;
        for (const at::Tensor* p : {sums, bias, &gamma, beta})
            if (p && p->scalar_type() != at::kFloat) raise(PyExc_TypeError, "sums and parameters must be fp32");
        if (gamma.numel() != N || (beta && beta->numel() != N) || (bias && bias->numel() != N)) raise(PyExc_ValueError, "parameters must have the row length");
        if (sums && (sums->dim() != 3 || sums->size(1) != M || sums->size(2) != N)) raise(PyExc_ValueError, "sums must be [parts, rows, columns]");
        const int dt = dtype_code(res.scalar_type());
        const float eps = (float)number(arg[5]);
        at::Tensor c = sums ? result_like(res) : res, h = result_like(res);
        check([&] { return mhip_finish_norm(stream_of(res), f32(sums), sums ? (int)sums->size(0) : 0, f32(bias), res.data_ptr(), sums ? c.data_ptr() : nullptr,
                                            f32(&gamma), f32(beta), eps, h.data_ptr(), M, N, dt); });
        PyObject *a = THPVariable_Wrap(std::move(c)), *b = THPVariable_Wrap(std::move(h));
        PyObject* r = a && b ? PyTuple_Pack(2, a, b) : nullptr;
        Py_XDECREF(a);
        Py_XDECREF(b);
        return r;
    });
}

// causal_attention(qkv [B * S, 3 H D], B, H) -> [B * S, H D]: Q, K and V read in place
FUNCTION(causal_attention) {
    return guarded(n, 3, [&] {
        const at::Tensor& x = dense(arg[0]);
        const int64_t B = integer(arg[1]), H = integer(arg[2]);
        if (x.dim() != 2 || B < 1 || H < 1 || x.size(0) % B != 0 || x.size(1) % (3 * H) != 0) raise(PyExc_ValueError, "expected a projection [B * S, 3 H D]");
        const int64_t S = x.size(0) / B, d = x.size(1) / 3, D = d / H;
        const int dt = dtype_code(x.scalar_type());
        at::Tensor o = empty({B * S, d}, x.scalar_type(), x);
        const int64_t in[3] = {S * 3 * d, D, 3 * d}, strides[12] = {in[0], in[1], in[2], in[0], in[1], in[2], in[0], in[1], in[2], S * d, D, d};
        char* p = static_cast<char*>(x.data_ptr());
        const int64_t step = d * x.element_size();
        check([&] { return mhip_flash_attention_strided(stream_of(x), p, p + step, p + 2 * step, nullptr, o.data_ptr(), B, H, S, S, D,
                                                        (float)(1.0 / std::sqrt((double)D)), 1, 0, 0, dt, strides); });
        return THPVariable_Wrap(std::move(o));
    });
}

// attend_project_layer(qkv [B * S, 3 H D], weight fp32 [H D, N], bias, residual, B, H, (weights ahead)) -> [B * S, N]
FUNCTION(attend_project_layer) {
    return guarded(n, 7, [&] {
        const at::Tensor &x = dense(arg[0]), &w = dense(arg[1]);
        const at::Tensor *bias = optional_dense(arg[2]), *res = optional_dense(arg[3]);
        const int64_t B = integer(arg[4]), H = integer(arg[5]);
        if (x.dim() != 2 || B < 1 || H < 1 || x.size(0) % B != 0 || x.size(1) % (3 * H) != 0) raise(PyExc_ValueError, "expected a projection [B * S, 3 H D]");
        const int64_t S = x.size(0) / B, D = x.size(1) / 3 / H;
        if (w.dim() != 2 || w.size(0) != H * D) raise(PyExc_ValueError, "expected a weight [H D, N]");
        const int64_t M = x.size(0), N = w.size(1);
        for (const at::Tensor* p : {&w, bias})
            if (p && p->scalar_type() != at::kFloat) raise(PyExc_TypeError, "parameters must be fp32");
        if (bias && bias->numel() != N) raise(PyExc_ValueError, "bias must be [N]");
        if (res && (res->numel() != M * N || res->scalar_type() != x.scalar_type())) raise(PyExc_ValueError, "residual must have the result's size and dtype");
        const int dt = dtype_code(x.scalar_type());
        mhip_weights ahead[2] = {};
        const int n_ahead = weights_ahead(arg[6], ahead);
        at::Tensor c = empty({M, N}, x.scalar_type(), x);
        check([&] { return mhip_attend_project_layer(stream_of(x), x.data_ptr(), f32(&w), f32(bias), ptr(res), c.data_ptr(), B, S, H, D, N, dt, n_ahead, ahead); });
        return THPVariable_Wrap(std::move(c));
    });
}

// attend_project(qkv [B * S, 3 H D], weight fp32 [H D, N], B, H, (weights ahead)) -> fp32 [parts, B * S, N]
FUNCTION(attend_project) {
    return guarded(n, 5, [&] {
        const at::Tensor &x = dense(arg[0]), &w = dense(arg[1]);
        const int64_t B = integer(arg[2]), H = integer(arg[3]);
        if (x.dim() != 2 || B < 1 || H < 1 || x.size(0) % B != 0 || x.size(1) % (3 * H) != 0) raise(PyExc_ValueError, "expected a projection [B * S, 3 H D]");
        const int64_t S = x.size(0) / B, D = x.size(1) / 3 / H;
        if (w.dim() != 2 || w.size(0) != H * D) raise(PyExc_ValueError, "expected a weight [H D, N]");
        if (w.scalar_type() != at::kFloat) raise(PyExc_TypeError, "parameters must be fp32");
        const int dt = dtype_code(x.scalar_type());
        mhip_weights ahead[2] = {};
        const int n_ahead = weights_ahead(arg[4], ahead), parts = mhip_attend_project_parts(B, S, H, D, w.size(1), dt);
        at::Tensor c = empty({parts > 0 ? parts : 1, x.size(0), w.size(1)}, at::kFloat, x);
        check([&] { return mhip_attend_project(stream_of(x), x.data_ptr(), w.data_ptr<float>(), c.data_ptr<float>(), B, S, H, D, w.size(1), dt, n_ahead, ahead); });
        return THPVariable_Wrap(std::move(c));
    });
}

// flash_attention(q, k, v, scale or None, is_causal, mask, out)
FUNCTION(flash_attention) {
    return guarded(n, 7, [&] {
        const at::Tensor &q = tensor(arg[0]), &k = tensor(arg[1]), &v = tensor(arg[2]);
        const at::Tensor* given = arg[6] == Py_None ? nullptr : &tensor(arg[6]);
        const at::Tensor* views[4] = {&q, &k, &v, given};
        for (const at::Tensor* t : views)
            if (t && (!t->is_cuda() || t->dim() != 4 || t->stride(3) != 1))
                raise(PyExc_ValueError, "attention operands must be 4-D device tensors with a contiguous last axis");
        const at::Tensor* mask = optional_dense(arg[5]);
        if (k.sizes() != v.sizes() || q.size(0) != k.size(0) || q.size(1) != k.size(1) || q.size(3) != k.size(3))
            raise(PyExc_ValueError, "expected q [B,H,Sq,D] and k,v [B,H,Skv,D]");
        if (q.scalar_type() != k.scalar_type() || k.scalar_type() != v.scalar_type()) raise(PyExc_TypeError, "q, k, v dtypes differ");
        const int64_t B = q.size(0), H = q.size(1), Sq = q.size(2), D = q.size(3), Skv = k.size(2);
        const double scale = arg[3] == Py_None ? 1.0 / std::sqrt((double)D) : number(arg[3]);
        int64_t msb = 0, msh = 0;
        if (mask) {
            if (mask->scalar_type() != q.scalar_type()) raise(PyExc_TypeError, "mask dtype must match q");
            int64_t m[4] = {1, 1, 1, 1};
            const int64_t md = mask->dim();
            bool ok = md <= 4;
            for (int64_t d = 0; ok && d < md; d++) m[4 - md + d] = mask->size(d);
            if (!ok || m[2] != Sq || m[3] != Skv || (m[0] != 1 && m[0] != B) || (m[1] != 1 && m[1] != H))
                raise(PyExc_ValueError, "mask must broadcast to [B,H,Sq,Skv] with full last two dims");
            msh = m[1] == H ? Sq * Skv : 0;
            msb = m[0] == B ? m[1] * Sq * Skv : 0;
        }
        if (given && (given->sizes() != q.sizes() || given->scalar_type() != q.scalar_type())) raise(PyExc_ValueError, "out must have q's shape and dtype");
        at::Tensor o = given ? *given : empty(q.sizes(), q.scalar_type(), q);
        const bool causal = truth(arg[4]);
        const int dt = dtype_code(q.scalar_type());
        const bool packed = q.is_contiguous() && k.is_contiguous() && v.is_contiguous() && o.is_contiguous();
        int64_t strides[12];
        views[3] = &o;
        for (int t = 0; !packed && t < 4; t++)
            for (int d = 0; d < 3; d++) strides[3 * t + d] = views[t]->stride(d);
        const at::Tensor work = workspace(mhip_flash_attention_workspace(B, H, Sq, Skv, D, causal, dt), q);
        check([&] { return mhip_flash_attention_ws(stream_of(q), q.data_ptr(), k.data_ptr(), v.data_ptr(), ptr(mask), o.data_ptr(), B, H, Sq, Skv, D,
                                                   (float)scale, causal, msb, msh, dt, packed ? nullptr : strides, work.defined() ? work.data_ptr() : nullptr,
                                                   work.defined() ? work.numel() : 0); });
        return THPVariable_Wrap(std::move(o));
    });
}

// argmax(x, 64-bit indices?, with values?)
FUNCTION(argmax) {
    return guarded(n, 3, [&]() -> PyObject* {
        const at::Tensor& x = dense(arg[0]);
        const int64_t cols = last_size(x);
        const at::ScalarType it = truth(arg[1]) ? at::kLong : at::kInt;
        at::Tensor idx = empty(x.sizes().slice(0, x.dim() - 1), it, x), val;
        const bool values = truth(arg[2]);
        if (values) val = empty(x.sizes().slice(0, x.dim() - 1), x.scalar_type(), x);
        const int dt = dtype_code(x.scalar_type()), idt = dtype_code(it);
        check([&] { return mhip_argmax(stream_of(x), x.data_ptr(), idx.data_ptr(), values ? val.data_ptr() : nullptr, cols ? x.numel() / cols : 0, cols,
                          dt, idt); });
        if (!values) return THPVariable_Wrap(std::move(idx));
        PyObject *a = THPVariable_Wrap(std::move(idx)), *b = THPVariable_Wrap(std::move(val));
        PyObject* r = a && b ? PyTuple_Pack(2, a, b) : nullptr;
        Py_XDECREF(a);
        Py_XDECREF(b);
        return r;
    });
}

// bind(error type)
FUNCTION(bind) {
    return guarded(n, 1, [&]() -> PyObject* {
        Py_INCREF(arg[0]);
        Py_XSETREF(g_error, arg[0]);
        Py_RETURN_NONE;
    });
}

#define ENTRY(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {ENTRY(softmax), ENTRY(layer_norm), ENTRY(rms_norm), ENTRY(bias_gelu), ENTRY(matmul), ENTRY(linear), ENTRY(linear_layer), ENTRY(matmul_sums), ENTRY(tied_head), ENTRY(finish_norm), ENTRY(causal_attention), ENTRY(attend_project), ENTRY(attend_project_layer),
                          ENTRY(flash_attention), ENTRY(argmax), ENTRY(bind), {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__native(void) { return PyModule_Create(&kModule); }
