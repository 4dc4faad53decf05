// The Python face's usual calls, in one native call each: check the operands, allocate the result and the workspace with torch's allocator, call the C ABI.
//
// What a small product or layer took was the host: 8.2 us for a product, of which its launch is 4 (torch.empty 1.7, filling the descriptor, the workspace
// query and the call through ctypes, the checks in Python), 12 us for a convolution of one launch, 23 for its two gradients.  Every function here takes
// the plain forms only (exact tensors in device memory, contiguous or a transposed matrix, whole-number options) and returns None for everything else,
// errors included: functional.py then goes its general way, which raises them.  A non-zero status of the C ABI comes back as an int.
// us a call through ctypes | so: a small product 8.2 | 4.8, linear 8.3 | 5.1, a convolution of one tap 12.4 | 5.6, its gradients 22.6 | 14.3.
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>

#include "../../include/ntgemm.h"

namespace {

struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

int ntg_dtype(at::ScalarType t) {
    switch (t) {
    case at::kHalf: return NTG_FLOAT16;
    case at::kBFloat16: return NTG_BFLOAT16;
    case at::kFloat: return NTG_FLOAT32;
    case at::kDouble: return NTG_FLOAT64;
    case at::kChar: return NTG_INT8;
    case at::kShort: return NTG_INT16;
    case at::kInt: return NTG_INT32;
    case at::kLong: return NTG_INT64;
    case at::kByte: return NTG_UINT8;
    default: return -1;
    }
}

// Modes see torch's own calls only on the general way.
bool modes_active() { return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled(); }

// a plain tensor in device memory (no subclass, no wrapper without storage)
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() ? &t : nullptr;
}

at::Tensor fresh(at::IntArrayRef size, const at::Tensor& like) { return at::empty(size, at::TensorOptions().dtype(like.scalar_type()).device(like.device())); }
at::Tensor bytes(int64_t n, const at::Tensor& like) { return at::empty({n}, at::TensorOptions().dtype(at::kByte).device(like.device())); }

bool whole(PyObject* o, int64_t& v) {
    if (!PyLong_CheckExact(o)) return false;
    int over = 0;
    v = PyLong_AsLongLongAndOverflow(o, &over);
    return over == 0;
}
// an option per axis: one number for all, or a tuple or list of as many
bool per_axis(PyObject* o, int nd, int64_t* v) {
    if (whole(o, v[0])) {
        for (int a = 1; a < nd; ++a) v[a] = v[0];
        return true;
    }
    if (nd < 2 || !(PyTuple_CheckExact(o) || PyList_CheckExact(o)) || PySequence_Fast_GET_SIZE(o) != nd) return false;
    for (int a = 0; a < nd; ++a)
        if (!whole(PySequence_Fast_GET_ITEM(o, a), v[a])) return false;
    return true;
}

// gemm(a, b, bias or None, transpose_a, transpose_b, relu, stream)
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 7 || modes_active()) Py_RETURN_NONE;
    const at::Tensor *a = plain(args[0]), *b = plain(args[1]), *bias = nullptr;
    if (!a || !b || a->dim() < 2 || b->dim() < 2 || a->scalar_type() != b->scalar_type()) Py_RETURN_NONE;
    const int dt = ntg_dtype(a->scalar_type());
    if (dt < 0) Py_RETURN_NONE;
    bool ta = args[3] == Py_True, tb = args[4] == Py_True;
    const bool relu = args[5] == Py_True;
    if ((!ta && args[3] != Py_False) || (!tb && args[4] != Py_False)) Py_RETURN_NONE;
    int64_t stream;
    if (!whole(args[6], stream)) Py_RETURN_NONE;
    const int64_t da = a->dim(), db = b->dim();
    // (a view that is a transposed matrix flips its flag; with a side of one both readings are right and the general way picks)
    const auto matrix = [](const at::Tensor& t, bool& flag) {
        if (t.is_contiguous()) return true;
        if (t.dim() != 2 || t.size(0) < 2 || t.size(1) < 2 || t.stride(0) != 1 || t.stride(1) != t.size(0)) return false;
        flag = !flag;
        return true;
    };
    int64_t ar = a->size(da - 2), ac = a->size(da - 1), br = b->size(db - 2), bc = b->size(db - 1);
    const bool fa = ta, fb = tb;
    if (!matrix(*a, ta) || !matrix(*b, tb)) Py_RETURN_NONE;
    const int64_t m = fa ? ac : ar, k = fa ? ar : ac, kb = fb ? bc : br, n = fb ? br : bc;
    if (k != kb || m <= 0 || n <= 0 || k <= 0) Py_RETURN_NONE;
    int64_t batch = 1;
    const at::Tensor& big = da >= db ? *a : *b;
    if (da > 2 && db > 2) {
        if (da != db) Py_RETURN_NONE;
        for (int64_t i = 0; i < da - 2; ++i)
            if (a->size(i) != b->size(i)) Py_RETURN_NONE;
    }
    c10::SmallVector<int64_t, 6> size;
    for (int64_t i = 0; i < big.dim() - 2; ++i) { size.push_back(big.size(i)); batch *= big.size(i); }
    size.push_back(m);
    size.push_back(n);
    if (batch <= 0) Py_RETURN_NONE;
    if (args[2] != Py_None) {
        bias = plain(args[2]);
        if (!bias || da != 2 || db != 2 || bias->dim() != 1 || bias->size(0) != n || !bias->is_contiguous() || bias->scalar_type() != a->scalar_type()) Py_RETURN_NONE;
    }
    ntg_gemm_desc d;
    std::memset(&d, 0, sizeof d);
    d.dtype = dt; d.transpose_a = ta; d.transpose_b = tb; d.c_mode = bias ? NTG_C_BIAS : NTG_C_OVERWRITE;
    d.m = m; d.k = k; d.n = n;
    d.batches = batch;
    d.stride_a = da > 2 || batch == 1 ? m * k : 0; d.stride_b = db > 2 || batch == 1 ? k * n : 0; d.stride_c = m * n;
    if (bias) { d.bias = bias->data_ptr(); d.bias_col_stride = 1; }
    at::Tensor c, ws;
    int status;
    {
        NoGil unlocked;
        c = fresh(size, *a);
        const int64_t need = ntg_gemm_workspace_bytes(&d);
        if (need > 0) {
            ws = bytes(need, *a);
            d.workspace = ws.data_ptr();
            d.workspace_bytes = need;
        }
        status = (relu ? ntg_gemm_relu_dev : ntg_gemm_dev)(&d, a->data_ptr(), b->data_ptr(), c.data_ptr(), reinterpret_cast<void*>(stream));
    }
    if (status) return PyLong_FromLong(status);
    return THPVariable_Wrap(std::move(c));
    END_HANDLE_TH_ERRORS
}

// ---- convolutions over one to three axes: [batch][channels][size], [out channels][channels / groups][kernel] ----
struct Geometry {
    int nd;
    int64_t B, C, O, groups, size[3], k[3], s[3], p[3], d[3], out[3];
};

// Options, sizes and kernels from here on go the general way, where no sum or product of them wraps: a padding of 2^63 - 1 must not come out as -1.
constexpr int64_t LARGE = int64_t(1) << 31;

bool options(Geometry& g, PyObject* stride, PyObject* padding, PyObject* dilation, PyObject* groups) {
    if (!per_axis(stride, g.nd, g.s) || !per_axis(padding, g.nd, g.p) || !per_axis(dilation, g.nd, g.d) || !whole(groups, g.groups) || g.groups < 1) return false;
    for (int a = 0; a < g.nd; ++a)
        if (g.s[a] < 1 || g.d[a] < 1 || g.p[a] < 0 || g.s[a] >= LARGE || g.d[a] >= LARGE || g.p[a] >= LARGE) return false;
    return true;
}
// image and kernel as they are given; the outputs' sizes
bool shapes(Geometry& g, at::IntArrayRef image, at::IntArrayRef kernel) {
    g.B = image[0]; g.C = image[1]; g.O = kernel[0];
    if (g.B < 1 || g.C < 1 || g.O < 1 || g.C % g.groups != 0 || kernel[1] != g.C / g.groups || g.O % g.groups != 0) return false;
    for (int a = 0; a < g.nd; ++a) {
        g.size[a] = image[2 + a]; g.k[a] = kernel[2 + a];
        if (g.size[a] >= LARGE || g.k[a] >= LARGE) return false;
        const int64_t reach = g.size[a] + 2 * g.p[a] - g.d[a] * (g.k[a] - 1) - 1;
        if (g.size[a] < 1 || g.k[a] < 1 || reach < 0) return false;
        g.out[a] = reach / g.s[a] + 1;
    }
    return true;
}
// the two-axis entry points' arguments (one axis: a single image row and tap row)
struct Two { int64_t h, w, kr, kc, sr, sc, pr, pc, dr, dc; };
Two two(const Geometry& g) {
    const int c = g.nd - 1;
    return {g.nd == 1 ? 1 : g.size[0], g.size[c], g.nd == 1 ? 1 : g.k[0], g.k[c], g.nd == 1 ? 1 : g.s[0], g.s[c], g.nd == 1 ? 0 : g.p[0], g.p[c], g.nd == 1 ? 1 : g.d[0], g.d[c]};
}
const at::Tensor* dense(PyObject* o, int nd) {
    const at::Tensor* t = plain(o);
    return t && t->dim() == nd + 2 && t->is_contiguous() ? t : nullptr;
}

constexpr int NOT_TAKEN = -1;
int forward(const Geometry& g, int dt, const at::Tensor& x, const at::Tensor& w, at::Tensor& y, void* stream) {
    c10::SmallVector<int64_t, 5> size = {g.B, g.O};
    for (int a = 0; a < g.nd; ++a) size.push_back(g.out[a]);
    if (g.nd < 3) {
        const Two t = two(g);
        const int64_t need = ntg_conv2d_fast_workspace_bytes(dt, g.B, g.C, t.h, t.w, g.O, t.kr, t.kc, t.sr, t.sc, t.pr, t.pc, t.dr, t.dc, g.groups);
        if (need < 0) return NOT_TAKEN;
        y = fresh(size, x);
        const at::Tensor ws = bytes(need > 0 ? need : 1, x);
        return ntg_conv2d_dev(dt, x.data_ptr(), w.data_ptr(), y.data_ptr(), ws.data_ptr(), need, g.B, g.C, t.h, t.w, g.O, t.kr, t.kc, t.sr, t.sc, t.pr, t.pc,
                              t.dr, t.dc, g.groups, stream);
    }
    const int64_t need = ntg_convnd_fast_workspace_bytes(dt, g.B, g.C, g.O, g.nd, g.size, g.k, g.s, g.p, g.d, g.groups, 0);
    if (need < 0) return NOT_TAKEN;
    y = fresh(size, x);
    const at::Tensor ws = bytes(need > 0 ? need : 1, x);
    return ntg_convnd_dev(dt, x.data_ptr(), w.data_ptr(), y.data_ptr(), ws.data_ptr(), need, g.B, g.C, g.O, g.nd, g.size, g.k, g.s, g.p, g.d, g.groups, stream);
}
// (dx is computed where want_dx; both are allocated here)
int gradients(const Geometry& g, int dt, const at::Tensor& x, const at::Tensor& w, const at::Tensor& dy, bool want_dx, at::Tensor& dx, at::Tensor& dw, void* stream) {
    const Two t = two(g);
    const int64_t need = g.nd < 3 ? ntg_conv2d_backward_workspace_bytes(dt, g.B, g.C, t.h, t.w, g.O, t.kr, t.kc, t.sr, t.sc, t.pr, t.pc, t.dr, t.dc, g.groups)
                                  : ntg_convnd_fast_workspace_bytes(dt, g.B, g.C, g.O, g.nd, g.size, g.k, g.s, g.p, g.d, g.groups, 1);
    if (need < 0) return NOT_TAKEN;
    if (want_dx) dx = fresh(x.sizes(), x);
    dw = fresh(w.sizes(), w);
    const at::Tensor ws = bytes(need > 0 ? need : 1, x);
    void* dxp = want_dx ? dx.data_ptr() : nullptr;
    if (g.nd < 3)
        return ntg_conv2d_backward_dev(dt, x.data_ptr(), w.data_ptr(), dy.data_ptr(), dxp, dw.data_ptr(), ws.data_ptr(), need, g.B, g.C, t.h, t.w, g.O, t.kr, t.kc,
                                       t.sr, t.sc, t.pr, t.pc, t.dr, t.dc, g.groups, 0, stream);
    return ntg_convnd_backward_dev(dt, x.data_ptr(), w.data_ptr(), dy.data_ptr(), dxp, dw.data_ptr(), ws.data_ptr(), need, g.B, g.C, g.O, g.nd, g.size, g.k, g.s,
                                   g.p, g.d, g.groups, 0, stream);
}

bool axes(PyObject* o, int& nd) {
    int64_t v;
    if (!whole(o, v) || v < 1 || v > 3) return false;
    nd = (int)v;
    return true;
}

// conv(axes, image, kernel, stride, padding, dilation, groups, stream)
PyObject* conv(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    Geometry g;
    int64_t stream;
    if (n_args != 8 || modes_active() || !axes(args[0], g.nd)) Py_RETURN_NONE;
    const at::Tensor *x = dense(args[1], g.nd), *w = dense(args[2], g.nd);
    if (!x || !w || x->scalar_type() != w->scalar_type() || !options(g, args[3], args[4], args[5], args[6]) || !whole(args[7], stream) ||
        !shapes(g, x->sizes(), w->sizes())) Py_RETURN_NONE;
    const int dt = ntg_dtype(x->scalar_type());
    if (dt < 0) Py_RETURN_NONE;
    at::Tensor y;
    int status;
    {
        NoGil unlocked;
        status = forward(g, dt, *x, *w, y, reinterpret_cast<void*>(stream));
    }
    if (status == NOT_TAKEN) Py_RETURN_NONE;
    if (status) return PyLong_FromLong(status);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

PyObject* pair(at::Tensor&& a, at::Tensor&& b) {
    PyObject* pa = THPVariable_Wrap(std::move(a));
    PyObject* pb = THPVariable_Wrap(std::move(b));
    PyObject* t = pa && pb ? PyTuple_Pack(2, pa, pb) : nullptr;
    Py_XDECREF(pa);
    Py_XDECREF(pb);
    return t;
}

// conv_backward(axes, image, kernel, grad, stride, padding, dilation, groups, stream)
PyObject* conv_backward(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    Geometry g;
    int64_t stream;
    if (n_args != 9 || modes_active() || !axes(args[0], g.nd)) Py_RETURN_NONE;
    const at::Tensor *x = dense(args[1], g.nd), *w = dense(args[2], g.nd), *dy = plain(args[3]);
    if (!x || !w || !dy || !dy->is_contiguous() || x->scalar_type() != w->scalar_type() || x->scalar_type() != dy->scalar_type() ||
        !options(g, args[4], args[5], args[6], args[7]) || !whole(args[8], stream) || !shapes(g, x->sizes(), w->sizes())) Py_RETURN_NONE;
    int64_t numel = g.B;
    bool wraps = __builtin_mul_overflow(numel, g.O, &numel);
    for (int a = 0; a < g.nd; ++a) wraps |= __builtin_mul_overflow(numel, g.out[a], &numel);
    const int dt = ntg_dtype(x->scalar_type());
    if (dt < 0 || wraps || dy->numel() != numel) Py_RETURN_NONE;
    at::Tensor dx, dw;
    int status;
    {
        NoGil unlocked;
        status = gradients(g, dt, *x, *w, *dy, true, dx, dw, reinterpret_cast<void*>(stream));
    }
    if (status == NOT_TAKEN) Py_RETURN_NONE;
    if (status) return PyLong_FromLong(status);
    return pair(std::move(dx), std::move(dw));
    END_HANDLE_TH_ERRORS
}

// conv_transpose(axes, image, kernel [Cin][Cout / groups][k], stride, padding, output_padding, dilation, groups, stream)
PyObject* conv_transpose(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    Geometry g;
    int64_t stream, op[3];
    if (n_args != 9 || modes_active() || !axes(args[0], g.nd)) Py_RETURN_NONE;
    const at::Tensor *x = dense(args[1], g.nd), *w = dense(args[2], g.nd);
    if (!x || !w || x->scalar_type() != w->scalar_type() || !options(g, args[3], args[4], args[6], args[7]) || !per_axis(args[5], g.nd, op) ||
        !whole(args[8], stream)) Py_RETURN_NONE;
    const int dt = ntg_dtype(x->scalar_type());
    g.B = x->size(0); g.C = x->size(1);
    if (dt < 0 || g.B < 1 || g.C < 1 || w->size(1) < 1 || w->size(0) != g.C || g.C % g.groups != 0) Py_RETURN_NONE;
    g.O = w->size(1) * g.groups;                                   // (at most the kernel's elements: groups <= its first size)
    c10::SmallVector<int64_t, 5> size = {g.B, g.O};
    for (int a = 0; a < g.nd; ++a) {
        g.size[a] = x->size(2 + a); g.k[a] = w->size(2 + a);
        if (g.size[a] >= LARGE || g.k[a] >= LARGE || op[a] >= LARGE) Py_RETURN_NONE;
        const int64_t out = (g.size[a] - 1) * g.s[a] - 2 * g.p[a] + g.d[a] * (g.k[a] - 1) + 1 + op[a];
        if (g.size[a] < 1 || g.k[a] < 1 || op[a] < 0 || out < 1) Py_RETURN_NONE;
        size.push_back(out);
    }
    const Two t = two(g);
    const int64_t or_ = g.nd == 1 ? 0 : op[0], oc = op[g.nd - 1];
    at::Tensor y;
    int status;
    {
        NoGil unlocked;
        const int64_t need = g.nd < 3 ? ntg_conv_transpose2d_workspace_bytes(dt, g.B, g.C, t.h, t.w, g.O, t.kr, t.kc, t.sr, t.sc, t.pr, t.pc, t.dr, t.dc, or_, oc, g.groups)
                                      : ntg_conv_transposend_workspace_bytes(dt, g.B, g.C, g.O, g.nd, g.size, g.k, g.s, g.p, g.d, op, g.groups);
        if (need < 0) status = NOT_TAKEN;
        else {
            y = fresh(size, *x);
            const at::Tensor ws = bytes(need > 0 ? need : 1, *x);
            status = g.nd < 3 ? ntg_conv_transpose2d_dev(dt, x->data_ptr(), w->data_ptr(), y.data_ptr(), ws.data_ptr(), need, g.B, g.C, t.h, t.w, g.O, t.kr, t.kc, t.sr,
                                                         t.sc, t.pr, t.pc, t.dr, t.dc, or_, oc, g.groups, reinterpret_cast<void*>(stream))
                              : ntg_conv_transposend_dev(dt, x->data_ptr(), w->data_ptr(), y.data_ptr(), ws.data_ptr(), need, g.B, g.C, g.O, g.nd, g.size, g.k, g.s, g.p,
                                                         g.d, op, g.groups, reinterpret_cast<void*>(stream));
        }
    }
    if (status == NOT_TAKEN) Py_RETURN_NONE;
    if (status) return PyLong_FromLong(status);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// conv_transpose_backward(axes, image, kernel, grad, stride, padding, dilation, groups, stream): d_image = conv(grad, kernel), d_kernel = the weight gradient of
// that convolution with image and output gradient exchanged
PyObject* conv_transpose_backward(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    Geometry g;
    int64_t stream;
    if (n_args != 9 || modes_active() || !axes(args[0], g.nd)) Py_RETURN_NONE;
    const at::Tensor *x = dense(args[1], g.nd), *w = dense(args[2], g.nd), *dy = dense(args[3], g.nd);
    if (!x || !w || !dy || x->scalar_type() != w->scalar_type() || x->scalar_type() != dy->scalar_type() || !options(g, args[4], args[5], args[6], args[7]) ||
        !whole(args[8], stream) || !shapes(g, dy->sizes(), w->sizes()) || x->size(0) != g.B || x->size(1) != g.O) Py_RETURN_NONE;
    for (int a = 0; a < g.nd; ++a)
        if (x->size(2 + a) != g.out[a]) Py_RETURN_NONE;
    const int dt = ntg_dtype(x->scalar_type());
    if (dt < 0) Py_RETURN_NONE;
    at::Tensor dx, dw, none;
    int status;
    {
        NoGil unlocked;
        status = forward(g, dt, *dy, *w, dx, reinterpret_cast<void*>(stream));
        if (status == 0) status = gradients(g, dt, *dy, *w, *x, false, none, dw, reinterpret_cast<void*>(stream));
    }
    if (status == NOT_TAKEN) Py_RETURN_NONE;
    if (status) return PyLong_FromLong(status);
    return pair(std::move(dx), std::move(dw));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"gemm", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(gemm)), METH_FASTCALL, nullptr},
    {"conv", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(conv)), METH_FASTCALL, nullptr},
    {"conv_backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(conv_backward)), METH_FASTCALL, nullptr},
    {"conv_transpose", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(conv_transpose)), METH_FASTCALL, nullptr},
    {"conv_transpose_backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(conv_transpose_backward)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_face", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__face() { return PyModule_Create(&module); }
