// CPython module ksmm_amd._native: the host side of KSLinear(algo='kernel') as one call.
//
// A layer on a small batch is done on the GPU in 5 to 15 us; the same call through Python checks,
// ctypes structures and torch.empty() took 20 to 30 us of host time.  Here the checks, the
// descriptors, the output and workspace tensors and the launch cost about 3 us.  Nothing is
// remembered between calls: pointers, sizes and types are read from the tensors each time.
//
// Every entry returns None when it does not take a call (an unusual argument, an error of the
// library, no memory): the caller then goes through ksmm_amd/kernel.py, which raises what is wrong
// with it.  The GIL is released from the first allocation on: both that and a launch can wait.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/ksmm_hip.h"

namespace {

int code_of(at::ScalarType t)
{
    switch (t) {
    case at::kFloat: return KSMM_F32;
    case at::kHalf: return KSMM_F16;
    case at::kFloat8_e4m3fn: return KSMM_FP8_E4M3;
    default: return -1;
    }
}

// makes a device current for the life of the object
struct DeviceScope {
    c10::DeviceIndex before = -1;
    explicit DeviceScope(c10::DeviceIndex want)
    {
        const c10::DeviceIndex now = c10::hip::current_device();
        if (now != want) {
            before = now;
            c10::hip::set_device(want);
        }
    }
    ~DeviceScope()
    {
        if (before >= 0) c10::hip::set_device(before);
    }
};

struct WithoutGil {
    PyThreadState *state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

struct Layer {
    ksmm_factor_desc f[KSMM_MAX_FACTORS];
    int n = 0;
    int64_t in_size = 0, out_size = 0;
};

// factor tensors, patterns (4-tuples) and scales (floats), lists of them; scales may be null: 1 each
bool read_layer(PyObject *params, PyObject *patterns, PyObject *scales, const at::Device &dev, Layer *l)
{
    if (!PyList_Check(params) || !PyList_Check(patterns) || (scales && !PyList_Check(scales))) return false;
    const Py_ssize_t n = PyList_GET_SIZE(params);
    if (n < 1 || n > KSMM_MAX_FACTORS || PyList_GET_SIZE(patterns) != n || (scales && PyList_GET_SIZE(scales) != n)) return false;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject *w = PyList_GET_ITEM(params, i), *p = PyList_GET_ITEM(patterns, i);
        if (!THPVariable_Check(w) || !PyTuple_Check(p) || PyTuple_GET_SIZE(p) != 4) return false;
        const at::Tensor &t = THPVariable_Unpack(w);
        int64_t v[4];
        for (int k = 0; k < 4; ++k) {
            v[k] = PyLong_AsLongLong(PyTuple_GET_ITEM(p, k));
            if (v[k] < 1 || v[k] > 0x7fffffff) return false;
        }
        ksmm_factor_desc &f = l->f[i];
        f.a = (int)v[0];
        f.b = (int)v[1];
        f.c = (int)v[2];
        f.d = (int)v[3];
        f.w_dtype = code_of(t.scalar_type());
        const double s = scales ? PyFloat_AsDouble(PyList_GET_ITEM(scales, i)) : 1.0;
        if (s == -1.0 && PyErr_Occurred()) return false;
        f.scale = (float)s;
        if (f.w_dtype < 0 || t.device() != dev || !t.is_contiguous() || t.dim() != 2 || t.size(0) != v[0] * v[2] * v[3] ||
            t.size(1) != v[1])
            return false;
        f.w = t.const_data_ptr();
        if (i == 0) l->in_size = v[0] * v[2] * v[3];
        l->out_size = v[0] * v[1] * v[3];
    }
    l->n = (int)n;
    return true;
}

// Shape of the result of a layer on x (batch-size-last: features first): false when x does not fit.
bool result_shape(const at::Tensor &x, bool bs_last, const Layer &l, int64_t *batch, c10::SmallVector<int64_t, 6> *shape)
{
    if (x.dim() < 1 || !x.is_contiguous() || x.numel() == 0) return false;
    const int64_t axis = bs_last ? 0 : x.dim() - 1;
    if (x.size(axis) != l.in_size) return false;
    shape->assign(x.sizes().begin(), x.sizes().end());
    (*shape)[axis] = l.out_size;
    if (bs_last && x.dim() == 1) shape->resize(1);
    *batch = x.numel() / l.in_size;
    return true;
}

// bias (None or a tensor) and activation (None or "gelu"); false: leave the call to Python
bool read_epilogue(PyObject *bias, PyObject *act, const at::Device &dev, at::ScalarType out, int64_t out_size, ksmm_epilogue *ep)
{
    ep->bias = nullptr;
    ep->act = KSMM_ACT_NONE;
    if (bias != Py_None) {
        if (!THPVariable_Check(bias)) return false;
        const at::Tensor &t = THPVariable_Unpack(bias);
        if (t.device() != dev || t.scalar_type() != out || !t.is_contiguous() || t.numel() != out_size) return false;
        ep->bias = t.const_data_ptr();
    }
    if (act != Py_None) {
        if (!PyUnicode_Check(act) || PyUnicode_CompareWithASCIIString(act, "gelu") != 0) return false;
        ep->act = KSMM_ACT_GELU;
    }
    return true;
}

// The whole layer without gradients: y = act(scale K_n .. K_1 x + bias), or KSMM error < 0.  quantise:
// x goes through e4m3 codes and a scale that the call finds itself.
int forward(const at::Tensor &x, const Layer &l, int64_t batch, const c10::SmallVector<int64_t, 6> &shape, bool bs_last,
            bool fuse, bool quantise, const ksmm_epilogue &ep, at::ScalarType out_type, at::Tensor *y)
{
    const int xd = code_of(x.scalar_type()), yd = code_of(out_type);
    void *const stream = c10::hip::getCurrentHIPStream(x.device().index()).stream();
    const ksmm_epilogue *const epilogue = ep.bias || ep.act ? &ep : nullptr;
    // chains of one launch need no workspace (1.7 us); they are of 16 x 16 blocks, or of two factors on small batches (asking
    // costs the others 0.4 us)
    if (fuse && !quantise && l.n > 1 && ((l.f[0].b == 16 && l.f[0].c == 16) || (l.n == 2 && l.f[0].d == 1 && batch <= 4096))) {
        at::Tensor out = at::empty(shape, x.options().dtype(out_type));
        const int rc = ksmm_chain_forward_fused(l.f, l.n, x.const_data_ptr(), out.mutable_data_ptr(), batch, xd, yd, bs_last, epilogue, stream);
        *y = std::move(out);
        if (rc != KSMM_ERR_BAD_ALGO) return rc;
    }
    const int64_t need = quantise ? ksmm_chain_quant_workspace(l.f, l.n, batch, xd, yd, bs_last)
                                  : ksmm_chain_workspace_layout(l.f, l.n, batch, xd, yd, bs_last);
    if (need < 0) return (int)need;
    if (!y->defined()) *y = at::empty(shape, x.options().dtype(out_type));
    at::Tensor ws;
    if (need > 0) ws = at::empty({need}, x.options().dtype(at::kByte));
    const auto run = quantise ? ksmm_chain_forward_quant : ksmm_chain_forward_ep;
    return run(l.f, l.n, x.const_data_ptr(), y->mutable_data_ptr(), need > 0 ? ws.mutable_data_ptr() : nullptr, need, batch, xd, yd,
               bs_last, fuse, epilogue, stream);
}

// infer(x, factors, patterns, bs_last, scales, fuse, bias, act, quantise) -> y or None
PyObject *py_infer(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (n != 9) {
        PyErr_SetString(PyExc_TypeError, "infer() takes 9 arguments");
        return nullptr;
    }
    try {
        if (!THPVariable_Check(args[0])) Py_RETURN_NONE;
        const at::Tensor &x = THPVariable_Unpack(args[0]);
        if (!x.is_cuda()) Py_RETURN_NONE;
        const bool bs_last = PyObject_IsTrue(args[3]) == 1, fuse = PyObject_IsTrue(args[5]) == 1, quantise = PyObject_IsTrue(args[8]) == 1;
        Layer l;
        int64_t batch;
        c10::SmallVector<int64_t, 6> shape;
        ksmm_epilogue ep;
        const bool taken = read_layer(args[1], args[2], args[4], x.device(), &l) && result_shape(x, bs_last, l, &batch, &shape);
        if (taken && code_of(x.scalar_type()) >= 0) {
            bool fp8 = false;
            for (int i = 0; i < l.n; ++i) fp8 |= l.f[i].w_dtype == KSMM_FP8_E4M3;
            const at::ScalarType out = fp8 ? at::kHalf : x.scalar_type();
            if (read_epilogue(args[6], args[7], x.device(), out, l.out_size, &ep)) {
                at::Tensor y;
                int status;
                {
                    WithoutGil released;
                    DeviceScope scope(x.device().index());
                    status = forward(x, l, batch, shape, bs_last, fuse, quantise, ep, out, &y);
                }
                if (status == KSMM_OK) return THPVariable_Wrap(std::move(y));
            }
        }
    } catch (const std::exception &) {
    }
    PyErr_Clear();
    Py_RETURN_NONE;
}

bool trainable(at::ScalarType t) { return t == at::kFloat || t == at::kHalf; }

// every factor of type t and in line with its neighbours (a chain's own check comes too late for the intermediates' sizes)
bool of_type(const Layer &l, at::ScalarType t)
{
    for (int i = 0; i < l.n; ++i) {
        if (l.f[i].w_dtype != code_of(t)) return false;
        if (i > 0 && (int64_t)l.f[i].a * l.f[i].c * l.f[i].d != (int64_t)l.f[i - 1].a * l.f[i - 1].b * l.f[i - 1].d) return false;
    }
    return true;
}

PyObject *wrapped(const at::Tensor &t)
{
    if (t.defined()) return THPVariable_Wrap(t);
    Py_RETURN_NONE;
}

// train_forward(x, factors, patterns, bs_last, bias, act) -> (y, what each factor but the first was applied to.., z) or
// None; z is what the activation was applied to (None without one).
PyObject *py_train_forward(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    if (n_args != 6) {
        PyErr_SetString(PyExc_TypeError, "train_forward() takes 6 arguments");
        return nullptr;
    }
    try {
        if (!THPVariable_Check(args[0])) Py_RETURN_NONE;
        const at::Tensor &x = THPVariable_Unpack(args[0]);
        const bool bs_last = PyObject_IsTrue(args[3]) == 1;
        Layer l;
        int64_t batch;
        c10::SmallVector<int64_t, 6> shape;
        ksmm_epilogue ep;
        if (x.is_cuda() && x.dim() == 2 && trainable(x.scalar_type()) && read_layer(args[1], args[2], nullptr, x.device(), &l) &&
            of_type(l, x.scalar_type()) && result_shape(x, bs_last, l, &batch, &shape) &&
            read_epilogue(args[4], args[5], x.device(), x.scalar_type(), l.out_size, &ep)) {
            const int dt = code_of(x.scalar_type());
            at::Tensor out[KSMM_MAX_FACTORS], y;
            int status = KSMM_OK;
            {
                WithoutGil released;
                DeviceScope scope(x.device().index());
                void *const stream = c10::hip::getCurrentHIPStream(x.device().index()).stream();
                const ksmm_epilogue bias_only{ep.bias, KSMM_ACT_NONE};
                const void *in = x.const_data_ptr();
                for (int i = 0; i < l.n && status == KSMM_OK; ++i) {
                    const ksmm_factor_desc &f = l.f[i];
                    const int64_t size = (int64_t)f.a * f.b * f.d;
                    const int64_t need = ksmm_factor_workspace(batch, f.a, f.b, f.c, f.d, dt, dt, dt, bs_last);
                    if (need < 0) {
                        status = (int)need;
                        break;
                    }
                    out[i] = at::empty({bs_last ? size : batch, bs_last ? batch : size}, x.options());
                    at::Tensor ws;
                    if (need > 0) ws = at::empty({need}, x.options().dtype(at::kByte));
                    status = ksmm_factor_forward_ep(in, f.w, out[i].mutable_data_ptr(), batch, f.a, f.b, f.c, f.d, dt, dt, dt, bs_last, 1.f,
                                                    i + 1 == l.n && ep.bias ? &bias_only : nullptr,
                                                    need > 0 ? ws.mutable_data_ptr() : nullptr, need, stream);
                    in = out[i].const_data_ptr();
                }
                if (status == KSMM_OK) y = ep.act ? at::gelu(out[l.n - 1]) : out[l.n - 1];
            }
            if (status == KSMM_OK) {
                PyObject *r = PyTuple_New(l.n + 1);
                if (!r) return nullptr;
                PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(y));
                for (int i = 0; i + 1 < l.n; ++i) PyTuple_SET_ITEM(r, i + 1, THPVariable_Wrap(out[i]));
                PyTuple_SET_ITEM(r, l.n, wrapped(ep.act ? out[l.n - 1] : at::Tensor()));
                return r;
            }
        }
    } catch (const std::exception &) {
    }
    PyErr_Clear();
    Py_RETURN_NONE;
}

// train_backward(grad, factors, patterns, inputs, z, bs_last, act, need_x, need_bias, need_factors) -> (grad_x, grad_bias, [grad_factors])
// or None; lists but for grad, z (None without an activation) and need_factors (a tuple).  What is not needed is None.
PyObject *py_train_backward(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    if (n_args != 10) {
        PyErr_SetString(PyExc_TypeError, "train_backward() takes 10 arguments");
        return nullptr;
    }
    try {
        if (!THPVariable_Check(args[0])) Py_RETURN_NONE;
        const at::Tensor &grad = THPVariable_Unpack(args[0]);
        const bool bs_last = PyObject_IsTrue(args[5]) == 1, need_x = PyObject_IsTrue(args[7]) == 1, need_bias = PyObject_IsTrue(args[8]) == 1;
        Layer l;
        ksmm_epilogue ep;
        bool taken = grad.is_cuda() && grad.dim() == 2 && grad.is_contiguous() && grad.numel() > 0 && trainable(grad.scalar_type()) &&
                     read_layer(args[1], args[2], nullptr, grad.device(), &l) && of_type(l, grad.scalar_type()) &&
                     read_epilogue(Py_None, args[6], grad.device(), grad.scalar_type(), l.out_size, &ep) &&
                     grad.size(bs_last ? 0 : 1) == l.out_size && PyList_Check(args[3]) && PyList_GET_SIZE(args[3]) == l.n &&
                     PyTuple_Check(args[9]) && PyTuple_GET_SIZE(args[9]) == l.n;
        const int64_t batch = taken ? grad.size(bs_last ? 1 : 0) : 0;
        const void *inputs[KSMM_MAX_FACTORS], *z = nullptr;
        bool need[KSMM_MAX_FACTORS];
        // a tensor of the pass: the gradient's type, as many features as factor i takes (i == n: as the layer gives)
        auto fits = [&](PyObject *o, int i, const void **p) {
            if (!THPVariable_Check(o)) return false;
            const at::Tensor &t = THPVariable_Unpack(o);
            const int64_t size = i == l.n ? l.out_size : (int64_t)l.f[i].a * l.f[i].c * l.f[i].d;
            *p = t.scalar_type() == grad.scalar_type() && t.device() == grad.device() && t.dim() == 2 && t.is_contiguous() &&
                         t.size(bs_last ? 0 : 1) == size && t.size(bs_last ? 1 : 0) == batch
                     ? t.const_data_ptr() : nullptr;
            return *p != nullptr;
        };
        for (int i = 0; taken && i < l.n; ++i) {
            need[i] = PyObject_IsTrue(PyTuple_GET_ITEM(args[9], i)) == 1;
            taken = fits(PyList_GET_ITEM(args[3], i), i, &inputs[i]);
        }
        if (taken && ep.act) taken = fits(args[4], l.n, &z);
        if (taken) {
            const int dt = code_of(grad.scalar_type());
            at::Tensor dx, dbias, dw[KSMM_MAX_FACTORS];
            int status;
            {
                WithoutGil released;
                DeviceScope scope(grad.device().index());
                const int64_t bytes = ksmm_layer_backward_workspace(l.f, l.n, batch, dt, bs_last, ep.act);
                status = bytes < 0 ? (int)bytes : KSMM_OK;
                if (status == KSMM_OK) {
                    const auto opts = grad.options();
                    void *to[KSMM_MAX_FACTORS];
                    if (need_x) dx = at::empty({bs_last ? l.in_size : batch, bs_last ? batch : l.in_size}, opts);
                    if (need_bias) dbias = bs_last ? at::empty({l.out_size, 1}, opts) : at::empty({l.out_size}, opts);
                    for (int i = 0; i < l.n; ++i) {
                        if (need[i]) dw[i] = at::empty({(int64_t)l.f[i].a * l.f[i].c * l.f[i].d, l.f[i].b}, opts);
                        to[i] = need[i] ? dw[i].mutable_data_ptr() : nullptr;
                    }
                    const at::Tensor ws = at::empty({bytes}, opts.dtype(at::kByte));
                    status = ksmm_layer_backward(l.f, l.n, inputs, z, grad.const_data_ptr(), need_x ? dx.mutable_data_ptr() : nullptr, to,
                                                 need_bias ? dbias.mutable_data_ptr() : nullptr, ws.mutable_data_ptr(), bytes, batch, dt,
                                                 bs_last, ep.act, c10::hip::getCurrentHIPStream(grad.device().index()).stream());
                }
            }
            if (status == KSMM_OK) {
                PyObject *ws = PyList_New(l.n);
                if (!ws) return nullptr;
                for (int i = 0; i < l.n; ++i) PyList_SET_ITEM(ws, i, wrapped(dw[i]));
                return Py_BuildValue("(NNN)", wrapped(dx), wrapped(dbias), ws);
            }
        }
    } catch (const std::exception &) {
    }
    PyErr_Clear();
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"train_forward", (PyCFunction)(void (*)(void))py_train_forward, METH_FASTCALL, "one layer, its intermediates kept"},
    {"train_backward", (PyCFunction)(void (*)(void))py_train_backward, METH_FASTCALL, "gradients of one layer"},
    {"infer", (PyCFunction)(void (*)(void))py_infer, METH_FASTCALL, "one layer without gradients"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
