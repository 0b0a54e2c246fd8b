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

// factor tensors (an iterable of them), patterns (tuple of 4-tuples) and scales (list of floats)
bool read_layer(PyObject *params, PyObject *patterns, PyObject *scales, const at::Device &dev, Layer *l)
{
    if (!PyList_Check(params) || !PyList_Check(patterns) || !PyList_Check(scales)) return false;
    const Py_ssize_t n = PyList_GET_SIZE(params);
    if (n < 1 || n > KSMM_MAX_FACTORS || PyList_GET_SIZE(patterns) != n || PyList_GET_SIZE(scales) != n) return false;
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
        const double s = PyFloat_AsDouble(PyList_GET_ITEM(scales, i));
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
    const int64_t need = quantise ? ksmm_chain_quant_workspace(l.f, l.n, batch, xd, yd, bs_last)
                                  : ksmm_chain_workspace_layout(l.f, l.n, batch, xd, yd, bs_last);
    if (need < 0) return (int)need;
    *y = at::empty(shape, x.options().dtype(out_type));
    at::Tensor ws;
    if (need > 0) ws = at::empty({need}, x.options().dtype(at::kByte));
    const auto run = quantise ? ksmm_chain_forward_quant : ksmm_chain_forward_ep;
    return run(l.f, l.n, x.const_data_ptr(), y->mutable_data_ptr(), need > 0 ? ws.mutable_data_ptr() : nullptr, need, batch, xd, yd,
               bs_last, fuse, ep.bias || ep.act ? &ep : nullptr, c10::hip::getCurrentHIPStream(x.device().index()).stream());
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

PyMethodDef methods[] = {
    {"infer", (PyCFunction)(void (*)(void))py_infer, METH_FASTCALL, "one layer without gradients"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
