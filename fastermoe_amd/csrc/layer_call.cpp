// Inference through the layer's call (fmoe_layer_forward), from Python's tensors to the enqueued kernels (host code).
//
// A decoding step is four kernels of 24 us in all.  Checking seven tensors, asking for the scratch block's size, allocating and
// converting the call's 31 arguments took Python 13 us of the 35 that it took to enqueue them, and so bounded the step; here that takes
// two.  What decides whether a layer may be called like this at all stays in Python.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/linear.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <cstdint>

#include "../../include/fmoe_hip.h"

namespace {

// the library's entry points, which Python has loaded (bind)
decltype(&fmoe_layer_sizes) layer_sizes = nullptr;
decltype(&fmoe_layer_forward) layer_forward = nullptr;

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return FMOE_F32;
        case at::kBFloat16: return FMOE_BF16;
        case at::kHalf: return FMOE_F16;
        default: return -1;
    }
}
bool on_16_bytes(const at::Tensor &t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }
void *pointer(const at::Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }

// The interpreter's lock, given back while this lives
struct WithoutLock {
    PyThreadState *state = PyEval_SaveThread();
    ~WithoutLock() { PyEval_RestoreThread(state); }
};

PyObject *bind(PyObject *, PyObject *args) {
    unsigned long long sizes, forward;
    if (!PyArg_ParseTuple(args, "KK", &sizes, &forward)) return nullptr;
    layer_sizes = reinterpret_cast<decltype(layer_sizes)>(static_cast<uintptr_t>(sizes));
    layer_forward = reinterpret_cast<decltype(layer_forward)>(static_cast<uintptr_t>(forward));
    Py_RETURN_NONE;
}

// infer(inp, gate_w, gate_b, score, pos, slot_to_row, table, w1, b1, w2, b2, top_k, activation, gate, stream): the output; None where
// the call does not take these tensors; a number, the library's status, where it failed.
constexpr Py_ssize_t kTensors = 11, kArgs = 15;
PyObject *infer(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != kArgs || layer_forward == nullptr) {
        PyErr_SetString(PyExc_TypeError, "infer: 15 arguments, after bind");
        return nullptr;
    }
    std::array<at::Tensor, kTensors> t;
    for (Py_ssize_t i = 0; i < kTensors; ++i) {
        if (args[i] == Py_None) continue;
        if (!THPVariable_Check(args[i])) {
            PyErr_SetString(PyExc_TypeError, "infer: tensors or None");
            return nullptr;
        }
        t[i] = THPVariable_Unpack(args[i]);
    }
    const auto &[given, gate_w, gate_b, score, pos, slot_to_row, table, w1, b1, w2, b2] = t;
    std::array<long long, kArgs - kTensors> number;
    for (size_t i = 0; i < number.size(); ++i) {
        number[i] = PyLong_AsLongLong(args[kTensors + i]);
        if (number[i] == -1 && PyErr_Occurred()) return nullptr;
    }
    const auto [top_k, activation, gate, stream] = number;

    if (!given.defined() || !w1.defined() || !w2.defined() || given.dim() != 2 || w1.dim() != 3 || !on_16_bytes(given)) Py_RETURN_NONE;
    const int dtype = dtype_code(given.scalar_type());
    if (dtype < 0) Py_RETURN_NONE;
    for (const at::Tensor *p : {&gate_w, &gate_b, &score, &w1, &b1, &w2, &b2})
        if (p->defined() && (p->scalar_type() != given.scalar_type() || p->device() != given.device() || !p->is_contiguous() || !on_16_bytes(*p)))
            Py_RETURN_NONE;
    const int64_t n = given.size(0), d = given.size(1), e = w1.size(0), h = w1.size(1);
    auto has = [](const at::Tensor &p, at::IntArrayRef sizes) { return !p.defined() || p.sizes() == sizes; };
    if (!has(w1, {e, h, d}) || !has(w2, {e, d, h}) || !has(b1, {e, h}) || !has(b2, {e, d}) || !has(gate_w, {e, d}) || !has(gate_b, {e})) Py_RETURN_NONE;
    int64_t sizes[3] = {};
    if (layer_sizes(n, d, h, e, top_k, dtype, (int)activation, 0, (int)gate, sizes) != 1) Py_RETURN_NONE;

    // Other threads of the interpreter go on from here, as they do in torch's own operators: an allocation may wait for the device, and the
    // library product of the logits, like the launches, for a full queue.
    at::Tensor out;
    int rc;
    {
        const WithoutLock no_lock;
        const at::Tensor inp = given.contiguous();
        const at::Tensor logits = gate == FMOE_GATE_LOGITS
                                      ? at::linear(inp, gate_w, gate_b.defined() ? std::optional<at::Tensor>(gate_b) : std::nullopt) : at::Tensor();
        const at::TensorOptions like = at::TensorOptions().dtype(inp.scalar_type()).device(inp.device());
        out = at::empty({n, d}, like);
        const at::Tensor scratch = at::empty({sizes[0]}, like.dtype(at::kByte));
        rc = layer_forward(pointer(inp), pointer(gate_w), pointer(gate_b), pointer(logits), pointer(w1), pointer(b1), pointer(w2), pointer(b2), nullptr,
                           pointer(score), (int64_t *)pointer(pos), (int64_t *)pointer(slot_to_row), pointer(table), nullptr, nullptr, nullptr,
                           pointer(out), n, d, h, e, top_k, dtype, (int)activation, 0, (int)gate, pointer(scratch), sizes[0],
                           reinterpret_cast<void *>(static_cast<uintptr_t>(stream)));
    }
    if (rc != FMOE_OK) return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "The addresses of fmoe_layer_sizes and fmoe_layer_forward."},
    {"infer", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(infer)), METH_FASTCALL, "A layer's output where nothing is differentiated."},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_layer_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__layer_call() {
    PyObject *m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddStringConstant(m, "built_for", FMOE_BUILT_FOR) < 0) Py_CLEAR(m);   // (torch's and Python's versions)
    return m;
}
