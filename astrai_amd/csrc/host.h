// Shared by host.cpp and host_mix.cpp: arguments of the native calls, torch's stream, outputs.
#pragma once

#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

namespace {

using at::Tensor;

// The argument's tensor, or null (None, another type, a subclass). None is one under torch.jit.trace, which would record the
// outputs' allocation and not what is written into them.
const Tensor* tensor_of(PyObject* o) {
    return THPVariable_CheckExact(o) && !torch::jit::tracer::isTracing() ? &THPVariable_Unpack(o) : nullptr;
}

// an optional tensor: false if the argument is something else
bool optional(PyObject* o, const Tensor*& t) {
    t = tensor_of(o);
    return t || o == Py_None;
}

bool whole(PyObject* o, int64_t& v) {
    int over = 1;
    v = PyLong_Check(o) ? PyLong_AsLongLongAndOverflow(o, &over) : 0;
    return !over;
}

bool real(PyObject* o, double& v) {
    int64_t i;
    if (PyFloat_Check(o)) v = PyFloat_AS_DOUBLE(o);
    else if (whole(o, i)) v = (double)i;
    else return false;
    return true;
}

bool plain(const Tensor& t, c10::ScalarType type, c10::Device dev) {
    return t.scalar_type() == type && t.device() == dev && t.is_contiguous();
}

bool plain16(const Tensor& t, c10::ScalarType type, c10::Device dev) {
    return plain(t, type, dev) && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

void* stream_of(c10::Device dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

void* ptr(const Tensor* t) { return t ? t->data_ptr() : nullptr; }

// [..., n] from x [..., k]
Tensor output(const Tensor& x, int64_t n, c10::ScalarType type) {
    c10::SmallVector<int64_t, 5> sizes(x.sizes().begin(), x.sizes().end());
    sizes.back() = n;
    return at::empty(sizes, x.options().dtype(type).requires_grad(false));
}

// (other threads run while a launch waits for room in its queue)
template <class F>
int unlocked(F call) {
    struct Unlock {
        PyThreadState* const state = PyEval_SaveThread();
        ~Unlock() { PyEval_RestoreThread(state); }
    } unlock;
    return call();
}

// What this was built for, which the loader compares: the calls' arguments, the library's header, torch, Python.
#define ASTRAI_HOST_CALLS_VERSION 1
PyObject* with_built_for(PyObject* module, int abi_version) {
    PyObject* const what = module ? Py_BuildValue("(iiss)", ASTRAI_HOST_CALLS_VERSION, abi_version, ASTRAI_TORCH_VERSION,
                                                  ASTRAI_PYTHON_VERSION) : nullptr;
    if (what && PyModule_AddObject(module, "BUILT_FOR", what) == 0) return module;
    Py_XDECREF(what);
    Py_XDECREF(module);
    return nullptr;
}

#define ENTRY(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&name)), METH_FASTCALL, nullptr}

}  // namespace
