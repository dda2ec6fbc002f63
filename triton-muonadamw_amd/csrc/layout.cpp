// CPython module triton_muon_adamw._layout: what a cached launch plan assumes
// of the parameters and their gradients, read from the tensors natively.
//
// An optimizer step compares this with the plan's before it launches anything:
// addresses, element types, sizes and strides of every parameter that has a
// gradient and of the gradient.  In Python that is nine attribute reads, 0.5 us
// a parameter: more than the step itself for a set of small tensors (200 of
// them: 109 us a step, 93 of it this).
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/version.h>

#include <string>

namespace {

void put(std::string& s, int64_t v) { s.append(reinterpret_cast<const char*>(&v), sizeof(v)); }

void put_tensor(std::string& s, const at::Tensor& t) {
    put(s, reinterpret_cast<int64_t>(t.data_ptr()));
    put(s, (int64_t(t.scalar_type()) << 32) | t.dim());
    for (const int64_t n : t.sizes()) put(s, n);
    for (const int64_t n : t.strides()) put(s, n);
}

// layout(params) -> (active, key): the entries of the list that have a
// gradient, and their layouts as bytes.  None when an entry or its gradient is
// neither a plain Tensor nor a plain Parameter (a subclass may define its own
// attributes).
PyObject* layout(PyObject*, PyObject* params) {
    HANDLE_TH_ERRORS
    if (!PyList_CheckExact(params)) Py_RETURN_NONE;
    const Py_ssize_t n = PyList_GET_SIZE(params);
    THPObjectPtr active(PyList_New(0));
    if (!active) return nullptr;
    std::string key;
    key.reserve(size_t(n) * 112);
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(params); ++i) {
        PyObject* p = PyList_GET_ITEM(params, i);
        if (!THPVariable_CheckExact(p)) Py_RETURN_NONE;
        const at::Tensor& t = THPVariable_Unpack(p);
        const at::Tensor g = t.grad();
        if (!g.defined()) continue;
        THPObjectPtr gradient(THPVariable_Wrap(g));
        if (!gradient) return nullptr;
        if (!THPVariable_CheckExact(gradient.get())) Py_RETURN_NONE;
        if (PyList_Append(active.get(), p) != 0) return nullptr;
        put(key, reinterpret_cast<int64_t>(p));
        put_tensor(key, t);
        put_tensor(key, g);
    }
    THPObjectPtr bytes(PyBytes_FromStringAndSize(key.data(), Py_ssize_t(key.size())));
    if (!bytes) return nullptr;
    return PyTuple_Pack(2, active.get(), bytes.get());
    END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"layout", layout, METH_O, "layout(params) -> (parameters with a gradient, their layouts) or None"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_layout", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__layout() {
    THPObjectPtr m(PyModule_Create(&kModule));
    if (!m || PyModule_AddStringConstant(m.get(), "torch_version", TORCH_VERSION) != 0) return nullptr;
    return m.release();
}
