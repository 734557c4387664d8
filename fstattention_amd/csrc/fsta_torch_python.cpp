// The extension module `_fsta_torch`: the entry points of the package as plain C functions for calls that need nothing of
// torch's dispatcher (ordinary tensors on the GPU, no gradient, no mode that wants to see the call).  A call through the
// registered operator costs about 3 us of schema matching and boxing, and the lookup of the packed inputs another 1.5 us in
// Python; a launch of the smallest kernels takes less than that on the GPU.  Every function returns NotImplemented for a
// call it does not want to judge; the caller then takes the ordinary way, which also raises the errors.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/fsta.h"
#include "fsta_torch.h"

namespace {

PyObject* g_packed_type = nullptr;      // attention.PackedTreeMask
PyObject* g_packed_table = nullptr;     // attention._PACKED: id of a mask -> (weak reference, key, packed)

PyObject* not_implemented() { Py_RETURN_NOTIMPLEMENTED; }

// An ordinary torch.Tensor object (no subclass) in GPU memory
const at::Tensor* gpu_tensor(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has(c10::DispatchKey::Python) &&
                   !t.key_set().has(c10::DispatchKey::FuncTorchGradWrapper) && !t.key_set().has(c10::DispatchKey::FuncTorchBatched) &&
                   !t.is_conj() && !t.is_neg()
               ? &t
               : nullptr;
}

// Nobody has asked to see calls on tensors (modes, functorch, tracing)
bool plain_context() {
    const auto tls = c10::impl::tls_local_dispatch_key_set();
    return tls.included_ == c10::default_included_set && !at::impl::torch_function_mode_enabled();
}

bool wants_grad(const at::Tensor& t) { return t.requires_grad(); }

bool as_int(PyObject* o, int64_t* out) {
    if (!PyLong_Check(o)) return false;
    *out = PyLong_AsLongLong(o);
    if (*out == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

struct Packed {
    const at::Tensor *bits, *count, *plan;     // plan may be null
    int64_t block_m, max_ancestors, key_shift, key_limit;
    bool has_limit;
};

bool read_packed(PyObject* o, Packed* p) {
    if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != 7) return false;
    p->bits = gpu_tensor(PyTuple_GET_ITEM(o, 0));
    p->count = gpu_tensor(PyTuple_GET_ITEM(o, 1));
    PyObject* plan = PyTuple_GET_ITEM(o, 4);
    p->plan = plan == Py_None ? nullptr : gpu_tensor(plan);
    PyObject* limit = PyTuple_GET_ITEM(o, 6);
    p->has_limit = limit != Py_None;
    return p->bits && p->count && (plan == Py_None || p->plan) && as_int(PyTuple_GET_ITEM(o, 2), &p->block_m) &&
           as_int(PyTuple_GET_ITEM(o, 3), &p->max_ancestors) && as_int(PyTuple_GET_ITEM(o, 5), &p->key_shift) &&
           (!p->has_limit || as_int(limit, &p->key_limit));
}

// The packed form remembered for the bool tensor `mask`, if it is the one of these three tensors as they are now
// (attention.recall_packed and attention._cache_key, read from C); a borrowed reference or null.
PyObject* recall(PyObject* mask_obj, const at::Tensor& mask, const at::Tensor& a_idx, const at::Tensor& l_idx) {
    if (mask.is_inference() || a_idx.is_inference() || l_idx.is_inference()) return nullptr;
    PyObject* id = PyLong_FromVoidPtr(mask_obj);
    PyObject* entry = id ? PyDict_GetItem(g_packed_table, id) : nullptr;
    Py_XDECREF(id);
    if (!entry || !PyTuple_Check(entry) || PyTuple_GET_SIZE(entry) != 3) return nullptr;
    PyObject* ref = PyTuple_GET_ITEM(entry, 0);
    if (!PyWeakref_Check(ref) || PyWeakref_GET_OBJECT(ref) != mask_obj) return nullptr;
    PyObject* key = PyTuple_GET_ITEM(entry, 1);
    if (!PyTuple_Check(key) || PyTuple_GET_SIZE(key) != 6) return nullptr;
    const int64_t want[5] = {(int64_t)mask._version(), (int64_t)a_idx._version(), (int64_t)l_idx._version(),
                             (int64_t)(uintptr_t)a_idx.data_ptr(), (int64_t)(uintptr_t)l_idx.data_ptr()};
    for (int i = 0; i < 5; ++i) {
        int64_t v;
        if (!as_int(PyTuple_GET_ITEM(key, i), &v) || v != want[i]) return nullptr;
    }
    PyObject* shape = PyTuple_GET_ITEM(key, 5);
    if (!PyTuple_Check(shape) || PyTuple_GET_SIZE(shape) != mask.dim()) return nullptr;
    for (int64_t d = 0; d < mask.dim(); ++d) {
        int64_t v;
        if (!as_int(PyTuple_GET_ITEM(shape, d), &v) || v != mask.size(d)) return nullptr;
    }
    return PyTuple_GET_ITEM(entry, 2);
}

// attention(q, k, v, ancestor_idx, ancestor_mask, leaf_idx, sm_scale, BLOCK_M, MAX_ANCESTORS, out_dtype, return_lse, flags,
//           k_scale, v_scale): attention.fst_attention with its switches as FSTA_FLAG_* bits
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 14 || !g_packed_table || !plain_context()) return not_implemented();
    const at::Tensor *q = gpu_tensor(args[0]), *k = gpu_tensor(args[1]), *v = gpu_tensor(args[2]);
    const at::Tensor *a_idx = gpu_tensor(args[3]), *l_idx = gpu_tensor(args[5]);
    if (!q || !k || !v || !a_idx || !l_idx) return not_implemented();
    if (c10::GradMode::is_enabled() && (wants_grad(*q) || wants_grad(*k) || wants_grad(*v))) return not_implemented();
    if (q->dim() != 4 || k->dim() != 4 || v->dim() != 4) return not_implemented();
    const int64_t d = q->size(3);
    if (k->size(3) != d || v->size(3) != d || (d != 16 && d != 32 && d != 64 && d != 128)) return not_implemented();
    int64_t block_m, max_anc, flags;
    if (!as_int(args[7], &block_m) || !as_int(args[8], &max_anc) || !as_int(args[11], &flags) || block_m <= 0) return not_implemented();
    const double sm_scale = PyFloat_CheckExact(args[6]) ? PyFloat_AS_DOUBLE(args[6]) : PyFloat_AsDouble(args[6]);
    if (sm_scale == -1.0 && PyErr_Occurred()) {
        PyErr_Clear();
        return not_implemented();
    }
    const bool return_lse = args[10] == Py_True;
    if (!return_lse && args[10] != Py_False) return not_implemented();
    const int in_code = fsta_torch::dtype_code(q->scalar_type());
    int out_code = in_code;
    if (args[9] != Py_None) {
        if (!THPDtype_Check(args[9])) return not_implemented();
        out_code = fsta_torch::dtype_code(reinterpret_cast<THPDtype*>(args[9])->scalar_type);
    }
    if (in_code < 0 || out_code < 0) return not_implemented();

    Packed p;
    if (Py_TYPE(args[4]) == reinterpret_cast<PyTypeObject*>(g_packed_type)) {
        if (!read_packed(args[4], &p)) return not_implemented();
        if (p.plan && !p.has_limit && p.key_shift != k->size(2) - q->size(2)) return not_implemented();
    } else {
        const at::Tensor* mask = gpu_tensor(args[4]);
        if (!mask || mask->dim() != 3 || a_idx->dim() != 2 || mask->size(0) != a_idx->size(0) || mask->size(1) != block_m ||
            mask->size(2) != max_anc)
            return not_implemented();
        PyObject* packed = recall(args[4], *mask, *a_idx, *l_idx);
        if (!packed || !read_packed(packed, &p) || (p.has_limit && p.key_limit != k->size(2))) return not_implemented();
    }
    if (p.block_m != block_m || p.max_ancestors != max_anc) return not_implemented();
    c10::optional<at::Tensor> k_scale, v_scale;
    for (int i = 0; i < 2; ++i)
        if (args[12 + i] != Py_None) {
            const at::Tensor* s = gpu_tensor(args[12 + i]);
            if (!s) return not_implemented();
            (i ? v_scale : k_scale) = *s;
        }
    try {
        const auto out = fsta_torch::attention_fwd(*q, *k, *v, *a_idx, *p.bits, *p.count, *l_idx,
                                                   p.plan ? c10::optional<at::Tensor>(*p.plan) : c10::nullopt, p.key_shift, sm_scale,
                                                   block_m, max_anc, out_code, return_lse, flags, k_scale, v_scale);
        PyObject* o = THPVariable_Wrap(std::get<0>(out));
        if (!o || !return_lse) return o;
        PyObject* lse = THPVariable_Wrap(std::get<1>(out));
        PyObject* both = lse ? PyTuple_Pack(2, o, lse) : nullptr;
        Py_DECREF(o);
        Py_XDECREF(lse);
        return both;
    } catch (const std::exception&) {
        return not_implemented();      // (the ordinary way meets the same condition and raises it)
    }
}

// setup(PackedTreeMask, packed_table)
PyObject* setup(PyObject*, PyObject* args) {
    PyObject *type, *table;
    if (!PyArg_ParseTuple(args, "OO!", &type, &PyDict_Type, &table)) return nullptr;
    Py_INCREF(type);
    Py_INCREF(table);
    Py_XSETREF(g_packed_type, type);
    Py_XSETREF(g_packed_table, table);
    Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&attention)), METH_FASTCALL, nullptr},
    {"setup", &setup, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fsta_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fsta_torch(void) { return PyModule_Create(&kModule); }
