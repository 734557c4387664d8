// The extension module `_fsta_torch`: the entry points of the package as plain C functions for calls that need nothing of
// torch's dispatcher (ordinary tensors on the GPU, no gradient, no mode that wants to see the call).  A call through the
// registered operator costs about 3 us of schema matching and boxing, and the lookup of the packed inputs another 1.5 us in
// Python; a launch of the smallest kernels takes less than that on the GPU.  Every function returns NotImplemented for a
// call it does not want to judge; the caller then takes the ordinary way, which also raises the errors.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/record_function.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <pybind11/pybind11.h>

#include <cstring>

#include "../../include/fsta.h"
#include "fsta_torch.h"

using fsta_torch::fresh;

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

// Nobody stands between the dispatcher and the kernels (dispatch modes, functorch, tracing).  Inference mode only takes
// ADInplaceOrView out of the default set, which looks after views of and writes to arguments: there are none here.
bool plain_dispatch() {
    const auto included = c10::impl::tls_local_dispatch_key_set().included_ | c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView);
    return included == c10::default_included_set;
}
// .. and nobody has asked to see calls from Python
bool plain_context() { return plain_dispatch() && !at::impl::torch_function_mode_enabled(); }

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

// Profilers and other observers see a call under the name of the registered operator
__attribute__((noinline)) void report(c10::optional<at::RecordFunction>& seen, at::StepCallbacks&& callbacks, const at::Tensor& q,
                                      const at::Tensor& k, const at::Tensor& v, const at::Tensor& a_idx, const Packed& p,
                                      const at::Tensor& l_idx) {
    seen.emplace(std::move(callbacks));
    if (seen->needsInputs()) {
        const c10::IValue inputs[] = {q, k, v, a_idx, *p.bits, *p.count, l_idx};
        seen->before("fsta::attention_fwd", c10::ArrayRef<const c10::IValue>(inputs, 7));
    } else {
        seen->before("fsta::attention_fwd");
    }
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
        c10::optional<at::RecordFunction> seen;
        if (auto callbacks = at::getStepCallbacksUnlessEmpty(at::RecordScope::FUNCTION))
            report(seen, std::move(*callbacks), *q, *k, *v, *a_idx, p, *l_idx);
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

// ---- front-end of a decoding step (integer work; outputs are new tensors, arguments are checked in precompute.py) -------
// A return code of the library other than FSTA_OK comes back as a Python int.

const at::Tensor& tensor_arg(PyObject* o) {
    TORCH_CHECK_TYPE(THPVariable_Check(o), "expected a torch.Tensor");
    return THPVariable_Unpack(o);
}

int64_t int_arg(PyObject* o) {
    int64_t v;
    TORCH_CHECK_TYPE(as_int(o, &v), "expected an int");
    return v;
}

struct OnStream {      // the tensors' device and torch's current stream on it
    explicit OnStream(const at::Tensor& t)
        : guard(t.device()), stream(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream()) {}
    const c10::hip::HIPGuardMasqueradingAsCUDA guard;
    const hipStream_t stream;
};

// The status word of a call: the caller's or a zeroed one
at::Tensor status_word(PyObject* given, const at::Tensor& like) {
    return given != Py_None ? tensor_arg(given) : at::zeros({1}, like.options().dtype(at::kInt));
}

template <class... T> PyObject* as_tuple(const T&... tensors) {      // undefined tensors become None
    PyObject* tuple = PyTuple_New(sizeof...(T));
    if (!tuple) return nullptr;
    Py_ssize_t i = 0;
    auto put = [&](const at::Tensor& t) {
        PyObject* o = t.defined() ? THPVariable_Wrap(t) : (Py_INCREF(Py_None), Py_None);
        PyTuple_SET_ITEM(tuple, i++, o);
        return o != nullptr;
    };
    if ((put(tensors) && ...)) return tuple;
    Py_DECREF(tuple);
    return nullptr;
}

// Watches the words of fsta_precompute_from_parents_flags until all of them are set (a wait for the stream costs 10 us more
// than the kernel takes).  Asks the runtime now and then, so that a launch that failed ends the wait with its error.
long watch_flags(const volatile int32_t* words, int64_t n, hipStream_t stream) {
    long found = 0;
    int spins = 0;
    bool drained = false;
    for (int64_t j = 0; j < n;) {
        if (const int32_t word = words[j]) {
            found |= word >> 1;
            ++j;
            continue;
        }
        TORCH_CHECK(!drained, "kernel_inputs_from_parents_gpu: the kernel ended without reporting");
        if (++spins % 4096 == 0) {
            const hipError_t err = hipStreamQuery(stream);
            TORCH_CHECK(err == hipSuccess || err == hipErrorNotReady, "kernel_inputs_from_parents_gpu: ", hipGetErrorString(err));
            drained = err == hipSuccess;      // (the word is looked at once more)
        }
        __builtin_ia32_pause();
    }
    return found;
}

template <class T> T* data_or_null(const at::Tensor& t) { return t.defined() ? static_cast<T*>(t.data_ptr()) : nullptr; }

// dfs_order(parent, light_first, read_status, status or None) -> (perm, rank, status)
PyObject* dfs_order(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n_args == 4, "dfs_order takes 4 arguments");
    const at::Tensor parent = tensor_arg(args[0]).contiguous();
    const OnStream on(parent);
    const int64_t n = parent.size(0);
    at::Tensor perm = fresh({n}, at::kLong, parent), rank = fresh({n}, at::kLong, parent);
    // (a status word that nobody reads is one int more of workspace)
    const int64_t ints = (int64_t)FSTA_DFS_ORDER_WORKSPACE_INTS(n);
    at::Tensor work = fresh({ints + 1}, at::kInt, parent), status;
    if (args[3] != Py_None || args[2] == Py_True) status = status_word(args[3], parent);
    uint32_t* word = status.defined() ? static_cast<uint32_t*>(status.data_ptr()) : reinterpret_cast<uint32_t*>(work.data_ptr<int32_t>() + ints);
    const int rc = fsta_dfs_order(parent.data_ptr<int64_t>(), n, args[1] == Py_True, perm.data_ptr<int64_t>(), rank.data_ptr<int64_t>(),
                                  work.data_ptr<int32_t>(), word, on.stream);
    return rc != FSTA_OK ? PyLong_FromLong(rc) : as_tuple(perm, rank, status);
    END_HANDLE_TH_ERRORS
}

// renumber_parents(parent, rank) -> new_parent
PyObject* renumber_parents(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n_args == 2, "renumber_parents takes 2 arguments");
    const at::Tensor parent = tensor_arg(args[0]).contiguous(), rank = tensor_arg(args[1]).contiguous();
    const OnStream on(parent);
    at::Tensor out = fresh(parent.sizes(), at::kLong, parent);
    const int rc = fsta_renumber_parents(parent.data_ptr<int64_t>(), rank.data_ptr<int64_t>(), parent.size(0), out.data_ptr<int64_t>(),
                                         on.stream);
    return rc != FSTA_OK ? PyLong_FromLong(rc) : THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// inputs_from_parents(parent, block_m, max_ancestors, width, check, want_bool_mask, want_lineage, status or None)
//   -> (ancestor_idx, ancestor_mask, leaf_idx, mask_bits, anc_count, plan, lineage, level_lookup, status), bits
// `check` (then no status word is used or returned): waits until every block has reported, bits are the FSTA_PRE_* conditions;
// else 0
PyObject* inputs_from_parents(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n_args == 8, "inputs_from_parents takes 8 arguments");
    const at::Tensor parent = tensor_arg(args[0]).contiguous();
    const int64_t n = parent.size(0), block_m = int_arg(args[1]), max_anc = int_arg(args[2]), width = int_arg(args[3]);
    const bool check = args[4] == Py_True, want_mask = args[5] == Py_True, want_lineage = args[6] == Py_True;
    TORCH_CHECK_VALUE(block_m > 0 && block_m <= INT32_MAX && max_anc > 0 && max_anc <= INT32_MAX && width > 0,
                      "block_m, max_ancestors and width must be positive");
    const OnStream on(parent);
    if (check) {      // (before anything is recorded: a replay would report into memory that has gone to others)
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        TORCH_CHECK(hipStreamIsCapturing(on.stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone,
                    "kernel_inputs_from_parents_gpu: check=True waits for the GPU, which a stream that is being captured does not");
    }
    const int64_t nb = (n + block_m - 1) / block_m;
    at::Tensor a_idx = fresh({nb, max_anc}, at::kLong, parent), l_idx = fresh({nb, block_m}, at::kLong, parent), a_mask, lineage, level, plan;
    if (want_mask) a_mask = fresh({nb, block_m, max_anc}, at::kBool, parent);
    at::Tensor bits = fresh({nb, (int64_t)fsta_mask_words((int32_t)max_anc), block_m}, at::kInt, parent), count = fresh({nb}, at::kInt, parent);
    const size_t plan_bytes = fsta_block_plan_bytes((int32_t)nb, (int32_t)block_m, (int32_t)max_anc);
    if (plan_bytes) plan = fresh({(int64_t)(plan_bytes / 4)}, at::kInt, parent);
    if (want_lineage) {
        lineage = fresh({n, width}, at::kLong, parent);
        level = fresh({n}, at::kLong, parent);
    }
    // A caller that waits is told through pinned host memory, a word per block; a word in device memory is for those that
    // look later.
    at::Tensor flags, status;
    if (check && nb > 0) {
        flags = at::empty({nb}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
        memset(flags.data_ptr(), 0, (size_t)nb * sizeof(int32_t));
    }
    if (!check) status = status_word(args[7], parent);
    const int rc = fsta_precompute_from_parents_flags(
        parent.data_ptr<int64_t>(), n, width, (int32_t)block_m, (int32_t)max_anc, 1, data_or_null<int64_t>(lineage),
        data_or_null<int64_t>(level), a_idx.data_ptr<int64_t>(), data_or_null<uint8_t>(a_mask), l_idx.data_ptr<int64_t>(),
        static_cast<uint32_t*>(bits.data_ptr()), count.data_ptr<int32_t>(), data_or_null<uint32_t>(plan),
        data_or_null<uint32_t>(status), data_or_null<uint32_t>(flags), on.stream);
    if (rc != FSTA_OK) return PyLong_FromLong(rc);
    long found = 0;
    if (check && nb > 0) {
        pybind11::gil_scoped_release no_gil;
        found = watch_flags(flags.data_ptr<int32_t>(), nb, on.stream);
    }
    PyObject* tensors = as_tuple(a_idx, a_mask, l_idx, bits, count, plan, lineage, level, status);
    return tensors ? Py_BuildValue("Nl", tensors, found) : nullptr;
    END_HANDLE_TH_ERRORS
}

// medusa_parents(probs, n, read_status, status or None) -> (parent, status)
PyObject* medusa_parents(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n_args == 4, "medusa_parents takes 4 arguments");
    const at::Tensor probs = tensor_arg(args[0]).contiguous();
    const int64_t n = int_arg(args[1]);
    const OnStream on(probs);
    const int32_t depths = (int32_t)probs.size(0), topk = (int32_t)probs.size(1);
    const int32_t code = probs.scalar_type() == at::kFloat ? FSTA_F32 : FSTA_F64;
    at::Tensor parent = fresh({n}, at::kLong, probs);
    at::Tensor status = args[3] != Py_None || args[2] == Py_True ? status_word(args[3], probs) : fresh({1}, at::kInt, probs);
    const size_t need = fsta_medusa_workspace_bytes(depths, topk);
    at::Tensor work;      // (stream-ordered: free again after the launches)
    if (need) work = fresh({(int64_t)need}, at::kByte, probs);
    uint32_t* word = static_cast<uint32_t*>(status.data_ptr());
    const int rc = need ? fsta_medusa_tree_ws(probs.data_ptr(), code, depths, topk, (int32_t)n, parent.data_ptr<int64_t>(), word,
                                              work.data_ptr(), need, on.stream)
                        : fsta_medusa_tree(probs.data_ptr(), code, depths, topk, (int32_t)n, parent.data_ptr<int64_t>(), word, on.stream);
    return rc != FSTA_OK ? PyLong_FromLong(rc) : as_tuple(parent, status);
    END_HANDLE_TH_ERRORS
}

// shift_index(ancestor_idx, leaf_idx, shift) -> both with `shift` added to the entries that are not negative; NotImplemented
// for anything but ordinary int64 tensors on one GPU
PyObject* shift_index(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 3 || !plain_context()) return not_implemented();
    const at::Tensor *a = gpu_tensor(args[0]), *b = gpu_tensor(args[1]);
    int64_t shift;
    if (!a || !b || a->scalar_type() != at::kLong || b->scalar_type() != at::kLong || a->device() != b->device() || !as_int(args[2], &shift))
        return not_implemented();
    const at::Tensor ac = a->contiguous(), bc = b->contiguous();
    const OnStream on(ac);
    at::Tensor out_a = fresh(ac.sizes(), at::kLong, ac), out_b = fresh(bc.sizes(), at::kLong, bc);
    const int rc = fsta_shift_index(ac.data_ptr<int64_t>(), ac.numel(), bc.data_ptr<int64_t>(), bc.numel(), shift,
                                    out_a.data_ptr<int64_t>(), out_b.data_ptr<int64_t>(), on.stream);
    return rc != FSTA_OK ? not_implemented() : as_tuple(out_a, out_b);
    END_HANDLE_TH_ERRORS
}

// quantizes(k, v): True if the operator for the 8-bit storage, whose only implementation is a kernel, takes both: ordinary GPU
// tensors of one shape and type, in slices of whole 16-byte pieces, that nobody transforms, traces below the dispatcher or
// differentiates, in either direction.  (A mode that watches calls from Python, such as a default device, sees the operator.)
PyObject* quantizes(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n_args == 2, "quantizes takes 2 arguments");
    if (!plain_dispatch()) Py_RETURN_FALSE;
    const at::Tensor* t[2];
    for (int i = 0; i < 2; ++i) {
        t[i] = gpu_tensor(args[i]);
        if (!t[i] || (c10::GradMode::is_enabled() && wants_grad(*t[i])) || t[i]->_fw_grad(0).defined()) Py_RETURN_FALSE;
    }
    const at::Tensor &k = *t[0], &v = *t[1];
    if (k.dim() != 4 || v.sizes() != k.sizes() || v.device() != k.device() || v.scalar_type() != k.scalar_type() ||
        fsta_torch::dtype_code(k.scalar_type()) < 0 || k.numel() == 0 || k.size(2) * k.size(3) % 16 != 0 ||
        k.size(0) * k.size(1) > (int64_t)1 << 20 ||      // (a workgroup of 1024 threads per slice of both: a grid ends at 2^32)
        (uintptr_t)k.data_ptr() % 16 != 0 || (uintptr_t)v.data_ptr() % 16 != 0)
        Py_RETURN_FALSE;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
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

#define FSTA_FASTCALL(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&f)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    FSTA_FASTCALL(attention),
    FSTA_FASTCALL(dfs_order),
    FSTA_FASTCALL(renumber_parents),
    FSTA_FASTCALL(inputs_from_parents),
    FSTA_FASTCALL(medusa_parents),
    FSTA_FASTCALL(shift_index),
    FSTA_FASTCALL(quantizes),
    {"setup", &setup, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fsta_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fsta_torch(void) { return PyModule_Create(&kModule); }
