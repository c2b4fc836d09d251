// _pylist: one walk over a Python list of tensors, in C++.
//
// The three functions of torchft/quantization.py walk their tensor list on every call
// (_prepare_quantize_fp8, quantization.py:462-515: device, dtype, dimensions, shapes,
// strides, addresses).  In Python that walk costs about half a microsecond per tensor and
// check, milliseconds for a list of 10 000 tensors whose kernels take 50 us.  scan() makes
// all the checks against the arrays of a cached plan and collects the addresses in one
// pass of a few nanoseconds per tensor.  It decides nothing on its own: any tensor that
// does not match sends the caller back to the Python walk, which builds a new plan or
// raises the reference's assertion.
//
// Host code only; built with the host compiler against the Python and libtorch headers
// (torchft_amd/_build.py).  Not part of libtftq.so, whose C ABI has no Python or torch
// types.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <algorithm>
#include <utility>
#include <vector>

#include <torch/csrc/autograd/python_variable.h>

#include <ATen/core/Tensor.h>

namespace {

// A tensor is three objects one behind the other (the Python object, the tensor, its storage), and a
// walk that asks for each when it needs it waits for memory three times per tensor.  The objects of
// the tensors ahead are asked for before their turn.  (Inlined by force: with two callers the compiler
// makes it a call per tensor, and a pass of three walks over 10 000 tensors took 250 us instead of 230.)
constexpr Py_ssize_t AHEAD = 8;
__attribute__((always_inline)) inline void fetch_ahead(PyObject *list, Py_ssize_t i, Py_ssize_t n, bool storages)
{
    if (i + 3 * AHEAD < n) __builtin_prefetch(PyList_GET_ITEM(list, i + 3 * AHEAD));
    if (i + 2 * AHEAD < n) {
        PyObject *o = PyList_GET_ITEM(list, i + 2 * AHEAD);
        if (THPVariable_CheckExact(o)) {
            const char *impl = reinterpret_cast<const char *>(THPVariable_Unpack(o).unsafeGetTensorImpl());
            __builtin_prefetch(impl);
            __builtin_prefetch(impl + 64);
            __builtin_prefetch(impl + 128);
        }
    }
    if (storages && i + AHEAD < n) {
        PyObject *o = PyList_GET_ITEM(list, i + AHEAD);
        if (THPVariable_CheckExact(o)) {
            const at::Tensor &t = THPVariable_Unpack(o);
            if (t.defined()) __builtin_prefetch(t.unsafeGetTensorImpl()->unsafe_storage().unsafeGetStorageImpl());
        }
    }
}

// scan(tensors, dtype, device, shapes, strides, pointers, n) -> int
//   tensors   a list
//   dtype     0 = float32, 1 = float16, 2 = bfloat16 (the TFTQ_* codes of tftq.h)
//   device    ordinal of the GPU every tensor must be on (-1: host memory; the tests of this
//             walk run where there is no GPU)
//   shapes    address of int64[n][2]: the sizes every tensor must have
//   strides   address of int64[n][2]: the strides every tensor must have
//   pointers  address of uint64[n] that receives the tensors' addresses (0: not wanted)
//   n         length the list must have
// Returns n when every element is a plain 2-D tensor of that dtype on that device with
// those sizes and strides (or the 1-D tensor that unsqueeze(1) turns into such a one); the index of the first element that is not, otherwise (the
// addresses before it have then been written); -1 when `tensors` is not a list of n elements.
PyObject *scan(PyObject *, PyObject *args)
{
    PyObject *list = nullptr;
    int dtype_code = 0, device = 0;
    unsigned long long a_shapes = 0, a_strides = 0, a_pointers = 0;
    Py_ssize_t n = 0;
    if (!PyArg_ParseTuple(args, "OiiKKKn", &list, &dtype_code, &device, &a_shapes, &a_strides, &a_pointers, &n))
        return nullptr;
    if (!PyList_CheckExact(list) || PyList_GET_SIZE(list) != n) return PyLong_FromLong(-1);
    const at::ScalarType want = dtype_code == 0   ? at::kFloat
                                : dtype_code == 1 ? at::kHalf
                                                  : at::kBFloat16;
    const int64_t *shapes = reinterpret_cast<const int64_t *>(static_cast<uintptr_t>(a_shapes));
    const int64_t *strides = reinterpret_cast<const int64_t *>(static_cast<uintptr_t>(a_strides));
    uint64_t *pointers = reinterpret_cast<uint64_t *>(static_cast<uintptr_t>(a_pointers));
    Py_ssize_t i = 0;
    try {
        for (; i < n; i++) {
            fetch_ahead(list, i, n, pointers != nullptr);
            PyObject *o = PyList_GET_ITEM(list, i);
            if (!THPVariable_CheckExact(o) && !THPVariable_Check(o)) break;
            const at::Tensor &t = THPVariable_Unpack(o);
            // tensor subclasses that intercept operations (fake, functional, distributed
            // tensors) answer for themselves in Python
            if (!t.defined() || t.unsafeGetTensorImpl()->is_python_dispatch()) break;
            const int64_t dim = t.dim();
            if ((dim != 2 && dim != 1) || t.scalar_type() != want) break;
            const c10::Device d = t.device();
            if (device >= 0 ? (!d.is_cuda() || d.index() != device) : !d.is_cpu()) break;
            const c10::IntArrayRef sz = t.sizes(), st = t.strides();
            // a 1-D tensor of k elements stands for its [k, 1] view (quantization.py:487-488)
            if (sz[0] != shapes[2 * i] || (dim == 2 ? sz[1] : 1) != shapes[2 * i + 1]) break;
            if (st[0] != strides[2 * i] || (dim == 2 ? st[1] : 1) != strides[2 * i + 1]) break;
            if (pointers) pointers[i] = static_cast<uint64_t>(reinterpret_cast<uintptr_t>(t.data_ptr()));
        }
    } catch (...) {
        // whatever this tensor is, the Python walk will say it in the reference's words
    }
    return PyLong_FromSsize_t(i);
}

// describe(tensors, most) -> (key, device, pointers) or None
// For a list of 1 to `most` (at most 64) plain 2-D tensors of one of the three dtypes on one device:
// bytes that differ for lists of other lengths, dtypes, devices, sizes or strides, the device's
// ordinal (-1: host memory) and the tensors' addresses as the bytes of an array of uint64.  None
// for anything else.
PyObject *describe(PyObject *, PyObject *args)
{
    constexpr Py_ssize_t MOST = 64;
    PyObject *list = nullptr;
    Py_ssize_t most = 0;
    if (!PyArg_ParseTuple(args, "On", &list, &most)) return nullptr;
    if (most > MOST) most = MOST;
    const Py_ssize_t n = PyList_CheckExact(list) ? PyList_GET_SIZE(list) : 0;
    if (n < 1 || n > most) Py_RETURN_NONE;
    int64_t key[2 + 4 * MOST];
    uint64_t pointers[MOST];
    int64_t device = 0;
    try {
        for (Py_ssize_t i = 0; i < n; i++) {
            PyObject *o = PyList_GET_ITEM(list, i);
            if (!THPVariable_CheckExact(o)) Py_RETURN_NONE;
            const at::Tensor &t = THPVariable_Unpack(o);
            if (!t.defined() || t.unsafeGetTensorImpl()->is_python_dispatch() || t.dim() != 2) Py_RETURN_NONE;
            const c10::Device d = t.device();
            if (!d.is_cuda() && !d.is_cpu()) Py_RETURN_NONE;
            const int64_t dtype = static_cast<int64_t>(t.scalar_type()), at_device = d.is_cuda() ? d.index() : -1;
            if (i == 0) {
                if (t.scalar_type() != at::kFloat && t.scalar_type() != at::kHalf && t.scalar_type() != at::kBFloat16) Py_RETURN_NONE;
                key[0] = dtype;
                key[1] = device = at_device;
            }
            if (dtype != key[0] || at_device != device) Py_RETURN_NONE;
            const c10::IntArrayRef sz = t.sizes(), st = t.strides();
            int64_t *k = key + 2 + 4 * i;
            k[0] = sz[0];
            k[1] = sz[1];
            k[2] = st[0];
            k[3] = st[1];
            pointers[i] = static_cast<uint64_t>(reinterpret_cast<uintptr_t>(t.data_ptr()));
        }
    } catch (...) {
        Py_RETURN_NONE;  // whatever this tensor is, the Python walk will say it in the reference's words
    }
    return Py_BuildValue("(y#iy#)", reinterpret_cast<const char *>(key), static_cast<Py_ssize_t>((2 + 4 * n) * 8),
                         static_cast<int>(device), reinterpret_cast<const char *>(pointers), static_cast<Py_ssize_t>(n * 8));
}

// Tensors that stand for others.
constexpr c10::DispatchKeySet WRAPPERS({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                        c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::BatchedNestedTensor,
                                        c10::DispatchKey::Functionalize});

// in_place(owners, pieces, known) -> addresses, or None
// The owners' addresses as a list of ints, if a kernel may read and write the owners, all at once, as
// the elements of `pieces` (as many plain contiguous tensors), and `known` itself if they are the
// addresses that this list holds.  None where only a copy does that: tensors of another type, dtype,
// device or shape than their piece, that are not contiguous, that autograd or functorch follows, that
// were made in inference mode, that have their sign in a flag or no memory, and owners that share
// memory.
PyObject *in_place(PyObject *, PyObject *args)
{
    PyObject *owners = nullptr, *pieces = nullptr, *known = nullptr;
    if (!PyArg_ParseTuple(args, "O!O!O", &PyList_Type, &owners, &PyList_Type, &pieces, &known)) return nullptr;
    const Py_ssize_t n = PyList_GET_SIZE(owners);
    if (PyList_GET_SIZE(pieces) != n) Py_RETURN_NONE;
    bool same = PyList_CheckExact(known) && PyList_GET_SIZE(known) == n;
    std::vector<std::pair<uintptr_t, uintptr_t>> spans;
    PyObject *out = nullptr;
    try {
        spans.reserve(static_cast<size_t>(n));
        for (Py_ssize_t i = 0; i < n; i++) {
            fetch_ahead(owners, i, n, true);
            PyObject *o = PyList_GET_ITEM(owners, i), *q = PyList_GET_ITEM(pieces, i);
            if (!THPVariable_CheckExact(o) || !THPVariable_Check(q)) Py_RETURN_NONE;
            const at::Tensor &t = THPVariable_Unpack(o), &piece = THPVariable_Unpack(q);
            if (!t.defined() || t.key_set().has_any(WRAPPERS) || !t.has_storage() || t.layout() != at::kStrided ||
                t.scalar_type() != piece.scalar_type() || t.device() != piece.device() ||
                t.sizes() != piece.sizes() || !t.is_contiguous() || t.requires_grad() || t.is_neg() || t.is_inference())
                Py_RETURN_NONE;
            const uintptr_t at = reinterpret_cast<uintptr_t>(t.data_ptr());
            if (at == 0 && t.numel() != 0) Py_RETURN_NONE;
            spans.emplace_back(at, at + t.nbytes());
            same = same && PyLong_AsUnsignedLongLong(PyList_GET_ITEM(known, i)) == at;
        }
        if (same) {  // looked at when they were written down
            Py_INCREF(known);
            return known;
        }
        out = PyList_New(n);
        if (!out) return nullptr;
        for (Py_ssize_t i = 0; i < n; i++) {
            PyObject *a = PyLong_FromUnsignedLongLong(spans[static_cast<size_t>(i)].first);
            if (!a) {
                Py_DECREF(out);
                return nullptr;
            }
            PyList_SET_ITEM(out, i, a);
        }
        std::sort(spans.begin(), spans.end());
        uintptr_t end = 0;
        for (const auto &span : spans) {
            if (span.first == span.second) continue;
            if (span.first < end) {
                Py_DECREF(out);
                Py_RETURN_NONE;
            }
            end = span.second;
        }
        return out;
    } catch (...) {  // a tensor that answers none of this
        Py_XDECREF(out);
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

PyMethodDef methods[] = {
    {"in_place", in_place, METH_VARARGS,
     "in_place(owners, pieces, known): the owners' addresses if kernels may work on them in place of the pieces, or None"},
    {"describe", describe, METH_VARARGS,
     "describe(tensors, most): (bytes that tell lists apart, device, addresses) of a short list of 2-D tensors, or None"},
    {"scan", scan, METH_VARARGS,
     "scan(tensors, dtype, device, shapes, strides, pointers, n): check a list of tensors against a plan's "
     "arrays and collect their addresses; returns n, the index of the first mismatch, or -1"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pylist", "C++ walk over lists of tensors", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

#ifndef TFTQ_PYLIST_ID
#define TFTQ_PYLIST_ID "unknown"
#endif

PyMODINIT_FUNC PyInit__pylist(void)
{
    PyObject *m = PyModule_Create(&module);
    // identifies the source the module was built from (a hash that the build passes in)
    if (m && PyModule_AddStringConstant(m, "BUILD_ID", TFTQ_PYLIST_ID) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
