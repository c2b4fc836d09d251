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
// For a short list whose plan is known the same module makes the whole call of a named function:
// describes the list, finds the plan, looks the packed buffer over (or allocates it) and calls the
// launch function of libtftq.so, whose address it has been given (bind).  Anything out of the
// ordinary gives None, and Python does the call in its own steps, with its own words for what is wrong.
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

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

namespace {

// A tensor is three objects one behind the other (the Python object, the tensor, its storage), and a
// walk that asks for each when it needs it waits for memory three times per tensor.  The objects of
// the tensors ahead are asked for before their turn; the tensor's first 64 bytes lead to its storage.
// (Inlined by force: with two callers the compiler makes it a call per tensor, and a pass of three
// walks over 10 000 tensors took 250 us instead of 230.)
constexpr Py_ssize_t AHEAD = 8;
__attribute__((always_inline)) inline void fetch_ahead(PyObject *const *items, Py_ssize_t i, Py_ssize_t n, PyTypeObject *plain, bool storages)
{
    if (i + 3 * AHEAD >= n) return;
    __builtin_prefetch(items[i + 3 * AHEAD]);
    PyObject *o = items[i + 2 * AHEAD];
    if (Py_TYPE(o) == plain) {
        const char *impl = reinterpret_cast<const char *>(THPVariable_Unpack(o).unsafeGetTensorImpl());
        if (storages) __builtin_prefetch(impl);
        __builtin_prefetch(impl + 64);
        __builtin_prefetch(impl + 128);
    }
    if (!storages) return;
    o = items[i + AHEAD];
    if (Py_TYPE(o) == plain) {
        const at::Tensor &t = THPVariable_Unpack(o);
        if (t.defined()) __builtin_prefetch(t.unsafeGetTensorImpl()->unsafe_storage().unsafeGetStorageImpl());
    }
}
inline PyTypeObject *plain_type() { return reinterpret_cast<PyTypeObject *>(THPVariableClass); }

// The loop of scan() (below): the index of the first tensor that does not match, or n.  Every look at
// a tensor is one that the compiler can make without a call: a pass of three walks over 10 000 tensors,
// two of them for the addresses, 239 -> 211 us.
template <bool POINTERS>
Py_ssize_t walk(PyObject *list, Py_ssize_t n, c10::Device device, caffe2::TypeMeta dtype, const int64_t *shapes,
                const int64_t *strides, uint64_t *pointers)
{
    PyObject *const *items = reinterpret_cast<PyListObject *>(list)->ob_item;
    PyTypeObject *const plain = plain_type();
    const uint64_t esz = dtype.itemsize();
    // tensors side by side are often views of one storage, whose address is then asked for once
    const c10::StorageImpl *storage = nullptr;
    uint64_t base = 0;
    for (Py_ssize_t i = 0; i < n; i++) {
        fetch_ahead(items, i, n, plain, POINTERS);
        PyObject *o = items[i];
        if (Py_TYPE(o) != plain && !THPVariable_Check(o)) return i;
        const at::Tensor &t = THPVariable_Unpack(o);
        // tensor subclasses that intercept operations (fake, functional, distributed
        // tensors) answer for themselves in Python
        if (!t.defined()) return i;
        c10::TensorImpl *impl = t.unsafeGetTensorImpl();
        if (impl->is_python_dispatch() || impl->dtype() != dtype || impl->device() != device) return i;
        const c10::IntArrayRef size = impl->sizes();
        const int64_t dim = static_cast<int64_t>(size.size());
        if (dim != 2 && dim != 1) return i;
        const int64_t *sz = size.data(), *st = impl->strides().data();
        const int64_t *shape = shapes + 2 * i, *stride = strides + 2 * i;
        // a 1-D tensor of k elements stands for its [k, 1] view (quantization.py:487-488)
        const int64_t n1 = dim == 2 ? sz[1] : 1, s1 = dim == 2 ? st[1] : 1;
        if (((sz[0] ^ shape[0]) | (n1 ^ shape[1]) | (st[0] ^ stride[0]) | (s1 ^ stride[1])) != 0) return i;
        if (!POINTERS) continue;
        if (impl->has_storage() && sz[0] != 0 && n1 != 0) {
            c10::StorageImpl *own = impl->unsafe_storage().unsafeGetStorageImpl();
            if (own != storage) {
                base = static_cast<uint64_t>(reinterpret_cast<uintptr_t>(own->mutable_data()));
                storage = own;
            }
            pointers[i] = base + static_cast<uint64_t>(impl->storage_offset()) * esz;
        } else {
            pointers[i] = static_cast<uint64_t>(reinterpret_cast<uintptr_t>(t.data_ptr()));
        }
    }
    return n;
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
// those sizes and strides (or the 1-D tensor that unsqueeze(1) turns into such a one); the index of the first element that is not, otherwise (0
// where a tensor answers with an exception); -1 when `tensors` is not a list of n elements.
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
    const c10::Device on = device >= 0 ? c10::Device(c10::kCUDA, static_cast<c10::DeviceIndex>(device)) : c10::Device(c10::kCPU);
    const int64_t *shapes = reinterpret_cast<const int64_t *>(static_cast<uintptr_t>(a_shapes));
    const int64_t *strides = reinterpret_cast<const int64_t *>(static_cast<uintptr_t>(a_strides));
    uint64_t *pointers = reinterpret_cast<uint64_t *>(static_cast<uintptr_t>(a_pointers));
    Py_ssize_t i = 0;
    try {
        const caffe2::TypeMeta meta = c10::scalarTypeToTypeMeta(want);
        i = pointers ? walk<true>(list, n, on, meta, shapes, strides, pointers)
                     : walk<false>(list, n, on, meta, shapes, strides, nullptr);
    } catch (...) {
        // whatever this list holds, the Python walk will say it in the reference's words
    }
    return PyLong_FromSsize_t(i);
}

// A list of 1 to `most` (at most 64) plain 2-D tensors of one of the three dtypes on one device.
struct ShortList {
    static constexpr Py_ssize_t MOST = 64;
    Py_ssize_t n = 0;
    int64_t device = 0;            // ordinal; -1: host memory
    int64_t key[2 + 4 * MOST];     // differs for lists of other lengths, dtypes, devices, sizes or strides
    uint64_t pointers[MOST];       // the tensors' addresses
    Py_ssize_t key_bytes() const { return (2 + 4 * n) * 8; }

    bool describe(PyObject *list, Py_ssize_t most)
    {
        if (most > MOST) most = MOST;
        n = PyList_CheckExact(list) ? PyList_GET_SIZE(list) : 0;
        if (n < 1 || n > most) return false;
        try {
            for (Py_ssize_t i = 0; i < n; i++) {
                PyObject *o = PyList_GET_ITEM(list, i);
                if (!THPVariable_CheckExact(o)) return false;
                const at::Tensor &t = THPVariable_Unpack(o);
                if (!t.defined() || t.unsafeGetTensorImpl()->is_python_dispatch() || t.dim() != 2) return false;
                const c10::Device d = t.device();
                if (!d.is_cuda() && !d.is_cpu()) return false;
                const int64_t dtype = static_cast<int64_t>(t.scalar_type()), at_device = d.is_cuda() ? d.index() : -1;
                if (i == 0) {
                    if (t.scalar_type() != at::kFloat && t.scalar_type() != at::kHalf && t.scalar_type() != at::kBFloat16) return false;
                    key[0] = dtype;
                    key[1] = device = at_device;
                }
                if (dtype != key[0] || at_device != device) return false;
                const c10::IntArrayRef sz = t.sizes(), st = t.strides();
                int64_t *k = key + 2 + 4 * i;
                k[0] = sz[0];
                k[1] = sz[1];
                k[2] = st[0];
                k[3] = st[1];
                pointers[i] = static_cast<uint64_t>(reinterpret_cast<uintptr_t>(t.data_ptr()));
            }
        } catch (...) {
            return false;  // whatever this tensor is, the Python walk will say it in the reference's words
        }
        return true;
    }
};

// describe(tensors, most) -> (key, device, pointers) or None
// What a ShortList holds, key and pointers as bytes.  None for anything that is not such a list.
PyObject *describe(PyObject *, PyObject *args)
{
    PyObject *list = nullptr;
    Py_ssize_t most = 0;
    if (!PyArg_ParseTuple(args, "On", &list, &most)) return nullptr;
    ShortList l;
    if (!l.describe(list, most)) Py_RETURN_NONE;
    return Py_BuildValue("(y#iy#)", reinterpret_cast<const char *>(l.key), l.key_bytes(), static_cast<int>(l.device),
                         reinterpret_cast<const char *>(l.pointers), l.n * 8);
}

// ---------------------------------------------------------------------------
// whole calls
// ---------------------------------------------------------------------------
// What libtftq.so launches with (tftq.h), and what says which stream is current.
struct {
    int (*quantize)(const void *plan, const void *const *tensors, const void *table, void *pointers, void *packed,
                    int64_t packed_bytes, int device, void *stream) = nullptr;
    int (*reduce)(const void *plan, const void *table, void *packed, int64_t packed_bytes, int rank, int is_avg, int device,
                  void *stream) = nullptr;
    int (*dequantize)(const void *plan, void *const *tensors, const void *table, void *pointers, const void *packed,
                      int64_t packed_bytes, int device, void *stream) = nullptr;
    int (*dequantize_scaled)(const void *plan, void *const *tensors, const void *table, void *pointers, const void *packed,
                             int64_t packed_bytes, float post_scale, int device, void *stream) = nullptr;
    PyObject *raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream
} library;

PyObject *name_address, *name_output_size, *name_used;

// A plan (quantization._Plan) for one call.
struct Plan {
    PyObject *object = nullptr;  // owned
    const void *address = nullptr;
    int64_t output_size = 0;
    ~Plan() { Py_XDECREF(object); }

    bool read(PyObject *plan)
    {
        Py_INCREF(plan);
        object = plan;
        PyObject *a = PyObject_GetAttr(plan, name_address), *b = PyObject_GetAttr(plan, name_output_size);
        if (a && b) {
            address = reinterpret_cast<const void *>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLong(a)));
            output_size = PyLong_AsLongLong(b);
        }
        Py_XDECREF(a);
        Py_XDECREF(b);
        if (PyErr_Occurred()) PyErr_Clear();
        return address != nullptr;
    }
    // The plan that `plans` (quantization._short_plans) has for the list.
    bool find(PyObject *plans, const ShortList &l, PyObject *ws)
    {
        if (!PyLong_CheckExact(ws) || !PyDict_CheckExact(plans)) return false;
        PyObject *key = PyBytes_FromStringAndSize(reinterpret_cast<const char *>(l.key), l.key_bytes());
        PyObject *pair = key ? PyTuple_Pack(2, key, ws) : nullptr;
        PyObject *plan = pair ? PyDict_GetItemWithError(plans, pair) : nullptr;  // borrowed
        const bool found = plan && read(plan) && PyObject_SetAttr(plan, name_used, Py_True) == 0;
        Py_XDECREF(pair);
        Py_XDECREF(key);
        if (PyErr_Occurred()) PyErr_Clear();
        return found;
    }
};

// Whether this thread's operations go straight to the tensors: modes that intercept them (a tracer, a
// fake mode) see what Python does.
bool plain_calls()
{
    return library.quantize && !at::impl::torch_function_mode_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set();
}

bool current_stream(int64_t device, void **stream)
{
    PyObject *index = PyLong_FromLongLong(device);
    PyObject *raw = index ? PyObject_CallOneArg(library.raw_stream, index) : nullptr;
    Py_XDECREF(index);
    if (raw) *stream = reinterpret_cast<void *>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLong(raw)));
    Py_XDECREF(raw);
    if (!PyErr_Occurred()) return true;
    PyErr_Clear();
    return false;
}

// The address of a packed buffer that _check_packed has nothing to say about.
bool packed_buffer(PyObject *o, int64_t device, int64_t bytes, void **address)
{
    if (!THPVariable_CheckExact(o)) return false;
    try {
        const at::Tensor &t = THPVariable_Unpack(o);
        if (!t.defined() || t.unsafeGetTensorImpl()->is_python_dispatch() || t.dim() < 1 || t.scalar_type() != at::kByte ||
            t.size(0) != bytes || !t.is_contiguous() || !t.device().is_cuda() || t.device().index() != device)
            return false;
        *address = t.data_ptr();
    } catch (...) {
        return false;
    }
    return true;
}

// Leaves the interpreter to other threads for the lifetime of the object, exceptions included.
struct WithoutInterpreter {
    PyThreadState *state = PyEval_SaveThread();
    ~WithoutInterpreter() { PyEval_RestoreThread(state); }
};

PyObject *launch_quantize(const Plan &plan, const void *const *tensors, int64_t device)
{
    void *stream = nullptr;
    if (!current_stream(device, &stream)) Py_RETURN_NONE;
    try {
        at::Tensor out;
        int rc;
        {
            // The allocation too: it may have to wait for work on the GPU, and what ends that wait (the
            // abort of a collective whose peer is gone, say) may be another thread's to do.
            WithoutInterpreter others_run;
            out = at::empty({plan.output_size}, at::TensorOptions(at::kByte).device(c10::Device(c10::kCUDA, static_cast<c10::DeviceIndex>(device))));
            rc = library.quantize(plan.address, tensors, nullptr, nullptr, out.data_ptr(), plan.output_size, static_cast<int>(device), stream);
        }
        return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(std::move(out));
    } catch (...) {  // out of memory, say: Python says so
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

PyObject *launch_reduce(const Plan &plan, PyObject *o, PyObject *rank, PyObject *is_avg, int64_t device)
{
    void *stream = nullptr, *packed = nullptr;
    if (!PyLong_CheckExact(rank) || !PyLong_CheckExact(is_avg) || !packed_buffer(o, device, plan.output_size, &packed)) Py_RETURN_NONE;
    int overflow = 0;
    const long r = PyLong_AsLongAndOverflow(rank, &overflow), avg = PyLong_AsLong(is_avg);
    if (overflow || r != static_cast<int>(r) || !current_stream(device, &stream)) Py_RETURN_NONE;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = library.reduce(plan.address, nullptr, packed, plan.output_size, static_cast<int>(r), avg != 0, static_cast<int>(device), stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

// post_scale: None or a float
PyObject *launch_dequantize(const Plan &plan, void *const *tensors, PyObject *o, PyObject *post_scale, int64_t device)
{
    void *stream = nullptr, *packed = nullptr;
    if ((post_scale != Py_None && !PyFloat_CheckExact(post_scale)) || !packed_buffer(o, device, plan.output_size, &packed) ||
        !current_stream(device, &stream))
        Py_RETURN_NONE;
    const float scale = post_scale == Py_None ? 1.0f : static_cast<float>(PyFloat_AS_DOUBLE(post_scale));
    int rc;
    Py_BEGIN_ALLOW_THREADS
    if (post_scale == Py_None)
        rc = library.dequantize(plan.address, tensors, nullptr, nullptr, packed, plan.output_size, static_cast<int>(device), stream);
    else
        rc = library.dequantize_scaled(plan.address, tensors, nullptr, nullptr, packed, plan.output_size, scale, static_cast<int>(device), stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

bool arguments(const char *what, Py_ssize_t got, Py_ssize_t want)
{
    if (got == want) return true;
    PyErr_Format(PyExc_TypeError, "%s takes %zd arguments", what, want);
    return false;
}

// quantize(tensors, most, ws, plans) -> the packed tensor, the error code of tftq_quantize, or None
PyObject *quantize(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (!arguments("quantize", n, 4)) return nullptr;
    ShortList l;
    Plan plan;
    if (!plain_calls() || !l.describe(args[0], PyLong_AsSsize_t(args[1])) || l.device < 0 || !plan.find(args[3], l, args[2])) Py_RETURN_NONE;
    return launch_quantize(plan, reinterpret_cast<const void *const *>(l.pointers), l.device);
}

// reduce(tensors, most, ws, plans, packed, rank, is_avg) -> the code of tftq_reduce, or None
PyObject *reduce(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (!arguments("reduce", n, 7)) return nullptr;
    ShortList l;
    Plan plan;
    if (!plain_calls() || !l.describe(args[0], PyLong_AsSsize_t(args[1])) || l.device < 0 || !plan.find(args[3], l, args[2])) Py_RETURN_NONE;
    return launch_reduce(plan, args[4], args[5], args[6], l.device);
}

// dequantize(tensors, most, ws, plans, packed, post_scale) -> the code of tftq_dequantize(_scaled), or None
PyObject *dequantize(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (!arguments("dequantize", n, 6)) return nullptr;
    ShortList l;
    Plan plan;
    if (!plain_calls() || !l.describe(args[0], PyLong_AsSsize_t(args[1])) || l.device < 0 || !plan.find(args[3], l, args[2])) Py_RETURN_NONE;
    return launch_dequantize(plan, reinterpret_cast<void *const *>(l.pointers), args[4], args[5], l.device);
}

// The same for a prepared bucket of a short list, whose plan and addresses (`pointers`: of the host
// array that holds them) are known.
// bucket_quantize(plan, device, pointers), bucket_reduce(plan, device, packed, rank, is_avg),
// bucket_dequantize(plan, device, pointers, packed, post_scale)
PyObject *bucket_quantize(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (!arguments("bucket_quantize", n, 3)) return nullptr;
    Plan plan;
    if (!plain_calls() || !plan.read(args[0])) Py_RETURN_NONE;
    return launch_quantize(plan, reinterpret_cast<const void *const *>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLong(args[2]))),
                           PyLong_AsLongLong(args[1]));
}
PyObject *bucket_reduce(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (!arguments("bucket_reduce", n, 5)) return nullptr;
    Plan plan;
    if (!plain_calls() || !plan.read(args[0])) Py_RETURN_NONE;
    return launch_reduce(plan, args[2], args[3], args[4], PyLong_AsLongLong(args[1]));
}
PyObject *bucket_dequantize(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (!arguments("bucket_dequantize", n, 5)) return nullptr;
    Plan plan;
    if (!plain_calls() || !plan.read(args[0])) Py_RETURN_NONE;
    return launch_dequantize(plan, reinterpret_cast<void *const *>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLong(args[2]))),
                             args[3], args[4], PyLong_AsLongLong(args[1]));
}

// bind(quantize, reduce, dequantize, dequantize_scaled, raw_stream): the addresses of libtftq.so's
// functions and the callable that says which stream of a device is current.
PyObject *bind(PyObject *, PyObject *args)
{
    unsigned long long q = 0, r = 0, d = 0, ds = 0;
    PyObject *raw = nullptr;
    if (!PyArg_ParseTuple(args, "KKKKO", &q, &r, &d, &ds, &raw)) return nullptr;
    Py_INCREF(raw);
    Py_XDECREF(library.raw_stream);
    library.raw_stream = raw;
    library.reduce = reinterpret_cast<decltype(library.reduce)>(static_cast<uintptr_t>(r));
    library.dequantize = reinterpret_cast<decltype(library.dequantize)>(static_cast<uintptr_t>(d));
    library.dequantize_scaled = reinterpret_cast<decltype(library.dequantize_scaled)>(static_cast<uintptr_t>(ds));
    library.quantize = reinterpret_cast<decltype(library.quantize)>(static_cast<uintptr_t>(q));
    Py_RETURN_NONE;
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
        PyObject *const *items = reinterpret_cast<PyListObject *>(owners)->ob_item;
        PyTypeObject *const plain = plain_type();
        spans.reserve(static_cast<size_t>(n));
        for (Py_ssize_t i = 0; i < n; i++) {
            fetch_ahead(items, i, n, plain, true);
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

PyCFunction fast(PyObject *(*f)(PyObject *, PyObject *const *, Py_ssize_t)) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "bind(quantize, reduce, dequantize, dequantize_scaled, raw_stream): the functions of whole calls"},
    {"quantize", fast(quantize), METH_FASTCALL, "quantize(tensors, most, ws, plans): fused_quantize_into_fp8 of a short list, or None"},
    {"reduce", fast(reduce), METH_FASTCALL, "reduce(tensors, most, ws, plans, packed, rank, is_avg): fused_reduce_fp8, or None"},
    {"dequantize", fast(dequantize), METH_FASTCALL,
     "dequantize(tensors, most, ws, plans, packed, post_scale): fused_dequantize_from_fp8, or None"},
    {"bucket_quantize", fast(bucket_quantize), METH_FASTCALL, "bucket_quantize(plan, device, pointers)"},
    {"bucket_reduce", fast(bucket_reduce), METH_FASTCALL, "bucket_reduce(plan, device, packed, rank, is_avg)"},
    {"bucket_dequantize", fast(bucket_dequantize), METH_FASTCALL, "bucket_dequantize(plan, device, pointers, packed, post_scale)"},
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
    name_address = PyUnicode_InternFromString("address");
    name_output_size = PyUnicode_InternFromString("output_size");
    name_used = PyUnicode_InternFromString("used");
    if (!name_address || !name_output_size || !name_used) return nullptr;
    PyObject *m = PyModule_Create(&module);
    // identifies the source the module was built from (a hash that the build passes in)
    if (m && PyModule_AddStringConstant(m, "BUILD_ID", TFTQ_PYLIST_ID) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
