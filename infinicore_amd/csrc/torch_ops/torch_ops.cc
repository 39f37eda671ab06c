// The calls of infinicore_amd/ops.py on their way from torch tensors to the C API of libinfiniop.so: output allocation,
// plan lookup by the tensors' metadata, pointers, current stream, call. What the reference does there in C++
// (src/infinicore/ops/paged_attention/paged_attention_infiniop.cc:16-58). In Python this took longer than the kernels of
// a small call (us a pass, in Python / here): rotation, cache write and decode of one sequence of 1 023 tokens 26.9 / 12.6, of
// four prompts of 19 - 250 24.1 / 16.8; a small decode alone 12.1 / 6.6; a first call with new metadata 71 / 36.
//
// A plan (operator descriptor) is made by a Python function the first time its metadata is seen and kept in a cache
// bounded by least recent use; device and stream are part of the key. Scratch of a call:
//   * prefill: from torch's allocator for this call alone, given back when its kernels are enqueued, as torch's own
//     operators do. Calls of several threads never share it, under capture it comes from the graph's pool, and a hundred
//     plans (one per prompt shape) do not hold tens of MB each beside a KV pool that was sized without them.
//   * decode: kept by the plan, because a call leaves in it where its first tiles were for the next call (the next layer of
//     a step). Threads that make the same call on one stream take turns (the launches of one call would otherwise interleave
//     with the other's between partial rows and merge). Calls under capture have a buffer from the graph's pool, one per
//     capture, which lives as long as the graph, whatever becomes of the plan.
// The cache is only touched with the interpreter lock held; the lock is given up during the call into the library, and a
// shared pointer keeps the plan alive until the call is back, whoever evicts it meanwhile.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstring>
#include <memory>
#include <mutex>
#include <vector>

#include "infinicore/lru_cache.h"

namespace {

using infinicore_amd::LruCache;
using infinicore_amd::MetaKey;
using infinicore_amd::MetaKeyHash;

// The operators, by the number ops.py knows them by.
struct Operator {
    int tensors;
    int device_tensor;  // the tensor that says which device (and must be on one)
    bool has_out;       // tensors[0] is the output, allocated here where it is None
    bool last_optional; // the last tensor may be None
    bool keeps_scratch; // its scratch is worth keeping from call to call
};
constexpr Operator kOperators[] = {
    {7, 1, true, true, true},     // paged_attention: out, q, k_cache, v_cache, block_tables, cache_lens, alibi_slopes
    {8, 1, true, true, false},    // paged_attention_prefill: ... seq_lens, cum_seq_lens_q, alibi_slopes
    {5, 2, false, false, false},  // paged_caching: k_cache, v_cache, k, v, slot_mapping
    {8, 2, false, false, false},  // rope_paged_caching: ... slot_mapping, pos_ids, sin_table, cos_table
    {10, 4, false, false, false}, // the same with q_out, q in front
    {5, 2, false, false, false},  // kv_caching: k_cache, v_cache, k, v, past_kv_lengths
};
constexpr int kNumOperators = sizeof(kOperators) / sizeof(kOperators[0]);
constexpr int kMaxTensors = 10;

using SetDevice = int (*)(int, int);
struct Library {
    void *run[kNumOperators];
    SetDevice set_device;
    int device_type;
    bool ready;
};
Library g_library{};

std::vector<PyObject *> g_retired; // plans nobody uses any more, to be closed where Python code may run

struct Entry {
    PyObject *plan = nullptr;
    void *descriptor = nullptr;
    size_t workspace_bytes = 0;
    std::mutex turn; // of the calls that use the buffers
    c10::DataPtr scratch, captured_scratch;
    unsigned long long capture = 0; // that captured_scratch belongs to
    ~Entry() {
        if (plan != nullptr) {
            g_retired.push_back(plan);
        }
    }
};
using EntryPtr = std::shared_ptr<Entry>;
using Cache = LruCache<MetaKey, EntryPtr, MetaKeyHash>;

Cache &cache() {
    static Cache *const c = new Cache(100); // never destroyed: its plans hold Python objects
    return *c;
}

// Closes retired plans. With an error already set, theirs are reported and dropped.
void closeRetired() {
    while (!g_retired.empty()) {
        PyObject *plan = g_retired.back();
        g_retired.pop_back();
        PyObject *type, *value, *trace;
        PyErr_Fetch(&type, &value, &trace);
        PyObject *r = PyObject_CallMethod(plan, "close", nullptr);
        if (r == nullptr) {
            PyErr_WriteUnraisable(plan);
        }
        Py_XDECREF(r);
        Py_DECREF(plan);
        PyErr_Restore(type, value, trace);
    }
}

bool readPlan(PyObject *plan, Entry &entry) {
    auto number = [&](const char *name, unsigned long long &out) {
        PyObject *x = PyObject_GetAttrString(plan, name);
        if (x == nullptr) {
            return false;
        }
        out = PyLong_AsUnsignedLongLong(x);
        Py_DECREF(x);
        return !PyErr_Occurred();
    };
    unsigned long long descriptor = 0, bytes = 0;
    if (!number("descriptor_address", descriptor) || !number("workspace_bytes", bytes)) {
        return false;
    }
    entry.descriptor = reinterpret_cast<void *>(static_cast<uintptr_t>(descriptor));
    entry.workspace_bytes = static_cast<size_t>(bytes);
    entry.plan = plan; // the reference goes with it
    return true;
}

int callLibrary(int kind, const Entry &e, void *workspace, void *const *p, void *stream) {
    using V = void *;
    using C = const void *;
    void *const fn = g_library.run[kind];
    switch (kind) {
    case 0: return reinterpret_cast<int (*)(V, V, size_t, V, C, C, C, C, C, C, V)>(fn)(e.descriptor, workspace, e.workspace_bytes, p[0], p[1], p[2], p[3], p[4], p[5], p[6], stream);
    case 1: return reinterpret_cast<int (*)(V, V, size_t, V, C, C, C, C, C, C, C, V)>(fn)(e.descriptor, workspace, e.workspace_bytes, p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], stream);
    case 3: return reinterpret_cast<int (*)(V, V, size_t, V, V, C, C, C, C, C, C, V)>(fn)(e.descriptor, workspace, e.workspace_bytes, p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], stream);
    case 4: return reinterpret_cast<int (*)(V, V, size_t, V, C, V, V, C, C, C, C, C, C, V)>(fn)(e.descriptor, workspace, e.workspace_bytes, p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], stream);
    default: return reinterpret_cast<int (*)(V, V, size_t, V, V, C, C, C, V)>(fn)(e.descriptor, workspace, e.workspace_bytes, p[0], p[1], p[2], p[3], p[4], stream);
    }
}

struct WithoutInterpreterLock {
    PyThreadState *const state = PyEval_SaveThread();
    ~WithoutInterpreterLock() { PyEval_RestoreThread(state); }
};

// The capture a stream is part of; 0 where it is not capturing.
unsigned long long captureOf(hipStream_t stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    if (stream == nullptr) { // cannot be captured, and may not be asked while another stream is
        return 0;
    }
    if (hipStreamGetCaptureInfo(stream, &status, &id) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return status == hipStreamCaptureStatusActive ? id : 0;
}

// setup(run function addresses, address of infinirtSetDevice, device type, plans kept)
PyObject *setup(PyObject *, PyObject *args) {
    PyObject *functions;
    unsigned long long set_device;
    int device_type;
    Py_ssize_t capacity;
    if (!PyArg_ParseTuple(args, "O!Kin", &PyTuple_Type, &functions, &set_device, &device_type, &capacity)) {
        return nullptr;
    }
    if (PyTuple_GET_SIZE(functions) != kNumOperators) {
        PyErr_SetString(PyExc_ValueError, "one function per operator expected");
        return nullptr;
    }
    for (int i = 0; i < kNumOperators; ++i) {
        g_library.run[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(functions, i));
    }
    if (PyErr_Occurred()) {
        return nullptr;
    }
    g_library.set_device = reinterpret_cast<SetDevice>(static_cast<uintptr_t>(set_device));
    g_library.device_type = device_type;
    g_library.ready = true;
    cache().setCapacity(static_cast<size_t>(capacity));
    Py_RETURN_NONE;
}

// call(operator, number, make, tensor or None ...) -> the first tensor, or the status as a number where it says failure
// `number` is the scale or the algorithm; make(number, *tensors) returns a plan, called when there is none yet.
PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    const long kind = nargs >= 3 ? PyLong_AsLong(args[0]) : -1;
    if (kind < 0 || kind >= kNumOperators || nargs != 3 + kOperators[kind].tensors || !g_library.ready) {
        if (!PyErr_Occurred()) {
            PyErr_SetString(PyExc_TypeError, "call(operator, number, make, tensors...)");
        }
        return nullptr;
    }
    const Operator &op = kOperators[kind];
    const double number = PyFloat_AsDouble(args[1]);
    if (number == -1.0 && PyErr_Occurred()) {
        return nullptr;
    }
    const at::Tensor *t[kMaxTensors];
    for (int i = 0; i < op.tensors; ++i) {
        PyObject *x = args[3 + i];
        if (x == Py_None && ((i == 0 && op.has_out) || (i == op.tensors - 1 && op.last_optional))) {
            t[i] = nullptr;
        } else if (THPVariable_Check(x)) {
            t[i] = &THPVariable_Unpack(x);
        } else {
            PyErr_Format(PyExc_TypeError, "a tensor expected, not %s", Py_TYPE(x)->tp_name);
            return nullptr;
        }
    }
    const at::Tensor &on = *t[op.device_tensor];
    if (!on.is_cuda()) {
        PyErr_SetString(PyExc_ValueError, "infinicore_amd.ops works on CUDA (HIP) tensors only; there is no host fallback");
        return nullptr;
    }
    const c10::DeviceIndex device = on.device().index();
    at::Tensor allocated;
    if (op.has_out && t[0] == nullptr) {
        if (t[3]->dim() == 0) {
            PyErr_SetString(PyExc_IndexError, "v_cache has no dimensions");
            return nullptr;
        }
        // (a query without dimensions is refused by the operator, with its status)
        c10::DimVector shape(on.sizes().begin(), on.sizes().begin() + std::max<int64_t>(on.dim() - 1, 0));
        shape.push_back(t[3]->size(-1));
        allocated = at::empty(shape, at::TensorOptions().dtype(on.scalar_type()).device(on.device()));
        t[0] = &allocated;
    }
    const hipStream_t stream = c10::hip::getCurrentHIPStream(device).stream();

    MetaKey key;
    key.words.reserve(128);
    int64_t bits;
    std::memcpy(&bits, &number, sizeof(bits));
    key.add(kind);
    key.add(device);
    key.add(static_cast<int64_t>(reinterpret_cast<uintptr_t>(stream)));
    key.add(bits);
    void *pointers[kMaxTensors];
    for (int i = 0; i < op.tensors; ++i) {
        if (t[i] == nullptr) {
            key.add(-1);
            pointers[i] = nullptr;
            continue;
        }
        key.add(static_cast<int64_t>(t[i]->scalar_type()));
        key.add(t[i]->dim());
        const auto sizes = t[i]->sizes(), strides = t[i]->strides();
        key.words.insert(key.words.end(), sizes.begin(), sizes.end());
        key.words.insert(key.words.end(), strides.begin(), strides.end());
        pointers[i] = t[i]->data_ptr();
    }

    EntryPtr entry;
    if (auto found = cache().get(key)) {
        entry = std::move(*found);
    } else {
        std::vector<PyObject *> make_args(1 + op.tensors);
        make_args[0] = args[1];
        for (int i = 0; i < op.tensors; ++i) {
            make_args[1 + i] = args[3 + i];
        }
        PyObject *wrapped = nullptr;
        if (allocated.defined()) {
            wrapped = THPVariable_Wrap(allocated);
            if (wrapped == nullptr) {
                return nullptr;
            }
            make_args[1] = wrapped;
        }
        PyObject *plan = PyObject_Vectorcall(args[2], make_args.data(), make_args.size(), nullptr);
        Py_XDECREF(wrapped);
        if (plan == nullptr) {
            return nullptr;
        }
        entry = std::make_shared<Entry>();
        if (!readPlan(plan, *entry)) {
            Py_DECREF(plan);
            return nullptr;
        }
        if (auto raced = cache().get(key)) { // another thread made one while this one was in Python
            entry = std::move(*raced);
        } else {
            cache().put(key, entry);
        }
    }

    int status;
    {
        const WithoutInterpreterLock unlocked; // (also while an allocation waits for the device)
        status = g_library.set_device(g_library.device_type, device);
        const auto allocate = [&] { return c10::hip::HIPCachingAllocator::get()->allocate(entry->workspace_bytes); }; // of the current stream
        if (status == 0 && entry->workspace_bytes == 0) {
            status = callLibrary(static_cast<int>(kind), *entry, nullptr, pointers, stream);
        } else if (status == 0 && !op.keeps_scratch) {
            const c10::DataPtr scratch = allocate();
            status = callLibrary(static_cast<int>(kind), *entry, scratch.get(), pointers, stream);
        } else if (status == 0) {
            const unsigned long long capture = captureOf(stream);
            const std::lock_guard<std::mutex> lock(entry->turn);
            c10::DataPtr &scratch = capture != 0 ? entry->captured_scratch : entry->scratch;
            if (capture != 0 && capture != entry->capture) {
                scratch.clear();
                entry->capture = capture;
            }
            if (!scratch) {
                scratch = allocate();
            }
            status = callLibrary(static_cast<int>(kind), *entry, scratch.get(), pointers, stream);
        }
    }
    entry.reset();
    if (!g_retired.empty()) {
        closeRetired();
    }
    PyObject *first;
    if (allocated.defined()) {
        first = THPVariable_Wrap(allocated);
        if (first == nullptr) {
            return nullptr;
        }
    } else {
        first = args[3];
        Py_INCREF(first);
    }
    if (status != 0) {
        Py_DECREF(first);
        return PyLong_FromLong(status);
    }
    return first;
    END_HANDLE_TH_ERRORS
}

PyObject *clear(PyObject *, PyObject *) {
    cache().clear();
    closeRetired();
    Py_RETURN_NONE;
}

PyObject *size(PyObject *, PyObject *) { return PyLong_FromSize_t(cache().size()); }

PyMethodDef kMethods[] = {
    {"setup", setup, METH_VARARGS, nullptr},
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call)), METH_FASTCALL, nullptr},
    {"clear", clear, METH_NOARGS, nullptr},
    {"size", size, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_torch_ops", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

} // namespace

extern "C" __attribute__((visibility("default"))) PyObject *PyInit__torch_ops() { return PyModule_Create(&kModule); }
