// The host side of one-token appends in native code: what kvcomp_amd.compute._packed_append and KVCompCtx._tail_append ask of
// their tensors, and the launch, without a Python call per question.  A generated token costs a model two of these calls per layer,
// and the kernels behind them take a microsecond or three: the questions took longer than the kernels.
//
// A function returns 1 when it has queued its kernel and 0, having done nothing, for anything but plain tensors that the kernel
// takes: the callers' own code decides then.  Below 0: what the library returned.  What only Python knows (tangents being carried
// along, a trace being taken) the callers ask first.  The library is called without the interpreter's lock: a launch waits while its
// stream's queue is full (some 2700 appends behind a kernel that runs on), and Python's other threads run on meanwhile.
// A one-token append of the simulated cache takes the host 8.6 us with it (13.2 without), one of a context 5.0 (6.6), launches included.
//
//   append_dense(k, v, cos, sin, k_cache, v_cache, at)   kvc_append_dense
//   append_rows(tail, at, rows, row_bytes)               kvc_copy_rows of all of `rows` to `at` rows into `tail`
//   first_encode(counted, ...)                           a first store from the wait for its symbol counts to the encode's launch
//
// Host C++ only, over the C ABI of include/kvcomp_hip.h.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>

#include <algorithm>

#include "kvcomp_hip.h"

namespace {

// `call` without the interpreter's lock, which it is not to need; what it returned as this module's functions say it
template <class F> PyObject *unlocked(F call)
{
    int rc;
    {
        const pybind11::gil_scoped_release released;
        rc = call();
    }
    return PyLong_FromLong(rc == 0 ? 1 : rc < 0 ? rc : -rc);
}
void *stream_of(const at::Tensor &t) { return (void *)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// a tensor of no class of its own (those answer for themselves), with memory of its own behind it
const at::Tensor *plain(PyObject *o)
{
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() && !t.is_neg() && !t.is_conj() ? &t : nullptr;
}

bool recorded(const at::Tensor &t) { return t.requires_grad() && c10::GradMode::is_enabled(); }
uint64_t at_of(const at::Tensor &t) { return (uint64_t)(uintptr_t)t.data_ptr(); }

// the conditions of kvcomp_amd.compute._append_job and _packed_append
PyObject *append_dense(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 7, "append_dense(k, v, cos, sin, k_cache, v_cache, at)");
    const at::Tensor *k = plain(args[0]), *v = plain(args[1]), *kc = plain(args[4]), *vc = plain(args[5]);
    if (!k || !v || !kc || !vc || k->dim() != 4 || kc->dim() != 4) return PyLong_FromLong(0);
    const auto device = k->device();
    const auto shape = k->sizes(), held = kc->sizes();
    for (const at::Tensor *t : {k, v, kc, vc})
        if (t->scalar_type() != at::kHalf || t->device() != device || recorded(*t)) return PyLong_FromLong(0);
    const int64_t B = shape[0], H = shape[1], T = shape[2], D = shape[3];
    if (v->sizes() != shape || D % 2 != 0 || k->stride(3) != 1 || v->stride(3) != 1) return PyLong_FromLong(0);
    if (held[0] != B || held[1] != H || held[3] != D || vc->sizes() != held || !kc->is_contiguous() || !vc->is_contiguous()) return PyLong_FromLong(0);
    kvc_append_job job = {};
    if (args[2] != Py_None) {
        const at::Tensor *cos = plain(args[2]), *sin = plain(args[3]);
        if (!cos || !sin) return PyLong_FromLong(0);
        for (const at::Tensor *t : {cos, sin})
            if (t->scalar_type() != at::kHalf || t->device() != device || t->dim() != 3 || recorded(*t) || t->stride(2) != 1) return PyLong_FromLong(0);
        const auto angles = cos->sizes();
        if (sin->sizes() != angles || angles[1] != T || angles[2] != D || (angles[0] != 1 && angles[0] != B)) return PyLong_FromLong(0);
        job.d_cos = (decltype(job.d_cos))(uintptr_t)at_of(*cos);
        job.d_sin = (decltype(job.d_sin))(uintptr_t)at_of(*sin);
        job.cos_stride_b = angles[0] == 1 ? 0 : cos->stride(0);
        job.cos_stride_t = cos->stride(1);
        job.sin_stride_b = angles[0] == 1 ? 0 : sin->stride(0);
        job.sin_stride_t = sin->stride(1);
    }
    const int64_t at = PyLong_AsLongLong(args[6]);
    if (at == -1 && PyErr_Occurred()) return nullptr;
    job.d_k = (decltype(job.d_k))(uintptr_t)at_of(*k);
    job.d_v = (decltype(job.d_v))(uintptr_t)at_of(*v);
    job.d_k_cache = (decltype(job.d_k_cache))(uintptr_t)at_of(*kc);
    job.d_v_cache = (decltype(job.d_v_cache))(uintptr_t)at_of(*vc);
    job.batch = B;
    job.heads = H;
    job.tokens = T;
    job.head_dim = D;
    job.capacity = held[2];
    job.at = at;
    job.k_stride_b = k->stride(0);
    job.k_stride_h = k->stride(1);
    job.k_stride_t = k->stride(2);
    job.v_stride_b = v->stride(0);
    job.v_stride_h = v->stride(1);
    job.v_stride_t = v->stride(2);
    const c10::DeviceGuard guard(device);
    void *stream = stream_of(*k);
    return unlocked([&] { return kvc_append_dense(&job, stream); });
    END_HANDLE_TH_ERRORS
}

// the conditions of KVCompCtx._tail_append
PyObject *append_rows(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 4, "append_rows(tail, at, rows, row_bytes)");
    const at::Tensor *tail = plain(args[0]), *rows = plain(args[2]);
    if (!tail || !rows || rows->dim() != 4 || rows->device() != tail->device() || rows->scalar_type() != at::kHalf ||
        tail->scalar_type() != at::kHalf || !rows->is_contiguous() || !tail->is_contiguous() || rows->requires_grad() || tail->requires_grad())
        return PyLong_FromLong(0);
    const int64_t at = PyLong_AsLongLong(args[1]), row_bytes = PyLong_AsLongLong(args[3]);
    if ((at == -1 || row_bytes == -1) && PyErr_Occurred()) return nullptr;
    const int64_t bytes = rows->numel() * 2;
    if (bytes == 0 || row_bytes <= 0 || bytes % row_bytes != 0 || at < 0 || at * row_bytes + bytes > tail->numel() * 2) return PyLong_FromLong(0);
    const uint64_t to = at_of(*tail) + (uint64_t)(at * row_bytes), from = at_of(*rows);
    if (((to | from | (uint64_t)row_bytes) & 15) != 0) return PyLong_FromLong(0);
    const c10::DeviceGuard guard(tail->device());
    void *stream = stream_of(*tail);
    return unlocked([&] { return kvc_copy_rows((void *)(uintptr_t)to, (const void *)(uintptr_t)from, bytes, stream); });
    END_HANDLE_TH_ERRORS
}

// While the host is between a first store's counts and its encode the GPU has nothing to do, and this was some 20 us of Python (views
// of the codebook's parts, the payload buffer, the job, three calls).  Here it is the codebook (3 us), an allocation and the launches.
// (counted, smoothed_symbols, book, job, scratch, prepared, place, table_at, vectors, outcome, number, stream); book, job, scratch and
// outcome are addresses, place is the tensor for the decode tables with the codebook's parts from table_at on.  Returns (what
// kvc_counted_codebook returned, what kvc_encode_queue_book did, the payload's most bytes, its buffer or None): None where the codebook is
// not one for it (more than sixteen symbols, codes of more than seven bits), and nothing is queued then.
PyObject *first_encode(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 12, "first_encode takes twelve arguments");
    int64_t v[12] = {};
    for (int i = 0; i < 12; i++) {
        if (i == 6) continue;
        v[i] = (int64_t)PyLong_AsUnsignedLongLongMask(args[i]);
        if (PyErr_Occurred()) return nullptr;
    }
    const at::Tensor *place = plain(args[6]);
    TORCH_CHECK(place && place->scalar_type() == at::kByte && place->is_contiguous(), "place: a device uint8 tensor");
    const c10::DeviceGuard guard(place->device());
    kvc_codebook *book = (kvc_codebook *)(uintptr_t)v[2];
    kvc_encode_job *job = (kvc_encode_job *)(uintptr_t)v[3];
    void *stream = (void *)(uintptr_t)v[11];
    int counted_rc, queue_rc = 0;
    int64_t most = 0;
    at::Tensor payload;
    {
        const pybind11::gil_scoped_release released;
        counted_rc = kvc_counted_codebook((void *)(uintptr_t)v[0], (int)v[1], book, stream);
        if (!counted_rc && book->encode_bytes > 0 && book->encode_bytes <= 16 * 8 && book->max_code_bits <= 7 &&
            place->numel() >= v[7] + (book->encode_bytes + 15) / 16 * 16 + book->decode_bytes) {
            // (the same room for growing as any buffer of a context's)
            most = book->payload_bits / 8 + v[8] + 1;
            payload = at::empty({most + std::max<int64_t>(most / 4, 16)}, place->options());
            job->d_encoded = (uint8_t *)payload.data_ptr();
            job->encoded_cap = most;
            uint8_t *lut = (uint8_t *)place->data_ptr();
            queue_rc = kvc_encode_queue_book(job, (void *)(uintptr_t)v[4], (int)v[5], book, lut + v[7], lut, (uint32_t *)(uintptr_t)v[9], (uint32_t)v[10], stream);
        }
    }
    PyObject *buffer = payload.defined() ? THPVariable_Wrap(payload) : (Py_INCREF(Py_None), Py_None);
    if (!buffer) return nullptr;
    return Py_BuildValue("iiLN", counted_rc, queue_rc, (long long)most, buffer);
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"first_encode", (PyCFunction)(void (*)())first_encode, METH_FASTCALL, "a first store's codebook and the encode with it"},
    {"append_dense", (PyCFunction)(void (*)())append_dense, METH_FASTCALL, "kvc_append_dense where it takes the tensors; whether it did"},
    {"append_rows", (PyCFunction)(void (*)())append_rows, METH_FASTCALL, "kvc_copy_rows where it takes the tensors; whether it did"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "kvcomp_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_kvcomp_host(void) { return PyModule_Create(&module); }
