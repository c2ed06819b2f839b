// The host side of a quantizer call in native code: output tensors, job records, submission, straight-through graph nodes.
//
// A call on a small tensor is bound by the host.  Written in Python, a converted matrix cost 6 us -- two allocations, the
// record of its job as a tuple and again as a ctypes structure, the reference that keeps each tensor alive -- and a
// straight-through node of torch.autograd.Function 41 us forward and backward, for a kernel of 3 us.  The functions here do
// the same with the same torch calls (an allocation, the current stream, a graph node) and record or submit the same mq_job;
// for the quantizers that converters call on every matrix, the checks and sizes as well.
//
// They take ordinary tensors only: of class Tensor or Parameter, dense, on the GPU, with no mode, transform, tracer or
// forward-mode level active that would have to see the operation.  For anything else they return None (or False) and the
// caller goes on in Python, which is where every argument is checked and every refusal is worded.
#include <ATen/Context.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <vector>

#include "../../../include/miles_quant.h"

namespace {

PyObject* g_error = nullptr;      // MilesQuantError

using Owned = pybind11::object;
Owned owned(PyObject* o) { return pybind11::reinterpret_steal<Owned>(o); }

// ---- which tensors and which moments are ordinary ------------------------------------------------------------------
const c10::DispatchKeySet& special_keys() {
    using c10::DispatchKey;
    static const c10::DispatchKeySet keys({DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::PythonDispatcher,
                                           DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::FuncTorchDynamicLayerBackMode,
                                           DispatchKey::FuncTorchGradWrapper, DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchVmapMode,
                                           DispatchKey::Batched, DispatchKey::VmapMode, DispatchKey::Functionalize, DispatchKey::Conjugate,
                                           DispatchKey::Negative, DispatchKey::ZeroTensor, DispatchKey::Tracer, DispatchKey::DeferredInit});
    return keys;
}
bool ordinary_moment() {
    return !c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled() && !torch::jit::tracer::isTracing() &&
           !c10::impl::tls_local_dispatch_key_set().included_.has_any(special_keys());
}
// the tensor of an object that is an ordinary one, else null
const at::Tensor* ordinary(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.is_quantized() && !t.key_set().has_any(special_keys()) ? &t : nullptr;
}
hipStream_t stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
int dtype_code(at::ScalarType t) { return t == at::kBFloat16 ? MQ_BF16 : t == at::kHalf ? MQ_F16 : t == at::kFloat ? MQ_F32 : -1; }

// at::empty on the device of `like`, without the dispatcher (0.3 us a call), whose modes and transforms no ordinary moment has;
// where uninitialised memory is to be filled, that is the dispatched function's business
at::Tensor make(at::IntArrayRef sizes, at::ScalarType dtype, const at::Tensor& like) {
    if (at::globalContext().deterministicAlgorithms()) return at::empty(sizes, like.options().dtype(dtype).requires_grad(false));
    return at::Tensor(at::detail::empty_cuda(sizes, dtype, like.device(), c10::nullopt));
}

// at::empty_like of a tensor whose memory is one run
at::Tensor make_like(const at::Tensor& x) {
    at::Tensor y = make(x.sizes(), x.scalar_type(), x);
    return y.strides() == x.strides() ? y : at::empty_like(x);      // (dimensions of size 1 have any stride)
}

PyObject* failed() {
    PyErr_SetString(g_error ? g_error : PyExc_RuntimeError, mq_last_error());
    return nullptr;
}

// ---- job lists -------------------------------------------------------------------------------------------------------
// The jobs of a `deferred()` block and the tensors they name.  The block's Python object takes them over (`take`) when it has
// to look at them or to add one of its own.
struct Recorder {
    PyObject_HEAD
    std::vector<mq_job>* jobs;
    std::vector<at::Tensor>* held;
    c10::DeviceIndex device;          // of the first job's input
};
// What jobs of this thread do: run at once, join the list of a block, or (a recording that a caller keeps) be left to Python.
struct Scope {
    Recorder* recorder = nullptr;
    bool recording = false;
};
thread_local Scope t_scope;

void recorder_free(PyObject* self) {
    Recorder* r = (Recorder*)self;
    delete r->jobs;
    delete r->held;
    PyTypeObject* type = Py_TYPE(self);
    type->tp_free(self);
    Py_DECREF(type);
}
PyObject* recorder_new(PyTypeObject* type, PyObject*, PyObject*) {
    Recorder* r = (Recorder*)type->tp_alloc(type, 0);
    if (!r) return nullptr;
    r->jobs = new std::vector<mq_job>();
    r->held = new std::vector<at::Tensor>();
    r->device = -1;
    return (PyObject*)r;
}
Py_ssize_t recorder_length(PyObject* self) { return (Py_ssize_t)((Recorder*)self)->jobs->size(); }
PyObject* address(const void* p) { return p ? PyLong_FromVoidPtr(const_cast<void*>(p)) : Py_NewRef(Py_None); }
// (records as tuples in the order of mq_job's fields, tensors, device index): the list is empty afterwards
PyObject* recorder_take(PyObject* self, PyObject*) {
    HANDLE_TH_ERRORS
    Recorder* r = (Recorder*)self;
    const Owned records = owned(PyList_New((Py_ssize_t)r->jobs->size())), held = owned(PyList_New((Py_ssize_t)r->held->size()));
    if (!records || !held) return nullptr;
    for (size_t i = 0; i < r->jobs->size(); i++) {
        const mq_job& j = (*r->jobs)[i];
        PyObject* t = Py_BuildValue("(iiNNNNNLLLiiLL)", j.kind, j.dtype, address(j.in), address(j.out), address(j.scale), address(j.aux),
                                    address(j.aux2), (long long)j.rows, (long long)j.cols, (long long)j.ld, j.p0, j.p1,
                                    (long long)j.rows_per_block, (long long)j.block_stride);
        if (!t) return nullptr;
        PyList_SET_ITEM(records.ptr(), (Py_ssize_t)i, t);
    }
    for (size_t i = 0; i < r->held->size(); i++) PyList_SET_ITEM(held.ptr(), (Py_ssize_t)i, THPVariable_Wrap((*r->held)[i]));
    r->jobs->clear();
    r->held->clear();
    return Py_BuildValue("(OOi)", records.ptr(), held.ptr(), (int)r->device);
    END_HANDLE_TH_ERRORS
}
// how many of the recorded jobs are of one of the given kinds (a bit mask)
PyObject* recorder_count(PyObject* self, PyObject* mask_arg) {
    const unsigned long long mask = PyLong_AsUnsignedLongLong(mask_arg);
    if (PyErr_Occurred()) return nullptr;
    Py_ssize_t n = 0;
    for (const mq_job& j : *((Recorder*)self)->jobs) n += (mask >> j.kind) & 1;
    return PyLong_FromSsize_t(n);
}
// submits the list as it is
PyObject* recorder_run(PyObject* self, PyObject*) {
    HANDLE_TH_ERRORS
    Recorder* r = (Recorder*)self;
    int rc = MQ_OK;
    if (!r->jobs->empty()) {
        hipStream_t stream = c10::hip::getCurrentHIPStream(r->device).stream();
        pybind11::gil_scoped_release no_gil;
        rc = mq_run_jobs(r->jobs->data(), (int64_t)r->jobs->size(), stream);
    }
    if (rc != MQ_OK) return failed();
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}
PyMethodDef recorder_methods[] = {{"take", recorder_take, METH_NOARGS, nullptr},
                                  {"count", recorder_count, METH_O, nullptr},
                                  {"run", recorder_run, METH_NOARGS, nullptr},
                                  {nullptr, nullptr, 0, nullptr}};
PyType_Slot recorder_slots[] = {{Py_tp_new, (void*)recorder_new},
                                {Py_tp_dealloc, (void*)recorder_free},
                                {Py_sq_length, (void*)recorder_length},
                                {Py_tp_methods, recorder_methods},
                                {0, nullptr}};
PyType_Spec recorder_spec = {"mq_host.Recorder", sizeof(Recorder), 0, Py_TPFLAGS_DEFAULT, recorder_slots};
PyTypeObject* g_recorder_type = nullptr;

// enter(recorder | None): jobs of this thread join that list, or (None) are left to Python; leave(): they run at once again
PyObject* scope_enter(PyObject*, PyObject* o) {
    Scope next;
    if (o == Py_None) next.recording = true;
    else if (Py_TYPE(o) == g_recorder_type) next.recorder = (Recorder*)Py_NewRef(o);
    else return PyErr_Format(PyExc_TypeError, "enter: a Recorder or None");
    Py_XDECREF((PyObject*)t_scope.recorder);
    t_scope = next;
    Py_RETURN_NONE;
}
PyObject* scope_leave(PyObject*, PyObject*) {
    Py_XDECREF((PyObject*)t_scope.recorder);
    t_scope = Scope{};
    Py_RETURN_NONE;
}

// false, and no error set, for what is no integer of 64 bits: the call goes back to Python
bool integer(PyObject* o, int64_t& v) {
    v = PyLong_AsLongLong(o);
    if (v != -1 || !PyErr_Occurred()) return true;
    PyErr_Clear();
    return false;
}
// Records the jobs, which name `in` and `named`, or runs them; false with the error set if they are refused.
bool place(const mq_job* jobs, size_t count, const at::Tensor& in, const at::Tensor* const* named, int n) {
    if (t_scope.recorder) {
        Recorder& r = *t_scope.recorder;
        if (r.jobs->empty() && r.device < 0) r.device = in.device().index();
        r.jobs->insert(r.jobs->end(), jobs, jobs + count);
        r.held->push_back(in);
        for (int i = 0; i < n; i++)
            if (named[i]) r.held->push_back(*named[i]);
        return true;
    }
    int rc;
    {
        hipStream_t stream = stream_of(in);
        pybind11::gil_scoped_release no_gil;
        rc = mq_run_jobs(jobs, (int64_t)count, stream);
    }
    if (rc != MQ_OK) failed();
    return rc == MQ_OK;
}
void* data(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }

// submit(kind, dtype | None, in, out, scale, aux, aux2, rows, cols, ld, p0, p1, rows_per_block, block_stride) -> handled?
// (dtype None: that of `in`)
PyObject* submit(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 14) return PyErr_Format(PyExc_TypeError, "submit: 14 arguments");
    if (t_scope.recording) Py_RETURN_FALSE;
    const at::Tensor* in = ordinary(a[2]);
    if (!in || !ordinary_moment()) Py_RETURN_FALSE;
    const at::Tensor* named[4] = {};
    for (int i = 0; i < 4; i++)
        if (a[3 + i] != Py_None && !(named[i] = ordinary(a[3 + i]))) Py_RETURN_FALSE;
    if (!named[0]) Py_RETURN_FALSE;
    int64_t v[9];
    for (int i = 0; i < 7; i++)
        if (!integer(a[7 + i], v[i])) Py_RETURN_FALSE;
    if (!integer(a[0], v[7])) Py_RETURN_FALSE;
    if (a[1] == Py_None) v[8] = dtype_code(in->scalar_type()) < 0 ? 0 : dtype_code(in->scalar_type());
    else if (!integer(a[1], v[8])) Py_RETURN_FALSE;
    const mq_job job{(int32_t)v[7], (int32_t)v[8], in->data_ptr(), data(named[0]), data(named[1]), data(named[2]), data(named[3]),
                     v[0], v[1], v[2], (int32_t)v[3], (int32_t)v[4], v[5], v[6]};
    if (!place(&job, 1, *in, named, 4)) return nullptr;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// one output to make: (dtype, *sizes)
struct Spec {
    at::ScalarType dtype;
    c10::SmallVector<int64_t, 4> sizes;
};
bool spec_of(PyObject* o, Spec& s) {
    if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) < 1 || !THPDtype_Check(PyTuple_GET_ITEM(o, 0))) return false;
    s.dtype = ((THPDtype*)PyTuple_GET_ITEM(o, 0))->scalar_type;
    for (Py_ssize_t i = 1; i < PyTuple_GET_SIZE(o); i++) {
        int64_t v;
        if (!integer(PyTuple_GET_ITEM(o, i), v)) return false;
        s.sizes.push_back(v);
    }
    return true;
}
// Makes the outputs that `make` names, places the job on them (`aux_in` in the place of aux) and returns those that `kept` names.
PyObject* made_by(mq_job job, const at::Tensor& in, const at::Tensor* aux_in, const Spec (&spec)[4], const bool (&making)[4], const bool (&kept)[4]) {
    at::Tensor made[4];
    {
        pybind11::gil_scoped_release no_gil;      // (the allocator may wait for another thread)
        for (int i = 0; i < 4; i++)
            if (making[i]) made[i] = make(spec[i].sizes, spec[i].dtype, in);
    }
    const at::Tensor* named[4] = {making[0] ? &made[0] : nullptr, making[1] ? &made[1] : nullptr, aux_in ? aux_in : making[2] ? &made[2] : nullptr,
                                  making[3] ? &made[3] : nullptr};
    job.in = in.data_ptr();
    job.out = data(named[0]);
    job.scale = data(named[1]);
    job.aux = data(named[2]);
    job.aux2 = data(named[3]);
    if (!place(&job, 1, in, named, 4)) return nullptr;
    int count = 0;
    for (int i = 0; i < 4; i++) count += kept[i];
    Owned result = owned(PyTuple_New(count));
    if (!result) return nullptr;
    for (int i = 0, at = 0; i < 4; i++)
        if (kept[i]) PyTuple_SET_ITEM(result.ptr(), at++, THPVariable_Wrap(std::move(made[i])));
    return result.release().ptr();
}
// produce(kind, dtype | None, in, aux_in | None, rows, cols, ld, p0, p1, out, scale, aux, aux2) -> the tensors made, or None
// `out` .. `aux2` are (dtype, *sizes) or None; `aux_in` is a tensor that takes the place of `aux` in the job.
PyObject* produce(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 13) return PyErr_Format(PyExc_TypeError, "produce: 13 arguments");
    if (t_scope.recording) Py_RETURN_NONE;
    const at::Tensor* in = ordinary(a[2]);
    if (!in || !ordinary_moment()) Py_RETURN_NONE;
    const at::Tensor* aux_in = nullptr;
    if (a[3] != Py_None && !(aux_in = ordinary(a[3]))) Py_RETURN_NONE;
    int64_t v[7];
    for (int i = 0; i < 5; i++)
        if (!integer(a[4 + i], v[i])) Py_RETURN_NONE;
    if (!integer(a[0], v[5])) Py_RETURN_NONE;
    if (a[1] == Py_None) v[6] = dtype_code(in->scalar_type()) < 0 ? 0 : dtype_code(in->scalar_type());
    else if (!integer(a[1], v[6])) Py_RETURN_NONE;
    Spec spec[4];
    bool making[4];
    for (int i = 0; i < 4; i++) {
        making[i] = a[9 + i] != Py_None;
        if (making[i] && !spec_of(a[9 + i], spec[i])) Py_RETURN_NONE;
    }
    return made_by(mq_job{(int32_t)v[5], (int32_t)v[6], nullptr, nullptr, nullptr, nullptr, nullptr, v[0], v[1], v[2], (int32_t)v[3], (int32_t)v[4], 0, 0},
                   *in, aux_in, spec, making, making);
    END_HANDLE_TH_ERRORS
}

// ---- whole quantizers: the checks, sizes and job of one matrix ---------------------------------------------------------
// Each takes the usual form of its argument (see `plain`) and answers None for every other one, and for whatever it would
// have to refuse: the Python function goes on then, with the same job for what it accepts.  A recorded call, us, in
// Python and here: block FP8 3.6 / 1.8, MXFP8 3.6 / 1.7, INT4 3.4 / 1.9, with zero points 5.5 / 3.1, FP8 back to bf16 2.4 / 1.1, most of
// what is left its allocations; a stack of NVFP4 matrices, for each of them, 3.4 / 0.1.
bool recordable() { return !t_scope.recording && ordinary_moment(); }
// an ordinary tensor with elements whose memory is one run
const at::Tensor* plain(PyObject* o) {
    const at::Tensor* t = ordinary(o);
    return t && t->numel() > 0 && t->is_contiguous() ? t : nullptr;
}
const at::Tensor* plain_weight(PyObject* o) {
    const at::Tensor* t = plain(o);
    return t && t->dim() > 0 && dtype_code(t->scalar_type()) >= 0 ? t : nullptr;
}
// an ordinary weight matrix with elements, its rows any distance apart
const at::Tensor* weight_rows(PyObject* o) {
    const at::Tensor* t = ordinary(o);
    return t && t->dim() == 2 && t->numel() > 0 && t->stride(1) == 1 && dtype_code(t->scalar_type()) >= 0 ? t : nullptr;
}
bool positive(PyObject* o, int64_t& v) { return integer(o, v) && v > 0 && v <= 0x7FFFFFFF; }
// the sizes of t with the last one replaced
c10::SmallVector<int64_t, 4> sizes_to(const at::Tensor& t, int64_t last) {
    c10::SmallVector<int64_t, 4> sizes(t.sizes().begin(), t.sizes().end());
    sizes.back() = last;
    return sizes;
}
mq_job job_of(int kind, int dtype, int64_t rows, int64_t cols, int64_t ld, int64_t p0 = 0, int64_t p1 = 0) {
    return mq_job{kind, dtype, nullptr, nullptr, nullptr, nullptr, nullptr, rows, cols, ld, (int32_t)p0, (int32_t)p1, 0, 0};
}
constexpr bool kOne[4] = {true, false, false, false}, kTwo[4] = {true, true, false, false}, kThree[4] = {true, true, true, false},
               kFour[4] = {true, true, true, true}, kPackedZeros[4] = {true, true, false, true};

// block_fp8(weight, block_size)
PyObject* block_fp8(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor* w = n == 2 && recordable() ? weight_rows(a[0]) : nullptr;
    int64_t bn, bk;
    if (!w || !(PyList_CheckExact(a[1]) || PyTuple_CheckExact(a[1])) || PySequence_Fast_GET_SIZE(a[1]) < 2) Py_RETURN_NONE;
    if (!positive(PySequence_Fast_GET_ITEM(a[1], 0), bn) || !positive(PySequence_Fast_GET_ITEM(a[1], 1), bk)) Py_RETURN_NONE;
    const int64_t N = w->size(0), K = w->size(1);
    const Spec spec[4] = {{at::kFloat8_e4m3fn, {N, K}}, {at::kFloat, {(N + bn - 1) / bn, (K + bk - 1) / bk}}};
    return made_by(job_of(MQ_JOB_FP8_BLOCK, dtype_code(w->scalar_type()), N, K, w->stride(0), bn, bk), *w, nullptr, spec, kTwo, kTwo);
    END_HANDLE_TH_ERRORS
}
// scaled_fp8(weight, per_channel, floor bits of bf16, of fp16, of fp32)
PyObject* scaled_fp8(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor* w = n == 5 && recordable() ? weight_rows(a[0]) : nullptr;
    int64_t per_channel, floor_bits[3];
    if (!w || !integer(a[1], per_channel)) Py_RETURN_NONE;
    for (int i = 0; i < 3; i++)
        if (!integer(a[2 + i], floor_bits[i])) Py_RETURN_NONE;
    const int code = dtype_code(w->scalar_type());
    const int64_t N = w->size(0), K = w->size(1), unit = code == MQ_F32 ? 4 : 8;
    const bool held = per_channel && K >= unit && K <= 4096 * unit;      // rows of 16-byte units are held in registers: no workspace
    Spec spec[4] = {{at::kFloat8_e4m3fn, {N, K}}, {at::kFloat, {1}}, {at::kInt, {N > MQ_FP8_SCALED_WORDS ? N : MQ_FP8_SCALED_WORDS}}};
    if (per_channel) spec[1].sizes = {N, 1};
    const int64_t bits = floor_bits[code == MQ_BF16 ? 0 : code == MQ_F16 ? 1 : 2];
    return made_by(job_of(MQ_JOB_FP8_SCALED, code, N, K, w->stride(0), bits, per_channel != 0), *w, nullptr, spec, held ? kTwo : kThree, kTwo);
    END_HANDLE_TH_ERRORS
}
// mxfp8(weight)
PyObject* mxfp8(PyObject*, PyObject* o) {
    HANDLE_TH_ERRORS
    const at::Tensor* w = recordable() ? plain_weight(o) : nullptr;
    if (!w || w->size(-1) % 32 != 0) Py_RETURN_NONE;
    const int64_t K = w->size(-1);
    const Spec spec[4] = {{at::kFloat8_e4m3fn, sizes_to(*w, K)}, {at::kByte, sizes_to(*w, K / 32)}};
    return made_by(job_of(MQ_JOB_MXFP8, dtype_code(w->scalar_type()), w->numel() / K, K, K), *w, nullptr, spec, kTwo, kTwo);
    END_HANDLE_TH_ERRORS
}
// mxfp4(weight, group)
PyObject* mxfp4(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor* w = n == 2 && recordable() ? plain_weight(a[0]) : nullptr;
    int64_t group;
    if (!w || !positive(a[1], group) || w->size(-1) % group != 0 || w->size(-1) % 2 != 0) Py_RETURN_NONE;
    const int64_t K = w->size(-1);
    const Spec spec[4] = {{at::kByte, sizes_to(*w, K / 2)}, {at::kByte, sizes_to(*w, K / group)}};
    return made_by(job_of(MQ_JOB_MXFP4, dtype_code(w->scalar_type()), w->numel() / K, K, K, group), *w, nullptr, spec, kTwo, kTwo);
    END_HANDLE_TH_ERRORS
}
// int4(weight, group, symmetric) -> (words, scales) or (words, scales, packed zero points)
PyObject* int4(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor* w = n == 3 && recordable() ? plain_weight(a[0]) : nullptr;
    int64_t group;
    if (!w || w->dim() != 2 || !positive(a[1], group) || !PyBool_Check(a[2])) Py_RETURN_NONE;
    const bool symmetric = a[2] == Py_True;
    const int64_t M = w->size(0), K = w->size(1), groups = K / group;
    if (K % group != 0 || K % 8 != 0 || (!symmetric && (group % 8 != 0 || M % 8 != 0))) Py_RETURN_NONE;
    const Spec spec[4] = {{at::kInt, {M, K / 8}}, {w->scalar_type(), {M, groups}}, {at::kByte, {M, groups}}, {at::kInt, {groups, M / 8}}};
    return made_by(job_of(symmetric ? MQ_JOB_INT4_PACK : MQ_JOB_INT4_PACK_ASYM, dtype_code(w->scalar_type()), M, K, K, group), *w, nullptr, spec,
                   symmetric ? kTwo : kFour, symmetric ? kTwo : kPackedZeros);
    END_HANDLE_TH_ERRORS
}
// fp8_dequant(codes, scales, block) -> (values,)
PyObject* fp8_dequant(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor *x = n == 3 && recordable() ? plain(a[0]) : nullptr, *s = x ? plain(a[1]) : nullptr;
    int64_t block;
    if (!s || x->scalar_type() != at::kFloat8_e4m3fn || x->dim() != 2 || s->dim() != 2 || s->scalar_type() != at::kFloat || !positive(a[2], block))
        Py_RETURN_NONE;
    const int64_t M = x->size(0), N = x->size(1);
    const Spec spec[4] = {{at::kBFloat16, {M, N}}};
    return made_by(job_of(MQ_JOB_FP8_DEQUANT, 0, M, N, N, block), *x, s, spec, kOne, kOne);
    END_HANDLE_TH_ERRORS
}
// mxfp4_dequant(codes, scales, group) -> (values,)
PyObject* mxfp4_dequant(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor *x = n == 3 && recordable() ? plain(a[0]) : nullptr, *s = x ? plain(a[1]) : nullptr;
    int64_t group;
    if (!s || x->dim() == 0 || x->scalar_type() != at::kByte || s->scalar_type() != at::kByte || s->device() != x->device() || !positive(a[2], group))
        Py_RETURN_NONE;
    const int64_t numel = x->numel() * 2;
    if (numel % group != 0 || s->numel() != numel / group) Py_RETURN_NONE;
    const Spec spec[4] = {{at::kBFloat16, sizes_to(*x, x->size(-1) * 2)}};
    return made_by(job_of(MQ_JOB_MXFP4_DEQUANT, 0, 1, numel, numel, group), *x, s, spec, kOne, kOne);
    END_HANDLE_TH_ERRORS
}
// fp8_to_mxfp8(codes, tile scales)
PyObject* fp8_to_mxfp8(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor *x = n == 2 && recordable() ? plain(a[0]) : nullptr, *s = x ? plain(a[1]) : nullptr;
    if (!s || x->dim() != 2 || s->dim() != 2 || s->scalar_type() != at::kFloat || (x->scalar_type() != at::kFloat8_e4m3fn && x->scalar_type() != at::kByte))
        Py_RETURN_NONE;
    const int64_t N = x->size(0), K = x->size(1);
    if (K % 32 != 0 || s->size(0) < (N + 127) / 128 || s->size(1) < (K + 127) / 128) Py_RETURN_NONE;
    const Spec spec[4] = {{at::kFloat8_e4m3fn, {N, K}}, {at::kByte, {N, K / 32}}};
    return made_by(job_of(MQ_JOB_FP8_TO_MXFP8, 0, N, K, s->size(1)), *x, s, spec, kTwo, kTwo);
    END_HANDLE_TH_ERRORS
}
// mxfp4_to_fp8(codes, scale bytes)
PyObject* mxfp4_to_fp8(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor *x = n == 2 && recordable() ? plain(a[0]) : nullptr, *s = x ? plain(a[1]) : nullptr;
    if (!s || x->dim() != 2 || s->dim() != 2 || x->scalar_type() != at::kChar || s->element_size() != 1 || (uintptr_t)x->data_ptr() % 16 != 0)
        Py_RETURN_NONE;
    const int64_t M = x->size(0), K = x->size(1) * 2;
    if (M % 128 != 0 || K % 128 != 0 || s->size(0) != M || s->size(1) != K / 32) Py_RETURN_NONE;
    const Spec spec[4] = {{at::kFloat8_e4m3fn, {M, K}}, {at::kFloat, {M / 128, K / 128}}};
    return made_by(job_of(MQ_JOB_MXFP4_TO_FP8, 0, M, K, K), *x, s, spec, kTwo, kTwo);
    END_HANDLE_TH_ERRORS
}
// int4_unpack(words, scales, (rows, columns), group) -> (values,)
PyObject* int4_unpack(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor *x = n == 4 && recordable() ? plain(a[0]) : nullptr, *s = x ? plain(a[1]) : nullptr;
    int64_t M, K, group;
    if (!s || x->dim() != 2 || x->scalar_type() != at::kInt || dtype_code(s->scalar_type()) < 0 || s->dim() == 0) Py_RETURN_NONE;
    if (!PyTuple_CheckExact(a[2]) || PyTuple_GET_SIZE(a[2]) != 2 || !positive(PyTuple_GET_ITEM(a[2], 0), M) || !positive(PyTuple_GET_ITEM(a[2], 1), K) ||
        !positive(a[3], group))
        Py_RETURN_NONE;
    if (x->size(0) != M || x->size(1) != (K + 7) / 8 || K % group != 0 || s->numel() != M * (K / group)) Py_RETURN_NONE;
    const Spec spec[4] = {{at::kBFloat16, {M, K}}};
    return made_by(job_of(MQ_JOB_INT4_UNPACK, dtype_code(s->scalar_type()), M, K, K, group), *x, s, spec, kOne, kOne);
    END_HANDLE_TH_ERRORS
}
// nvfp4_stack(weights [n, M, K], e4m3_max, flags, words of a record) -> (codes, block scales, global scales): a job for each
// matrix, all in one list
PyObject* nvfp4_stack(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor* w = n == 4 && recordable() ? plain_weight(a[0]) : nullptr;
    int64_t e4m3_max, flags, words;
    if (!w || w->dim() != 3 || w->size(2) % 16 != 0 || !integer(a[1], e4m3_max) || !integer(a[2], flags) || !positive(a[3], words)) Py_RETURN_NONE;
    const int64_t count = w->size(0), M = w->size(1), K = w->size(2);
    at::Tensor q, s, g, records;
    std::vector<mq_job> jobs;
    {
        pybind11::gil_scoped_release no_gil;
        q = make({count, M, K / 2}, at::kByte, *w);
        s = make({count, M, K / 16}, at::kFloat8_e4m3fn, *w);
        g = make({count}, at::kFloat, *w);
        records = make({count, words}, at::kInt, *w);
        jobs.reserve((size_t)count);
        for (int64_t i = 0; i < count; i++) {
            mq_job job = job_of(MQ_JOB_NVFP4, dtype_code(w->scalar_type()), M, K, K, e4m3_max, flags);
            job.in = (const char*)w->data_ptr() + i * M * K * w->element_size();
            job.out = (char*)q.data_ptr() + i * M * (K / 2);
            job.scale = (char*)s.data_ptr() + i * M * (K / 16);
            job.aux = (char*)records.data_ptr() + i * words * 4;
            job.aux2 = (char*)g.data_ptr() + i * 4;
            jobs.push_back(job);
        }
    }
    const at::Tensor* const named[4] = {&q, &s, &records, &g};
    if (!place(jobs.data(), jobs.size(), *w, named, 4)) return nullptr;
    return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(q)), THPVariable_Wrap(std::move(s)), THPVariable_Wrap(std::move(g)));
    END_HANDLE_TH_ERRORS
}

// ---- calls that are no jobs: only where no list is being made ---------------------------------------------------------
bool listing() { return t_scope.recorder || t_scope.recording; }

// act_quant(x, block, flags, scale dtype) -> (codes, scales) or None; x contiguous, its last dimension a multiple of block
PyObject* act_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4) return PyErr_Format(PyExc_TypeError, "act_quant: 4 arguments");
    const at::Tensor* x = ordinary(a[0]);
    int64_t block, flags;
    if (!x || listing() || !ordinary_moment() || !x->is_contiguous() || x->dim() == 0 || dtype_code(x->scalar_type()) < 0) Py_RETURN_NONE;
    if (!integer(a[1], block) || !integer(a[2], flags)) Py_RETURN_NONE;
    if (block <= 0 || block > 0x7FFFFFFF || x->size(-1) % block != 0 || !THPDtype_Check(a[3])) Py_RETURN_NONE;
    c10::SmallVector<int64_t, 4> sizes(x->sizes().begin(), x->sizes().end());
    sizes.back() /= block;
    at::Tensor y, s;
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        s = make(sizes, ((THPDtype*)a[3])->scalar_type, *x);
        y = make(x->sizes(), at::kFloat8_e4m3fn, *x);
        rc = mq_fp8_act_quant(x->data_ptr(), dtype_code(x->scalar_type()), y.data_ptr(), s.data_ptr(), x->numel(), (int)block, (int)flags, stream_of(*x));
    }
    if (rc != MQ_OK) return failed();
    return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(y)), THPVariable_Wrap(std::move(s)));
    END_HANDLE_TH_ERRORS
}

// The image of x in front, the gradient handed back as it comes (a torch.autograd.Function of the same two lines takes the
// Python path).
struct StraightThrough : torch::autograd::Function<StraightThrough> {
    static at::Tensor forward(torch::autograd::AutogradContext*, const at::Tensor&, const at::Tensor* image) { return *image; }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext*, torch::autograd::variable_list grads) {
        return {grads[0], at::Tensor()};
    }
};
at::Tensor with_gradient_through(const at::Tensor& x, const at::Tensor& image) {
    return at::GradMode::is_enabled() && x.requires_grad() ? StraightThrough::apply(x, &image) : image;
}
// an ordinary tensor that an image of the same layout is made of
bool imageable(const at::Tensor* x) {
    return x && x->is_contiguous() && x->dim() > 0 && !x->_fw_grad(0).defined();
}
// fake_quant(x, mode, block): mq_fake_quant with the gradient handed through, or None
PyObject* fake_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3) return PyErr_Format(PyExc_TypeError, "fake_quant: 3 arguments");
    const at::Tensor* x = ordinary(a[0]);
    int64_t mode, block;
    if (listing() || !ordinary_moment() || !imageable(x) || dtype_code(x->scalar_type()) < 0) Py_RETURN_NONE;
    if (!integer(a[1], mode) || !integer(a[2], block)) Py_RETURN_NONE;
    if (block <= 0 || x->size(-1) % block != 0) Py_RETURN_NONE;
    at::Tensor y;
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        at::NoGradGuard no_grad;
        y = make_like(*x);
        rc = mq_fake_quant(x->data_ptr(), dtype_code(x->scalar_type()), y.data_ptr(), x->numel(), (int)mode, stream_of(*x));
    }
    if (rc != MQ_OK) return failed();
    return THPVariable_Wrap(with_gradient_through(*x, y));
    END_HANDLE_TH_ERRORS
}
// simulate(x, block, flags): mq_fp8_act_quant cast back in place, with the gradient handed through, or None
PyObject* simulate(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3) return PyErr_Format(PyExc_TypeError, "simulate: 3 arguments");
    const at::Tensor* x = ordinary(a[0]);
    int64_t block, flags;
    if (listing() || !ordinary_moment() || !imageable(x) || dtype_code(x->scalar_type()) < 0) Py_RETURN_NONE;
    if (!integer(a[1], block) || !integer(a[2], flags)) Py_RETURN_NONE;
    if (block <= 0 || block > 0x7FFFFFFF || x->size(-1) % block != 0) Py_RETURN_NONE;
    c10::SmallVector<int64_t, 4> sizes(x->sizes().begin(), x->sizes().end());
    sizes.back() /= block;
    at::Tensor y;
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        at::NoGradGuard no_grad;
        y = make_like(*x);
        const at::Tensor s = make(sizes, at::kFloat, *x);
        rc = mq_fp8_act_quant(x->data_ptr(), dtype_code(x->scalar_type()), y.data_ptr(), s.data_ptr(), x->numel(), (int)block, (int)flags, stream_of(*x));
    }
    if (rc != MQ_OK) return failed();
    return THPVariable_Wrap(with_gradient_through(*x, y));
    END_HANDLE_TH_ERRORS
}
// nvfp4_images(weights, block, words, e4m3_max, flags): the NVFP4 images of a list of matrices that can share launches (one
// 16-bit dtype, one device, contiguous, whole blocks, 16-byte aligned), a node for each, or None
PyObject* nvfp4_images(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5) return PyErr_Format(PyExc_TypeError, "nvfp4_images: 5 arguments");
    if (!PyList_Check(a[0]) || listing() || !ordinary_moment()) Py_RETURN_NONE;
    int64_t block, words, e4m3_max, flags;
    if (!integer(a[1], block) || !integer(a[2], words) || !integer(a[3], e4m3_max) || !integer(a[4], flags)) Py_RETURN_NONE;
    std::vector<at::Tensor> weights, images;
    std::vector<mq_fake_quant_item> items;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[0]); i++) {
        const at::Tensor* w = ordinary(PyList_GET_ITEM(a[0], i));
        if (!imageable(w) || (w->scalar_type() != at::kBFloat16 && w->scalar_type() != at::kHalf) || w->dim() != 2 || w->numel() == 0 ||
            w->size(1) % block != 0 || (uintptr_t)w->data_ptr() % 16 != 0)
            Py_RETURN_NONE;
        if (!weights.empty() && (w->scalar_type() != weights[0].scalar_type() || w->device() != weights[0].device())) Py_RETURN_NONE;
        weights.push_back(*w);
    }
    if (weights.empty()) Py_RETURN_NONE;
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        at::NoGradGuard no_grad;
        images.reserve(weights.size());
        items.reserve(weights.size());
        for (const at::Tensor& w : weights) {
            images.push_back(make_like(w));
            items.push_back(mq_fake_quant_item{w.data_ptr(), images.back().data_ptr(), w.numel()});
        }
        const at::Tensor partials = make({(int64_t)weights.size() * words}, at::kInt, weights[0]);
        rc = mq_nvfp4_fake_quant(items.data(), (int64_t)items.size(), dtype_code(weights[0].scalar_type()), partials.data_ptr(), (int)e4m3_max,
                                 (int)flags, stream_of(weights[0]));
    }
    if (rc != MQ_OK) return failed();
    Owned result = owned(PyList_New((Py_ssize_t)weights.size()));
    if (!result) return nullptr;
    for (size_t i = 0; i < weights.size(); i++)
        PyList_SET_ITEM(result.ptr(), (Py_ssize_t)i, THPVariable_Wrap(with_gradient_through(weights[i], images[i])));
    return result.release().ptr();
    END_HANDLE_TH_ERRORS
}
// int4_fake(x, block_m, block_n, symmetric) -> (values, scale, zero) or None
PyObject* int4_fake(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4) return PyErr_Format(PyExc_TypeError, "int4_fake: 4 arguments");
    const at::Tensor* x = ordinary(a[0]);
    int64_t bm, bn, sym;
    if (!x || listing() || !ordinary_moment() || x->dim() != 2 || !x->is_contiguous() || dtype_code(x->scalar_type()) < 0) Py_RETURN_NONE;
    if (!integer(a[1], bm) || !integer(a[2], bn) || !integer(a[3], sym)) Py_RETURN_NONE;
    if (bm <= 0 || bn <= 0 || bm > 0x7FFFFFFF || bn > 0x7FFFFFFF) Py_RETURN_NONE;
    at::Tensor y, s, z;
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        at::NoGradGuard no_grad;
        const int64_t M = x->size(0), N = x->size(1);
        y = make_like(*x);
        s = make({(M + bm - 1) / bm, (N + bn - 1) / bn}, x->scalar_type(), *x);
        z = make(s.sizes(), x->scalar_type(), *x);
        rc = mq_int4_fake_quant(x->data_ptr(), dtype_code(x->scalar_type()), y.data_ptr(), s.data_ptr(), z.data_ptr(), M, N, (int)bm, (int)bn,
                                (int)sym, stream_of(*x));
    }
    if (rc != MQ_OK) {
        PyErr_SetString(PyExc_RuntimeError, mq_last_error());
        return nullptr;
    }
    return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(y)), THPVariable_Wrap(std::move(s)), THPVariable_Wrap(std::move(z)));
    END_HANDLE_TH_ERRORS
}

// set_error(exception class): what a refusal by the library raises
PyObject* set_error(PyObject*, PyObject* o) {
    Py_XSETREF(g_error, Py_NewRef(o));
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"set_error", set_error, METH_O, nullptr},
                         {"enter", scope_enter, METH_O, nullptr},
                         {"leave", scope_leave, METH_NOARGS, nullptr},
                         {"submit", (PyCFunction)(void*)submit, METH_FASTCALL, nullptr},
                         {"produce", (PyCFunction)(void*)produce, METH_FASTCALL, nullptr},
                         {"block_fp8", (PyCFunction)(void*)block_fp8, METH_FASTCALL, nullptr},
                         {"scaled_fp8", (PyCFunction)(void*)scaled_fp8, METH_FASTCALL, nullptr},
                         {"mxfp8", mxfp8, METH_O, nullptr},
                         {"mxfp4", (PyCFunction)(void*)mxfp4, METH_FASTCALL, nullptr},
                         {"int4", (PyCFunction)(void*)int4, METH_FASTCALL, nullptr},
                         {"fp8_dequant", (PyCFunction)(void*)fp8_dequant, METH_FASTCALL, nullptr},
                         {"mxfp4_dequant", (PyCFunction)(void*)mxfp4_dequant, METH_FASTCALL, nullptr},
                         {"fp8_to_mxfp8", (PyCFunction)(void*)fp8_to_mxfp8, METH_FASTCALL, nullptr},
                         {"mxfp4_to_fp8", (PyCFunction)(void*)mxfp4_to_fp8, METH_FASTCALL, nullptr},
                         {"int4_unpack", (PyCFunction)(void*)int4_unpack, METH_FASTCALL, nullptr},
                         {"nvfp4_stack", (PyCFunction)(void*)nvfp4_stack, METH_FASTCALL, nullptr},
                         {"act_quant", (PyCFunction)(void*)act_quant, METH_FASTCALL, nullptr},
                         {"fake_quant", (PyCFunction)(void*)fake_quant, METH_FASTCALL, nullptr},
                         {"simulate", (PyCFunction)(void*)simulate, METH_FASTCALL, nullptr},
                         {"nvfp4_images", (PyCFunction)(void*)nvfp4_images, METH_FASTCALL, nullptr},
                         {"int4_fake", (PyCFunction)(void*)int4_fake, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "mq_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_mq_host() {
    PyObject* m = PyModule_Create(&module);
    if (!m) return nullptr;
    g_recorder_type = (PyTypeObject*)PyType_FromSpec(&recorder_spec);
    if (!g_recorder_type || PyModule_AddObjectRef(m, "Recorder", (PyObject*)g_recorder_type) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
