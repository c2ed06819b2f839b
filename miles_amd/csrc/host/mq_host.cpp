// The host side of a quantizer call in native code: output tensors, job records, submission, straight-through graph nodes.
//
// A call on a small tensor is bound by the host.  Written in Python, a converted matrix cost 6 us -- two allocations, the
// record of its job as a tuple and again as a ctypes structure, the reference that keeps each tensor alive -- and a
// straight-through node of torch.autograd.Function 41 us forward and backward, for a kernel of 3 us.  The functions here do
// the same with the same torch calls (at::empty, the current stream, a graph node) and record or submit the same mq_job.
//
// They take ordinary tensors only: of class Tensor or Parameter, dense, on the GPU, with no mode, transform, tracer or
// forward-mode level active that would have to see the operation.  For anything else they return None (or False) and the
// caller goes on in Python, which is where every argument is checked and every refusal is worded.
#include <ATen/PythonTorchFunctionTLS.h>
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
// Records the job or runs it; false with the error set if it is refused.
bool place(const mq_job& job, const at::Tensor& in, const at::Tensor* const* named, int n) {
    if (t_scope.recorder) {
        Recorder& r = *t_scope.recorder;
        if (r.jobs->empty() && r.device < 0) r.device = in.device().index();
        r.jobs->push_back(job);
        r.held->push_back(in);
        for (int i = 0; i < n; i++)
            if (named[i]) r.held->push_back(*named[i]);
        return true;
    }
    int rc;
    {
        hipStream_t stream = stream_of(in);
        pybind11::gil_scoped_release no_gil;
        rc = mq_run_jobs(&job, 1, stream);
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
    if (!place(job, *in, named, 4)) return nullptr;
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
    bool make[4];
    int count = 0;
    for (int i = 0; i < 4; i++) {
        make[i] = a[9 + i] != Py_None;
        if (make[i] && !spec_of(a[9 + i], spec[i])) Py_RETURN_NONE;
        count += make[i];
    }
    at::Tensor made[4];
    {
        pybind11::gil_scoped_release no_gil;      // (the allocator may wait for another thread)
        for (int i = 0; i < 4; i++)
            if (make[i]) made[i] = at::empty(spec[i].sizes, in->options().dtype(spec[i].dtype).requires_grad(false));
    }
    const at::Tensor* named[4] = {make[0] ? &made[0] : nullptr, make[1] ? &made[1] : nullptr, aux_in ? aux_in : make[2] ? &made[2] : nullptr,
                                  make[3] ? &made[3] : nullptr};
    const mq_job job{(int32_t)v[5], (int32_t)v[6], in->data_ptr(), data(named[0]), data(named[1]), data(named[2]), data(named[3]),
                     v[0], v[1], v[2], (int32_t)v[3], (int32_t)v[4], 0, 0};
    if (!place(job, *in, named, 4)) return nullptr;
    Owned result = owned(PyTuple_New(count));
    if (!result) return nullptr;
    for (int i = 0, at = 0; i < 4; i++)
        if (make[i]) PyTuple_SET_ITEM(result.ptr(), at++, THPVariable_Wrap(std::move(made[i])));
    return result.release().ptr();
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
        const auto options = x->options().requires_grad(false);
        s = at::empty(sizes, options.dtype(((THPDtype*)a[3])->scalar_type));
        y = at::empty(x->sizes(), options.dtype(at::kFloat8_e4m3fn));
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
        y = at::empty_like(*x);
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
        y = at::empty_like(*x);
        const at::Tensor s = at::empty(sizes, x->options().dtype(at::kFloat).requires_grad(false));
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
            images.push_back(at::empty_like(w));
            items.push_back(mq_fake_quant_item{w.data_ptr(), images.back().data_ptr(), w.numel()});
        }
        const at::Tensor partials = at::empty({(int64_t)weights.size() * words}, weights[0].options().dtype(at::kInt).requires_grad(false));
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
        y = at::empty_like(*x);
        s = at::empty({(M + bm - 1) / bm, (N + bn - 1) / bn}, x->options().requires_grad(false));
        z = at::empty_like(s);
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
