// The per-call path of the Python binding (tensor_amd/capi.py) in native code: output and workspace allocation, the
// current stream and the C ABI call, for the entry points a program calls once per layer.
//
// What bounds a small layer is this path, not the GPU: its kernel and launch take 4 us, the same call through ctypes took
// 9.6 us on the host (torch.cuda.current_stream() 2.9, torch.empty from Python 1.5, ctypes argument conversion and four
// geometry queries the rest). Tensors come from torch's allocator on the current stream, as before; the GIL is released
// around the C ABI call, as ctypes does.
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/Context.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty.h>
#include <ATen/record_function.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>

#include <stdexcept>
#include <string>

#include "../../include/otter_hip_int8.h"

namespace {

PyObject* g_error = nullptr;  // capi.HipError

PyObject* raise_status(int rc) {
    PyObject* args = Py_BuildValue("(is)", rc, otter_hip_last_error());
    if (args) PyErr_SetObject(g_error ? g_error : PyExc_RuntimeError, args);
    Py_XDECREF(args);
    return nullptr;
}

// one reader for the positional arguments of a call; the first failure sets the Python error and sticks
struct Args {
    PyObject* const* a;
    bool ok = true;
    long num(int i) {
        if (!ok) return 0;
        const long v = PyLong_AsLong(a[i]);
        if (v == -1 && PyErr_Occurred()) ok = false;
        return v;
    }
    double real(int i) {
        if (!ok) return 0;
        const double v = PyFloat_AsDouble(a[i]);
        if (v == -1.0 && PyErr_Occurred()) ok = false;
        return v;
    }
    template <typename T>
    T* handle(int i) {
        if (!ok || a[i] == Py_None) return nullptr;  // a closed layer: the C ABI refuses the null handle
        void* p = PyLong_AsVoidPtr(a[i]);
        if (!p && PyErr_Occurred()) ok = false;
        return static_cast<T*>(p);
    }
    const at::Tensor* tensor(int i) {  // null for None
        if (!ok || a[i] == Py_None) return nullptr;
        if (!THPVariable_Check(a[i])) {
            PyErr_SetString(PyExc_TypeError, "a torch tensor expected");
            ok = false;
            return nullptr;
        }
        return &THPVariable_Unpack(a[i]);
    }
};

// An allocation. The dispatcher in front of it costs 0.5 us of a call's 4.6, so it is left out where nothing can be listening: no
// dispatch mode or transform of this thread, no profiler, and no deterministic filling of new memory.
at::Tensor device_empty(int64_t count, at::ScalarType dt, long device) {
    const c10::Device where(c10::DeviceType::CUDA, (c10::DeviceIndex)device);
    if (c10::impl::tls_local_dispatch_key_set().included_ == c10::default_included_set && !at::hasCallbacks() &&
        !at::globalContext().deterministicAlgorithms())
        return at::detail::empty_cuda({count}, dt, where, std::nullopt);
    return at::empty({count}, at::TensorOptions().dtype(dt).device(where));
}
at::ScalarType type_of_layout(int layout) {
    return layout <= OTTER_HIP_F32_P8 ? at::kFloat : layout <= OTTER_HIP_I8_P8 ? at::kChar : at::kInt;
}
void* stream_now() { return (void*)c10::hip::getCurrentHIPStream().stream(); }
size_t bytes_of(const at::Tensor& t) { return (size_t)t.numel() * t.element_size(); }

// A workspace that the library asks for from within a call, on this thread and without the interpreter's lock. Allocated in front of
// every call on an fp32 blob it was 0.4 us of the 5.2 that a small layer takes, for launches that quantize for themselves.
struct Workspace {
    long device;
    at::Tensor made;
    std::string error;
    bool no_memory = false;  // the error is the lack of memory: a layer may do without
    static void* make(void* self_, size_t bytes) {
        auto* self = static_cast<Workspace*>(self_);
        const PyGILState_STATE lock = PyGILState_Ensure();  // (a dispatch mode runs Python)
        void* p = nullptr;
        try {
            self->made = device_empty((int64_t)bytes, at::kChar, self->device);
            p = self->made.data_ptr();
        } catch (const c10::OutOfMemoryError& e) {
            self->fails(e.what(), true);
        } catch (python_error& e) {
            e.persist();  // (out of the interpreter, where it would outlive a call that does without)
            self->fails(e.what(), lack_of_memory(e.type));
        } catch (const std::exception& e) {
            self->fails(e.what(), false);
        }
        PyGILState_Release(lock);
        return p;
    }
    static bool lack_of_memory(PyObject* type) {  // torch.OutOfMemoryError, the form that it has behind a dispatch mode
        PyObject* const torch = PyImport_ImportModule("torch");
        PyObject* const of = torch ? PyObject_GetAttrString(torch, "OutOfMemoryError") : nullptr;
        const bool is = of && type && PyErr_GivenExceptionMatches(type, of);
        Py_XDECREF(of), Py_XDECREF(torch), PyErr_Clear();
        return is;
    }
    void fails(const char* what, bool memory) { error = *what ? what : "no workspace", no_memory = memory; }
};

#define NEED(n)                                                                 \
    if (nargs != (n)) {                                                         \
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");          \
        return nullptr;                                                         \
    }

// the tensor behind `given`, or a new one when the caller gave none
PyObject* result(PyObject* given, const at::Tensor& t) {
    if (given != Py_None) {
        Py_INCREF(given);
        return given;
    }
    return THPVariable_Wrap(t);
}

// (handle, K, x, in_layout, n, h, w, out_layout or None, out or None, workspace or None, device)
PyObject* conv_forward(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    NEED(11)
    try {
        Args g{a};
        auto* h = g.handle<otter_hip_conv_t>(0);
        const long K = g.num(1);
        const at::Tensor* x = g.tensor(2);
        const int in_layout = (int)g.num(3), n = (int)g.num(4), ih = (int)g.num(5), iw = (int)g.num(6);
        const int out_layout = a[7] == Py_None ? otter_hip_conv_default_out_layout(h) : (int)g.num(7);
        const at::Tensor *out = g.tensor(8), *ws = g.tensor(9);
        const long device = g.num(10);
        if (!g.ok) return nullptr;
        if (out_layout < 0) return raise_status(out_layout);
        int oh = 0, ow = 0;
        int rc = otter_hip_conv_output_shape(h, ih, iw, &oh, &ow);
        if (rc) return raise_status(rc);
        at::Tensor made;
        Workspace made_ws{device};
        if (!out) out = &(made = device_empty((int64_t)n * K * oh * ow, type_of_layout(out_layout), device));
        void* stream = stream_now();
        const void* px = x ? x->data_ptr() : nullptr;
        void *po = out->data_ptr(), *pw = ws ? ws->data_ptr() : nullptr;
        const size_t wb = ws ? bytes_of(*ws) : 0;
        Py_BEGIN_ALLOW_THREADS
        rc = ws ? otter_hip_conv_forward(h, px, in_layout, n, ih, iw, po, out_layout, pw, wb, stream)
                : otter_hip_conv_forward_making(h, px, in_layout, n, ih, iw, po, out_layout, Workspace::make, &made_ws, stream);
        Py_END_ALLOW_THREADS
        if (!made_ws.error.empty() && (rc || !made_ws.no_memory)) throw std::runtime_error(made_ws.error);
        if (rc) return raise_status(rc);
        return result(a[8], *out);
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// (handles, K of the last layer, x, n, h, w, out or None, workspace or None, device)
PyObject* conv_chain(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    NEED(9)
    try {
        Args g{a};
        PyObject* seq = PySequence_Fast(a[0], "a sequence of layer handles expected");
        if (!seq) return nullptr;
        std::vector<const otter_hip_conv_t*> hs((size_t)PySequence_Fast_GET_SIZE(seq));
        Args gh{PySequence_Fast_ITEMS(seq)};
        for (size_t i = 0; i < hs.size(); ++i) hs[i] = gh.handle<otter_hip_conv_t>((int)i);
        Py_DECREF(seq);
        const long K = g.num(1);
        const at::Tensor* x = g.tensor(2);
        const int n = (int)g.num(3), ih = (int)g.num(4), iw = (int)g.num(5);
        const at::Tensor *out = g.tensor(6), *ws = g.tensor(7);
        const long device = g.num(8);
        if (!g.ok || !gh.ok) return nullptr;
        int rc, oh = ih, ow = iw;
        for (const auto* h : hs)
            if ((rc = otter_hip_conv_output_shape(h, oh, ow, &oh, &ow))) return raise_status(rc);
        at::Tensor made, made_ws;
        if (!ws) {
            const size_t need = otter_hip_conv_chain_workspace_bytes(hs.data(), (int)hs.size(), n, ih, iw);
            if (need) ws = &(made_ws = device_empty((int64_t)need, at::kChar, device));
        }
        if (!out) out = &(made = device_empty((int64_t)n * K * oh * ow, at::kChar, device));
        void* stream = stream_now();
        const void* px = x ? x->data_ptr() : nullptr;
        void *po = out->data_ptr(), *pw = ws ? ws->data_ptr() : nullptr;
        const size_t wb = ws ? bytes_of(*ws) : 0;
        Py_BEGIN_ALLOW_THREADS
        rc = otter_hip_conv_chain_forward(hs.data(), (int)hs.size(), px, n, ih, iw, po, pw, wb, stream);
        Py_END_ALLOW_THREADS
        if (rc) return raise_status(rc);
        return result(a[6], *out);
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// The form of a block that a single call runs in, or 0: as otter_hip_conv_block_launches says. The cost models of
// otter_hip_conv_block_fastest are of the launches alone; of the host's time one launch takes 6.5 us a call, two 8.5 and three 11.
// Their choice is taken where it is no more launches (128 -> 768 -> 128 on one 13x13 image 11.4 us a call in three, 8.3 in two;
// 160 -> 960 -> 208 on 25 8x8 images 15.9 and 11.7). For more of them the two blobs between the layers have to be beyond 4 MB (two
// launches) and 12 MB (three), which keep the GPU busy for longer than that: 112 -> 672 -> 112 on 33 22x22 images 30.3 us in one, 24.7 in
// three; but 64 -> 384 -> 64 on 58 14x14 images, with 8.7 MB, 11.4 in one and 14.2 in three, and 24 -> 144 -> 40 on 49 10x9 images 8.9
// and 11. A workspace that is given has to hold them. (workspace: its bytes, < 0: none; *bytes: what the form needs)
int block_form(const otter_hip_conv_t* e, const otter_hip_conv_t* d, const otter_hip_conv_t* p, int n, int h, int w, int64_t workspace,
               size_t* bytes) {
    const int as_is = otter_hip_conv_block_launches(e, d, p, n, h, w);
    int form = as_is < 1 ? 0 : otter_hip_conv_block_fastest(e, d, p, n, h, w);
    if (form < 1) return 0;
    *bytes = otter_hip_conv_block_form_workspace_bytes(e, d, p, form, n, h, w);
    if (form > as_is && *bytes < ((size_t)(form == 2 ? 4 : 12) << 20))
        *bytes = otter_hip_conv_block_form_workspace_bytes(e, d, p, form = as_is, n, h, w);
    return workspace >= 0 && (size_t)workspace < *bytes ? 0 : form;
}

// (expand, depthwise, project, K, out_layout, x, n, h, w, residual or None, q_scale or None, q_round_mode, out or None,
//  q or None, workspace or None, device) -> (out, q or None)
PyObject* conv_block(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    NEED(16)
    try {
        Args g{a};
        const auto *e = g.handle<otter_hip_conv_t>(0), *d = g.handle<otter_hip_conv_t>(1), *p = g.handle<otter_hip_conv_t>(2);
        const long K = g.num(3);
        const int out_layout = (int)g.num(4);
        const at::Tensor* x = g.tensor(5);
        const int n = (int)g.num(6), ih = (int)g.num(7), iw = (int)g.num(8);
        const at::Tensor* res = g.tensor(9);
        const bool with_q = a[10] != Py_None;
        const float q_scale = with_q ? (float)g.real(10) : 0.f;
        const int q_round = (int)g.num(11);
        const at::Tensor *out = g.tensor(12), *q = g.tensor(13), *ws = g.tensor(14);
        const long device = g.num(15);
        if (!g.ok) return nullptr;
        int rc, oh = ih, ow = iw;
        for (const auto* h : {e, d, p})
            if ((rc = otter_hip_conv_output_shape(h, oh, ow, &oh, &ow))) return raise_status(rc);
        const int64_t count = (int64_t)n * K * oh * ow;
        at::Tensor made, made_q, made_ws;
        if (!out) out = &(made = device_empty(count, type_of_layout(out_layout), device));
        if (!q && with_q) q = &(made_q = device_empty(count, at::kChar, device));
        size_t need = 0;
        const bool usual = out_layout == OTTER_HIP_F32_P4 || out_layout == OTTER_HIP_I8_P8;  // (any other rules out a single launch)
        const int form = usual ? block_form(e, d, p, n, ih, iw, ws ? (int64_t)bytes_of(*ws) : -1, &need) : 0;
        if (!ws && !form) need = otter_hip_conv_block_layout_workspace_bytes(e, d, p, out_layout, n, ih, iw);
        if (!ws && need) ws = &(made_ws = device_empty((int64_t)need, at::kChar, device));
        void* stream = stream_now();
        const void* px = x ? x->data_ptr() : nullptr;
        const float* pr = res ? (const float*)res->data_ptr() : nullptr;
        void *po = out->data_ptr(), *pq = q ? q->data_ptr() : nullptr, *pw = ws ? ws->data_ptr() : nullptr;
        const size_t wb = ws ? bytes_of(*ws) : 0;
        Py_BEGIN_ALLOW_THREADS
        rc = form ? otter_hip_conv_block_forward_form(e, d, p, form, px, n, ih, iw, pr, po, out_layout, pq, q_scale, q_round, pw, wb, stream)
                      : otter_hip_conv_block_forward(e, d, p, px, n, ih, iw, pr, po, out_layout, pq, q_scale, q_round, pw, wb, stream);
        Py_END_ALLOW_THREADS
        if (rc) return raise_status(rc);
        PyObject* o = result(a[12], *out);
        PyObject* qo = nullptr;
        if (q) qo = result(a[13], *q);
        else Py_INCREF(qo = Py_None);
        if (!o || !qo) {
            Py_XDECREF(o), Py_XDECREF(qo);
            return nullptr;
        }
        PyObject* pair = PyTuple_New(2);
        if (!pair) {
            Py_DECREF(o), Py_DECREF(qo);
            return nullptr;
        }
        PyTuple_SET_ITEM(pair, 0, o);
        PyTuple_SET_ITEM(pair, 1, qo);
        return pair;
    } catch (const std::exception& ex) {
        PyErr_SetString(PyExc_RuntimeError, ex.what());
        return nullptr;
    }
}

// the current stream as an integer
PyObject* current_stream(PyObject*, PyObject*) { return PyLong_FromVoidPtr(stream_now()); }

PyObject* set_error(PyObject*, PyObject* type) {
    Py_INCREF(type);
    Py_XDECREF(g_error);
    g_error = type;
    Py_RETURN_NONE;
}

#define FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(conv_forward), FAST(conv_chain), FAST(conv_block),
                         {"current_stream", current_stream, METH_NOARGS, nullptr},
                         {"set_error", set_error, METH_O, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_otter_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__otter_binding(void) { return PyModule_Create(&module); }
