// The module call from Python, in C: what calling a ``QuantLinear`` does in the common case, and the bound product it runs.
//
// An eager decode step is a chain of calls of a few microseconds each: the kernel of one takes 4 to 7 us.  The way to it
// alone (nn.Module.__call__, forward's reshapes of a 3-D input, the crossing into a TorchScript class, the dispatcher's
// at::empty) took 7 us of host time on top of the 2.4 us of the launch itself.
// Here the call is one C function of the type: it looks the bound product of the row count up in the module's routes,
// checks that the module and its buffers are as they were when the route was decided, allocates y in the shape of x
// and launches.  Measured (one row, 4096 x 4096, us of host time per call of a 3-D x): 9.6 before, 3.8 now.
// Everything else (another dtype or layout, a gradient wanted, hooks, tracing, a subclass, a row count not seen
// before) goes to nn.Module.__call__ and from there to forward, as ever.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/object_ptr.h>

#include <new>

#include "binding.h"

namespace {

using namespace gptq_torch;

// ---- the bound product: BoundCall(kind, a, b, c, d, e, bias, bits, group_size, M, K, N), called with x
struct BoundCall {
    PyObject_HEAD
    Bound q;
};

PyTypeObject *g_bound_type = nullptr;

// an x that q takes as it is: fp16, dense rows of K, M of them in all, and aligned for the kernels' 16-byte loads
bool takes(const Bound &q, const Tensor &x)
{
    return x.is_cuda() && x.layout() == at::kStrided && x.has_storage() && x.scalar_type() == at::kHalf && x.dim() >= 1 &&
           x.size(-1) == q.K && x.numel() == (int64_t)q.M * q.K && x.is_contiguous() && x.get_device() == q.a.get_device() &&
           (uintptr_t)x.data_ptr() % 16 == 0;
}

// Lets other Python threads run meanwhile: an allocation or a launch can wait for the GPU, and waits for the lock of a
// workspace whose holder may itself be waiting for the interpreter (an allocator that records Python stacks).
struct WithoutInterpreter {
    PyThreadState *const state = PyEval_SaveThread();
    ~WithoutInterpreter() { PyEval_RestoreThread(state); }
};

PyObject *apply(const Bound &q, const Tensor &x)
{
    Tensor y;
    {
        const WithoutInterpreter free;
        const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
        c10::SmallVector<int64_t, 6> sizes(x.sizes().begin(), x.sizes().end());
        sizes.back() = q.N;
        y = at::detail::empty_cuda(sizes, at::kHalf, x.device(), std::nullopt);
        void *stream = (void *)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.get_device()).stream();
        raise(q.launch(x, y.data_ptr(), stream), "gptq_hip product", q.M, q.K, q.N, q.bits, q.group_size);
    }
    return THPVariable_Wrap(std::move(y));
}

OptTensor tensor_or_none(PyObject *o, const char *name)
{
    if (o == Py_None) return std::nullopt;
    TORCH_CHECK(THPVariable_Check(o), name, " must be a tensor or None");
    return THPVariable_Unpack(o);
}

PyObject *bound_new(PyTypeObject *type, PyObject *args, PyObject *)
{
    HANDLE_TH_ERRORS
    int kind, bits, gs, M, K, N;
    PyObject *a, *b, *c, *d, *e, *bias;
    if (!PyArg_ParseTuple(args, "iOOOOOOiiiii", &kind, &a, &b, &c, &d, &e, &bias, &bits, &gs, &M, &K, &N)) return nullptr;
    TORCH_CHECK(kind >= 0 && kind <= 2, "kind must be 0 (checkpoint tensors), 1 (sorted copy) or 2 (tiled copy)");
    Bound q;
    q.kind = kind, q.bits = bits, q.group_size = gs, q.M = M, q.K = K, q.N = N;
    const OptTensor ta = tensor_or_none(a, "a"), tb = tensor_or_none(b, "b"), tc = tensor_or_none(c, "c");
    TORCH_CHECK(ta && tb && (kind == 2 || tc), "the layer's tensors are missing");
    q.a = *ta, q.b = *tb, q.c = tc ? *tc : Tensor();
    q.d = tensor_or_none(d, "d"), q.e = tensor_or_none(e, "e"), q.bias = tensor_or_none(bias, "bias");
    TORCH_CHECK(kind != 1 || q.d, "the sorted copy needs its kmap");
    check_bound(q);
    raise(q.choose(), "gptq_hip plan", M, K, N, bits, gs);
    PyObject *self = type->tp_alloc(type, 0);
    if (!self) return nullptr;
    new (&((BoundCall *)self)->q) Bound(std::move(q));
    return self;
    END_HANDLE_TH_ERRORS
}

void bound_dealloc(PyObject *self)
{
    PyTypeObject *type = Py_TYPE(self);
    ((BoundCall *)self)->q.~Bound();
    type->tp_free(self);
    Py_DECREF(type);
}

PyObject *bound_call(PyObject *self, PyObject *args, PyObject *kwargs);

PyType_Slot bound_slots[] = {{Py_tp_new, (void *)bound_new},
                             {Py_tp_dealloc, (void *)bound_dealloc},
                             {Py_tp_call, (void *)bound_call},
                             {Py_tp_doc, (void *)"a layer's constant tensors bound to one row count; call it with x"},
                             {0, nullptr}};
PyType_Spec bound_spec = {"gptq_hip_call.BoundCall", sizeof(BoundCall), 0, Py_TPFLAGS_DEFAULT, bound_slots};

// ---- the call of a QuantLinear
// The function stands in the type's tp_call slot, beside the methods: QuantLinear.__call__ is still nn.Module's, for tracers
// and compilers that follow the methods.  Python fills the slot anew, with the ordinary call, whenever a __call__ is set on
// the class or on nn.Module; the first product called the ordinary way after that was undone brings the function back.
PyTypeObject *g_module_type = nullptr;   // the class the function was installed on; a subclass takes the ordinary way
ternaryfunc g_ordinary = nullptr;        // Python's own function of the slot: looks __call__ up and calls it
PyObject *g_nn_module = nullptr;         // torch.nn.Module
PyObject *g_global_hooks[4] = {};        // the four dicts of hooks on every module
PyObject *g_forward = nullptr, *g_nn_call = nullptr, *g_nn_call_impl = nullptr;   // the methods that the function stands for
PyObject *s_call, *s_call_impl, *s_routes, *s_buffers, *s_forward, *s_hooks[4], *s_watched[4], *s_compiled;

// whether a call of a module would still run them: none replaced or added on the class or on nn.Module
bool methods_untouched()
{
    PyObject *own = g_module_type->tp_dict, *nn = ((PyTypeObject *)g_nn_module)->tp_dict;
    return PyDict_GetItem(own, s_forward) == g_forward && PyDict_GetItem(nn, s_call) == g_nn_call &&
           PyDict_GetItem(nn, s_call_impl) == g_nn_call_impl && !PyDict_GetItem(own, s_call) && !PyDict_GetItem(own, s_call_impl);
}

// The bound product of a call of `self` with x (a new reference), or nullptr where the ordinary way has to decide.
PyObject *route_of(PyObject *self, const Tensor &x)
{
    if (x.dim() < 1 || x.size(-1) < 1 || (x.requires_grad() && c10::GradMode::is_enabled())) return nullptr;
    if (c10::impl::TorchDispatchModeTLS::any_modes_set() || torch::jit::tracer::isTracing()) return nullptr;
    PyObject **dictp = _PyObject_GetDictPtr(self);
    if (!dictp || !*dictp) return nullptr;
    PyObject *dict = *dictp;
    for (PyObject *h : g_global_hooks)
        if (PyDict_GET_SIZE(h) != 0) return nullptr;
    for (PyObject *name : s_hooks) {
        PyObject *h = PyDict_GetItem(dict, name);
        if (!h || !PyDict_Check(h) || PyDict_GET_SIZE(h) != 0) return nullptr;
    }
    // (a forward set on the instance, as offload hooks do, or a compiled call)
    if (PyDict_GetItem(dict, s_forward) || PyDict_GetItem(dict, s_call_impl) || PyDict_GetItem(dict, s_compiled)) return nullptr;
    if (!methods_untouched()) return nullptr;
    PyObject *routes = PyDict_GetItem(dict, s_routes), *buffers = PyDict_GetItem(dict, s_buffers);
    if (!routes || !PyDict_Check(routes) || !buffers || !PyDict_Check(buffers)) return nullptr;
    PyObject *rows = PyLong_FromLongLong((long long)(x.numel() / x.size(-1)));
    if (!rows) {
        PyErr_Clear();
        return nullptr;
    }
    PyObject *r = PyDict_GetItem(routes, rows);
    Py_DECREF(rows);
    if (!r || !PyTuple_Check(r) || PyTuple_GET_SIZE(r) != 4) return nullptr;
    PyObject *watched = PyTuple_GET_ITEM(r, 0), *fn = PyTuple_GET_ITEM(r, 3);
    if (Py_TYPE(fn) != g_bound_type || !PyTuple_Check(watched) || PyTuple_GET_SIZE(watched) != 4) return nullptr;
    // the same buffer objects, not written since (QuantLinear._fresh)
    int64_t versions = 0;
    for (int i = 0; i < 4; i++) {
        PyObject *t = PyTuple_GET_ITEM(watched, i);
        if (PyDict_GetItem(buffers, s_watched[i]) != t || !THPVariable_Check(t)) return nullptr;
        const Tensor &v = THPVariable_Unpack(t);
        if (v.is_inference()) return nullptr;
        versions += v._version();
    }
    if (PyLong_AsLongLong(PyTuple_GET_ITEM(r, 1)) != versions) return nullptr;
    if (!takes(((BoundCall *)fn)->q, x)) return nullptr;
    Py_INCREF(fn);
    return fn;
}

PyObject *module_call(PyObject *self, PyObject *args, PyObject *kwargs)
{
    HANDLE_TH_ERRORS
    if (PyTuple_GET_SIZE(args) == 1 && (!kwargs || PyDict_GET_SIZE(kwargs) == 0) && Py_TYPE(self) == g_module_type &&
        THPVariable_CheckExact(PyTuple_GET_ITEM(args, 0))) {
        const Tensor &x = THPVariable_Unpack(PyTuple_GET_ITEM(args, 0));
        if (PyObject *fn = route_of(self, x)) {
            const THPObjectPtr hold(fn);
            return apply(((BoundCall *)fn)->q, x);
        }
    }
    return g_ordinary(self, args, kwargs);
    END_HANDLE_TH_ERRORS
}

PyObject *bound_call(PyObject *self, PyObject *args, PyObject *kwargs)
{
    HANDLE_TH_ERRORS
    if (g_module_type && g_module_type->tp_call == g_ordinary && methods_untouched()) g_module_type->tp_call = module_call;
    const Bound &q = ((BoundCall *)self)->q;
    TORCH_CHECK(PyTuple_GET_SIZE(args) == 1 && (!kwargs || PyDict_GET_SIZE(kwargs) == 0) && THPVariable_Check(PyTuple_GET_ITEM(args, 0)),
                "one tensor is expected");
    const Tensor x = THPVariable_Unpack(PyTuple_GET_ITEM(args, 0));
    // what is recorded or handled by something else (torch.jit.trace, dispatch modes, tensor subclasses) is the operator
    if (!THPVariable_CheckExact(PyTuple_GET_ITEM(args, 0)) || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
        torch::jit::tracer::isTracing())
        return THPVariable_Wrap(dispatch(q, x));
    TORCH_CHECK(x.is_cuda() && x.device() == q.a.device(), "x is on ", x.device(), ", the layer on ", q.a.device(),
                ": the GPTQ kernels run on a ROCm GPU only and there is no CPU fallback");
    const Tensor rows = x.is_contiguous() ? aligned(x) : x;
    TORCH_CHECK(takes(q, rows), "x must be a contiguous fp16 tensor of ", q.M, " rows of ", q.K);
    return apply(q, rows);
    END_HANDLE_TH_ERRORS
}

// aside(fn, *args): fn(*args) hidden from torch.jit.trace and from dispatch modes.  A layer decides its routes and prepares its
// copies so: a recording that holds the allocations of a copy, and not the kernels that fill it, replays on empty memory.
PyObject *aside(PyObject *, PyObject *args)
{
    HANDLE_TH_ERRORS
    if (PyTuple_GET_SIZE(args) < 1) {
        PyErr_SetString(PyExc_TypeError, "a callable is expected");
        return nullptr;
    }
    THPObjectPtr rest(PyTuple_GetSlice(args, 1, PyTuple_GET_SIZE(args)));
    if (!rest) return nullptr;
    PyObject *fn = PyTuple_GET_ITEM(args, 0);
    if (!c10::impl::TorchDispatchModeTLS::any_modes_set() && !torch::jit::tracer::isTracing()) return PyObject_CallObject(fn, rest.get());
    struct Untraced {
        std::shared_ptr<torch::jit::tracer::TracingState> state = torch::jit::tracer::getTracingState();
        Untraced() { torch::jit::tracer::setTracingState(nullptr); }
        ~Untraced() { torch::jit::tracer::setTracingState(state); }
    } untraced;
    const c10::impl::ExcludeDispatchKeyGuard no_modes(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot}));
    return PyObject_CallObject(fn, rest.get());
    END_HANDLE_TH_ERRORS
}

// install(cls): makes module_call what runs when an instance of cls is called
PyObject *install(PyObject *, PyObject *cls)
{
    HANDLE_TH_ERRORS
    if (!PyType_Check(cls)) {
        PyErr_SetString(PyExc_TypeError, "a class is expected");
        return nullptr;
    }
    THPObjectPtr mod(PyImport_ImportModule("torch.nn.modules.module"));
    if (!mod) return nullptr;
    static const char *const globals[4] = {"_global_backward_pre_hooks", "_global_backward_hooks", "_global_forward_hooks",
                                           "_global_forward_pre_hooks"};
    for (int i = 0; i < 4; i++) {
        g_global_hooks[i] = PyObject_GetAttrString(mod.get(), globals[i]);   // kept for the life of the process
        if (!g_global_hooks[i]) return nullptr;
        if (!PyDict_Check(g_global_hooks[i])) {
            PyErr_SetString(PyExc_TypeError, globals[i]);
            return nullptr;
        }
    }
    if (!(g_nn_module = PyObject_GetAttrString(mod.get(), "Module"))) return nullptr;
    g_forward = PyDict_GetItem(((PyTypeObject *)cls)->tp_dict, s_forward);
    g_nn_call = PyDict_GetItem(((PyTypeObject *)g_nn_module)->tp_dict, s_call);
    g_nn_call_impl = PyDict_GetItem(((PyTypeObject *)g_nn_module)->tp_dict, s_call_impl);
    if (!g_forward || !g_nn_call || !g_nn_call_impl) {
        PyErr_SetString(PyExc_TypeError, "a class with a forward of its own, derived from nn.Module, is expected");
        return nullptr;
    }
    for (PyObject *method : {g_forward, g_nn_call, g_nn_call_impl}) Py_INCREF(method);
    Py_INCREF(cls);
    g_module_type = (PyTypeObject *)cls;
    if (g_module_type->tp_call != module_call) {
        g_ordinary = g_module_type->tp_call;
        g_module_type->tp_call = module_call;
    }
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

PyMethodDef functions[] = {{"aside", aside, METH_VARARGS, "aside(fn, *args): fn(*args), hidden from tracing and dispatch modes."},
                           {"install", install, METH_O, "Makes the call in C the one of a QuantLinear class."}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "gptq_hip_call", "the QuantLinear call in C", -1, functions};

}  // namespace

PyMODINIT_FUNC PyInit_gptq_hip_call()
{
    auto intern = [](const char *s) { return PyUnicode_InternFromString(s); };
    s_call = intern("__call__"), s_routes = intern("_routes"), s_buffers = intern("_buffers"), s_forward = intern("forward");
    s_call_impl = intern("_call_impl");
    s_compiled = intern("_compiled_call_impl");
    static const char *const hooks[4] = {"_backward_hooks", "_backward_pre_hooks", "_forward_hooks", "_forward_pre_hooks"};
    static const char *const watched[4] = {"qweight", "qzeros", "scales", "g_idx"};
    for (int i = 0; i < 4; i++) s_hooks[i] = intern(hooks[i]), s_watched[i] = intern(watched[i]);
    PyObject *m = PyModule_Create(&module_def);
    if (!m) return nullptr;
    g_bound_type = (PyTypeObject *)PyType_FromSpec(&bound_spec);
    if (!g_bound_type) return nullptr;
    Py_INCREF(g_bound_type);
    if (PyModule_AddObject(m, "BoundCall", (PyObject *)g_bound_type) != 0) return nullptr;
    return m;
}
