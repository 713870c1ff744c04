// The host side of a mixer call: quamba_amd._host.Plan.
//
// One decode step of one sequence is four to six kernels of 3-5 us; gathering the layer's tensors, checking that nothing
// has changed and filling the parameter block cost 13-17 us of that in Python.  A Plan holds the parameter block of a
// layer (qa_mamba1_* / qa_mamba2_*, include/quamba_amd.h) together with what it was made from - the sub-modules, their
// buffers (the tensor objects and their addresses), the scalars they carry, their hooks - and run() verifies all of it,
// allocates output and workspace, and enqueues the layer.
//
// run(hidden, conv_state, ssm_state, step) returns the output tensor; None when the library call does not cover these
// arguments (the mixer then runs its modules one by one); False when the layer is not the one the plan was made from any
// more; a status code when the library refused.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <map>
#include <tuple>
#include <vector>

#include "../../include/quamba_amd.h"

namespace {

struct Buffer {
    PyObject* object;          // a tensor or None
    const void* address;
};

struct Module {
    PyObject *name, *module, *dict, *buffers_dict;
    std::vector<Buffer> buffers;
};

struct Scalar {
    PyObject *dict, *key, *value;
};

using Forward = int (*)(const void*, void*);
using Workspace = int64_t (*)(const void*, int);

struct State {
    PyObject* modules = nullptr;               // the mixer's own dict of sub-modules
    std::vector<Module> parts;
    std::vector<Scalar> scalars;
    std::vector<PyObject*> no_hooks;           // dicts that have to be empty: global hooks
    bool usable = false;
    int family = 1;
    QaMamba1Params m1;
    QaMamba2Params m2;
    Forward fns[2] = {nullptr, nullptr};
    Workspace workspace = nullptr;
    std::vector<int64_t> ssm_shape;
    int64_t conv_dim = 0, widths[2][2] = {{0, 0}, {0, 0}};
    int64_t d_model = 0, n_out = 0, pad_out = 0;
    at::Device device = at::Device(at::kCPU);
    PyObject *get_device = nullptr, *set_device = nullptr, *get_stream = nullptr, *oom = nullptr;
    std::map<std::tuple<int64_t, int64_t, int>, int64_t> bytes;
};

struct PlanObject {
    PyObject_HEAD
    State* s;
};

PyObject *s_buffers, *s_hooks, *s_pre_hooks;   // interned attribute names

const void* address_of(PyObject* t) { return t == Py_None ? nullptr : THPVariable_Unpack(t).const_data_ptr(); }

// ---- making a plan ------------------------------------------------------------------------------------------------
PyObject* keep(PyObject* o) {
    Py_XINCREF(o);
    return o;
}

void plan_free(State* s) {
    if (!s) return;
    Py_XDECREF(s->modules);
    for (auto& m : s->parts) {
        Py_XDECREF(m.name); Py_XDECREF(m.module); Py_XDECREF(m.dict); Py_XDECREF(m.buffers_dict);
        for (auto& b : m.buffers) Py_XDECREF(b.object);
    }
    for (auto& c : s->scalars) { Py_XDECREF(c.dict); Py_XDECREF(c.key); Py_XDECREF(c.value); }
    for (PyObject* d : s->no_hooks) Py_XDECREF(d);
    Py_XDECREF(s->get_device); Py_XDECREF(s->set_device); Py_XDECREF(s->get_stream); Py_XDECREF(s->oom);
    delete s;
}

// Plan(modules_dict, names, scalars, global_hook_dicts, native): scalars are (dict, key) pairs; native is None for a layer
// the library does not cover, or (family, block bytes, (forward, step, workspace) addresses, (conv channels, state shape,
// (forward widths, step widths)), output padding, a tensor on the layer's device, (get_device, set_device, get_stream, out-of-memory error)).
int plan_init(PlanObject* self, PyObject* args, PyObject*) {
    PyObject *modules, *names, *scalars, *hooks, *native;
    if (!PyArg_ParseTuple(args, "O!O!O!O!O", &PyDict_Type, &modules, &PyTuple_Type, &names, &PyTuple_Type, &scalars, &PyTuple_Type, &hooks, &native)) return -1;
    State* s = new State;
    plan_free(self->s);
    self->s = s;
    s->modules = keep(modules);
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(names); ++i) {
        Module m = {};
        m.name = keep(PyTuple_GET_ITEM(names, i));
        m.module = keep(PyDict_GetItem(modules, m.name));
        m.dict = m.module ? PyObject_GenericGetDict(m.module, nullptr) : nullptr;
        m.buffers_dict = m.dict ? keep(PyDict_GetItem(m.dict, s_buffers)) : nullptr;
        s->parts.push_back(m);
        if (!m.buffers_dict || !PyDict_Check(m.buffers_dict)) {
            PyErr_SetString(PyExc_TypeError, "not a module of the layer");
            return -1;
        }
        PyObject *key, *value;
        Py_ssize_t pos = 0;
        while (PyDict_Next(m.buffers_dict, &pos, &key, &value)) {
            if (value != Py_None && !THPVariable_Check(value)) {
                PyErr_SetString(PyExc_TypeError, "a buffer that is no tensor");
                return -1;
            }
            s->parts.back().buffers.push_back({keep(value), address_of(value)});
        }
    }
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(scalars); ++i) {
        PyObject *dict, *key;
        if (!PyArg_ParseTuple(PyTuple_GET_ITEM(scalars, i), "O!O", &PyDict_Type, &dict, &key)) return -1;
        s->scalars.push_back({keep(dict), keep(key), keep(PyDict_GetItem(dict, key))});
    }
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(hooks); ++i) s->no_hooks.push_back(keep(PyTuple_GET_ITEM(hooks, i)));
    if (native == Py_None) return 0;

    const char* block;
    Py_ssize_t block_len;
    unsigned long long fwd, step, ws;
    long long conv_dim, f0, f1, t0, t1, pad;
    PyObject *shape, *anchor;
    if (!PyArg_ParseTuple(native, "iy#(KKK)(LO!((LL)(LL)))LO(OOOO)", &s->family, &block, &block_len, &fwd, &step, &ws, &conv_dim, &PyTuple_Type, &shape,
                          &f0, &f1, &t0, &t1, &pad, &anchor, &s->get_device, &s->set_device, &s->get_stream, &s->oom)) {
        s->get_device = s->set_device = s->get_stream = s->oom = nullptr;
        return -1;
    }
    keep(s->get_device); keep(s->set_device); keep(s->get_stream); keep(s->oom);
    const size_t want = s->family == 1 ? sizeof(QaMamba1Params) : sizeof(QaMamba2Params);
    if (static_cast<size_t>(block_len) != want || !THPVariable_Check(anchor)) {
        PyErr_SetString(PyExc_TypeError, "not a parameter block of this layer");
        return -1;
    }
    if (s->family == 1) std::memcpy(&s->m1, block, want);
    else std::memcpy(&s->m2, block, want);
    s->fns[0] = reinterpret_cast<Forward>(static_cast<uintptr_t>(fwd));
    s->fns[1] = reinterpret_cast<Forward>(static_cast<uintptr_t>(step));
    s->workspace = reinterpret_cast<Workspace>(static_cast<uintptr_t>(ws));
    s->conv_dim = conv_dim;
    s->widths[0][0] = f0; s->widths[0][1] = f1; s->widths[1][0] = t0; s->widths[1][1] = t1;
    s->pad_out = pad;
    s->d_model = s->family == 1 ? s->m1.d_model : s->m2.d_model;
    s->n_out = s->family == 1 ? s->m1.out_proj.n : s->m2.out_proj.n;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(shape); ++i) s->ssm_shape.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(shape, i)));
    s->device = THPVariable_Unpack(anchor).device();
    s->usable = true;
    return 0;
}

// ---- using it -----------------------------------------------------------------------------------------------------
bool same_value(PyObject* a, PyObject* b) {
    if (a == b) return true;
    if (!a || !b) return false;
    if (PyFloat_CheckExact(a) && PyFloat_CheckExact(b)) return PyFloat_AS_DOUBLE(a) == PyFloat_AS_DOUBLE(b);
    if (PyLong_CheckExact(a) && PyLong_CheckExact(b)) return PyObject_RichCompareBool(a, b, Py_EQ) == 1;
    return false;
}

bool hooked(PyObject* dict, PyObject* name) {
    PyObject* d = PyDict_GetItem(dict, name);
    return d && PyDict_Check(d) && PyDict_GET_SIZE(d) != 0;
}

// 1: the layer the plan was made from; 0: it has changed; -1: unchanged but hooked
int verify(const State& s) {
    bool with_hooks = false;
    for (PyObject* d : s.no_hooks) with_hooks = with_hooks || PyDict_GET_SIZE(d) != 0;
    for (const Module& m : s.parts) {
        if (PyDict_GetItem(s.modules, m.name) != m.module || PyDict_GetItem(m.dict, s_buffers) != m.buffers_dict) return 0;
        if (PyDict_GET_SIZE(m.buffers_dict) != static_cast<Py_ssize_t>(m.buffers.size())) return 0;
        PyObject *key, *value;
        Py_ssize_t pos = 0;
        size_t i = 0;
        while (PyDict_Next(m.buffers_dict, &pos, &key, &value)) {
            const Buffer& b = m.buffers[i++];
            if (value != b.object || (value != Py_None && address_of(value) != b.address)) return 0;
        }
        with_hooks = with_hooks || hooked(m.dict, s_hooks) || hooked(m.dict, s_pre_hooks);
    }
    for (const Scalar& c : s.scalars)
        if (!same_value(PyDict_GetItem(c.dict, c.key), c.value)) return 0;
    return with_hooks ? -1 : 1;
}

template <class Params>
PyObject* enqueue(State& s, Params p, const at::Tensor& hidden, PyObject* conv_o, PyObject* ssm_o, int step) {
    const int64_t batch = hidden.size(0), len = hidden.size(1);
    p.batch = static_cast<int32_t>(batch);
    p.seqlen = static_cast<int32_t>(len);
    p.hidden = hidden.const_data_ptr<int8_t>();
    if (conv_o != Py_None) {
        const at::Tensor& c = THPVariable_Unpack(conv_o);
        if (c.scalar_type() != at::kChar || c.device() != s.device || c.dim() != 3 || c.size(0) != batch || c.size(1) != s.conv_dim ||
            (c.size(2) != s.widths[step][0] && c.size(2) != s.widths[step][1])) Py_RETURN_NONE;
        p.conv_state = c.data_ptr<int8_t>();
        p.conv_state_len = static_cast<int32_t>(c.size(2));
        p.conv_state_batch_stride = c.stride(0); p.conv_state_c_stride = c.stride(1); p.conv_state_l_stride = c.stride(2);
    }
    if (ssm_o != Py_None) {
        const at::Tensor& t = THPVariable_Unpack(ssm_o);
        const bool fp32 = t.scalar_type() == at::kFloat;
        if ((!fp32 && t.scalar_type() != at::kChar) || t.device() != s.device || !t.is_contiguous() || t.size(0) != batch ||
            !t.sizes().slice(1).equals(s.ssm_shape)) Py_RETURN_NONE;
        p.ssm_state = t.data_ptr();
        p.state_is_fp32 = fp32;
        if (reinterpret_cast<uintptr_t>(p.ssm_state) % 16 != 0) Py_RETURN_NONE;
    }
    auto& bytes = s.bytes;
    const auto key = std::make_tuple(batch, len, step);
    auto it = bytes.find(key);
    if (it == bytes.end()) {
        if (bytes.size() >= 256) bytes.clear();
        it = bytes.emplace(key, s.workspace(&p, step)).first;
    }
    if (it->second <= 0) Py_RETURN_NONE;
    const auto opts = at::TensorOptions().device(s.device);
    at::Tensor out = at::empty({batch, len, s.n_out}, opts.dtype(at::kHalf));
    at::Tensor ws = at::empty({it->second}, opts.dtype(at::kByte));
    p.out = out.data_ptr();
    p.workspace = ws.data_ptr();
    p.workspace_bytes = it->second;
    PyObject* stream_o = PyObject_CallFunction(s.get_stream, "i", static_cast<int>(s.device.index()));
    if (!stream_o) return nullptr;
    void* stream = PyLong_AsVoidPtr(stream_o);
    Py_DECREF(stream_o);
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = s.fns[step](&p, stream);
    Py_END_ALLOW_THREADS
    if (status != QA_OK) return PyLong_FromLong(status);
    if (s.pad_out) out = out.narrow(2, 0, s.n_out - s.pad_out);
    return THPVariable_Wrap(out);
}

PyObject* run_on_device(State& s, PyObject* hidden_o, PyObject* conv_o, PyObject* ssm_o, int step) {
    const at::Tensor& hidden = THPVariable_Unpack(hidden_o);
    if (hidden.scalar_type() != at::kChar || hidden.device() != s.device || hidden.dim() != 3 || !hidden.is_contiguous() ||
        hidden.size(2) != s.d_model || hidden.size(0) == 0 || hidden.size(1) == 0 || hidden.size(0) > 65535 || hidden.size(1) > 0x7fffffff) Py_RETURN_NONE;
    PyObject* at_o = PyObject_CallNoArgs(s.get_device);
    if (!at_o) return nullptr;
    const long at_dev = PyLong_AsLong(at_o);
    Py_DECREF(at_o);
    const bool move = at_dev != s.device.index();
    if (move) {
        PyObject* r = PyObject_CallFunction(s.set_device, "i", static_cast<int>(s.device.index()));
        if (!r) return nullptr;
        Py_DECREF(r);
    }
    PyObject* out = s.family == 1 ? enqueue(s, s.m1, hidden, conv_o, ssm_o, step) : enqueue(s, s.m2, hidden, conv_o, ssm_o, step);
    if (move) {
        PyObject *type, *value, *trace;
        PyErr_Fetch(&type, &value, &trace);
        PyObject* r = PyObject_CallFunction(s.set_device, "l", at_dev);
        Py_XDECREF(r);
        PyErr_Restore(type, value, trace);
    }
    return out;
}

PyObject* plan_run(PlanObject* self, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 4 || !self->s) {
        PyErr_SetString(PyExc_TypeError, "run(hidden, conv_state, ssm_state, step)");
        return nullptr;
    }
    State& s = *self->s;
    const int step = PyObject_IsTrue(args[3]);
    if (step < 0) return nullptr;
    const int same = verify(s);
    if (same == 0) Py_RETURN_FALSE;
    if (same < 0 || !s.usable || !THPVariable_Check(args[0])) Py_RETURN_NONE;
    for (int i = 1; i < 3; ++i)
        if (args[i] != Py_None && !THPVariable_Check(args[i])) Py_RETURN_NONE;
    try {
        return run_on_device(s, args[0], args[1], args[2], step);
    } catch (const c10::OutOfMemoryError& e) {
        PyErr_SetString(s.oom, e.what_without_backtrace());
        return nullptr;
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// Copies and pickles of a layer start without a plan.
PyObject* plan_reduce(PyObject*, PyObject*) { return Py_BuildValue("(O())", reinterpret_cast<PyObject*>(Py_TYPE(Py_None))); }

void plan_dealloc(PlanObject* self) {
    plan_free(self->s);
    Py_TYPE(self)->tp_free(reinterpret_cast<PyObject*>(self));
}

PyMethodDef plan_methods[] = {
    {"run", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(plan_run)), METH_FASTCALL, "Enqueues the layer."},
    {"__reduce__", plan_reduce, METH_NOARGS, "Pickles as None."},
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject PlanType = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", "Host side of the mixers' library calls.", -1, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    s_buffers = PyUnicode_InternFromString("_buffers");
    s_hooks = PyUnicode_InternFromString("_forward_hooks");
    s_pre_hooks = PyUnicode_InternFromString("_forward_pre_hooks");
    PlanType.tp_name = "quamba_amd._host.Plan";
    PlanType.tp_basicsize = sizeof(PlanObject);
    PlanType.tp_flags = Py_TPFLAGS_DEFAULT;
    PlanType.tp_new = PyType_GenericNew;
    PlanType.tp_init = reinterpret_cast<initproc>(plan_init);
    PlanType.tp_dealloc = reinterpret_cast<destructor>(plan_dealloc);
    PlanType.tp_methods = plan_methods;
    if (PyType_Ready(&PlanType) < 0) return nullptr;
    PyObject* m = PyModule_Create(&module_def);
    if (!m) return nullptr;
    Py_INCREF(&PlanType);
    if (PyModule_AddObject(m, "Plan", reinterpret_cast<PyObject*>(&PlanType)) < 0) return nullptr;
    if (PyModule_AddIntConstant(m, "ABI_VERSION", QA_ABI_VERSION) < 0) return nullptr;      // of the blocks a plan holds
    return m;
}
