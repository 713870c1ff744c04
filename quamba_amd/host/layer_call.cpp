// The host side of a mixer call: quamba_amd._host.Plan.
//
// One decode step of one sequence is four to six kernels of 3-5 us; gathering the layer's tensors, checking that nothing
// has changed and filling the parameter block cost 13-17 us of that in Python.  A Plan holds the parameter block of a
// layer (qa_mamba1_* / qa_mamba2_*, include/quamba_amd.h) together with what it was made from, and run() verifies all of it,
// allocates output and workspace, and enqueues the layer.
//
// What it was made from is a list of dicts - the mixer's sub-modules, and of each of them its attributes, buffers and
// parameters - as they were, entry by entry: a tensor whose address is in the block is in one of them wherever the module
// keeps it, the entry keeps it alive, and every call compares the entries with what the dicts hold now (values by identity,
// numbers by value, tensors by their address as well).  The modules' classes belong to it too: another function in the place
// of a method is another layer.
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

struct Entry {
    PyObject *key, *value;
    bool tensor;
    const void* address;       // of a tensor's memory
};

struct Watch {
    PyObject* dict;
    uint64_t version;
    bool entire;                   // held entry by entry (a class is not, where its dict has a version)
    std::vector<Entry> entries;
};

// The number the interpreter gives a dict anew with every change of it (0: this interpreter has none).
uint64_t version_of(PyObject* dict) {
#if PY_VERSION_HEX < 0x030C0000
    return reinterpret_cast<PyDictObject*>(dict)->ma_version_tag;
#else
    return 0;
#endif
}

using Forward = int (*)(const void*, void*);
using Workspace = int64_t (*)(const void*, int);

struct State {
    std::vector<Watch> watches;
    std::vector<Entry> tensors;                // the entries that are tensors, once more (borrowed)
    std::vector<PyObject*> no_hooks;           // dicts that have to be empty: hooks
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

// Where a tensor's memory is.  One that only stands for others (under vmap, say, or a fake one) has none of its own: a layer
// that holds such a tensor runs module by module.
const char kNoMemory = 0;
const void* address_of(PyObject* t) noexcept {
    try {
        return THPVariable_Unpack(t).const_data_ptr();
    } catch (...) {
        return &kNoMemory;
    }
}

// ---- making a plan ------------------------------------------------------------------------------------------------
PyObject* keep(PyObject* o) {
    Py_XINCREF(o);
    return o;
}

void plan_free(State* s) {
    if (!s) return;
    for (auto& w : s->watches) {
        Py_XDECREF(w.dict);
        for (auto& e : w.entries) { Py_XDECREF(e.key); Py_XDECREF(e.value); }
    }
    for (PyObject* d : s->no_hooks) Py_XDECREF(d);
    Py_XDECREF(s->get_device); Py_XDECREF(s->set_device); Py_XDECREF(s->get_stream); Py_XDECREF(s->oom);
    delete s;
}

// Plan(watched, hooks, native): the dicts and classes the layer was made from, the dicts that have to be empty, and None for a layer the
// library does not cover, or (family, block bytes, (forward, step, workspace) addresses, (conv channels, state shape,
// (forward widths, step widths)), output padding, a tensor on the layer's device, (get_device, set_device, get_stream, out-of-memory error)).
int make_plan(PlanObject* self, PyObject* args) {
    PyObject *watched, *hooks, *native;
    if (!PyArg_ParseTuple(args, "O!O!O", &PyTuple_Type, &watched, &PyTuple_Type, &hooks, &native)) return -1;
    for (PyObject* dicts : {watched, hooks})
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(dicts); ++i)
            if (!PyDict_Check(PyTuple_GET_ITEM(dicts, i)) && (dicts == hooks || !PyType_Check(PyTuple_GET_ITEM(dicts, i)))) {
                PyErr_SetString(PyExc_TypeError, "a plan is made from dicts and classes");
                return -1;
            }
    State* s = new State;
    plan_free(self->s);
    self->s = s;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(watched); ++i) {
        PyObject* from = PyTuple_GET_ITEM(watched, i);
        PyObject* dict = keep(PyType_Check(from) ? reinterpret_cast<PyTypeObject*>(from)->tp_dict : from);
        s->watches.push_back({dict, version_of(dict), dict == from || version_of(dict) == 0, {}});
        if (!s->watches.back().entire) continue;
        s->watches.back().entries.reserve(PyDict_GET_SIZE(dict));
        PyObject *key, *value;
        Py_ssize_t pos = 0;
        while (PyDict_Next(dict, &pos, &key, &value)) {
            // (by type: THPVariable_Check asks the metaclass about everything that is no tensor)
            const bool tensor = PyObject_TypeCheck(value, reinterpret_cast<PyTypeObject*>(THPVariableClass));
            s->watches.back().entries.push_back({keep(key), keep(value), tensor, tensor ? address_of(value) : nullptr});
            if (tensor) s->tensors.push_back(s->watches.back().entries.back());
        }
    }
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(hooks); ++i) s->no_hooks.push_back(keep(PyTuple_GET_ITEM(hooks, i)));
    if (native == Py_None) return 0;
    if (!PyTuple_Check(native)) {
        PyErr_SetString(PyExc_TypeError, "the native part of a plan is a tuple or None");
        return -1;
    }

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
    if (PyErr_Occurred()) return -1;
    s->device = THPVariable_Unpack(anchor).device();
    s->usable = true;
    for (const Entry& e : s->tensors) s->usable = s->usable && e.address != &kNoMemory;
    return 0;
}

// No C++ exception passes through the interpreter.
template <class Result, class Body>
Result guarded(const State* s, Result failed, Body&& body) {
    try {
        return body();
    } catch (const c10::OutOfMemoryError& e) {
        PyErr_SetString(s && s->oom ? s->oom : PyExc_MemoryError, e.what_without_backtrace());
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    } catch (...) {
        PyErr_SetString(PyExc_RuntimeError, "unknown C++ exception");
    }
    return failed;
}

int plan_init(PlanObject* self, PyObject* args, PyObject*) {
    return guarded(nullptr, -1, [&] { return make_plan(self, args); });
}

// ---- using it -----------------------------------------------------------------------------------------------------
bool same_value(PyObject* a, PyObject* b) {
    if (a == b) return true;
    if (PyFloat_CheckExact(a) && PyFloat_CheckExact(b)) return PyFloat_AS_DOUBLE(a) == PyFloat_AS_DOUBLE(b);
    if (PyLong_CheckExact(a) && PyLong_CheckExact(b)) return PyObject_RichCompareBool(a, b, Py_EQ) == 1;
    return false;
}

// The dict holds what it held.  (Most calls end at the version; scanning the twenty dicts of a layer takes about 1 us.)
bool same_entries(Watch& w) {
    const uint64_t version = version_of(w.dict);
    if (version && version == w.version) return true;
    if (!w.entire) return false;
    if (PyDict_GET_SIZE(w.dict) != static_cast<Py_ssize_t>(w.entries.size())) return false;
    PyObject *key, *value;
    Py_ssize_t pos = 0;
    const Entry* e = w.entries.data();
    for (; PyDict_Next(w.dict, &pos, &key, &value); ++e)
        if (key != e->key || !same_value(value, e->value)) return false;
    w.version = version;
    return true;
}

// 1: the layer the plan was made from; 0: it has changed; -1: unchanged but hooked
int verify(State& s) {
    for (Watch& w : s.watches)
        if (!same_entries(w)) return 0;
    for (const Entry& e : s.tensors)
        if (address_of(e.value) != e.address) return 0;
    for (PyObject* d : s.no_hooks)
        if (PyDict_GET_SIZE(d) != 0) return -1;
    return 1;
}

template <class Params>
PyObject* enqueue(State& s, Params p, const at::Tensor& hidden, PyObject* conv_o, PyObject* ssm_o, int step) {
    const int64_t batch = hidden.size(0), len = hidden.size(1);
    p.batch = static_cast<int32_t>(batch);
    p.seqlen = static_cast<int32_t>(len);
    p.hidden = hidden.const_data_ptr<int8_t>();
    if (reinterpret_cast<uintptr_t>(p.hidden) % 16 != 0) Py_RETURN_NONE;
    if (conv_o != Py_None) {
        const at::Tensor& c = THPVariable_Unpack(conv_o);
        if (c.scalar_type() != at::kChar || c.device() != s.device || c.dim() != 3 || c.size(0) != batch || c.size(1) != s.conv_dim ||
            (c.size(2) != s.widths[step][0] && c.size(2) != s.widths[step][1])) Py_RETURN_NONE;
        // (rows that lie on each other: the modules' copy refuses them)
        for (int i = 0; i < 3; ++i)
            if (c.stride(i) == 0 && c.size(i) > 1) Py_RETURN_NONE;
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

// The layer's device for as long as this stands, however the call ends.
class OnDevice {
  public:
    explicit OnDevice(const State& s) : s_(s) {
        PyObject* at = PyObject_CallNoArgs(s.get_device);
        if (!at) return;
        back_ = PyLong_AsLong(at);
        Py_DECREF(at);
        if (PyErr_Occurred()) return;
        ok = back_ == s.device.index();
        if (!ok) ok = moved_ = set(s.device.index());
    }
    ~OnDevice() {
        if (!moved_) return;
        PyObject *type, *value, *trace;
        PyErr_Fetch(&type, &value, &trace);
        if (!set(back_)) PyErr_WriteUnraisable(s_.set_device);
        PyErr_Restore(type, value, trace);
    }
    OnDevice(const OnDevice&) = delete;
    bool ok = false;               // otherwise an error is set

  private:
    bool set(long device) {
        PyObject* r = PyObject_CallFunction(s_.set_device, "l", device);
        Py_XDECREF(r);
        return r != nullptr;
    }
    const State& s_;
    long back_ = 0;
    bool moved_ = false;
};

PyObject* run_on_device(State& s, PyObject* hidden_o, PyObject* conv_o, PyObject* ssm_o, int step) {
    const at::Tensor& hidden = THPVariable_Unpack(hidden_o);
    if (hidden.scalar_type() != at::kChar || hidden.device() != s.device || hidden.dim() != 3 || !hidden.is_contiguous() ||
        hidden.size(2) != s.d_model || hidden.size(0) == 0 || hidden.size(1) == 0 || hidden.size(0) > 65535 || hidden.size(1) > 0x7fffffff) Py_RETURN_NONE;
    const OnDevice on(s);
    if (!on.ok) return nullptr;
    return s.family == 1 ? enqueue(s, s.m1, hidden, conv_o, ssm_o, step) : enqueue(s, s.m2, hidden, conv_o, ssm_o, step);
}

PyObject* plan_run(PlanObject* self, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 4 || !self->s) {
        PyErr_SetString(PyExc_TypeError, "run(hidden, conv_state, ssm_state, step)");
        return nullptr;
    }
    State& s = *self->s;
    const int step = PyObject_IsTrue(args[3]);
    if (step < 0) return nullptr;
    return guarded(&s, static_cast<PyObject*>(nullptr), [&]() -> PyObject* {
        const int same = verify(s);
        if (same == 0) Py_RETURN_FALSE;
        if (same < 0 || !s.usable || !THPVariable_Check(args[0])) Py_RETURN_NONE;
        for (int i = 1; i < 3; ++i)
            if (args[i] != Py_None && !THPVariable_Check(args[i])) Py_RETURN_NONE;
        return run_on_device(s, args[0], args[1], args[2], step);
    });
}

// Copies and pickles of a layer start without a plan.
PyObject* plan_reduce(PyObject*, PyObject*) { return Py_BuildValue("(O())", reinterpret_cast<PyObject*>(Py_TYPE(Py_None))); }

// (an attribute of a sub-module may lead back to the mixer and from there to the plan)
int plan_traverse(PlanObject* self, visitproc visit, void* arg) {
    if (!self->s) return 0;
    for (const Watch& w : self->s->watches) {
        Py_VISIT(w.dict);
        for (const Entry& e : w.entries) { Py_VISIT(e.key); Py_VISIT(e.value); }
    }
    for (PyObject* d : self->s->no_hooks) Py_VISIT(d);
    for (PyObject* o : {self->s->get_device, self->s->set_device, self->s->get_stream, self->s->oom}) Py_VISIT(o);
    return 0;
}

int plan_clear(PlanObject* self) {
    State* s = self->s;
    self->s = nullptr;
    plan_free(s);
    return 0;
}

void plan_dealloc(PlanObject* self) {
    PyObject_GC_UnTrack(self);
    plan_clear(self);
    Py_TYPE(self)->tp_free(reinterpret_cast<PyObject*>(self));
}

PyMethodDef plan_methods[] = {
    {"run", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(plan_run)), METH_FASTCALL, "Enqueues the layer."},
    {"__reduce__", plan_reduce, METH_NOARGS, "Pickles as None."},
    {nullptr, nullptr, 0, nullptr}};

// class_version(cls): the version of a class's own dict (0: none)
PyObject* class_version(PyObject*, PyObject* cls) {
    if (!PyType_Check(cls)) {
        PyErr_SetString(PyExc_TypeError, "class_version(cls)");
        return nullptr;
    }
    return PyLong_FromUnsignedLongLong(version_of(reinterpret_cast<PyTypeObject*>(cls)->tp_dict));
}

PyMethodDef module_methods[] = {{"class_version", class_version, METH_O, "Version of a class's own dict."}, {nullptr, nullptr, 0, nullptr}};

PyTypeObject PlanType = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", "Host side of the mixers' library calls.", -1, module_methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    PlanType.tp_name = "quamba_amd._host.Plan";
    PlanType.tp_basicsize = sizeof(PlanObject);
    PlanType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC;
    PlanType.tp_new = PyType_GenericNew;
    PlanType.tp_traverse = reinterpret_cast<traverseproc>(plan_traverse);
    PlanType.tp_clear = reinterpret_cast<inquiry>(plan_clear);
    PlanType.tp_free = PyObject_GC_Del;
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
