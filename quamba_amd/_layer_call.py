"""One library call per mixer call: qa_mamba1_* / qa_mamba2_* behind the mixers.

A mixer's weights, scales and sizes are gathered into the library's parameter block once and kept, in a native object
(quamba_amd._host.Plan, host/layer_call.cpp), for as long as its sub-modules and everything they hold - attributes, buffers
and parameters, tensors with their addresses - are the ones the block was made from; running the plan verifies that,
allocates output and workspace and enqueues the layer.  Mixers, tensors or states the library call does not cover (other
sub-module classes or replaced methods, forward hooks, views with gaps, unusual sizes) yield None, and the mixer runs its
modules one by one.
"""
import ctypes as C
import functools
import numbers

import torch
import torch.nn.modules.module as _module

from . import _lib
from .linear import _AlphaHooks, _W4A8Base

_host = None


def _plan_class():
    """quamba_amd._host.Plan; raises if the extension is not built (there is no fallback)."""
    global _host
    if _host is None:
        try:
            from . import _host as native
        except ImportError as e:
            raise RuntimeError("quamba_amd/_host.so is missing or does not load: build it with `python -m quamba_amd.build`") from e
        if getattr(native, "ABI_VERSION", None) != _lib.ABI_VERSION:
            raise RuntimeError("quamba_amd/_host.so is built for another layout of the parameter blocks: rebuild it with "
                               "`python -m quamba_amd.build --force`")
        _host = native
    return _host.Plan


class _Unsupported(Exception):
    pass


def _need(cond):
    if not cond:
        raise _Unsupported


def _held(module):
    """name -> what the module holds under it, as attribute access finds it (in a third of its time; a layer has some fifty)."""
    own = module.__dict__
    parameters, buffers = own["_parameters"], own["_buffers"]

    def get(name):
        return own[name] if name in own else parameters[name] if name in parameters else buffers[name]
    return get


def _ptr(t, dtype, numel, device, align=1):
    """Address of a dense tensor of `numel` elements on the layer's device (None stays None)."""
    if t is None:
        return None
    if t.dtype is not dtype or t.numel() != numel or t.device != device or not t.is_contiguous():
        raise _Unsupported
    try:
        a = t.data_ptr()
    except RuntimeError as e:                  # no memory of its own (under vmap, say)
        raise _Unsupported from e
    if a % align:
        raise _Unsupported
    return a


def _number(v):
    """A value that goes into the block as a number: one that only changes by becoming another object.  (A tensor or an array
    of one element can change in place, which the plan would not see: the modules read it on every call.)"""
    _need(type(v) in (float, int, bool) or isinstance(v, numbers.Real))
    return v


def linear_block(lin, device):
    """QaLinearParams of one of the linear modules."""
    p, held = _lib.QaLinearParams(), _held(lin)
    weight = held("weight")
    if isinstance(lin, _W4A8Base):
        n, k, s_group = lin.size_n, lin.size_k, held("s_group")
        p.n, p.k, p.bits, p.col_numel = n, k, 4, n
        p.weight = _ptr(weight, torch.uint8, n * (k // 2), device, 16)
        p.s_group = _ptr(s_group, torch.float16, (k // 128) * n, device) if s_group.numel() else None
        p.col_scale = _ptr(held("s_channel"), torch.float32, n, device)
        p.row_scale = _ptr(held("input_scale"), torch.float32, 1, device)
        _need(k % 128 == 0)
    else:
        n, k, b = lin.out_features + lin.pad_out, lin.in_features, held("b")
        cols = b.numel()
        p.n, p.k, p.bits, p.col_numel = n, k, 8, cols
        _need(weight.shape == (k, n) and cols in (1, n))
        p.weight = _ptr(weight.t(), torch.int8, n * k, device, 16)
        p.col_scale = _ptr(b, torch.float32, cols, device)
        p.row_scale = _ptr(held("a"), torch.float32, 1, device)
        if isinstance(lin, _AlphaHooks):
            p.row_rule, p.alpha = _lib.QA_ROW_ALPHA, _number(lin.alpha)
        else:
            p.row_rule = _lib.QA_ROW_HALF_AWAY
    return p


_ENTRIES = {}          # family -> addresses of its entry points in the loaded library


def _native(mixer):
    """What quamba_amd._host.Plan takes for a mixer the library covers."""
    device = mixer.out_proj.weight.device
    _need(device.type == "cuda")
    block, dims = mixer._native_block(device)
    lib = _lib.lib()
    family = 1 if type(block) is _lib.QaMamba1Params else 2
    if family not in _ENTRIES:
        _ENTRIES[family] = tuple(C.cast(getattr(lib, f"qa_mamba{family}{s}"), C.c_void_p).value for s in ("_forward", "_step", "_workspace_bytes"))
    runtime = (torch.cuda.current_device, torch.cuda.set_device, torch._C._cuda_getCurrentRawStream, torch.cuda.OutOfMemoryError)
    return family, bytes(block), _ENTRIES[family], dims, mixer.out_proj.pad_out, mixer.out_proj.weight, runtime


# The classes whose methods the library call stands for, as they were when this package was imported: what each of them
# holds itself, and the names under which it and its bases hold something callable; and the version of what it held when it
# was last found so.
_HELD, _CALLABLE, _SEEN = {}, {}, {}


def remember(*classes):
    """The library call stands for the methods of these classes as they are now."""
    for cls in classes:
        _CALLABLE[cls] = frozenset(n for n in dir(cls) if callable(getattr(cls, n, None)))
        for c in cls.__mro__:
            if c.__module__.split(".")[0] == __package__ or c is torch.nn.Module:
                _HELD[c] = dict(vars(c))


def _code_of(held):
    return {n: f for n, f in held.items() if callable(f) or isinstance(f, (classmethod, staticmethod, property))}


@functools.lru_cache(maxsize=64)
def _classes_of(types):
    """The remembered classes among these and their bases."""
    return tuple({c: None for t in types for c in t.__mro__ if c in _HELD})


def _own_code(modules, classes):
    """Whether calling the modules' methods runs the code of their classes: no method replaced on the instance (as offloading
    and tracing tools wrap modules) or on the class, no compiled form in their place."""
    _plan_class()
    for c in classes:
        version = _host.class_version(c)
        if version and _SEEN.get(c) == version:
            continue
        if vars(c) != _HELD[c] and _code_of(vars(c)) != _code_of(_HELD[c]):
            return False
        _SEEN[c] = version
    return all(type(m) in _CALLABLE and _CALLABLE[type(m)].isdisjoint(m.__dict__) and m.__dict__.get("_compiled_call_impl") is None for m in modules)


def _make(mixer):
    """The mixer's plan (one that only ever yields None where the library does not cover the mixer)."""
    mods = mixer._native_modules()
    if mods is None:                           # (whatever stands there need not be held together like an ordinary module)
        return _plan_class()((mixer._modules,), (), None)
    watched = [mixer._modules]
    hooks = [getattr(_module, k) for k in ("_global_forward_hooks", "_global_forward_pre_hooks")]
    for m in mods:
        held = m.__dict__
        watched += [held, held["_buffers"], held["_parameters"]]
        hooks += [held["_forward_hooks"], held["_forward_pre_hooks"]]
    classes = _classes_of(tuple(map(type, mods)))
    watched += classes
    try:
        _need(_own_code(mods, classes))
        native = _native(mixer)
    except _Unsupported:
        native = None
    return _plan_class()(tuple(watched), tuple(hooks), native)


def call(mixer, hidden, conv_state, ssm_state, step):
    """The layer's output fp16 (batch, seqlen, outputs), or None where the library call does not apply."""
    plan = mixer.__dict__.get("_plan")
    out = plan.run(hidden, conv_state, ssm_state, step) if plan is not None else False
    if out is False:
        plan = mixer.__dict__["_plan"] = _make(mixer)
        out = plan.run(hidden, conv_state, ssm_state, step)
        if out is False:
            return None
    if type(out) is int:
        _lib.check(out, "mixer step" if step else "mixer forward")
    return out
