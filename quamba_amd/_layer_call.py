"""One library call per mixer call: the parameter blocks of qa_mamba1_* / qa_mamba2_*.

A mixer's weights, scales and sizes are gathered into a ctypes block once and kept for as long as its sub-modules,
their buffers (the tensor objects and their addresses) and their Python-float scales are the ones the block was made
from; each call copies the block, adds its own tensors and enqueues the whole layer.  Mixers, tensors or states the
library calls do not cover (other sub-module classes, forward hooks, views with gaps, unusual sizes) yield None, and
the mixer runs its modules one by one.
"""
import ctypes as C

import torch
import torch.nn.modules.module as _module

from . import _lib

_STATE_DTYPES = (torch.int8, torch.float32)


def _none():
    return None


class Plan:
    """A gathered block and what it was gathered from.  Copies and pickles of a mixer start without one."""
    __slots__ = ("key", "tensors", "block", "size", "device", "fns", "workspace", "pad_out", "n_out", "dims")

    def __reduce__(self):
        return (_none, ())

    def __deepcopy__(self, memo):
        return None


def _key(mixer, mods):
    """What a plan depends on: sub-modules and buffers by identity and address, the scalars they carry by value."""
    bufs = [t for md in mods for t in md._buffers.values()]
    return ([id(md) for md in mods], [id(t) for t in bufs], [t.data_ptr() for t in bufs if t is not None], mixer._scalars()), bufs


class _Unsupported(Exception):
    pass


def _need(cond):
    if not cond:
        raise _Unsupported


def _ptr(t, dtype, numel, device, align=1):
    """Address of a dense tensor of `numel` elements on the plan's device (None stays None)."""
    if t is None:
        return None
    _need(t.dtype == dtype and t.numel() == numel and t.device == device and t.is_contiguous())
    a = t.data_ptr()
    _need(a % align == 0)
    return a


def linear_block(lin, device):
    """QaLinearParams of one of the linear modules."""
    p = _lib.QaLinearParams()
    if hasattr(lin, "s_group"):
        n, k = lin.size_n, lin.size_k
        p.n, p.k, p.bits, p.col_numel = n, k, 4, n
        p.weight = _ptr(lin.weight, torch.uint8, n * (k // 2), device, 16)
        p.s_group = _ptr(lin.s_group, torch.float16, (k // 128) * n, device) if lin.s_group.numel() else None
        p.col_scale = _ptr(lin.s_channel, torch.float32, n, device)
        p.row_scale = _ptr(lin.input_scale, torch.float32, 1, device)
        _need(k % 128 == 0)
    else:
        n, k = lin.out_features + lin.pad_out, lin.in_features
        p.n, p.k, p.bits, p.col_numel = n, k, 8, lin.b.numel()
        _need(tuple(lin.weight.shape) == (k, n) and p.col_numel in (1, n))
        p.weight = _ptr(lin.weight.t(), torch.int8, n * k, device, 16)
        p.col_scale = _ptr(lin.b, torch.float32, lin.b.numel(), device)
        p.row_scale = _ptr(lin.a, torch.float32, 1, device)
        if hasattr(lin, "alpha"):
            p.row_rule, p.alpha = _lib.QA_ROW_ALPHA, lin.alpha
        else:
            p.row_rule = _lib.QA_ROW_HALF_AWAY
    return p


def _plan(mixer):
    """The mixer's plan, made anew when anything it was made from has changed; None where there is none."""
    mods = mixer._native_modules()
    if mods is None or _module._has_any_global_hook():
        return None
    for md in mods:
        if md._forward_hooks or md._forward_pre_hooks:
            return None
    plan = mixer.__dict__.get("_plan")
    key, bufs = _key(mixer, mods)
    if plan is not None and plan.key == key:
        return plan
    plan = Plan()
    plan.key, plan.tensors, plan.workspace = key, (mods, bufs), {}
    try:
        plan.device = mixer.out_proj.weight.device
        _need(plan.device.type == "cuda")
        plan.block, plan.dims = mixer._native_block(plan.device)
    except _Unsupported:
        plan.block = None
    else:
        plan.size = type(plan.block)
        family = "qa_mamba1" if plan.size is _lib.QaMamba1Params else "qa_mamba2"
        lib = _lib.lib()
        plan.fns = tuple(getattr(lib, family + s) for s in ("_forward", "_step", "_workspace_bytes"))
        plan.pad_out, plan.n_out = mixer.out_proj.pad_out, plan.block.out_proj.n
    mixer.__dict__["_plan"] = plan
    return plan


def call(mixer, hidden, conv_state, ssm_state, step):
    """The layer's output (tokens, outputs) fp16, or None where the library call does not apply."""
    plan = _plan(mixer)
    if plan is None or plan.block is None:
        return None
    batch, seqlen, d_model = hidden.shape
    conv_dim, state_shape, widths = plan.dims
    if hidden.dtype is not torch.int8 or hidden.device != plan.device or not hidden.is_contiguous() or batch == 0 or seqlen == 0:
        return None
    block = plan.size.from_buffer_copy(plan.block)
    if d_model != block.d_model:
        return None
    if conv_state is not None:
        s = conv_state.shape
        if (conv_state.dtype is not torch.int8 or conv_state.device != plan.device or len(s) != 3 or s[0] != batch
                or s[1] != conv_dim or s[2] not in widths[step]):
            return None
        block.conv_state, block.conv_state_len = conv_state.data_ptr(), s[2]
        block.conv_state_batch_stride, block.conv_state_c_stride, block.conv_state_l_stride = conv_state.stride()
    if ssm_state is not None:
        if (ssm_state.dtype not in _STATE_DTYPES or ssm_state.device != plan.device or ssm_state.shape[1:] != state_shape
                or ssm_state.shape[0] != batch or not ssm_state.is_contiguous() or ssm_state.data_ptr() % 16):
            return None
        block.ssm_state, block.state_is_fp32 = ssm_state.data_ptr(), ssm_state.dtype is torch.float32
    block.batch, block.seqlen, block.hidden = batch, seqlen, hidden.data_ptr()
    ref = C.byref(block)
    key = (batch, seqlen, step)
    nbytes = plan.workspace.get(key)
    if nbytes is None:
        nbytes = plan.fns[2](ref, step)
        if len(plan.workspace) >= 256:
            plan.workspace.clear()
        plan.workspace[key] = nbytes
    if nbytes == 0:
        return None
    out = torch.empty((batch * seqlen, plan.n_out), dtype=torch.float16, device=plan.device)
    workspace = torch.empty((nbytes,), dtype=torch.uint8, device=plan.device)
    block.out, block.workspace, block.workspace_bytes = out.data_ptr(), workspace.data_ptr(), nbytes
    index = plan.device.index
    if torch.cuda.current_device() == index:
        status = plan.fns[step](ref, torch._C._cuda_getCurrentRawStream(index))
    else:
        with torch.cuda.device(index):
            status = plan.fns[step](ref, torch._C._cuda_getCurrentRawStream(index))
    if status:
        _lib.check(status, "mixer step" if step else "mixer forward")
    return out[:, :-plan.pad_out] if plan.pad_out else out
