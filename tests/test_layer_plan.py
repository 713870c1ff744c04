"""The plan behind a mixer call (quamba_amd._host.Plan) on the host alone: what it notices about a layer, what it keeps."""
import ctypes as C
import gc
import weakref

import numpy as np
import pytest
import torch
import torch.nn as nn

from quamba_amd import W4A8QMamba, W4A8QMamba2, W8A8QMamba, W8A8QMamba2, _layer_call, _lib

MIXERS = [W8A8QMamba, W4A8QMamba, W8A8QMamba2, W4A8QMamba2]
HIDDEN = torch.zeros(1, 1, 256, dtype=torch.int8)


def _mixer(cls):
    if cls in (W8A8QMamba, W4A8QMamba):
        return cls(256, 16, 4, device="cpu")
    return cls(256, 64, 4, 2, 64, ngroups=2, chunk_size=64, device="cpu", x_nhead_group=2, x_ndim_group=2)


def _unchanged(plan):
    """None: the plan's layer (which the library does not cover, on the CPU); False: not that layer any more."""
    return plan.run(HIDDEN, None, None, False) is None


def _tensors(mixer):
    return [(m, name) for m in mixer._modules.values() for name, t in m._buffers.items() if t is not None]


@pytest.mark.parametrize("cls", MIXERS)
@pytest.mark.parametrize("held", ["buffer", "parameter", "attribute"])
def test_every_tensor_is_watched_wherever_the_module_holds_it(cls, held):
    m = _mixer(cls)

    def hold(module, name, t):
        for d in (module._buffers, module._parameters, module.__dict__):
            d.pop(name, None)
        if held == "buffer":
            module.register_buffer(name, t)
        elif held == "parameter":
            module.register_parameter(name, nn.Parameter(t, requires_grad=False))
        else:
            module.__dict__[name] = t

    for module, name in _tensors(m):
        hold(module, name, getattr(module, name))
    plan = _layer_call._make(m)
    assert _unchanged(plan)
    for module, name in _tensors(m) + [(mod, n) for mod in m._modules.values() for n, t in {**mod._parameters, **mod.__dict__}.items() if torch.is_tensor(t)]:
        old = getattr(module, name)
        gone = weakref.ref(old)
        new = old.clone().contiguous()
        if held == "attribute":
            module.__dict__[name] = new
        else:
            setattr(module, name, nn.Parameter(new, requires_grad=False) if held == "parameter" else new)
        del old, new
        assert not _unchanged(plan), name
        assert gone() is not None, f"{name}: its address is in the plan's block"
        plan = _layer_call._make(m)
        assert _unchanged(plan), name


@pytest.mark.parametrize("cls", [W8A8QMamba, W8A8QMamba2])
def test_replaced_modules_numbers_and_memory_are_seen(cls):
    m = _mixer(cls)
    plan = _layer_call._make(m)
    m.had.x_H_scale = float(m.had.x_H_scale) + 0.0           # another object, the same number
    assert _unchanged(plan)
    m.had.x_H_scale = 3.0
    assert not _unchanged(plan)
    plan = _layer_call._make(m)
    m.out_proj.weight.data = m.out_proj.weight.clone()       # the same object, other memory
    assert not _unchanged(plan)
    plan = _layer_call._make(m)
    m.had = type(m.had)(m.had.dim)
    assert not _unchanged(plan)


def test_other_modules_in_the_mixer():
    """In the place of one of its own: the modules run, whatever it is made of.  Beside them: nothing to the call."""
    m = _mixer(W8A8QMamba)
    stock = m.had
    m.had = torch.jit.script(nn.Identity())                  # (keeps no dicts of buffers and parameters)
    plan = _layer_call._make(m)
    assert _unchanged(plan) and m._native_modules() is None
    m.had = stock
    assert not _unchanged(plan)
    m.observer = nn.Linear(1, 1)
    m.observer.forward = lambda x: x
    native = []
    kept, _layer_call._native = _layer_call._native, lambda mixer: native.append(mixer)
    try:
        _layer_call._make(m)
    finally:
        _layer_call._native = kept
    assert native == [m]


def test_a_plan_does_not_keep_its_mixer():
    m = _mixer(W8A8QMamba)
    m.__dict__["_plan"] = _layer_call._make(m)
    m.conv1d.__dict__["owner"] = m                           # leads from the plan back to the mixer
    m.__dict__["_plan"] = _layer_call._make(m)
    gone = weakref.ref(m)
    del m
    gc.collect()
    assert gone() is None


@pytest.mark.parametrize("cls", MIXERS)
def test_a_tensor_without_memory_of_its_own(cls):
    """Under vmap a buffer stands for a batch of tensors and has no address: the plan yields to the modules (once, and
    without a plan made anew on each call), and an existing plan sees the exchange."""
    m = _mixer(cls)
    plan = _layer_call._make(m)
    held = m.out_proj._buffers["weight"]
    seen = []

    def body(w):
        m.out_proj._buffers["weight"] = w
        inner = _layer_call._make(m)
        seen.extend([_unchanged(plan), _unchanged(inner), _layer_call.call(m, HIDDEN, None, None, False), _unchanged(m.__dict__["_plan"])])
        return w

    torch.vmap(body)(torch.stack([held, held]))
    m.out_proj._buffers["weight"] = held
    assert seen == [False, True, None, True]
    assert not _unchanged(m.__dict__["_plan"])


def test_a_plan_made_of_the_wrong_things_is_an_error():
    plan = _layer_call._plan_class()
    for args in ((), ((), ()), ((), (), 3), ((3,), (), None), ((), (3,), None), ((), (), (1, b"", (1, 2, 3)))):
        with pytest.raises(TypeError):
            plan(*args)
    with pytest.raises(TypeError):
        plan.__new__(plan).run(HIDDEN, None, None, False)


@pytest.mark.parametrize("cls", MIXERS)
def test_a_number_that_can_change_in_place_is_left_to_the_modules(cls):
    m = _mixer(cls)
    cpu = torch.device("cpu")
    m._native_block(cpu)
    names = [("had", "x_H_scale"), ("had", "had_scale"), ("out_proj", "alpha")] + (
        [("norm", "z_scale"), ("norm", "eps"), ("conv1d", "x_scale"), ("conv1d", "wB_scale"), ("conv1d", "bC_scale"), ("qchunk_scan", "dt_limit")]
        if hasattr(m, "norm") else [("conv1d", n) for n in ("input_scale", "weight_scale", "bias_scale", "output_scale")])
    for module, name in names:
        md = m._modules[module]
        if name not in md.__dict__:
            continue                                         # (4-bit projections have no alpha)
        kept = getattr(md, name)
        for held in ([torch.tensor(v) for v in (kept, 1.0)] if name != "dt_limit" else [[0.0, 1.0], (torch.tensor(0.0), 1.0)]):
            setattr(md, name, held)
            with pytest.raises(_layer_call._Unsupported):
                m._native_block(cpu)
        setattr(md, name, kept)
    m._native_block(cpu)
    m.had.x_H_scale = np.float32(0.5)                        # (a number like any other)
    m._native_block(cpu)


class _Runtime:
    """A plan over host functions in place of the library's and the device's, for what the plan does around them."""
    FORWARD = C.CFUNCTYPE(C.c_int, C.POINTER(_lib.QaMamba1Params), C.c_void_p)
    WORKSPACE = C.CFUNCTYPE(C.c_int64, C.POINTER(_lib.QaMamba1Params), C.c_int)

    def __init__(self, status=0, workspace=256, stream=0, current=3):
        self.current, self.calls, self.blocks = current, [], []
        self.device, self.stream = current, stream
        self.fns = self.FORWARD(lambda p, s: self.enter("forward", p, status)), self.FORWARD(lambda p, s: self.enter("step", p, status))
        self.workspace = self.WORKSPACE(lambda p, step: workspace)
        block = _lib.QaMamba1Params()
        block.d_model, block.out_proj.n = 256, 256
        addresses = tuple(C.cast(f, C.c_void_p).value for f in self.fns + (self.workspace,))
        runtime = (lambda: self.device, self.set_device, self.get_stream, MemoryError)
        self.plan = _layer_call._plan_class()((), (), (1, bytes(block), addresses, (512, (512, 16), ((4, 3), (4, 3))), 0, torch.empty(0), runtime))

    def enter(self, what, p, status):
        self.calls.append((what, self.device))
        self.blocks.append(_lib.QaMamba1Params.from_buffer_copy(p.contents))
        return status

    def set_device(self, index):
        self.device = index

    def get_stream(self, index):
        if isinstance(self.stream, Exception):
            raise self.stream
        return self.stream


def test_hidden_states_the_products_cannot_read_go_to_the_modules():
    """Contiguous but not 16-byte aligned: refused before anything is enqueued, whatever the token count."""
    r = _Runtime()
    room = torch.zeros(5 * 256 + 16, dtype=torch.int8)
    start = -room.data_ptr() % 16
    for tokens, offset in ((1, 1), (3, 8), (5, 4)):
        h = room[start + offset:][:tokens * 256].view(1, tokens, 256)
        assert h.is_contiguous() and r.plan.run(h, None, None, False) is None and not r.calls
    assert torch.is_tensor(r.plan.run(room[start:][:256].view(1, 1, 256), None, None, False))


def test_states_the_call_does_not_write():
    r = _Runtime()
    conv, ssm = torch.zeros(1, 512, 4, dtype=torch.int8), torch.zeros(1, 512, 16)
    assert torch.is_tensor(r.plan.run(HIDDEN, conv, ssm, False)) and r.blocks[-1].state_is_fp32 == 1 and r.blocks[-1].conv_state == conv.data_ptr()
    assert torch.is_tensor(r.plan.run(HIDDEN, conv[..., 1:], ssm.to(torch.int8), True)) and r.blocks[-1].conv_state_len == 3
    room = torch.zeros(512 * 16 + 4)
    off = room[(-room.data_ptr() // 4) % 4 + 1:][:512 * 16].view(1, 512, 16)
    for c, s in ((conv[:, :1].expand(1, 512, 4), ssm), (conv[:, :511], ssm), (conv.float(), ssm), (conv.expand(2, 512, 4), ssm), (conv[..., :2], ssm),
                 (conv, ssm.half()), (conv, ssm.transpose(1, 2).contiguous().transpose(1, 2)), (conv, ssm[:, :511]), (conv, off)):
        for step in (False, True):
            assert r.plan.run(HIDDEN, c, s, step) is None
    assert len(r.calls) == 2


def test_the_current_device_comes_back_however_the_call_ends():
    here = -1                                                # (the index of a device without one)
    r = _Runtime()
    assert r.plan.run(HIDDEN, None, None, False).shape == (1, 1, 256) and r.calls == [("forward", here)] and r.device == 3
    r = _Runtime(status=-5)
    assert r.plan.run(HIDDEN, None, None, True) == -5 and r.calls == [("step", here)] and r.device == 3
    r = _Runtime(workspace=1 << 60)                          # more than there is: the allocation throws
    with pytest.raises(RuntimeError):
        r.plan.run(HIDDEN, None, None, False)
    assert not r.calls and r.device == 3
    r = _Runtime(stream=KeyError("no stream"))
    with pytest.raises(KeyError):
        r.plan.run(HIDDEN, None, None, False)
    assert r.device == 3
    r = _Runtime(current=here)                               # on the layer's device already
    assert torch.is_tensor(r.plan.run(HIDDEN, None, None, False)) and r.device == here
    r = _Runtime()
    assert r.plan.run(HIDDEN.float(), None, None, False) is None and not r.calls and r.device == 3


def _own_code(*modules):
    return _layer_call._own_code(modules, _layer_call._classes_of(tuple(map(type, modules))))


def _public(module):
    return [n for c in type(module).__mro__ if c.__module__.startswith("quamba_amd") for n, f in vars(c).items() if callable(f) and not n.startswith("__")]


@pytest.mark.parametrize("cls", MIXERS)
def test_a_method_replaced_on_a_module_is_another_layer(cls):
    m = _mixer(cls)
    assert _own_code(*m._modules.values())
    for module in m._modules.values():
        names = _public(module)
        assert "forward" in names
        for name in names + ["_call_impl", "_compiled_call_impl"]:
            plan = _layer_call._make(m)
            assert _unchanged(plan) and _own_code(module)
            module.__dict__[name] = lambda *a, **k: None
            assert not _unchanged(plan) and not _own_code(module), name
            del module.__dict__[name]
    plan = _layer_call._make(m)
    m.had.transform_fn = lambda x, s: x
    assert not _unchanged(plan)


@pytest.mark.parametrize("cls", MIXERS)
def test_a_method_replaced_on_a_class_is_another_layer(cls, monkeypatch):
    m = _mixer(cls)
    for module in m._modules.values():
        for c in (type(module), torch.nn.Module):
            name = "forward" if c is not torch.nn.Module else "__call__"
            plan = _layer_call._make(m)
            assert _unchanged(plan) and _own_code(module)
            with monkeypatch.context() as patch:
                patch.setattr(c, name, lambda *a, **k: None)
                assert not _unchanged(plan) and not _own_code(module)
            assert _own_code(module)
