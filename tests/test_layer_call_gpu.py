"""The library call that enqueues a whole layer against the same layer run module by module: token counts around the
edges of the scan's tiles and segments, both state types, states of three and four codes, one row (the single-row
rules of the projections) and many; and what the call leaves to the modules."""
import ctypes

import pytest
import torch

from quamba_amd import W4A8QMamba, W4A8QMamba2, W8A8QMamba, W8A8QMamba2, _layer_call, _lib
from quamba_amd.linear import W8A8B8O8LinearParallel
from tests import test_mixer_variants_gpu as variants
from tests.test_mixer_variants_gpu import _mamba2, _ri

pytestmark = pytest.mark.gpu


def _mamba1(cls, dev, seed, d_model=256):
    sized = lambda width, *a, **k: cls(d_model, *a, **k)       # (the shared builder is for one width)
    return variants._mamba1(sized, dev, seed)


MIXERS = [(W8A8QMamba, _mamba1), (W4A8QMamba, _mamba1), (W8A8QMamba2, _mamba2), (W4A8QMamba2, _mamba2)]


def _states(m, dev, g, batch, dtype, width):
    dim = m.conv1d.weight.shape[0]
    conv = _ri(dev, g, batch, width, dim).transpose(1, 2) if hasattr(m, "qchunk_scan") else _ri(dev, g, batch, dim, width)
    shape = (batch, m.nheads, m.headdim, m.d_state) if hasattr(m, "qchunk_scan") else (batch, m.d_inner, m.d_state)
    ssm = _ri(dev, g, *shape) if dtype == torch.int8 else torch.randn(shape, device=dev, generator=g) * 0.1
    return conv, ssm


def _close(got, want, conv, ssm):
    scale = float(want.float().abs().max()) + 1e-6
    diff = (got.float() - want.float()).abs()
    # fp16 scan outputs may differ in the last place, and int8 codes made of them by one step
    assert float(diff.max()) <= 2e-2 * scale and float(diff.mean()) <= 1e-3 * scale
    assert torch.equal(conv[0], conv[1])
    a, b = ssm[0].float(), ssm[1].float()
    if ssm[0].dtype == torch.int8:
        assert float((a - b).abs().max()) <= 1 and float((a != b).float().mean()) <= 5e-3
    else:
        assert float((a - b).abs().max()) <= 1e-3 * float(b.abs().max())


@pytest.mark.parametrize("cls,build", MIXERS)
@pytest.mark.parametrize("batch,seqlen,dtype,width", [(1, 1, torch.int8, 4), (1, 3, torch.float32, 3), (3, 33, torch.int8, 4),
                                                      (2, 64, torch.float32, 4), (1, 257, torch.int8, 3), (2, 1029, torch.float32, 4)])
def test_forward(dev, cls, build, batch, seqlen, dtype, width):
    m, g = build(cls, dev, seed=seqlen)
    width = 4 if hasattr(m, "qchunk_scan") else width            # (the second family's forward takes the whole window)
    h = _ri(dev, g, batch, seqlen, 256)
    conv, ssm = _states(m, dev, g, batch, dtype, width)
    conv2, ssm2 = conv.clone(), ssm.clone()
    out = _layer_call.call(m, h, conv, ssm, False)
    assert out is not None, "the library call has to take this"
    want = m._forward_modules(h, conv2, ssm2)
    _close(out, want, (conv, conv2), (ssm, ssm2))
    assert torch.equal(m.forward(h), out)          # without states


@pytest.mark.parametrize("cls,build", MIXERS)
@pytest.mark.parametrize("batch,dtype,width", [(1, torch.int8, 4), (1, torch.float32, 3), (7, torch.int8, 4), (33, torch.float32, 4), (70, torch.int8, 3)])
def test_step(dev, cls, build, batch, dtype, width):
    m, g = build(cls, dev, seed=batch)
    h = _ri(dev, g, batch, 1, 256)
    conv, ssm = _states(m, dev, g, batch, dtype, width)
    conv2, ssm2 = conv.clone(), ssm.clone()
    out = _layer_call.call(m, h, conv, ssm, True)
    assert out is not None, "the library call has to take this"
    want = m._step_modules(h, conv2, ssm2)
    _close(out[:, 0], want, (conv, conv2), (ssm, ssm2))


@pytest.mark.parametrize("d_model", [768, 2048, 2560])
def test_step_of_a_wide_layer(dev, d_model):
    """in_proj and the conv in one launch, with the weight rows' K split over waves (2048) and not (768); for one row the
    transform and out_proj in one launch, with 12, 1 and 40 column blocks."""
    m, g = _mamba1(W8A8QMamba, dev, seed=1, d_model=d_model)
    for batch in (1, 5):
        h = _ri(dev, g, batch, 1, d_model)
        conv, ssm = _states(m, dev, g, batch, torch.int8, 4)
        conv2, ssm2 = conv.clone(), ssm.clone()
        out = _layer_call.call(m, h, conv, ssm, True)
        _close(out[:, 0], m._step_modules(h, conv2, ssm2), (conv, conv2), (ssm, ssm2))


def test_step_with_a_dt_proj_that_rounds_half_away(dev):
    """One row's rule of the parallel linear, which a caller of the C ABI may name for any projection: half of the step sizes'
    codes sit at a tie."""
    m, g = _mamba1(W8A8QMamba, dev, seed=1)
    lin, other = m.dt_proj, W8A8B8O8LinearParallel(m.dt_proj.in_features, m.dt_proj.out_features, device=dev)
    for t in (lin, other):
        t._set_weight(_ri(dev, torch.Generator(device=dev).manual_seed(2), t.out_features, t.in_features, lo=-1, hi=2))
        t.a, t.b = torch.ones(1, 1, device=dev), torch.full((1, t.b.numel()), 0.5, device=dev)
    h = _ri(dev, g, 1, 1, 256)
    conv, ssm = _states(m, dev, g, 1, torch.float32, 4)
    states = [(conv.clone(), ssm.clone()) for _ in range(3)]
    p = _lib.QaMamba1Params.from_buffer_copy(_layer_call._native(m)[1])
    p.batch = p.seqlen = p.state_is_fp32 = 1
    p.dt_proj.row_rule = _lib.QA_ROW_HALF_AWAY
    p.conv_state_batch_stride, p.conv_state_c_stride, p.conv_state_l_stride = conv.stride()
    out = torch.empty(1, 1, p.out_proj.n, dtype=torch.float16, device=dev)
    p.workspace_bytes = _lib.lib().qa_mamba1_workspace_bytes(ctypes.byref(p), 1)
    work = torch.empty(p.workspace_bytes, dtype=torch.uint8, device=dev)
    p.hidden, p.out, p.conv_state, p.ssm_state, p.workspace = (t.data_ptr() for t in (h, out, *states[0], work))
    _lib.check(_lib.lib().qa_mamba1_step(ctypes.byref(p), _lib.current_stream(dev)), "mamba1_step")
    even = m._step_modules(h, *states[1])
    m.dt_proj = other
    want = m._step_modules(h, *states[2])
    _close(out[:, 0], want, *zip(states[0], states[2]))
    assert not torch.equal(even, want) and float((states[1][1] - states[2][1]).abs().max()) > 1e-2 * float(ssm.abs().max())


@pytest.mark.parametrize("cls,d_model,batch,width", [(W8A8QMamba, 768, 3, 4), (W8A8QMamba, 2560, 30, 4), (W8A8QMamba, 2560, 61, 4), (W8A8QMamba, 2560, 20, 3),
                                                     (W4A8QMamba, 2560, 24, 4), (W4A8QMamba, 2560, 61, 4), (W8A8QMamba2, 768, 9, 4),
                                                     (W8A8QMamba2, 2560, 17, 3), (W8A8QMamba, 3072, 2, 4),
                                                     (W8A8QMamba, 1024, 4, 4), (W4A8QMamba, 1536, 6, 4), (W4A8QMamba2, 2048, 40, 4), (W4A8QMamba2, 4096, 63, 4)])
def test_step_of_many_sequences(dev, cls, d_model, batch, width):
    """in_proj and the conv in one launch for more than two rows: tiles of the product (each of them in
    test_kernel_choice_gpu.py), with one and two passes over its sums, the conv's state by channel and by step (three and four codes),
    rows and columns with remainders; in the first family dt_proj in the state update's launch, ranks of 48 to 192, one to four
    entries a wave."""
    dtype = torch.float32 if batch % 2 == 0 else torch.int8
    second = cls in (W8A8QMamba2, W4A8QMamba2)
    sized = lambda d, *a, **k: cls(d_model, *a, **k)
    m, g = (_mamba2 if second else variants._mamba1)(sized, dev, seed=batch)
    if second:
        heads = m.nheads // 2
        m.conv1d.x_head_group_range = m.qchunk_scan.x_head_group_range = torch.tensor([[1, heads], [3, heads]], dtype=torch.int32, device=dev)
    h = _ri(dev, g, batch, 1, d_model)
    conv, ssm = _states(m, dev, g, batch, dtype, width)
    conv2, ssm2 = conv.clone(), ssm.clone()
    out = _layer_call.call(m, h, conv, ssm, True)
    assert out is not None
    _close(out[:, 0], m._step_modules(h, conv2, ssm2), (conv, conv2), (ssm, ssm2))


@pytest.mark.parametrize("batch,seqlen", [(1, 0), (5, 0), (2, 37), (3, 900)])
@pytest.mark.parametrize("norm_first", [False, True])
def test_norm_of_whole_rows_of_4096(dev, batch, seqlen, norm_first):
    """One norm group a row, in the transform's launch: one row, a few, more than the chip holds workgroups (seqlen 0: a step)."""
    m, g = _mamba2(lambda d, *a, **k: W8A8QMamba2(2048, *a, **{**k, "ngroups": 1}), dev, seed=batch)
    m.norm.norm_before_gate = norm_first
    c, q = m.conv1d, m.qchunk_scan                                 # (the tables of two groups: the first one's)
    c.x_out_scales, c.B_out_scales, c.C_out_scales = c.x_out_scales[:1], c.B_out_scales[:1], c.C_out_scales[:1]
    c.x_head_group_range = torch.tensor([[1, m.nheads]], dtype=torch.int32, device=dev)
    c.x_dim_group_range = c.x_dim_group_range[:1].contiguous()
    q.x_scales, q.B_scale, q.C_scale = c.x_out_scales, c.B_out_scales, c.C_out_scales
    q.x_head_group_range, q.x_dim_group_range = c.x_head_group_range, c.x_dim_group_range
    q.ssm_state_scale = q.ssm_state_scale[:1].contiguous()
    step = seqlen == 0
    h = _ri(dev, g, batch, max(seqlen, 1), 2048)
    conv, ssm = _states(m, dev, g, batch, torch.float32, 4)
    conv2, ssm2 = conv.clone(), ssm.clone()
    out = _layer_call.call(m, h, conv, ssm, step)
    assert out is not None and m.norm.group_size in (None, 4096)
    _close(out[:, 0] if step else out, m._step_modules(h, conv2, ssm2) if step else m._forward_modules(h, conv2, ssm2), (conv, conv2), (ssm, ssm2))


@pytest.mark.parametrize("d_model,batch,seqlen", [(768, 1, 65), (768, 16, 33), (1536, 1, 515), (1536, 12, 70), (2560, 16, 31), (3072, 3, 100)])
def test_forward_of_a_wide_layer(dev, d_model, batch, seqlen):
    """dt_proj inside the scan: ranks of 48, 96, 160 and 192, the time over waves, eight and four lanes per channel, both at once."""
    m, g = _mamba1(W8A8QMamba, dev, seed=seqlen, d_model=d_model)
    h = _ri(dev, g, batch, seqlen, d_model)
    conv, ssm = _states(m, dev, g, batch, torch.float32, 4)
    conv2, ssm2 = conv.clone(), ssm.clone()
    out = _layer_call.call(m, h, conv, ssm, False)
    want = m._forward_modules(h, conv2, ssm2)
    _close(out, want, (conv, conv2), (ssm, ssm2))


@pytest.mark.parametrize("cls,build", MIXERS[:1] + MIXERS[3:])
def test_changed_modules_are_seen(dev, cls, build):
    m, g = build(cls, dev, seed=5)
    h = _ri(dev, g, 2, 20, 256)
    first = m.forward(h)
    m.had.x_H_scale *= 2.0                                     # a scale, by value
    second = m.forward(h)
    assert not torch.equal(first, second) and torch.equal(second, m._forward_modules(h, None, None))
    m.conv1d.weight = m.conv1d.weight.flip(0).contiguous()     # a buffer, by identity
    third = m.forward(h)
    assert not torch.equal(third, second) and torch.equal(third, m._forward_modules(h, None, None))
    seen = []
    hook = m.conv1d.register_forward_hook(lambda *a: seen.append(1))
    assert torch.equal(m.forward(h), third) and seen           # hooked modules run one by one
    hook.remove()


@pytest.mark.parametrize("cls,build", MIXERS)
def test_weights_held_as_parameters_are_followed(dev, cls, build):
    """A weight that is a Parameter (no buffer) when the first call is made, replaced before the second."""
    m, g = build(cls, dev, seed=6)
    h = _ri(dev, g, 2, 20, 256)
    outs = []
    for turn in range(3):
        w = m.out_proj.weight
        # (int8 weights are the transposed view of contiguous rows)
        w = w.roll(turn, 0) if w.dtype == torch.uint8 else w.t().roll(turn, 0).contiguous().t()
        if turn == 0:
            del m.out_proj._buffers["weight"]
        m.out_proj.weight = torch.nn.Parameter(w, requires_grad=False)
        outs.append(_layer_call.call(m, h, None, None, False))
        want = m._forward_modules(h, None, None)
        # (as in _close: fp16 scan outputs may differ in the last place; other rows of the weight differ by the whole range)
        assert outs[-1] is not None and float((outs[-1].float() - want.float()).abs().max()) <= 2e-2 * float(want.float().abs().max()), turn
        del w
    assert not torch.equal(outs[0], outs[1]) and not torch.equal(outs[1], outs[2])


@pytest.mark.parametrize("cls,build", MIXERS)
def test_replaced_methods_are_called(dev, cls, build, monkeypatch):
    m, g = build(cls, dev, seed=7)
    h = _ri(dev, g, 2, 20, 256)
    first, seen = m.forward(h), []

    def noting(f):
        return lambda *a, **k: (seen.append(f), f(*a, **k))[1]

    def runs_the_modules():
        seen.clear()
        out = m.forward(h)
        # (as in _close: fp16 scan outputs may differ in the last place)
        assert seen and float((out.float() - first.float()).abs().max()) <= 2e-2 * float(first.float().abs().max())

    m.conv1d.forward = noting(m.conv1d.forward)                # on the instance
    runs_the_modules()
    del m.conv1d.forward
    m.out_proj._call_impl = noting(m.out_proj._call_impl)
    runs_the_modules()
    del m.out_proj._call_impl
    if not hasattr(m, "norm"):
        kept = m.had.transform_fn
        m.had.transform_fn = noting(kept)
        runs_the_modules()
        m.had.transform_fn = kept
    with monkeypatch.context() as patch:                       # on the class
        patch.setattr(type(m.conv1d), "forward", noting(type(m.conv1d).forward))
        runs_the_modules()
    seen.clear()
    assert torch.equal(m.forward(h), first) and not seen and _layer_call.call(m, h, None, None, False) is not None


@pytest.mark.parametrize("cls,build", MIXERS)
def test_unaligned_hidden_states(dev, cls, build):
    """Contiguous, 8 bytes off: the W8A8 Mamba1 forward pads token counts that are no multiple of 16 and so takes it; where the
    modules refuse it, so does the mixer, with the states as they were."""
    m, g = build(cls, dev, seed=8)
    for batch, seqlen in ((2, 21), (1, 32)):
        h = torch.empty(batch * seqlen * 256 + 8, dtype=torch.int8, device=dev)[8:].view(batch, seqlen, 256)
        h.copy_(_ri(dev, g, batch, seqlen, 256))
        assert h.is_contiguous() and h.data_ptr() % 16 == 8
        if cls is W8A8QMamba and seqlen == 21:
            want = m.forward(h.clone())
            assert float((m.forward(h).float() - want.float()).abs().max()) <= 2e-2 * float(want.float().abs().max())
        else:
            with pytest.raises(RuntimeError):
                m.forward(h)
    conv, ssm = _states(m, dev, g, 2, torch.int8, 4)
    kept = conv.clone(), ssm.clone()
    with pytest.raises(RuntimeError):
        m.step(h[:, :2].reshape(2, 1, 256), conv, ssm)
    assert torch.equal(conv, kept[0]) and torch.equal(ssm, kept[1])


@pytest.mark.parametrize("cls,build", MIXERS)
def test_a_scale_held_as_a_tensor_may_change_in_place(dev, cls, build):
    m, g = build(cls, dev, seed=9)
    h = _ri(dev, g, 2, 20, 256)
    want = [m.forward(h)]
    m.had.x_H_scale *= 2.0
    want.append(m.forward(h))
    m.had.x_H_scale = torch.tensor(m.had.x_H_scale / 2.0)
    got = [m.forward(h)]
    m.had.x_H_scale.mul_(2.0)
    got.append(m.forward(h))
    for a, b in zip(got, want):                              # (as in _close: fp16 scan outputs may differ in the last place)
        assert float((a.float() - b.float()).abs().max()) <= 2e-2 * float(b.float().abs().max())
    assert not torch.equal(got[0], got[1])
