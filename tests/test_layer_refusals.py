"""The layer calls of the C ABI refuse what one of their kernels would refuse before the first launch: a step advances both
states in place and could not be made again another way.  Nothing here is launched: every block is wrong in one place."""
import ctypes as C

import pytest

from quamba_amd import _lib

NULL, SHAPE, STRIDE, UNSUPPORTED = -1, -2, -3, -4
AT = 1 << 20                                                 # an aligned address that is never read


def _linear(n, k, bits=8):
    p = _lib.QaLinearParams()
    p.n, p.k, p.bits, p.col_numel, p.alpha = n, k, bits, 1 if bits == 8 else n, 1.0
    p.weight = p.col_scale = p.row_scale = AT
    p.s_group = AT if bits == 4 else None
    return p


def _call_fields(p):
    p.batch, p.seqlen, p.conv_state_len, p.d_conv = 2, 1, 4, 4
    p.hidden = p.out = p.conv_state = p.ssm_state = p.workspace = AT
    p.workspace_bytes = 1 << 40
    return p


def _mamba1():
    p = _call_fields(_lib.QaMamba1Params())
    p.d_model, p.d_inner, p.d_state, p.dt_rank = 256, 512, 16, 16
    p.in_proj, p.x_proj, p.dt_proj, p.out_proj = _linear(1024, 256), _linear(48, 512), _linear(512, 16), _linear(256, 512)
    for name in ("conv_weight", "A_log", "D", "dt_bias", "A_scale", "D_scale", "dt_bias_scale", "u_scale", "dt_scale", "B_scale", "C_scale",
                 "z_scale", "ssm_state_scale"):
        setattr(p, name, AT)
    return p


def _mamba2():
    p = _call_fields(_lib.QaMamba2Params())
    p.d_model, p.d_inner, p.d_state, p.headdim, p.ngroups, p.chunk_size, p.norm_group_size = 256, 512, 64, 64, 1, 64, 512
    p.in_proj, p.out_proj = _linear(1168, 256), _linear(256, 512)
    for name in ("conv_weight", "x_out_scales", "B_out_scales", "C_out_scales", "A_log", "D", "A_log_scale", "D_scale", "dt_scale", "x_scales",
                 "B_scale", "C_scale", "ssm_state_scale", "norm_weight"):
        setattr(p, name, AT)
    return p


def _set(*path_and_value):
    *path, value = path_and_value

    def change(p):
        for name in path[:-1]:
            p = getattr(p, name)
        setattr(p, path[-1], value)
    return change


BOTH = [
    (_set("hidden", AT + 8), STRIDE), (_set("workspace", AT + 16), STRIDE), (_set("workspace_bytes", 1), STRIDE), (_set("out", None), NULL),
    (_set("in_proj", "weight", AT + 8), STRIDE), (_set("out_proj", "weight", AT + 4), STRIDE), (_set("out_proj", "weight", None), NULL),
    (_set("out_proj", "row_scale", None), NULL), (_set("out_proj", "col_numel", 7), SHAPE), (_set("conv_state_len", 5), SHAPE),
    (_set("D_scale", None), NULL), (_set("dt_scale", None), NULL), (_set("B_scale", None), NULL),
    (_set("C_scale", None), NULL),
]
MAMBA1 = [(_set("A_scale", None), NULL), (_set("u_scale", None), NULL), (_set("z_scale", None), NULL), (_set("dt_bias_scale", None), NULL),
          (_set("ssm_state_scale", None), NULL), (_set("dt_proj", "bits", 4), SHAPE)]
MAMBA2 = [(_set("A_log_scale", None), NULL), (_set("x_scales", None), NULL), (_set("norm_weight", AT + 8), STRIDE), (_set("norm_group_size", 4), UNSUPPORTED),
          (_set("ssm_state_scale", None), NULL), (_set("nhead_groups", 2), NULL), (_set("conv_head_range", AT), NULL)]


@pytest.mark.parametrize("call", ["forward", "step"])
@pytest.mark.parametrize("family,build,change,status", [(1, _mamba1, *c) for c in BOTH + MAMBA1] + [(2, _mamba2, *c) for c in BOTH + MAMBA2])
def test_refused_before_the_first_launch(family, build, change, status, call):
    p = build()
    change(p)
    assert getattr(_lib.lib(), f"qa_mamba{family}_{call}")(C.byref(p), None) == status


def test_the_step_sizes_made_in_the_scan_need_no_workspace():
    """A codes' section for them only where dt_proj is a product of its own."""
    l, tokens = _lib.lib(), 8 * 640
    p = _mamba1()
    p.batch, p.seqlen = 8, 640
    in_scan = l.qa_mamba1_workspace_bytes(C.byref(p), 0)
    p.x_proj, p.dt_rank, p.dt_proj = _linear(240, 512), 208, _linear(512, 208)             # a rank the scan does not take
    assert l.qa_mamba1_workspace_bytes(C.byref(p), 0) - in_scan == tokens * (240 - 48) + tokens * 512


def test_sizes_no_kernel_takes_need_no_workspace():
    """Zero bytes: the caller runs the operators one by one, or tells its user."""
    l = _lib.lib()
    wide = lambda p: (setattr(p, "d_inner", 112), setattr(p, "in_proj", _linear(224, 256)), setattr(p, "x_proj", _linear(48, 112)),
                      setattr(p, "dt_proj", _linear(112, 16)), setattr(p, "out_proj", _linear(256, 112)))
    rank = lambda p: (setattr(p, "dt_rank", 20), setattr(p, "dt_proj", _linear(512, 20)), setattr(p, "x_proj", _linear(64, 512)))
    tokens = lambda p: (setattr(p, "batch", 4096), setattr(p, "seqlen", 4096))          # rows * columns past 32-bit offsets
    for change in (wide, rank, tokens):
        p = _mamba1()
        assert l.qa_mamba1_workspace_bytes(C.byref(p), 0) > 0
        change(p)
        assert l.qa_mamba1_workspace_bytes(C.byref(p), 0) == 0 and l.qa_mamba1_workspace_bytes(C.byref(p), 1) == 0
        assert l.qa_mamba1_forward(C.byref(p), None) in (SHAPE, UNSUPPORTED)
    for name, value, forward, step in (("chunk_size", 2048, False, True), ("headdim", 512, False, True), ("norm_group_size", 4, False, False), ("d_state", 512, True, False)):
        p = _mamba2()
        assert l.qa_mamba2_workspace_bytes(C.byref(p), 0) > 0 and l.qa_mamba2_workspace_bytes(C.byref(p), 1) > 0
        setattr(p, name, value)
        p.in_proj = _linear(2064, 256)                       # (columns enough for either)
        assert (l.qa_mamba2_workspace_bytes(C.byref(p), 0) > 0) == forward and (l.qa_mamba2_workspace_bytes(C.byref(p), 1) > 0) == step, name
