"""Performance cases: the four quantized mixers, prefill and decode, as a generation loop calls them.

A case is one call of a mixer on a token batch: ``forward`` over a prompt that also leaves the conv and the recurrent
state behind for decoding (prefill), or ``step`` over one token per sequence that advances both states in place
(decode).  One such call runs every operator of the package on the way: the projections (W8A8 or W4A8), the causal
conv, the selective scan or the SSD chunk scan (or their single-step forms), the gated norm, the Hadamard rotation.

Sizes are those of the model configurations that the benchmark and the tests use (widths 768 ... 2560, for the second
family also 4096 with eight groups); prompts have any length, so lengths that are no multiple of anything are drawn as
often as round ones.
"""
import math

import torch

from quamba_amd import W4A8QMamba, W4A8QMamba2, W8A8QMamba, W8A8QMamba2

MIXERS = {(1, 8): W8A8QMamba, (1, 4): W4A8QMamba, (2, 8): W8A8QMamba2, (2, 4): W4A8QMamba2}
STATE_DTYPES = {"int8": torch.int8, "fp32": torch.float32}
WIDTHS = {1: (768, 1024, 1536, 2048, 2560), 2: (768, 1024, 1536, 2048, 2560, 4096)}
D_STATE = {1: 16, 2: 128}
D_CONV, HEADDIM, CHUNK = 4, 64, 256
HEAD_GROUPS = DIM_GROUPS = 4                # grouped scales of x in the second family


def _case(name, family, bits, phase, d_model, batch, seqlen, state):
    case = {"family": family, "bits": bits, "phase": phase, "d_model": d_model, "batch": batch, "seqlen": seqlen, "state": state}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one user at a prompt, smallest model: the latency of a token (launches and host work count)
        _case("m1 w8 decode 1 x 768", 1, 8, "decode", 768, 1, 1, "int8"),
        # one user, largest model of the family, 4-bit weights: streaming the weights
        _case("m1 w4 decode 1 x 2560", 1, 4, "decode", 2560, 1, 1, "int8"),
        # a serving batch with the recurrent state kept in fp32 (the benchmark's decode configuration)
        _case("m1 w8 decode 64 x 2560", 1, 8, "decode", 2560, 64, 1, "fp32"),
        # one short prompt, smallest model (the first configuration of the benchmark)
        _case("m1 w8 prefill 1x512 x 768", 1, 8, "prefill", 768, 1, 512, "fp32"),
        # the benchmark's headline configuration, with the projections that lie between its four kernels
        _case("m1 w8 prefill 8x2048 x 2560", 1, 8, "prefill", 2560, 8, 2048, "fp32"),
        # a few prompts padded to the longest of them, a length that is a multiple of nothing
        _case("m1 w8 prefill 3x1021 x 2560", 1, 8, "prefill", 2560, 3, 1021, "int8"),
        # one prompt of odd length, 4-bit weights, a model in the middle of the range
        _case("m1 w4 prefill 1x777 x 1536", 1, 4, "prefill", 1536, 1, 777, "int8"),
        # second family: one user, 4-bit weights, largest model
        _case("m2 w4 decode 1 x 4096", 2, 4, "decode", 4096, 1, 1, "int8"),
        # a serving batch of the largest model: the fp32 states are most of the bytes
        _case("m2 w4 decode 64 x 4096", 2, 4, "decode", 4096, 64, 1, "fp32"),
        # one prompt of odd length
        _case("m2 w8 prefill 1x1531 x 2560", 2, 8, "prefill", 2560, 1, 1531, "int8"),
        # long prompts (the benchmark's chunk-scan configuration as a whole layer)
        _case("m2 w8 prefill 4x4096 x 2560", 2, 8, "prefill", 2560, 4, 4096, "fp32"),
        # the largest layer (the benchmark's W4A8 configuration)
        _case("m2 w4 prefill 16x1024 x 4096", 2, 4, "prefill", 4096, 16, 1024, "int8"),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    family, bits = rng.choice((1, 2)), rng.choice((8, 4))
    phase, state = rng.choice(("prefill", "decode")), rng.choice(("int8", "fp32"))
    d_model = rng.choice(WIDTHS[family])
    if phase == "decode":
        return _case(None, family, bits, phase, d_model, _log_uniform(rng, 1, 128), 1, state)
    seqlen = _log_uniform(rng, 16, 4096)
    if rng.random() < 0.5:
        seqlen = max(16, seqlen // 16 * 16)
    batch = _log_uniform(rng, 1, max(1, min(16, 12288 // seqlen)))
    return _case(None, family, bits, phase, d_model, batch, seqlen, state)


# ---------------------------------------------------------------------------------------------------------------------
# A mixer with random weights and the scales a calibration would give it
# ---------------------------------------------------------------------------------------------------------------------
class _Maker:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.dev = torch.device("cuda")
        self.g = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device=self.dev)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device=self.dev) * (hi - lo) + lo

    def codes(self, std, *shape):
        """int8 codes of normally distributed values, calibrated so that few of them saturate."""
        return (self.normal(*shape) * std).round_().clamp_(-127, 127).to(torch.int8)

    def quantized(self, x):
        scale = float(x.abs().max()) / 127
        return (x / scale).round().to(torch.int8), scale

    def activations(self, *shape):
        """N(0, 1) with one channel in a hundred 20 times as large, quantized by the largest value."""
        x = self.normal(*shape)
        outlier = torch.randperm(shape[-1], generator=self.g, device=self.dev)[: -(-shape[-1] // 100)]
        x[..., outlier] *= 20.0
        return self.quantized(x)

    def scalar(self, v):
        return torch.tensor(float(v), dtype=torch.float32, device=self.dev)


ACT_STD = 25.0      # standard deviation of the codes of a calibrated activation (the largest of many is near 127)
W_STD = 25.0        # the same for weights


def _fill_linear(mk, lin, in_rms, gain, spread=1.0):
    """Random weights; an output whose standard deviation is ``gain`` when the input codes have root mean square
    ``in_rms``.  ``spread``: the range of the per-channel scales where the layer has them."""
    k = lin.in_features
    if hasattr(lin, "s_group"):
        nib = lambda: (mk.normal(lin.size_n, k // 2) * 2.6 + 8.0).round_().clamp_(0, 15).to(torch.uint8)
        lin.weight = nib() | (nib() << 4)
        lin.s_group = mk.uniform(6.0, 12.0, k // 128, lin.size_n).half()
        unit = gain / (math.sqrt(k) * in_rms * 2.6 * 9.2)
        lin.input_scale = mk.scalar(0.05)
        lin.s_channel = mk.uniform(1.0 / spread, spread, 1, lin.size_n) * (unit / 0.05)
    else:
        n = lin.out_features + lin.pad_out
        w = mk.codes(W_STD, n, k)
        w[lin.out_features:] = 0
        lin.weight = w.t()
        unit = gain / (math.sqrt(k) * in_rms * W_STD)
        lin.a = torch.full((1, 1), 0.05, device=mk.dev)
        if lin.b.numel() > 1:
            lin.b = mk.uniform(1.0 / spread, spread, 1, n) * (unit / 0.05)
        else:
            lin.b = torch.full((1, 1), unit / 0.05, device=mk.dev)
        lin.alpha = float(lin.a * lin.b.reshape(-1)[0])


def _inverse_softplus(y):
    return y + torch.log(-torch.expm1(-y))


def _step_size_bias(mk, n):
    return _inverse_softplus(torch.exp(mk.uniform(math.log(1e-3), math.log(1e-1), n)))


IN_SCALE = 0.04       # in_proj's output: values of unit variance
CONV_SCALE = 0.035    # the conv's output after SiLU: 4.4 is the largest code
CONV_RMS = 12.0       # root mean square of its codes
DT_SCALE = 0.03       # the step sizes' offset before softplus


def _conv(mk, n):
    w, ws = mk.quantized(mk.uniform(-0.5, 0.5, n, D_CONV))
    b, bs = mk.quantized(mk.uniform(-0.5, 0.5, n))
    return w, ws, b, bs


def _mixer1(mk, case, hidden_rms):
    m = MIXERS[1, case["bits"]](case["d_model"], D_STATE[1], D_CONV, device=mk.dev, state_dtype=STATE_DTYPES[case["state"]])
    _fill_linear(mk, m.in_proj, hidden_rms, ACT_STD)
    _fill_linear(mk, m.x_proj, CONV_RMS, ACT_STD)
    _fill_linear(mk, m.dt_proj, ACT_STD, ACT_STD)
    _fill_linear(mk, m.out_proj, ACT_STD, 1.0)
    c = m.conv1d
    c.weight, c.weight_scale, c.bias, c.bias_scale = _conv(mk, m.d_inner)
    c.input_scale, c.output_scale = IN_SCALE, CONV_SCALE
    s = m.selective_scan
    s.A_log, a_scale = mk.quantized(torch.log(mk.uniform(1.0, 16.0, m.d_inner, D_STATE[1])))
    s.D, d_scale = mk.quantized(torch.ones(m.d_inner, device=mk.dev))
    s.dt_bias, db_scale = mk.quantized(_step_size_bias(mk, m.d_inner))
    for name, v in (("A_scale", a_scale), ("D_scale", d_scale), ("dt_bias_scale", db_scale), ("u_scale", CONV_SCALE),
                    ("dt_scale", DT_SCALE), ("B_scale", 0.04), ("C_scale", 0.04), ("z_scale", IN_SCALE), ("ssm_state_scale", 0.01)):
        setattr(s, name, mk.scalar(v))
    m.had.x_H_scale = 0.02
    return m


def _mixer2(mk, case, hidden_rms):
    groups = 8 if case["d_model"] == 4096 else 1
    m = MIXERS[2, case["bits"]](case["d_model"], D_STATE[2], D_CONV, 2, HEADDIM, ngroups=groups, chunk_size=CHUNK, device=mk.dev,
                                state_dtype=STATE_DTYPES[case["state"]], x_nhead_group=HEAD_GROUPS, x_ndim_group=DIM_GROUPS)
    _fill_linear(mk, m.in_proj, hidden_rms, ACT_STD, spread=1.2)
    _fill_linear(mk, m.out_proj, ACT_STD, 1.0, spread=1.2)
    bc, c = groups * D_STATE[2], m.conv1d
    parts = [_conv(mk, n) for n in (m.d_ssm, bc, bc)]
    c.weight, c.bias = torch.cat([p[0] for p in parts]), torch.cat([p[2] for p in parts])
    c.wx_scale, c.wB_scale, c.wC_scale = (p[1] for p in parts)
    c.bx_scale, c.bB_scale, c.bC_scale = (p[3] for p in parts)
    c.x_scale = c.B_scale = c.C_scale = IN_SCALE
    ends = lambda total, n: torch.arange(1, n + 1, dtype=torch.int32, device=mk.dev) * (total // n)
    c.x_head_group_range = ends(m.nheads // groups, HEAD_GROUPS).repeat(groups, 1)
    c.x_dim_group_range = ends(HEADDIM, DIM_GROUPS).repeat(groups, HEAD_GROUPS, 1)
    c.x_out_scales = mk.uniform(0.8, 1.2, groups, HEAD_GROUPS, DIM_GROUPS) * CONV_SCALE
    c.B_out_scales, c.C_out_scales = (mk.uniform(0.9, 1.1, groups) * CONV_SCALE for _ in range(2))
    s = m.qchunk_scan
    s.A_log, a_scale = mk.quantized(mk.uniform(0.0, math.log(16.0), m.nheads))
    s.D, d_scale = mk.quantized(torch.ones(m.nheads, device=mk.dev))
    s.dt_bias = _step_size_bias(mk, m.nheads).half()
    s.A_log_scale, s.D_scale, s.dt_scale = mk.scalar(a_scale), mk.scalar(d_scale), mk.scalar(DT_SCALE)
    s.x_scales, s.B_scale, s.C_scale = c.x_out_scales, c.B_out_scales, c.C_out_scales
    s.x_head_group_range, s.x_dim_group_range = c.x_head_group_range, c.x_dim_group_range
    s.ssm_state_scale = mk.uniform(0.8, 1.2, groups, HEAD_GROUPS, DIM_GROUPS, D_STATE[2]) * 2e-3
    m.norm.weight = (1.0 + 0.1 * mk.normal(m.d_ssm)).half()
    m.norm.z_scale = IN_SCALE
    m.had.x_H_scale = 0.045
    return m


def prepare(case, seed):
    mk = _Maker(seed)
    hidden, _ = mk.activations(case["batch"], case["seqlen"], case["d_model"])
    hidden_rms = float(hidden.float().square().mean().sqrt())
    m = (_mixer1 if case["family"] == 1 else _mixer2)(mk, case, hidden_rms)
    conv_state, ssm_state = m.allocate_inference_cache(case["batch"])
    if case["phase"] == "decode":
        # the states that a prompt left behind
        conv_state.copy_(mk.codes(ACT_STD, *conv_state.shape))
        if ssm_state.dtype == torch.int8:
            ssm_state.copy_(mk.codes(ACT_STD, *ssm_state.shape))
        else:
            ssm_state.copy_(mk.normal(*ssm_state.shape) * 0.1)
    return {"mixer": m, "hidden": hidden, "conv_state": conv_state, "ssm_state": ssm_state, "decode": case["phase"] == "decode"}


def run(state):
    m, conv_state, ssm_state = state["mixer"], state["conv_state"], state["ssm_state"]
    if state["decode"]:
        out, conv_state, ssm_state = m.step(state["hidden"], conv_state, ssm_state)
    else:
        out = m(state["hidden"], conv_state=conv_state, ssm_state=ssm_state)
    return {"out": out, "conv_state": conv_state, "ssm_state": ssm_state}


def work(case):
    """Weights, inputs and outputs once; the projections' products and the recurrence (a multiplication by the decay
    and two multiply-adds per channel, state and token)."""
    d, tokens, n = case["d_model"], case["batch"] * case["seqlen"], D_STATE[case["family"]]
    inner = 2 * d
    wide = case["bits"] / 8 * (1 + 1 / 32 if case["bits"] == 4 else 1)     # bytes a weight (with its share of the group scales)
    if case["family"] == 1:
        rank = math.ceil(d / 16)
        sized = d * 2 * inner + inner * (rank + 2 * n) + inner * d
        weights, products = sized * wide + rank * inner, sized + rank * inner
        small = inner * (D_CONV + 1 + n + 2)
        conv_dim = inner
    else:
        groups = 8 if d == 4096 else 1
        sized = d * (2 * inner + 2 * groups * n + inner // HEADDIM) + inner * d
        weights, products = sized * wide, sized
        conv_dim = inner + 2 * groups * n
        small = conv_dim * (D_CONV + 1) + 2 * inner
    state = case["batch"] * (inner * n * (4 if case["state"] == "fp32" else 1) + conv_dim * D_CONV)
    if case["phase"] == "decode":
        state *= 2
    return {"bytes": weights + small + state + tokens * d * 3, "flops": 2.0 * tokens * products + 5.0 * tokens * inner * n}


def tolerance(case):
    """The scan's fp16 output (and the order of its sums) may differ in its last place; a few of the int8 codes made
    from it then sit on the other side of a tie, before out_proj and in an int8 recurrent state."""
    return {"rel": 1e-2, "max": 0.1, "differ": 5e-3}
