"""The step size codes that the scan of a layer call makes itself, to the bit.  They are not written anywhere, so the scan is
made to show them: with a decay of exp(-100) and less the fp32 state after a prompt is B * (step size * u) of its last step
alone, and the step sizes of neighbouring codes are at least 0.7 % apart.  Prompts of every length up to more than a tile of
steps put that last step at every place of a tile."""
import pytest
import torch

from quamba_amd import W8A8QMamba, _layer_call
from tests import launched
from tests.test_layer_call_gpu import _mamba1
from tests.test_mixer_variants_gpu import _ri

pytestmark = pytest.mark.gpu

DT_SCALE, A_LOG_SCALE = 0.05, 0.1


def _codes_of_the_modules(m, h):
    """u, dt and B codes of the last step, one operator after the other."""
    x = m.conv1d(m.in_proj.to_seqlen_last(h).chunk(2, dim=1)[0])
    rows = m.x_proj(x.transpose(1, 2).contiguous())
    dt = m.dt_proj.to_seqlen_last(rows[..., :m.dt_rank].contiguous())
    return x[:, :, -1], dt[:, :, -1], rows[:, -1, m.dt_rank:m.dt_rank + m.d_state]


def _mixer(dev, d_model, batch, dt_rank="auto"):
    m, g = _mamba1(lambda d, *a, **k: W8A8QMamba(d, *a, dt_rank=dt_rank, **k), dev, seed=d_model + batch, d_model=d_model)
    s = m.selective_scan
    s.A_log = torch.full_like(s.A_log, 127)                    # A = -exp(12.7): step sizes from 1.6e-3 up decay by exp(-500)
    s.A_scale, s.dt_scale = torch.tensor(A_LOG_SCALE, device=dev), torch.tensor(DT_SCALE, device=dev)
    s.dt_bias = torch.zeros_like(s.dt_bias)
    m.dt_proj.b = m.dt_proj.b * 6                              # codes over the whole range
    return m, g


def _last_codes(m, g, dev, batch, lengths, kernels=None):
    """kernels: one more length -> what the scan's kernels are called."""
    s = m.selective_scan
    table = torch.nn.functional.softplus(torch.arange(-128, 128, device=dev, dtype=torch.float64) * DT_SCALE)
    shown = 0
    for seqlen in lengths:
        h = _ri(dev, g, batch, seqlen, m.d_model)
        ssm = torch.zeros(batch, m.d_inner, m.d_state, device=dev)
        out, names = launched.kernels(lambda: _layer_call.call(m, h, None, ssm, False)) if kernels else (_layer_call.call(m, h, None, ssm, False), [])
        assert out is not None, "the library call has to take this"
        if kernels:
            launched.expect(names, *kernels[seqlen])
        u, dt, B = _codes_of_the_modules(m, h)
        n = B.abs().float().argmax(1)                          # (the absolute value of -128 is not an int8)
        Bn = B.gather(1, n[:, None])[:, 0]
        found = ssm.double().gather(2, n[:, None, None].expand(batch, m.d_inner, 1))[..., 0]
        unit = float(s.u_scale) * u.double() * (float(s.B_scale) * Bn.double())[:, None]
        tells = unit != 0
        step = found[tells] / unit[tells]
        code = (step[:, None] - table).abs().argmin(1) - 128
        assert torch.equal(code, dt[tells].long()), seqlen
        assert float((step / table[code + 128] - 1).abs().max()) < 1e-5
        shown += int(tells.sum())
    assert shown > 100 * len(lengths) and len(set(dt.flatten().tolist())) > 100


# ranks 16, 48, 96, 128, 160, 192; the time over the waves of a workgroup, eight and four lanes per channel, both kinds at once
@pytest.mark.parametrize("d_model,batch,lengths", [
    (256, 2, list(range(1, 40)) + [515]), (768, 1, list(range(1, 70)) + [513, 1030]), (1536, 1, list(range(30, 70)) + [777]),
    (2048, 9, list(range(1, 40))), (2560, 8, list(range(1, 40)) + [129]), (2560, 16, [1, 31, 32, 33, 70]), (3072, 3, list(range(1, 40)) + [600])])
def test_codes(dev, d_model, batch, lengths):
    _last_codes(*_mixer(dev, d_model, batch), dev, batch, lengths)


# The time over waves of four and of eight lanes, with one, two and three 64-code pieces of the rank (64, 128 and 192 too: no remainder), up to
# twelve and up to sixteen waves: lengths around a wave's steps, a block of all waves and several blocks, whose later ones have the rows of
# dt_proj's input requested during the block before.  Ranks that belong to no default width reach what narrow layers of a high rank do.
FOUR, EIGHT, SIXTEEN = ("scan_waves_kernel<4, 12, true, {}>",), ("scan_waves_kernel<8, 12, true, {}>",), ("scan_waves_kernel<8, 16, true, {}>",)
SEGMENTS = ("scan_tm_kernel<8, false, false, {}>", "scan_tm_kernel<8, true, true, {}>")


@pytest.mark.parametrize("d_model,dt_rank,batch,lengths", [
    (768, "auto", 2, {97: FOUR, 112: FOUR, 113: FOUR, 200: FOUR}), (768, "auto", 1, {500: SIXTEEN, 512: SIXTEEN, 513: EIGHT, 1000: SIXTEEN, 1024: SIXTEEN, 1025: EIGHT, 1500: SIXTEEN}),
    (1024, "auto", 1, {400: SIXTEEN, 1000: SIXTEEN}),
    (1536, "auto", 1, {37: FOUR, 48: FOUR, 49: FOUR, 300: FOUR, 777: FOUR}), (1536, "auto", 2, {67: EIGHT, 96: EIGHT, 97: EIGHT, 400: EIGHT, 511: EIGHT}),
    (2560, "auto", 1, {34: FOUR, 48: FOUR, 49: FOUR, 64: FOUR, 65: EIGHT, 97: EIGHT, 256: EIGHT, 257: FOUR, 300: FOUR, 700: EIGHT, 769: EIGHT}),
    (3072, "auto", 1, {512: EIGHT, 515: EIGHT}),
    (768, 96, 1, {500: SIXTEEN, 1023: SIXTEEN}), (768, 128, 1, {512: SIXTEEN, 1024: SIXTEEN}), (768, 160, 1, {500: SIXTEEN, 1000: SIXTEEN, 1500: SIXTEEN}),
    (256, "auto", 1, {1024: SEGMENTS, 1500: SEGMENTS}), (256, "auto", 2, {1088: SEGMENTS, 1300: SEGMENTS, 2000: SEGMENTS}),
    (256, 96, 1, {1500: SEGMENTS}), (256, 160, 2, {1300: SEGMENTS})])
def test_codes_over_waves_and_segments(dev, d_model, dt_rank, batch, lengths):
    m, g = _mixer(dev, d_model, batch, dt_rank)
    pieces = (m.dt_rank + 63) // 64
    _last_codes(m, g, dev, batch, lengths, {n: [k.format(pieces) for k in kernels] for n, kernels in lengths.items()})
