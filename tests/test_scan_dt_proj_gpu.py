"""The step size codes that the scan of a layer call makes itself, to the bit.  They are not written anywhere, so the scan is
made to show them: with a decay of exp(-100) and less the fp32 state after a prompt is B * (step size * u) of its last step
alone, and the step sizes of neighbouring codes are at least 0.7 % apart.  Prompts of every length up to more than a tile of
steps put that last step at every place of a tile."""
import pytest
import torch

from quamba_amd import W8A8QMamba, _layer_call
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


# ranks 16, 48, 96, 128, 160, 192; sixteen and eight lanes per channel, segments, four lanes, both kinds at once
@pytest.mark.parametrize("d_model,batch,lengths", [
    (256, 2, list(range(1, 40)) + [515]), (768, 1, list(range(1, 70)) + [513, 1030]), (1536, 1, list(range(30, 70)) + [777]),
    (2048, 9, list(range(1, 40))), (2560, 8, list(range(1, 40)) + [129]), (2560, 16, [1, 31, 32, 33, 70]), (3072, 3, list(range(1, 40)) + [600])])
def test_codes(dev, d_model, batch, lengths):
    m, g = _mamba1(W8A8QMamba, dev, seed=d_model + batch, d_model=d_model)
    s = m.selective_scan
    s.A_log = torch.full_like(s.A_log, 127)                    # A = -exp(12.7): step sizes from 1.6e-3 up decay by exp(-500)
    s.A_scale, s.dt_scale = torch.tensor(A_LOG_SCALE, device=dev), torch.tensor(DT_SCALE, device=dev)
    s.dt_bias = torch.zeros_like(s.dt_bias)
    m.dt_proj.b = m.dt_proj.b * 6                              # codes over the whole range
    table = torch.nn.functional.softplus(torch.arange(-128, 128, device=dev, dtype=torch.float64) * DT_SCALE)
    shown = 0
    for seqlen in lengths:
        h = _ri(dev, g, batch, seqlen, d_model)
        ssm = torch.zeros(batch, m.d_inner, m.d_state, device=dev)
        assert _layer_call.call(m, h, None, ssm, False) is not None, "the library call has to take this"
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
