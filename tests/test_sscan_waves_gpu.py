"""The scan that cuts the time over the waves of a workgroup, with named lanes and waves: one wave, the most there can be, lengths
of a step, around a wave's steps, around a block of all waves and of several blocks, channel counts that are no multiple of a
workgroup's.  Against the seqlen-major scan (which test_sscan_gpu.py holds to the oracle), with the bars of
test_sscan_token_major_gpu.py."""
import pytest
import torch

from quamba_amd import ops
from tests import launched
from tests.test_sscan_token_major_gpu import _inputs, _token_major

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes,waves", [(4, 1), (4, 5), (4, 12), (8, 1), (8, 4), (8, 16)])
@pytest.mark.parametrize("batch,dim,dtype,with_z", [(1, 4, torch.float32, True), (2, 148, torch.int8, True), (1, 300, torch.float32, False)])
def test_waves(dev, lanes, waves, batch, dim, dtype, with_z):
    steps = 16 if lanes == 4 else 32
    block = steps * waves
    for seqlen in sorted({1, steps - 1, steps + 1, block - 1, block, block + 1, 2 * block + steps, 3 * block + 3}):
        d, s = _inputs(dev, batch, dim, seqlen, seed=dim + seqlen)
        rows = lambda a: a.transpose(1, 2).contiguous()
        B, Cm = rows(d["bc"][:, :, 8:24])[:, None], rows(d["bc"][:, :, 24:40])[:, None]
        want, st = ops.sscan_fwd(rows(d["u"]), s["u"], rows(d["dt"]), s["dt"], d["A"], s["A"], B, s["B"], Cm, s["C"], s["st"], d["D"], s["D"],
                                 rows(d["z"]) if with_z else None, s["z"] if with_z else None, d["db"], s["db"], True, state_dtype=dtype)
        out, state = _token_major(d, s, dtype, with_z, 0, (64 if lanes == 4 else 96) + waves - 1)
        assert bool(((out.float() - want.float()).abs() <= 1e-3 + 2e-3 * want.float().abs()).all()), seqlen
        a, b = state.float(), st[:, :, 0].float()
        if dtype == torch.int8:
            assert float((a - b).abs().max()) <= 1
        else:
            assert float((a - b).abs().max()) <= 1e-4 * float(b.abs().max())


@pytest.mark.parametrize("dim,seqlen", [(1536, 300), (512, 90), (5120, 40)])
@pytest.mark.parametrize("sizes", [range(-127, -60), range(-127, 128)])
def test_step_sizes_below_zero(dev, dim, seqlen, sizes):
    """Without softplus decays may grow without bounds, and a state that is zero until the last step stays zero: the grown product of many
    decays must not meet it.  (Growth of exp(1.3 x 11) a step, 88 is the largest exponent of fp32.)"""
    d, s = _inputs(dev, 1, dim, seqlen, seed=dim)
    g = torch.Generator(device=dev).manual_seed(seqlen)
    d["u"][:, :-1] = 0
    d["dt"] = torch.randint(sizes.start, sizes.stop, d["dt"].shape, dtype=torch.int8, device=dev, generator=g)
    d["A"].fill_(120)
    s["dt"], s["db"] = s["dt"] / 3, s["db"] / 100
    (out, state), names = launched.kernels(lambda: _token_major(d, s, torch.float32, True, 0, softplus=0))
    step = s["dt"] * d["dt"][:, -1].double() + s["db"] * d["db"].double()
    want = (step * s["u"] * d["u"][:, -1].double())[..., None] * s["B"] * d["bc"][:, -1, None, 8:24].double()
    assert float((state - want).abs().max()) <= 1e-5 * float(want.abs().max())
    assert not bool(out[:, :-1].any()) and bool(out.isfinite().all())
    launched.expect(names, "scan_tm_kernel<8, true, true, 0>")


def _in_64_bits(d, s):
    """Outputs and last state of the scan, one step after the other."""
    f = lambda k, codes: s[k].double() * codes.double()
    u, B, C, A = f("u", d["u"]), f("B", d["bc"][:, :, 8:24]), f("C", d["bc"][:, :, 24:40]), -torch.exp(f("A", d["A"]))
    dt = torch.nn.functional.softplus(f("dt", d["dt"]) + f("db", d["db"]))
    h, ys = torch.zeros(*u.shape[::2], 16, dtype=torch.float64, device=u.device), []
    for t in range(u.shape[1]):
        h = h * torch.exp(dt[:, t, :, None] * A) + (dt[:, t] * u[:, t])[..., None] * B[:, t, None]
        ys.append((h * C[:, t, None]).sum(-1))
    z = f("z", d["z"])
    return (torch.stack(ys, 1) + f("D", d["D"]) * u) * z * torch.sigmoid(z), h


@pytest.mark.parametrize("batch,dim,seqlen", [(1, 1536, 512), (2, 512, 1100), (1, 3072, 77)])
def test_error_against_64_bits(dev, batch, dim, seqlen):
    """Cut over waves the sums are no less exact than in one pass: outputs as near as fp16 rounds them (2.1e-4; what fp32 adds is beyond
    the fourth figure), states within what the order of fp32 sums changes (1.4 to 1.9e-7 in one pass, 0.8 to 1.0 of that over waves)."""
    d, s = _inputs(dev, batch, dim, seqlen, seed=seqlen)
    d["db"].fill_(-127)                                        # (step sizes of 0.007 to 0.08: states that remember hundreds of steps)
    s["dt"] = s["dt"] / 3
    y, h = _in_64_bits(d, s)
    off = lambda got, want: float((got.double() - want).norm() / want.norm())
    one_pass = off(_token_major(d, s, torch.float32, True, 0, 8)[1], h)
    for lanes in (16, 64 + 3, 64 + 11, 96 + 7, 96 + 15):
        out, state = _token_major(d, s, torch.float32, True, 0, lanes)
        assert off(out, y) <= 1.01 * off(y.half(), y), lanes
        assert off(state, h) <= 1.1 * one_pass, (lanes, off(state, h), one_pass)
