"""The forward xBC conv with its grouped output scales looked up across a wave, against the kernel of one thread per output that takes
any alignment: edges of the tables, of the channel blocks and of the runs of steps."""
import ctypes

import pytest
import torch

from quamba_amd import _lib
from tests import launched

pytestmark = pytest.mark.gpu


def _ends(count, total, g):
    """`count` increasing ends, the last one `total`."""
    return sorted(torch.randperm(total - 1, generator=g)[: count - 1].add(1).tolist()) + [total]


# batch, seqlen, ssd groups, heads a group, headdim, d_state, head groups, dim groups; the kernel's output scales
CASES = [(1, 5, 1, 24, 64, 128, 4, 4, 1), (1, 1531, 1, 80, 64, 128, 4, 4, 1), (2, 300, 8, 16, 64, 128, 8, 8, 1), (3, 1000, 1, 32, 64, 128, 1, 1, 1), (1, 77, 1, 9, 128, 64, 3, 5, 1),
         (2, 130, 2, 64, 4, 16, 8, 3, 1), (1, 64, 3, 1, 256, 8, 1, 8, 1), (4, 700, 1, 7, 32, 4, 5, 2, 1), (2, 9, 1, 3, 16, 12, 2, 7, 1), (3, 4, 1, 1, 8, 4, 1, 2, 1),
         (1, 40, 2, 3, 64, 128, 2, 2, 2), (1, 40, 1, 6, 96, 128, 2, 2, 2), (1, 40, 1, 12, 64, 128, 9, 2, 2)]


@pytest.mark.parametrize("batch,seqlen,groups,heads,headdim,d_state,hg,dg,kind", CASES)
@pytest.mark.parametrize("silu,bias", [(1, True), (0, False)])
def test_grouped_scales_across_a_wave(dev, batch, seqlen, groups, heads, headdim, d_state, hg, dg, kind, silu, bias):
    g = torch.Generator().manual_seed(batch * seqlen + headdim)
    x_dim, bc = groups * heads * headdim, groups * d_state
    dim = x_dim + 2 * bc
    codes = lambda *shape: torch.randint(-128, 128, shape, dtype=torch.int8, generator=g).to(dev)
    xBC, w, b = codes(batch, seqlen, dim), codes(dim, 4), codes(dim)
    scales = [(torch.rand(n, generator=g) * 0.05 + 0.003).to(dev) for n in (groups * hg * dg, groups, groups)]
    hr = torch.tensor([e for _ in range(groups) for e in _ends(hg, max(heads, hg), g)], dtype=torch.int32, device=dev)
    dr = torch.tensor([e for _ in range(groups * hg) for e in _ends(dg, max(headdim, dg), g)], dtype=torch.int32, device=dev)
    hr.view(groups, hg)[:, -1] = heads

    def run(pad):                                          # a pad of one byte: no aligned words, the general kernel
        outs = [torch.full((batch, seqlen, n + pad), 99, dtype=torch.int8, device=dev) for n in (x_dim, bc, bc)]
        p = _lib.QaConv2Params()
        p.batch, p.dim, p.seqlen, p.width, p.silu_activation, p.x_dim, p.x_headdim, p.d_state, p.n_groups = batch, dim, seqlen, 4, silu, x_dim, headdim, d_state, groups
        p.nhead_groups, p.ndim_groups, p.conv_state_len = hg, dg, 4
        p.xBC_batch_stride, p.xBC_l_stride, p.xBC_c_stride = seqlen * dim, dim, 1
        for name, t in zip("xBC", outs):
            setattr(p, name + "_batch_stride", t.stride(0)); setattr(p, name + "_l_stride", t.stride(1)); setattr(p, name + "_c_stride", 1); setattr(p, name, t.data_ptr())
        p.weight_c_stride, p.weight_width_stride = 4, 1
        p.xBC, p.weight, p.bias = xBC.data_ptr(), w.data_ptr(), b.data_ptr() if bias else None
        p.x_out_scales, p.B_out_scales, p.C_out_scales, p.x_head_group_range, p.x_dim_group_range = (t.data_ptr() for t in (*scales, hr, dr))
        p.scale_x, p.scale_B, p.scale_C, p.scale_wx, p.scale_wB, p.scale_wC, p.scale_bx, p.scale_bB, p.scale_bC = 0.02, 0.021, 0.022, 0.005, 0.006, 0.007, 0.004, 0.005, 0.006
        _, names = launched.kernels(lambda: _lib.check(_lib.lib().qa_quamba2_conv1d_fwd(ctypes.byref(p), _lib.current_stream(dev)), "conv2"))
        return [t[..., :n] for t, n in zip(outs, (x_dim, bc, bc))], names

    want, _ = run(1)
    got, names = run(0)
    launched.expect(names, f"conv2_fwd_kernel<{'true' if silu else 'false'}, true, {kind}, ")
    for a, c in zip(got, want):
        assert torch.equal(a, c)
