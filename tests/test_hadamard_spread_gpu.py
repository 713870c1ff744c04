"""Rows of 12 or 40 times 128 columns at the numbers of rows where the launch changes the waves that it wants on a SIMD: the bits of the
general transform (a row that begins off 16 bytes takes it), and with the norm in front those of the two kernels apart."""
import ctypes

import pytest
import torch

from quamba_amd import _lib, ops
from tests import launched

pytestmark = pytest.mark.gpu


def _waves(rows, dim, fused):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    return 1 if fused and dim == 5120 and rows <= 2 * cus else 3 if 4 * cus < rows <= 6 * cus else 8


@pytest.mark.parametrize("dim,s", [(1536, 12), (5120, 40)])
@pytest.mark.parametrize("rows", [129, 512, 513, 1024, 1025, 1536, 1537, 2100])
@pytest.mark.parametrize("mode", ["plain", "gate first", "gate last", "no gate"])
def test_rows_per_compute_unit(dev, rows, dim, s, mode):
    g = torch.Generator(device=dev).manual_seed(rows + dim)
    x = (torch.randn(rows, dim, device=dev, generator=g) * 2).half()
    w = (torch.rand(dim, device=dev, generator=g) + 0.5).half()
    z = torch.randint(-128, 128, (rows, dim), dtype=torch.int8, device=dev, generator=g)
    gated, first, fuse = mode.startswith("gate"), mode != "gate last", ["plain", "gate first", "gate last", "no gate"].index(mode)
    y = x if mode == "plain" else ops.qlayer_normgated_fwd(x, w, None, 1e-5, z_scale=0.03 if gated else None, q_z=z if gated else None, group_size=dim,
                                                           norm_before_gate=not first, use_float16_output=True)[0]
    apart = torch.empty(rows, dim + 8, dtype=torch.half, device=dev)[:, 1:dim + 1]
    apart.copy_(y)
    n, h = _lib.QaNormGatedParams(), _lib.QaHadamardParams()
    want, got = torch.empty_like(z), torch.empty_like(z)
    h.rows, h.dim, h.scale, h.out_row_stride, h.x_row_stride, h.x, h.out = rows, dim, 0.7, dim, dim + 8, apart.data_ptr(), want.data_ptr()
    _lib.check(_lib.lib().qa_hadamard_quant(ctypes.byref(h), _lib.current_stream(dev)), "general")
    h.x_row_stride, h.x, h.out = dim, x.data_ptr(), got.data_ptr()
    n.rows, n.dim, n.group_size, n.norm_before_gate, n.eps, n.z_scale = rows, dim, dim, int(not first), 1e-5, 0.03
    n.x_row_stride, n.z_row_stride, n.x, n.weight, n.qz = dim, dim, x.data_ptr(), w.data_ptr(), z.data_ptr() if gated else None

    def call():
        if mode == "plain":
            _lib.check(_lib.lib().qa_hadamard_quant(ctypes.byref(h), _lib.current_stream(dev)), "hadamard")
        else:
            _lib.check(_lib.lib().qa_rmsnorm_gated_hadamard_quant(ctypes.byref(n), ctypes.byref(h), _lib.current_stream(dev)), "norm_hadamard")
    _, names = launched.kernels(call)
    launched.expect(names, f"hadamard_sm_kernel<{s}, 7, __half, {fuse}, {_waves(rows, dim, fuse != 0)}>")
    assert int(want.abs().max()) > 20
    assert torch.equal(got, want)
