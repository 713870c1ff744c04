"""qa_rmsnorm_gated_hadamard_quant on rows of 12 or 40 times 128 or 256 columns with one norm group: the bits of the two
kernels it replaces, one after the other."""
import ctypes

import numpy as np
import pytest
import torch

from quamba_amd import _lib, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [1536, 3072, 5120, 10240])
@pytest.mark.parametrize("rows,gated,norm_first", [(1, True, False), (130, True, False), (37, True, True), (300, False, False)])
def test_whole_row_norm_and_hadamard(dev, dim, rows, gated, norm_first):
    g = np.random.default_rng(dim + rows)
    x = torch.from_numpy((g.standard_normal((rows, dim)) * 2).astype(np.float16)).to(dev)
    w = torch.from_numpy(g.uniform(0.5, 1.5, dim).astype(np.float16)).to(dev)
    z = torch.from_numpy(g.integers(-128, 128, (rows, dim + 64)).astype(np.int8)).to(dev)
    y = ops.qlayer_normgated_fwd(x, w, None, 1e-5, z_scale=0.03 if gated else None, q_z=z[:, :dim] if gated else None, group_size=dim,
                                 norm_before_gate=norm_first, use_float16_output=True)[0]
    want = ops.hadamard_quant(y, 0.7)
    got = torch.empty((rows, dim), dtype=torch.int8, device=dev)
    n, h = _lib.QaNormGatedParams(), _lib.QaHadamardParams()
    n.rows, n.dim, n.group_size, n.norm_before_gate, n.eps, n.z_scale = rows, dim, dim, int(norm_first), 1e-5, 0.03
    n.x_row_stride, n.z_row_stride = dim, dim + 64
    n.x, n.weight, n.qz = x.data_ptr(), w.data_ptr(), z.data_ptr() if gated else None
    h.rows, h.dim, h.scale, h.out_row_stride, h.out = rows, dim, 0.7, dim, got.data_ptr()
    _lib.check(_lib.lib().qa_rmsnorm_gated_hadamard_quant(ctypes.byref(n), ctypes.byref(h), _lib.current_stream(dev)), "norm_hadamard")
    assert int(want.abs().max()) > 40
    assert torch.equal(got, want)
