"""Products with up to eight activation rows against the oracle: one, two and four waves per four weight rows, K and N that
leave remainders in the lane pieces and the row groups, every row count the kernel is compiled for (seven and eight rows, and three
and four of many weights, go to the kernel that splits K)."""
import numpy as np
import pytest
import torch

import oracle
from quamba_amd import ops
from quamba_amd import w4a8_utils as wu

pytestmark = pytest.mark.gpu
ROWS = [1, 2, 3, 4, 7, 8]


def _t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


@pytest.mark.parametrize("N,K", [(5, 16), (130, 1040), (4097, 1536), (4098, 2064), (11270, 1024)])
def test_int8_weights(dev, N, K):
    for M in ROWS:
        g = np.random.default_rng(M + N + K)
        a, w = g.integers(-128, 128, (M, K)).astype(np.int8), g.integers(-128, 128, (N, K)).astype(np.int8)
        sa, sb = np.float32([0.02]), (g.uniform(0.5, 1.5, N) * 0.6 / np.sqrt(K)).astype(np.float32)
        _, f16, i8 = oracle.gemm_w8a8(a, w, sa, sb)
        for want, dtype in ((i8, torch.int8), (f16.astype(np.float16), torch.float16)):
            got = torch.empty((M, N), dtype=dtype, device=dev)
            ops.scaled_mm_dq(got, _t(a, dev), _t(w, dev).t(), _t(sa, dev), _t(sb, dev))
            np.testing.assert_array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("N,K", [(64, 128), (1028, 2176), (5124, 2048), (11272, 1152)])
def test_4_bit_weights(dev, N, K):
    for M in ROWS:
        g = np.random.default_rng(M + N + K)
        a, codes = g.integers(-128, 128, (M, K)).astype(np.int8), g.integers(0, 16, (N, K)).astype(np.uint8)
        sg = g.uniform(2.0, 15.8, (K // 128, N)).astype(np.float16)
        sc, st = (g.uniform(0.5, 1.5, N) * 0.06 / np.sqrt(K) / 8).astype(np.float32), g.uniform(0.5, 1.5, M).astype(np.float32)
        want = oracle.gemm_w4a8(a, codes, sg, sc, st)[3]
        packed = wu.pack_w4a8(torch.from_numpy(codes.T.astype(np.int32))).to(dev)
        got = ops.w4a8o8_gemm(_t(a, dev), packed, _t(st, dev), _t(sc[None], dev), _t(sg, dev), None, M, N, K)
        np.testing.assert_array_equal(got.cpu().numpy(), want)
