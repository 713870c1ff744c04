"""Every tile the W8A8 and W4A8 products choose from, at sizes with remainders in rows, columns and K, against the oracle."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from quamba_amd import _lib, ops
from quamba_amd import w4a8_utils as wu

pytestmark = pytest.mark.gpu


def _t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


# K over the waves (the first three), 128 x 64, 128 x 128, 128 x 256 in one round and in three, 256 x 256
@pytest.mark.parametrize("M,N,K", [(130, 60, 272), (9, 2100, 2064), (300, 1000, 528), (900, 1200, 400), (1000, 2100, 384), (2100, 2100, 272),
                                   (4700, 4700, 144), (4000, 4000, 160), (4200, 4900, 128)])
@pytest.mark.parametrize("order", [0, 1])
def test_int8_weights(dev, M, N, K, order):
    g = np.random.default_rng(M + N + K)
    a, w = g.integers(-128, 128, (M, K)).astype(np.int8), g.integers(-128, 128, (N, K)).astype(np.int8)
    sa, sb = (g.uniform(0.5, 1.5, M) * 0.02).astype(np.float32), (g.uniform(0.5, 1.5, N) * 0.6 / np.sqrt(K)).astype(np.float32)
    acc = oracle.gemm_w8a8(a, w, sa, sb)[0].astype(np.float32)
    v = sb[None] * (sa[:, None] * acc) if order else sa[:, None] * (sb[None] * acc)
    want = np.clip(np.rint(v), -128, 127).astype(np.int8)
    got = torch.empty((M, N), dtype=torch.int8, device=dev)
    ta, tw, tsa, tsb = _t(a, dev), _t(w, dev), _t(sa, dev), _t(sb, dev)
    p = _lib.QaGemmW8A8Params()
    p.m, p.n, p.k, p.a_scale_numel, p.w_scale_numel, p.scale_order = M, N, K, M, N, order
    p.lda = p.ldw = K
    p.ldd = N
    p.a, p.w, p.a_scale, p.w_scale, p.d = (t.data_ptr() for t in (ta, tw, tsa, tsb, got))
    _lib.check(_lib.lib().qa_gemm_w8a8(ctypes.byref(p), _lib.current_stream(dev)), "gemm_w8a8")
    np.testing.assert_array_equal(got.cpu().numpy(), want)


# few outputs, rows and columns with remainders: K over the waves, of one unit, part of one and two, and with a ring of units that goes
# round
@pytest.mark.parametrize("M,N,K", [(9, 5, 16), (17, 33, 80), (16, 48, 6160), (100, 30, 12304), (256, 250, 144), (257, 250, 144)])
@pytest.mark.parametrize("order", [0, 1])
def test_int8_weights_of_few_outputs(dev, M, N, K, order):
    test_int8_weights(dev, M, N, K, order)


# workgroups that start at points of their own in K: few columns, a row block each (9 k tiles, the third turn of 7 passes their end);
# tiles of 256 x 256, an XCD each (20 and 25 k tiles; the 320-wide ones are in test_kernel_choice_gpu.py); beside them 128 x 256 tiles
# and K with part of a tile, which start at the beginning
@pytest.mark.parametrize("M,N,K", [(11000, 130, 1152), (11000, 192, 1024), (11000, 130, 1168), (4090, 4080, 3200), (4200, 10300, 2560), (4800, 5100, 3072),
                                   (5100, 4800, 3072), (4200, 4300, 3216)])
@pytest.mark.parametrize("order,dtype", [(0, torch.int8), (1, torch.int8), (0, torch.float16), (0, torch.bfloat16)])
def test_starting_points_in_k(dev, M, N, K, order, dtype):
    test_large_tiles_over_a_long_k(dev, M, N, K, order, dtype)


# K over the waves of a workgroup: as many 128-byte units of K as waves, one more, the ring of two units round several times, all
# with and without a remainder of K; then other tiles, at the K where the dispatch takes them (200 x 2510 is in 64 x 64 tiles without
# it, 61 x 18500 in 128 x 128; every one, and units for a part of the waves only, in test_kernel_choice_gpu.py)
@pytest.mark.parametrize("M,N,K", [(m, n, k) for m, n in [(9, 200), (20, 1000), (70, 1900)] for k in (16, 128, 1008, 1024, 1040, 2048, 2064, 3200, 4112)] +
                         [(16, 4201, 2192), (3, 12210, 2176), (64, 6001, 2192), (200, 2510, 2176), (61, 18500, 2064)])
@pytest.mark.parametrize("order,dtype", [(0, torch.int8), (1, torch.int8), (0, torch.float16), (0, torch.bfloat16)])
def test_k_split_over_the_waves(dev, M, N, K, order, dtype):
    test_large_tiles_over_a_long_k(dev, M, N, K, order, dtype)


# the same with 4-bit weights, groups of 128 and one scale per channel; an odd number of columns, group scales two bytes off a word
@pytest.mark.parametrize("M,N,K", [(9, 200, 128), (9, 201, 1024), (33, 500, 1152), (20, 1000, 4352), (16, 4201, 2176), (3, 12210, 2176), (70, 1900, 1280),
                                   (64, 6001, 2176), (30, 20001, 2176), (61, 10201, 2176), (64, 18500, 2048), (130, 60, 2176)])
@pytest.mark.parametrize("grouped", [True, False])
@pytest.mark.parametrize("dtype", [torch.int8, torch.float16])
def test_k_split_over_the_waves_with_4_bits(dev, M, N, K, grouped, dtype):
    """Codes times a group scale are exact in fp32, so rounding them there is the single rounding of the expansion."""
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a = torch.randint(-128, 128, (M, K), dtype=torch.int8, device=dev, generator=g)
    codes = torch.randint(0, 16, (N, K), dtype=torch.uint8, device=dev, generator=g)
    words = codes.view(N, K // 8, 2, 4)
    packed = (words[:, :, 0] | words[:, :, 1] << 4).reshape(N, K // 2).contiguous()
    scales = torch.empty(K // 128 * N + 1, dtype=torch.float16, device=dev)
    sg = scales[1:].view(K // 128, N)
    sg.copy_(torch.rand(sg.shape, device=dev, generator=g) * 13 + 2)
    if grouped:
        w8 = ((codes.float() - 8) * sg.t().float().repeat_interleave(128, 1)).round().double()
    else:
        w8 = (codes.to(torch.int8) << 4).double()
    sc, st = (torch.rand(N, device=dev, generator=g) + 0.5) * 0.006 / K ** 0.5, torch.rand(M, device=dev, generator=g) + 0.5
    v = st[:, None] * (sc * (a.double() @ w8.t()).float())
    want = v.round().clamp(-128, 127).to(torch.int8) if dtype == torch.int8 else v.half()
    got = torch.empty((M, N), dtype=dtype, device=dev)
    p = _lib.QaGemmW4A8Params()
    p.m, p.n, p.k, p.tok_scale_numel, p.group_size, p.lda, p.ldd = M, N, K, M, 128 if grouped else -1, K, N
    p.out_type = _lib.QA_OUT_I8 if dtype == torch.int8 else _lib.QA_OUT_F16
    p.a, p.w_packed, p.s_channel, p.s_token, p.d = (t.data_ptr() for t in (a, packed, sc, st, got))
    p.s_group = sg.data_ptr() if grouped else None
    _lib.check(_lib.lib().qa_gemm_w4a8(ctypes.byref(p), _lib.current_stream(dev)), "gemm_w4a8")
    assert torch.equal(got, want)


# K over the waves in 16 x 16 to 32 x 48, 64 x 128, 128 x 128, 192 x 128, expanded once
@pytest.mark.parametrize("M,N,K,workspace", [(70, 200, 2176, False), (100, 1000, 384, False), (130, 2050, 1664, False), (250, 2500, 1152, False),
                                             (600, 2100, 256, False), (300, 4200, 1664, False), (70, 9000, 128, False), (700, 3100, 1152, False),
                                             (900, 6100, 128, False), (950, 6100, 896, False), (4000, 3300, 1664, False), (4000, 3300, 1664, True)])
def test_4_bit_weights(dev, M, N, K, workspace):
    g = np.random.default_rng(M + N + K)
    a, codes = g.integers(-128, 128, (M, K)).astype(np.int8), g.integers(0, 16, (N, K)).astype(np.uint8)
    sg = g.uniform(2.0, 15.8, (K // 128, N)).astype(np.float16)
    sc, st = (g.uniform(0.5, 1.5, N) * 0.06 / np.sqrt(K) / 8).astype(np.float32), g.uniform(0.5, 1.5, M).astype(np.float32)
    want = oracle.gemm_w4a8(a, codes, sg, sc, st)[3]
    packed = wu.pack_w4a8(torch.from_numpy(codes.T.astype(np.int32))).to(dev)
    rows, ops.W4A8_EXPAND_ONCE_ROWS = ops.W4A8_EXPAND_ONCE_ROWS, 65 if workspace else 1 << 30
    try:
        got = ops.w4a8o8_gemm(_t(a, dev), packed, _t(st, dev), _t(sc[None], dev), _t(sg, dev), None, M, N, K)
    finally:
        ops.W4A8_EXPAND_ONCE_ROWS = rows
    np.testing.assert_array_equal(got.cpu().numpy(), want)


# 128 x 128 with four stages, 128 x 256 with three, 256 x 256, 256 x 320 and 320 x 256 with two: K of as many k tiles as there
# are stages and one more, and of so many that the ring of stages goes round several times, with and without a remainder
LARGE = [(1500, 2500), (1500, 5000), (4090, 4090), (4090, 5100), (5100, 4090)]


@pytest.mark.parametrize("M,N", LARGE)
@pytest.mark.parametrize("K", [384, 512, 640, 1712, 2560])
@pytest.mark.parametrize("order,dtype", [(0, torch.int8), (1, torch.int8), (0, torch.float16), (0, torch.bfloat16)])
def test_large_tiles_over_a_long_k(dev, M, N, K, order, dtype):
    """Sums of integers below 2^53 are exact in float64 whatever their order, the epilogue is two fp32 products and a rounding."""
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a, w = (torch.randint(-128, 128, s, dtype=torch.int8, device=dev, generator=g) for s in ((M, K), (N, K)))
    sa, sb = torch.rand(M, device=dev, generator=g) * 0.02 + 0.01, (torch.rand(N, device=dev, generator=g) + 0.5) * 0.6 / K ** 0.5
    acc = (a.double() @ w.double().t()).float()
    v = sb * (sa[:, None] * acc) if order else sa[:, None] * (sb * acc)
    want = v.round().clamp(-128, 127).to(torch.int8) if dtype == torch.int8 else v.to(dtype)
    got = torch.empty((M, N), dtype=dtype, device=dev)
    p = _lib.QaGemmW8A8Params()
    p.m, p.n, p.k, p.a_scale_numel, p.w_scale_numel, p.scale_order = M, N, K, M, N, order
    p.out_type = {torch.int8: _lib.QA_OUT_I8, torch.float16: _lib.QA_OUT_F16, torch.bfloat16: _lib.QA_OUT_BF16}[dtype]
    p.lda = p.ldw = K
    p.ldd = N
    p.a, p.w, p.a_scale, p.w_scale, p.d = (t.data_ptr() for t in (a, w, sa, sb, got))
    _lib.check(_lib.lib().qa_gemm_w8a8(ctypes.byref(p), _lib.current_stream(dev)), "gemm_w8a8")
    assert torch.equal(got, want)
    if dtype == torch.int8:
        assert int(want.max()) - int(want.min()) > 100


@pytest.mark.parametrize("M,N,K", [(9, 37, 1040), (64, 300, 640), (65, 300, 640), (1500, 2500, 1712)])
def test_the_single_row_rules_with_many_rows(dev, M, N, K):
    """16 x 16 with K over the waves and 128 x 128 with two stages: the host's scalar, and rounding half away from zero."""
    g = torch.Generator(device=dev).manual_seed(K)
    a, w = (torch.randint(-128, 128, s, dtype=torch.int8, device=dev, generator=g) for s in ((M, K), (N, K)))
    acc = (a.double() @ w.double().t()).float()
    got = torch.empty((M, N), dtype=torch.int8, device=dev)
    p = _lib.QaGemmW8A8Params()
    p.m, p.n, p.k, p.a_scale_numel, p.w_scale_numel = M, N, K, 1, N
    p.lda = p.ldw = K
    p.ldd = N
    alpha = torch.tensor(0.012 / K ** 0.5, device=dev)
    p.use_alpha, p.alpha = 1, float(alpha)
    p.a, p.w, p.d = a.data_ptr(), w.data_ptr(), got.data_ptr()
    _lib.check(_lib.lib().qa_gemm_w8a8(ctypes.byref(p), _lib.current_stream(dev)), "gemm_w8a8")
    assert torch.equal(got, (alpha * acc).round().clamp(-128, 127).to(torch.int8))
    sa, sb = torch.tensor([0.5], device=dev), (torch.rand(N, device=dev, generator=g) + 0.5) * 0.025 / K ** 0.5
    p.use_alpha, p.round_mode, p.a_scale, p.w_scale = 0, _lib.QA_ROUND_HALF_AWAY, sa.data_ptr(), sb.data_ptr()
    _lib.check(_lib.lib().qa_gemm_w8a8(ctypes.byref(p), _lib.current_stream(dev)), "gemm_w8a8")
    v = ((sb * sa) * acc).double()
    assert torch.equal(got, (v.sign() * (v.abs() + 0.5).floor()).clamp(-128, 127).to(torch.int8))
