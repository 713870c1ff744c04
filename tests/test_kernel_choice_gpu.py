"""Every kernel that the products and a layer's calls choose from by cost, at a size where the choice falls on it: the result
against an exact one, and the kernel that ran by its name, so that another choice does not leave one without a test."""
import ctypes

import pytest
import torch

from quamba_amd import W4A8QMamba, W4A8QMamba2, W8A8QMamba, W8A8QMamba2, _layer_call, _lib
from tests import launched
from tests import test_gemm_tiles_gpu as tiles
from tests import test_layer_call_gpu as layers
from tests import test_mixer_variants_gpu as variants

pytestmark = pytest.mark.gpu
OUT = {torch.int8: _lib.QA_OUT_I8, torch.float16: _lib.QA_OUT_F16, torch.bfloat16: _lib.QA_OUT_BF16}

# (M, N, K) -> what the kernel's name starts with, its output type, order of the scales and starting points in K left out.
# K of one and of some 128-byte units, units for a part of the waves only, with and without a remainder
SPLIT_INT8 = [((9, 5, 16), "16, 16, 2"), ((9, 3071, 96), "16, 16, 2"), ((300, 1000, 528), "32, 48, 1"), ((9, 2001, 400), "16, 16, 2"), ((70, 200, 528), "16, 16, 2"),
              ((16, 4201, 2192), "16, 32, 1"), ((5, 12210, 2176), "16, 48, 1"), ((40, 4001, 400), "32, 32, 1"), ((70, 1900, 1040), "32, 32, 1"), ((64, 6001, 2192), "32, 48, 1"), ((20, 20001, 2176), "32, 80, 1"),
              ((17, 18003, 2064), "32, 80, 1"), ((71, 9001, 5136), "64, 80, 1")]
TILES_INT8 = [((300, 3000, 16), "1, 1, 2, 2, 4", False), ((600, 1000, 528), "1, 1, 2, 2, 4", False), ((900, 1200, 400), "1, 1, 4, 2, 4", False),
              ((1500, 2500, 656), "2, 1, 2, 4, 4", False), ((61, 18500, 2064), "2, 1, 2, 4, 4", False), ((11000, 130, 1152), "2, 1, 2, 4, 4", True),
              ((1100, 5000, 528), "3, 1, 2, 4, 3", False), ((770, 6001, 16), "3, 1, 2, 4, 3", False), ((1500, 5000, 528), "2, 2, 2, 4, 3", False),
              ((4090, 5100, 528), "2, 5, 4, 2, 2", False), ((4090, 5100, 3200), "2, 5, 4, 2, 2", True), ((5100, 4090, 528), "5, 2, 2, 4, 2", False),
              ((5100, 4090, 3200), "5, 2, 2, 4, 2", True), ((4090, 4090, 528), "4, 2, 2, 4, 2", False), ((4090, 4080, 3200), "4, 2, 2, 4, 2", True)]
GEMV_INT8 = [((m, n, k), f"{m + (m == 3)}, {waves}") for m in (1, 2, 3, 4) for n, k, waves in ((201, 1040, 1), (4002, 1552, 4), (5003, 2064, 2), (201, 8336, 4))]


@pytest.mark.parametrize("size,shape", SPLIT_INT8)
@pytest.mark.parametrize("order,dtype", [(0, torch.int8), (1, torch.int8), (0, torch.float16), (0, torch.bfloat16)])
def test_int8_split_over_k(dev, size, shape, order, dtype):
    _, names = launched.kernels(lambda: _int8(dev, *size, order, dtype))
    launched.expect(names, f"gemm_split_kernel<8, {shape}, {OUT[dtype]}, 0>")


@pytest.mark.parametrize("size,shape,turn", TILES_INT8)
@pytest.mark.parametrize("order,dtype", [(order, dtype) for order in (0, 1) for dtype in OUT])
def test_int8_tiles(dev, size, shape, turn, order, dtype):
    _, names = launched.kernels(lambda: _int8(dev, *size, order, dtype))
    launched.expect(names, f"gemm_w8a8_kernel<{shape}, {OUT[dtype]}, false, {'true' if order else 'false'}, {'true' if turn else 'false'}>")


@pytest.mark.parametrize("size,shape", GEMV_INT8)
@pytest.mark.parametrize("order,dtype", [(1, torch.int8), (0, torch.int8), (0, torch.float16), (0, torch.bfloat16)])
def test_int8_dot_products(dev, size, shape, order, dtype):
    _, names = launched.kernels(lambda: _int8(dev, *size, order, dtype))
    launched.expect(names, f"gemv_kernel<8, {shape}, ")


def _int8(dev, M, N, K, order, dtype):
    """As test_large_tiles_over_a_long_k, for few outputs too."""
    if M * N > 100000:
        return tiles.test_large_tiles_over_a_long_k(dev, M, N, K, order, dtype)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a, w = (torch.randint(-128, 128, s, dtype=torch.int8, device=dev, generator=g) for s in ((M, K), (N, K)))
    sa, sb = torch.rand(M, device=dev, generator=g) * 0.02 + 0.01, (torch.rand(N, device=dev, generator=g) + 0.5) * 0.6 / K ** 0.5
    acc = (a.double() @ w.double().t()).float()
    v = sb * (sa[:, None] * acc) if order else sa[:, None] * (sb * acc)
    got = torch.empty((M, N), dtype=dtype, device=dev)
    p = _lib.QaGemmW8A8Params()
    p.m, p.n, p.k, p.a_scale_numel, p.w_scale_numel, p.scale_order, p.out_type = M, N, K, M, N, order, OUT[dtype]
    p.lda = p.ldw = K
    p.ldd = N
    p.a, p.w, p.a_scale, p.w_scale, p.d = (t.data_ptr() for t in (a, w, sa, sb, got))
    _lib.check(_lib.lib().qa_gemm_w8a8(ctypes.byref(p), _lib.current_stream(dev)), "gemm_w8a8")
    assert torch.equal(got, v.round().clamp(-128, 127).to(torch.int8) if dtype == torch.int8 else v.to(dtype))


def _four_bits(dev, M, N, K, grouped, dtype, transposed=False, workspace=False):
    """Codes times a group scale are exact in fp32, so rounding them there is the single rounding of the expansion; sums of integers
    below 2^53 are exact in float64."""
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a = torch.randint(-128, 128, (M, K), dtype=torch.int8, device=dev, generator=g)
    codes = torch.randint(0, 16, (N, K), dtype=torch.uint8, device=dev, generator=g)
    words = codes.view(N, K // 8, 2, 4)
    packed = (words[:, :, 0] | words[:, :, 1] << 4).reshape(N, K // 2).contiguous()
    sg = (torch.rand(K // 128, N, device=dev, generator=g) * 13 + 2).half()
    w8 = ((codes.float() - 8) * sg.t().float().repeat_interleave(128, 1)).round().double() if grouped else (codes.to(torch.int8) << 4).double()
    sc, st = (torch.rand(N, device=dev, generator=g) + 0.5) * 0.006 / K ** 0.5, torch.rand(M, device=dev, generator=g) + 0.5
    v = st[:, None] * (sc * (a.double() @ w8.t()).float())
    want = v.round().clamp(-128, 127).to(torch.int8) if dtype == torch.int8 else v.half()
    got = torch.empty((N, M) if transposed else (M, N), dtype=dtype, device=dev)
    p = _lib.QaGemmW4A8Params()
    p.m, p.n, p.k, p.tok_scale_numel, p.group_size, p.lda, p.ldd = M, N, K, M, 128 if grouped else -1, K, M if transposed else N
    p.out_type, p.output_transpose = OUT[dtype], int(transposed)
    p.a, p.w_packed, p.s_channel, p.s_token, p.d = (t.data_ptr() for t in (a, packed, sc, st, got))
    p.s_group = sg.data_ptr() if grouped else None
    space = torch.empty(N * K if workspace else 0, dtype=torch.int8, device=dev)
    if workspace:
        p.w8_workspace, p.w8_workspace_bytes = space.data_ptr(), space.numel()
    _lib.check(_lib.lib().qa_gemm_w4a8(ctypes.byref(p), _lib.current_stream(dev)), "gemm_w4a8")
    assert torch.equal(got, want.t() if transposed else want)


FOUR_BITS = [((9, 201, 128), "split_kernel<4, 16, 16, 2"), ((16, 4201, 1152), "split_kernel<4, 16, 32, 1"), ((5, 12210, 2176), "split_kernel<4, 16, 48, 1"),
             ((70, 1900, 1280), "split_kernel<4, 32, 32, 1"), ((64, 6001, 2176), "split_kernel<4, 32, 48, 1"), ((30, 20001, 2176), "split_kernel<4, 32, 80, 1"),
             ((61, 10201, 2176), "split_kernel<4, 64, 48, 1"), ((64, 18500, 2048), "split_kernel<4, 64, 80, 1"), ((200, 4001, 640), "w4a8_kernel<{}"),
             ((900, 1536, 768), "w4a8_reg_kernel<2, 4, 256, {}"), ((900, 2561, 768), "w4a8_reg_kernel<4, 4, 128, {}"),
             ((777, 6144, 1536), "w4a8_reg_kernel<6, 4, 128, {}"),
             # some rounds of split tiles, and far more rows than columns: tiles that stream K, or fewer rows a split tile
             ((200, 3071, 768), "w4a8_kernel<{}"), ((1531, 768, 1536), "w4a8_reg_kernel<2, 4, 256, {}"), ((6000, 128, 3072), "w4a8_kernel<{}"),
             ((4096, 160, 4096), "split_kernel<4, 32, 80, 1")]


@pytest.mark.parametrize("size,shape", FOUR_BITS)
@pytest.mark.parametrize("grouped", [True, False])
@pytest.mark.parametrize("dtype", [torch.int8, torch.float16])
def test_four_bits(dev, size, shape, grouped, dtype):
    _, names = launched.kernels(lambda: _four_bits(dev, *size, grouped, dtype))
    launched.expect(names, f"gemm_{shape.format('true' if grouped else 'false')}, {OUT[dtype]}")


@pytest.mark.parametrize("dtype", [torch.int8, torch.float16])
def test_four_bits_expanded_once(dev, dtype):
    _, names = launched.kernels(lambda: _four_bits(dev, 4000, 3300, 1664, True, dtype, workspace=True))
    launched.expect(names, "w4_expand_kernel", "gemm_w8a8_kernel<")


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K,waves", [(204, 1152, 1), (4004, 1664, 4), (4100, 2176, 2), (204, 8320, 4)])
@pytest.mark.parametrize("dtype", [torch.int8, torch.float16])
def test_four_bits_dot_products(dev, M, N, K, waves, dtype):
    _, names = launched.kernels(lambda: _four_bits(dev, M, N, K, True, dtype))
    launched.expect(names, f"gemv_kernel<4, {M + (M == 3)}, {waves}, ")


@pytest.mark.parametrize("M,shape", [(5, "1, 1, "), (40, "1, 4, ")])
@pytest.mark.parametrize("N,K,waves", [(330, 1152, 4), (330, 2176, 8)])
@pytest.mark.parametrize("dtype", [torch.int8, torch.float16])
def test_four_bits_transposed(dev, M, shape, N, K, waves, dtype):
    _, names = launched.kernels(lambda: _four_bits(dev, M, N, K, True, dtype, transposed=True))
    launched.expect(names, f"gemm_w4a8_skinny_kernel<{shape}{waves}, ")


def _layer(cls, dev, d_model, seed):
    second = cls in (W8A8QMamba2, W4A8QMamba2)
    m, g = (variants._mamba2 if second else variants._mamba1)(lambda d, *a, **k: cls(d_model, *a, **k), dev, seed=seed)
    if second:
        heads = m.nheads // 2
        m.conv1d.x_head_group_range = m.qchunk_scan.x_head_group_range = torch.tensor([[1, heads], [3, heads]], dtype=torch.int32, device=dev)
    return m, g


# in_proj of a decode step with the conv behind it in one launch: every tile, the conv's state by channel (its last argument 1) and by
# step (2), rows and columns with remainders
STEPS = [(W8A8QMamba, 256, 7, "8, 16, 16, 2, 0, 1"), (W8A8QMamba, 512, 61, "8, 16, 32, 1, 0, 1"), (W8A8QMamba, 2560, 5, "8, 16, 48, 1, 0, 1"),
         (W8A8QMamba, 512, 67, "8, 32, 32, 1, 0, 1"), (W8A8QMamba, 1536, 20, "8, 32, 32, 1, 0, 1"), (W8A8QMamba, 768, 83, "8, 32, 48, 1, 0, 1"),
         (W8A8QMamba, 1536, 67, "8, 32, 80, 1, 0, 1"),
         (W4A8QMamba, 256, 7, "4, 16, 16, 2, 0, 1"), (W4A8QMamba, 256, 66, "4, 16, 32, 1, 0, 1"), (W4A8QMamba, 2560, 5, "4, 16, 48, 1, 0, 1"),
         (W4A8QMamba, 512, 67, "4, 32, 32, 1, 0, 1"), (W4A8QMamba, 768, 83, "4, 32, 48, 1, 0, 1"), (W4A8QMamba, 1536, 67, "4, 64, 48, 1, 0, 1"),
         (W4A8QMamba, 2560, 99, "4, 64, 80, 1, 0, 1"), (W4A8QMamba, 2048, 65, "4, 32, 32, 1, 0, 1"),
         (W8A8QMamba2, 256, 7, "8, 16, 16, 2, 0, 2"), (W8A8QMamba2, 512, 47, "8, 16, 32, 1, 0, 2"), (W8A8QMamba2, 2048, 5, "8, 16, 48, 1, 0, 2"),
         (W8A8QMamba2, 256, 99, "8, 32, 32, 1, 0, 2"), (W8A8QMamba2, 768, 67, "8, 32, 48, 1, 0, 2"), (W8A8QMamba2, 1536, 66, "8, 32, 80, 1, 0, 2"),
         (W8A8QMamba2, 2048, 97, "8, 64, 80, 1, 0, 2"),
         (W4A8QMamba2, 256, 7, "4, 16, 16, 2, 0, 2"), (W4A8QMamba2, 256, 51, "4, 16, 32, 1, 0, 2"), (W4A8QMamba2, 2048, 5, "4, 16, 48, 1, 0, 2"),
         (W4A8QMamba2, 256, 98, "4, 32, 32, 1, 0, 2"), (W4A8QMamba2, 512, 115, "4, 32, 48, 1, 0, 2"), (W4A8QMamba2, 4096, 25, "4, 32, 80, 1, 0, 2"),
         (W4A8QMamba2, 2048, 35, "4, 64, 48, 1, 0, 2"), (W4A8QMamba2, 4096, 33, "4, 64, 80, 1, 0, 2")]


@pytest.mark.parametrize("cls,d_model,batch,shape", STEPS)
def test_in_proj_with_the_conv_behind_it(dev, cls, d_model, batch, shape):
    _step(dev, cls, d_model, batch, torch.int8 if batch % 2 else torch.float32, f"gemm_split_kernel<{shape}>")


# a product in three rounds of workgroups would wait for the conv in each of them: a launch of its own
@pytest.mark.parametrize("cls,d_model,batch", [(W8A8QMamba, 2048, 65), (W8A8QMamba2, 2560, 33), (W4A8QMamba2, 4096, 65)])
def test_the_conv_of_many_rows(dev, cls, d_model, batch):
    _step(dev, cls, d_model, batch, torch.int8, "conv2_update4_kernel")


# few rows: dot products with the conv behind them, a wave and two for four weight rows; the recurrence of one, two and more
# sequences with states of both types; for one row the transform inside out_proj's launch, 12, 1 and 40 column blocks
@pytest.mark.parametrize("cls,d_model,batch,dtype,names", [
    (W8A8QMamba, 768, 2, torch.int8, ["gemv_kernel<8, 2, 1, 3, 0, true>", "mamba1_step_kernel<2, false>"]),
    (W8A8QMamba, 2048, 2, torch.float32, ["gemv_kernel<8, 2, 2, 2, 0, true>", "mamba1_step_kernel<2, true>"]),
    (W8A8QMamba, 2048, 3, torch.int8, ["gemv_kernel<8, 4, 2, 2, 0, true>", "mamba1_step_kernel<4, false>"]),
    (W4A8QMamba, 768, 1, torch.float32, ["gemv_kernel<4, 1, 1, 2, 0, true>", "mamba1_step_kernel<1, true>", "gemv_rotated_kernel<4, 12>"]),
    (W4A8QMamba, 2048, 1, torch.int8, ["gemv_kernel<4, 1, 2, 1, 0, true>", "mamba1_step_kernel<1, false>", "gemv_rotated_kernel<4, 1>"]),
    (W4A8QMamba, 2048, 2, torch.int8, ["gemv_kernel<4, 2, 2, 1, 0, true>"]),
    (W4A8QMamba, 2560, 1, torch.int8, ["gemv_rotated_kernel<4, 40>"]),
    (W8A8QMamba, 1536, 1, torch.int8, ["gemv_rotated_kernel<8, 12>"]),
    # the conv's output scales from tables; a state by step
    (W8A8QMamba2, 768, 1, torch.int8, ["gemv_conv_tables_kernel<8, 1, 1, 4>"]), (W8A8QMamba2, 2048, 2, torch.float32, ["gemv_conv_tables_kernel<8, 2, 2, 2>"]),
    (W8A8QMamba2, 256, 3, torch.int8, ["gemv_conv_tables_kernel<8, 4, 1, 3>"]), (W4A8QMamba2, 4096, 1, torch.int8, ["gemv_conv_tables_kernel<4, 1, 1, 2>"]),
    (W4A8QMamba2, 2048, 2, torch.float32, ["gemv_conv_tables_kernel<4, 2, 2, 1>"]), (W4A8QMamba2, 768, 4, torch.int8, ["gemv_conv_tables_kernel<4, 4, 1, 2>"])])
def test_step_of_few_rows(dev, cls, d_model, batch, dtype, names):
    _step(dev, cls, d_model, batch, dtype, *names)


# 4-bit weights with one scale per channel and no groups: products by tiles of their own, the conv behind them
@pytest.mark.parametrize("cls,d_model,batch,shape", [(W4A8QMamba, 512, 3, "4, 16, 16, 2, 0, 1"), (W4A8QMamba, 512, 7, "4, 16, 16, 2, 0, 1"), (W4A8QMamba, 1536, 67, "4, 64, 48, 1, 0, 1"),
                                                     (W4A8QMamba2, 256, 50, "4, 16, 32, 1, 0, 2"), (W4A8QMamba2, 512, 115, "4, 32, 48, 1, 0, 2")])
def test_in_proj_without_group_scales(dev, cls, d_model, batch, shape):
    _step(dev, cls, d_model, batch, torch.float32, f"gemm_split_kernel<{shape}>", per_channel=True)


# a conv state whose codes of a channel are one word, in buffers that are not the package's own: channels eight bytes apart behind a
# base of four, the second family's by channel
@pytest.mark.parametrize("apart", [4, 8])
@pytest.mark.parametrize("cls,d_model,batch,name", [
    (W8A8QMamba, 768, 1, "gemv_kernel<8, 1, 1, 4, 0, true>"), (W8A8QMamba, 2048, 2, "gemv_kernel<8, 2, 2, 2, 0, true>"), (W4A8QMamba, 768, 2, "gemv_kernel<4, 2, 1, 2, 0, true>"),
    (W8A8QMamba2, 768, 1, "gemv_conv_words_kernel<8, 1, 1, 4>"), (W8A8QMamba2, 256, 3, "gemv_conv_words_kernel<8, 4, 1, 3>"),
    (W4A8QMamba2, 2048, 2, "gemv_conv_words_kernel<4, 2, 2, 1>"), (W4A8QMamba2, 4096, 1, "gemv_conv_words_kernel<4, 1, 1, 2>")])
def test_step_with_a_state_of_words(dev, cls, d_model, batch, name, apart):
    def view(conv):
        buf = torch.zeros(4 + batch * conv.shape[1] * apart, dtype=torch.int8, device=dev)
        v = buf[4:].view(batch, conv.shape[1], apart)[..., :4]
        return v.copy_(conv)
    _step(dev, cls, d_model, batch, torch.int8, name, conv_view=view)


def _step(dev, cls, d_model, batch, dtype, *names, per_channel=False, conv_view=lambda conv: conv):
    m, g = _layer(cls, dev, d_model, batch)
    if per_channel:
        m.in_proj.s_group = torch.empty((0, m.in_proj.size_n), dtype=torch.float16, device=dev)
        variants._fill_linear(m.in_proj, dev, g, 40.0)
    h = variants._ri(dev, g, batch, 1, d_model)
    conv, ssm = layers._states(m, dev, g, batch, dtype, 4)
    conv2, ssm2 = conv.clone(), ssm.clone()
    conv = conv_view(conv)
    out, ran = launched.kernels(lambda: _layer_call.call(m, h, conv, ssm, True))
    assert out is not None
    layers._close(out[:, 0], m._step_modules(h, conv2, ssm2), (conv, conv2), (ssm, ssm2))
    launched.expect(ran, *names)


# the scan of a prompt with dt_proj inside it, ranks of 16, 48, 64, 80, 96 and 160: four lanes a channel, both kinds of workgroup,
# segments, eight lanes, the time over the waves of a workgroup
@pytest.mark.parametrize("d_model,batch,seqlen,names", [
    (1024, 16, 33, ["scan_tm_kernel<4, true, true, 1>"]), (1280, 16, 35, ["scan_tm_mixed_kernel<true, 2>"]), (2560, 8, 37, ["scan_tm_mixed_kernel<true, 3>"]),
    (256, 1, 1500, ["scan_tm_kernel<8, false, false, 1>", "scan_tm_kernel<8, true, true, 1>"]), (2560, 3, 515, ["scan_tm_kernel<8, true, true, 3>"]),
    (1536, 1, 37, ["scan_waves_kernel<4, 12, true, 2>"]), (2560, 1, 700, ["scan_waves_kernel<8, 12, true, 3>"]), (768, 1, 515, ["scan_waves_kernel<8, 12, true, 1>"]),
    (768, 1, 500, ["scan_waves_kernel<8, 16, true, 1>"]), (768, 1, 1024, ["scan_waves_kernel<8, 16, true, 1>"]), (2560, 1, 48, ["scan_waves_kernel<4, 12, true, 3>"]),
    (2560, 1, 300, ["scan_waves_kernel<4, 12, true, 3>"]), (1536, 2, 67, ["scan_waves_kernel<8, 12, true, 2>"]), (1536, 2, 400, ["scan_waves_kernel<8, 12, true, 2>"]),
    (3072, 1, 515, ["scan_waves_kernel<8, 12, true, 3>"]), (256, 2, 1300, ["scan_tm_kernel<8, false, false, 1>", "scan_tm_kernel<8, true, true, 1>"])])
def test_scan_of_a_layer(dev, d_model, batch, seqlen, names):
    m, g = _layer(W8A8QMamba, dev, d_model, seqlen)
    h = variants._ri(dev, g, batch, seqlen, d_model)
    conv, ssm = layers._states(m, dev, g, batch, torch.float32, 4)
    conv2, ssm2 = conv.clone(), ssm.clone()
    out, ran = launched.kernels(lambda: _layer_call.call(m, h, conv, ssm, False))
    layers._close(out, m._forward_modules(h, conv2, ssm2), (conv, conv2), (ssm, ssm2))
    launched.expect(ran, *names)
