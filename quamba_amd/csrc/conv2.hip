// Mamba2 xBC conv: depthwise causal conv1d (+SiLU) over the concatenated [x | B | C] channels of
// in_proj's output, requantised into three int8 tensors with per-part input/weight/bias scales and
// grouped output scales.
//
// Arithmetic (reference csrc/causal_conv1d/quamba2_conv1d_fwd_kernel.cuh:215-246, update kernel
// quamba2_conv1d_update_kernel.cuh:134-143):
//   forward   v = fma(s_w*s_in, sum_w W[c,w]*x[t-(k-1-w)], s_b*bias[c])
//   update    v = s_b*bias[c];  v = fma((s_w*s_in)*W[c,w], x[..], v) per tap, after shifting the state
//   then v = v / (1 + exp(-v)) if silu, q = sat8(round_half_away(v / s_out[c]))
// s_out[c] for an x channel is found through the cumulative head-group / dim-group end indices of
// its ssd group (fwd kernel :151-189), for B and C channels it is the ssd group's scale (:190-212).
//
// Layout and mapping: activations are channel-contiguous (batch, seqlen, dim).  A lane owns four
// neighbouring channels and walks a run of time steps: one dword load per step (a wave reads 256
// contiguous bytes), the last four inputs of each channel are kept as a packed byte window updated
// with one byte permute, the taps are one packed int8 dot product per output (exact), the epilogue
// is the cheap-with-exact-fallback route shared with the Mamba1 conv, one dword store per step.
#include "conv2_common.hpp"
#include "mixer_common.hpp"

#include <type_traits>

namespace qa {
namespace {

constexpr int kThreads = 256;

// What a lane takes of the channels' operands is requested in one straight run behind the inputs: where ways with and without
// loads meet the compiler waits for every load in flight, the inputs among them, and the look-up of an output scale - the
// head's group, the channel's group in it, their scale - was three trips to memory one after the other.  Now a wave requests the whole
// table and looks it up across its lanes.  Bound by vector issue (some 55 instructions for four outputs, of which the exponential and the
// reciprocal are a third) and, in short runs, by that set-up.  In a layer, kernel times in turn on one card, us before and after: one
// scale 1 x 512 x 1536 channels 5.2 -> 4.6, 1 x 777 x 3072 5.9 -> 4.9, 3 x 1021 x 5120 15.4 -> 13.2, 8 x 2048 x 5120 55.6 -> 50.5; tables 1 x 500 x 5376
// 7.3 -> 6.3, 3 x 1000 x 2304 12.0 -> 9.7, 1 x 1531 x 5376 11.8 -> 11.0, 4 x 4096 x 5376 60.7 -> 57.7, 16 x 1024 x 10240 105 -> 98.  Of this the sums as
// floats (dot4_float) are 52.7 -> 50.5 at 8 x 2048 x 5120, 103 -> 98 at 16 x 1024 x 10240, 6.5 -> 6.3 at 1 x 500 x 5376 and nothing at 3 x 1021; runs of 6, 12,
// 24 and 48 steps 9.9 -> 9.7 at 3 x 1000 x 2304, 6.4 -> 6.3 at 1 x 500 x 5376, 20.1 -> 19.7 at 1 x 12000 x 1792, elsewhere nothing; the rest is the
// straight run.  (One copy of the exact route in a loop over a lane's outputs instead of four, a third of the code: 48.4 -> 53.6 at 8 x 2048
// x 5120 on another card.)
enum ScaleKind { kOneScale, kTables, kWalk };

// grid: x = blocks of 256 channels, y = blocks of 4 runs of `run` steps (one run per wave), z = batch
// PACKED: four taps a channel, back to back: the lane's taps are one 16-byte piece, its biases one word.  SCALES kOneScale: one
// output scale for all (the Mamba1 conv); kTables: up to 8 x 8 of an ssd group, whose channels are whole waves; kWalk: anything.
// BATCH: loads in flight per lane.
template <bool SILU, bool PACKED, ScaleKind SCALES, int BATCH>
__global__ __launch_bounds__(kThreads) void conv2_fwd_kernel(QaConv2Params p, int run) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));   // the same in every lane: the step
                                                                                          // counters below stay in scalar registers
    const int wave_ch = blockIdx.x * 256, ch0 = wave_ch + lane * 4;
    const int b = blockIdx.z;
    const int t0 = (blockIdx.y * 4 + wave) * run;
    if (t0 >= p.seqlen || (SCALES != kTables && ch0 >= p.dim)) return;
    const int t_end = min(t0 + run, p.seqlen);
    // (the tables are looked up by the whole wave: lanes past the last channel take that one's operands and store nothing)
    const int ch = SCALES == kTables ? min(ch0, p.dim - 4) : ch0;

    // uniform row addresses and one offset per lane: the address arithmetic stays in scalar registers
    const int8_t* const src = p.xBC + b * p.xBC_batch_stride;
    const uint32_t at_ch = static_cast<uint32_t>(ch);
    auto input = [&](int t) {
        int64_t row = t * p.xBC_l_stride;
        asm("" : "+s"(row));                                  // (the compiler would add the lane's offset first, and multiply in vector registers)
        return *reinterpret_cast<const uint32_t*>(src + row + at_ch);
    };
    uint32_t hist[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) hist[i] = input(max(t0 - 3 + i, 0));
    // the loads of the next batch of steps are in flight while the current batch is worked on
    uint32_t d[BATCH], dn[BATCH];
    auto fetch = [&](int tb, uint32_t (&dst)[BATCH]) {
#pragma unroll
        for (int i = 0; i < BATCH; ++i) dst[i] = input(min(tb + i, p.seqlen - 1));      // in range for every lane; steps past the end are never used
    };
    fetch(t0, dn);

    const Part part = part_of(p, ch);          // the four channels of a lane never straddle two parts
    uint32_t taps[4], bias4 = 0u;
    if constexpr (PACKED) {
        const uint4 w = *reinterpret_cast<const uint4*>(p.weight + ch * 4);
        bias4 = *reinterpret_cast<const uint32_t*>(p.bias ? p.bias + ch : p.weight);
        taps[0] = w.x; taps[1] = w.y; taps[2] = w.z; taps[3] = w.w;
    }
    float s_out[4], inv_s_out[4], table = 0.0f, own = 0.0f;
    int head_end = 0, dim_end = 0;
    if constexpr (SCALES == kTables) {
        // lane 8 h + d: head group h, group d of its channels; the table is that of the wave's first channel
        const int g = p.n_groups > 1 && wave_ch < p.x_dim ? wave_ch / (p.x_dim / p.n_groups) : 0;
        const int entry = (g * p.nhead_groups + min(lane >> 3, p.nhead_groups - 1)) * p.ndim_groups + min(lane & 7, p.ndim_groups - 1);
        table = p.x_out_scales[entry];
        dim_end = p.x_dim_group_range[entry];
        head_end = p.x_head_group_range[g * p.nhead_groups + min(lane & 7, p.nhead_groups - 1)];
        const float* const group = part.index == 0 ? p.x_out_scales : part.index == 1 ? p.B_out_scales : p.C_out_scales;
        own = group[part.index == 0 || p.n_groups == 1 ? 0 : (ch - part.offset) / p.d_state];
    }
    if constexpr (SCALES != kWalk) __builtin_amdgcn_sched_barrier(0);
    float bias_f[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if constexpr (PACKED) {
            bias_f[e] = p.bias ? part.s_bias * static_cast<float>(static_cast<int8_t>(bias4 >> (8 * e))) : 0.0f;
        } else {
            taps[e] = pack_taps(p.weight + (ch + e) * p.weight_c_stride, p.weight_width_stride, p.width);
            bias_f[e] = p.bias ? part.s_bias * static_cast<float>(p.bias[ch + e]) : 0.0f;
        }
    }
    if constexpr (SCALES == kOneScale) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s_out[e] = p.x_out_scale;
    } else if constexpr (SCALES == kTables) {
        // (a wave begins a head or lies in one: 256 channels are whole heads of 4 .. 256, a power of two)
        const int shift = __builtin_ctz(p.x_headdim), in_group = p.n_groups > 1 ? wave_ch % (p.x_dim / p.n_groups) : wave_ch;
        const int head = (in_group + lane * 4) >> shift, first = (lane * 4) & (p.x_headdim - 1);
        int hg = 0, dg[4] = {};
#pragma unroll
        for (int j = 0; j < 7; ++j) hg += static_cast<int>(j < p.nhead_groups - 1) & static_cast<int>(head >= __builtin_amdgcn_readlane(head_end, j));
#pragma unroll
        for (int j = 0; j < 7; ++j) {
            const int end = __builtin_amdgcn_ds_bpermute(4 * (8 * hg + j), dim_end);
#pragma unroll
            for (int e = 0; e < 4; ++e) dg[e] += static_cast<int>(j < p.ndim_groups - 1) & static_cast<int>(first + e >= end);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float s = __int_as_float(__builtin_amdgcn_ds_bpermute(4 * (8 * hg + dg[e]), __float_as_int(table)));
            s_out[e] = part.index == 0 ? s : own;
        }
        if (ch0 >= p.dim) return;
    } else {
        out_scales4_of(p, part, ch, s_out);
    }
    bool exact_only[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        inv_s_out[e] = 1.0f / s_out[e];
        exact_only[e] = conv_needs_exact_route(s_out[e]);
    }
    const ConvQuantRegs kq(__builtin_fminf(__builtin_fminf(s_out[0], s_out[1]), __builtin_fminf(s_out[2], s_out[3])));
    int64_t out_ls, out_cs;
    int8_t* out = out_ptr(p, part, b, ch0, &out_ls, &out_cs);

    const int dot_magic = dot4_magic();
    // byte j of win[e] holds x[t-3+j] of channel ch0+e
    uint32_t win[4] = {0u, 0u, 0u, 0u};
    auto push = [&](uint32_t d) {
        win[0] = __builtin_amdgcn_perm(d, win[0], 0x04030201u);
        win[1] = __builtin_amdgcn_perm(d, win[1], 0x05030201u);
        win[2] = __builtin_amdgcn_perm(d, win[2], 0x06030201u);
        win[3] = __builtin_amdgcn_perm(d, win[3], 0x07030201u);
    };
#pragma unroll
    for (int i = 0; i < 3; ++i) push(t0 - 3 + i >= 0 ? hist[i] : 0u);
    int8_t* out_at = out + t0 * out_ls;             // walks on by one step's stride (the stride differs from lane to lane: a
                                                    // product per step would be a 64-bit multiplication in vector registers)
    for (int tb = t0; tb < t_end; tb += BATCH) {
#pragma unroll
        for (int i = 0; i < BATCH; ++i) d[i] = dn[i];
        if (tb + BATCH < t_end) fetch(tb + BATCH, dn);
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            if (tb + i >= t_end) break;
            push(d[i]);
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(part.s_in, dot4_float(win[e], taps[e], dot_magic), bias_f[e]);
            *reinterpret_cast<uint32_t*>(out_at) = conv_quant4(v, s_out, inv_s_out, SILU, exact_only, kq);
            out_at += out_ls;
        }
    }
    // the wave that reaches the end leaves the last inputs of its channels (still in the caches) in the conv state
    if (p.conv_state && t_end == p.seqlen) {
        int8_t* st = p.conv_state + b * p.conv_state_batch_stride + ch0 * p.conv_state_c_stride;
        const bool words = p.conv_state_c_stride == 1 && (reinterpret_cast<uintptr_t>(st) & 3u) == 0 && p.conv_state_l_stride % 4 == 0;
        for (int i = 0; i < p.conv_state_len; ++i) {
            const int t = p.seqlen - p.conv_state_len + i;
            const uint32_t v = t >= 0 ? input(t) : 0u;
            if (words) {
                *reinterpret_cast<uint32_t*>(st + i * p.conv_state_l_stride) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) st[e * p.conv_state_c_stride + i * p.conv_state_l_stride] = static_cast<int8_t>(v >> (8 * e));
            }
        }
    }
}

// Any alignment: one thread per output element, same arithmetic.
__global__ __launch_bounds__(kThreads) void conv2_fwd_generic_kernel(QaConv2Params p) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    const int64_t total = static_cast<int64_t>(p.batch) * p.dim * p.seqlen;
    if (idx >= total) return;
    const int ch = static_cast<int>(idx % p.dim);
    const int t = static_cast<int>((idx / p.dim) % p.seqlen);
    const int b = static_cast<int>(idx / (static_cast<int64_t>(p.seqlen) * p.dim));
    const Part part = part_of(p, ch);
    const int8_t* src = p.xBC + b * p.xBC_batch_stride + ch * p.xBC_c_stride;
    const int8_t* w = p.weight + ch * p.weight_c_stride;
    float acc = 0.0f;
    for (int k = 0; k < p.width; ++k) {
        const int ti = t - (p.width - 1 - k);
        const float xv = ti >= 0 ? static_cast<float>(src[ti * p.xBC_l_stride]) : 0.0f;
        acc += static_cast<float>(w[k * p.weight_width_stride]) * xv;      // exact integers
    }
    const float bias_f = p.bias ? part.s_bias * static_cast<float>(p.bias[ch]) : 0.0f;
    const float v = __builtin_fmaf(part.s_in, acc, bias_f);
    int64_t out_ls, out_cs;
    int8_t* out = out_ptr(p, part, b, ch, &out_ls, &out_cs);
    out[t * out_ls] = conv_epilogue(v, out_scale_of(p, part, ch), p.silu_activation);
}

__global__ __launch_bounds__(kThreads) void conv2_update_kernel(QaConv2Params p) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (idx >= static_cast<int64_t>(p.batch) * p.dim) return;
    const int ch = static_cast<int>(idx % p.dim);
    const int b = static_cast<int>(idx / p.dim);
    int8_t* st = p.conv_state + b * p.conv_state_batch_stride + ch * p.conv_state_c_stride;
    const int8_t* w = p.weight + ch * p.weight_c_stride;
    const int width = p.width;
    const int slen = p.conv_state_len;            // width (slot 0 is dropped) or width-1
    const int drop = slen - (width - 1);
    // four taps and a state of four codes, each in one aligned word (the Mamba2 layer's own buffers): one load and one
    // store per row instead of one per code
    const bool w_word = width == 4 && p.weight_width_stride == 1 && aligned4(w);
    const bool s_word = slen == 4 && p.conv_state_l_stride == 1 && aligned4(st);
    __attribute__((aligned(4))) int8_t xs[4], ws[4] = {0, 0, 0, 0};
    const int8_t x_new = p.xBC[b * p.xBC_batch_stride + ch * p.xBC_c_stride];
    if (w_word) {
        *reinterpret_cast<uint32_t*>(ws) = *reinterpret_cast<const uint32_t*>(w);
    } else {
        for (int i = 0; i < width; ++i) ws[i] = w[i * p.weight_width_stride];
    }
    if (s_word) {
        const uint32_t win = (*reinterpret_cast<const uint32_t*>(st) >> 8) | (static_cast<uint32_t>(static_cast<uint8_t>(x_new)) << 24);
        *reinterpret_cast<uint32_t*>(st) = win;                    // the whole window is the new state
        *reinterpret_cast<uint32_t*>(xs) = win;
    } else {
        for (int i = 0; i < width - 1; ++i) xs[i] = st[(i + drop) * p.conv_state_l_stride];
        xs[width - 1] = x_new;
        for (int i = 0; i < slen; ++i) st[i * p.conv_state_l_stride] = xs[i + (width - slen)];
    }
    const Part part = part_of(p, ch);
    float v = p.bias ? part.s_bias * static_cast<float>(p.bias[ch]) : 0.0f;
    for (int i = 0; i < width; ++i) v = __builtin_fmaf(part.s_in * static_cast<float>(ws[i]), static_cast<float>(xs[i]), v);
    int64_t out_ls, out_cs;
    int8_t* out = out_ptr(p, part, b, ch, &out_ls, &out_cs);
    out[0] = conv_epilogue(v, out_scale_of(p, part, ch), p.silu_activation);
}

// The single-step update of four neighbouring channels per lane, as conv_step4 makes it behind a product.  The parts of it in
// their own order, the state's stores ahead of the scales' look-up: put together from conv_quad and conv_step4 the kernel took 3.89 us
// for 3.84 (mean of 60 sizes, 1 .. 200 sequences of 512 .. 10240 channels; up to 0.2 with the state in rows).
// grid: x quads of channels, y batch.
template <bool CHANNEL_ROWS>
__global__ __launch_bounds__(kThreads) void conv2_update4_kernel(QaConv2Params p) {
    const int ch0 = (blockIdx.x * kThreads + threadIdx.x) * 4, b = blockIdx.y;
    if (ch0 >= p.dim) return;
    int8_t* st = p.conv_state + b * p.conv_state_batch_stride + ch0 * p.conv_state_c_stride;
    const uint32_t x_new = *reinterpret_cast<const uint32_t*>(p.xBC + b * p.xBC_batch_stride + ch0);
    const uint4 w = *reinterpret_cast<const uint4*>(p.weight + ch0 * 4);
    const uint32_t taps[4] = {w.x, w.y, w.z, w.w};
    const uint32_t b4 = p.bias ? *reinterpret_cast<const uint32_t*>(p.bias + ch0) : 0u;
    uint32_t win[4];                                              // byte j of win[e]: input t - 3 + j of channel ch0 + e
    if constexpr (CHANNEL_ROWS) {
        const int drop = p.conv_state_len - 3;
        uint32_t d[4];
#pragma unroll
        for (int i = 0; i < 3; ++i) d[i] = *reinterpret_cast<const uint32_t*>(st + (drop + i) * p.conv_state_l_stride);
        d[3] = x_new;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i >= 4 - p.conv_state_len) *reinterpret_cast<uint32_t*>(st + (i - (4 - p.conv_state_len)) * p.conv_state_l_stride) = d[i];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t pick = 0x0c0c0000u | ((4u + e) << 8) | e;     // byte e of two words, side by side
            win[e] = __builtin_amdgcn_perm(d[1], d[0], pick) | (__builtin_amdgcn_perm(d[3], d[2], pick) << 16);
        }
    } else {
        const uint4 h = *reinterpret_cast<const uint4*>(st);
        const uint32_t held[4] = {h.x, h.y, h.z, h.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) win[e] = (held[e] >> 8) | (((x_new >> (8 * e)) & 0xffu) << 24);
        *reinterpret_cast<uint4*>(st) = make_uint4(win[0], win[1], win[2], win[3]);
    }
    const Part part = part_of(p, ch0);
    float s_out[4], inv_s_out[4], v[4];
    bool exact_only[4];
    out_scales4_of(p, part, ch0, s_out);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        inv_s_out[e] = 1.0f / s_out[e];
        exact_only[e] = conv_needs_exact_route(s_out[e]);
        v[e] = part.s_bias * static_cast<float>(static_cast<int8_t>(b4 >> (8 * e)));
#pragma unroll
        for (int i = 0; i < 4; ++i)
            v[e] = __builtin_fmaf(part.s_in * static_cast<float>(static_cast<int8_t>(taps[e] >> (8 * i))), static_cast<float>(static_cast<int8_t>(win[e] >> (8 * i))), v[e]);
    }
    const ConvQuantRegs kq(__builtin_fminf(__builtin_fminf(s_out[0], s_out[1]), __builtin_fminf(s_out[2], s_out[3])));
    int64_t out_ls, out_cs;
    *reinterpret_cast<uint32_t*>(out_ptr(p, part, b, ch0, &out_ls, &out_cs)) = conv_quant4(v, s_out, inv_s_out, p.silu_activation, exact_only, kq);
}

int validate(const QaConv2Params* p, bool update) {
    if (!p) return QA_ERR_NULL;
    if (p->batch < 0 || p->dim < 0 || p->seqlen < 0 || p->batch > 65535) return QA_ERR_SHAPE;
    // (a call over no elements may pass null tensors)
    const bool empty = p->batch == 0 || p->dim == 0 || (!update && p->seqlen == 0);
    if (!empty && (!p->xBC || !p->weight || !p->x || !p->B || !p->C)) return QA_ERR_NULL;
    if (!empty && (!p->x_out_scales || !p->B_out_scales || !p->C_out_scales)) return QA_ERR_NULL;
    if ((p->x_head_group_range == nullptr) != (p->x_dim_group_range == nullptr)) return QA_ERR_NULL;
    if (!empty && update && !p->conv_state) return QA_ERR_NULL;
    if (p->width < 2 || p->width > 4) return QA_ERR_SHAPE;
    if (p->x_dim < 0 || p->x_headdim < 1 || p->d_state < 1 || p->n_groups < 1) return QA_ERR_SHAPE;
    if (p->x_dim % p->x_headdim != 0 || p->x_dim % p->n_groups != 0) return QA_ERR_SHAPE;
    if (p->x_dim + 2 * p->d_state * p->n_groups != p->dim) return QA_ERR_SHAPE;
    if (p->x_head_group_range && (p->nhead_groups < 1 || p->ndim_groups < 1)) return QA_ERR_SHAPE;
    if (update && p->conv_state_len != p->width && p->conv_state_len != p->width - 1) return QA_ERR_SHAPE;
    return QA_OK;
}

}  // namespace
}  // namespace qa

namespace qa {
int conv_channel_last_fwd(const QaConv2Params& p, hipStream_t stream) {
    const bool packed = p.width == 4 && p.weight_width_stride == 1 && p.weight_c_stride == 4 && aligned16(p.weight) && aligned4(p.bias);
    const bool one_scale = packed && !p.x_out_scales;
    const bool tables = packed && p.x_out_scales && p.x_head_group_range && p.x_dim_group_range && p.nhead_groups <= 8 && p.ndim_groups <= 8 && p.x_headdim % 4 == 0 &&
                        256 % p.x_headdim == 0 && p.d_state % 4 == 0 && (p.n_groups == 1 || p.x_dim / p.n_groups % 256 == 0) && p.x_dim > 0 && p.B_out_scales && p.C_out_scales;
    // Steps per wave: 4 to 256, whichever takes the busiest SIMD's waves the shortest: in ns about 145 a step and for a wave's
    // set-up (taps, scales, the three inputs ahead) 100 with one output scale and 400 with tables, and 160 a step of the last wave with
    // nobody beside it.  Measured in a layer with runs of 4, 6, 8, 12, 16, 24, 32 steps, us: one scale 1 x 512 x 1536 channels 4.6, 4.6, 5.4, 5.8,
    // 6.9, 8.1, 10.0; 3 x 1021 x 5120 13.4, 14.0, 14.9, 16.0, 15.6, 16.3, 16.0; 4 x 1500 x 2048 11.8, 12.1, 11.7, 12.4, 12.4, 12.7, 14.7; tables 1 x 1531 x
    // 5376 11.8, 12.0, 11.6, 12.2, 11.6, 13.9, 14.6; 3 x 1000 x 2304 10.0, 9.8, 10.4, 10.8, 10.5, 12.5, 12.5; 4 x 4096 x 5376 (a faster card than that of the figures at the top) 62, 54, 52, 51, 49, 50, 50.  The
    // choice is at most 4 % behind the best run.  Anything else: 250, and two and three taps, which come byte by byte, 350 and 100 a step (over
    // 148 sizes of each the choice is 0.2 % behind the best power of two and 0.3 with fewer taps).
    int run = 4;
    {
        const int64_t ch_blocks = (p.dim + 255) / 256, simds = 4LL * compute_units();
        const int set_up = one_scale ? 100 : tables ? 400 : p.width == 4 ? 250 : 350, alone = p.width == 4 ? 160 : 100;
        int64_t best = -1;
        for (int r : {4, 6, 8, 12, 16, 24, 32, 48, 64, 128, 256}) {
            if (!one_scale && !tables && (r & (r - 1))) continue;
            const int64_t waves = ch_blocks * (((p.seqlen + r - 1) / r + 3) / 4 * 4) * p.batch;
            const int64_t cost = (waves + simds - 1) / simds * (145 * r + set_up) + alone * r;
            if (best < 0 || cost < best || (p.seqlen + 4LL * run - 1) / (4 * run) > 65535) { best = cost; run = r; }
        }
    }
    const int64_t run_blocks = (p.seqlen + 4 * run - 1) / (4 * run);
    if (run_blocks > 65535) return QA_ERR_SHAPE;
    dim3 grid((p.dim + 255) / 256, static_cast<unsigned>(run_blocks), p.batch);
    auto with = [&](auto silu_c) {
        constexpr bool kSilu = decltype(silu_c)::value;
        auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, stream, p, run); };
        auto by_run = [&](auto scales_c) {
            constexpr ScaleKind kScales = decltype(scales_c)::value;
            if (run == 4) go(conv2_fwd_kernel<kSilu, true, kScales, 4>);
            else if (run == 6) go(conv2_fwd_kernel<kSilu, true, kScales, 6>);
            else go(conv2_fwd_kernel<kSilu, true, kScales, 8>);
        };
        if (one_scale) by_run(std::integral_constant<ScaleKind, kOneScale>{});
        else if (tables) by_run(std::integral_constant<ScaleKind, kTables>{});
        else if (packed) go(conv2_fwd_kernel<kSilu, true, kWalk, 8>);
        else go(conv2_fwd_kernel<kSilu, false, kWalk, 8>);
    };
    if (p.silu_activation) with(std::true_type{});
    else with(std::false_type{});
    return check_launch();
}
}  // namespace qa

namespace qa {
int conv_single_update(const QaConv2Params& p, hipStream_t stream) {
    const bool words = conv_words_ok(p) && p.xBC_c_stride == 1 && p.xBC_batch_stride % 4 == 0 && aligned4(p.xBC);
    const dim3 grid4(static_cast<unsigned>((p.dim / 4 + kThreads - 1) / kThreads), static_cast<unsigned>(p.batch));
    if (words && conv_state_in_rows(p)) {
        hipLaunchKernelGGL(conv2_update4_kernel<true>, grid4, dim3(kThreads), 0, stream, p);
        return check_launch();
    }
    if (words && conv_state_in_words(p)) {
        hipLaunchKernelGGL(conv2_update4_kernel<false>, grid4, dim3(kThreads), 0, stream, p);
        return check_launch();
    }
    const int64_t blocks = (static_cast<int64_t>(p.batch) * p.dim + kThreads - 1) / kThreads;
    if (blocks > 0x7fffffffLL) return QA_ERR_SHAPE;
    hipLaunchKernelGGL(conv2_update_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, stream, p);
    return check_launch();
}
}  // namespace qa

extern "C" int qa_quamba2_conv1d_fwd(const QaConv2Params* p, void* stream_) {
    using namespace qa;
    const int st = validate(p, false);
    if (st != QA_OK) return st;
    if (p->xBC_c_stride != 1 || p->x_c_stride != 1 || p->B_c_stride != 1 || p->C_c_stride != 1) return QA_ERR_STRIDE;
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const int64_t total = static_cast<int64_t>(p->batch) * p->dim * p->seqlen;
    if (total == 0) return QA_OK;
    const int bc = p->d_state * p->n_groups;
    auto mult4 = [](int64_t v) { return v % 4 == 0; };
    const bool vec = p->x_dim % 4 == 0 && bc % 4 == 0 && aligned4(p->xBC) && aligned4(p->x) && aligned4(p->B) &&
                     aligned4(p->C) && mult4(p->xBC_batch_stride) && mult4(p->xBC_l_stride) &&
                     mult4(p->x_batch_stride) && mult4(p->x_l_stride) && mult4(p->B_batch_stride) &&
                     mult4(p->B_l_stride) && mult4(p->C_batch_stride) && mult4(p->C_l_stride);
    if (vec) return conv_channel_last_fwd(*p, stream);
    if (p->conv_state) return QA_ERR_STRIDE;                      // (written by the kernel for aligned rows only)
    const int64_t blocks = (total + kThreads - 1) / kThreads;
    if (blocks > 0x7fffffffLL) return QA_ERR_SHAPE;
    hipLaunchKernelGGL(conv2_fwd_generic_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, stream, *p);
    return check_launch();
}

extern "C" int qa_quamba2_conv1d_update(const QaConv2Params* p, void* stream_) {
    using namespace qa;
    const int st = validate(p, true);
    if (st != QA_OK) return st;
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const int64_t total = static_cast<int64_t>(p->batch) * p->dim;
    if (total == 0) return QA_OK;
    return conv_single_update(*p, stream);
}
