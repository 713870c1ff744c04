// The channels of the Mamba2 xBC conv: which part a channel belongs to, its scales, where its output goes.
#pragma once
#include "conv_common.hpp"

namespace qa {

struct Part {
    int index;        // 0 = x, 1 = B, 2 = C
    int offset;       // first channel of the part inside xBC
    float s_in;       // weight scale * input scale
    float s_bias;
};

__device__ __forceinline__ Part part_of(const QaConv2Params& p, int ch) {
    const int bc = p.d_state * p.n_groups;
    Part r;
    if (ch < p.x_dim) {
        r.index = 0; r.offset = 0; r.s_in = p.scale_wx * p.scale_x; r.s_bias = p.scale_bx;
    } else if (ch < p.x_dim + bc) {
        r.index = 1; r.offset = p.x_dim; r.s_in = p.scale_wB * p.scale_B; r.s_bias = p.scale_bB;
    } else {
        r.index = 2; r.offset = p.x_dim + bc; r.s_in = p.scale_wC * p.scale_C; r.s_bias = p.scale_bC;
    }
    return r;
}

// Output scale of channel `ch`; the range walk is the reference's (first range that contains the index).
__device__ __forceinline__ float out_scale_of(const QaConv2Params& p, const Part& part, int ch) {
    if (!p.x_out_scales) return p.x_out_scale;          // one host-side scale: the Mamba1 conv
    const bool grouped = p.x_head_group_range != nullptr && p.x_dim_group_range != nullptr;
    if (part.index != 0) {
        const float* s = part.index == 1 ? p.B_out_scales : p.C_out_scales;
        return grouped ? s[(ch - part.offset) / p.d_state] : s[0];
    }
    if (!grouped) return p.x_out_scales[0];
    const int group_size = p.x_dim / p.n_groups;
    const int g = ch / group_size;
    const int head = (ch % group_size) / p.x_headdim;
    const int d = ch % p.x_headdim;
    const float* scales = p.x_out_scales + g * p.nhead_groups * p.ndim_groups;
    const int32_t* hr = p.x_head_group_range + g * p.nhead_groups;
    const int32_t* dr = p.x_dim_group_range + g * p.nhead_groups * p.ndim_groups;
    float s = 0.0f;
    int h_start = 0;
    for (int hg = 0; hg < p.nhead_groups; ++hg) {
        if (h_start <= head && head < hr[hg]) {
            int d_start = 0;
            for (int dg = 0; dg < p.ndim_groups; ++dg) {
                if (d_start <= d && d < dr[hg * p.ndim_groups + dg]) {
                    s = scales[hg * p.ndim_groups + dg];
                    break;
                }
                d_start = dr[hg * p.ndim_groups + dg];
            }
            break;
        }
        h_start = hr[hg];
    }
    return s;
}

// The same for the four channels ch .. ch + 3 (of one part, ch a multiple of four).  Range tables of up to kRangeUnroll
// entries and whole quads of channels per head: every entry of a level is requested at once - three round trips instead
// of a chain of up to a dozen dependent loads per channel, which took longer than a short run's steps.
constexpr int kRangeUnroll = 8;
__device__ __forceinline__ void out_scales4_of(const QaConv2Params& p, const Part& part, int ch, float (&s)[4]) {
    const bool grouped = p.x_head_group_range != nullptr && p.x_dim_group_range != nullptr;
    if (!p.x_out_scales || !grouped || part.index != 0) {
        // one scale, or one per ssd group
        if (!p.x_out_scales || !grouped) {
            const float one = out_scale_of(p, part, ch);
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] = one;
        } else {
            const float* scales = part.index == 1 ? p.B_out_scales : p.C_out_scales;
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] = scales[(ch + e - part.offset) / p.d_state];
        }
        return;
    }
    if (p.nhead_groups > kRangeUnroll || p.ndim_groups > kRangeUnroll || p.x_headdim % 4 != 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = out_scale_of(p, part, ch + e);
        return;
    }
    const int group_size = p.x_dim / p.n_groups, g = ch / group_size, head = (ch % group_size) / p.x_headdim, d = ch % p.x_headdim;
    const int32_t* hr = p.x_head_group_range + g * p.nhead_groups;
    int ends[kRangeUnroll], hg = 0;
#pragma unroll
    for (int j = 0; j < kRangeUnroll - 1; ++j) ends[j] = hr[min(j, p.nhead_groups - 1)];
#pragma unroll
    for (int j = 0; j < kRangeUnroll - 1; ++j) hg += j < p.nhead_groups - 1 && head >= ends[j] ? 1 : 0;
    const int row = (g * p.nhead_groups + hg) * p.ndim_groups;
#pragma unroll
    for (int j = 0; j < kRangeUnroll - 1; ++j) ends[j] = p.x_dim_group_range[row + min(j, p.ndim_groups - 1)];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        int dg = 0;
#pragma unroll
        for (int j = 0; j < kRangeUnroll - 1; ++j) dg += j < p.ndim_groups - 1 && d + e >= ends[j] ? 1 : 0;
        s[e] = p.x_out_scales[row + dg];
    }
}

__device__ __forceinline__ int8_t* out_ptr(const QaConv2Params& p, const Part& part, int b, int ch,
                                            int64_t* l_stride, int64_t* c_stride) {
    const int local = ch - part.offset;
    if (part.index == 0) { *l_stride = p.x_l_stride; *c_stride = p.x_c_stride; return p.x + b * p.x_batch_stride + local * p.x_c_stride; }
    if (part.index == 1) { *l_stride = p.B_l_stride; *c_stride = p.B_c_stride; return p.B + b * p.B_batch_stride + local * p.B_c_stride; }
    *l_stride = p.C_l_stride; *c_stride = p.C_c_stride;
    return p.C + b * p.C_batch_stride + local * p.C_c_stride;
}

// The single-step update of four neighbouring channels of a part, for words in every operand: four taps a channel back to
// back, inputs and outputs with unit channel stride, and a state that is either channel-contiguous (a word per step: the
// Mamba2 layer's buffer) or four codes a channel (a 16-byte piece: the Mamba1 layer's).
// What the four channels bring, the same for every row: taps and bias already scaled (a product of some rows makes them once a
// column and hands them to the rows' threads: int8 64 x 10240 x 2560 11.8 -> 11.4 us, 4 bits 32 x 18560 x 4096 17.2 -> 16.3).
struct alignas(16) ConvQuad {
    float taps[4][4], bias[4], s_out[4];
};
__device__ __forceinline__ ConvQuad conv_quad(const QaConv2Params& p, const Part& part, int ch0) {
    ConvQuad q;
    const uint4 w = *reinterpret_cast<const uint4*>(p.weight + ch0 * 4);
    const uint32_t bias = p.bias ? *reinterpret_cast<const uint32_t*>(p.bias + ch0) : 0u, taps[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        q.bias[e] = part.s_bias * static_cast<float>(static_cast<int8_t>(bias >> (8 * e)));
#pragma unroll
        for (int i = 0; i < 4; ++i) q.taps[e][i] = part.s_in * static_cast<float>(static_cast<int8_t>(taps[e] >> (8 * i)));
    }
    out_scales4_of(p, part, ch0, q.s_out);
    return q;
}
// the state, as loaded: a word per step of the three that the window keeps, or a word per channel
template <bool CHANNEL_ROWS>
struct ConvHeld {
    uint32_t w[CHANNEL_ROWS ? 3 : 4];
};
template <bool CHANNEL_ROWS>
__device__ __forceinline__ ConvHeld<CHANNEL_ROWS> conv_held4(const QaConv2Params& p, int b, int ch0) {
    const int8_t* st = p.conv_state + b * p.conv_state_batch_stride + ch0 * p.conv_state_c_stride;
    ConvHeld<CHANNEL_ROWS> h;
    if constexpr (CHANNEL_ROWS) {
#pragma unroll
        for (int i = 0; i < 3; ++i) h.w[i] = *reinterpret_cast<const uint32_t*>(st + (p.conv_state_len - 3 + i) * p.conv_state_l_stride);
    } else {
        const uint4 v = *reinterpret_cast<const uint4*>(st);
        h.w[0] = v.x; h.w[1] = v.y; h.w[2] = v.z; h.w[3] = v.w;
    }
    return h;
}
// x_new: the new inputs, a byte per channel.  The state moves on; returns the four outputs.
template <bool CHANNEL_ROWS>
__device__ __forceinline__ uint32_t conv_step4(const QaConv2Params& p, int b, int ch0, const ConvQuad& q, const ConvHeld<CHANNEL_ROWS>& h, uint32_t x_new) {
    int8_t* st = p.conv_state + b * p.conv_state_batch_stride + ch0 * p.conv_state_c_stride;
    uint32_t win[4];                                              // byte j of win[e]: input t - 3 + j of channel ch0 + e
    if constexpr (CHANNEL_ROWS) {
        const uint32_t d[4] = {h.w[0], h.w[1], h.w[2], x_new};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i >= 4 - p.conv_state_len) *reinterpret_cast<uint32_t*>(st + (i - (4 - p.conv_state_len)) * p.conv_state_l_stride) = d[i];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t pick = 0x0c0c0000u | ((4u + e) << 8) | e;     // byte e of two words, side by side
            win[e] = __builtin_amdgcn_perm(d[1], d[0], pick) | (__builtin_amdgcn_perm(d[3], d[2], pick) << 16);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) win[e] = (h.w[e] >> 8) | (((x_new >> (8 * e)) & 0xffu) << 24);
        *reinterpret_cast<uint4*>(st) = make_uint4(win[0], win[1], win[2], win[3]);
    }
    float inv_s_out[4], v[4];
    bool exact_only[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        inv_s_out[e] = p.silu_activation ? 0.0f : 1.0f / q.s_out[e];     // (SiLU divides by both at once)
        exact_only[e] = conv_needs_exact_route(q.s_out[e]);
        v[e] = q.bias[e];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[e] = __builtin_fmaf(q.taps[e][i], static_cast<float>(static_cast<int8_t>(win[e] >> (8 * i))), v[e]);
    }
    const ConvQuantRegs kq(__builtin_fminf(__builtin_fminf(q.s_out[0], q.s_out[1]), __builtin_fminf(q.s_out[2], q.s_out[3])));
    return conv_quant4(v, q.s_out, inv_s_out, p.silu_activation, exact_only, kq);
}
// the layouts these take: words everywhere but in the state and in the inputs ...
inline bool conv_words_ok(const QaConv2Params& p) {
    auto mult4 = [](int64_t v) { return v % 4 == 0; };
    return p.width == 4 && p.weight_width_stride == 1 && p.weight_c_stride == 4 && aligned16(p.weight) && aligned4(p.bias) && mult4(p.x_dim) &&
           p.x_c_stride == 1 && mult4(p.x_batch_stride) && aligned4(p.x) &&
           (p.x_dim == p.dim ||                                   // (the Mamba1 conv: no B and C parts)
            (mult4(static_cast<int64_t>(p.d_state) * p.n_groups) && p.B_c_stride == 1 && mult4(p.B_batch_stride) && aligned4(p.B) && p.C_c_stride == 1 && mult4(p.C_batch_stride) && aligned4(p.C)));
}
// ... and the two layouts of the state
inline bool conv_state_in_rows(const QaConv2Params& p) { return p.conv_state_c_stride == 1 && p.conv_state_l_stride % 4 == 0 && p.conv_state_batch_stride % 4 == 0 && aligned4(p.conv_state); }
inline bool conv_state_in_words(const QaConv2Params& p) {
    return p.conv_state_len == 4 && p.conv_state_l_stride == 1 && p.conv_state_c_stride == 4 && p.conv_state_batch_stride % 16 == 0 && aligned16(p.conv_state);
}

}  // namespace qa
