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

}  // namespace qa
