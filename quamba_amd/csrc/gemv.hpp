// Products with very few activation rows (one decode step of a few sequences): see gemv.hip.
#pragma once
#include "qa_common.hpp"

namespace qa {

constexpr int kGemvRows = 8;
constexpr int kGemvConvGroups = 8;     // head groups and dim groups of the conv's output scales, at most

enum GemvRule {
    kGemvRowOuter = 0,     // s_row * (s_col * acc)
    kGemvColOuter = 1,     // s_col * (s_row * acc)
    kGemvAlpha = 2,        // alpha * acc
    kGemvHalfAway = 3,     // (s_col * s_row) * acc
};

struct GemvParams {
    int m, n, k, bits;
    int out_type;          // QaOutType
    int rule, half_away;   // half_away: int8 results round half away from zero
    int row_numel, col_numel;
    float alpha;
    int64_t lda, ldw, ldd; // ldw: bytes between the rows of w
    const int8_t* a;
    const void* w;
    const __half* s_group; // 4 bits: (k / 128, n)
    const float* row_scale;
    const float* col_scale;
    void* d;
};

// The output columns ch0 .. ch0 + conv.dim - 1 are the input of a causal conv's single-step update (width 4): the conv
// state moves on, the conv's int8 output goes where `conv` says, and the columns themselves are not stored.
struct GemvConv {
    int ch0;
    QaConv2Params conv;
};
// (four columns a wave: whole quads of channels, inside one part and one head; taps as one word)
inline bool gemv_conv_ok(const GemvConv& f) {
    const QaConv2Params& c = f.conv;
    return c.width == 4 && c.weight_width_stride == 1 && c.weight_c_stride == 4 && aligned4(c.weight) && f.ch0 % 4 == 0 && c.dim % 4 == 0 &&
           c.x_dim % 4 == 0 && c.x_headdim % 4 == 0 && (c.x_dim == c.dim || (c.d_state * c.n_groups) % 4 == 0) &&
           c.nhead_groups <= kGemvConvGroups && c.ndim_groups <= kGemvConvGroups;
}

int gemv_launch(const GemvParams& p, const GemvConv* conv, hipStream_t stream);

// One activation row that is made on the spot: sat8(round_half_away(H y * had_scale)) of a row y of k fp16 values
// (qa_hadamard_quant); fp16 results.  QA_ERR_UNSUPPORTED: not for these sizes (the caller then makes the two calls).
struct GemvRotate {
    const __half* y;
    float had_scale;
};
int gemv_rotated_launch(const GemvParams& p, const GemvRotate& r, hipStream_t stream);

}  // namespace qa
