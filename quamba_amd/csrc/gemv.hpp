// Products with few activation rows (a decode step): one to four of them in gemv.hip, more in gemm_split.hpp.
#pragma once
#include "qa_common.hpp"

#include <algorithm>

namespace qa {

constexpr int kGemvRows = 4;
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

// The same as the kernels take it.  What a launch costs the host grows with its arguments - 2.8 us up to 64 bytes, 3.4 at 128, 3.7
// at 256, 3.9 at 512 - and a decode step of one or two sequences is as long as its launches.  (Row pitches fit an int: qa_gemm_w8a8,
// qa_gemm_w4a8 and a layer call's checks refuse operands of 0x70000000 bytes and more.)
struct GemvArgs {
    const int8_t* a;
    const void* w;
    const __half* s_group;
    const float* row_scale;
    const float* col_scale;
    void* d;
    int64_t ldd;
    int m, n, k, lda, ldw;
    float alpha;
    uint8_t rule, half_away, one_row_scale, one_col_scale;
    explicit GemvArgs(const GemvParams& p)
        : a(p.a), w(p.w), s_group(p.s_group), row_scale(p.row_scale), col_scale(p.col_scale), d(p.d), ldd(p.ldd), m(p.m), n(p.n), k(p.k),
          lda(static_cast<int>(p.lda)), ldw(static_cast<int>(p.ldw)), alpha(p.alpha), rule(static_cast<uint8_t>(p.rule)),
          half_away(p.half_away != 0), one_row_scale(p.row_numel == 1), one_col_scale(p.col_numel == 1) {}
};

// The output columns ch0 .. ch0 + conv.dim - 1 are the input of a causal conv's single-step update (width 4): the conv
// state moves on, the conv's int8 output goes where `conv` says, and the columns themselves are not stored.
struct GemvConv {
    int ch0;
    QaConv2Params conv;
};
struct NoGemvConv {};
// (four columns a wave: whole quads of channels, inside one part and one head; taps as one word)
inline bool gemv_conv_ok(const GemvConv& f) {
    const QaConv2Params& c = f.conv;
    return c.width == 4 && c.weight_width_stride == 1 && c.weight_c_stride == 4 && aligned4(c.weight) && f.ch0 % 4 == 0 && c.dim % 4 == 0 &&
           c.x_dim % 4 == 0 && c.x_headdim % 4 == 0 && (c.x_dim == c.dim || (c.d_state * c.n_groups) % 4 == 0) &&
           c.nhead_groups <= kGemvConvGroups && c.ndim_groups <= kGemvConvGroups;
}
// a state of four codes that is one word, whatever lies between the channels' words
inline bool gemv_state_in_words(const QaConv2Params& c) {
    return c.conv_state_len == 4 && c.conv_state_l_stride == 1 && c.conv_state_c_stride % 4 == 0 && c.conv_state_batch_stride % 4 == 0 && aligned4(c.conv_state);
}

int gemv_launch(const GemvParams& p, const GemvConv* conv, hipStream_t stream);

// gemm_split_w8.hip, gemm_split_w4.hip: K over the eight waves of a workgroup, in one of these tiles.  What a launch takes, in
// us with `units` of 128 codes of K, is 2.9 and rounds (of one workgroup per CU) x (fixed + per_unit x units), as measured over
// 1 .. 12288 rows of 32 .. 20000 columns and K from 128 to 8192, the weights in the L2s and beyond them; the fixed part is
// the sums of the larger tiles, which all meet at the end (negative: another tile is always the faster one).
struct SplitShape {
    int rows, cols;
    float fixed[2], per_unit[2];       // int8, 4 bits
};
constexpr SplitShape kSplitShapes[] = {
    {16, 16, {0.0f, 0.0f}, {0.045f, 0.045f}}, {16, 32, {0.0f, 0.0f}, {0.07f, 0.075f}},  {16, 48, {0.0f, 0.0f}, {0.1f, 0.115f}},
    {32, 32, {0.0f, 0.0f}, {0.09f, 0.1f}},    {32, 48, {0.3f, 0.2f}, {0.125f, 0.135f}}, {32, 80, {1.2f, 1.0f}, {0.155f, 0.22f}},
    {64, 48, {-1.0f, 1.6f}, {0.0f, 0.165f}}, {64, 80, {2.6f, 2.5f}, {0.2f, 0.31f}},
};
struct SplitChoice {
    int shape;
    float us, rounds;
};
inline SplitChoice split_choice(int bits, int m, int n, int k, int cus, bool conv = false) {
    SplitChoice best = {-1, 1e30f, 0.0f};
    for (int i = 0; i < static_cast<int>(sizeof(kSplitShapes) / sizeof(kSplitShapes[0])); ++i) {
        const SplitShape& s = kSplitShapes[i];
        if (s.fixed[bits == 4] < 0.0f) continue;
        const int64_t tiles = static_cast<int64_t>((m + s.rows - 1) / s.rows) * ((n + s.cols - 1) / s.cols);
        const float rounds = static_cast<float>((tiles + cus - 1) / cus), units = static_cast<float>((k + 127) / 128);
        // 4 bits: workgroups that share a CU expand their codes at the same time, which tells from two of the large tiles and from five of the
        // others on: 777 x 2560 x 5120 33.4 us by 64 x 48, 28.0 expanded once; 777 x 1536 x 3072 17.3 by 64 x 48, 18.3 by 32 x 32, 16.9 in
        // 64 x 128 tiles; 100 x 18560 x 4096 37.5 by 64 x 80, 25.4 in 128 x 128 tiles.  With far more rows than columns hardly anyone
        // shares the rows: 4096 x 160 x 4096 and 4096 x 192 x 4096 21.1 and 21.5 by 64 x 48, 14.8 and 15.0 in 64 x 64 tiles, 6000 x 128 x 3072
        // 14.1 by 32 x 32, 11.9 in tiles.
        // 8 bits: with more rows than columns the workgroups each fetch rows of their own from memory, most of all when a CU has
        // several: 2400 x 192 x 5120 14.8 us in two rounds of 32 x 32, 12.5 by 32 x 80, 11.0 in 64 x 64 tiles; 2400 x 160 x 4096 11.4 in
        // two rounds, 8.7 in tiles, 3000 x 128 x 3072 9.5 and 7.5 - but 1800 x 192 x 5120 10.0 by 32 x 48, 11.0 in tiles.
        // Both: each round ends in sums of its own, which tells where K is short: 4 bits 200 x 3072 x 768 6.4 in three rounds of 32 x 32,
        // 5.1 in 64 x 64 tiles, 1531 x 768 x 1536 10.7 in three of 32 x 48, 9.6 in 64 x 128; int8 777 x 1536 x 48 7.0 in five of 32 x 32,
        // 4.4 in 128 x 64 tiles.  From K = 3072 on the price is the better one without them (4 bits 16 x 18560 x 4096 10.6 in three
        // rounds, 11.8 in two), and a conv behind the product is priced by the round as it is.
        float crowd = 1.0f;
        if (bits == 4 && rounds > (s.rows == 64 ? 1.0f : 4.0f)) crowd = 1.3f;
        if (bits == 4 && m / 4 > n) crowd = s.rows == 64 ? 1.8f : 1.3f;
        if (bits == 8 && m > n) crowd = rounds > 1.0f ? 1.6f : 1.2f;
        const float more = conv || k > 2048 ? 0.0f : 0.4f * (rounds - 1.0f);
        const float us = 2.9f + more + rounds * crowd * (s.fixed[bits == 4] + s.per_unit[bits == 4] * units);
        if (tiles <= 0x7fffffff && us < best.us) best = {i, us, rounds};
    }
    return best;
}
// Operands as the products' entry points take them (16-byte aligned rows; K a multiple of 16, or of 128 with 4 bits; with 8
// bits every offset below 2^31).  4 bits: a tile's rows and the group scales (null: per channel) are addressed with 32 bits.
inline bool split_addressable_w4(int n, int k) { return 40LL * k <= 0x7fffffffLL && static_cast<int64_t>(n) * (k / 128) < 1 << 29; }
int split_launch_w8(const GemvParams& p, int shape, const GemvConv* conv, hipStream_t stream);
int split_launch_w4(const GemvParams& p, int shape, const GemvConv* conv, hipStream_t stream);

// us of the products' launches without it, where one round of their tiles is enough (else far more): gemm_w8a8.hip, gemm_w4a8.hip
float tiles_us_w8(int m, int n, int k, int cus);
float tiles_us_w4(int m, int n, int k, int cus);

// Which of the two a product of up to kGemvRows rows takes.  A row is work for the vector units in gemv.hip and free in a
// block of sixteen here, but a launch of small size is the faster one there: one and two rows, and three and four while the
// weights are few (in a layer, us with three and four rows, gemv against split: int8 8192 x 2048 with the conv 5.2 against 6.8, 2048 x
// 4096 3.6 / 4.6, 10240 x 2560 8.0 / 7.7; 4 bits 6144 x 1536 with the conv 5.7 / 6.1, 10240 x 2560 10.3 / 7.5, 8416 x 2048 11.4 / 8.0, 192 x
// 5120 3.2 / 4.4).  Five to eight rows, where a row more takes twice the registers, are the faster ones here with any weights (alone, weights
// from beyond the L2s: int8 1536 x 48 and 2048 x 4096 the same 4.2, 8192 x 2048 6.4 / 4.8, 10240 x 2560 9.2 / 6.2; 4 bits 192 x 5120 4.2 / 4.3,
// 3072 x 768 5.0 / 4.2, 2048 x 4096 5.8 / 4.2, 18560 x 4096 18.4 / 11.1).
inline bool gemv_is_faster(int bits, int m, int n, int k) { return m <= 2 || (m <= kGemvRows && static_cast<int64_t>(n) * k < (bits == 8 ? 20000000 : 10000000)); }

// One activation row that is made on the spot: sat8(round_half_away(H y * had_scale)) of a row y of k fp16 values
// (qa_hadamard_quant); fp16 results.  QA_ERR_UNSUPPORTED: not for these sizes (the caller then makes the two calls).
struct GemvRotate {
    const __half* y;
    float had_scale;
};
int gemv_rotated_launch(const GemvParams& p, const GemvRotate& r, hipStream_t stream);

}  // namespace qa
