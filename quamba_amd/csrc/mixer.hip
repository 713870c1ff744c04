// The assembled mixers: one library call enqueues every kernel of a layer call.
//
// What a small call costs is the host: seven to nine launches, each behind its own argument checks, tensor
// allocations and stream lookups in the caller's language (about 22 us each from Python against 3-5 us of kernel at
// one token).  Here the intermediates are sections of one workspace and the launches follow each other at the
// runtime's own pace.
//
// Layout: activations stay row-major (token, channel) from in_proj to out_proj.  The conv walks time with four
// channels per lane, the scan stages token-major rows, x_proj and dt_proj are plain row-major products - so no second
// copy of the conv's output, no transposition of B and C, no padding of the token count, and prompts of any length
// run on the same kernels.
//
// A call is refused before its first launch or not at all (validate, ready): a step advances both states in place, and one
// that stopped half way could not be made again another way.
#include "conv2_common.hpp"
#include "gemv.hpp"
#include "hadamard_core.hpp"
#include "mixer_common.hpp"
#include "ssd_common.hpp"

#include <algorithm>

namespace qa {
namespace {

constexpr int kExpandOnceRows = 65;       // from this many rows on the product may want the 4-bit weights expanded once (qa_gemm_w4a8 decides)

// Sections of the workspace, each 256-byte aligned.
struct Carver {
    uint8_t* base;
    int64_t off = 0;
    template <typename T>
    T* take(int64_t bytes) {
        T* r = base ? reinterpret_cast<T*>(base + off) : nullptr;
        off = (off + bytes + 255) & ~int64_t(255);
        return r;
    }
};

struct Scratch {
    void* p;
    int64_t bytes;
};

int64_t expanded_bytes(const QaLinearParams& w, int64_t rows) {
    return w.bits == 4 && rows >= kExpandOnceRows ? static_cast<int64_t>(w.n) * w.k : 0;
}

// d (rows, w.n) = the projection of a (rows, w.k).  channel_scale_last: the association of the transposed call
// (to_seqlen_last), whose products and bits the row-major one reproduces.
int project(const QaLinearParams& w, const int8_t* a, int64_t lda, int rows, void* d, int out_type, bool channel_scale_last,
            const Scratch& w8, void* stream) {
    if (w.bits == 4) {
        QaGemmW4A8Params p = {};
        p.m = rows; p.n = w.n; p.k = w.k;
        p.group_size = w.s_group ? 128 : -1;
        p.out_type = out_type;
        p.tok_scale_numel = 1;
        p.lda = lda; p.ldd = w.n;
        p.a = a; p.w_packed = static_cast<const uint8_t*>(w.weight); p.s_group = w.s_group;
        p.s_channel = w.col_scale; p.s_token = w.row_scale; p.d = d;
        if (expanded_bytes(w, rows)) { p.w8_workspace = w8.p; p.w8_workspace_bytes = w8.bytes; }
        return qa_gemm_w4a8(&p, stream);
    }
    QaGemmW8A8Params p = {};
    p.m = rows; p.n = w.n; p.k = w.k;
    p.out_type = out_type;
    p.lda = lda; p.ldw = w.k; p.ldd = w.n;
    p.a = a; p.w = static_cast<const int8_t*>(w.weight); p.d = d;
    p.a_scale = w.row_scale; p.w_scale = w.col_scale;
    p.a_scale_numel = 1; p.w_scale_numel = w.col_numel;
    if (channel_scale_last) {
        p.scale_order = 1;
    } else if (rows == 1 && w.row_rule == QA_ROW_ALPHA) {
        p.use_alpha = 1;
        p.alpha = w.alpha;
    } else if (rows == 1 && w.row_rule == QA_ROW_HALF_AWAY) {
        p.round_mode = QA_ROUND_HALF_AWAY;
    }
    return qa_gemm_w8a8(&p, stream);
}

// what the products would refuse: `rows` rows of activations, lda apart and 16-byte aligned, against w
int linear_check(const QaLinearParams& w, int64_t rows, int64_t lda) {
    if ((w.bits != 8 && w.bits != 4) || w.n < 1 || w.k < 1 || !w.weight || !w.col_scale || !w.row_scale) return QA_ERR_NULL;
    if (w.k % (w.bits == 8 ? 16 : 128) != 0 || (w.bits == 8 && w.col_numel != 1 && w.col_numel != w.n)) return QA_ERR_SHAPE;
    if (lda % 16 != 0 || lda < w.k || !aligned16(w.weight)) return QA_ERR_STRIDE;
    // 32-bit offsets (4-bit weights from the tile's first row)
    const int64_t weights = static_cast<int64_t>(w.n) * w.k;
    if (rows * lda >= 0x70000000LL || (w.bits == 8 ? weights >= 0x70000000LL : 64LL * w.k > 0x7fffffffLL || weights > 64LL * 0x7fffff00LL)) return QA_ERR_SHAPE;
    return QA_OK;
}

int hadamard_check(int dim) { return dim <= 32768 && hadamard_shape(dim).s != 0 ? QA_OK : QA_ERR_UNSUPPORTED; }

constexpr int64_t kConvSteps = 65535LL * 4 * 256;       // of a sequence: the grid of the forward conv

// in_proj of a decode step with the conv's step behind it in one launch (QA_ERR_UNSUPPORTED: two launches).  Behind a product
// that splits K the conv takes 0.3 us and 1.1 per four outputs of a thread, on the few waves that hold the sums, in each round of
// workgroups; 0.8 with 4-bit weights in tiles of up to 32 x 32, of which a CU has two at a time, one at its conv and one at its
// product.  A launch of its own takes 4.0, with grouped scales, whose table is walked first, 5.5 - and the product may then be
// another, faster one (us, apart -> together: int8 16 x 10240 x 2560 11.3 -> 8.6, 64 x 10240 x 2560 11.2 -> 10.8, 128 x 10240 x 2560
// 14.2 -> 15.9; 4 bits 24 x 10240 x 2560 9.9 -> 8.1, 40 x 8480 x 2048 12.4 -> 10.9, 64 x 18560 x 4096 33 -> 31; in three and four rounds
// int8 65 x 8192 x 2048 10.0 -> 12.3, 33 x 10576 x 2560 11.5 -> 13.2, 4 bits 65 x 18560 x 4096 30.5 -> 37.4, but 65 x 8192 x 2048
// 13.5 -> 11.8, 65 x 10576 x 2560 17.7 -> 16.1).
int project_conv(const QaLinearParams& w, const int8_t* a, int64_t lda, int rows, int8_t* d, int ch0, const QaConv2Params& conv, void* stream) {
    const GemvConv f = {ch0, conv};
    if (!gemv_conv_ok(f)) return QA_ERR_UNSUPPORTED;
    if (w.k % 16 != 0 || lda % 16 != 0 || !aligned16(a) || !aligned16(w.weight)) return QA_ERR_UNSUPPORTED;
    GemvParams g = {};
    g.m = rows; g.n = w.n; g.k = w.k; g.bits = w.bits;
    g.out_type = QA_OUT_I8;
    g.rule = kGemvRowOuter;
    if (w.bits == 8 && rows == 1 && w.row_rule == QA_ROW_ALPHA) { g.rule = kGemvAlpha; g.alpha = w.alpha; }
    if (w.bits == 8 && rows == 1 && w.row_rule == QA_ROW_HALF_AWAY) { g.rule = kGemvHalfAway; g.half_away = 1; }
    g.row_numel = 1; g.col_numel = w.bits == 4 ? w.n : w.col_numel;
    g.lda = lda; g.ldw = w.bits == 4 ? w.k / 2 : w.k; g.ldd = w.n;
    g.a = a; g.w = w.weight; g.s_group = static_cast<const __half*>(w.s_group);
    g.row_scale = w.row_scale; g.col_scale = w.col_scale; g.d = d;
    if (w.bits == 4 && (w.k % 128 != 0 || !split_addressable_w4(w.n, w.k))) return QA_ERR_UNSUPPORTED;
    const bool dot_products = w.bits == 8 || (w.s_group && w.n % 4 == 0 && (reinterpret_cast<uintptr_t>(w.s_group) & 7u) == 0);
    if (gemv_is_faster(w.bits, rows, w.n, w.k) && dot_products) return gemv_launch(g, &f, static_cast<hipStream_t>(stream));
    // (words in every operand and in the columns that are stored)
    if (!conv_words_ok(conv) || !(conv_state_in_words(conv) || conv_state_in_rows(conv)) || w.n % 4 != 0 || !aligned4(d)) return QA_ERR_UNSUPPORTED;
    const int cus = compute_units();
    const SplitChoice split = split_choice(w.bits, rows, w.n, w.k, cus, true);
    const float tiles = w.bits == 8 ? tiles_us_w8(rows, w.n, w.k, cus) : tiles_us_w4(rows, w.n, w.k, cus);
    const SplitShape& shape = kSplitShapes[split.shape];
    const int quads = (shape.rows * shape.cols / 4 + 511) / 512;
    const float of_conv = w.bits == 4 && shape.rows * shape.cols <= 32 * 32 ? 0.8f : 0.3f + 1.1f * static_cast<float>(quads);
    if (split.us + split.rounds * of_conv > std::min(split.us, tiles) + (conv.x_head_group_range ? 5.5f : 4.0f)) return QA_ERR_UNSUPPORTED;
    return w.bits == 8 ? split_launch_w8(g, split.shape, &f, static_cast<hipStream_t>(stream)) : split_launch_w4(g, split.shape, &f, static_cast<hipStream_t>(stream));
}

int hadamard(const void* y, int8_t* out, int rows, int dim, float scale, void* stream) {
    QaHadamardParams h = {};
    h.rows = rows; h.dim = dim; h.in_type = 0; h.scale = scale;
    h.x_row_stride = dim; h.out_row_stride = dim;
    h.x = y; h.out = out;
    return qa_hadamard_quant(&h, stream);
}

// out_proj of one row with the transform that makes its activations in the same launch (QA_ERR_UNSUPPORTED: apart)
int project_rotated(const QaLinearParams& w, const GemvRotate& r, void* out, void* stream) {
    if (w.bits == 4 && !w.s_group) return QA_ERR_UNSUPPORTED;
    GemvParams g = {};
    g.m = 1; g.n = w.n; g.k = w.k; g.bits = w.bits;
    g.out_type = QA_OUT_F16;
    g.rule = kGemvRowOuter;
    if (w.bits == 8 && w.row_rule == QA_ROW_ALPHA) { g.rule = kGemvAlpha; g.alpha = w.alpha; }
    if (w.bits == 8 && w.row_rule == QA_ROW_HALF_AWAY) g.rule = kGemvHalfAway;
    g.row_numel = 1; g.col_numel = w.bits == 4 ? w.n : w.col_numel;
    g.ldw = w.bits == 4 ? w.k / 2 : w.k; g.ldd = w.n;
    g.w = w.weight; g.s_group = static_cast<const __half*>(w.s_group);
    g.row_scale = w.row_scale; g.col_scale = w.col_scale; g.d = out;
    return gemv_rotated_launch(g, r, static_cast<hipStream_t>(stream));
}

#define QA_TRY(call)                       \
    do {                                   \
        const int st_ = (call);            \
        if (st_ != QA_OK) return st_;      \
    } while (0)

// ---------------------------------------------------------------------------------------------
// Mamba1
// ---------------------------------------------------------------------------------------------
struct Mamba1Buffers {
    int8_t *xz, *x, *x_dbl, *dt, *yq;
    __half* y;
    Scratch w8, scan;
    int64_t total;
};

QaSScanParams scan_sizes(const QaMamba1Params& p) {
    QaSScanParams s = {};
    s.batch = p.batch; s.dim = p.d_inner; s.seqlen = p.seqlen; s.dstate = p.d_state; s.n_groups = 1;
    s.delta_softplus = p.delta_softplus;                                       // (the workspace goes with it, sscan_tm.hip)
    return s;
}

// dt_proj inside the scan (sscan_tm.hip) or as a product of its own
bool dt_in_scan(const QaMamba1Params& p) {
    return p.dt_proj.bits == 8 && p.dt_proj.k <= kSscanDtRank && p.x_proj.n % 16 == 0 && p.seqlen * static_cast<int64_t>(p.x_proj.n) < 1 << 30;
}

Mamba1Buffers carve(const QaMamba1Params& p, void* base, bool step) {
    const int64_t t = static_cast<int64_t>(p.batch) * p.seqlen;
    Carver c{static_cast<uint8_t*>(base)};
    Mamba1Buffers b;
    b.xz = c.take<int8_t>(t * p.in_proj.n);
    b.x = c.take<int8_t>(t * p.d_inner);
    b.x_dbl = c.take<int8_t>(t * p.x_proj.n);
    b.dt = c.take<int8_t>(!step && dt_in_scan(p) ? 0 : t * p.dt_proj.n);       // (8 x 2048 tokens of 5120 channels: 84 MB)
    b.yq = c.take<int8_t>(t * p.d_inner);
    b.y = c.take<__half>(t * p.d_inner * 2);
    b.w8.bytes = std::max(std::max(expanded_bytes(p.in_proj, t), expanded_bytes(p.x_proj, t)),
                          std::max(expanded_bytes(p.dt_proj, t), expanded_bytes(p.out_proj, t)));
    b.w8.p = c.take<uint8_t>(b.w8.bytes);
    b.scan.bytes = step ? 0 : sscan_token_major_workspace(scan_sizes(p));
    b.scan.p = c.take<uint8_t>(b.scan.bytes);
    b.total = c.off;
    return b;
}

// the Mamba1 conv in the terms of the Mamba2 one: every channel an x channel, one output scale
QaConv2Params conv_of(const QaMamba1Params& p, const Mamba1Buffers& b) {
    QaConv2Params c = {};
    const int64_t len = p.seqlen;
    const int d = p.d_inner;
    c.batch = p.batch; c.dim = d; c.seqlen = p.seqlen; c.width = p.d_conv;
    c.silu_activation = 1;
    c.x_dim = d; c.x_headdim = d; c.d_state = 1; c.n_groups = 1;
    c.conv_state_len = p.conv_state_len;
    c.xBC_batch_stride = len * 2 * d; c.xBC_l_stride = 2 * d; c.xBC_c_stride = 1;
    c.x_batch_stride = len * d; c.x_l_stride = d; c.x_c_stride = 1;
    c.weight_c_stride = p.d_conv; c.weight_width_stride = 1;
    c.conv_state_batch_stride = p.conv_state_batch_stride; c.conv_state_c_stride = p.conv_state_c_stride; c.conv_state_l_stride = p.conv_state_l_stride;
    c.xBC = b.xz; c.weight = p.conv_weight; c.bias = p.conv_bias; c.x = b.x; c.conv_state = p.conv_state;
    c.scale_x = p.conv_scale_x; c.scale_wx = p.conv_scale_w; c.scale_bx = p.conv_scale_b; c.x_out_scale = p.conv_scale_out;
    return c;
}

int validate(const QaMamba1Params* p) {
    if (!p) return QA_ERR_NULL;
    if (p->batch < 1 || p->seqlen < 1 || p->batch > 65535 || p->seqlen > kConvSteps || static_cast<int64_t>(p->batch) * p->seqlen > 0x7fffffff) return QA_ERR_SHAPE;
    if (p->d_state != 16 || p->d_conv < 2 || p->d_conv > 4 || p->d_inner < 16 || p->d_inner % 16 != 0 || p->dt_rank % 4 != 0) return QA_ERR_UNSUPPORTED;
    if (p->in_proj.k != p->d_model || p->in_proj.n != 2 * p->d_inner || p->x_proj.k != p->d_inner ||
        p->x_proj.n < p->dt_rank + 2 * p->d_state || p->x_proj.n % 4 != 0 || p->dt_proj.k != p->dt_rank ||
        p->dt_proj.n != p->d_inner || p->out_proj.k != p->d_inner) return QA_ERR_SHAPE;
    if (p->conv_state_len != p->d_conv && p->conv_state_len != p->d_conv - 1) return QA_ERR_SHAPE;
    const int64_t t = static_cast<int64_t>(p->batch) * p->seqlen;
    QA_TRY(linear_check(p->in_proj, t, p->d_model));
    QA_TRY(linear_check(p->x_proj, t, p->d_inner));
    QA_TRY(linear_check(p->dt_proj, t, p->x_proj.n));
    QA_TRY(linear_check(p->out_proj, t, p->d_inner));
    return hadamard_check(p->d_inner);
}

SscanDtProj scan_dt_of(const QaMamba1Params& p, const Mamba1Buffers& b) {
    const QaLinearParams& w = p.dt_proj;
    const int64_t dbl = p.x_proj.n;
    return {static_cast<const int8_t*>(w.weight), b.x_dbl, p.seqlen * dbl, dbl, w.row_scale, w.col_scale, w.k, w.col_numel};
}

QaSScanParams scan_of(const QaMamba1Params& p, const Mamba1Buffers& b) {
    QaSScanParams s = scan_sizes(p);
    const int64_t dbl = p.x_proj.n, len = p.seqlen, d = p.d_inner;
    s.token_major = 1;
    s.u_batch_stride = len * d; s.u_l_stride = d; s.u_d_stride = 1;
    s.delta_batch_stride = len * d; s.delta_l_stride = d; s.delta_d_stride = 1;
    s.z_batch_stride = len * 2 * d; s.z_l_stride = 2 * d; s.z_d_stride = 1;
    s.B_batch_stride = s.C_batch_stride = len * dbl;
    s.B_l_stride = s.C_l_stride = dbl;
    s.B_dstate_stride = s.C_dstate_stride = 1;
    s.A_d_stride = p.d_state; s.A_dstate_stride = 1;
    s.out_batch_stride = len * d; s.out_l_stride = d; s.out_d_stride = 1;
    s.u = b.x; s.delta = b.dt; s.A_log = p.A_log; s.B = b.x_dbl + p.dt_rank; s.C = s.B + p.d_state;
    s.D = p.D; s.delta_bias = p.dt_bias; s.z = b.xz + d;
    s.scale_u = p.u_scale; s.scale_delta = p.dt_scale; s.scale_A = p.A_scale; s.scale_B = p.B_scale; s.scale_C = p.C_scale;
    s.scale_D = p.D_scale; s.scale_delta_bias = p.dt_bias_scale; s.scale_z = p.z_scale; s.scale_ssm_state = p.ssm_state_scale;
    s.out = b.y;
    if (p.state_is_fp32) s.last_state_f32 = static_cast<float*>(p.ssm_state);
    else s.last_state_i8 = static_cast<int8_t*>(p.ssm_state);
    s.workspace = b.scan.p; s.workspace_bytes = b.scan.bytes;
    return s;
}

QaSsmUpdateParams update_of(const QaMamba1Params& p, const Mamba1Buffers& b) {
    QaSsmUpdateParams u = {};
    const int64_t d = p.d_inner;
    u.batch = p.batch; u.nheads = 1; u.dim = p.d_inner; u.dstate = p.d_state; u.ngroups = 1;
    u.dt_softplus = p.delta_softplus;
    u.state_is_fp32 = p.state_is_fp32;
    u.state_batch_stride = d * p.d_state; u.state_head_stride = u.state_batch_stride;
    u.state_dim_stride = p.d_state; u.state_dstate_stride = 1;
    u.x_batch_stride = u.x_head_stride = d; u.x_dim_stride = 1;
    u.dt_batch_stride = u.dt_head_stride = d; u.dt_dim_stride = 1;
    u.dt_bias_head_stride = d; u.dt_bias_dim_stride = 1;
    u.A_head_stride = u.state_batch_stride; u.A_dim_stride = p.d_state; u.A_dstate_stride = 1;
    u.B_batch_stride = u.B_group_stride = p.x_proj.n; u.B_dstate_stride = 1;
    u.C_batch_stride = u.C_group_stride = p.x_proj.n; u.C_dstate_stride = 1;
    u.D_head_stride = d; u.D_dim_stride = 1;
    u.z_batch_stride = u.z_head_stride = 2 * d; u.z_dim_stride = 1;
    u.out_batch_stride = u.out_head_stride = d; u.out_dim_stride = 1;
    u.state = p.ssm_state; u.x = b.x; u.dt = b.dt; u.dt_bias = p.dt_bias; u.A_log = p.A_log;
    u.B = b.x_dbl + p.dt_rank; u.C = u.B + p.d_state; u.D = p.D; u.z = b.xz + d;
    u.x_scale = p.u_scale; u.dt_scale = p.dt_scale; u.dt_bias_scale = p.dt_bias_scale; u.A_log_scale = p.A_scale;
    u.state_scale = p.ssm_state_scale; u.B_scale = p.B_scale; u.C_scale = p.C_scale; u.D_scale = p.D_scale; u.z_scale = p.z_scale;
    u.out = b.y;
    return u;
}

// b: the workspace's sections
int ready(const QaMamba1Params* p, bool step, Mamba1Buffers& b) {
    QA_TRY(validate(p));
    if (!p->hidden || !p->out || !p->workspace || !p->conv_weight || !p->A_log) return QA_ERR_NULL;
    if (step && (!p->conv_state || !p->ssm_state)) return QA_ERR_NULL;
    if (step && p->seqlen != 1) return QA_ERR_SHAPE;
    b = carve(*p, p->workspace, step);
    if (p->workspace_bytes < b.total || (reinterpret_cast<uintptr_t>(p->workspace) & 255u) || !aligned16(p->hidden)) return QA_ERR_STRIDE;
    if (step) return ssm_update_check(update_of(*p, b));
    const SscanDtProj dt = scan_dt_of(*p, b);
    return sscan_token_major_check(scan_of(*p, b), dt_in_scan(*p) ? &dt : nullptr);
}

// ---------------------------------------------------------------------------------------------
// Mamba2
// ---------------------------------------------------------------------------------------------
struct Mamba2Buffers {
    int8_t *zxbcdt, *x, *B, *C, *yq;
    __half *y, *yn;
    Scratch w8, ssd;
    int64_t total;
};

int heads_of(const QaMamba2Params& p) { return p.d_inner / p.headdim; }

bool norm_fuses(const QaMamba2Params& p) { return norm_hadamard_fuses(p.d_inner, p.norm_group_size); }

QaSsdParams ssd_sizes(const QaMamba2Params& p) {
    QaSsdParams s = {};
    s.batch = p.batch; s.seqlen = p.seqlen; s.nheads = heads_of(p); s.headdim = p.headdim; s.dstate = p.d_state;
    s.ngroups = p.ngroups; s.chunk_size = p.chunk_size;
    return s;
}

Mamba2Buffers carve(const QaMamba2Params& p, void* base, bool step) {
    const int64_t t = static_cast<int64_t>(p.batch) * p.seqlen, bc = static_cast<int64_t>(p.ngroups) * p.d_state;
    Carver c{static_cast<uint8_t*>(base)};
    Mamba2Buffers b;
    b.zxbcdt = c.take<int8_t>(t * p.in_proj.n);
    b.x = c.take<int8_t>(t * p.d_inner);
    b.B = c.take<int8_t>(t * bc);
    b.C = c.take<int8_t>(t * bc);
    b.yq = c.take<int8_t>(t * p.d_inner);
    b.y = c.take<__half>(t * p.d_inner * 2);
    b.yn = c.take<__half>(norm_fuses(p) ? 0 : t * p.d_inner * 2);
    b.w8.bytes = std::max(expanded_bytes(p.in_proj, t), expanded_bytes(p.out_proj, t));
    b.w8.p = c.take<uint8_t>(b.w8.bytes);
    b.ssd.bytes = step ? 0 : ssd_workspace_layout(ssd_sizes(p)).total + ssd_workspace_layout(ssd_sizes(p)).sums_bytes;
    b.ssd.p = c.take<uint8_t>(b.ssd.bytes);
    b.total = c.off;
    return b;
}

int validate(const QaMamba2Params* p, bool step) {
    if (!p) return QA_ERR_NULL;
    if (p->batch < 1 || p->seqlen < 1 || p->batch > 65535 || p->seqlen > kConvSteps || static_cast<int64_t>(p->batch) * p->seqlen > 0x7fffffff) return QA_ERR_SHAPE;
    if (p->d_inner < 16 || p->headdim < 1 || p->d_inner % p->headdim != 0 || p->ngroups < 1 || heads_of(*p) % p->ngroups != 0) return QA_ERR_SHAPE;
    if (p->d_conv < 2 || p->d_conv > 4 || p->d_inner % 16 != 0 || p->d_state < 1 || (p->ngroups * p->d_state) % 4 != 0) return QA_ERR_UNSUPPORTED;
    // the limits of the scan (qa_ssd_chunk_scan_fwd) and of the state update
    if (step ? p->d_state > 256 || heads_of(*p) > 65535 : p->headdim > 256 || p->d_state > 1024 || p->chunk_size < 1 || p->chunk_size > 1024) return QA_ERR_UNSUPPORTED;
    const int64_t used = 2LL * p->d_inner + 2LL * p->ngroups * p->d_state + heads_of(*p);
    if (p->in_proj.k != p->d_model || p->in_proj.n < used || p->in_proj.n % 8 != 0 || p->out_proj.k != p->d_inner) return QA_ERR_SHAPE;
    if (p->conv_state_len != p->d_conv && p->conv_state_len != p->d_conv - 1) return QA_ERR_SHAPE;
    if (p->norm_group_size < 1 || p->d_inner % p->norm_group_size != 0) return QA_ERR_SHAPE;
    if (p->norm_group_size % 8 != 0 || p->norm_group_size > kNormGroup) return QA_ERR_UNSUPPORTED;
    const int64_t t = static_cast<int64_t>(p->batch) * p->seqlen;
    QA_TRY(linear_check(p->in_proj, t, p->d_model));
    QA_TRY(linear_check(p->out_proj, t, p->d_inner));
    return hadamard_check(p->d_inner);
}

QaConv2Params conv2_of(const QaMamba2Params& p, const Mamba2Buffers& b) {
    QaConv2Params c = {};
    const int64_t bc = static_cast<int64_t>(p.ngroups) * p.d_state, len = p.seqlen;
    c.batch = p.batch; c.dim = static_cast<int>(p.d_inner + 2 * bc); c.seqlen = p.seqlen; c.width = p.d_conv;
    c.silu_activation = 1;
    c.x_dim = p.d_inner; c.x_headdim = p.headdim; c.d_state = p.d_state; c.n_groups = p.ngroups;
    c.nhead_groups = p.conv_nhead_groups; c.ndim_groups = p.conv_ndim_groups;
    c.conv_state_len = p.conv_state_len;
    c.xBC_batch_stride = len * p.in_proj.n; c.xBC_l_stride = p.in_proj.n; c.xBC_c_stride = 1;
    c.x_batch_stride = len * p.d_inner; c.x_l_stride = p.d_inner; c.x_c_stride = 1;
    c.B_batch_stride = len * bc; c.B_l_stride = bc; c.B_c_stride = 1;
    c.C_batch_stride = len * bc; c.C_l_stride = bc; c.C_c_stride = 1;
    c.weight_c_stride = p.d_conv; c.weight_width_stride = 1;
    c.conv_state_batch_stride = p.conv_state_batch_stride; c.conv_state_c_stride = p.conv_state_c_stride; c.conv_state_l_stride = p.conv_state_l_stride;
    c.xBC = b.zxbcdt + p.d_inner; c.weight = p.conv_weight; c.bias = p.conv_bias;
    c.x = b.x; c.B = b.B; c.C = b.C; c.conv_state = p.conv_state;
    c.x_out_scales = p.x_out_scales; c.B_out_scales = p.B_out_scales; c.C_out_scales = p.C_out_scales;
    c.x_head_group_range = p.conv_head_range; c.x_dim_group_range = p.conv_dim_range;
    c.scale_x = p.scale_x; c.scale_B = p.scale_B; c.scale_C = p.scale_C;
    c.scale_wx = p.scale_wx; c.scale_wB = p.scale_wB; c.scale_wC = p.scale_wC;
    c.scale_bx = p.scale_bx; c.scale_bB = p.scale_bB; c.scale_bC = p.scale_bC;
    return c;
}

QaSsdParams ssd_of(const QaMamba2Params& p, const Mamba2Buffers& b) {
    QaSsdParams s = ssd_sizes(p);
    s.dt_softplus = p.delta_softplus;
    s.D_has_hdim = p.D_has_hdim;
    s.nhead_groups = p.nhead_groups; s.ndim_groups = p.ndim_groups;
    s.final_state_is_fp32 = p.state_is_fp32;
    s.dt_row_stride = p.in_proj.n;
    s.dt_min = p.dt_min; s.dt_max = p.dt_max;
    s.x = b.x; s.B = b.B; s.C = b.C;
    s.dt = b.zxbcdt + 2 * p.d_inner + 2 * p.ngroups * p.d_state;
    s.A_log = p.A_log; s.D = p.D; s.dt_bias = p.dt_bias;
    s.x_scale = p.x_scales; s.dt_scale = p.dt_scale; s.A_log_scale = p.A_log_scale; s.B_scale = p.B_scale; s.C_scale = p.C_scale;
    s.D_scale = p.D_scale; s.state_scale = p.ssm_state_scale;
    s.x_head_group_range = p.head_range; s.x_dim_group_range = p.dim_range;
    s.out = b.y; s.final_states = p.ssm_state;
    s.workspace = b.ssd.p; s.workspace_bytes = b.ssd.bytes;
    return s;
}

QaSsmUpdateParams update_of(const QaMamba2Params& p, const Mamba2Buffers& b) {
    QaSsmUpdateParams u = {};
    const int heads = heads_of(p);
    const int64_t bc = static_cast<int64_t>(p.ngroups) * p.d_state;
    u.batch = p.batch; u.nheads = heads; u.dim = p.headdim; u.dstate = p.d_state; u.ngroups = p.ngroups;
    u.dt_softplus = p.delta_softplus;
    u.state_is_fp32 = p.state_is_fp32;
    u.dt_bias_is_fp16 = 1;
    u.nhead_groups = p.nhead_groups; u.ndim_groups = p.ndim_groups;
    u.state_dstate_stride = 1; u.state_dim_stride = p.d_state;
    u.state_head_stride = static_cast<int64_t>(p.headdim) * p.d_state; u.state_batch_stride = u.state_head_stride * heads;
    u.x_batch_stride = p.d_inner; u.x_head_stride = p.headdim; u.x_dim_stride = 1;
    u.dt_batch_stride = p.in_proj.n; u.dt_head_stride = 1;
    u.dt_bias_head_stride = 1;
    u.A_head_stride = 1;
    u.B_batch_stride = u.C_batch_stride = bc; u.B_group_stride = u.C_group_stride = p.d_state; u.B_dstate_stride = u.C_dstate_stride = 1;
    u.D_head_stride = p.D_has_hdim ? p.headdim : 1; u.D_dim_stride = p.D_has_hdim ? 1 : 0;
    u.out_batch_stride = p.d_inner; u.out_head_stride = p.headdim; u.out_dim_stride = 1;
    u.state = p.ssm_state; u.x = b.x; u.dt = b.zxbcdt + 2 * p.d_inner + 2 * bc; u.dt_bias = p.dt_bias; u.A_log = p.A_log;
    u.B = b.B; u.C = b.C; u.D = p.D;
    u.x_scale = p.x_scales; u.dt_scale = p.dt_scale; u.A_log_scale = p.A_log_scale; u.state_scale = p.ssm_state_scale;
    u.B_scale = p.B_scale; u.C_scale = p.C_scale; u.D_scale = p.D_scale;
    u.x_head_group_range = p.head_range; u.x_dim_group_range = p.dim_range;
    u.out = b.y;
    return u;
}

int ready(const QaMamba2Params* p, bool step, Mamba2Buffers& b) {
    QA_TRY(validate(p, step));
    if (!p->hidden || !p->out || !p->workspace || !p->conv_weight || !p->A_log || !p->norm_weight) return QA_ERR_NULL;
    if (!p->x_out_scales || !p->B_out_scales || !p->C_out_scales) return QA_ERR_NULL;
    if ((p->conv_head_range == nullptr) != (p->conv_dim_range == nullptr)) return QA_ERR_NULL;
    if (p->conv_head_range && (p->conv_nhead_groups < 1 || p->conv_ndim_groups < 1)) return QA_ERR_SHAPE;
    if (step && (!p->conv_state || !p->ssm_state)) return QA_ERR_NULL;
    if (step && p->seqlen != 1) return QA_ERR_SHAPE;
    b = carve(*p, p->workspace, step);
    if (p->workspace_bytes < b.total || (reinterpret_cast<uintptr_t>(p->workspace) & 255u) || !aligned16(p->hidden) || !aligned16(p->norm_weight)) return QA_ERR_STRIDE;
    return step ? ssm_update_check(update_of(*p, b)) : ssd_check(ssd_of(*p, b));
}

// gated norm, Hadamard rotation and quantisation, out_proj
int mamba2_tail(const QaMamba2Params& p, const Mamba2Buffers& b, void* stream) {
    const int rows = p.batch * p.seqlen;
    QaNormGatedParams n = {};
    n.rows = rows; n.dim = p.d_inner; n.group_size = p.norm_group_size;
    n.norm_before_gate = p.norm_before_gate; n.out_mode = 0;
    n.eps = p.norm_eps; n.z_scale = p.norm_z_scale;
    n.x_row_stride = p.d_inner; n.z_row_stride = p.in_proj.n; n.out_row_stride = p.d_inner;
    n.x = b.y; n.weight = p.norm_weight; n.qz = b.zxbcdt; n.out = b.yn;
    if (norm_fuses(p)) {
        QaHadamardParams h = {};
        h.rows = rows; h.dim = p.d_inner; h.scale = p.had_scale; h.out_row_stride = p.d_inner; h.out = b.yq;
        QA_TRY(norm_hadamard_quant(&n, &h, true, stream));
    } else {
        QA_TRY(qa_rmsnorm_gated(&n, stream));
        QA_TRY(hadamard(b.yn, b.yq, rows, p.d_inner, p.had_scale, stream));
    }
    return project(p.out_proj, b.yq, p.d_inner, rows, p.out, QA_OUT_F16, false, b.w8, stream);
}

}  // namespace
}  // namespace qa

extern "C" int64_t qa_mamba1_workspace_bytes(const QaMamba1Params* p, int step) {
    using namespace qa;
    return validate(p) == QA_OK ? carve(*p, nullptr, step != 0).total : 0;
}

extern "C" int qa_mamba1_forward(const QaMamba1Params* p, void* stream) {
    using namespace qa;
    Mamba1Buffers b;
    QA_TRY(ready(p, false, b));
    const int rows = p->batch * p->seqlen, d = p->d_inner;
    QA_TRY(project(p->in_proj, p->hidden, p->d_model, rows, b.xz, QA_OUT_I8, true, b.w8, stream));

    QA_TRY(conv_channel_last_fwd(conv_of(*p, b), static_cast<hipStream_t>(stream)));

    QA_TRY(project(p->x_proj, b.x, d, rows, b.x_dbl, QA_OUT_I8, false, b.w8, stream));
    const bool fused_dt = dt_in_scan(*p);
    if (!fused_dt) QA_TRY(project(p->dt_proj, b.x_dbl, p->x_proj.n, rows, b.dt, QA_OUT_I8, true, b.w8, stream));
    const SscanDtProj dt = scan_dt_of(*p, b);
    QA_TRY(sscan_token_major_fwd(scan_of(*p, b), fused_dt ? &dt : nullptr, static_cast<hipStream_t>(stream)));

    QA_TRY(hadamard(b.y, b.yq, rows, d, p->had_scale, stream));
    return project(p->out_proj, b.yq, d, rows, p->out, QA_OUT_F16, false, b.w8, stream);
}

extern "C" int qa_mamba1_step(const QaMamba1Params* p, void* stream) {
    using namespace qa;
    Mamba1Buffers b;
    QA_TRY(ready(p, true, b));
    const int rows = p->batch, d = p->d_inner;
    const int fused = project_conv(p->in_proj, p->hidden, p->d_model, rows, b.xz, 0, conv_of(*p, b), stream);
    if (fused == QA_ERR_UNSUPPORTED) {
        QA_TRY(project(p->in_proj, p->hidden, p->d_model, rows, b.xz, QA_OUT_I8, false, b.w8, stream));
        QA_TRY(conv_single_update(conv_of(*p, b), static_cast<hipStream_t>(stream)));
    } else if (fused != QA_OK) {
        return fused;
    }

    QA_TRY(project(p->x_proj, b.x, d, rows, b.x_dbl, QA_OUT_I8, false, b.w8, stream));

    const QaSsmUpdateParams u = update_of(*p, b);
    const QaLinearParams& dt = p->dt_proj;
    int st = QA_ERR_UNSUPPORTED;
    if (dt.bits == 8 && !(rows == 1 && dt.row_rule == QA_ROW_HALF_AWAY)) {                // (codes rounded half to even)
        const SsmDtProj proj = {static_cast<const int8_t*>(dt.weight), b.x_dbl, p->x_proj.n, dt.row_scale, dt.col_scale, dt.k / 16, dt.col_numel,
                                rows == 1 && dt.row_rule == QA_ROW_ALPHA, dt.alpha};
        st = mamba1_step(u, proj, static_cast<hipStream_t>(stream));
    }
    if (st == QA_ERR_UNSUPPORTED) {
        QA_TRY(project(dt, b.x_dbl, p->x_proj.n, rows, b.dt, QA_OUT_I8, false, b.w8, stream));
        st = qa_ssm_state_update(&u, stream);
    }
    QA_TRY(st);

    if (rows == 1) {
        const GemvRotate r = {b.y, p->had_scale};
        st = project_rotated(p->out_proj, r, p->out, stream);
        if (st != QA_ERR_UNSUPPORTED) return st;
    }
    QA_TRY(hadamard(b.y, b.yq, rows, d, p->had_scale, stream));
    return project(p->out_proj, b.yq, d, rows, p->out, QA_OUT_F16, false, b.w8, stream);
}

extern "C" int64_t qa_mamba2_workspace_bytes(const QaMamba2Params* p, int step) {
    using namespace qa;
    return validate(p, step != 0) == QA_OK ? carve(*p, nullptr, step != 0).total : 0;
}

extern "C" int qa_mamba2_forward(const QaMamba2Params* p, void* stream) {
    using namespace qa;
    Mamba2Buffers b;
    QA_TRY(ready(p, false, b));
    const int rows = p->batch * p->seqlen;
    QA_TRY(project(p->in_proj, p->hidden, p->d_model, rows, b.zxbcdt, QA_OUT_I8, false, b.w8, stream));
    QA_TRY(conv_channel_last_fwd(conv2_of(*p, b), static_cast<hipStream_t>(stream)));
    const QaSsdParams s = ssd_of(*p, b);
    QA_TRY(qa_ssd_chunk_scan_fwd(&s, stream));
    return mamba2_tail(*p, b, stream);
}

extern "C" int qa_mamba2_step(const QaMamba2Params* p, void* stream) {
    using namespace qa;
    Mamba2Buffers b;
    QA_TRY(ready(p, true, b));
    const int rows = p->batch;
    const QaConv2Params c = conv2_of(*p, b);
    const int fused = project_conv(p->in_proj, p->hidden, p->d_model, rows, b.zxbcdt, p->d_inner, c, stream);
    if (fused == QA_ERR_UNSUPPORTED) {
        QA_TRY(project(p->in_proj, p->hidden, p->d_model, rows, b.zxbcdt, QA_OUT_I8, false, b.w8, stream));
        QA_TRY(qa_quamba2_conv1d_update(&c, stream));
    } else if (fused != QA_OK) {
        return fused;
    }
    const QaSsmUpdateParams u = update_of(*p, b);
    QA_TRY(qa_ssm_state_update(&u, stream));
    return mamba2_tail(*p, b, stream);
}
