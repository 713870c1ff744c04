// Up to four activation rows against a weight matrix: a stream over the weights.
//
// A wave owns four rows of the weight and the whole of K: a lane takes 16 bytes of each row out of every 1024 (int8: 16
// codes; 4 bits: 32 codes), so a load of the wave is 1 KB in one piece, and the loads of up to four such pieces of all
// four rows go out before the first is used; a piece is multiplied as it arrives.  The matrix cores have nothing to give
// here - a tile of 16 activation rows would be three quarters or more empty - and their fragments would have to pass through
// LDS; the products are 4-way int8 dot products in the lane that loaded the codes, and LDS is not used at all.  The lanes'
// partial sums meet through lane swaps (two stages, four values at a time) and row permutes.
//
// Bound by the memory round trips of a short kernel, not by bandwidth: 1 x 10240 x 2560 with 4-bit weights (13 MB)
// 10.2 us as a 32-column matrix-core tile per workgroup.
//
// With a conv behind the product (GemvConv) the wave that holds a conv channel's new input also makes its conv step: the
// operands of that step are requested with the weights, and a launch and a round trip through memory are saved.
#include "conv2_common.hpp"
#include "gemm_core.hpp"
#include "gemv.hpp"
#include "hadamard_core.hpp"
#include "w4_expand.hpp"

namespace qa {
namespace {

using gemm::v4u;
using gemm::quant8;
using gemm::one_f16_or_bf16;

constexpr int kRows = 4;               // weight rows per wave

// a, b: one value per lane each -> the lower half of the wave holds the sums of a over lane pairs (l, l + 32), the upper
// half those of b
__device__ __forceinline__ int fold32(int a, int b) {
    const auto r = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(a), static_cast<unsigned>(b), false, false);
    return static_cast<int>(r[0]) + static_cast<int>(r[1]);
}
// the same for the even and odd rows of sixteen lanes
__device__ __forceinline__ int fold16(int a, int b) {
    const auto r = __builtin_amdgcn_permlane16_swap(static_cast<unsigned>(a), static_cast<unsigned>(b), false, false);
    return static_cast<int>(r[0]) + static_cast<int>(r[1]);
}
// sum over a row of sixteen lanes, in every lane of it
__device__ __forceinline__ int row_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, true);       // lane ^ 1
    v += __builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, true);       // lane ^ 2
    v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true);      // mirrored in half a row
    v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true);      // mirrored in the row
    return v;
}

// The conv behind a product: one output scale and a state of a word per channel (Mamba1's layer), output scales from tables and such
// a state, or anything.  A word may stand anywhere on four bytes: read code by code (channels 4 and 8 bytes apart, one row, us) int8
// 10240 x 2560 5.8 -> 6.25, 4 bits 6.1 -> 6.7, with tables int8 10576 x 2560 6.3 -> 6.5, 4 bits two rows 6320 x 1536 4.6 -> 4.9.
enum ConvKind { kNoConv, kConvOneScale, kConvTablesWords, kConvTables };
constexpr bool words_held(ConvKind c) { return c == kConvOneScale || c == kConvTablesWords; }

// What a conv step takes of the conv's operands, requested behind the weights by every wave in one straight run: a branch
// around loads leaves the compiler unsure how many are in flight, and it waits for all of them, the weights among them, where the
// ways meet.  (Waves without conv channels read the operands of some that are.)
//
// The output scale of four channels, neighbours in one part and one head (out_scale_of in conv2_common.hpp): every lane requests its
// share of the tables of the channels' group at once, and the search in them is a few ballots when the sums are there.  As three scalar
// loads one after the other, each the index of the next, it held up the products of the weights that came first (in a layer, one row, us:
// int8 10448 x 2560 8.2 -> 6.5, 3352 x 768 4.6 -> 4.1; 4 bits 18560 x 4096 13.5 -> 12.9, 6280 x 1536 5.7 -> 5.0; two rows 10448 x 2560
// 9.7 -> 8.6).
struct ConvOperands {
    uint32_t taps, held;   // the last three codes of the lane's channel, the oldest in byte 0
    uint8_t codes[3];      // the same as they are loaded where the state is no word
    int8_t bias;
    float scale;           // in_table: of head group lane / 8, dim group lane % 8; else of the lane's own channel
    int head_end, dim_end; // in_table: where head group `lane` ends, and that dim group
    bool in_table;
};
// ch: the wave's first channel; mine: the lane's; st: the state of that
template <ConvKind CONV>
__device__ __forceinline__ ConvOperands request_conv(const QaConv2Params& p, const Part& part, int ch, int mine, const int8_t* st, int lane) {
    ConvOperands r;
    r.taps = *reinterpret_cast<const uint32_t*>(p.weight + mine * 4);
    r.bias = *(p.bias ? p.bias + mine : p.weight);
    if constexpr (words_held(CONV)) {
        r.held = *reinterpret_cast<const uint32_t*>(st);
    } else {
        const int drop = p.conv_state_len - 3;
#pragma unroll
        for (int i = 0; i < 3; ++i) r.codes[i] = static_cast<uint8_t>(st[(drop + i) * p.conv_state_l_stride]);
    }
    if constexpr (CONV == kConvOneScale) return r;
    const bool grouped = p.x_out_scales && p.x_head_group_range != nullptr && p.x_dim_group_range != nullptr;
    r.in_table = grouped && part.index == 0;
    int g = 0, own = 0;
    if (r.in_table && p.n_groups > 1) g = ch / (p.x_dim / p.n_groups);
    if (grouped && part.index != 0) own = (mine - part.offset) / p.d_state;
    const int row = r.in_table ? (g * p.nhead_groups + min(lane >> 3, p.nhead_groups - 1)) * p.ndim_groups + min(lane & 7, p.ndim_groups - 1) : own;
    const float* const any = reinterpret_cast<const float*>(p.weight);         // (something to read)
    const float* scales = part.index == 0 ? p.x_out_scales : part.index == 1 ? p.B_out_scales : p.C_out_scales;
    r.scale = (p.x_out_scales ? scales : any)[row];
    r.head_end = (r.in_table ? p.x_head_group_range : reinterpret_cast<const int32_t*>(any))[r.in_table ? g * p.nhead_groups + min(lane, p.nhead_groups - 1) : 0];
    r.dim_end = (r.in_table ? p.x_dim_group_range : reinterpret_cast<const int32_t*>(any))[r.in_table ? row : 0];
    return r;
}
// the output scale of channel ch + which, ch the wave's first (all lanes of the wave active)
__device__ __forceinline__ float found_out_scale(const QaConv2Params& p, const ConvOperands& r, int ch, int which, int lane) {
    static_assert(kGemvConvGroups == 8, "eight lanes a head group");
    if (!p.x_out_scales) return p.x_out_scale;
    if (!r.in_table) return r.scale;
    const int head = ch % (p.x_dim / p.n_groups) / p.x_headdim, d = ch % p.x_headdim;
    const int hg = __popcll(__builtin_amdgcn_ballot_w64(lane < p.nhead_groups - 1 && head >= r.head_end));
    float found = 0.0f;
#pragma unroll
    for (int e = 0; e < kRows; ++e) {
        const uint64_t beyond = __builtin_amdgcn_ballot_w64((lane & 7) < p.ndim_groups - 1 && d + e >= r.dim_end);
        const int at = 8 * hg + __popcll((beyond >> (8 * hg)) & 0xff);
        const float s = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(r.scale), at));
        found = which == e ? s : found;
    }
    return found;
}

// BATCH: pieces of K (1 KB of each weight row) whose loads are in flight together.  KS: waves of the workgroup that share
// four rows, a contiguous part of K each.
template <int BITS, int M, int KS, int BATCH, int OUT, ConvKind CONV, class Conv>
__device__ __forceinline__ void gemv_body(const GemvArgs& p, const Conv& f) {
    constexpr int V = kRows * M, PER = V / 4;                    // values of the wave, and per lane after two folds
    constexpr int kLaneCodes = BITS == 8 ? 16 : 32, kPieceCodes = 64 * kLaneCodes, AQ = kLaneCodes / 16;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)), part_k = wave % KS;
    int n0 = (blockIdx.x * (static_cast<int>(blockDim.x) / (64 * KS)) + wave / KS) * kRows;
    if (KS == 1 && n0 >= p.n) return;
    if constexpr (CONV != kNoConv) {
        // the conv's columns go first: their waves have a step more to make when the sums are there
        const int last = (p.n + kRows - 1) / kRows * kRows;
        if (n0 < last) n0 += n0 + f.ch0 < last ? f.ch0 : f.ch0 - last;
    }
    // this wave's part of K
    const int share = (p.k / kLaneCodes + KS - 1) / KS * kLaneCodes;
    const int k_first = part_k * share, k_end = min(k_first + share, p.k);

    const uint8_t* w_row[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) w_row[r] = static_cast<const uint8_t*>(p.w) + static_cast<int64_t>(min(n0 + r, p.n - 1)) * p.ldw;
    const int pieces = (k_end - k_first + kPieceCodes - 1) / kPieceCodes;
    v4u fw[BATCH][kRows], fa[BATCH][M][AQ];
    uint2 fs[BATCH];
    auto load = [&](int c, int b) __attribute__((always_inline)) {
        // (lanes past the end read the row's start; their activations are zeroed below)
        const int k0 = k_first + c * kPieceCodes + lane * kLaneCodes, kk = k0 < k_end ? k0 : 0;
#pragma unroll
        for (int r = 0; r < kRows; ++r) fw[b][r] = *reinterpret_cast<const v4u*>(w_row[r] + kk * BITS / 8);
        if constexpr (BITS == 4) fs[b] = *reinterpret_cast<const uint2*>(p.s_group + static_cast<int64_t>(kk / 128) * p.n + min(n0, p.n - 4));
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int8_t* a = p.a + min(m, p.m - 1) * p.lda + kk;
#pragma unroll
            for (int q = 0; q < AQ; ++q) fa[b][m][q] = *reinterpret_cast<const v4u*>(a + 16 * q);
        }
    };
    int acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = 0;
    auto multiply = [&](int c, int b) __attribute__((always_inline)) {
        const bool in = k_first + c * kPieceCodes + lane * kLaneCodes < k_end;
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int q = 0; q < AQ; ++q) fa[b][m][q] = in ? fa[b][m][q] : v4u{0u, 0u, 0u, 0u};
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            if constexpr (BITS == 8) {
#pragma unroll
                for (int m = 0; m < M; ++m)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        acc[m * kRows + r] = __builtin_amdgcn_sdot4(static_cast<int>(fw[b][r][q]), static_cast<int>(fa[b][m][0][q]), acc[m * kRows + r], false);
            } else {
                const uint32_t pair = r & 2 ? fs[b].y : fs[b].x;
                const uint32_t one = r & 1 ? pair >> 16 : pair & 0xffffu;
                const __half2 s2 = bits_h2(one | (one << 16));
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint2 e = expand_grouped(fw[b][r][q], s2);
#pragma unroll
                    for (int m = 0; m < M; ++m) {
                        int& s = acc[m * kRows + r];
                        s = __builtin_amdgcn_sdot4(static_cast<int>(e.x), static_cast<int>(fa[b][m][q / 2][2 * (q & 1)]), s, false);
                        s = __builtin_amdgcn_sdot4(static_cast<int>(e.y), static_cast<int>(fa[b][m][q / 2][2 * (q & 1) + 1]), s, false);
                    }
                }
            }
        }
    };

    // the value this lane finishes: row `lane / 16` of four, `lane % 16` < PER
    const int quarter = lane >> 4, slot = lane & 15;
    const int value = (quarter >> 1) * (V / 2) + (quarter & 1) * PER + min(slot, PER - 1);
    const int my_m = min(value / kRows, p.m - 1), my_n = min(n0 + value % kRows, p.n - 1);
    const bool mine = slot < PER && value / kRows < p.m && n0 + value % kRows < p.n;
    float s_row = 0.0f, s_col = 0.0f;
    // (the four columns of a wave are all conv channels, of one part and one head, or none is)
    bool conv_col = false;
    int ch0 = 0, ch = 0;                                         // the wave's first channel, the lane's
    Part part = {};
    ConvOperands conv;
    int8_t* st = nullptr;
    // the scales and the conv's operands, behind the weights
    auto request_rest = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        const float* const any = reinterpret_cast<const float*>(p.a);          // (the rule without scales reads something)
        s_row = p.rule == kGemvAlpha ? p.alpha : p.row_scale[p.one_row_scale ? 0 : my_m];
        s_col = p.rule == kGemvAlpha ? *any : p.col_scale[p.one_col_scale ? 0 : my_n];
        if constexpr (CONV != kNoConv) {
            const QaConv2Params& c = f.conv;
            conv_col = n0 >= f.ch0 && n0 < f.ch0 + c.dim;
            ch0 = conv_col ? n0 - f.ch0 : 0;
            ch = conv_col ? my_n - f.ch0 : value % kRows;
            part = part_of(c, ch0);
            st = c.conv_state + my_m * c.conv_state_batch_stride + ch * c.conv_state_c_stride;
            conv = request_conv<CONV>(c, part, ch0, ch, st, lane);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // all loads of a batch, then its products in their order: one straight run for each number of pieces
    auto batch = [&](auto p_c, int c0, bool first) __attribute__((always_inline)) {
        constexpr int P = decltype(p_c)::value;
#pragma unroll
        for (int b = 0; b < P; ++b) load(c0 + b, b);
        if (first) request_rest();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < P; ++b) multiply(c0 + b, b);
    };
    bool done = false;
    static_for<1, BATCH>([&](auto p_c) {
        if (!done && pieces == decltype(p_c)::value) {
            batch(p_c, 0, true);
            done = true;
        }
    });
    if (!done) {
        batch(std::integral_constant<int, BATCH>{}, 0, true);
        // (pieces past the last one are lanes past the end)
        for (int c0 = BATCH; c0 < pieces; c0 += BATCH) batch(std::integral_constant<int, BATCH>{}, c0, false);
    }

    int half[V / 2], sum = 0;
#pragma unroll
    for (int v = 0; v < V / 2; ++v) half[v] = fold32(acc[v], acc[v + V / 2]);
#pragma unroll
    for (int v = 0; v < PER; ++v) {
        const int s = row_sum(fold16(half[v], half[v + PER]));
        sum = slot == v ? s : sum;
    }
    if constexpr (KS > 1) {
        __shared__ int parts[4][64];
        if (part_k) parts[wave][lane] = sum;
        __syncthreads();
        if (part_k) return;
#pragma unroll
        for (int i = 1; i < KS; ++i) sum += parts[wave + i][lane];
    }
    float c_out_scale = 1.0f;
    if constexpr (CONV == kConvOneScale) c_out_scale = f.conv.x_out_scale;
    else if constexpr (CONV != kNoConv) if (conv_col) c_out_scale = found_out_scale(f.conv, conv, ch0, value % kRows, lane);
    if (!mine) return;
    const float accf = static_cast<float>(sum);
    float y = p.rule == kGemvHalfAway ? (s_col * s_row) * accf : p.rule == kGemvColOuter ? s_col * (s_row * accf)
            : p.rule == kGemvAlpha ? s_row * accf : s_row * (s_col * accf);
    asm volatile("" : "+v"(y));                                  // the fp32 product is rounded on its own
    if constexpr (OUT == QA_OUT_I8) {
        const int8_t q = static_cast<int8_t>(quant8(y, p.half_away ? QA_ROUND_HALF_AWAY : QA_ROUND_RNE));
        if constexpr (CONV != kNoConv) if (conv_col) {
            const QaConv2Params& c = f.conv;
            const uint32_t kept = words_held(CONV) ? conv.held >> 8 : conv.codes[0] | (conv.codes[1] << 8) | (conv.codes[2] << 16);
            const uint32_t win = kept | (static_cast<uint32_t>(static_cast<uint8_t>(q)) << 24);
            if constexpr (words_held(CONV)) {
                *reinterpret_cast<uint32_t*>(st) = win;
            } else {
                for (int i = 0; i < c.conv_state_len; ++i) st[i * c.conv_state_l_stride] = static_cast<int8_t>(win >> (8 * (i + 4 - c.conv_state_len)));
            }
            float v = c.bias ? part.s_bias * static_cast<float>(conv.bias) : 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v = __builtin_fmaf(part.s_in * static_cast<float>(static_cast<int8_t>(conv.taps >> (8 * i))), static_cast<float>(static_cast<int8_t>(win >> (8 * i))), v);
            int64_t ls, cs;
            const ConvQuantRegs kq(c_out_scale);
            out_ptr(c, part, my_m, ch, &ls, &cs)[0] = static_cast<int8_t>(conv_quant(v, c_out_scale, 1.0f / c_out_scale, c.silu_activation,
                                                                                     conv_needs_exact_route(c_out_scale), kq));
            return;
        }
        static_cast<int8_t*>(p.d)[my_m * p.ldd + my_n] = q;
    } else {
        static_cast<uint16_t*>(p.d)[my_m * p.ldd + my_n] = one_f16_or_bf16<OUT>(y);
    }
}

template <int BITS, int M, int KS, int BATCH, int OUT, bool CONV>
__global__ __launch_bounds__(256) void gemv_kernel(GemvArgs p, std::conditional_t<CONV, GemvConv, NoGemvConv> f) {
    gemv_body<BITS, M, KS, BATCH, OUT, CONV ? kConvOneScale : kNoConv>(p, f);
}
template <int BITS, int M, int KS, int BATCH>
__global__ __launch_bounds__(256) void gemv_conv_words_kernel(GemvArgs p, GemvConv f) {
    gemv_body<BITS, M, KS, BATCH, QA_OUT_I8, kConvTablesWords>(p, f);
}
template <int BITS, int M, int KS, int BATCH>
__global__ __launch_bounds__(256) void gemv_conv_tables_kernel(GemvArgs p, GemvConv f) {
    gemv_body<BITS, M, KS, BATCH, QA_OUT_I8, kConvTables>(p, f);
}

template <int BITS, int M, int KS, int BATCH>
int launch(const GemvParams& p, const GemvConv* conv, hipStream_t stream) {
    const int64_t groups = (static_cast<int64_t>(p.n) + kRows - 1) / kRows;
    const int per_block = KS > 1 || groups >= 1024 ? 4 : 1;      // waves; few waves: a workgroup each, spread over the part
    const dim3 grid(static_cast<unsigned>((groups * KS + per_block - 1) / per_block)), block(64 * per_block);
    const GemvArgs args(p);
    const NoGemvConv none = {};
    const bool words = conv && gemv_state_in_words(conv->conv);
    if (words && !conv->conv.x_out_scales) hipLaunchKernelGGL((gemv_kernel<BITS, M, KS, BATCH, QA_OUT_I8, true>), grid, block, 0, stream, args, *conv);
    else if (words) hipLaunchKernelGGL((gemv_conv_words_kernel<BITS, M, KS, BATCH>), grid, block, 0, stream, args, *conv);
    else if (conv) hipLaunchKernelGGL((gemv_conv_tables_kernel<BITS, M, KS, BATCH>), grid, block, 0, stream, args, *conv);
    else if (p.out_type == QA_OUT_I8) hipLaunchKernelGGL((gemv_kernel<BITS, M, KS, BATCH, QA_OUT_I8, false>), grid, block, 0, stream, args, none);
    else if (p.out_type == QA_OUT_F16) hipLaunchKernelGGL((gemv_kernel<BITS, M, KS, BATCH, QA_OUT_F16, false>), grid, block, 0, stream, args, none);
    else hipLaunchKernelGGL((gemv_kernel<BITS, M, KS, BATCH, QA_OUT_BF16, false>), grid, block, 0, stream, args, none);
    return check_launch();
}

// Waves per four rows.  A wave alone works through its rows' K at the pace of one wave's latencies, so K is split while the
// rows alone leave the SIMDs short of waves (measured, us for 1 / 2 / 4 waves at one activation row: 4 bits 2560 x 5120 5.9 /
// 5.8 / 4.9, 4096 x 8192 8.7 / 7.1 / 6.9, 10240 x 2560 7.4 / 6.5 / 9.1, 18560 x 4096 11.5 / 11.0 / 15.3; int8 192 x 5120
// 2.7 / 2.8 / 2.6, 10240 x 2560 7.0 / 6.5 / 6.9); past about 5000 waves more of them only repeat the prologue.
template <int BITS, int M, int B1, int B2, int B4>
int pick(const GemvParams& p, const GemvConv* conv, hipStream_t stream) {
    const int64_t groups = (static_cast<int64_t>(p.n) + kRows - 1) / kRows;
    if (groups <= 1024 && p.k >= 1536) return launch<BITS, M, 4, B4>(p, conv, stream);
    if (groups <= 2816 && p.k >= 2048) return launch<BITS, M, 2, B2>(p, conv, stream);
    return launch<BITS, M, 1, B1>(p, conv, stream);
}
// ---------------------------------------------------------------------------------------------
// One activation row that the kernel makes itself: the Hadamard transform and quantisation that as a launch of its own keeps
// one workgroup busy for 3 to 5 us while the weights wait.  Here every workgroup transforms the row in its own LDS, in the
// order of the stand-alone kernel and so to the same bits, with its share of the weights on the way.  Eight waves a workgroup
// and at most about one workgroup per CU, so that no CU transforms the row twice; KS waves share four weight rows.  A decode
// step of one sequence (one launch less to make and to wait for): d_inner 1536 21.0 -> 18.0 us, 3072 20.5 -> 17.3, 4096 21.9
// -> 19.7, 5120 25.7 -> 23.6; 8192 33.5 -> 34.0, so up to 5120 only.  The transform is most of the kernel: with the first three
// index bits in the registers the row arrives in and the outputs of a lane chosen for their common beginnings (s_point_quantised) the
// launch takes 2560 x 5120 with 4 bits 9.6 -> 8.9 us, int8 8.2 -> 7.3, 768 x 1536 4.8 -> 4.4.  (With the gated norm in front as well it was slower
// than the two kernels at every width.)
// ---------------------------------------------------------------------------------------------
constexpr int kRotThreads = 512, kRotWaves = kRotThreads / 64, kRotDim = 5120;

struct RotShape {
    int log_m, ks;
};

template <int BITS, int S>
__global__ __launch_bounds__(kRotThreads) void gemv_rotated_kernel(GemvArgs p, GemvRotate r, RotShape shape) {
    constexpr int kLaneCodes = BITS == 8 ? 16 : 32, kPieceCodes = 64 * kLaneCodes, AQ = kLaneCodes / 16, BATCH = BITS == 8 ? 4 : 2;
    extern __shared__ __attribute__((aligned(16))) float buf[];
    __shared__ int parts[kRotWaves][64];
    const int tid = threadIdx.x, lane = tid & 63, dim = p.k;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ks = shape.ks, part_k = wave % ks;
    const int n0 = (blockIdx.x * (kRotWaves / ks) + wave / ks) * kRows;
    int8_t* codes = reinterpret_cast<int8_t*>(buf + (dim + (dim >> 5) + 4) / 4 * 4);
    const int share = (dim / kLaneCodes + ks - 1) / ks * kLaneCodes;
    const int k_first = part_k * share, k_end = min(k_first + share, dim);
    const int pieces = (k_end - k_first + kPieceCodes - 1) / kPieceCodes;

    const uint8_t* w_row[kRows];
#pragma unroll
    for (int q = 0; q < kRows; ++q) w_row[q] = static_cast<const uint8_t*>(p.w) + static_cast<int64_t>(min(n0 + q, p.n - 1)) * p.ldw;
    v4u fw[BATCH][kRows];
    uint2 fs[BATCH];
    auto load = [&](int c0) {
#pragma unroll
        for (int b = 0; b < BATCH; ++b) {
            const int k0 = k_first + (c0 + b) * kPieceCodes + lane * kLaneCodes, kk = k0 < k_end ? k0 : 0;
#pragma unroll
            for (int q = 0; q < kRows; ++q) fw[b][q] = *reinterpret_cast<const v4u*>(w_row[q] + kk * BITS / 8);
            if constexpr (BITS == 4) fs[b] = *reinterpret_cast<const uint2*>(p.s_group + static_cast<int64_t>(kk / 128) * p.n + min(n0, p.n - 4));
            if (c0 + b + 1 >= pieces) break;
        }
    };
    // The row first: loads return in order, and what waits for it must not wait for the weights
    constexpr int kRowPieces = (kRotDim / 8 + kRotThreads - 1) / kRotThreads;
    uint4 yr[kRowPieces];
#pragma unroll
    for (int i = 0; i < kRowPieces; ++i)
        if ((tid + i * kRotThreads) * 8 < dim) yr[i] = *reinterpret_cast<const uint4*>(r.y + (tid + i * kRotThreads) * 8);
    __builtin_amdgcn_sched_barrier(0);
    load(0);
    const int quarter = lane >> 4, my_n = min(n0 + quarter, p.n - 1);
    const bool mine = (lane & 15) == 0 && n0 + quarter < p.n;
    const float s_row = p.rule == kGemvAlpha ? p.alpha : p.row_scale[0];
    const float s_col = p.rule == kGemvAlpha ? 1.0f : p.col_scale[p.one_col_scale ? 0 : my_n];
    __builtin_amdgcn_sched_barrier(0);

#pragma unroll
    for (int i = 0; i < kRowPieces; ++i) {
        const int e0 = (tid + i * kRotThreads) * 8;
        if (e0 < dim) {
            // index bits 0-2 in the registers the row arrives in
            const __half* h = reinterpret_cast<const __half*>(&yr[i]);
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = __half2float(h[j]);
#pragma unroll
            for (int s = 1; s < 8; s <<= 1) {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    if (j & s) continue;
                    const float a = v[j], c = v[j | s];
                    v[j] = a + c;
                    v[j | s] = a - c;
                }
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) buf[phys(e0 + j)] = v[j];
        }
    }
    __syncthreads();
    fwht_passes<kRotThreads, __half>(buf, nullptr, dim, shape.log_m, true, tid, 3);
    if constexpr (S > 1) {
        s_point_quantised<S, kRotThreads, 4>(buf, codes, shape.log_m, r.had_scale, tid);
    } else {
        for (int e0 = tid * 16; e0 < dim; e0 += kRotThreads * 16) {
            uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int j = 0; j < 16; ++j) w[j >> 2] |= static_cast<uint32_t>(sat8_half_away(buf[phys(e0 + j)] * r.had_scale) & 0xff) << (8 * (j & 3));
            *reinterpret_cast<uint4*>(codes + e0) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
    __syncthreads();

    int acc[kRows] = {0, 0, 0, 0};
    for (int c0 = 0; c0 < pieces; c0 += BATCH) {
        if (c0) load(c0);
#pragma unroll
        for (int b = 0; b < BATCH; ++b) {
            if (c0 + b >= pieces) break;
            const int k0 = k_first + (c0 + b) * kPieceCodes + lane * kLaneCodes;
            v4u fa[AQ];
#pragma unroll
            for (int q = 0; q < AQ; ++q) fa[q] = k0 < k_end ? *reinterpret_cast<const v4u*>(codes + k0 + 16 * q) : v4u{0u, 0u, 0u, 0u};
#pragma unroll
            for (int row = 0; row < kRows; ++row) {
                if constexpr (BITS == 8) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) acc[row] = __builtin_amdgcn_sdot4(static_cast<int>(fw[b][row][q]), static_cast<int>(fa[0][q]), acc[row], false);
                } else {
                    const uint32_t pair = row & 2 ? fs[b].y : fs[b].x;
                    const uint32_t one = row & 1 ? pair >> 16 : pair & 0xffffu;
                    const __half2 s2 = bits_h2(one | (one << 16));
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint2 e = expand_grouped(fw[b][row][q], s2);
                        acc[row] = __builtin_amdgcn_sdot4(static_cast<int>(e.x), static_cast<int>(fa[q / 2][2 * (q & 1)]), acc[row], false);
                        acc[row] = __builtin_amdgcn_sdot4(static_cast<int>(e.y), static_cast<int>(fa[q / 2][2 * (q & 1) + 1]), acc[row], false);
                    }
                }
            }
        }
    }
    int sum = row_sum(fold16(fold32(acc[0], acc[2]), fold32(acc[1], acc[3])));          // of row `lane / 16`
    if (ks > 1) {
        if (part_k) parts[wave][lane] = sum;
        __syncthreads();
        if (part_k) return;
        for (int i = 1; i < ks; ++i) sum += parts[wave + i][lane];
    }
    if (!mine) return;
    const float accf = static_cast<float>(sum);
    float y = p.rule == kGemvHalfAway ? (s_col * s_row) * accf : p.rule == kGemvColOuter ? s_col * (s_row * accf)
            : p.rule == kGemvAlpha ? s_row * accf : s_row * (s_col * accf);
    asm volatile("" : "+v"(y));                                  // the fp32 product is rounded on its own
    static_cast<uint16_t*>(p.d)[my_n] = one_f16_or_bf16<QA_OUT_F16>(y);
}
}  // namespace

int gemv_launch(const GemvParams& p, const GemvConv* conv, hipStream_t stream) {
    if (p.bits == 8) {
        if (p.m == 1) return pick<8, 1, 4, 2, 2>(p, conv, stream);
        if (p.m == 2) return pick<8, 2, 3, 2, 2>(p, conv, stream);
        return pick<8, 4, 3, 2, 2>(p, conv, stream);
    }
    if (p.m == 1) return pick<4, 1, 2, 1, 1>(p, conv, stream);
    if (p.m == 2) return pick<4, 2, 2, 1, 1>(p, conv, stream);
    return pick<4, 4, 2, 1, 1>(p, conv, stream);
}

int gemv_rotated_launch(const GemvParams& p, const GemvRotate& r, hipStream_t stream) {
    const HadamardShape h = hadamard_shape(p.k);
    const int64_t groups = (static_cast<int64_t>(p.n) + kRows - 1) / kRows;
    if (p.m != 1 || p.out_type != QA_OUT_F16 || h.s == 0 || h.log_m < 5 || p.k > kRotDim || groups > 2048) return QA_ERR_UNSUPPORTED;
    if (!aligned16(r.y) || !aligned16(p.w) || p.ldw % 16 != 0 || (p.bits == 4 && (p.k % 128 != 0 || p.n % 4 != 0 || (reinterpret_cast<uintptr_t>(p.s_group) & 7u)))) return QA_ERR_UNSUPPORTED;
    const RotShape shape = {h.log_m, groups <= 512 ? 4 : groups <= 1024 ? 2 : 1};
    const int per_block = kRotWaves / shape.ks;
    const dim3 grid(static_cast<unsigned>((groups + per_block - 1) / per_block));
    const int lds = (p.k + (p.k >> 5) + 4) / 4 * 16 + p.k;           // (below 64 KB)
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kRotThreads), lds, stream, GemvArgs(p), r, shape);
        return check_launch();
    };
    if (p.bits == 8) return h.s == 12 ? go(gemv_rotated_kernel<8, 12>) : h.s == 40 ? go(gemv_rotated_kernel<8, 40>) : go(gemv_rotated_kernel<8, 1>);
    return h.s == 12 ? go(gemv_rotated_kernel<4, 12>) : h.s == 40 ? go(gemv_rotated_kernel<4, 40>) : go(gemv_rotated_kernel<4, 1>);
}

}  // namespace qa
