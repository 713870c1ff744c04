// Products of some activation rows, up to 64 a workgroup (the projections of a decode batch or a short prompt): BM x BN
// outputs, K over the workgroup's eight waves, 128 codes of every row at a time; int8 or 4-bit weights.
//
// What bounds them is how fast the CUs fetch their operands, the trips to memory that wait for each other and, with 4-bit
// weights, the expansion of the codes.  A wave keeps the partial sums of the whole tile: an operand fragment serves all of
// the other operand's blocks, and a code is expanded once per BM rows.  All that it needs for a unit of K goes straight to
// its own part of LDS, whole lines with consecutive lanes along a row (fragments of 16x16x64 fetched into registers directly
// touch sixteen rows with consecutive lanes, which a CU takes at about 16 bytes a clock), and from there to registers; the
// next unit is on its way during the arithmetic and no barrier stands between the waves.  4-bit codes are expanded in the
// lane whose fragment they become: the order of K within a unit is free, so a lane's fragments are the 32 codes of one
// 16-byte piece and the activations are read to match.  The waves' sums meet in LDS in the place of the units; a thread then
// finishes single outputs, neighbours along a row.
//
// Before, one kernel of 16 x 16 with fragments fetched into registers by sixteen waves, and 32 x 32 tiles staged through
// registers, the 4-bit codes expanded on the way (rows x outputs x K, us): int8 64 x 192 x 5120 6.7 -> 3.8, 16 x 2560 x 5120 6.9 ->
// 4.8, 64 x 2560 x 5120 7.8 -> 6.6, 200 x 2560 x 5120 11.8 -> 10.2; 4 bits 24 x 192 x 5120 7.4 -> 4.4, 24 x 2560 x 5120 8.1 -> 5.9,
// 64 x 4096 x 8192 12.3 -> 9.3, 24 x 10240 x 2560 9.7 -> 6.4, 64 x 18560 x 4096 18.6 -> 16.6.  What is left of a small one is the
// launch (2.9); the large ones wait for their units, of which a CU holds 100 KB at a time (int8 64 x 10240 x 2560: 64 x 64
// tiles that stream K past one ring take 7.2, 64 x 48 of these 9.4).  With 4-bit weights the fragment reads conflict in LDS, 1.6 to 2.2
// cycles per active one (int8 32 x 32 none, 32 x 80 0.7).
//
// With a conv behind the product (GemvConv) a thread that has the new inputs of four channels makes their conv step as well:
// the state arrives during the product, and a launch and a round trip through memory are saved.
#pragma once
#include "conv2_common.hpp"
#include "gemm_core.hpp"
#include "gemv.hpp"
#include "w4_expand.hpp"

namespace qa {
namespace split {

using namespace gemm;

template <int BITS, int BM, int BN, int DEPTH>
struct Cfg {
    static constexpr int kWaves = 8, kThreads = 64 * kWaves, kRowBlocks = BM / 16, kColBlocks = BN / 16;
    static constexpr int kAReq = BM / 8, kWReq = BN * BITS / 64;                       // requests of 1 KB per unit
    static constexpr int kAtW = BM * kBK, kAtScales = kAtW + kWReq * 1024;             // of a unit: activations, weights, group scales
    static constexpr int kUnit = kAtScales + (BITS == 4 ? kColBlocks * 256 : 0);
    static constexpr int kPitch = BN + 4;                                              // words a row of sums: sixteen rows cover all banks
    // the sums meet in one pass, or two where the rows of all eight waves do not fit
    static constexpr int kPassRows = kWaves * BM * kPitch * 4 <= 120 * 1024 ? BM : BM / 2, kPasses = BM / kPassRows;
    static constexpr int kPass = kPassRows * BN, kOutputs = (kPass + kThreads - 1) / kThreads;  // outputs per pass, and per thread
    static constexpr int kRing = kWaves * DEPTH * kUnit, kSums = kWaves * kPassRows * kPitch * 4;
    static constexpr int kColScales = (BN + 63) / 64 * 64, kRowScales = 64;
    static constexpr int kScalesAt = kRing > kSums ? kRing : kSums;
    static constexpr int kColumnsAt = (kScalesAt + (kColScales + kRowScales) * 4 + 15) / 16 * 16;
    static constexpr int kLdsBytes = kColumnsAt + BN / 4 * static_cast<int>(sizeof(ConvQuad));
    static constexpr int kQuads = (kPass / 4 + kThreads - 1) / kThreads;               // of outputs in a pass, per thread
    static_assert(BM <= 64 && BN <= 256 && kLdsBytes <= 160 * 1024, "tile shape");
};

enum ConvKind { kNoConv, kConvWords, kConvRows };       // the layouts of the conv's state (conv_state_in_words, conv_state_in_rows)

template <int BITS, int BM, int BN, int DEPTH, int OUT, ConvKind CONV>
__global__ __launch_bounds__((Cfg<BITS, BM, BN, DEPTH>::kThreads)) void gemm_split_kernel(GemvArgs p, std::conditional_t<CONV != kNoConv, GemvConv, NoGemvConv> f) {
    using C = Cfg<BITS, BM, BN, DEPTH>;
    __shared__ __attribute__((aligned(16))) uint8_t lds[C::kLdsBytes];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int m0, n0;
    split_tile_of_workgroup<BM, BN>(blockIdx.x, p.m, p.n, m0, n0);
    const int units = (p.k + kBK - 1) / kBK, my_units = (units - wave + C::kWaves - 1) / C::kWaves;        // units wave, wave + 8, ...
    const bool grouped = BITS == 4 && p.s_group != nullptr;
    const uint32_t lds_base = lds_offset_of(lds);

    // the tile's scales, ahead of the first units (rows and columns outside read zero)
    float* const s_col = reinterpret_cast<float*>(lds + C::kScalesAt);
    float* const s_row = s_col + C::kColScales;
    if (p.rule != kGemvAlpha) {
        const v4i rsrc_c = make_rsrc(p.col_scale, (p.one_col_scale ? 1 : p.n) * 4), rsrc_r = make_rsrc(p.row_scale, (p.one_row_scale ? 1 : p.m) * 4);
#pragma unroll
        for (int i = 0; i < (C::kColScales + C::kRowScales) / 64; ++i) {
            if (i % C::kWaves != wave) continue;
            if (i < C::kColScales / 64) buffer_load_lds_b32(rsrc_c, lds_base + C::kScalesAt + i * 256, p.one_col_scale ? 0 : (n0 + i * 64 + lane) * 4);
            else buffer_load_lds_b32(rsrc_r, lds_base + C::kScalesAt + i * 256, p.one_row_scale ? 0 : (m0 + lane) * 4);
        }
    }

    const int ldw = p.ldw;
    const v4i rsrc_a = make_rsrc(p.a, static_cast<int>((static_cast<int64_t>(p.m) - 1) * p.lda + p.k));
    const v4i rsrc_w = make_rsrc(static_cast<const uint8_t*>(p.w) + static_cast<int64_t>(n0) * ldw, (min(BN, p.n - n0) - 1) * ldw + p.k * BITS / 8);
    TileLoader<C::kAReq> load_a;
    load_a.template init<1>(m0, p.m, p.lda, 0, lane);
    TileLoader<BITS == 8 ? C::kWReq : 1> load_w;
    if constexpr (BITS == 8) load_w.template init<1>(0, p.n - n0, ldw, 0, lane);
    // packed weights: request b fetches rows 16 b + l / 4; a row's four pieces are exchanged by bits 2 and 3 of the row, so
    // that sixteen rows of one column of pieces cover all banks
    const int w_off = BITS == 4 ? (lane >> 2) * ldw + ((lane & 3) ^ ((lane >> 4) & 3)) * 16 : 0;
    // group scales are fetched as aligned words of two; `s_first` is the first scale's place in the first word
    const uintptr_t s_addr = reinterpret_cast<uintptr_t>(p.s_group);
    const int s_first = static_cast<int>((s_addr >> 1) & 1);
    v4i rsrc_s = {};
    if (grouped) rsrc_s = make_rsrc(reinterpret_cast<const void*>(s_addr & ~uintptr_t{3}), static_cast<int>((static_cast<int64_t>(units) * p.n + s_first + 1) / 2 * 4));
    int s_at[C::kColBlocks];                                       // index of this lane's row's scale of unit 0
#pragma unroll
    for (int b = 0; b < C::kColBlocks; ++b) s_at[b] = s_first + min(n0 + 16 * b + (lane & 15), p.n - 1);
    uint8_t* const mine = lds + wave * DEPTH * C::kUnit;
    const uint32_t at = lds_base + wave * DEPTH * C::kUnit;
    auto issue = [&](int u, int slot) {
        const int unit = wave + u * C::kWaves, k0 = unit * kBK;
        const uint32_t to = at + slot * C::kUnit;
        if constexpr (BITS == 8) {
            load_w.template issue<1>(rsrc_w, k0, p.k, to + C::kAtW, 0);
            load_a.template issue<1>(rsrc_a, k0, p.k, to, 0);
        } else {                                                   // (K is whole units)
#pragma unroll
            for (int b = 0; b < C::kColBlocks; ++b) {
                buffer_load_lds_b128(rsrc_w, to + C::kAtW + b * 1024, w_off + 16 * b * ldw, unit * (kBK / 2));
                if (grouped) buffer_load_lds_b32(rsrc_s, to + C::kAtScales + b * 256, ((s_at[b] + unit * p.n) << 1) & ~3);
            }
#pragma unroll
            for (int r = 0; r < C::kAReq; ++r) load_a.template issue_whole<1>(r, rsrc_a, k0, to, 0);
        }
    };
    auto arrived = [&](bool all) {                                 // the oldest unit on its way (or all of them)
        constexpr int kReq = C::kAReq + C::kWReq;
        if (all) __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        else if (grouped) __builtin_amdgcn_s_waitcnt(vmcnt_imm((DEPTH - 1) * (kReq + C::kColBlocks)));
        else __builtin_amdgcn_s_waitcnt(vmcnt_imm((DEPTH - 1) * kReq));
        wave_lds_sync();
    };
#pragma unroll
    for (int u = 0; u < DEPTH; ++u)
        if (u < my_units) issue(u, u);

    // With a conv a thread finishes four neighbouring outputs at a time: quad t = tid + q * kThreads of a pass, row t / (BN / 4).
    // The conv state of its row and channels is on its way from here on.
    ConvHeld<CONV == kConvRows> held[CONV ? C::kPasses : 1][CONV ? C::kQuads : 1];
    ConvQuad* const quads = reinterpret_cast<ConvQuad*>(lds + C::kColumnsAt);
    auto is_conv = [&](int n) {
        if constexpr (CONV != kNoConv) return n >= f.ch0 && n < f.ch0 + f.conv.dim;
        else return false;
    };
    if constexpr (CONV != kNoConv) {
        const QaConv2Params& c = f.conv;
#pragma unroll
        for (int i = 0; i < C::kPasses; ++i)
#pragma unroll
            for (int q = 0; q < C::kQuads; ++q) {
                // (columns and rows that are not the conv's read some that are)
                const int t = tid + q * C::kThreads, ch = min(max(n0 + t % (BN / 4) * 4 - f.ch0, 0), c.dim - 4);
                held[i][q] = conv_held4<CONV == kConvRows>(c, min(m0 + C::kPassRows * i + t / (BN / 4), p.m - 1), ch);
            }
        // the columns' taps and scales (a chain of loads), by the last wave, which has the fewest units
        const int quad = tid - (C::kThreads - 64), n = n0 + 4 * quad;
        if (quad >= 0 && quad < BN / 4 && is_conv(n)) quads[quad] = conv_quad(c, part_of(c, n - f.ch0), n - f.ch0);
    }

    v4i acc[C::kRowBlocks][C::kColBlocks];
#pragma unroll
    for (int i = 0; i < C::kRowBlocks; ++i)
#pragma unroll
        for (int b = 0; b < C::kColBlocks; ++b) acc[i][b] = v4i{0, 0, 0, 0};
    const int frow = lane & 15, quarter = lane >> 4;
    // A 16-byte read of LDS takes lanes 0 .. 3, 12 .. 15 and 20 .. 27 together, of the next 32 the same, then the others: rows 0 .. 3 and 12 .. 15
    // of one quarter with rows 4 .. 11 of the next.  Of packed weights a quarter of the wave has two chunks of activations, so with its
    // pieces in their order neighbours' chunks fall on the same banks; 0, 3, 2, 1 do not (conflicts 2.2 cycles per active one -> 0; 64 x 18560 x 4096
    // 16.7 -> 16.5 us, 64 x 4096 x 8192 8.8 -> 8.6, others the same).
    const int piece = BITS == 4 ? 3 * quarter & 3 : quarter;
    for (int base = 0; base < my_units; base += DEPTH) {
        static_for<0, DEPTH>([&](auto slot_c) {
            constexpr int slot = decltype(slot_c)::value;
            const int u = base + slot;
            if (u >= my_units) return;
            arrived(DEPTH == 1 || u + DEPTH > my_units);
            const uint8_t* from = mine + slot * C::kUnit;
            v4i fa[2][C::kRowBlocks], fw[BITS == 8 ? 2 : 1][BITS == 8 ? C::kColBlocks : 1];
            v4u packed[BITS == 4 ? C::kColBlocks : 1];
            uint32_t pair[BITS == 4 ? C::kColBlocks : 1];
#pragma unroll
            for (int b = 0; b < C::kColBlocks; ++b) {
                if constexpr (BITS == 4) {
                    packed[b] = *reinterpret_cast<const v4u*>(from + C::kAtW + b * 1024 + frow * 64 + (piece ^ ((frow >> 2) & 3)) * 16);
                    pair[b] = *reinterpret_cast<const uint32_t*>(from + C::kAtScales + b * 256 + lane * 4);
                } else {
#pragma unroll
                    for (int step = 0; step < 2; ++step)
                        fw[step][b] = *reinterpret_cast<const v4i*>(from + C::kAtW + (b * 16 + frow) * kBK + swz(frow, 4 * step + quarter) * 16);
                }
            }
#pragma unroll
            for (int step = 0; step < 2; ++step)
#pragma unroll
                for (int i = 0; i < C::kRowBlocks; ++i)
                    fa[step][i] = *reinterpret_cast<const v4i*>(from + (i * 16 + frow) * kBK + swz(frow, BITS == 8 ? 4 * step + piece : 2 * piece + step) * 16);
            // all of it is in registers before the slot is given away
            __builtin_amdgcn_s_waitcnt(0xc07f);                    // lgkmcnt(0)
            __builtin_amdgcn_sched_barrier(0);
            const int unit = wave + u * C::kWaves;
            if (u + DEPTH < my_units) issue(u + DEPTH, slot);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = 0; b < C::kColBlocks; ++b) {
                uint2 e[4];
                if constexpr (BITS == 4) {
                    if (grouped) {
                        const uint32_t one = ((s_at[b] + unit * p.n) & 1 ? pair[b] >> 16 : pair[b] & 0xffffu) * 0x10001u;
#pragma unroll
                        for (int w = 0; w < 4; ++w) e[w] = expand_grouped(packed[b][w], bits_h2(one));
                    } else {
#pragma unroll
                        for (int w = 0; w < 4; ++w) e[w] = expand_per_channel(packed[b][w]);
                    }
                }
#pragma unroll
                for (int step = 0; step < 2; ++step) {
                    v4i fb;
                    if constexpr (BITS == 8) fb = fw[step][b];
                    else fb = v4i{static_cast<int>(e[2 * step].x), static_cast<int>(e[2 * step].y), static_cast<int>(e[2 * step + 1].x), static_cast<int>(e[2 * step + 1].y)};
#pragma unroll
                    for (int i = 0; i < C::kRowBlocks; ++i) acc[i][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb, fa[step][i], acc[i][b], 0, 0, 0);
                }
            }
        });
    }

    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));                      // (the scales of a wave without units)
    __syncthreads();                                               // every wave is done with its units
    int* const sums = reinterpret_cast<int*>(lds);
#pragma unroll
    for (int i = 0; i < C::kPasses; ++i) {
        if (i > 0) __syncthreads();                                // the pass before has been read
        // lane l holds row l % 16, columns 4 (l / 16) .. + 3 of a block
#pragma unroll
        for (int r = 0; r < C::kPassRows / 16; ++r)
#pragma unroll
            for (int b = 0; b < C::kColBlocks; ++b)
                *reinterpret_cast<v4i*>(&sums[(wave * C::kPassRows + r * 16 + frow) * C::kPitch + b * 16 + 4 * quarter]) = acc[i * (C::kPassRows / 16) + r][b];
        __syncthreads();
        auto scaled = [&](int sum, int row, int col) {
            const float accf = static_cast<float>(sum), sr = s_row[C::kPassRows * i + row], sc = s_col[col];
            float y;
            if (p.rule == kGemvAlpha) y = p.alpha * accf;
            else if (p.rule == kGemvColOuter) y = sc * (sr * accf);
            else if (p.rule == kGemvHalfAway) y = (sc * sr) * accf;
            else y = sr * (sc * accf);
            asm volatile("" : "+v"(y));                            // the fp32 product is rounded on its own
            return y;
        };
        if constexpr (CONV != kNoConv) {
#pragma unroll
            for (int q = 0; q < C::kQuads; ++q) {
                const int t = tid + q * C::kThreads, row = t / (BN / 4), quad = t % (BN / 4), m = m0 + C::kPassRows * i + row, n = n0 + 4 * quad;
                if (t >= C::kPass / 4 || m >= p.m || n >= p.n) continue;
                v4i sum = {0, 0, 0, 0};
#pragma unroll
                for (int x = 0; x < C::kWaves; ++x) sum += *reinterpret_cast<const v4i*>(&sums[(x * C::kPassRows + row) * C::kPitch + 4 * quad]);
                uint32_t word = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) word |= static_cast<uint32_t>(quant8(scaled(sum[e], row, 4 * quad + e), QA_ROUND_RNE) & 0xff) << (8 * e);
                if (!is_conv(n)) {
                    *reinterpret_cast<uint32_t*>(static_cast<int8_t*>(p.d) + m * p.ldd + n) = word;
                    continue;
                }
                const Part part = part_of(f.conv, n - f.ch0);
                int64_t ls, cs;
                *reinterpret_cast<uint32_t*>(out_ptr(f.conv, part, m, n - f.ch0, &ls, &cs)) = conv_step4<CONV == kConvRows>(f.conv, m, n - f.ch0, quads[quad], held[i][q], word);
            }
            continue;
        }
#pragma unroll
        for (int o = 0; o < C::kOutputs; ++o) {
            const int t = tid + o * C::kThreads, row = t / BN, col = t % BN, m = m0 + C::kPassRows * i + row, n = n0 + col;
            if (t >= C::kPass || m >= p.m || n >= p.n) continue;
            int sum = 0;
#pragma unroll
            for (int x = 0; x < C::kWaves; ++x) sum += sums[(x * C::kPassRows + row) * C::kPitch + col];
            const float y = scaled(sum, row, col);
            if constexpr (OUT == QA_OUT_I8) {
                static_cast<int8_t*>(p.d)[m * p.ldd + n] = static_cast<int8_t>(quant8(y, p.half_away ? QA_ROUND_HALF_AWAY : QA_ROUND_RNE));
            } else {
                static_cast<uint16_t*>(p.d)[m * p.ldd + n] = one_f16_or_bf16<OUT>(y);
            }
        }
    }
}

template <int BITS, int BM, int BN, int DEPTH>
int launch(const GemvParams& p, const GemvConv* conv, hipStream_t stream) {
    using C = Cfg<BITS, BM, BN, DEPTH>;
    const int64_t blocks = static_cast<int64_t>((p.m + BM - 1) / BM) * ((p.n + BN - 1) / BN);
    const GemvArgs args(p);
    auto go = [&](auto kernel, const auto& f) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(C::kThreads), 0, stream, args, f);
        return check_launch();
    };
    if (conv) return conv_state_in_words(conv->conv) ? go(gemm_split_kernel<BITS, BM, BN, DEPTH, QA_OUT_I8, kConvWords>, *conv) : go(gemm_split_kernel<BITS, BM, BN, DEPTH, QA_OUT_I8, kConvRows>, *conv);
    const NoGemvConv none = {};
    if (p.out_type == QA_OUT_F16) return go(gemm_split_kernel<BITS, BM, BN, DEPTH, QA_OUT_F16, kNoConv>, none);
    if constexpr (BITS == 8) { if (p.out_type == QA_OUT_BF16) return go(gemm_split_kernel<BITS, BM, BN, DEPTH, QA_OUT_BF16, kNoConv>, none); }
    return go(gemm_split_kernel<BITS, BM, BN, DEPTH, QA_OUT_I8, kNoConv>, none);
}

// the tile shapes in the order of kSplitShapes
template <int BITS>
int launch_shape(const GemvParams& p, int shape, const GemvConv* conv, hipStream_t stream) {
    switch (shape) {
        case 0: return launch<BITS, 16, 16, 2>(p, conv, stream);
        case 1: return launch<BITS, 16, 32, 1>(p, conv, stream);
        case 2: return launch<BITS, 16, 48, 1>(p, conv, stream);
        case 3: return launch<BITS, 32, 32, 1>(p, conv, stream);
        case 4: return launch<BITS, 32, 48, 1>(p, conv, stream);
        case 5: return launch<BITS, 32, 80, 1>(p, conv, stream);
        case 6: if constexpr (BITS == 4) return launch<BITS, 64, 48, 1>(p, conv, stream); else break;
        case 7: return launch<BITS, 64, 80, 1>(p, conv, stream);
    }
    return QA_ERR_UNSUPPORTED;
}

}  // namespace split
}  // namespace qa
