// W4A8 GEMM: int8 activations x 4-bit weights with group-wise (128) fp16 scales or per-channel
// scaling, on the int8 matrix cores.
//
//   grouped:      w8[n,k] = int8( rne( (code - 8) * s_group[k/128, n] ) )      one fp16 FMA, one rounding
//   per-channel:  w8[n,k] = 16 * signed_nibble(code)
//   acc[m,n] = sum_k a[m,k] * w8[n,k] (int32);  d = cast( (float(acc) * s_channel[n]) * s_token[m|0] )
// Reference arithmetic: csrc/linear/marlin_qqq_gemm_kernel.cuh:125-178 (dequant), :744-749 (fp16
// epilogue), marlin_qqq_gemm_kernel_o8.cuh:107-116 (int8 epilogue, round-half-even saturating).
//
// Weight storage (this library's own): uint8 (N, K/2).  Each aligned group of 8 codes of a row is
// one 32-bit word whose byte i holds code[8w+i] in the low nibble and code[8w+4+i] in the high
// nibble, so that the fp16 exponent trick below yields the int8 bytes in k order.
// The expansion to int8 is arithmetic in registers: (word & 0x000f000f) | 0x6400_6400 is the half2 (1024+c0, 1024+c2);
// subtracting 1032 gives c-8 exactly; one packed FMA with the group scale and the constant 1280 leaves rne((c-8)*s) as a
// two's-complement byte in the low byte of each half; v_perm gathers four of them: fifteen vector instructions for eight
// codes and lane, four to five cycles each, where a product of 32 x 32 x 32 takes 32 cycles of the matrix cores.  How often
// a code is expanded - once per row block of the output - and on how many of the chip's SIMDs at once is what the kernels
// below trade: every one of them is bound by it from about a hundred activation rows on.
#include "gemm_core.hpp"
#include "gemv.hpp"
#include "w4_expand.hpp"

#include <algorithm>
#include <cmath>

namespace qa {
namespace {

using namespace gemm;

// The tile kernel, 64 x 64 outputs over four waves of 32 x 32.  Everything that comes from memory goes straight to LDS, STAGES - 1 tiles ahead and counted by hand: the
// activations as the fragments want them, the packed weights and their group scales as each thread's own 16 bytes and word
// (no other lane reads those: they are registers that a load in flight does not occupy).  During the multiplications of tile
// t a thread expands its codes of tile t + 1, a word behind every multiplication, into the one of two int8 weight
// tiles that is not being read: the vector units work in the shadow of the matrix cores.  (Behind all multiplications of a
// tile instead, with a tile's loads issued one tile ahead, a 64 x 64 tile on a CU of its own took 0.67 us per 128 of K; now
// 0.38, of which the expansion is 0.15 and the LDS traffic of fragments, codes and tiles about as much.)
struct W4Tile {
    static constexpr int kStages = 3;
    using C = Cfg<1, 1, 2, 2, kStages>;
    static constexpr int kSlots = kStages - 1;                     // tiles of packed weights
    static constexpr int kABytes = C::kBM * kBK, kWBytes = C::kBN * kBK;
    static constexpr int kPackedBytes = C::kBN * (kBK / 2), kScaleBytes = C::kThreads * 4;      // a thread: 16 bytes (32 codes), a word
    static constexpr int kScalesAt = kStages * kABytes + 2 * kWBytes + kSlots * (kPackedBytes + kScaleBytes);
    static constexpr int kLdsBytes = kScalesAt + TileScales<C::kBM, C::kBN, C::kWaves>::kBytes;
    static_assert(kPackedBytes == 16 * C::kThreads && epilogue_lds_bytes<1, 1, C::kWaves>() <= kScalesAt, "tile shape");
};

template <bool GROUPED, int OUT>
__global__ __launch_bounds__(W4Tile::C::kThreads) void gemm_w4a8_kernel(QaGemmW4A8Params p) {
    using W = W4Tile;
    using C = W::C;
    constexpr int BM = C::kBM, BN = C::kBN, WAVES = C::kWaves, STAGES = W::kStages;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int tiles_m = (p.m + BM - 1) / BM, tiles_n = (p.n + BN - 1) / BN;
    int tile_m, tile_n;
    tile_of_workgroup<BM, BN>(blockIdx.x, tiles_m, tiles_n, tile_m, tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int k_tiles = p.k / kBK, ldw = p.k / 2;

    const uint32_t lds_base = lds_offset_of(lds);
    TileScales<BM, BN, WAVES>::request(lds_base + W::kScalesAt, p.s_token, p.tok_scale_numel, p.m, m0, p.s_channel, p.n, p.n, n0, wave, lane);
    constexpr int kAtW = STAGES * W::kABytes, kAtPacked = kAtW + 2 * W::kWBytes, kAtScale = kAtPacked + W::kSlots * W::kPackedBytes;
    const v4i rsrc_a = make_rsrc(p.a, static_cast<int>((static_cast<int64_t>(p.m) - 1) * p.lda + p.k));
    const v4i rsrc_w = make_rsrc(p.w_packed + static_cast<int64_t>(n0) * ldw, min(BN, p.n - n0) * ldw);
    // group scales are fetched as aligned words of two; `s_first` is the first scale's place in the first word
    const uintptr_t s_addr = reinterpret_cast<uintptr_t>(p.s_group);
    const int s_first = static_cast<int>((s_addr >> 1) & 1);
    v4i rsrc_s = {};
    if constexpr (GROUPED) rsrc_s = make_rsrc(reinterpret_cast<const void*>(s_addr & ~uintptr_t{3}), static_cast<int>((static_cast<int64_t>(k_tiles) * p.n + s_first + 1) / 2 * 4));
    // (K is whole tiles: a tile is an offset the whole wave shares.  Requests past the last tile repeat it.)
    TileLoader<C::kAInstr> load_a;
    load_a.template init<WAVES>(m0, p.m, p.lda, wave, lane);
    const int last = k_tiles - 1;
    auto issue_a = [&](int r, int tile, int stage) {
        buffer_load_lds_b128(rsrc_a, lds_base + stage * W::kABytes + (r * WAVES + wave) * 1024, load_a.voff[r], min(tile, last) * kBK);
    };

    // this thread's packed chunk of the weight tile: row tid / 4, codes 32 (tid % 4) .. + 31
    const int row = tid >> 2, quarter = tid & 3;
    const int w_off = row * ldw + quarter * 16, s_col = s_first + min(n0 + row, p.n - 1);
    uint32_t s_pick = 0x01000100u + (s_col & 1) * 0x02020202u;     // the half of the fetched word, twice
    uint8_t* const to_w[2] = {lds + kAtW + row * kBK + swz(row, 2 * quarter) * 16, lds + kAtW + row * kBK + swz(row, 2 * quarter + 1) * 16};
    const uint32_t s_flip = p.n & 1 ? 0x02020202u : 0u;
    auto issue_w = [&](int tile, int slot) {
        const int t = min(tile, last);
        buffer_load_lds_b128(rsrc_w, lds_base + kAtPacked + slot * W::kPackedBytes + wave * 1024, w_off, t * (kBK / 2));
        if constexpr (GROUPED) buffer_load_lds_b32(rsrc_s, lds_base + kAtScale + slot * W::kScaleBytes + wave * 256, ((s_col + t * p.n) << 1) & ~3);
    };
    uint4 wreg;
    __half2 s2;
    auto fetch_w = [&](int slot) {                         // tile after tile
        wreg = *reinterpret_cast<const uint4*>(lds + kAtPacked + slot * W::kPackedBytes + tid * 16);
        if constexpr (GROUPED) {
            const uint32_t word = *reinterpret_cast<const uint32_t*>(lds + kAtScale + slot * W::kScaleBytes + tid * 4);
            s2 = bits_h2(__builtin_amdgcn_perm(word, word, s_pick));
            s_pick ^= s_flip;
        }
    };
    // word `w` of this thread's four (a pair is written when its second one is done)
    uint2 done;
    auto expand_w = [&](int w, int to) {
        const uint32_t packed = w == 0 ? wreg.x : w == 1 ? wreg.y : w == 2 ? wreg.z : wreg.w;
        const uint2 e = GROUPED ? expand_grouped(packed, s2) : expand_per_channel(packed);
        if (w % 2 == 0) done = e;
        else *reinterpret_cast<uint4*>(to_w[w / 2] + to * W::kWBytes) = make_uint4(done.x, done.y, e.x, e.y);
    };

    v16i acc[1][1];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][0][r] = 0;

    if (k_tiles > 0) {
        // Requests go out in the order W(0) A(0) W(1) A(1) ..., the first tile's weights being expanded before the loop
        issue_w(0, 0);
#pragma unroll
        for (int s = 0; s < STAGES - 1; ++s) {
#pragma unroll
            for (int r = 0; r < C::kAInstr; ++r) issue_a(r, s, s);
            if (s + 1 < STAGES - 1) issue_w(s + 1, s + 1);
        }
        constexpr int kLoads = C::kAInstr + (GROUPED ? 2 : 1);                 // requests of a wave per tile
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((STAGES - 2) * kLoads + C::kAInstr));
        wave_lds_sync();
        fetch_w(0);
#pragma unroll
        for (int w = 0; w < 4; ++w) expand_w(w, 0);
        __builtin_amdgcn_sched_barrier(0);
        issue_w(STAGES - 1, 0);
        const int frow = lane & 31, fhalf = lane >> 5;
        constexpr int kUnroll = 6;                                             // whole turns of stages, slots and weight tiles
        static_assert(kUnroll % STAGES == 0 && kUnroll % W::kSlots == 0 && kUnroll % 2 == 0 && C::kAInstr <= 4, "a request behind each of four multiplications");
        for (int base = 0; base < k_tiles; base += kUnroll) {
            static_for<0, kUnroll>([&](auto u_c) {
                constexpr int u = decltype(u_c)::value;
                const int kt = base + u;
                if (kt >= k_tiles) return;
                __builtin_amdgcn_s_waitcnt(vmcnt_imm((STAGES - 2) * kLoads));   // A(kt) and W(kt + 1) are here
                __syncthreads();
                fetch_w((u + 1) % W::kSlots);
                __builtin_amdgcn_sched_barrier(0);
                mma_tile_paced(lds + (u % STAGES) * W::kABytes + wm * 32 * kBK, lds + kAtW + (u % 2) * W::kWBytes + wn * 32 * kBK, frow, fhalf, acc[0][0],
                               [&](int step) {
                                   // (the fragments of the multiplication before this were read after fetch_w's
                                   // words, so these are in their registers and the slot they came from is free)
                                   if (step == 0) issue_w(kt + STAGES, (u + STAGES) % W::kSlots);
                                   if (step < C::kAInstr) issue_a(step, kt + STAGES - 1, (u + STAGES - 1) % STAGES);
                                   expand_w(step, (u + 1) % 2);
                               });
            });
        }
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    __syncthreads();

    Epilogue e;
    e.use_alpha = 0; e.alpha = 0.0f; e.round_mode = QA_ROUND_RNE; e.col_outer = 0;
    e.ldd = p.ldd; e.d = p.d;
    epilogue<1, 1, OUT, false, false>(e, acc, lds, p.m, p.n, m0 + wm * 32, n0 + wn * 32, wave, lane,
                                      reinterpret_cast<const float*>(lds + W::kScalesAt), BN + wm * 32, wn * 32);
}

template <int OUT>
int launch_tile(const QaGemmW4A8Params& p, hipStream_t stream) {
    using W = W4Tile;
    using C = W::C;
    const int64_t tiles = static_cast<int64_t>((p.m + C::kBM - 1) / C::kBM) * ((p.n + C::kBN - 1) / C::kBN);
    if (tiles > 0x7fffffffLL || static_cast<int64_t>(C::kBN) * p.k > 0x7fffffffLL || static_cast<int64_t>(p.n) * p.k > 64LL * 0x7fffff00LL) return QA_ERR_SHAPE;
    static_assert(W::kLdsBytes <= 65536, "more LDS than a launch gets by default");
    auto kernel = p.group_size > 0 ? gemm_w4a8_kernel<true, OUT> : gemm_w4a8_kernel<false, OUT>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(tiles)), dim3(C::kThreads), W::kLdsBytes, stream, p);
    return check_launch();
}

// ---------------------------------------------------------------------------------------------
// Weights that never pass through LDS.  A wave owns 32 output columns and all BM = 32 TM rows of the tile; the packed codes
// go from memory into the registers of the lane whose fragment they become, and are expanded there between the
// multiplications.  A tile of K is KT codes (KT / 2 for either half of the lanes, which is 32 or 64 consecutive bytes of a
// packed row - the order of K inside a tile is free as long as both operands agree); weights are requested two tiles ahead
// (registers in three sets), activations one, straight to LDS.  The four waves share the activations.  No code is expanded
// twice in a tile and none costs LDS bandwidth, so this goes further than the tile kernel above: 777 x 6144 x 1536 in 192
// rows takes 16.0 us, in 64 x 64 tiles 20.9 and did 22.8 in the 128 x 128 tiles it replaces.
// ---------------------------------------------------------------------------------------------
template <int TM, int NW, int KT>
struct RegCfg {
    static constexpr int kThreads = 64 * NW;
    static constexpr int kBM = 32 * TM, kBN = 32 * NW;
    static constexpr int kRowChunks = KT / 16;
    static constexpr int kABytes = kBM * KT;
    static constexpr int kAInstr = kABytes / 1024 / NW;            // direct-to-LDS requests of a wave per tile
    static constexpr int kWLoads = KT / 64;                        // 16-byte pieces of packed weights per lane and tile
    // what a row's 16-byte pieces are exchanged by: sixteen neighbouring rows of one column of pieces then cover all banks
    __device__ static __forceinline__ int exchange(int row) { return KT == 256 ? row & 15 : (row >> 1) & 7; }
    static constexpr int kEpilogue = epilogue_lds_bytes<TM, 1, NW>();
    static constexpr int kScalesAt = 2 * kABytes > kEpilogue ? 2 * kABytes : kEpilogue;
    static constexpr int kLdsBytes = kScalesAt + TileScales<kBM, kBN, NW>::kBytes;
};

template <int TM, int NW, int KT, bool GROUPED, int OUT, bool TRANS>
__global__ __launch_bounds__(64 * NW) void gemm_w4a8_reg_kernel(QaGemmW4A8Params p) {
    using R = RegCfg<TM, NW, KT>;
    static_assert(R::kAInstr * NW * 1024 == R::kABytes && (KT == 128 || KT == 256), "tile shape");
    constexpr int kOob = 0x7ffffff0;                               // beyond any buffer: the load returns zeros
    constexpr int kSteps = KT / 32, kSets = 3, kLoads = R::kWLoads + (GROUPED ? 1 : 0);
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int frow = lane & 31, fhalf = lane >> 5;
    const int tiles_m = (p.m + R::kBM - 1) / R::kBM, tiles_n = (p.n + R::kBN - 1) / R::kBN;
    int tile_m, tile_n;
    tile_of_workgroup<R::kBM, R::kBN>(blockIdx.x, tiles_m, tiles_n, tile_m, tile_n);
    const int m0 = tile_m * R::kBM, n0 = tile_n * R::kBN + wave * 32;
    const int ldw = p.k / 2, k_tiles = (p.k + KT - 1) / KT;

    // activations: request j of a wave fills LDS bytes [(j NW + wave) 1024, + 1024) of the tile, i.e. 1024 / KT rows
    const v4i rsrc_a = make_rsrc(p.a, static_cast<int>((static_cast<int64_t>(p.m) - 1) * p.lda + p.k));
    const uint32_t lds_a = lds_offset_of(lds);
    TileScales<R::kBM, R::kBN, NW>::request(lds_a + R::kScalesAt, p.s_token, p.tok_scale_numel, p.m, m0, p.s_channel, p.n, p.n, tile_n * R::kBN, wave, lane);
    int a_off[R::kAInstr], a_k[R::kAInstr];
#pragma unroll
    for (int j = 0; j < R::kAInstr; ++j) {
        const int piece = (j * NW + wave) * 64 + lane, row = piece / R::kRowChunks, c = (piece % R::kRowChunks) ^ R::exchange(row);
        a_k[j] = c * 16;
        a_off[j] = m0 + row < p.m ? static_cast<int>((m0 + row) * p.lda) + c * 16 : 0x70000000;
    }
    auto issue_a = [&](int tile, int stage) {
        const int k0 = min(tile, k_tiles - 1) * KT;                                  // (past the last tile: that one again)
#pragma unroll
        for (int j = 0; j < R::kAInstr; ++j) {
            const int off = KT == 128 || k0 + a_k[j] < p.k ? a_off[j] : kOob;        // (K is a multiple of 128)
            buffer_load_lds_b128(rsrc_a, lds_a + stage * R::kABytes + (j * NW + wave) * 1024, off, k0);
        }
    };

    // weights: this lane's row, its half of the tile's codes
    const int rows_left = p.n - n0;
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w_packed) + static_cast<int64_t>(n0) * ldw, 0,
                                                                           rows_left > 0 ? min(32, rows_left) * ldw : 0, kRsrcFlags);
    const __half* sg = GROUPED ? static_cast<const __half*>(p.s_group) + min(n0 + frow, p.n - 1) : nullptr;
    v4u fw[kSets][R::kWLoads];
    uint16_t fs[kSets];
    auto load_w = [&](int t, auto set_c) {
        constexpr int set = decltype(set_c)::value;
        const int tile = min(t, k_tiles - 1);
#pragma unroll
        for (int l = 0; l < R::kWLoads; ++l) fw[set][l] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, frow * ldw + fhalf * (KT / 4) + tile * (KT / 2) + 16 * l, 0, 0);
        if constexpr (GROUPED) fs[set] = __half_as_ushort(sg[static_cast<int64_t>(min(KT == 256 ? 2 * tile + fhalf : tile, p.k / 128 - 1)) * p.n]);
    };

    v16i acc[1][TM];
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][j][r] = 0;

    if (k_tiles > 0) {
        load_w(0, std::integral_constant<int, 0>{});
        __builtin_amdgcn_sched_barrier(0);
        issue_a(0, 0);
        load_w(1, std::integral_constant<int, 1>{});
        for (int base = 0; base < k_tiles; base += 6) {
            static_for<0, 6>([&](auto u_c) {
                constexpr int u = decltype(u_c)::value, set = u % kSets, stage = u % 2;
                const int tile = base + u;
                if (tile >= k_tiles) return;
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_waitcnt(vmcnt_imm(kLoads));     // this tile's activations (and weights) are here
                __syncthreads();
                const uint8_t* sa = lds + stage * R::kABytes;
                v4i fa[2][TM], w8[2];
                auto fetch = [&](int kk) {
#pragma unroll
                    for (int j = 0; j < TM; ++j) {
                        const int row = j * 32 + frow, c = (fhalf * kSteps + kk) ^ R::exchange(row);
                        fa[kk & 1][j] = *reinterpret_cast<const v4i*>(sa + row * KT + c * 16);
                    }
                };
                __half2 s2;
                auto expand = [&](int kk, int half) {
                    const v4u piece = fw[set][kk / 2];
                    const uint32_t word = piece[2 * (kk & 1) + half];
                    const uint2 e = GROUPED ? expand_grouped(word, s2) : expand_per_channel(word);
                    w8[kk & 1][2 * half] = static_cast<int>(e.x);
                    w8[kk & 1][2 * half + 1] = static_cast<int>(e.y);
                };
                fetch(0);
                if constexpr (GROUPED) s2 = bits_h2(static_cast<uint32_t>(fs[set]) * 0x10001u);
#pragma unroll
                for (int l = 0; l < R::kWLoads; ++l) asm volatile("" : "+v"(fw[set][l]));      // (all of the set is waited for here)
                expand(0, 0);
                expand(0, 1);
                __builtin_amdgcn_sched_barrier(0);
                // activations before weights: the wait for the next tile's weights then never includes the tile after it
                issue_a(tile + 1, stage ^ 1);
                load_w(tile + 2, std::integral_constant<int, (u + 2) % kSets>{});
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int kk = 0; kk < kSteps; ++kk) {
                    if (kk + 1 < kSteps) fetch(kk + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int x = 0; x < TM; ++x) {
                        acc[0][x] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w8[kk & 1], fa[kk & 1][x], acc[0][x], 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        if (kk + 1 < kSteps) {
#pragma unroll
                            for (int w = x * 2 / TM; w < (x + 1) * 2 / TM; ++w) expand(kk + 1, w);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            });
        }
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    __syncthreads();

    Epilogue e;
    e.use_alpha = 0; e.alpha = 0.0f; e.round_mode = QA_ROUND_RNE; e.col_outer = 0;
    e.ldd = p.ldd; e.d = p.d;
    epilogue<TM, 1, OUT, false, TRANS>(e, acc, lds, p.m, p.n, m0, n0, wave, lane, reinterpret_cast<const float*>(lds + R::kScalesAt), R::kBN, wave * 32);
}

template <int TM, int NW, int KT, int OUT, bool TRANS>
int launch_reg_one(const QaGemmW4A8Params& p, hipStream_t stream) {
    using R = RegCfg<TM, NW, KT>;
    const int64_t tiles = static_cast<int64_t>((p.m + R::kBM - 1) / R::kBM) * ((p.n + R::kBN - 1) / R::kBN);
    if (tiles > 0x7fffffffLL || 16LL * p.k > 0x7fffffffLL) return QA_ERR_SHAPE;
    auto kernel = p.group_size > 0 ? gemm_w4a8_reg_kernel<TM, NW, KT, true, OUT, TRANS> : gemm_w4a8_reg_kernel<TM, NW, KT, false, OUT, TRANS>;
    if (R::kLdsBytes > 65536) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                R::kLdsBytes) != hipSuccess) {
            return check_launch();
        }
    }
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(tiles)), dim3(R::kThreads), R::kLdsBytes, stream, p);
    return check_launch();
}

template <int TM, int NW, int KT>
int launch_reg(const QaGemmW4A8Params& p, hipStream_t stream) {
    return p.out_type == QA_OUT_I8 ? launch_reg_one<TM, NW, KT, QA_OUT_I8, false>(p, stream) : launch_reg_one<TM, NW, KT, QA_OUT_F16, false>(p, stream);
}

// ---------------------------------------------------------------------------------------------
// Few activation rows, transposed output: a stream over the packed weights.  A workgroup
// owns 32 output columns and all rows; its WAVES waves split K between them in interleaved pieces
// of 256 codes, i.e. one full 128-byte line of packed weights per row.  A wave fetches a piece with
// eight lanes per row (DEPTH pieces in flight in registers), expands its 32 codes per lane to int8
// and passes them through a staging area in LDS that is private to the wave; the activation tiles
// take the same route, one 128-byte half at a time.  Partial sums meet in LDS at the end.
// ---------------------------------------------------------------------------------------------
template <int TM, int WAVES>
constexpr int skinny_lds_bytes() { return WAVES * (2 + TM) * 32 * kBK + TM * 16 * 64 * 4; }      // (2 + TM) tiles per wave, TM reduction blocks

// Adds the waves' partial accumulators in `red` (TM*16*64 ints, zeroed by the caller before any
// barrier it has passed), then every thread scales and writes four columns of one row.
// Lane l of the accumulator layout holds row (l & 31) and, in registers 4q..4q+3, the columns
// 8q + 4*(l >> 5) + (0..3): one unit = (row block, q, lane).
template <int TM, int OUT>
__device__ __forceinline__ void skinny_reduce_store(const QaGemmW4A8Params& p, v16i (&acc)[TM], int* red, int m0, int n0, int tid, int threads) {
    const int lane = tid & 63;
    __syncthreads();                                       // red is zero
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            __hip_atomic_fetch_add(&red[(j * 16 + r) * 64 + lane], acc[j][r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __syncthreads();
    for (int u = tid; u < TM * 4 * 64; u += threads) {
        const int ul = u & 63, j = u >> 8, q = (u >> 6) & 3;
        const int mm = m0 + j * 32 + (ul & 31), nn = n0 + 8 * q + 4 * (ul >> 5);
        if (mm >= p.m || nn >= p.n) continue;
        const float s_row = p.s_token[p.tok_scale_numel == 1 ? 0 : mm];
        for (int t = 0; t < min(4, p.n - nn); ++t) {
            float v = s_row * (p.s_channel[nn + t] * static_cast<float>(red[(j * 16 + q * 4 + t) * 64 + ul]));
            asm volatile("" : "+v"(v));                    // the fp32 product is rounded on its own
            const int64_t at = static_cast<int64_t>(nn + t) * p.ldd + mm;
            if (OUT == QA_OUT_I8) static_cast<int8_t*>(p.d)[at] = static_cast<int8_t>(quant8(v, QA_ROUND_RNE));
            else static_cast<uint16_t*>(p.d)[at] = one_f16_or_bf16<OUT>(v);
        }
    }
}

template <int TM, int AI, int WAVES, int DEPTH, int OUT>
__global__ __launch_bounds__(64 * WAVES) void gemm_w4a8_skinny_kernel(QaGemmW4A8Params p) {
    constexpr int kThreads = 64 * WAVES;
    constexpr int kOob = 0x7ffffff0;                       // beyond any buffer: the load returns zeros
    constexpr int kTile = 32 * kBK;
    constexpr int kPiece = 2 * kBK;                        // codes per row and piece
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    int* red = reinterpret_cast<int*>(lds + WAVES * (2 + TM) * kTile);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int frow = lane & 31, fhalf = lane >> 5;
    int m0, n0;
    split_tile_of_workgroup<32 * TM, 32>(blockIdx.x, p.m, p.n, m0, n0);
    const bool grouped = p.group_size > 0;
    for (int i = tid; i < TM * 16 * 64; i += kThreads) red[i] = 0;
    uint8_t* stage = lds + wave * ((2 + TM) * kTile);          // two weight halves, TM activation tiles
    if (AI < 4) {
        // only the first 8*AI rows of an activation tile are ever fetched (M <= 8*AI): the rest stays zero
        for (int i = lane; i < TM * kTile / 16; i += 64) reinterpret_cast<v4u*>(stage + 2 * kTile)[i] = v4u{0u, 0u, 0u, 0u};
    }

    const int ldw = p.k / 2;
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(p.w_packed), 0, static_cast<int>(static_cast<int64_t>(p.n) * ldw), kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(p.a), 0, static_cast<int>((static_cast<int64_t>(p.m) - 1) * p.lda + p.k), kRsrcFlags);
    // fetch mapping: instruction i, lane l -> tile row 8i + l/8, 16-byte chunk l%8.  A packed chunk is
    // 32 codes: chunks 0..3 expand into the first 128-code half of the piece, 4..7 into the second.
    const int lrow = lane >> 3, lchunk = lane & 7;
    const int my_half = lchunk >> 2, my_c0 = (lchunk & 3) * 2;
    int w_off[4], a_off[TM][AI], s_col[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = n0 + 8 * i + lrow;
        w_off[i] = row < p.n ? row * ldw + lchunk * 16 : -1;
        s_col[i] = min(row, p.n - 1);
        if (i < AI) {
#pragma unroll
            for (int j = 0; j < TM; ++j) {
                const int arow = m0 + j * 32 + 8 * i + lrow;
                a_off[j][i] = arow < p.m ? static_cast<int>(arow * p.lda) + lchunk * 16 : -1;
            }
        }
    }
    const __half* sg = static_cast<const __half*>(p.s_group);
    const int n_groups = p.k / kBK;

    const int pieces = (p.k + kPiece - 1) / kPiece;
    const int my_pieces = (pieces - wave + WAVES - 1) / WAVES;
    v4u fw[DEPTH][4], fa[DEPTH][2][TM][AI];
    __half fs[DEPTH][4];
    auto load = [&](int i_piece, auto buf_c) {
        constexpr int buf = decltype(buf_c)::value;
        const int k0 = (wave + i_piece * WAVES) * kPiece;
        const bool w_ok = k0 + lchunk * 32 < p.k;
        const int group = min(k0 / kBK + my_half, n_groups - 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            fw[buf][i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, (w_ok && w_off[i] >= 0) ? w_off[i] + k0 / 2 : kOob, 0, 0);
            if (grouped) fs[buf][i] = sg[static_cast<int64_t>(group) * p.n + s_col[i]];
            if (i < AI) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bool a_k_ok = k0 + h * kBK + lchunk * 16 < p.k;
#pragma unroll
                    for (int j = 0; j < TM; ++j) {
                        fa[buf][h][j][i] = __builtin_amdgcn_raw_buffer_load_b128(
                            rsrc_a, (a_k_ok && a_off[j][i] >= 0) ? a_off[j][i] + k0 + h * kBK : kOob, 0, 0);
                    }
                }
            }
        }
    };

    v16i acc[TM];
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0;

    static_for<0, DEPTH - 1>([&](auto s) {
        if (decltype(s)::value < my_pieces) load(decltype(s)::value, s);
    });
    for (int base = 0; base < my_pieces; base += DEPTH) {
        static_for<0, DEPTH>([&](auto s_c) {
            constexpr int s = decltype(s_c)::value;
            if (base + s + DEPTH - 1 < my_pieces) load(base + s + DEPTH - 1, std::integral_constant<int, (s + DEPTH - 1) % DEPTH>{});
            if (base + s < my_pieces) {
                // expand this lane's 32 codes per fetched row into its half of the staged weights
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t w[4] = {fw[s][i].x, fw[s][i].y, fw[s][i].z, fw[s][i].w};
                    uint2 e[4];
                    if (grouped) {
                        const __half2 s2 = __half2half2(fs[s][i]);
#pragma unroll
                        for (int t = 0; t < 4; ++t) e[t] = expand_grouped(w[t], s2);
                    } else {
#pragma unroll
                        for (int t = 0; t < 4; ++t) e[t] = expand_per_channel(w[t]);
                    }
                    const int row = 8 * i + lrow;
                    uint8_t* dst = stage + my_half * kTile + row * kBK;
                    *reinterpret_cast<v4u*>(dst + swz(row, my_c0) * 16) = v4u{e[0].x, e[0].y, e[1].x, e[1].y};
                    *reinterpret_cast<v4u*>(dst + swz(row, my_c0 + 1) * 16) = v4u{e[2].x, e[2].y, e[3].x, e[3].y};
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
#pragma unroll
                    for (int i = 0; i < AI; ++i) {
                        const int row = 8 * i + lrow;
#pragma unroll
                        for (int j = 0; j < TM; ++j)
                            *reinterpret_cast<v4u*>(stage + (2 + j) * kTile + row * kBK + swz(row, lchunk) * 16) = fa[s][h][j][i];
                    }
                    wave_lds_sync();
#pragma unroll
                    for (int kk = 0; kk < 4; ++kk) {
                        const int off = frow * kBK + swz(frow, kk * 2 + fhalf) * 16;
                        const v4i bw = *reinterpret_cast<const v4i*>(stage + h * kTile + off);
#pragma unroll
                        for (int j = 0; j < TM; ++j) {
                            const v4i ba = *reinterpret_cast<const v4i*>(stage + (2 + j) * kTile + off);
                            acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bw, ba, acc[j], 0, 0, 0);
                        }
                    }
                    wave_lds_sync();
                }
            }
        });
    }

    skinny_reduce_store<TM, OUT>(p, acc, red, m0, n0, tid, kThreads);
}

template <int TM, int AI, int WAVES, int DEPTH, int OUT>
int launch_skinny_one(const QaGemmW4A8Params& p, hipStream_t stream) {
    constexpr int kLds = skinny_lds_bytes<TM, WAVES>();
    auto kernel = gemm_w4a8_skinny_kernel<TM, AI, WAVES, DEPTH, OUT>;
    if (kLds > 65536) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                kLds) != hipSuccess) {
            return check_launch();
        }
    }
    const int64_t blocks = static_cast<int64_t>((p.m + 32 * TM - 1) / (32 * TM)) * ((p.n + 31) / 32);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(64 * WAVES), kLds, stream, p);
    return check_launch();
}

template <int TM, int AI, int WAVES, int DEPTH>
int launch_skinny(const QaGemmW4A8Params& p, hipStream_t stream) {
    return p.out_type == QA_OUT_I8 ? launch_skinny_one<TM, AI, WAVES, DEPTH, QA_OUT_I8>(p, stream) : launch_skinny_one<TM, AI, WAVES, DEPTH, QA_OUT_F16>(p, stream);
}

int64_t tiles_of(const QaGemmW4A8Params& p, int64_t bm, int64_t bn) { return ((p.m + bm - 1) / bm) * ((p.n + bn - 1) / bn); }

int dispatch_skinny(const QaGemmW4A8Params& p, int cus, hipStream_t stream) {
    // eight waves share K when there is at most a workgroup per CU and K is long, else four
    const bool wide = tiles_of(p, 32, 32) <= cus && p.k >= 2048;
    // activation rows are fetched eight at a time: up to 8 rows need one fetch per tile, up to 32 four
    if (p.m <= 8) return wide ? launch_skinny<1, 1, 8, 3>(p, stream) : launch_skinny<1, 1, 4, 3>(p, stream);
    return wide ? launch_skinny<1, 4, 8, 2>(p, stream) : launch_skinny<1, 4, 4, 2>(p, stream);
}

// ---------------------------------------------------------------------------------------------
// The weights expanded to int8 once: w8 (N, K) row-major, the layout the int8 x int8 kernel reads.
// One thread = 32 codes (16 packed bytes in, 32 bytes out), with the same expansion as the fused kernel.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void w4_expand_kernel(QaGemmW4A8Params p, int8_t* w8) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int per_row = p.k / 32;
    if (idx >= static_cast<int64_t>(p.n) * per_row) return;
    const int n = static_cast<int>(idx / per_row), piece = static_cast<int>(idx % per_row);
    const uint4 v = *reinterpret_cast<const uint4*>(p.w_packed + static_cast<int64_t>(n) * (p.k / 2) + piece * 16);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    uint2 e[4];
    if (p.group_size > 0) {
        const __half sc = static_cast<const __half*>(p.s_group)[static_cast<int64_t>(piece / 4) * p.n + n];
        const __half2 s2 = __half2half2(sc);
#pragma unroll
        for (int t = 0; t < 4; ++t) e[t] = expand_grouped(w[t], s2);
    } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) e[t] = expand_per_channel(w[t]);
    }
    int8_t* dst = w8 + static_cast<int64_t>(n) * p.k + piece * 32;
    *reinterpret_cast<uint4*>(dst) = make_uint4(e[0].x, e[0].y, e[1].x, e[1].y);
    *reinterpret_cast<uint4*>(dst + 16) = make_uint4(e[2].x, e[2].y, e[3].x, e[3].y);
}

// Which kernel a product without transposed output takes: the one whose cost, in microseconds as measured over 16 .. 4096
// rows of 768 .. 18560 columns and K from 768 to 8192, is the least.  A launch goes in rounds of one workgroup per CU, and
// r workgroups on the busiest CU take a fixed time and one that grows with r per 128 of K; the kernels differ in the size of
// their tiles - large ones expand each code fewer times, small ones spread over the chip earlier - and the weights expanded
// once, in a pass of their own, cost that pass.
enum Way { kWaySplit, kWay64x64, kWay64x128, kWay128x128, kWay192x128, kWayExpandOnce };
struct WayChoice {
    int way;
    double us;
    void offer(int w, double cost) {
        if (cost < us) *this = {w, cost};
    }
};

WayChoice cheapest_tile(int m, int n, int k, int cus) {
    const double k_tiles = k / 128;
    auto rounds = [&](int64_t bm, int64_t bn) { return static_cast<double>((((m + bm - 1) / bm) * ((n + bn - 1) / bn) + cus - 1) / cus); };
    WayChoice best = {kWay128x128, 1e30};
    best.offer(kWay64x64, 3.0 + k_tiles * (0.10 + 0.28 * rounds(64, 64)));
    best.offer(kWay64x128, 3.0 + k_tiles * (0.08 + 0.42 * rounds(64, 128)));
    best.offer(kWay128x128, 3.0 + k_tiles * std::max(0.73, 0.10 + 0.57 * rounds(128, 128)));
    best.offer(kWay192x128, 3.0 + k_tiles * (0.05 + 0.84 * rounds(192, 128)));
    return best;
}

int cheapest_way(const QaGemmW4A8Params& p, int cus, const SplitChoice& split, bool expandable) {
    WayChoice best = cheapest_tile(p.m, p.n, p.k, cus);
    if (split.shape >= 0) best.offer(kWaySplit, split.us);
    if (expandable) {
        // (the int8 x int8 kernel's own estimate up to a round of its 128 x 256 tiles, see there, with weights that come from the
        // pass before: 777 x 2560 x 5120 takes 6.6 + 21.4 us; a round of 192 x 128 there against one here 2000 x 2560 x 5120 36.4 and 39.1,
        // 2500 x 2048 x 4096 29.1 and 32.1, 3300 x 1536 x 3072 23.5 and 25.4; beyond, 3600 x 4096 x 1024 5.6 + 17.8, 26.0 in 128 x 128 tiles,
        // 8800 x 3072 x 768 5.5 + 26.3 and 33.9)
        const double rounds = static_cast<double>((tiles_of(p, 256, 256) + cus - 1) / cus);
        const double w8 = tiles_of(p, 128, 256) <= cus ? tiles_us_w8(p.m, p.n, p.k, cus) + 0.6 : 2.4 + 1.55 * rounds * (p.k / 128);
        best.offer(kWayExpandOnce, 5.1 + static_cast<double>(p.n) * p.k / 3.1e6 + w8);
    }
    return best.way;
}

}  // namespace

float tiles_us_w4(int m, int n, int k, int cus) { return static_cast<float>(cheapest_tile(m, n, k, cus).us); }

}  // namespace qa

extern "C" int qa_gemm_w4a8(const QaGemmW4A8Params* p, void* stream_) {
    using namespace qa;
    if (!p) return QA_ERR_NULL;
    if (p->m < 0 || p->n < 0 || p->k < 0) return QA_ERR_SHAPE;
    const bool empty = p->m == 0 || p->n == 0;                      // (an output without elements: tensors may be null)
    if (!empty && (!p->a || !p->w_packed || !p->s_channel || !p->s_token || !p->d)) return QA_ERR_NULL;
    if (p->group_size != 128 && p->group_size != -1) return QA_ERR_UNSUPPORTED;
    if (!empty && p->group_size == 128 && !p->s_group) return QA_ERR_NULL;
    if (p->out_type != QA_OUT_I8 && p->out_type != QA_OUT_F16) return QA_ERR_UNSUPPORTED;
    if (p->tok_scale_numel != 1 && p->tok_scale_numel != p->m) return QA_ERR_SHAPE;
    if (p->k % 128 != 0) return QA_ERR_SHAPE;                       // whole 128-code groups / k tiles
    if (p->lda % 16 != 0 || p->lda < p->k || !aligned16(p->a) || !aligned16(p->w_packed)) return QA_ERR_STRIDE;
    if (p->ldd < (p->output_transpose ? p->m : p->n)) return QA_ERR_STRIDE;
    if (p->m == 0 || p->n == 0) return QA_OK;
    if (static_cast<int64_t>(p->m) * p->lda >= 0x70000000LL) return QA_ERR_SHAPE;
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const bool addressable = static_cast<int64_t>(p->n) * (p->k / 2) < 0x70000000LL;
    const int64_t w8_bytes = static_cast<int64_t>(p->n) * p->k;
    const bool expandable = p->w8_workspace && p->w8_workspace_bytes >= w8_bytes && aligned16(p->w8_workspace) && w8_bytes < 0x70000000LL;
    const int cus = compute_units();
    if (p->output_transpose && p->m <= 64 && addressable) return dispatch_skinny(*p, cus, stream);
    if (!p->output_transpose) {
        GemvParams g = {};
        g.m = p->m; g.n = p->n; g.k = p->k; g.bits = 4;
        g.out_type = p->out_type;
        g.rule = kGemvRowOuter;
        g.row_numel = p->tok_scale_numel; g.col_numel = p->n;
        g.lda = p->lda; g.ldw = p->k / 2; g.ldd = p->ldd;
        g.a = p->a; g.w = p->w_packed; g.s_group = p->group_size == 128 ? static_cast<const __half*>(p->s_group) : nullptr;
        g.row_scale = p->s_token; g.col_scale = p->s_channel; g.d = p->d;
        if (gemv_is_faster(4, p->m, p->n, p->k) && g.s_group && p->n % 4 == 0 && (reinterpret_cast<uintptr_t>(p->s_group) & 7u) == 0) return gemv_launch(g, nullptr, stream);
        const SplitChoice split = split_addressable_w4(p->n, p->k) ? split_choice(4, p->m, p->n, p->k, cus) : SplitChoice{-1, 0.0f, 0.0f};
        const int way = cheapest_way(*p, cus, split, expandable);
        if (way == kWaySplit) return split_launch_w4(g, split.shape, nullptr, stream);
        if (way == kWay64x64) return p->out_type == QA_OUT_I8 ? launch_tile<QA_OUT_I8>(*p, stream) : launch_tile<QA_OUT_F16>(*p, stream);
        if (way == kWay64x128) return launch_reg<2, 4, 256>(*p, stream);
        if (way == kWay128x128) return launch_reg<4, 4, 128>(*p, stream);
        if (way == kWay192x128) return launch_reg<6, 4, 128>(*p, stream);
    }
    if (expandable && (!p->output_transpose || p->n > 64)) {
        int8_t* w8 = static_cast<int8_t*>(p->w8_workspace);
        const int64_t threads = static_cast<int64_t>(p->n) * (p->k / 32);
        hipLaunchKernelGGL(w4_expand_kernel, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0, stream, *p, w8);
        // (acc * s_channel[n]) * s_token[m] and s_token[m] * (s_channel[n] * acc) round the same two products
        QaGemmW8A8Params q = {};
        q.k = p->k; q.ldd = p->ldd; q.d = p->d;
        q.out_type = p->out_type;
        q.round_mode = QA_ROUND_RNE;
        if (!p->output_transpose) {
            q.m = p->m; q.n = p->n;
            q.lda = p->lda; q.ldw = p->k;
            q.a = p->a; q.w = w8;
            q.a_scale = p->s_token; q.a_scale_numel = p->tok_scale_numel;
            q.w_scale = p->s_channel; q.w_scale_numel = p->n;
        } else {
            // the (N,M) output is the product with the operands' roles exchanged; the column scale (the
            // token's) is then applied last, which keeps the association s_token * (s_channel * acc)
            q.m = p->n; q.n = p->m;
            q.lda = p->k; q.ldw = p->lda;
            q.a = w8; q.w = p->a;
            q.a_scale = p->s_channel; q.a_scale_numel = p->n;
            q.w_scale = p->s_token; q.w_scale_numel = p->tok_scale_numel;
            q.scale_order = 1;
        }
        return qa_gemm_w8a8(&q, stream_);
    }
    return p->out_type == QA_OUT_I8 ? launch_reg_one<4, 4, 128, QA_OUT_I8, true>(*p, stream) : launch_reg_one<4, 4, 128, QA_OUT_F16, true>(*p, stream);
}
