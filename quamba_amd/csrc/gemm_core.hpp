// Shared int8-MFMA GEMM core for the W8A8 and W4A8 linears (gfx950).
//
//   acc[m,n] = sum_k a[m,k] * w[n,k]   (int32)      a: (M,K) int8, K-contiguous
//   d[m,n]   = cast(s_row[m|0] * (s_col[n|0] * float(acc)))          w: (N,K) int8, K-contiguous (W8A8)
//                                                                       or 4-bit codes + group scales (W4A8)
// Structure: WGM x WGN waves per workgroup, each wave TM x TN blocks of 32 x 32 (v_mfma_i32_32x32x32_i8, or
// v_mfma_i32_16x16x64_i8 in the main loop of tiles of 128 x 128 and more, see RotatedMma); block
// tile (WGM*TM*32) x (WGN*TN*32) x 128 k-bytes.  The k extent of 128 bytes is one full cache line
// per operand row: measured on MI355X, 64-byte row pieces halve the L1 load rate.  Operand tiles live
// in LDS as rows of eight 16-byte chunks, the chunk index XOR-swizzled with bits 1..3 of the row
// (measured conflict-free for the 32-row x 16-byte fragment reads).  int8 operands go global -> LDS
// directly (buffer_load ... lds, 16 bytes per lane, out-of-range lanes deliver zeros), so no
// registers are spent on staging and the next tile is in flight while the current one is multiplied.
// The 4-bit operand passes through registers, is expanded to int8 there and stored to the same
// layout.  The weight fragment is the MFMA "A" operand, so a lane ends up with four consecutive
// output columns of one row; the epilogue scales, converts, stages through LDS (privately per wave)
// and writes 16-byte pieces of output rows (or of output columns for the transposed layout).
#pragma once
#include "qa_common.hpp"

namespace qa {
namespace gemm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

constexpr int kBK = 128;                 // k-bytes per tile row
constexpr int kChunks = kBK / 16;        // 16-byte chunks per tile row
constexpr int kRsrcFlags = 0x00020000;   // raw buffer, 32-bit data format

__device__ __forceinline__ int swz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

// s_waitcnt immediate for "at most n vector-memory operations outstanding" (gfx9 encoding),
// leaving the LDS/scalar and export counters unconstrained.
__host__ __device__ constexpr int vmcnt_imm(int n) { return (n & 0xf) | ((n >> 4) << 14) | (0x7 << 4) | (0xf << 8); }

// round (half-even or half-away) and saturate to int8, returned in the low byte of an int
__device__ __forceinline__ int quant8(float v, int round_mode) {
    const float r = round_mode == QA_ROUND_RNE ? __builtin_rintf(v) : __builtin_roundf(v);
    // med3 returns -128 for NaN inputs as min(max(r,-128),127) would
    return static_cast<int>(__builtin_amdgcn_fmed3f(r, -128.0f, 127.0f));
}

// Four values -> four int8 bytes (round half to even, saturating) in one word.  Clamping to the
// integers -128 and 127 first does not change the rounded result; adding 1.5 * 2^23 then rounds to
// nearest-even in the addition itself and leaves the two's-complement byte in the low 8 bits.  The additions of the
// second to fourth value write that low byte straight into its place in the word (sub-dword destination select,
// the other bytes preserved), so no byte permutes are needed.
__device__ __forceinline__ uint32_t pack4_rne_sat8(float v0, float v1, float v2, float v3) {
    const float magic = 12582912.0f;
    const float c1 = __builtin_amdgcn_fmed3f(v1, -128.0f, 127.0f), c2 = __builtin_amdgcn_fmed3f(v2, -128.0f, 127.0f);
    const float c3 = __builtin_amdgcn_fmed3f(v3, -128.0f, 127.0f);
    uint32_t word = __float_as_uint(__builtin_amdgcn_fmed3f(v0, -128.0f, 127.0f) + magic);   // byte 0; bytes 1..3 replaced below
    asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(word) : "v"(c1), "v"(magic));
    asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_2 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(word) : "v"(c2), "v"(magic));
    asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_3 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(word) : "v"(c3), "v"(magic));
    return word;
}

// Two fp32 values -> two 16-bit floats of the output type (round to nearest even) in one word; bf16 rounds on the
// bit pattern: add 0x7fff plus the lowest kept bit, keep the high half (NaN payloads are not preserved).
__device__ __forceinline__ uint32_t bf16_bits(float v) {
    const uint32_t u = __float_as_uint(v);
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}
template <int OUT>
__device__ __forceinline__ uint32_t pack2_f16_or_bf16(float v0, float v1) {
    if (OUT == QA_OUT_BF16) return bf16_bits(v0) | (bf16_bits(v1) << 16);
    const __half2 h = __floats2half2_rn(v0, v1);
    return *reinterpret_cast<const uint32_t*>(&h);
}
template <int OUT>
__device__ __forceinline__ uint16_t one_f16_or_bf16(float v) {
    if (OUT == QA_OUT_BF16) return static_cast<uint16_t>(bf16_bits(v));
    const __half h = __float2half(v);
    return *reinterpret_cast<const uint16_t*>(&h);
}

struct Epilogue {
    int use_alpha;            // d = cast(alpha * acc)
    float alpha;
    int round_mode;           // QaRound
    int col_outer;            // d = cast(s_col * (s_row * acc)) instead of s_row * (s_col * acc)
    int64_t ldd;
    void* d;
};

template <int TM, int TN, int WGM, int WGN, int STAGES>
struct Cfg {
    static constexpr int kWaves = WGM * WGN;
    static constexpr int kThreads = 64 * kWaves;
    static constexpr int kBM = WGM * TM * 32;
    static constexpr int kBN = WGN * TN * 32;
    static constexpr int kAInstr = kBM * kChunks / kThreads;   // direct-to-LDS loads per thread per tile
    static constexpr int kWInstr = kBN * kChunks / kThreads;
    static constexpr int kStageBytes = (kBM + kBN) * kBK;
    static constexpr int kLdsBytes = STAGES * kStageBytes;
};

// Output tile of workgroup `linear`.  Workgroups go to the eight XCDs (each with an L2 of its own) in turn by linear
// index, and with one workgroup per CU a launch runs in rounds of 256.  The tiles an XCD works on at the same time
// should share operand panels, so that its L2 fetches each panel once per round: the 32 workgroups an XCD gets in a
// round take 32 consecutive positions of an order that walks the tile grid in bands of BAND m-tiles, n-tile by
// n-tile - a block of BAND x 32/BAND tiles, whatever the tile counts are (the natural m-first order does that only
// when the number of m-tiles is a multiple of eight).  BAND is 4 or 8, whichever makes the block's operand rows
// (BAND BM + 32/BAND BN) fewer.  The workgroups past the last full round keep the band order as it is.
template <int BM, int BN>
__device__ __forceinline__ void tile_of_workgroup(int linear, int tiles_m, int tiles_n, int& tm, int& tn) {
    constexpr int kXcds = 8, kPerXcd = 32, kRound = kXcds * kPerXcd, kBand = BN > BM ? 8 : 4;
    const int tiles = tiles_m * tiles_n;
    int g = linear;
    if (linear < tiles / kRound * kRound) {
        const int xcd = linear % kXcds, pos = linear / kXcds;
        g = ((pos / kPerXcd) * kXcds + xcd) * kPerXcd + pos % kPerXcd;
    }
    const int per_band = kBand * tiles_n;
    const int band = g / per_band, in_band = g % per_band;
    const int rows = min(kBand, tiles_m - band * kBand);          // the last band may be narrower
    tm = band * kBand + in_band % rows;
    tn = in_band / rows;
}

// Raw buffer descriptor (base, stride 0, num_records bytes) held in four scalar registers.
__device__ __forceinline__ v4i make_rsrc(const void* base, int num_bytes) {
    const uint64_t addr = reinterpret_cast<uint64_t>(base);
    v4i r;
    r.x = __builtin_amdgcn_readfirstlane(static_cast<int>(addr & 0xffffffffu));
    r.y = __builtin_amdgcn_readfirstlane(static_cast<int>((addr >> 32) & 0xffffu));
    r.z = __builtin_amdgcn_readfirstlane(num_bytes);
    r.w = __builtin_amdgcn_readfirstlane(kRsrcFlags);
    return r;
}

// 16 bytes per lane from buffer offset `voff` straight into LDS at lds_addr + lane*16 (lds_addr is
// wave-uniform; `soff`, also uniform, is added to the offset); lanes whose offset is outside the buffer deliver zeros.  Written as assembly so
// that the vector-memory counter stays under this kernel's control: a tile's loads stay in flight
// during the arithmetic and are waited for with an explicit s_waitcnt just before the barrier.
__device__ __forceinline__ void buffer_load_lds_b128(v4i rsrc, uint32_t lds_addr, int voff, int soff = 0) {
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory");
}

// The same with 4 bytes per lane.
__device__ __forceinline__ void buffer_load_lds_b32(v4i rsrc, uint32_t lds_addr, int voff) {
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, 0 offen lds"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(rsrc)
                 : "memory");
}

__device__ __forceinline__ uint32_t lds_offset_of(const void* p) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t)p));
}

// Per-lane addressing of one int8 operand tile (ROWS x 128 bytes) for the direct-to-LDS loads:
// instruction g = j*waves + wave fills LDS bytes [g*1024, +1024) of the tile, lane l the slot
// g*64 + l = (row, physical chunk); the lane fetches the logical chunk that the swizzle maps there.
template <int INSTR>
struct TileLoader {
    int voff[INSTR];     // byte offset at k0 = 0 (0x70000000 for rows outside the matrix)
    int kc[INSTR];       // k offset of the chunk inside the tile
    template <int WAVES>
    __device__ __forceinline__ void init(int row0, int rows_total, int64_t ld, int wave, int lane) {
#pragma unroll
        for (int j = 0; j < INSTR; ++j) {
            const int slot = (j * WAVES + wave) * 64 + lane, row = slot / kChunks, c = swz(row, slot % kChunks);
            kc[j] = c * 16;
            voff[j] = row0 + row < rows_total ? static_cast<int>((row0 + row) * ld) + c * 16 : 0x70000000;
        }
    }
    template <int WAVES>
    __device__ __forceinline__ void issue_one(int j, v4i rsrc, int k0, int k_end, uint32_t dst, int wave) const {
        const int off = (k0 + kc[j] < k_end) ? voff[j] + k0 : 0x7ffffff0;
        buffer_load_lds_b128(rsrc, dst + (j * WAVES + wave) * 1024, off);
    }
    // a tile whose 128 bytes all lie inside K
    template <int WAVES>
    __device__ __forceinline__ void issue_whole(int j, v4i rsrc, int k0, uint32_t dst, int wave) const {
        buffer_load_lds_b128(rsrc, dst + (j * WAVES + wave) * 1024, voff[j], k0);
    }
    template <int WAVES>
    __device__ __forceinline__ void issue(v4i rsrc, int k0, int k_end, uint32_t dst, int wave) const {
#pragma unroll
        for (int j = 0; j < INSTR; ++j) {
            const int off = (k0 + kc[j] < k_end) ? voff[j] + k0 : 0x7ffffff0;
            buffer_load_lds_b128(rsrc, dst + (j * WAVES + wave) * 1024, off);
        }
    }
};

// Accumulates one 128-byte k tile of one 32 x 32 block with the instruction order pinned: sa / sw point at this wave's rows of
// the staged operands.  A lone multiplication per step does not cover the time its fragments take: three of the four steps'
// are requested ahead of the first one, the last behind it in program order, and `hook(step)` runs after every multiplication:
// the caller places its global -> LDS requests for the next tile there, one at a time, so that the wave never waits on a full
// memory queue with multiplications behind it in program order.  sched_barrier keeps the compiler from regrouping.
template <class Hook>
__device__ __forceinline__ void mma_tile_paced(const uint8_t* sa, const uint8_t* sw, int frow, int fhalf, v16i& acc, Hook&& hook) {
    constexpr int kSteps = kBK / 32, kAhead = 3;
    v4i fa[kSteps], fw[kSteps];
    auto fetch = [&](int kk) {
        const int at = frow * kBK + swz(frow, kk * 2 + fhalf) * 16;
        fw[kk] = *reinterpret_cast<const v4i*>(sw + at);
        fa[kk] = *reinterpret_cast<const v4i*>(sa + at);
    };
#pragma unroll
    for (int kk = 0; kk < kAhead; ++kk) fetch(kk);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk < kSteps; ++kk) {
        if (kk + kAhead < kSteps) fetch(kk + kAhead);
        __builtin_amdgcn_sched_barrier(0);
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fw[kk], fa[kk], acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        hook(kk);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The main loop of the large tiles, on v_mfma_i32_16x16x64_i8.  These launches run at the power limit of the part - their
// clock is what the energy of a multiplication leaves - and registers full of random int8 operands multiply at 4.0 POP/s
// with this shape against 3.3 with 32x32x32 (both 4.9 with zeros): half as many accumulators are read and written per product.
//
// A k tile of 128 bytes is two steps of 64.  Of the two operands' fragments (16 rows x 64 bytes) a wave keeps the smaller
// set, `held`, for a whole step and walks through the other one, a fragment at a time with all held ones: `Walk` is true when
// the w operand is walked.  A walked fragment is fetched three positions ahead into a ring of four, the held ones of the next
// step during the last three positions of a step, each fetch behind a multiplication of its own - fetched in a block
// between the steps they left the matrix pipe idle (256 x 256 tiles, K 8192: 158900 -> 144000 cycles).  The barrier
// stands where the last fetch from this tile's stage has been made, three positions before the end: there the wave waits for its own
// global -> LDS requests and meets the others, so the next tile's stage is complete and this one may be overwritten.
// IN_FLIGHT: requests, the last ones made, that need not be complete at the barrier (those of tiles after the next).
// `hook(idx)` runs after every multiplication, idx counted from the barrier, through kPerTile; the caller places its
// requests behind the multiplications it chooses.
// Against 32x32x32 with block fetches (rows x outputs x K, us): 16384 x 18560 x 4096 1030 -> 965, 16384 x 4096 x 8192
// 434 -> 388, 16384 x 10240 x 2560 375 -> 333.  Four waves of 128 x 128 instead of eight of 128 x 64 or so read a third less from
// LDS, but one wave per SIMD does not hide its own requests: 520 us where the eight take 388.
template <int TM, int TN>
struct RotatedMma {
    static constexpr bool kWalkW = TN > TM;
    static constexpr int kHeld = 2 * (kWalkW ? TM : TN), kWalk = 2 * (kWalkW ? TN : TM), kRing = 4, kAhead = 3;
    static constexpr int kPerTile = 2 * kWalk * kHeld, kBehindBarrier = kAhead * kHeld;     // multiplications
    static_assert(2 * kWalk % kRing == 0 && kAhead < kWalk && kHeld <= kAhead * (kHeld - 1), "the order of the fetches");
    v4i acc[2 * TN][2 * TM];      // lane l: row 16 j + (l & 15), columns 16 i + 4 (l >> 4) + 0..3
    v4i held[2][kHeld], ring[kRing];
    int at;                       // this lane's 16 bytes of fragment 0, step 0, in a stage's rows

    __device__ __forceinline__ void init(int lane) {
        at = (lane & 15) * kBK + swz(lane & 15, lane >> 4) * 16;
#pragma unroll
        for (int i = 0; i < 2 * TN; ++i)
#pragma unroll
            for (int j = 0; j < 2 * TM; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    }
    // step 1 is four chunks further, which the swizzle turns into an exchange of bit 6
    __device__ __forceinline__ v4i fragment(const uint8_t* rows, int step, int f) const {
        return *reinterpret_cast<const v4i*>(rows + ((at ^ (step * 64)) + f * 16 * kBK));
    }
    // sa / sw: this wave's rows of the first tile's stage
    __device__ __forceinline__ void start(const uint8_t* sa, const uint8_t* sw) {
#pragma unroll
        for (int h = 0; h < kHeld; ++h) held[0][h] = fragment(kWalkW ? sa : sw, 0, h);
#pragma unroll
        for (int g = 0; g < kAhead; ++g) ring[g] = fragment(kWalkW ? sw : sa, 0, g);
    }
    template <int IN_FLIGHT, class Hook>
    __device__ __forceinline__ void tile(const uint8_t* sa, const uint8_t* sw, const uint8_t* na, const uint8_t* nw, Hook&& hook) {
        const uint8_t* const h0 = kWalkW ? sa : sw;
        const uint8_t* const h1 = kWalkW ? na : nw;
        const uint8_t* const w0 = kWalkW ? sw : sa;
        const uint8_t* const w1 = kWalkW ? nw : na;
#pragma unroll
        for (int g = 0; g < 2 * kWalk; ++g) {
            const int step = g / kWalk, pos = g % kWalk, from_end = kWalk - pos;
            if (g == 2 * kWalk - kAhead) {
                __builtin_amdgcn_s_waitcnt(vmcnt_imm(IN_FLIGHT));
                __syncthreads();
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int h = 0; h < kHeld; ++h) {
                const int x = g % 2 ? kHeld - 1 - h : h;               // there and back: one operand stays at every turn, 0.7 % of the time
                v4i& c = kWalkW ? acc[pos][x] : acc[x][pos];
                c = __builtin_amdgcn_mfma_i32_16x16x64_i8(kWalkW ? ring[g % kRing] : held[step][x], kWalkW ? held[step][x] : ring[g % kRing], c, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (h == 0) {
                    const int n = g + kAhead;
                    ring[n % kRing] = n < 2 * kWalk ? fragment(w0, n / kWalk, n % kWalk) : fragment(w1, 0, n - 2 * kWalk);
                } else if (from_end <= kAhead) {
                    const int f = (kAhead - from_end) * (kHeld - 1) + h - 1;
                    if (f < kHeld) held[1 - step][f] = step == 0 ? fragment(h0, 1, f) : fragment(h1, 0, f);
                }
                hook((g * kHeld + h + kBehindBarrier) % kPerTile);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
};

// Orders this wave's LDS writes before its later LDS reads (the staging area is private to the
// wave, and one wave's LDS operations execute in order, so no workgroup barrier is needed).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The scales of a workgroup's tile, BN column scales and BM row scales, fetched into LDS in front of everything else: loaded
// where they are used, they cost the end of every tile two memory round trips and, with a scale per column, 150 instructions
// of addresses.  (One scale for all columns or rows is read into each of its places; rows and columns outside read zero.)
template <int BM, int BN, int WAVES>
struct TileScales {
    static constexpr int kBytes = (BM + BN) * 4;
    static_assert(BM % 64 == 0 || BM == 32, "whole requests");
    // call once before the first tile's requests; complete with them
    static __device__ __forceinline__ void request(uint32_t lds_addr, const float* row_scale, int row_numel, int m, int m0, const float* col_scale, int col_numel, int n, int n0, int wave, int lane) {
        constexpr int kCols = BN / 64, kRows = (BM + 63) / 64;
        const v4i rsrc_c = make_rsrc(col_scale, (col_numel == 1 ? 1 : n) * 4), rsrc_r = make_rsrc(row_scale, (row_numel == 1 ? 1 : m) * 4);
#pragma unroll
        for (int i = 0; i < kCols + kRows; ++i) {
            if (i % WAVES != wave) continue;
            if (i < kCols) buffer_load_lds_b32(rsrc_c, lds_addr + i * 256, col_numel == 1 ? 0 : (n0 + i * 64 + lane) * 4);
            else buffer_load_lds_b32(rsrc_r, lds_addr + BN * 4 + (i - kCols) * 256, row_numel == 1 ? 0 : (m0 + (i - kCols) * 64 + lane) * 4);
        }
    }
};

// Accumulators as the two matrix instructions leave them, seen as quads: in quad u of row block b a lane holds four
// consecutive output columns, from column_of(u), of row row_of() of the block.  Of 32x32x32: acc[i][j], row l & 31 of block
// j, columns i*32 + 8*(r/4) + 4*(l/32) + (r%4) in register r; of 16x16x64: acc[i][j], row l & 15, columns i*16 + 4*(l/16) + r.
template <class V>
struct QuadView {
    static constexpr int kRows = sizeof(V) == 16 ? 16 : 32, kQuadsPer = sizeof(V) / 16;
    template <int NI, int NJ>
    static __device__ __forceinline__ float value(const V (&acc)[NI][NJ], int u, int b, int t) { return static_cast<float>(acc[u / kQuadsPer][b][u % kQuadsPer * 4 + t]); }
    static __device__ __forceinline__ int row_of(int lane) { return lane & (kRows - 1); }
    static __device__ __forceinline__ int column_of(int u, int lane) { return kRows == 16 ? u * 16 + 4 * (lane >> 4) : u / 4 * 32 + 8 * (u % 4) + 4 * (lane >> 5); }
};

// FLEX = false compiles the common rule only (d = cast_rne(s_row * (s_col * acc))); FLEX = true also
// honours use_alpha and the round-half-away GEMV rule at run time.  TRANS selects the (N,M) output.
// COL_OUTER (the column scale applied last) is a compile-time choice: selecting the association per
// element costs two extra instructions on each of the 128 outputs of a lane.
// s_lds: the scales of the workgroup's tile in LDS (TileScales), this wave's first row and column at row_at and col_at.
template <int TM, int TN, int OUT, bool FLEX, bool TRANS, bool COL_OUTER = false, class V, int NI, int NJ>
__device__ __forceinline__ void epilogue(const Epilogue& e, V (&acc)[NI][NJ], uint8_t* lds, int m, int n,
                                         int wave_m0, int wave_n0, int wave, int lane, const float* s_lds, int row_at, int col_at) {
    using Q = QuadView<V>;
    constexpr int kElt = OUT == QA_OUT_I8 ? 1 : 2, kQuads = TN * 32 / (256 / Q::kRows) , kRowBlocks = TM * 32 / Q::kRows;
    static_assert(NI * Q::kQuadsPer == kQuads && NJ == kRowBlocks, "accumulators of another tile");
    const bool vec_ok = (e.ldd * kElt) % 16 == 0 && aligned16(e.d);
    const bool use_alpha = FLEX && e.use_alpha;
    const bool away = FLEX && e.round_mode == QA_ROUND_HALF_AWAY;
    const int round_mode = FLEX ? e.round_mode : QA_ROUND_RNE;

    float s_col[kQuads][4];
#pragma unroll
    for (int u = 0; u < kQuads; ++u) {
        const float4 v = *reinterpret_cast<const float4*>(s_lds + col_at + Q::column_of(u, lane));
        s_col[u][0] = v.x; s_col[u][1] = v.y; s_col[u][2] = v.z; s_col[u][3] = v.w;
    }
    float s_row[kRowBlocks];
#pragma unroll
    for (int b = 0; b < kRowBlocks; ++b) s_row[b] = use_alpha ? e.alpha : s_lds[row_at + b * Q::kRows + Q::row_of(lane)];
    auto scaled = [&](int u, int b, int t) -> float {
        const float accf = Q::value(acc, u, b, t);
        float v;
        if (use_alpha) v = s_row[b] * accf;
        // GEMV rule (round-half-away mode): the two scales are multiplied first
        else if (COL_OUTER) v = s_col[u][t] * (s_row[b] * accf);
        else v = away ? (s_col[u][t] * s_row[b]) * accf : s_row[b] * (s_col[u][t] * accf);
        // keep the fp32 product a value of its own: folding the multiply into a mixed-precision
        // convert would round once instead of twice and change the fp16 result in rare cases
        asm volatile("" : "+v"(v));
        return v;
    };

    if constexpr (!TRANS) {
        constexpr int kPitch = TN * 32 * kElt + 16;
        uint8_t* stg = lds + wave * (32 * kPitch);
        // a tile that lies inside the output altogether: no bounds to look at, 32-bit offsets from one address
        const bool whole = vec_ok && wave_m0 + TM * 32 <= m && wave_n0 + TN * 32 <= n && e.ldd * kElt < (1 << 23);
        uint8_t* const first = static_cast<uint8_t*>(e.d) + (static_cast<int64_t>(wave_m0) * e.ldd + wave_n0) * kElt;
        const uint32_t row_bytes = static_cast<uint32_t>(e.ldd * kElt);
#pragma unroll
        for (int j = 0; j < TM; ++j) {
#pragma unroll
            for (int sub = 0; sub < 32 / Q::kRows; ++sub) {
                const int b = j * (32 / Q::kRows) + sub, row = sub * Q::kRows + Q::row_of(lane);
#pragma unroll
                for (int u = 0; u < kQuads; ++u) {
                    const int nl = Q::column_of(u, lane);
                    const float v0 = scaled(u, b, 0), v1 = scaled(u, b, 1);
                    const float v2 = scaled(u, b, 2), v3 = scaled(u, b, 3);
                    if (OUT == QA_OUT_I8) {
                        uint32_t word;
                        if (!away) {
                            word = pack4_rne_sat8(v0, v1, v2, v3);
                        } else {
                            const uint32_t b0 = quant8(v0, round_mode) & 0xff, b1 = quant8(v1, round_mode) & 0xff;
                            const uint32_t b2 = quant8(v2, round_mode) & 0xff, b3 = quant8(v3, round_mode);
                            word = b0 | (b1 << 8) | (b2 << 16) | (b3 << 24);
                        }
                        *reinterpret_cast<uint32_t*>(stg + row * kPitch + nl) = word;
                    } else {
                        uint2 pk;
                        pk.x = pack2_f16_or_bf16<OUT>(v0, v1);
                        pk.y = pack2_f16_or_bf16<OUT>(v2, v3);
                        *reinterpret_cast<uint2*>(stg + row * kPitch + nl * 2) = pk;
                    }
                }
            }
            wave_lds_sync();
            constexpr int kPiecesPerRow = TN * 32 * kElt / 16;
            if (whole) {
#pragma unroll
                for (int piece = lane; piece < 32 * kPiecesPerRow; piece += 64) {
                    const uint32_t r = piece / kPiecesPerRow, cb = (piece % kPiecesPerRow) * 16;
                    *reinterpret_cast<uint4*>(first + ((j * 32 + r) * row_bytes + cb)) = *reinterpret_cast<const uint4*>(stg + r * kPitch + cb);
                }
                wave_lds_sync();
                continue;
            }
#pragma unroll
            for (int piece = lane; piece < 32 * kPiecesPerRow; piece += 64) {
                const int r = piece / kPiecesPerRow, cb = (piece % kPiecesPerRow) * 16;
                const int mm2 = wave_m0 + j * 32 + r;
                const int nn = wave_n0 + cb / kElt;
                if (mm2 >= m || nn >= n) continue;
                uint8_t* dst = static_cast<uint8_t*>(e.d) + (static_cast<int64_t>(mm2) * e.ldd + nn) * kElt;
                const uint4 val = *reinterpret_cast<const uint4*>(stg + r * kPitch + cb);
                if (vec_ok && nn + 16 / kElt <= n) {
                    *reinterpret_cast<uint4*>(dst) = val;
                } else {
                    const uint8_t* src = reinterpret_cast<const uint8_t*>(&val);
                    const int nbytes = min(16, (n - nn) * kElt);
                    for (int t = 0; t < nbytes; ++t) dst[t] = src[t];
                }
            }
            wave_lds_sync();
        }
    } else {
        // transposed output d[n][m]: stage 32 columns n x (TM*32) rows m per pass
        static_assert(Q::kRows == 32, "only of 32x32x32");
        const int frow = lane & 31, fhalf = lane >> 5;
        constexpr int kPitch = TM * 32 * kElt + 16;
        uint8_t* stg = lds + wave * (32 * kPitch);
#pragma unroll
        for (int i = 0; i < TN; ++i) {
#pragma unroll
            for (int j = 0; j < TM; ++j) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const int nl = 8 * q + 4 * fhalf + t;          // column inside this 32-column tile
                        const float v = scaled(i * 4 + q, j, t);
                        if (OUT == QA_OUT_I8) {
                            *reinterpret_cast<int8_t*>(stg + nl * kPitch + j * 32 + frow) =
                                static_cast<int8_t>(quant8(v, round_mode));
                        } else {
                            *reinterpret_cast<uint16_t*>(stg + nl * kPitch + (j * 32 + frow) * 2) = one_f16_or_bf16<OUT>(v);
                        }
                    }
                }
            }
            wave_lds_sync();
            constexpr int kPiecesPerRow = TM * 32 * kElt / 16;
#pragma unroll
            for (int piece = lane; piece < 32 * kPiecesPerRow; piece += 64) {
                const int r = piece / kPiecesPerRow, cb = (piece % kPiecesPerRow) * 16;
                const int nn = wave_n0 + i * 32 + r;
                const int mm2 = wave_m0 + cb / kElt;
                if (nn >= n || mm2 >= m) continue;
                uint8_t* dst = static_cast<uint8_t*>(e.d) + (static_cast<int64_t>(nn) * e.ldd + mm2) * kElt;
                const uint4 val = *reinterpret_cast<const uint4*>(stg + r * kPitch + cb);
                if (vec_ok && mm2 + 16 / kElt <= m) {
                    *reinterpret_cast<uint4*>(dst) = val;
                } else {
                    const uint8_t* src = reinterpret_cast<const uint8_t*>(&val);
                    const int nbytes = min(16, (m - mm2) * kElt);
                    for (int t = 0; t < nbytes; ++t) dst[t] = src[t];
                }
            }
            wave_lds_sync();
        }
    }
}

// Largest epilogue staging footprint (fp16, either orientation) must fit in the operand stages.
template <int TM, int TN, int WAVES>
constexpr int epilogue_lds_bytes() {
    return WAVES * 32 * ((TM > TN ? TM : TN) * 32 * 2 + 16);
}

// Tile of workgroup `linear`, row blocks of BM by column blocks of BN.  With many column blocks the row blocks of one of
// them go to one XCD (eight workgroups apart), whose L2 then holds their weights.
template <int BM, int BN = BM>
__device__ __forceinline__ void split_tile_of_workgroup(int linear, int m, int n, int& m0, int& n0) {
    const int blocks_m = (m + BM - 1) / BM, blocks_n = (n + BN - 1) / BN, whole = blocks_n / 8 * 8 * blocks_m;
    if (linear < whole) {
        n0 = ((linear / (8 * blocks_m)) * 8 + linear % 8) * BN;
        m0 = (linear / 8) % blocks_m * BM;
    } else {
        const int rest = linear - whole, columns = blocks_n % 8;
        n0 = (blocks_n / 8 * 8 + rest % columns) * BN;
        m0 = rest / columns * BM;
    }
}

}  // namespace gemm
}  // namespace qa
