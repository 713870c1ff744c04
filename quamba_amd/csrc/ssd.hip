// Mamba2 quantized SSD chunk scan (prefill) for gfx950.
//
// Stages and arithmetic follow the reference's Triton pipeline (quamba/triton/quant_ssd_combined.py
// :61-77, grouped :146-162); see each kernel for the file it restates.  fp16 operands rounded where the
// reference rounds them, fp32 accumulation, as there; the one pure int8 contraction (C B^T) runs on the
// int8 matrix cores inside the chunk scan and stays in fp32 registers.
//   cumsum      dt = clamp(softplus(s_dt q_dt + dt_bias)), dA_cs = within-chunk cumsum(dt * A)
//   state       S_c[p,n] = sum_k f16(x^[k,p]) f16(B^[k,n] exp(dA_last - dA_k) dt_k)   (fp16 MFMA)
//               P_0 = 0, P_{c+1} = exp(dA_last,c) P_c + S_c in registers; P_c stored in fp16; final state fp32 / int8
//   chunk_scan  CB[m,k] = (s_C s_B) * sum_n q_C[m,n] q_B[k,n]                       (int8 MFMA, at and below the diagonal)
//               y[m,p] = exp(dA_m) sum_n f16(C^[m,n]) f16(P_c[p,n]) + sum_{k<=m} f16(CB[m,k] e^{dA_m-dA_k} dt_k) f16(x^[k,p])
//               + D x^[m,p], optional z gate, fp16 out                               (fp16 MFMA)
// Both fp16 contractions over the time index need x (and B) with time as the fastest-moving index,
// while memory has channels fastest; the tiles are transposed once on the way into LDS and then read as
// 16-byte MFMA operands.
#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>

#include "mixer_common.hpp"
#include "ssd_common.hpp"

namespace qa {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kP = 64;          // head dimension of these kernels
__device__ __forceinline__ float fexp(float x) { return ssd_exp(x); }
__device__ __forceinline__ int8_t byte_of(uint32_t w, int j) { return static_cast<int8_t>((w >> (8 * j)) & 0xffu); }

// ---------------------------------------------------------------------------------------------
// Stage 1 (quamba/triton/quant_chunk_cumsum.py:56-70).  A workgroup takes kCumHeads heads of one chunk.  Memory has the heads
// of a step side by side and the steps a row of the projection apart, so a thread fetches all its heads of one step at
// once and hands them through LDS to the waves, one head each at 256 steps: there a lane has chunk_size/64 consecutive
// steps, and an inclusive scan runs across the lanes.  With a wave per head that gathers its own steps every load touches
// 64 lines for a byte each.  The tables per channel are written by workgroups of their own in front, one wave per
// head: their walk over the groups is as long as the rest and stood in front of it in the waves of the first chunk.
// 4 x 4096 steps of 80 heads 12.7 -> 10.8 us, 1 x 1531 of 80 7.4 -> 5.7 us, 16 x 1024 of 128 17.7 -> 16.5 us,
// of which the softplus (130 instructions for 64 steps) is about 9.
// ---------------------------------------------------------------------------------------------
constexpr int kCumHeads = 4;

// the step size of an int8 code with its bias
__device__ __forceinline__ float step_size(const QaSsdParams& p, float s_dt, int8_t code, float bias) {
    float v = s_dt * static_cast<float>(code) + bias;
    if (p.dt_softplus) v = v <= 20.0f ? log1pf(expf(v)) : v;
    return fminf(fmaxf(v, p.dt_min), p.dt_max);
}
__device__ __forceinline__ float decay_rate(const QaSsdParams& p, int h) { return -expf(*p.A_log_scale * static_cast<float>(p.A_log[h])); }
// In a whole wave, a lane with E consecutive step sizes of a chunk: the inclusive sums of dt A from the chunk's start.
template <int E>
__device__ __forceinline__ void chunk_cumsum(const float (&dtv)[E], float A, int lane, float (&cs)[E]) {
    float local = 0.0f;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        local += dtv[e] * A;
        cs[e] = local;
    }
    // exclusive prefix of the lane totals
    float incl = local;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const float up = __shfl_up(incl, off);
        if (lane >= off) incl += up;
    }
    const float before = incl - local;
#pragma unroll
    for (int e = 0; e < E; ++e) cs[e] = before + cs[e];
}

template <int Q>
__global__ __launch_bounds__(Q) void ssd_cumsum_kernel(QaSsdParams p, float* dt_out, float* dA_out, float* xs_out, int32_t* srow_out, int nc) {
    constexpr int E = Q / 64;                          // steps per lane, and waves
    __shared__ __align__(16) float dt_s[kCumHeads][Q];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int table_groups = (p.nheads + E - 1) / E;
    const int item = static_cast<int>(blockIdx.x) - table_groups;
    if (item < 0) {
        const int h = blockIdx.x * E + wave;
        if (h < p.nheads) ssd_write_channel_tables(p, h, lane, xs_out, srow_out);
        return;
    }
    const int bc = item % (p.batch * nc), h0 = item / (p.batch * nc) * kCumHeads;
    const int b = bc / nc, c = bc % nc;
    {
        const int t = c * Q + static_cast<int>(threadIdx.x);
        const int64_t di = (static_cast<int64_t>(b) * p.seqlen + min(t, p.seqlen - 1)) * ssd_dt_stride(p) + h0;
        float v[kCumHeads], bias[kCumHeads];
        // asked for together with the steps: behind the branches of the softplus each would be a wait of its own
#pragma unroll
        for (int j = 0; j < kCumHeads; ++j) {
            bias[j] = !p.dt_is_fp32 && p.dt_bias ? __half2float(static_cast<const __half*>(p.dt_bias)[min(h0 + j, p.nheads - 1)]) : 0.0f;
        }
        if (p.dt_is_fp32) {
#pragma unroll
            for (int j = 0; j < kCumHeads; ++j) v[j] = h0 + j < p.nheads ? static_cast<const float*>(p.dt)[di + j] : 0.0f;
        } else {
            const int8_t* q = static_cast<const int8_t*>(p.dt);
            uint32_t w = 0;
            if (((reinterpret_cast<uintptr_t>(q) | static_cast<unsigned>(ssd_dt_stride(p)) | static_cast<unsigned>(p.nheads)) & 3u) == 0) {
                w = *reinterpret_cast<const uint32_t*>(q + di);
            } else {
#pragma unroll
                for (int j = 0; j < kCumHeads; ++j) w |= h0 + j < p.nheads ? static_cast<uint32_t>(static_cast<uint8_t>(q[di + j])) << (8 * j) : 0u;
            }
            const float s_dt = *p.dt_scale;
#pragma unroll
            for (int j = 0; j < kCumHeads; ++j) v[j] = step_size(p, s_dt, byte_of(w, j), bias[j]);
        }
#pragma unroll
        for (int j = 0; j < kCumHeads; ++j) dt_s[j][threadIdx.x] = t < p.seqlen ? v[j] : 0.0f;
    }
    float A[(kCumHeads + E - 1) / E];
#pragma unroll
    for (int j = wave, i = 0; i < static_cast<int>(sizeof(A) / 4); j += E, ++i) A[i] = decay_rate(p, min(h0 + j, p.nheads - 1));
    __syncthreads();
#pragma unroll
    for (int i = 0; i < static_cast<int>(sizeof(A) / 4); ++i) {
        const int j = wave + i * E, h = h0 + j;
        if (h >= p.nheads) return;
        float dtv[E], run[E];
#pragma unroll
        for (int e = 0; e < E; ++e) dtv[e] = dt_s[j][lane * E + e];
        chunk_cumsum<E>(dtv, A[i], lane, run);
        const int64_t row = ((static_cast<int64_t>(b) * p.nheads + h) * nc + c) * Q + lane * E;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            dt_out[row + e] = dtv[e];
            dA_out[row + e] = run[e];
        }
    }
}

// ---------------------------------------------------------------------------------------------
// The fp16 contractions run on v_mfma_f32_16x16x32_f16 with the operands rounded to fp16 where the reference
// rounds them, so that the products agree and only the order of the fp32 sums differs:
//   S_c[p,n] = sum_k f16(x^[k,p]) f16(B^[k,n] exp(dA_last - dA_k) dt_k);   P_{c+1} = exp(dA_last) P_c + S_c
//   y[m,p]   = exp(dA_m) sum_n f16(C^[m,n]) f16(P_c[p,n])                                  (term 1)
//            + sum_{k<=m} f16(CB[m,k] exp(dA_m - dA_k) dt_k) f16(x^[k,p])                  (term 2)
//            + x^[m,p] D, optional z gate, fp16 out
// Both contractions over the time index need x with time as the fastest-moving index, while memory has channels
// fastest.  A thread transposes 4x4 blocks on the way into LDS: four dword loads (sixteen lanes cover the 64
// bytes of a row), four 8-byte stores.  The rows of the transposed tile are kept in the order
//   slot(p) = 16 (p % 4) + p / 4
// so that the sixteen lanes of one store write sixteen neighbouring rows (all banks, instead of every fourth row)
// and an MFMA tile, sixteen neighbouring rows, holds the channels p = 4 i + tile (i = 0..15): a lane then owns
// four neighbouring channels of an output row, which leave as one 8-byte store without passing through LDS.
// int8 values enter as biased bytes u = q + 128 (one xor per dword): s q = fma(u, s, -128 s) exactly, with the
// byte-to-float conversion in a single instruction.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ v4f mfma16(v8h a, v8h b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ float ubyte_of(uint32_t w, int j) { return static_cast<float>((w >> (8 * j)) & 0xffu); }
// float(int8 byte j of w) in one instruction (left to itself the compiler shifts and sign-extends the byte out first)
__device__ __forceinline__ float sbyte_of(uint32_t w, int j) {
    float r;
    switch (j) {
        case 0: asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(r) : "v"(w)); break;
        case 1: asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(r) : "v"(w)); break;
        case 2: asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(r) : "v"(w)); break;
        default: asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(r) : "v"(w)); break;
    }
    return r;
}
// fp16 of a value that is an fp32 number already.  The empty asm separates the conversion from the multiplication that made the
// value: where the compiler merges the two into a mixed-precision instruction the exact product is rounded once, which is another
// number at some ties, and which of the kernels' values it does so with changes with the code around them.
__device__ __forceinline__ _Float16 rounded(float v) {
    asm("" : "+v"(v));
    return static_cast<_Float16>(v);
}
constexpr uint32_t kBias = 0x80808080u;
__device__ __forceinline__ uint32_t word_of(const uint4& v, int d) { return d == 0 ? v.x : d == 1 ? v.y : d == 2 ? v.z : v.w; }
__device__ __forceinline__ float lane_of(const float4& v, int d) { return d == 0 ? v.x : d == 1 ? v.y : d == 2 ? v.z : v.w; }

// A thread's share of a chunk's x tile, steps 4 kb .. 4 kb + 3 of the CH (8 or 16) channels from c0 on (four loads of as many
// bytes), goes to the transposed fp16 tile: CH 8-byte stores, rows in slot order.
template <int CH>
struct XShare { uint32_t w[CH / 4]; };
template <int CH>
__device__ __forceinline__ XShare<CH> load_x_share(const int8_t* from) {
    XShare<CH> r;
    if constexpr (CH == 16) {
        const uint4 v = *reinterpret_cast<const uint4*>(from);
        r.w[0] = v.x; r.w[1] = v.y; r.w[2] = v.z; r.w[3] = v.w;
    } else {
        const uint2 v = *reinterpret_cast<const uint2*>(from);
        r.w[0] = v.x; r.w[1] = v.y;
    }
    return r;
}
// Where the transposed x tile of both kernels has its 16-byte pieces: rows without a pad, the pieces exchanged by the row, so that the
// rows of an operand read (and of the transposing stores) fall into different banks.
template <int Q>
struct XPlaces {
    static __device__ __forceinline__ int turn(int row) { return Q == 64 ? (row >> 1) & 7 : row & 15; }
    static __device__ __forceinline__ int x_at(int row, int piece) { return row * Q + ((piece ^ turn(row)) << 3); }
    // piece 4 ks + lq of a row from piece lq < 4: exchanged within sixteen (eight) pieces, past those further on
    static constexpr int kPieces = Q == 64 ? 8 : 16;
    static constexpr int x_turned(int ks) { return 4 * ks % kPieces * 8; }
    static constexpr int x_past(int ks) { return 4 * ks / kPieces * kPieces * 8; }
};

// `put(row, v)`: the four steps of a row of that tile
template <int CH, class Put>
__device__ __forceinline__ void stage_x_share(const XShare<CH> (&xr)[4], const float* xs, int c0, Put&& put) {
#pragma unroll
    for (int d = 0; d < CH / 4; ++d) {
        const float4 s4 = *reinterpret_cast<const float4*>(xs + c0 + 4 * d);
        const uint32_t w0 = xr[0].w[d] ^ kBias, w1 = xr[1].w[d] ^ kBias, w2 = xr[2].w[d] ^ kBias, w3 = xr[3].w[d] ^ kBias;
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            const float sc = lane_of(s4, cc), nsc = -128.0f * sc;
            v4h v;
            v[0] = rounded(__builtin_fmaf(ubyte_of(w0, cc), sc, nsc));
            v[1] = rounded(__builtin_fmaf(ubyte_of(w1, cc), sc, nsc));
            v[2] = rounded(__builtin_fmaf(ubyte_of(w2, cc), sc, nsc));
            v[3] = rounded(__builtin_fmaf(ubyte_of(w3, cc), sc, nsc));
            put(cc * 16 + c0 / 4 + d, v);                                                // row slot(c0 + 4 d + cc)
        }
    }
}

// Workgroup L of a launch whose units (things that share operands through L2) should stay on one XCD: L -> XCD
// L % 8, position L / 8 there; `parts` consecutive positions are the parts of one (unit, head).
__device__ __forceinline__ void unit_head_part(int linear, int units, int hpg, int parts, int& unit, int& head_in_group, int& part) {
    if (units % 8 == 0) {
        const int xcd = linear % 8, pos = linear / 8;
        part = pos % parts;
        unit = (pos / parts / hpg) * 8 + xcd;
        head_in_group = (pos / parts) % hpg;
    } else {
        part = linear % parts;
        unit = linear / parts / hpg;
        head_in_group = (linear / parts) % hpg;
    }
}

// ---------------------------------------------------------------------------------------------
// Stages 2, 3 and 6 (quamba/triton/quant_chunk_state.py:76-89, quant_state_passing.py:60-83, quant_ssm_states.py
// :43,119): a workgroup of N / 16 waves per (batch, head) walks the chunks in order with the running state P
// (64 x N of headdim x dstate, fp32) in registers; the fp32 chunk states never travel
// through memory.  A wave owns 16 columns n and all rows p.  Its B operand, f16((s_B q_B[k,n]) w_k) with the
// per-head weight w_k = exp(dA_last - dA_k) dt_k, is built in registers from the transposed int8 B tile in LDS
// (8-byte reads); its A operand is the transposed x tile; both tiles are laid out against the banks (0.84 to 0.90 conflict cycles per
// active one are left, of 2.1).  The tiles of chunk c+1 are fetched into
// registers while chunk c is multiplied.  The state entering chunk c >= 1 is stored as fp16, rows in slot order.
// Bound by vector issue (converting x and B to fp16 operands) and by the LDS reads of the x tile, which every wave makes: with
// one workgroup for all N columns x is staged once: as a workgroup per 64 columns 16 x 1024 steps of 128 heads took 146 us, so
// 129; with the tiles padded by a piece a row (half of the LDS's busy cycles were conflicts) 129 -> 124, 4 x 4096 steps of 80 heads 104 -> 97, 1531
// steps 14.7 -> 13.4.  (Four waves of 32 columns instead of eight of 16 read x half as often and take 138: too few waves for the latencies
// of a chunk.  With s_B in the weight, q_B (s_B w_k), a product less per value: 128, but at fp16 ties another value than the
// reference's; the general kernels round the same one.)
// ---------------------------------------------------------------------------------------------
template <int N, int Q>
struct StateSmem : XPlaces<Q> {
    // A 16-byte read takes lanes 0 .. 3, 12 .. 15 and 20 .. 27 together, the other half of those 32 next: rows 0 .. 3 and 12 .. 15 of one piece
    // with rows 4 .. 11 of its neighbour.  Rows of x have no pad; their pieces are exchanged by the row, which keeps both halves apart
    // (and the transposing stores).  Rows of B are shifted by eight words and by four more past the eighth.
    static constexpr int BP = Q + 32;       // bytes per row of the transposed B tile
    __attribute__((aligned(16))) _Float16 xt[kP * Q];
    __attribute__((aligned(16))) int8_t b8[N * BP + N / 8 * 16];
    static __device__ __forceinline__ int b_at(int row, int k) { return row * BP + (row >> 3) * 16 + k; }
    __attribute__((aligned(16))) float w[Q];
    __attribute__((aligned(16))) float xs[kP];    // x scale per channel
    int32_t srow[kP];                             // the channel's row of the grouped state scales
};

template <int N, int Q, bool WALK>
__global__ __launch_bounds__(4 * N, N == 128 ? 4 : 3) void ssd_state_kernel(QaSsdParams p, float* dt_ws, float* dA_ws, __half* prev, float* sums, float* xs_ws,
                                                                              int32_t* srow_ws, int nc, int own_steps) {
    using S = StateSmem<N, Q>;
    extern __shared__ __attribute__((aligned(16))) unsigned char ssd_smem_raw[];
    S& sm = *reinterpret_cast<S*>(ssd_smem_raw);
    constexpr int kThreads = 4 * N;
    constexpr int CH = N == 128 ? 8 : 16;                         // channels of a thread's share of x
    constexpr int kSharesX = Q / 4 * (kP / CH), kSharesB = Q / 4 * (N / 16);
    static_assert(kSharesX <= kThreads && kSharesB <= kThreads && Q <= kThreads, "a thread stages at most one share of the chunk's tiles");

    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);    // the same in every lane: kept in a scalar register
    // a head of 64 s channels runs as s heads of 64 that share the head's step sizes, decay and skip weight: H, h count
    // those; hp is the head itself and ch0 the first of its channels this workgroup covers
    const int split = p.headdim / kP;
    const int G = p.ngroups, H = p.nheads * split, L = p.seqlen;
    int unit, hig, part;
    unit_head_part(blockIdx.x, p.batch * (WALK ? 1 : nc) * G, H / G, 1, unit, hig, part);
    const int h = (unit % G) * (H / G) + hig;
    const int hp = h / split, ch0 = (h % split) * kP;
    const int b = WALK ? unit / G : unit / (G * nc), my_chunk = WALK ? 0 : unit / G % nc;
    const int g = hp / (p.nheads / G);
    const bool grouped = p.nhead_groups > 0;
    const float sB = grouped ? p.B_scale[g] : p.B_scale[0];
    const uint32_t xrow = static_cast<uint32_t>(H) * kP;          // bytes between steps of x
    const uint32_t brow = static_cast<uint32_t>(G) * N;           // bytes between steps of B
    const int64_t rows0 = (static_cast<int64_t>(b) * p.nheads + hp) * nc;
    // this thread's share of a chunk's tiles: steps 4 kb .. 4 kb + 3 of CH channels of x and of sixteen state columns of B
    const int xc = tid % (kP / CH) * CH, xkb = tid / (kP / CH), bc = tid % (N / 16) * 16, bkb = tid / (N / 16);
    const bool mine_x = kSharesX == kThreads || tid < kSharesX, mine_b = kSharesB == kThreads || tid < kSharesB;
    const uint32_t voff_x = static_cast<uint32_t>(4 * xkb) * xrow + xc, voff_b = static_cast<uint32_t>(4 * bkb) * brow + bc;
    const bool steps_made = WALK || !own_steps;                   // step sizes, their sums and the tables: by ssd_cumsum_kernel
    if (steps_made && tid < kP) {
        sm.xs[tid] = xs_ws[hp * p.headdim + ch0 + tid];
        sm.srow[tid] = srow_ws[hp * p.headdim + ch0 + tid];
    }
    XShare<CH> xr[4];
    uint4 br[4];
    float r_dt = 0.0f, r_dA = 0.0f, r_last = 0.0f;
    int valid_loaded = Q;                                         // steps of the chunk whose tiles are in xr / br
    // One path for whole and ragged chunks: rows past the end of the sequence read the last row (the loads stay inside
    // the tensors) and are zeroed when the chunk is staged.  With a second, ragged path beside it the compiler merges
    // the two sets of destination registers by copies right behind the loads, i.e. waits for them where they are issued.
    auto load_chunk = [&](int c) {
        const int t0 = c * Q;
        const int valid = min(Q, L - t0);
        valid_loaded = valid;
        // uniform row addresses plus one per-thread offset: the address arithmetic stays in scalar registers
        const int8_t* xsrc = p.x + (static_cast<int64_t>(b) * L + t0) * xrow + static_cast<int64_t>(h) * kP;
        const int8_t* bsrc = p.B + (static_cast<int64_t>(b) * L + t0) * brow + static_cast<int64_t>(g) * N;
        const uint32_t last_x = static_cast<uint32_t>(valid - 1) * xrow + xc, last_b = static_cast<uint32_t>(valid - 1) * brow + bc;
        if (mine_x) {
#pragma unroll
            for (int r = 0; r < 4; ++r) xr[r] = load_x_share<CH>(xsrc + static_cast<uint64_t>(min(voff_x + static_cast<uint32_t>(r) * xrow, last_x)));
        }
        if (mine_b) {
#pragma unroll
            for (int r = 0; r < 4; ++r) br[r] = *reinterpret_cast<const uint4*>(bsrc + static_cast<uint64_t>(min(voff_b + static_cast<uint32_t>(r) * brow, last_b)));
        }
        if (steps_made) {
            const float* dA_row = dA_ws + (rows0 + c) * Q;
            r_last = dA_row[Q - 1];
            if (Q == kThreads || tid < Q) {
                r_dt = dt_ws[(rows0 + c) * Q + tid];
                r_dA = dA_row[tid];
            }
        }
    };
    auto stage_chunk = [&]() {
        if (valid_loaded < Q) {
            // ragged last chunk: steps past the end of the sequence count as zero
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (4 * xkb + r >= valid_loaded) xr[r] = XShare<CH>{};
                if (4 * bkb + r >= valid_loaded) br[r] = make_uint4(0u, 0u, 0u, 0u);
            }
        }
        if (mine_x) stage_x_share<CH>(xr, sm.xs, xc, [&](int row, const v4h& v) { *reinterpret_cast<v4h*>(&sm.xt[S::x_at(row, xkb >> 1) + 4 * (xkb & 1)]) = v; });
        if (mine_b) {
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                // 4x4 byte transpose: rows k (registers) x columns n (bytes) -> rows n x bytes k
                const uint32_t r0 = word_of(br[0], d), r1 = word_of(br[1], d), r2 = word_of(br[2], d), r3 = word_of(br[3], d);
                const uint32_t lo01 = __builtin_amdgcn_perm(r1, r0, 0x05010400u);   // r0.b0 r1.b0 r0.b1 r1.b1
                const uint32_t hi01 = __builtin_amdgcn_perm(r1, r0, 0x07030602u);   // r0.b2 r1.b2 r0.b3 r1.b3
                const uint32_t lo23 = __builtin_amdgcn_perm(r3, r2, 0x05010400u);
                const uint32_t hi23 = __builtin_amdgcn_perm(r3, r2, 0x07030602u);
                const int n4 = bc + 4 * d;
                *reinterpret_cast<uint32_t*>(&sm.b8[S::b_at(n4 + 0, bkb * 4)]) = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
                *reinterpret_cast<uint32_t*>(&sm.b8[S::b_at(n4 + 1, bkb * 4)]) = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
                *reinterpret_cast<uint32_t*>(&sm.b8[S::b_at(n4 + 2, bkb * 4)]) = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
                *reinterpret_cast<uint32_t*>(&sm.b8[S::b_at(n4 + 3, bkb * 4)]) = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
            }
        }
        if (steps_made && tid < Q) sm.w[tid] = fexp(r_last - r_dA) * r_dt;   // weight of step k in the chunk's state
    };

    // the running state: columns n = 16 wave + lane % 16; tile j, register r: channel p = 4 (4 (lane / 16) + r) + j
    const int n_col = 16 * wave + l16;
    v4f run[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) run[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    // the final state in the requested form
    auto store_final = [&](const v4f (&state)[4]) {
        if (p.final_states) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int pp = 4 * (4 * lq + r) + j;
                    const int64_t fo = ((static_cast<int64_t>(b) * H + h) * kP + pp) * N + n_col;
                    const float sv = state[j][r];
                    if (p.final_state_is_fp32) {
                        static_cast<float*>(p.final_states)[fo] = sv;
                    } else {
                        static_cast<int8_t*>(p.final_states)[fo] = ssd_quantize_state(p, sm.srow[pp], n_col, sv);
                    }
                }
        }
    };

    load_chunk(my_chunk);
    if (!steps_made) {
        // The chunk's step sizes, their sums and the channels' scales, which this workgroup needs before anyone else does, while its
        // tiles are on their way
        constexpr int E = Q / 64;
        __builtin_amdgcn_sched_barrier(0);
        if (wave == kThreads / 64 - 1) {
            const SsdChannel e = ssd_channel(p, hp, lane, ch0);
            sm.xs[lane] = e.xs;
            sm.srow[lane] = e.srow;
            if (b == 0 && my_chunk == 0) {
                xs_ws[hp * p.headdim + ch0 + lane] = e.xs;
                srow_ws[hp * p.headdim + ch0 + lane] = e.srow;
            }
        }
        if (tid < Q) {
            const int t = my_chunk * Q + tid;
            const int64_t at = (static_cast<int64_t>(b) * L + min(t, L - 1)) * ssd_dt_stride(p) + hp;
            float v;
            if (p.dt_is_fp32) {
                v = static_cast<const float*>(p.dt)[at];
            } else {
                const float bias = p.dt_bias ? __half2float(static_cast<const __half*>(p.dt_bias)[hp]) : 0.0f;
                v = step_size(p, *p.dt_scale, static_cast<const int8_t*>(p.dt)[at], bias);
            }
            sm.w[tid] = t < L ? v : 0.0f;
        }
        __syncthreads();
        if (wave == 0) {
            float dtv[E], cs[E];
#pragma unroll
            for (int e = 0; e < E; ++e) dtv[e] = sm.w[lane * E + e];
            chunk_cumsum<E>(dtv, decay_rate(p, hp), lane, cs);
            const float last = __shfl(cs[E - 1], 63);
            const int64_t row = (rows0 + my_chunk) * Q + lane * E;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                sm.w[lane * E + e] = fexp(last - cs[e]) * dtv[e];
                if (h % split == 0) {
                    dt_ws[row + e] = dtv[e];
                    dA_ws[row + e] = cs[e];
                }
            }
        }
    } else {
        __syncthreads();                                          // the table of x scales
    }
    stage_chunk();
    float dA_last = r_last;                                       // of the chunk about to be multiplied
    __syncthreads();

    const int chunks = WALK ? nc : 1;
    for (int c = 0; c < chunks; ++c) {
        const bool more = c + 1 < chunks;
        // in flight during the products.  Unconditional (the last chunk is requested once more and never staged): a
        // conditional request leaves the tile registers with two possible sources, which the compiler merges by
        // copies right behind the loads, i.e. by waiting for them where they are issued
        if constexpr (WALK) load_chunk(min(c + 1, nc - 1));
        __builtin_amdgcn_sched_barrier(0);                         // (the scheduler would sink the requests below the products)
        v4f accs[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) accs[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        int x_first = S::x_at(l16, lq);
        asm("" : "+v"(x_first));                                   // (four addresses kept over the chunks are four registers spilled)
#pragma unroll
        for (int ks = 0; ks < Q / 32; ++ks) {
            const int k0 = 32 * ks + 8 * lq;
            const uint2 b01 = *reinterpret_cast<const uint2*>(&sm.b8[S::b_at(16 * wave + l16, k0)]);
            const uint32_t b0 = b01.x, b1 = b01.y;
            const float4 w0 = *reinterpret_cast<const float4*>(&sm.w[k0]), w1 = *reinterpret_cast<const float4*>(&sm.w[k0 + 4]);
            v8h fx[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) fx[j] = *reinterpret_cast<const v8h*>(&sm.xt[(x_first ^ S::x_turned(ks)) + S::x_past(ks) + j * 16 * Q]);
            const float wk[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
            v8h bw;
#pragma unroll
            for (int e = 0; e < 8; ++e) bw[e] = rounded((sB * sbyte_of(e < 4 ? b0 : b1, e & 3)) * wk[e]);
#pragma unroll
            for (int j = 0; j < 4; ++j) accs[j] = mfma16(fx[j], bw, accs[j]);
        }
        if constexpr (!WALK) {
            if (nc == 1) {                                         // the only chunk's sums are the final state
                store_final(accs);
                return;
            }
            float* to = sums + (((static_cast<int64_t>(b) * nc + my_chunk) * H + h) * kP) * N + n_col;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) to[(j * 16 + 4 * lq + r) * N] = accs[j][r];
            return;
        }
        // P <- exp(dA_last) P + S
        const float decay = fexp(dA_last);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) run[j][r] = decay * run[j][r] + accs[j][r];
        if (more) {
            // the state entering chunk c + 1, in fp16 as the reference keeps it, rows in slot order
            __half* pst = prev + (((static_cast<int64_t>(b) * nc + c + 1) * H + h) * kP) * N + n_col;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) pst[(j * 16 + 4 * lq + r) * N] = __float2half(run[j][r]);
        }
        __syncthreads();                                           // every wave has read this chunk's tiles
        if (more) {
            stage_chunk();
            dA_last = r_last;
        }
        __syncthreads();
    }

    store_final(run);
}

// The same with few heads in flight: a workgroup per chunk (WALK false) leaves the chunk's own sums S_c in memory as fp32, rows
// in slot order, and this kernel runs the recurrence over them, four states a thread: the same values in the same order.
// (Up to kChainChunks chunks the chunk scan does it itself; of one chunk the sums are the final state.)
template <int N>
__global__ __launch_bounds__(256) void ssd_pass_kernel(QaSsdParams p, const float* dA_ws, __half* prev, const float* sums, const int32_t* srow_ws, int nc) {
    constexpr int kPieces = kP * N / 4;                           // of one head of 64 channels
    const int split = p.headdim / kP, H = p.nheads * split;
    const unsigned bh = blockIdx.x / (kPieces / 256);
    const int piece = (blockIdx.x % (kPieces / 256)) * 256 + threadIdx.x;
    const int b = bh / H, h = bh % H, hp = h / split, ch0 = (h % split) * kP;
    const int slot = piece / (N / 4), n = piece % (N / 4) * 4;
    const int64_t step = static_cast<int64_t>(H) * kP * N, first = ((static_cast<int64_t>(b) * nc) * H + h) * kP * N + piece * 4;
    const float* dA = dA_ws + (static_cast<int64_t>(b) * p.nheads + hp) * nc * p.chunk_size + p.chunk_size - 1;
    constexpr int kAhead = 8;
    float4 s[kAhead];
    float d[kAhead];
    auto load = [&](int c, int at) {
        const int cc = min(c, nc - 1);
        s[at] = *reinterpret_cast<const float4*>(sums + first + cc * step);
        d[at] = dA[static_cast<int64_t>(cc) * p.chunk_size];
    };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) load(i, i);
    float4 run = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int c0 = 0; c0 < nc; c0 += kAhead) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int c = c0 + i;
            if (c < nc) {
                const float decay = fexp(d[i]);
                run.x = decay * run.x + s[i].x;
                run.y = decay * run.y + s[i].y;
                run.z = decay * run.z + s[i].z;
                run.w = decay * run.w + s[i].w;
                load(c + kAhead, i);
                if (c + 1 < nc) {
                    v4h o;
                    o[0] = static_cast<_Float16>(run.x); o[1] = static_cast<_Float16>(run.y);
                    o[2] = static_cast<_Float16>(run.z); o[3] = static_cast<_Float16>(run.w);
                    *reinterpret_cast<v4h*>(prev + first + (c + 1) * step) = o;
                }
            }
        }
    }
    if (p.final_states) {
        const int pp = 4 * (slot % 16) + slot / 16;
        const int64_t fo = ((static_cast<int64_t>(b) * H + h) * kP + pp) * N + n;
        if (p.final_state_is_fp32) {
            *reinterpret_cast<float4*>(static_cast<float*>(p.final_states) + fo) = run;
        } else {
            const int srow = srow_ws[hp * p.headdim + ch0 + pp];
            const float v[4] = {run.x, run.y, run.z, run.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) static_cast<int8_t*>(p.final_states)[fo + i] = ssd_quantize_state(p, srow, n + i, v[i]);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Stages 4 and 5 (quamba/triton/quant_bmm_chunk.py:60-66, quant_chunk_scan.py:96-171): a workgroup of eight waves takes some
// heads of one (batch, chunk, group) in turn.  A wave owns whole 16-row m-tiles with all 64 channels, a long and a short
// causal range each (with sixteen tiles: 15 - w and w).
// C B^T never exists in memory: the chunk's B codes sit in LDS, a lane holds 32 codes of its row of C, and
// v_mfma_i32_16x16x64_i8 forms (C B^T)^T in 16 x 16 blocks - exact integers.  A block comes out with a lane per row m and four
// consecutive steps k, which is how the next product wants its first operand: two blocks (steps 4 q .. 4 q + 3 and 16 + 4 q
// .. 16 + 4 q + 3 of a 32-step piece, q = lane / 16) are the eight values of a lane, and the x operand is read from LDS in
// the same order (the order of the summation index is free as long as both operands agree).  The same codes of C, dequantised
// to fp16, are the first operand of term 1; a lane's codes are states 64 i + 16 q .. + 15, and the entering state is read in
// that order.  Below the diagonal the decay factors into exp(dA_m - R) (one exp per lane and piece, times s_C s_B) and exp(R -
// dA_k) dt_k (a table per workgroup) with R = dA at the last step of the piece, so that both exponents are <= 0; on the piece
// that holds the diagonal it is computed per element, in the reference's order: s_C s_B times the integer, the value the
// reference's bmm kernel stores, times exp, times dt_k.  While a head's last tile is computed, what the next head needs from
// memory is on its way to registers.  Moving a head's bytes (the entering state and x in, y out) and computing it take about
// as long as each other: 89 us of each for 4 x 4096 steps of 80 heads with nothing else in the kernel, and as a workgroup per
// head, two to a CU, they ran half one after the other.  Walking heads overlaps them and reads the codes of B and C once for
// all: 158 -> 127 us, 16 x 1024 of 128 257 -> 213, 1 x 1531 of 80 (a head each, so only the shorter code) 21.4 -> 19.7.  The
// walk has to stay inside 128 registers: with the next head requested ahead of the first tile, or the reads of LDS gathered in
// front of the products, some values spill, and waiting for a spilled one is waiting for the requests: 144 to 177 us.
// Two workgroups fit a CU's LDS with 128 states and chunks of 256 steps because the entering state and x take the same place:
// term 1 of both tiles runs first, x is staged from its registers after it.
// ---------------------------------------------------------------------------------------------
template <int N, int Q>
struct ScanSmem : XPlaces<Q> {
    static constexpr int NCH = N / 8;       // 16-byte pieces per row of the entering state
    static constexpr int SWZ = (NCH < 16 ? NCH : 16) - 1;
    static constexpr int BSWZ = (N / 16 < 8 ? N / 16 : 8) - 1;
    // of the head at hand; the entering state first, then x.  The state's rows have no padding: piece c of row r sits
    // at position c ^ (r & SWZ), so that the sixteen rows of an operand read fall into different banks
    union {
        __attribute__((aligned(16))) _Float16 xt[kP * Q];
        __attribute__((aligned(16))) _Float16 prev[kP][N];
    };
    __attribute__((aligned(16))) int8_t bq[Q][N];   // B codes; 16-byte piece c of row k at position c ^ (k & BSWZ)
    __attribute__((aligned(16))) float dt[Q];
    __attribute__((aligned(16))) float dA[Q];
    __attribute__((aligned(16))) float gk[Q];   // exp(dA[end of the 32-step piece] - dA_k) dt_k
    __attribute__((aligned(16))) float xs[kP];  // x scale per channel
    __attribute__((aligned(16))) float Dv[kP];  // skip weight per channel
    __attribute__((aligned(16))) float gate[256];   // SiLU(z_scale code) of the gate's 256 codes, indexed by the code's byte
};

constexpr int scan_waves_of(int Q) { return Q / 16 < 8 ? Q / 16 : 8; }

// One head, some in turn, or one whose entering state the workgroup makes itself from the chunks' own sums (the first chunk's
// workgroup then leaves the final state).
enum ScanMode { kScanOne, kScanWalk, kScanChain };
// With few chunks a workgroup per chunk and head reads the sums of the chunks before its own faster than a launch of its own passes
// the states on (pass and scan against the scan alone, us: 6 chunks of 80 heads 27.2 -> 21.0, 4 of 128 27.5 -> 22.6, 8 of 48 24.1 ->
// 20.4, 2 of 80 15.5 -> 15.8 and a launch less to make).  What is read grows with the square of the chunks - 16 of 80 heads read 300 MB -
// and with heads to walk the sums would have no registers.
constexpr int kChainChunks = 8;

template <int N, int Q, ScanMode MODE>
__global__ __launch_bounds__(64 * scan_waves_of(Q), 4) void ssd_chunk_scan_kernel(QaSsdParams p, const float* dt_ws, const float* dA_ws, const __half* prev, const float* sums,
                                                                                const float* xs_ws, const int32_t* srow_ws, int nc, int heads_each) {
    using S = ScanSmem<N, Q>;
    extern __shared__ __attribute__((aligned(16))) unsigned char ssd_smem_raw[];
    S& sm = *reinterpret_cast<S*>(ssd_smem_raw);
    constexpr int kWaves = scan_waves_of(Q);
    constexpr int kThreads = 64 * kWaves;
    constexpr int NMT = Q / 16;                                   // 16-row m-tiles of a chunk
    constexpr int TILES = NMT / kWaves;                           // per wave: 2 (Q 256), 1 (Q 128, 64)
    constexpr int PPC = kP * N / 8;                               // 16-byte pieces of the entering state
    constexpr int PB = PPC / kThreads;
    constexpr int BPC = Q * N / 16;                               // 16-byte pieces of the B codes
    constexpr int BB = BPC / kThreads;
    constexpr int CH = 8;                                         // channels of a thread's share of x
    constexpr int kShares = Q / 4 * (kP / CH);
    static_assert(kShares <= kThreads && Q <= kThreads, "a thread stages at most one share of the x tile");
    static_assert(PPC % kThreads == 0 && BPC % kThreads == 0, "whole shares per thread");
    static_assert(TILES <= 2, "a long and a short tile per wave");

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);    // the same in every lane: kept in a scalar register
    // (H, h, hp, ch0 as in the state kernel: heads of 64 s channels run as s heads of 64)
    const int split = p.headdim / kP;
    const int G = p.ngroups, H = p.nheads * split, L = p.seqlen;
    // the heads of one (batch, chunk, ssd group) read the same B and C codes: they go to one XCD.  Not where a workgroup reads
    // the chunks before its own: the last chunk's would all draw on one XCD's share of the memory
    int unit, unused, part;
    const int parts = (H / G + heads_each - 1) / heads_each;
    if constexpr (MODE == kScanChain) {
        unit = blockIdx.x / parts;
        part = blockIdx.x % parts;
    } else {
        unit_head_part(blockIdx.x, p.batch * nc * G, 1, parts, unit, unused, part);
    }
    const int g = unit % G;
    const int c = (unit / G) % nc;
    const int b = unit / (G * nc);
    const int h_first = g * (H / G) + part * heads_each, h_last = min(h_first + heads_each, (g + 1) * (H / G)) - 1;
    const bool grouped = p.nhead_groups > 0;
    const float sC = grouped ? p.C_scale[g] : p.C_scale[0];
    const float cb_scale = sC * (grouped ? p.B_scale[g] : p.B_scale[0]);
    const int t0 = c * Q;
    const int lim = min(Q, L - t0);
    const uint32_t xrow = static_cast<uint32_t>(H) * kP;          // bytes between steps of x
    const uint32_t crow = static_cast<uint32_t>(G) * N;           // bytes between steps of B and C
    const int64_t row0 = (static_cast<int64_t>(b) * L + t0) * xrow;
    const int8_t* Bbase = p.B + (static_cast<int64_t>(b) * L + t0) * crow + static_cast<int64_t>(g) * N;
    const int8_t* Cbase = p.C + (static_cast<int64_t>(b) * L + t0) * crow + static_cast<int64_t>(g) * N;
    const float D_scale = p.D ? *p.D_scale : 0.0f;
    const float z_scale = p.z ? *p.z_scale : 0.0f;

    // tile s of this wave
    auto tile_of = [&](int s) { return (s & 1) == 0 ? NMT - 1 - 8 * (s / 2) - wave : 8 * ((TILES - 1 - s) / 2) + wave; };

    // what a head needs from memory, fetched into registers while the head before it is computed.  Unconditional (the
    // last head is requested once more and never staged), and one path for whole and ragged chunks: rows past the end of
    // the sequence read the last row and are zeroed when the tile is staged.  With a second path beside it the compiler
    // merges the two sets of destination registers by copies right behind the loads, i.e. waits for them there.
    float r_dt = 0.0f, r_dA = 0.0f, r_xs = 0.0f, r_D = 0.0f;
    v4i r_prev[PB];
    // A lane's two groups of steps of a 32-step piece, 4 q and 16 + 4 q, share 16 bytes of the x tile: one read instead of two of 8 bytes,
    // and neighbouring threads store the two halves of a place.  (Against rows with a pad: 16 x 1024 steps of 128 heads 217 -> 209 us, 4 x
    // 4096 of 80 135 -> 134; the layers of 1531, 2 x 700 and 300 steps 1 %.  With the exchange but two reads of 8 bytes, which no longer
    // share an address: 228 and 144.)
    auto steps_of = [](int t) { return (t & ~7) | (t & 1) << 2 | (t & 6) >> 1; };
    XShare<CH> xr[4];                                             // steps 4 kb .. 4 kb + 3, channels xc .. xc + 7
    auto fetch_head = [&](int h, int tid) {
        const int xc = tid % (kP / CH) * CH, kb = steps_of(tid / (kP / CH));
        const int hp = h / split, ch0 = (h % split) * kP;
        if (Q == kThreads || tid < Q) {
            const int64_t row = ((static_cast<int64_t>(b) * p.nheads + hp) * nc + c) * Q;
            r_dt = dt_ws[row + tid];
            r_dA = dA_ws[row + tid];
        }
        if (tid < kP) {
            r_xs = xs_ws[hp * p.headdim + ch0 + tid];
            if (p.D) r_D = static_cast<float>(p.D_has_hdim ? p.D[hp * p.headdim + ch0 + tid] : p.D[hp]);
        }
        if constexpr (MODE != kScanChain) {
            // (the first chunk has no entering state: its slot of the workspace is read all the same and never used)
            const __half* pst = prev + ((static_cast<int64_t>(b) * nc + c) * H + h) * kP * N;
#pragma unroll
            for (int i = 0; i < PB; ++i) r_prev[i] = *reinterpret_cast<const v4i*>(pst + (tid + i * kThreads) * 8);
        }
        if (kShares == kThreads || tid < kShares) {
            const int8_t* from = p.x + row0 + static_cast<int64_t>(h) * kP;
            const uint32_t last_x = static_cast<uint32_t>(lim - 1) * xrow + xc, voff_x = static_cast<uint32_t>(4 * kb) * xrow + xc;
#pragma unroll
            for (int r = 0; r < 4; ++r) xr[r] = load_x_share<CH>(from + static_cast<uint64_t>(min(voff_x + static_cast<uint32_t>(r) * xrow, last_x)));
        }
    };

    // states 8 (tid + i kThreads) .. + 7 of the state entering chunk `end`, rows in slot order: the recurrence of ssd_pass_kernel, the
    // same values in the same order
    auto chain = [&](float (&run)[PB][8], int tid, int end) {
        constexpr int kAtOnce = 4;                                 // chunks requested together
        const int64_t step = static_cast<int64_t>(H) * kP * N;
        const float* from = sums + ((static_cast<int64_t>(b) * nc) * H + h_first) * kP * N + tid * 8;
        const float* dA_last = dA_ws + (static_cast<int64_t>(b) * p.nheads + h_first / split) * nc * Q + Q - 1;
#pragma unroll
        for (int i = 0; i < PB; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) run[i][e] = 0.0f;
        for (int c0 = 0; c0 < end; c0 += kAtOnce) {
            float4 sum[kAtOnce][PB][2];
            float d[kAtOnce];
#pragma unroll
            for (int k = 0; k < kAtOnce; ++k) {
                const int cc = min(c0 + k, end - 1);
                d[k] = dA_last[static_cast<int64_t>(cc) * Q];
#pragma unroll
                for (int i = 0; i < PB; ++i)
#pragma unroll
                    for (int q = 0; q < 2; ++q) sum[k][i][q] = *reinterpret_cast<const float4*>(from + cc * step + i * (8 * kThreads) + 4 * q);
            }
#pragma unroll
            for (int k = 0; k < kAtOnce; ++k) {
                if (c0 + k >= end) break;
                const float decay = fexp(d[k]);
#pragma unroll
                for (int i = 0; i < PB; ++i)
#pragma unroll
                    for (int e = 0; e < 8; ++e) run[i][e] = decay * run[i][e] + lane_of(sum[k][i][e / 4], e % 4);
            }
        }
    };

    // codes of C of this lane's rows: states 64 i + 16 q .. + 15 (rows past the end of the sequence read the last
    // row; nothing of theirs is stored)
    v4i cq[TILES][N / 64];
    {
        // every global read of the prologue is issued before the first LDS write, so that the workgroup waits once
        const int tid = threadIdx.x, l16 = tid & 15, lq = (tid & 63) >> 4;
        v4i r_b[BB];
#pragma unroll
        for (int i = 0; i < BB; ++i) {
            const int piece = tid + i * kThreads, k = piece / (N / 16), col = piece % (N / 16);
            r_b[i] = *reinterpret_cast<const v4i*>(Bbase + static_cast<uint32_t>(min(k, lim - 1)) * crow + 16 * col);
        }
#pragma unroll
        for (int s = 0; s < TILES; ++s) {
            const int8_t* cp = Cbase + static_cast<uint32_t>(min(tile_of(s) * 16 + l16, lim - 1)) * crow + 16 * lq;
#pragma unroll
            for (int i = 0; i < N / 64; ++i) cq[s][i] = *reinterpret_cast<const v4i*>(cp + 64 * i);
        }
        fetch_head(h_first, tid);
        if constexpr (MODE == kScanChain) {
            float run[PB][8];
            chain(run, tid, c);
#pragma unroll
            for (int i = 0; i < PB; ++i) {
                v8h o;
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = static_cast<_Float16>(run[i][e]);
                r_prev[i] = __builtin_bit_cast(v4i, o);
            }
        }
        if (p.z) {
            // the gate has 256 possible values: evaluated once per workgroup, looked up per output
            for (int i = tid; i < 256; i += kThreads) {
                const float zv = z_scale * static_cast<float>(static_cast<int8_t>(i));
                sm.gate[i] = zv * __builtin_amdgcn_rcpf(1.0f + fexp(-zv));
            }
        }
#pragma unroll
        for (int i = 0; i < BB; ++i) {
            const int piece = tid + i * kThreads, k = piece / (N / 16), col = piece % (N / 16);
            *reinterpret_cast<v4i*>(&sm.bq[k][(col ^ (k & S::BSWZ)) * 16]) = r_b[i];
        }
    }

    for (int h = h_first; h <= h_last; ++h) {
        const int8_t* xbase = p.x + row0 + static_cast<int64_t>(h) * kP;
        const int8_t* zbase = p.z + row0 + static_cast<int64_t>(h) * kP;       // only read if p.z
        // (opaque: the addresses of a head's steps, kept from head to head, are more than the registers hold, and so are the codes
        // of C as fp16)
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, l16 = lane & 15, lq = lane >> 4;
#pragma unroll
        for (int s = 0; s < TILES; ++s)
#pragma unroll
            for (int i = 0; i < N / 64; ++i) asm volatile("" : "+v"(cq[s][i]));
        __half* out = static_cast<__half*>(p.out) + row0 + static_cast<int64_t>(h) * kP;
        if (tid < kP) {
            sm.xs[tid] = r_xs;
            sm.Dv[tid] = D_scale * r_D;
        }
        if (tid < Q) {
            sm.dt[tid] = r_dt;
            sm.dA[tid] = r_dA;
            sm.gk[tid] = fexp(__shfl(r_dA, lane | 31) - r_dA) * r_dt;
        }
#pragma unroll
        for (int i = 0; i < PB; ++i) {
            const int piece = tid + i * kThreads, pr = piece / (N / 8), col = (piece % (N / 8)) * 8;
            *reinterpret_cast<v4i*>(&sm.prev[pr][col ^ ((pr & S::SWZ) * 8)]) = r_prev[i];
        }
        __syncthreads();

        // term 1 of every tile of the wave: C^ (rows m) x entering state (rows p), zero for the first chunk
        v4f acc[TILES][4];
#pragma unroll
        for (int s = 0; s < TILES; ++s) {
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[s][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            if (c > 0) {
                const int m0 = tile_of(s) * 16;
#pragma unroll
                for (int ks = 0; ks < N / 32; ++ks) {
                    const uint32_t w0 = static_cast<uint32_t>(cq[s][ks / 2][2 * (ks % 2)]), w1 = static_cast<uint32_t>(cq[s][ks / 2][2 * (ks % 2) + 1]);
                    v8h cf;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        cf[e] = rounded(sC * sbyte_of(w0, e));
                        cf[4 + e] = rounded(sC * sbyte_of(w1, e));
                    }
                    const int n0 = 64 * (ks / 2) + 16 * lq + 8 * (ks % 2);     // the states of those eight codes
                    v8h fs[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) fs[j] = *reinterpret_cast<const v8h*>(&sm.prev[j * 16 + l16][n0 ^ ((l16 & S::SWZ) * 8)]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[s][j] = mfma16(cf, fs[j], acc[s][j]);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float em = fexp(sm.dA[m0 + 4 * lq + r]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[s][j][r] *= em;
                }
            }
        }
        __syncthreads();                                               // everyone is done with the entering state
        if (kShares == kThreads || tid < kShares) {
            const int xc = tid % (kP / CH) * CH, kb = steps_of(tid / (kP / CH));
            if (lim < Q) {
                // ragged last chunk: steps past the end of the sequence count as zero
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (4 * kb + r >= lim) xr[r] = XShare<CH>{};
                }
            }
            stage_x_share<CH>(xr, sm.xs, xc, [&](int row, const v4h& v) { *reinterpret_cast<v4h*>(&sm.xt[S::x_at(row, (kb >> 1 & ~3) + (kb & 3)) + (kb & 4)]) = v; });
        }
        __syncthreads();

        // the short tile first, the next head's requests with the long one: by then the first tile's sums have left their registers
#pragma unroll
        for (int s = TILES - 1; s >= 0; --s) {
            if (MODE == kScanWalk && s == 0) {
                fetch_head(min(h + 1, h_last), tid);
                __builtin_amdgcn_sched_barrier(0);                     // (the scheduler would sink the requests below the products)
            }
            const int mt = tile_of(s);
            const int m0 = mt * 16;
            const int nks = (mt + 2) / 2;                               // 32-step pieces that reach row m0 + 15; the last holds the diagonal
            const int m_row = m0 + l16;                                 // row of this lane's first operands
            const float dA_m = sm.dA[m_row];
            // skip-term operands of this lane's four output rows
            // (requested now, used in the epilogue: nothing there waits for memory)
            uint32_t xq[4], zq[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t at = static_cast<uint32_t>(min(m0 + 4 * lq + r, lim - 1)) * xrow + 4 * l16;
                xq[r] = *reinterpret_cast<const uint32_t*>(xbase + at);
                if (p.z) zq[r] = *reinterpret_cast<const uint32_t*>(zbase + at);
            }
            // (C B^T)^T of a 16-step block of piece ks: a lane has four steps of its row
            auto cb_of = [&](int ks, int blk) {
                v4i cb = v4i{0, 0, 0, 0};
#pragma unroll
                for (int i = 0; i < N / 64; ++i) {
                    const v4i bo = *reinterpret_cast<const v4i*>(&sm.bq[32 * ks + 16 * blk + l16][((4 * i + lq) ^ (l16 & S::BSWZ)) * 16]);
                    cb = __builtin_amdgcn_mfma_i32_16x16x64_i8(bo, cq[s][i], cb, 0, 0, 0);
                }
                return cb;
            };
            // the weights of steps 32 ks + 4 q .. + 3 and 32 ks + 16 + 4 q .. + 3 times x
            const int x_first = S::x_at(l16, lq);
            auto times_x = [&](int ks, const float (&wv)[8]) {
                v8h fl;
#pragma unroll
                for (int e = 0; e < 8; ++e) fl[e] = rounded(wv[e]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const v8h fx = *reinterpret_cast<const v8h*>(&sm.xt[(x_first ^ S::x_turned(ks)) + S::x_past(ks) + j * 16 * Q]);
                    acc[s][j] = mfma16(fl, fx, acc[s][j]);
                }
            };
            float wv[8];
#pragma unroll 1
            for (int ks = 0; ks + 1 < nks; ++ks) {
                const int ka = 32 * ks + 4 * lq;
                const v4i cb[2] = {cb_of(ks, 0), cb_of(ks, 1)};
                const float4 g0 = *reinterpret_cast<const float4*>(&sm.gk[ka]), g1 = *reinterpret_cast<const float4*>(&sm.gk[ka + 16]);
                const float gk[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
                const float e_m = cb_scale * fexp(dA_m - sm.dA[32 * ks + 31]);       // the scale of C B^T rides with the row's decay
#pragma unroll
                for (int e = 0; e < 8; ++e) wv[e] = static_cast<float>(cb[e / 4][e % 4]) * (e_m * gk[e]);
                times_x(ks, wv);
            }
            // the piece with the diagonal: steps after row m do not count, nor does all of the second block of an even tile
            auto diagonal = [&](int blk) {
                const int ka = 32 * (nks - 1) + 16 * blk + 4 * lq;
                const v4i cb = cb_of(nks - 1, blk);
                const float4 a4 = *reinterpret_cast<const float4*>(&sm.dA[ka]), d4 = *reinterpret_cast<const float4*>(&sm.dt[ka]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float cv = ka + e <= m_row ? cb_scale * static_cast<float>(cb[e]) : 0.0f;
                    wv[4 * blk + e] = (cv * fexp(fminf(dA_m - lane_of(a4, e), 0.0f))) * lane_of(d4, e);
                }
            };
            diagonal(0);
            if (mt & 1) {
                diagonal(1);
            } else {
#pragma unroll
                for (int e = 4; e < 8; ++e) wv[e] = 0.0f;
            }
            times_x(nks - 1, wv);
            // Epilogue: acc[s][j][r] is row m0 + 4 (lane / 16) + r, channel 4 (lane % 16) + j
            const float4 xs4 = *reinterpret_cast<const float4*>(&sm.xs[4 * l16]), Dv4 = *reinterpret_cast<const float4*>(&sm.Dv[4 * l16]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + 4 * lq + r;
                if (m < lim) {
                    float y[4] = {acc[s][0][r], acc[s][1][r], acc[s][2][r], acc[s][3][r]};
                    if (p.D) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) y[j] = __builtin_fmaf(lane_of(xs4, j) * sbyte_of(xq[r], j), lane_of(Dv4, j), y[j]);
                    }
                    if (p.z) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) y[j] *= sm.gate[(zq[r] >> (8 * j)) & 0xffu];
                    }
                    v4h o;
#pragma unroll
                    for (int j = 0; j < 4; ++j) o[j] = static_cast<_Float16>(y[j]);
                    *reinterpret_cast<v4h*>(out + static_cast<uint32_t>(m) * xrow + 4 * l16) = o;
                }
            }
        }
        if constexpr (MODE == kScanWalk) __syncthreads();              // everyone is done with this head's tile and tables
    }
    if constexpr (MODE == kScanChain) {
        // the first chunk's workgroup, which had nothing to chain up, leaves the state after the last
        if (c > 0 || !p.final_states) return;
        const int tid = threadIdx.x;
        float run[PB][8];
        chain(run, tid, nc);
#pragma unroll
        for (int i = 0; i < PB; ++i) {
            const int piece = tid + i * kThreads, slot = piece / (N / 8), n = piece % (N / 8) * 8, pp = 4 * (slot % 16) + slot / 16;
            const int64_t at = ((static_cast<int64_t>(b) * H + h_first) * kP + pp) * N + n;
            const int srow = p.final_state_is_fp32 ? 0 : srow_ws[h_first / split * p.headdim + (h_first % split) * kP + pp];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (p.final_state_is_fp32) static_cast<float*>(p.final_states)[at + e] = run[i][e];
                else static_cast<int8_t*>(p.final_states)[at + e] = ssd_quantize_state(p, srow, n + e, run[i][e]);
            }
        }
    }
}

int validate(const QaSsdParams* p) {
    if (!p) return QA_ERR_NULL;
    if (p->batch < 0 || p->seqlen < 0 || p->nheads < 1 || p->ngroups < 1 || p->nheads % p->ngroups != 0) return QA_ERR_SHAPE;
    if (p->batch > 0 && p->seqlen > 0) {                          // (no steps: the tensors may be null)
        if (!p->x || !p->dt || !p->A_log || !p->B || !p->C || !p->out) return QA_ERR_NULL;
        if (!p->x_scale || !p->A_log_scale || !p->B_scale || !p->C_scale) return QA_ERR_NULL;
        if (!p->dt_is_fp32 && !p->dt_scale) return QA_ERR_NULL;
        if ((p->D && !p->D_scale) || (p->z && !p->z_scale)) return QA_ERR_NULL;
        if (p->final_states && !p->final_state_is_fp32 && !p->state_scale) return QA_ERR_NULL;
        if (p->nhead_groups > 0 && (!p->x_head_group_range || !p->x_dim_group_range || p->ndim_groups < 1)) return QA_ERR_NULL;
    }
    // what the general kernels take; the matrix-core kernels cover a subset (ssd_fast_shape)
    if (p->headdim < 1 || p->headdim > 256 || p->dstate < 1 || p->dstate > 1024 || p->chunk_size < 1 || p->chunk_size > 1024) return QA_ERR_UNSUPPORTED;
    const int64_t nc = (static_cast<int64_t>(p->seqlen) + p->chunk_size - 1) / p->chunk_size;
    if (ssd_fast_shape(*p)) {
        // every launch is a one-dimensional grid: one workgroup per (batch, chunk, head) or per (batch, head)
        const int64_t heads = static_cast<int64_t>(p->nheads) * (p->headdim / 64);       // heads of 64 channels
        if (static_cast<int64_t>(p->batch) * nc * heads > 0x7fffffffLL) return QA_ERR_SHAPE;
    } else {
        const int st = ssd_general_grid_check(*p);
        if (st != QA_OK) return st;
    }
    return QA_OK;
}

}  // namespace

int ssd_check(const QaSsdParams& p) { return validate(&p); }
}  // namespace qa

extern "C" int64_t qa_ssd_workspace_bytes(const QaSsdParams* p) {
    if (qa::validate(p) != QA_OK) return 0;
    const qa::SsdWorkspace ws = qa::ssd_workspace_layout(*p);
    return ws.total + ws.sums_bytes;
}

extern "C" int qa_ssd_chunk_scan_fwd(const QaSsdParams* p, void* stream_) {
    using namespace qa;
    const int st = validate(p);
    if (st != QA_OK) return st;
    if (p->batch == 0) return QA_OK;
    if (p->seqlen == 0) {
        // no steps: the state after them is the zero state the scan starts from
        const int64_t states = static_cast<int64_t>(p->batch) * p->nheads * p->headdim * p->dstate;
        return fill_zero(p->final_states, states * (p->final_state_is_fp32 ? 4 : 1), static_cast<hipStream_t>(stream_));
    }
    const SsdWorkspace ws = ssd_workspace_layout(*p);
    if (!p->workspace) return QA_ERR_NULL;
    if (p->workspace_bytes < ws.total || (reinterpret_cast<uintptr_t>(p->workspace) & 255u)) return QA_ERR_STRIDE;
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    uint8_t* base = static_cast<uint8_t*>(p->workspace);
    float* dt_ws = reinterpret_cast<float*>(base + ws.dt);
    float* dA_ws = reinterpret_cast<float*>(base + ws.dA);
    const int nc = (p->seqlen + p->chunk_size - 1) / p->chunk_size;
    const int64_t bch = static_cast<int64_t>(p->batch) * nc * p->nheads;

    __half* prev_ws = reinterpret_cast<__half*>(base + ws.prev);
    float* xs_ws = reinterpret_cast<float*>(base + ws.xs);
    int32_t* srow_ws = reinterpret_cast<int32_t*>(base + ws.srow);
    if (!ssd_fast_shape(*p)) {
        ssd_general_launch(*p, dt_ws, dA_ws, prev_ws, xs_ws, srow_ws, nc, stream);
        return check_launch();
    }
    const int heads64 = p->nheads * (p->headdim / 64);          // the kernels see a head of 64 s channels as s heads of 64
    int status = QA_OK;
    // more LDS than a kernel gets by default: raise the limit (idempotent)
    auto lds_ok = [&](const void* kernel, size_t lds) {
        if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) == hipSuccess) return true;
        status = check_launch();
        if (status == QA_OK) status = QA_ERR_LAUNCH;
        return false;
    };
    float* sums_ws = ws.sums_bytes && p->workspace_bytes >= ws.sums + ws.sums_bytes ? reinterpret_cast<float*>(base + ws.sums) : nullptr;
    auto launch = [&](auto n_c, auto q_c) {
        constexpr int N = decltype(n_c)::value, Q = decltype(q_c)::value, kScanThreads = 64 * scan_waves_of(Q);
        constexpr size_t kStateLds = sizeof(StateSmem<N, Q>), kScanLds = sizeof(ScanSmem<N, Q>);
        // Heads a scan workgroup walks: what takes the fewest of them one after the other in the places the chip has at once (sixteen
        // waves of up to 128 registers to a CU), a workgroup's start counted as a fifth of a head.  (A share of the heads for each
        // place, 10 and 6 of 16 in 640 workgroups on 512 places, took 8 x 1100 steps of 128 heads 169 us, 131 in
        // shares of two; 3000 steps of 128 heads 58.6 in shares of three, 47.4 of four; 3 x 1000 steps 54 and 46.)
        const int hpg = heads64 / p->ngroups, units = static_cast<int>(bch / p->nheads) * p->ngroups;
        const int64_t places = static_cast<int64_t>(compute_units()) * (1024 / kScanThreads);
        int heads_each = 1;
        int64_t least = -1;
        for (int parts = 1; parts <= hpg; ++parts) {
            const int each = (hpg + parts - 1) / parts;
            const int64_t cost = (static_cast<int64_t>(units) * ((hpg + each - 1) / each) + places - 1) / places * (5 * each + 1);
            if (least < 0 || cost < least) { least = cost; heads_each = each; }
        }
        const bool chain = sums_ws && heads_each == 1 && nc <= kChainChunks;
        auto scan_kernel = chain ? ssd_chunk_scan_kernel<N, Q, kScanChain> : heads_each == 1 ? ssd_chunk_scan_kernel<N, Q, kScanOne> : ssd_chunk_scan_kernel<N, Q, kScanWalk>;
        // With a workgroup per chunk and head these make the step sizes, too, in place of a launch in front: once per head instead of once
        // per four heads' line of bytes, which is cheaper up to some workgroups a CU (us of the two launches against the one:
        // 2 chunks of 24 heads 11.3 -> 7.4, 6 of 80 17.4 -> 13.7, 8 of 80 19.5 -> 17.4; 16 of 128 38.6 -> 41.7)
        const int64_t chunk_heads = static_cast<int64_t>(p->batch) * heads64 * nc;
        const int own_steps = (sums_ws || nc == 1) && chunk_heads <= 4LL * compute_units();
        const bool apart = sums_ws || (nc == 1 && own_steps);
        auto state_kernel = apart ? ssd_state_kernel<N, Q, false> : ssd_state_kernel<N, Q, true>;
        if (!lds_ok(reinterpret_cast<const void*>(state_kernel), kStateLds) || !lds_ok(reinterpret_cast<const void*>(scan_kernel), kScanLds)) return;
        if (!own_steps) {
            const int64_t tables = (p->nheads + Q / 64 - 1) / (Q / 64), heads = (p->nheads + kCumHeads - 1) / kCumHeads;
            hipLaunchKernelGGL(ssd_cumsum_kernel<Q>, dim3(static_cast<unsigned>(tables + heads * p->batch * nc)), dim3(Q), 0, stream, *p, dt_ws, dA_ws, xs_ws, srow_ws, nc);
        }
        hipLaunchKernelGGL(state_kernel, dim3(static_cast<unsigned>(apart ? chunk_heads : p->batch * heads64)), dim3(4 * N), kStateLds, stream, *p, dt_ws, dA_ws, prev_ws, sums_ws, xs_ws, srow_ws, nc,
                           own_steps);
        if (sums_ws && !chain)
            hipLaunchKernelGGL(ssd_pass_kernel<N>, dim3(static_cast<unsigned>(p->batch * heads64 * (N / 16))), dim3(256), 0, stream, *p, dA_ws, prev_ws, sums_ws, srow_ws, nc);
        hipLaunchKernelGGL(scan_kernel, dim3(static_cast<unsigned>(units * ((hpg + heads_each - 1) / heads_each))), dim3(kScanThreads), kScanLds, stream, *p, dt_ws, dA_ws, prev_ws, sums_ws, xs_ws,
                           srow_ws, nc, heads_each);
    };
#define QA_SSD_LAUNCH(N_, Q_) launch(std::integral_constant<int, N_>{}, std::integral_constant<int, Q_>{})
    if (p->dstate == 128) {
        if (p->chunk_size == 256) QA_SSD_LAUNCH(128, 256);
        else if (p->chunk_size == 128) QA_SSD_LAUNCH(128, 128);
        else QA_SSD_LAUNCH(128, 64);
    } else {
        if (p->chunk_size == 256) QA_SSD_LAUNCH(64, 256);
        else if (p->chunk_size == 128) QA_SSD_LAUNCH(64, 128);
        else QA_SSD_LAUNCH(64, 64);
    }
#undef QA_SSD_LAUNCH
    if (status != QA_OK) return status;
    return check_launch();
}

// ---------------------------------------------------------------------------------------------
// The same scan for callers that cannot allocate (code under HIP graph capture, serving loops and harnesses that
// forbid hipMalloc): the workspace is a fixed array in the device image instead of a caller's buffer.  Every GPU
// holds its own copy of the array at its own address, so the address is looked up once per device, with that
// device current, and kept.  In host code the array's name is only a handle for that lookup, never a pointer.
// ---------------------------------------------------------------------------------------------
namespace qa {
namespace {
constexpr int64_t kStaticScratchBytes = QA_SSD_STATIC_SCRATCH_BYTES;
constexpr int kMaxDevices = 64;
}  // namespace
}  // namespace qa

static __device__ __align__(256) unsigned char scratch[qa::kStaticScratchBytes];

namespace qa {
namespace {
std::mutex g_scratch_mutex;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device (null: the runtime refused the lookup).
void* static_scratch_of_current_device() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (ptr) return ptr;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    ptr = g_scratch_ptr[dev].load(std::memory_order_relaxed);
    if (ptr) return ptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        set_last_hip_error(static_cast<int>(e));
        return nullptr;
    }
    g_scratch_ptr[dev].store(ptr, std::memory_order_release);
    return ptr;
}
}  // namespace
}  // namespace qa

extern "C" int qa_ssd_chunk_scan_fwd_noalloc(const QaSsdParams* p, void* stream_) {
    using namespace qa;
    const int st = validate(p);
    if (st != QA_OK) return st;
    if (p->batch == 0 || p->seqlen == 0) return qa_ssd_chunk_scan_fwd(p, stream_);      // (nothing needs a workspace)
    if (ssd_workspace_layout(*p).total > kStaticScratchBytes) return QA_ERR_SCRATCH;
    void* ptr = static_scratch_of_current_device();
    if (!ptr) return QA_ERR_LAUNCH;
    QaSsdParams q = *p;
    q.workspace = ptr;
    q.workspace_bytes = kStaticScratchBytes;
    return qa_ssd_chunk_scan_fwd(&q, stream_);
}
