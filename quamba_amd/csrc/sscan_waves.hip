// Mamba1 int8 selective scan over token-major rows, sixteen states, the time cut over the waves of a workgroup: the scan of
// an assembled mixer where a wave for some channels each does not fill the chip (sscan_tm.hip chooses).  Arithmetic as in
// sscan_tm.hip (reference csrc/selective_scan/quant_sscan_fwd_kernel.cuh:110-293).
//
// A workgroup owns sixteen channels (eight with eight lanes a channel) and walks the sequence in blocks of T steps a wave.  In
// a block every wave scans its steps from a zero state, keeping the decays it evaluates in registers, and leaves its end
// state and the decay of all of its steps in LDS; after a barrier it chains its predecessors' up to the state it starts from,
// and goes over its steps once more, now with outputs: two multiply-adds a step and state, no exponential.  Everything but the
// waves' ends is a wave's own, so there is one barrier a block, and the bytes of the next block arrive during the second pass.
//
// What bounds it is vector issue, 570 instructions a wave of sixteen channels x sixteen steps (774 for eight x thirty-two), 76
// of them transcendental - a third more work than one pass takes - once there are three waves per SIMD, and with fewer the
// latencies of a block's phases.  What it replaces are one launch of eight or sixteen lanes a channel, which leaves waves of
// hundreds of dependent steps alone on their SIMDs, and two launches over segments, which evaluate step sizes and decays twice
// (prompts x steps x channels, us): 1 x 128 x 1536 8.9 -> 6.6, 1 x 300 x 1536 16.7 -> 10.0, 1 x 512 x 1536 18.9 -> 12.2, 1 x 777 x
// 3072 31.5 -> 27.7, 1 x 777 x 4096 39.5 -> 28.0, 2 x 1500 x 4096 111 -> 85, 4 x 2048 x 3072 191 -> 155; over 97 sizes 0.82 of the
// time before.  Sixteen waves of eight lanes just fit their registers; four lanes take 148, so at most twelve waves (forced into
// 128 they spill: 4 x 2048 x 5120 in twelve waves 242 us -> 297, in sixteen 271; 2 x 4000 x 2048 as the rule lays it out 91 -> 103).
//
// Other sums than one pass makes, in fp32 as there and no less exact: against 64 bits, at twelve sizes of 48 to 4000 steps x 1536 to 5120
// channels, end states are off by 1.4 to 1.6e-7 (2-norm, relative; one pass 1.4 to 1.9e-7, segments 1.4 to 1.9e-7, the more steps the
// more) and outputs by fp16's own 2.1e-4 with all of them.
#include "conv_common.hpp"
#include "gemm_core.hpp"
#include "mixer_common.hpp"
#include "sscan_common.hpp"
#include "sscan_waves.hpp"

#include <algorithm>

namespace qa {
namespace {

using gemm::v4i;
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int max_waves(int lanes) { return lanes == 4 ? 12 : kScanWavesMax; }

template <int NSPLIT>
struct WavesCfg {
    static constexpr int T = NSPLIT == 4 ? 16 : 32;        // steps of a wave
    static constexpr int NPL = 16 / NSPLIT;                // states per lane
    static constexpr int kCh = 64 / NSPLIT;                // channels
    static constexpr int kPitch = NSPLIT == 4 ? 20 : 40;   // floats per row of per-step values: rows written by four channels of
                                                           // sixteen steps, and read four steps of all channels, without conflicts
    static constexpr int kUzPitch = T + 4;                 // 16-bit (u | z << 8) codes per row
    static constexpr int kGroupPitch = 132;                // floats per group of four steps of B | C
    static constexpr int kOutPitch = kCh + 8;              // halves
    static constexpr int kSets = T / 16;                   // sixteen-step products of dt_proj
};

// what a wave keeps of its steps
template <class Cfg>
struct WaveRows {
    union {
        float d[Cfg::kCh][Cfg::kPitch];                    // step size: the second pass has the decays and needs it no more
        __half out[Cfg::T][Cfg::kOutPitch];
    };
    __attribute__((aligned(16))) float du[Cfg::kCh][Cfg::kPitch];              // step size x input code
    __attribute__((aligned(16))) float bc[Cfg::T / 4][Cfg::kGroupPitch];       // B | C of four steps by state
    __attribute__((aligned(16))) uint16_t uz[Cfg::kCh][Cfg::kUzPitch];
};

// what the waves share beside the ends of their steps; dt_proj's weights as 16-byte fragments of the lanes come behind it
struct Shared {
    float gate[256];                                       // SiLU gate per z code (indexed by the raw byte)
    float bias[16], dt_scale[16];                          // of the workgroup's channels
};

template <int NSPLIT>
constexpr int lds_bytes(int waves, int pieces) {
    using Cfg = WavesCfg<NSPLIT>;
    return waves * (static_cast<int>(sizeof(WaveRows<Cfg>)) + 2 * 2 * 64 * Cfg::NPL * 4) + 2 * 64 * Cfg::NPL * 4 + static_cast<int>(sizeof(Shared)) + pieces * 1024;
}

template <int N>
struct Floats {
    float v[N];
};
template <int N>
__device__ __forceinline__ Floats<N> load_floats(const float* at) {
    Floats<N> r;
    __builtin_memcpy(&r, __builtin_assume_aligned(at, 4 * N), sizeof(r));
    return r;
}
template <int N>
__device__ __forceinline__ void store_floats(float* at, const Floats<N>& r) { __builtin_memcpy(__builtin_assume_aligned(at, 4 * N), &r, sizeof(r)); }

// WAVES: the most that a workgroup may have
template <int NSPLIT, int WAVES, bool HAS_Z, int DTK>
__global__ __launch_bounds__(64 * WAVES) void scan_waves_kernel(QaSScanParams p, SscanDtProj dtp, int vec_out) {
    using Cfg = WavesCfg<NSPLIT>;
    constexpr int T = Cfg::T, NPL = Cfg::NPL, kCh = Cfg::kCh, kGroups = T / 4;
    constexpr bool kOuter = NSPLIT == 4;                   // B x (step size x input) on the matrix cores
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int waves = __builtin_amdgcn_readfirstlane(blockDim.x >> 6);
    WaveRows<Cfg>& sm = reinterpret_cast<WaveRows<Cfg>*>(lds)[wave];
    float* const ends = reinterpret_cast<float*>(lds + waves * sizeof(WaveRows<Cfg>));
    constexpr int kEnd = 64 * NPL;                                        // decays, then states of a wave
    float* const carry = ends + 2 * waves * 2 * kEnd;
    Shared& sh = *reinterpret_cast<Shared*>(carry + 2 * kEnd);
    v4i* const weights = reinterpret_cast<v4i*>(&sh + 1);

    // neighbouring workgroups share lines of every tensor: those of an XCD take neighbouring channels
    const int blocks = gridDim.x, per_xcd = blocks / 8;
    const int bx = blockIdx.x;
    const int cb = bx < 8 * per_xcd ? (bx % 8) * per_xcd + bx / 8 : bx;
    const int c0 = cb * kCh, b = blockIdx.y;
    const int c_local = lane % kCh;
    const int slice = (lane & 15) / kCh * 4 + (lane >> 4), qslice = slice & 3;
    const int c = c0 + c_local;
    const bool c_ok = c < p.dim;
    const int cc = c_ok ? c : p.dim - 1;
    const int L = p.seqlen, steps = waves * T, n_blocks = (L + steps - 1) / steps;
    const bool softplus = p.delta_softplus != 0;

    // this lane's share of a wave's steps: four channels of one step, the arrangement in which 16 x 16 products leave the
    // matrix cores
    const int g = lane >> 4, j = lane & 15;
    const int quad = NSPLIT == 4 ? g : g & 1;
    const int step = NSPLIT == 4 ? j : j + 16 * (g >> 1);
    const int lc4 = 4 * quad;
    const int ch4 = min(c0 + lc4, p.dim - 4);              // channels past the last read the last four; nothing of theirs is stored
    const int bc_step = lane >> 2, bc_word = lane & 3;

    const int8_t* const u_b = p.u + b * p.u_batch_stride;
    const int8_t* const z_b = HAS_Z ? p.z + b * p.z_batch_stride : nullptr;
    const int8_t* const d_b = DTK == 0 ? p.delta + b * p.delta_batch_stride : nullptr;
    const int8_t* const B_b = p.B + b * p.B_batch_stride;
    const int8_t* const C_b = p.C + b * p.C_batch_stride;
    const int8_t* const x_b = DTK ? dtp.x + b * dtp.x_batch_stride : nullptr;
    const uint32_t u_ls = static_cast<uint32_t>(p.u_l_stride), z_ls = HAS_Z ? static_cast<uint32_t>(p.z_l_stride) : 0, d_ls = DTK == 0 ? static_cast<uint32_t>(p.delta_l_stride) : 0;
    const uint32_t B_ls = static_cast<uint32_t>(p.B_l_stride), C_ls = static_cast<uint32_t>(p.C_l_stride), x_ls = DTK ? static_cast<uint32_t>(dtp.x_l_stride) : 0;

    uint32_t r_u, r_z = 0, r_d = 0, r_b[Cfg::kSets], r_c[Cfg::kSets];
    v4i r_x[DTK ? Cfg::kSets : 1][DTK ? DTK : 1];
    auto issue_loads = [&](int block) {                    // steps past the end read the last one
        const int t0 = min((block * waves + wave) * T, L - 1), last = min(T, L - t0) - 1;
        // (a wave-uniform address and 32-bit offsets)
        const uint32_t t = min(step, last);
        r_u = *reinterpret_cast<const uint32_t*>(u_b + static_cast<int64_t>(t0) * u_ls + (t * u_ls + ch4));
        if constexpr (DTK == 0) r_d = *reinterpret_cast<const uint32_t*>(d_b + static_cast<int64_t>(t0) * d_ls + (t * d_ls + ch4));
        if constexpr (HAS_Z) r_z = *reinterpret_cast<const uint32_t*>(z_b + static_cast<int64_t>(t0) * z_ls + (t * z_ls + ch4));
#pragma unroll
        for (int s = 0; s < Cfg::kSets; ++s) {
            const uint32_t tb = min(bc_step + 16 * s, last);
            r_b[s] = *reinterpret_cast<const uint32_t*>(B_b + static_cast<int64_t>(t0) * B_ls + (tb * B_ls + 4 * bc_word));
            r_c[s] = *reinterpret_cast<const uint32_t*>(C_b + static_cast<int64_t>(t0) * C_ls + (tb * C_ls + 4 * bc_word));
        }
    };
    auto issue_x = [&](int block) {
        if constexpr (DTK != 0) {
            const int t0 = min((block * waves + wave) * T, L - 1), last = min(T, L - t0) - 1;
#pragma unroll
            for (int s = 0; s < Cfg::kSets; ++s) {
                const uint32_t row = static_cast<uint32_t>(min(j + 16 * s, last)) * x_ls;
#pragma unroll
                for (int kb = 0; kb < DTK; ++kb) r_x[s][kb] = *reinterpret_cast<const v4i*>(x_b + static_cast<int64_t>(t0) * x_ls + (row + min(64 * kb + 16 * g, dtp.rank - 16)));
            }
        }
    };
    issue_loads(0);
    issue_x(0);

    // dt_proj's weights as the first operand: row j is channel j of the wave (again from the start when it has fewer)
    float dt_row = 0.0f;
    if constexpr (DTK != 0) {
        const int8_t* row = dtp.w + static_cast<int64_t>(min(c0 + j % kCh, p.dim - 1)) * dtp.rank;
        for (int kb = wave; kb < DTK; kb += waves) {
            v4i f = *reinterpret_cast<const v4i*>(row + min(64 * kb + 16 * g, dtp.rank - 16));
            if (64 * kb + 16 * g >= dtp.rank) f = v4i{0, 0, 0, 0};
            weights[kb * 64 + lane] = f;
        }
        dt_row = *dtp.row_scale;
    }
    uint32_t A_codes[NPL];
#pragma unroll
    for (int i = 0; i < NPL; ++i) A_codes[i] = static_cast<uint8_t>(p.A_log[cc * p.A_d_stride + (slice * NPL + i) * p.A_dstate_stride]);
    const float D_code = p.D ? static_cast<float>(p.D[cc]) : 0.0f;
    const float s_u = *p.scale_u, s_dt = *p.scale_delta, s_A = *p.scale_A, s_B = *p.scale_B, s_C = *p.scale_C;
    const float s_z = HAS_Z ? *p.scale_z : 0.0f, s_D = p.D ? *p.scale_D : 0.0f;
    const float D_u = (s_D * D_code) * s_u;                // skip weight per input code
    const float b_scale = s_B * s_u;                       // the input scale rides with B and D: (s_B q_B) (dt (s_u q_u))
    float A2[NPL];
#pragma unroll
    for (int i = 0; i < NPL; ++i) A2[i] = fmaxf(-expf(s_A * code_byte_to_float(A_codes[i], 0)) * kLog2e, -3.4e38f);     // (a decay of 1 for no time, always)
    if (tid < kCh) {
        const int at = min(c0 + tid, p.dim - 1);
        sh.bias[tid] = p.delta_bias ? *p.scale_delta_bias * static_cast<float>(p.delta_bias[at]) : 0.0f;
        if constexpr (DTK != 0) sh.dt_scale[tid] = dtp.col_scale[dtp.col_numel == 1 ? 0 : at];
    }
    if constexpr (HAS_Z) {
        for (int i = tid; i < 256; i += 64 * waves) sh.gate[i] = silu_gate(s_z * static_cast<float>(static_cast<int8_t>(i)));
    }

    auto stage = [&](int block) {
        float dv[4];
        const Floats<4> bias = load_floats<4>(&sh.bias[lc4]);
        if constexpr (DTK != 0) {
            const Floats<4> dt_col = load_floats<4>(&sh.dt_scale[lc4]);
            v4i acc[Cfg::kSets] = {};
#pragma unroll
            for (int kb = 0; kb < DTK; ++kb) {
                const v4i fw = weights[kb * 64 + lane];
#pragma unroll
                for (int s = 0; s < Cfg::kSets; ++s) acc[s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw, r_x[s][kb], acc[s], 0, 0, 0);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                int sum = acc[0][e];
                if constexpr (NSPLIT == 8) sum = g < 2 ? acc[0][e] : acc[1][e];
                float v = dt_col.v[e] * (dt_row * static_cast<float>(sum));
                v = __builtin_amdgcn_fmed3f(__builtin_rintf(v), -128.0f, 127.0f);              // the int8 code
                dv[e] = __builtin_fmaf(s_dt, v, bias.v[e]);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) dv[e] = __builtin_fmaf(s_dt, code_byte_to_float(r_d, e), bias.v[e]);
        }
        if (softplus) {
#pragma unroll
            for (int e = 0; e < 4; ++e) dv[e] = softplus20_flat(dv[e]);
        }
        const bool inside = (block * waves + wave) * T + step < L;     // steps past the end leave the state alone (a = 1, b = 0)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            dv[e] = inside ? dv[e] : 0.0f;
            sm.d[lc4 + e][step] = dv[e];
            sm.du[lc4 + e][step] = dv[e] * code_byte_to_float(r_u, e);
            sm.uz[lc4 + e][step] = static_cast<uint16_t>(__builtin_amdgcn_perm(r_z, r_u, 0x0c0c0400u + 0x0101u * e));
        }
#pragma unroll
        for (int s = 0; s < Cfg::kSets; ++s) {
            const int t = bc_step + 16 * s;
            float* const at = &sm.bc[t >> 2][16 * bc_word + (t & 3)];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                at[4 * e] = b_scale * code_byte_to_float(r_b[s], e);
                at[64 + 4 * e] = s_C * code_byte_to_float(r_c[s], e);
            }
        }
    };
    // B x (step size x input) of a group of four steps, value s NPL + n: step s, state n of this lane
    struct Products {
        float v[4 * NPL];
    };
    auto products = [&](int tq) {
        Products r;
        if constexpr (kOuter) {
            constexpr v16f zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            const v16f m = __builtin_amdgcn_mfma_f32_16x16x1f32(sm.bc[tq][4 * j + g], sm.du[c_local][4 * tq + g], zero, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 16; ++i) r.v[i] = m[i];
        } else {
            const Floats<4> du = load_floats<4>(&sm.du[c_local][4 * tq]);
#pragma unroll
            for (int n = 0; n < NPL; ++n) {
                const Floats<4> Bv = load_floats<4>(&sm.bc[tq][4 * (slice * NPL + n)]);
#pragma unroll
                for (int s = 0; s < 4; ++s) r.v[s * NPL + n] = Bv.v[s] * du.v[s];
            }
        }
        return r;
    };

    const int out_step = lane / (kCh / 4), out_ch = lane % (kCh / 4) * 4;
    const bool out_mine = c0 + out_ch < p.dim;             // (dim is a multiple of four)
    __half* const out_b = static_cast<__half*>(p.out) + b * p.out_batch_stride + (c0 + out_ch) * p.out_d_stride;
    const int out_col = slice >= 4 ? kCh + c_local : c_local;      // with eight lanes a channel only the first four's sums are complete
    float h[NPL];
    __syncthreads();                                       // what the waves share is complete
    for (int block = 0; block < n_blocks; ++block) {
        stage(block);
        gemm::wave_lds_sync();
        // from a zero state
        float a[kGroups][4][NPL], dt_sum = 0.0f;
#pragma unroll
        for (int i = 0; i < NPL; ++i) h[i] = 0.0f;
#pragma unroll
        for (int tq = 0; tq < kGroups; ++tq) {
            if constexpr (WAVES > 12) __builtin_amdgcn_sched_barrier(0);        // (one group's operands at a time beside the decays)
            const Floats<4> d = load_floats<4>(&sm.d[c_local][4 * tq]);
            const Products bdu = products(tq);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                dt_sum += d.v[s];
#pragma unroll
                for (int n = 0; n < NPL; ++n) {
                    a[tq][s][n] = fast_exp2(d.v[s] * A2[n]);
                    h[n] = __builtin_fmaf(a[tq][s][n], h[n], bdu.v[s * NPL + n]);
                }
            }
        }
        Floats<NPL> end_decay, end_state;
#pragma unroll
        for (int n = 0; n < NPL; ++n) {
            end_decay.v[n] = fast_exp2(dt_sum * A2[n]);
            end_state.v[n] = h[n];
        }
        float* const ends_now = ends + (block & 1) * waves * 2 * kEnd + lane * NPL;
        store_floats<NPL>(ends_now + wave * 2 * kEnd, end_decay);
        store_floats<NPL>(ends_now + wave * 2 * kEnd + kEnd, end_state);
        __syncthreads();
        // the state this wave starts from: the block's, then every predecessor's steps
#pragma unroll
        for (int n = 0; n < NPL; ++n) h[n] = 0.0f;
        if (block > 0) {
            const Floats<NPL> from = load_floats<NPL>(carry + ((block - 1) & 1) * kEnd + lane * NPL);
#pragma unroll
            for (int n = 0; n < NPL; ++n) h[n] = from.v[n];
        }
        // (four at a time: their reads wait together; those past this wave's place change nothing)
        for (int w0 = 0; w0 < wave; w0 += 4) {
            Floats<NPL> decay[4], state[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float* at = ends_now + min(w0 + i, waves - 1) * 2 * kEnd;
                decay[i] = load_floats<NPL>(at);
                state[i] = load_floats<NPL>(at + kEnd);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (w0 + i < wave) {
#pragma unroll
                    for (int n = 0; n < NPL; ++n) h[n] = __builtin_fmaf(decay[i].v[n], h[n], state[i].v[n]);
                }
        }
        if (wave == waves - 1) {
            Floats<NPL> to;
#pragma unroll
            for (int n = 0; n < NPL; ++n) to.v[n] = __builtin_fmaf(end_decay.v[n], h[n], end_state.v[n]);
            store_floats<NPL>(carry + (block & 1) * kEnd + lane * NPL, to);
        }
        issue_loads(block + 1);                            // (behind the last block: the last step, for nobody)
#pragma unroll
        for (int tq = 0; tq < kGroups; ++tq) {
            if constexpr (WAVES > 12) __builtin_amdgcn_sched_barrier(0);
            const uint32_t code = sm.uz[c_local][4 * tq + qslice];     // of the step this lane owns: u in byte 0, z in byte 1
            if (tq == (WAVES > 12 ? kGroups - 1 : 0)) issue_x(block + 1);         // (the decays' registers are free)
            const Products bdu = products(tq);
            float acc[4];
#pragma unroll
            for (int n = 0; n < NPL; ++n) {
                const Floats<4> Cv = load_floats<4>(&sm.bc[tq][64 + 4 * (slice * NPL + n)]);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    h[n] = __builtin_fmaf(a[tq][s][n], h[n], bdu.v[s * NPL + n]);
                    acc[s] = n == 0 ? h[n] * Cv.v[s] : __builtin_fmaf(h[n], Cv.v[s], acc[s]);
                }
            }
            // each of four lanes completes the step it owns: lanes 32, then 16 apart keep one half and hand the other over
            const auto fold32 = [](float x, float y) {
                const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
                return __uint_as_float(r[0]) + __uint_as_float(r[1]);
            };
            const float w02 = fold32(acc[0], acc[2]), w13 = fold32(acc[1], acc[3]);
            const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(w02), __float_as_uint(w13), false, false);
            float own_sum = __uint_as_float(r[0]) + __uint_as_float(r[1]);
            if constexpr (NSPLIT == 8) own_sum += row_from_up<8>(own_sum);
            float out_v = own_sum + D_u * code_byte_to_float(code, 0);
            if constexpr (HAS_Z) out_v *= sh.gate[code >> 8];
            sm.out[4 * tq + qslice][out_col] = __float2half(out_v);
        }
        gemm::wave_lds_sync();
        const int t = (block * waves + wave) * T + out_step;
        if (out_mine && t < L) {
            const uint2 v = *reinterpret_cast<const uint2*>(&sm.out[out_step][out_ch]);
            __half* const to = out_b + t * p.out_l_stride;
            if (vec_out) {
                *reinterpret_cast<uint2*>(to) = v;
            } else {
                const __half* from = reinterpret_cast<const __half*>(&v);
                for (int e = 0; e < 4; ++e) to[e * p.out_d_stride] = from[e];
            }
        }
        gemm::wave_lds_sync();                             // (the next block's rows come after this one's last reads)
    }
    if (wave == waves - 1 && c_ok) {                       // (steps past the end leave the state alone)
        const int64_t base = (static_cast<int64_t>(b) * p.dim + c) * 16 + slice * NPL;
        const float s_state = p.last_state_i8 ? *p.scale_ssm_state : 1.0f;
#pragma unroll
        for (int i = 0; i < NPL; ++i) {
            if (p.last_state_f32) p.last_state_f32[base + i] = h[i];
            if (p.last_state_i8) p.last_state_i8[base + i] = sat8_half_away(h[i] / s_state);
        }
    }
}

template <int NSPLIT, bool HAS_Z, int DTK>
int launch_one(const QaSScanParams& p, const SscanDtProj& dtp, int waves, hipStream_t stream) {
    using Cfg = WavesCfg<NSPLIT>;
    const int vec_out = p.out_d_stride == 1 && (reinterpret_cast<uintptr_t>(p.out) & 7u) == 0 && p.out_batch_stride % 4 == 0 && p.out_l_stride % 4 == 0;
    constexpr int kFew = max_waves(4), kMost = max_waves(NSPLIT);
    const auto kernel = waves <= kFew ? scan_waves_kernel<NSPLIT, kFew, HAS_Z, DTK> : scan_waves_kernel<NSPLIT, kMost, HAS_Z, DTK>;
    const int bytes = lds_bytes<NSPLIT>(waves, DTK);
    // more LDS than a kernel gets by default: the limit is the kernel's, the same for launches of any number of waves (other threads make theirs)
    const int limit = lds_bytes<NSPLIT>(waves <= kFew ? kFew : kMost, DTK);
    static_assert(lds_bytes<NSPLIT>(kMost, DTK) <= 160 * 1024, "LDS of a CU");
    if (bytes > 65536 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, limit) != hipSuccess) return check_launch();
    hipLaunchKernelGGL(kernel, dim3((p.dim + Cfg::kCh - 1) / Cfg::kCh, static_cast<unsigned>(p.batch)), dim3(64 * waves), bytes, stream, p, dtp, vec_out);
    return check_launch();
}

template <int NSPLIT>
int launch(const QaSScanParams& p, const SscanDtProj* dt, int waves, hipStream_t stream) {
    const SscanDtProj none = {};
    if (!dt) return p.z ? launch_one<NSPLIT, true, 0>(p, none, waves, stream) : launch_one<NSPLIT, false, 0>(p, none, waves, stream);
    if (dt->rank <= 64) return launch_one<NSPLIT, true, 1>(p, *dt, waves, stream);
    if (dt->rank <= 128) return launch_one<NSPLIT, true, 2>(p, *dt, waves, stream);
    return launch_one<NSPLIT, true, 3>(p, *dt, waves, stream);
}

}  // namespace

int sscan_waves_fwd(const QaSScanParams& p, const SscanDtProj* dt, int lanes, int waves, hipStream_t stream) {
    if ((lanes != 4 && lanes != 8) || waves < 1 || waves > max_waves(lanes)) return QA_ERR_UNSUPPORTED;
    return lanes == 4 ? launch<4>(p, dt, waves, stream) : launch<8>(p, dt, waves, stream);
}

// A block takes a time of its own, one for every wave that a SIMD holds and one for every predecessor that the last wave chains
// up; 956 launches of 1 ... 8 prompts of 16 ... 4096 steps x 512 ... 5120 channels lie within 6 % of this (rms), and the choice is the
// fastest launch or within 3 % of it in all of them.  While workgroups are no more than a SIMD has room for (three waves of these
// registers, four of sixteen-wave workgroups) nothing waits for a place; beyond, the one pass of sscan_tm.hip is the shorter one
// (3 x 1021 x 5120 106 us against 102, 8 x 512 x 2048 56 and 52), as it is for some short prompts (plan_of there).
ScanWavesPlan scan_waves_plan(const QaSScanParams& p, int cus) {
    const auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
    ScanWavesPlan best = {8, 0, kScanWavesNever};
    // (Without softplus step sizes may be negative, and the decay of all of a wave's steps beyond fp32 - a factor that nothing else would
    // make of them while the state is still zero: the product is no number then.)
    if (!p.delta_softplus) return best;
    for (const int lanes : {4, 8}) {
        const int64_t steps = lanes == 4 ? WavesCfg<4>::T : WavesCfg<8>::T, channels = lanes == 4 ? WavesCfg<4>::kCh : WavesCfg<8>::kCh;
        const int64_t per_cu = up(up(p.dim, channels) * p.batch, cus), pieces = up(p.seqlen, steps);
        for (int w = 1; w <= std::min<int64_t>(max_waves(lanes), pieces); ++w) {
            const int64_t per_simd = per_cu * up(w, 4), blocks = up(pieces, w);
            // (workgroups of other sizes share SIMDs unevenly)
            if (per_simd > (w <= 12 ? 3 : 4) || (per_cu > 1 && w % 4 != 0 && blocks > 1)) continue;
            // (three workgroups on a CU begin out of step with each other)
            const int64_t crowd = lanes == 4 && per_cu > 2 ? 1300 + 700 * std::min<int64_t>(blocks - 1, 2) : 0;
            const int64_t ns = 3590 + crowd + blocks * (lanes == 4 ? 1020 + 1030 * per_simd + 50 * w : 1550 + 1300 * per_simd + 40 * w);
            if (ns < best.ns) best = {lanes, w, ns};
        }
    }
    return best;
}

}  // namespace qa
