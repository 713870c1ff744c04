// Mamba1 int8 selective scan over token-major rows (channels contiguous), sixteen states: the scan inside the assembled
// mixer.  Arithmetic as in sscan.hip (reference csrc/selective_scan/quant_sscan_fwd_kernel.cuh:110-293).
//
// The walk is the one of sscan_fwd_pre_body: what does not depend on the state index is taken out of the time loop and
// evaluated while a tile of T steps is staged (step size with bias and softplus, step size x input, as fp32 rows in LDS); B
// and C are converted once per workgroup; the time loop is the recurrence alone.  What differs:
//
// Bound by vector issue: at 8 x 2048 steps x 5120 channels the recurrence is 16 exponentials (a quarter of the rate) and 64
// multiplies and adds per channel and step, 391 us of which about 300 are issue; the bytes would take 60.  With B x (step size
// x input) as matrix instructions and the sums over lanes by swaps 377 (16 x 512 x 5120, four lanes for all, 176 -> 168).
//
// Staging.  A wave stages its own channels with dword loads of four channels and one step.  Tails need no path of their
// own: steps past the end read the last step and get step size zero.
//
// Step sizes.  With SscanDtProj the codes of the step sizes are not read: dt_proj is a product of a tile's rows of x_proj's
// output (up to 192 codes, through LDS) with the weights of the wave's channels, two to twelve v_mfma_i32_16x16x64_i8 a tile
// with the weights in registers for good, and its result leaves the matrix cores exactly as the staging wants it - four
// channels of one step per lane.  The projection as a launch of its own took 47 us at 16384 tokens x 5120 channels and 13 at
// 3063 (nearly all of it writing the codes and reading them back); the scan with it takes 384 and 108 us, and took 384 and
// 107 with the codes read.
//
// Lanes.  NSPLIT lanes share a channel, 16 / NSPLIT states each: four when there are waves enough, eight when there are fewer -
// a wave's time is then set by its own latencies, and more, shorter waves hide more of them (64 steps of 1536 channels: 10.1 us
// with four lanes, 7.6 with eight).  With fewer still the time is cut over the waves of a workgroup (sscan_waves.hip).
//
// Segments.  Few channels of a long sequence leave most of the chip idle even so: the sequence is cut into segments that are
// scanned side by side, one pass for every segment's end state from a zero state and the sum of its step sizes (OUT false: no
// C, no outputs), one that starts every segment from the state its predecessors chain up to.  By the rule below (256 CUs) that is from
// 832 steps on with up to 1280 channels of one sequence or 1152 of two; wider layers are scanned over waves.  Step sizes that may be
// negative are not (scan_waves_plan), and take segments by the same costs in layers of up to 5120 channels (one sequence, from 576 steps on).
#include "conv_common.hpp"
#include "gemm_core.hpp"
#include "mixer_common.hpp"
#include "sscan_common.hpp"
#include "sscan_waves.hpp"

#include <algorithm>

namespace qa {
namespace {

constexpr int kThreads = 256;
using gemm::v4i;
typedef float v16f __attribute__((ext_vector_type(16)));

template <int NSPLIT>
struct TmCfg {
    static constexpr int T = 32;                           // steps per tile
    static constexpr int NPL = 16 / NSPLIT;                // states per lane
    static constexpr int kCh = kThreads / NSPLIT;          // channels per workgroup
    static constexpr int kWaveCh = 64 / NSPLIT;            // channels per wave
    static constexpr int kSteps = kWaveCh * T / 4 / 64;    // steps a lane stages per tile, of four channels
    static constexpr int kPitch = T + 4;                   // floats per row of per-step values
    static constexpr int kUzPitch = T + 4;                 // 16-bit (u | z << 8) codes per row
    static constexpr int kOutPitch = kCh + 8;              // halves; keeps rows 16-byte aligned
    static constexpr int kBcWords = T / 32;                // dwords of B / C codes a thread stages per tile
    static constexpr int kXSets = T / 16;                  // sixteen-step products per tile
};

template <class Cfg, int DTK>
struct TmSmem {
    __attribute__((aligned(16))) float d[Cfg::kCh][Cfg::kPitch];     // step size
    __attribute__((aligned(16))) float du[Cfg::kCh][Cfg::kPitch];    // step size x input code
    __attribute__((aligned(16))) uint16_t uz[Cfg::kCh][Cfg::kUzPitch];
    // the two tiles the waves share, twice each (one is scanned out of while the next is staged): B | C of four steps by
    // state, so that a lane reads four steps of a state with one 16-byte load
    __attribute__((aligned(16))) float bc[2][Cfg::T / 4][2][16][4];
    __attribute__((aligned(16))) __half out[2][Cfg::T][Cfg::kOutPitch];
    // x_proj's rows of two tiles, in pieces of 16 codes: piece (kb * T + row) * 4 + s holds codes 64 kb + 16 (s ^ (row / 4) % 4)
    __attribute__((aligned(16))) int8_t x[DTK ? 2 : 1][DTK ? DTK * Cfg::T * 64 : 16];
    float gate_table[256];             // SiLU gate per z code (indexed by the raw byte)
};

// DTK: 64-code pieces of dt_proj's K (0: the step size codes are read from p.delta).  SPREAD: a channel's lanes are 16 apart
// (and 8, when there are eight), not neighbours.
template <int NSPLIT, bool HAS_Z, bool OUT, int DTK, bool SPREAD>
__device__ __forceinline__ void scan_tm_body(const QaSScanParams& p, const SscanDtProj& dtp, int vec_out, int c0, int y, TmSmem<TmCfg<NSPLIT>, DTK>& sm) {
    using Cfg = TmCfg<NSPLIT>;
    constexpr int T = Cfg::T, NPL = Cfg::NPL, kCh = Cfg::kCh, kSteps = Cfg::kSteps;
    constexpr bool kOuter = NSPLIT == 4;                   // B x (step size x input) on the matrix cores
    static_assert(NSPLIT <= 8 && (SPREAD || !kOuter), "lanes as 16 x 16 products leave them");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int kWaveCh = Cfg::kWaveCh;
    const int c_local = SPREAD ? wave * kWaveCh + lane % kWaveCh : tid / NSPLIT;
    const int slice = SPREAD ? (lane & 15) / kWaveCh * 4 + (lane >> 4) : tid % NSPLIT, qslice = slice & 3;
    const int c = c0 + c_local;
    const bool c_ok = c < p.dim;
    const int cc = c_ok ? c : p.dim - 1;                   // clamped channel for parameter loads
    const int segments = max(p.segments, 1), per_entry = OUT ? segments : segments - 1;
    const int b = y / per_entry, seg_i = y - b * per_entry;
    const int t_base = seg_i * p.segment_len;              // (0 without segments)
    const int L = segments > 1 ? min(p.segment_len, p.seqlen - t_base) : p.seqlen;
    const int n_tiles = (L + T - 1) / T;
    const bool softplus = p.delta_softplus != 0;

    // This lane's share of a wave's tile: four channels from ch4 on, steps step0 .. step0 + kSteps - 1.  The arrangement is
    // the one in which 16 x 16 products leave the matrix cores: lane l holds rows 4 (l / 16) .. + 3 (channels) of column
    // l % 16 (steps).
    const int g = lane >> 4, j = lane & 15;
    const int quad = NSPLIT == 4 ? g : g & 1;
    const int step0 = NSPLIT == 4 ? 2 * j : j + 16 * (g >> 1);
    const int lc4 = wave * Cfg::kWaveCh + 4 * quad;
    const int ch4 = min(c0 + lc4, p.dim - 4);              // channels past the last read the last four; nothing of theirs is stored

    // Addresses: a wave-uniform pointer per tile and a lane's 32-bit offset in it (two scalar additions per tile; a 64-bit
    // multiply per load is eight quarter-rate instructions)
    const int8_t* u_at = p.u + b * p.u_batch_stride + t_base * p.u_l_stride;
    const int8_t* z_at = HAS_Z && OUT ? p.z + b * p.z_batch_stride + t_base * p.z_l_stride : nullptr;
    const int8_t* d_at = DTK == 0 ? p.delta + b * p.delta_batch_stride + t_base * p.delta_l_stride : nullptr;
    const int dw = tid & 7, bc_step = tid >> 3;            // B | C: dword tid % 8 of a step's sixteen B and sixteen C codes
    const int bc_ls = static_cast<int>(dw < 4 ? p.B_l_stride : p.C_l_stride);
    const int8_t* bc_at = (dw < 4 ? p.B + b * p.B_batch_stride + t_base * p.B_l_stride : p.C + b * p.C_batch_stride + t_base * p.C_l_stride) + 4 * (dw & 3);
    uint32_t off_u[kSteps], off_z[kSteps], off_d[kSteps], off_bc[Cfg::kBcWords];
    auto set_offsets = [&](int last) {                     // steps past `last` of a tile read that one
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            const int t = min(step0 + i, last);
            off_u[i] = t * static_cast<int>(p.u_l_stride) + ch4;
            if constexpr (HAS_Z && OUT) off_z[i] = t * static_cast<int>(p.z_l_stride) + ch4;
            if constexpr (DTK == 0) off_d[i] = t * static_cast<int>(p.delta_l_stride) + ch4;
        }
#pragma unroll
        for (int i = 0; i < Cfg::kBcWords; ++i) off_bc[i] = min(bc_step + 32 * i, last) * bc_ls;
    };
    set_offsets(T - 1);
    uint32_t r_u[kSteps], r_z[kSteps], r_d[kSteps], r_bc[Cfg::kBcWords];
    auto issue_loads = [&](int tile) {
        if ((tile + 1) * T > L) set_offsets(L - 1 - tile * T);          // (the last one: the offsets are not needed again)
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            r_u[i] = *reinterpret_cast<const uint32_t*>(u_at + off_u[i]);
            if constexpr (DTK == 0) r_d[i] = *reinterpret_cast<const uint32_t*>(d_at + off_d[i]);
            if constexpr (HAS_Z && OUT) r_z[i] = *reinterpret_cast<const uint32_t*>(z_at + off_z[i]);
        }
#pragma unroll
        for (int i = 0; i < Cfg::kBcWords; ++i) r_bc[i] = *reinterpret_cast<const uint32_t*>(bc_at + off_bc[i]);
        u_at += T * p.u_l_stride;
        if constexpr (DTK == 0) d_at += T * p.delta_l_stride;
        if constexpr (HAS_Z && OUT) z_at += T * p.z_l_stride;
        bc_at += static_cast<int64_t>(T) * bc_ls;
    };

    // dt_proj: x_proj's rows go straight to LDS, two tiles ahead (every wave reads all of them, so they have to pass a
    // barrier); the waves share the instructions.  Rows past the end read as zeros.
    constexpr int kXLoads = DTK ? (DTK * T * 4 / 64 + 3) / 4 : 1;
    const int x_ls = static_cast<int>(dtp.x_l_stride);
    v4i rsrc_x = {};
    int off_x[kXLoads];
    if constexpr (DTK != 0) {
        rsrc_x = gemm::make_rsrc(dtp.x + b * dtp.x_batch_stride + t_base * dtp.x_l_stride, (L - 1) * x_ls + dtp.rank);
#pragma unroll
        for (int i = 0; i < kXLoads; ++i) {
            const int piece = (4 * i + wave) * 64 + lane, row = piece / 4 % T, kb = piece / (4 * T);
            off_x[i] = row * x_ls + 64 * kb + 16 * ((piece & 3) ^ ((row >> 2) & 3));
        }
    }
    auto load_x = [&](int tile, int into) {
        if constexpr (DTK != 0) {
#pragma unroll
            for (int i = 0; i < kXLoads; ++i)
                if ((4 * i + wave) * 64 < DTK * T * 4) gemm::buffer_load_lds_b128(rsrc_x, gemm::lds_offset_of(sm.x[into]) + (4 * i + wave) * 1024, off_x[i] + tile * T * x_ls);
        }
    };

    load_x(0, 0);
    if (n_tiles > 1) load_x(1, 1);
    issue_loads(0);
    // dt_proj's weights as the first operand: row j is channel j of the wave (again from the start when it has fewer)
    v4i fw[DTK ? DTK : 1];
    float dt_col[4] = {}, dt_row = 0.0f;
    if constexpr (DTK != 0) {
        const int8_t* row = dtp.w + static_cast<int64_t>(min(c0 + wave * Cfg::kWaveCh + j % Cfg::kWaveCh, p.dim - 1)) * dtp.rank;
#pragma unroll
        for (int kb = 0; kb < DTK; ++kb) fw[kb] = *reinterpret_cast<const v4i*>(row + min(64 * kb + 16 * g, dtp.rank - 16));
#pragma unroll
        for (int e = 0; e < 4; ++e) dt_col[e] = dtp.col_scale[dtp.col_numel == 1 ? 0 : ch4 + e];
#pragma unroll
        for (int kb = 0; kb < DTK; ++kb)
            if (64 * kb + 16 * g >= dtp.rank) fw[kb] = v4i{0, 0, 0, 0};
        dt_row = *dtp.row_scale;
    }
    uint32_t db_codes = 0, A_codes[NPL];
    if (p.delta_bias) __builtin_memcpy(&db_codes, p.delta_bias + ch4, 4);
#pragma unroll
    for (int i = 0; i < NPL; ++i) A_codes[i] = static_cast<uint8_t>(p.A_log[cc * p.A_d_stride + (slice * NPL + i) * p.A_dstate_stride]);
    const float D_code = p.D ? static_cast<float>(p.D[cc]) : 0.0f;
    const float s_u = *p.scale_u, s_dt = *p.scale_delta, s_A = *p.scale_A, s_B = *p.scale_B, s_C = *p.scale_C;
    const float s_z = HAS_Z ? *p.scale_z : 0.0f, s_D = p.D ? *p.scale_D : 0.0f, s_db = p.delta_bias ? *p.scale_delta_bias : 0.0f;
    const float D_u = (s_D * D_code) * s_u;                // skip weight per input code
    const float bc_scale = dw < 4 ? s_B * s_u : s_C;       // the input scale rides with B and D: (s_B q_B) (dt (s_u q_u))
    float db4[4], dt_sum4[OUT ? 1 : 4] = {};
#pragma unroll
    for (int e = 0; e < 4; ++e) db4[e] = p.delta_bias ? s_db * code_byte_to_float(db_codes, e) : 0.0f;

    float A2[NPL], h[NPL];
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
        h[i] = 0.0f;
        A2[i] = -expf(s_A * code_byte_to_float(A_codes[i], 0)) * kLog2e;
    }
    if (OUT && seg_i > 0) {
        const int first = b * (segments - 1);
        for (int sp = first; sp < first + seg_i; ++sp) {
            const float sd = p.carry_dt_sum[static_cast<int64_t>(sp) * p.dim + cc];
#pragma unroll
            for (int i = 0; i < NPL; ++i)
                h[i] = __builtin_fmaf(fast_exp2(sd * A2[i]), h[i], p.carry_state[(static_cast<int64_t>(sp) * p.dim + cc) * 16 + slice * NPL + i]);
        }
    }

    // from the registers of issue_loads (and x of the same tile) into the wave's rows and copy `into` of the shared tile
    auto stage = [&](int tile, int into) {
        float dv[kSteps][4], duv[kSteps][4];
        if constexpr (DTK != 0) {
            v4i acc[Cfg::kXSets];
#pragma unroll
            for (int s = 0; s < Cfg::kXSets; ++s) {
                const int row = NSPLIT == 4 ? 2 * j + s : j + 16 * s;
                acc[s] = v4i{0, 0, 0, 0};
#pragma unroll
                for (int kb = 0; kb < DTK; ++kb) {
                    const v4i fx = *reinterpret_cast<const v4i*>(&sm.x[into][((kb * T + row) * 4 + (g ^ ((row >> 2) & 3))) * 16]);
                    acc[s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw[kb], fx, acc[s], 0, 0, 0);
                }
            }
#pragma unroll
            for (int i = 0; i < kSteps; ++i) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    int sum;
                    if constexpr (NSPLIT == 4) sum = acc[i][e];
                    else sum = g < 2 ? acc[0][e] : acc[1][e];
                    float v = dt_col[e] * (dt_row * static_cast<float>(sum));
                    v = __builtin_amdgcn_fmed3f(__builtin_rintf(v), -128.0f, 127.0f);          // the int8 code
                    dv[i][e] = __builtin_fmaf(s_dt, v, db4[e]);
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < kSteps; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) dv[i][e] = __builtin_fmaf(s_dt, code_byte_to_float(r_d[i], e), db4[e]);
        }
        if (softplus) {                  // one uniform branch per tile: the evaluations below overlap
#pragma unroll
            for (int i = 0; i < kSteps; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) dv[i][e] = softplus20_flat(dv[i][e]);
        }
        if ((tile + 1) * T > L) {
            // ragged last tile: steps past the end of the sequence must leave the state alone (a = 1, b = 0)
#pragma unroll
            for (int i = 0; i < kSteps; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) dv[i][e] = tile * T + step0 + i < L ? dv[i][e] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < kSteps; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (!OUT) dt_sum4[e] += dv[i][e];
                duv[i][e] = dv[i][e] * code_byte_to_float(r_u[i], e);
            }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (kSteps == 2) {
                *reinterpret_cast<float2*>(&sm.d[lc4 + e][step0]) = make_float2(dv[0][e], dv[1][e]);
                *reinterpret_cast<float2*>(&sm.du[lc4 + e][step0]) = make_float2(duv[0][e], duv[1][e]);
            } else {
                sm.d[lc4 + e][step0] = dv[0][e];
                sm.du[lc4 + e][step0] = duv[0][e];
            }
            if constexpr (OUT) {
                // (u z) of this channel's steps, bytewise
                const uint32_t pick = 0x0c0c0400u + 0x0101u * e;
                const uint32_t first = __builtin_amdgcn_perm(HAS_Z ? r_z[0] : 0u, r_u[0], pick);
                if constexpr (kSteps == 2) {
                    const uint32_t second = __builtin_amdgcn_perm(HAS_Z ? r_z[1] : 0u, r_u[1], pick);
                    *reinterpret_cast<uint32_t*>(&sm.uz[lc4 + e][step0]) = first | (second << 16);
                } else {
                    sm.uz[lc4 + e][step0] = static_cast<uint16_t>(first);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < Cfg::kBcWords; ++i) {
            const int t = bc_step + 32 * i;
#pragma unroll
            for (int e = 0; e < 4; ++e) sm.bc[into][t >> 2][dw >> 2][4 * (dw & 3) + e][t & 3] = bc_scale * code_byte_to_float(r_bc[i], e);
        }
    };

    // operands of one group of four steps
    struct Group {
        float d[4], du[kOuter ? 1 : 4], B[kOuter ? 1 : NPL][kOuter ? 1 : 4];
        v16f bdu;                       // with kOuter B x du instead, step s and state n of this lane in 4 s + n
        uint32_t code;                  // of the step this lane owns: u in byte 0, z in byte 1
    };
    // Four lanes per channel: these products on the matrix cores.  A 16 x 16 x 1 instruction of four blocks, a block per step,
    // multiplies the B of sixteen states (rows) with the du of sixteen channels (columns) and leaves four rows of a column - a
    // lane's states and channel - in each lane, rounded as the sixteen multiplications it stands for; a group's are made
    // during the group before.  The instruction keeps the vector units from about eight of their own (16 x 512 steps x 5120
    // channels 162 -> 157 us, 8 x 2048 x 4096 274 -> 263); with eight lanes per channel, where a group takes two of them for
    // eight multiplications, it loses (4 x 2048 x 5120 225 -> 256).
    struct Factors {                    // B of state j, du of this channel, both of step g
        float b, du;
    };
    auto fetch_factors = [&](Factors& o, int tq, int from) {
        o.b = sm.bc[from][tq][0][j][g];
        o.du = sm.du[c_local][tq * 4 + g];
    };
    auto multiply = [&](Group& o, const Factors& x) {
        constexpr v16f zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        o.bdu = __builtin_amdgcn_mfma_f32_16x16x1f32(x.b, x.du, zero, 0, 0, 0);
    };
    auto fetch = [&](Group& o, int tq, int from) {
        if constexpr (OUT) o.code = sm.uz[c_local][tq * 4 + qslice];
        const float4 d4 = *reinterpret_cast<const float4*>(&sm.d[c_local][tq * 4]);
        o.d[0] = d4.x; o.d[1] = d4.y; o.d[2] = d4.z; o.d[3] = d4.w;
        if constexpr (!kOuter) {
            const float4 du4 = *reinterpret_cast<const float4*>(&sm.du[c_local][tq * 4]);
            o.du[0] = du4.x; o.du[1] = du4.y; o.du[2] = du4.z; o.du[3] = du4.w;
#pragma unroll
            for (int n = 0; n < NPL; ++n) {
                const float4 Bv = *reinterpret_cast<const float4*>(sm.bc[from][tq][0][slice * NPL + n]);
                o.B[n][0] = Bv.x; o.B[n][1] = Bv.y; o.B[n][2] = Bv.z; o.B[n][3] = Bv.w;
            }
        }
    };
    // the column of the output tile a lane writes: with more than four lanes per channel only the first quad's sums are
    // complete (see below), the others go to the padding behind the row
    const int out_col = slice >= 4 ? kCh + (c_local & 7) : c_local;

    // All T / 4 groups of four steps, also of a ragged last tile: steps past the end have step size 0 and leave the state
    // alone, and their output rows are never stored.  The operands of a group are fetched while the group before is being
    // computed.
    auto compute = [&](int from) {
        __half* const out_at = &sm.out[from][qslice][out_col];
        Group grp[2];
        Factors fac[2];
        fetch(grp[0], 0, from);
        if constexpr (kOuter) {
            fetch_factors(fac[0], 0, from);
            fetch_factors(fac[1], 1, from);
            multiply(grp[0], fac[0]);
        }
#pragma unroll
        for (int tq = 0; tq < T / 4; ++tq) {
            Group& o = grp[tq & 1];
            float gate = 1.0f, C[NPL][4];
            if constexpr (OUT) {
                // (wanted last: the exponentials cover the time these take, and a third of the operands need no second set
                // of registers)
#pragma unroll
                for (int n = 0; n < NPL; ++n) {
                    const float4 Cv = *reinterpret_cast<const float4*>(sm.bc[from][tq][1][slice * NPL + n]);
                    C[n][0] = Cv.x; C[n][1] = Cv.y; C[n][2] = Cv.z; C[n][3] = Cv.w;
                }
                if constexpr (HAS_Z) gate = sm.gate_table[o.code >> 8];
            }
            if (tq + 1 < T / 4) fetch(grp[(tq + 1) & 1], tq + 1, from);
            if constexpr (kOuter) {
                if (tq + 2 < T / 4) fetch_factors(fac[tq & 1], tq + 2, from);
                if (tq + 1 < T / 4) multiply(grp[(tq + 1) & 1], fac[(tq + 1) & 1]);
            }
            // keep the reads above ahead of this group's arithmetic (the scheduler would sink them to their first use, and a
            // wave would then wait for LDS once or twice per group)
            __builtin_amdgcn_sched_barrier(0);
            float acc[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                acc[s] = 0.0f;
#pragma unroll
                for (int n = 0; n < NPL; ++n) {
                    const float a = fast_exp2(o.d[s] * A2[n]);
                    if constexpr (kOuter) h[n] = __builtin_fmaf(a, h[n], o.bdu[4 * s + n]);
                    else h[n] = __builtin_fmaf(a, h[n], o.B[n][s] * o.du[s]);
                    if constexpr (OUT) acc[s] = n == 0 ? h[n] * C[n][s] : __builtin_fmaf(h[n], C[n][s], acc[s]);
                }
            }
            if constexpr (!OUT) {
#pragma unroll
                for (int n = 0; n < NPL; ++n) asm volatile("" : "+v"(h[n]));      // (no output holds a group's arithmetic in its place)
                continue;
            }
            // each of four lanes completes the step it owns: a transposing reduction (keep one half, hand the other half over)
            // instead of four full ones.  Lanes 32 and 16 apart exchange halves with one swap for two values; neighbours, which
            // select what they keep and what they hand over, take half as many instructions again (four lanes 278 -> 274 us at
            // 8 x 2048 x 4096; both kinds of workgroup at 8 x 2048 x 5120 359 -> 351; eight lanes in a launch of their own, whose
            // waves wait for more than instructions, 3 x 1021 x 5120 100 -> 99 and short segments 13.0 -> 13.5: left as
            // neighbours).  The sums of a channel's other quads arrive by row shifts inside the additions.
            float own_sum;
            if constexpr (SPREAD) {
                const auto fold32 = [](float a, float b) {
                    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
                    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
                };
                const float w02 = fold32(acc[0], acc[2]), w13 = fold32(acc[1], acc[3]);
                const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(w02), __float_as_uint(w13), false, false);
                own_sum = __uint_as_float(r[0]) + __uint_as_float(r[1]);
                if constexpr (NSPLIT == 8) own_sum += row_from_up<8>(own_sum);
            } else {
                const bool odd = qslice & 1, hi = qslice & 2;
                const float w01 = (odd ? acc[1] : acc[0]) + quad_xor<1>(odd ? acc[0] : acc[1]);
                const float w23 = (odd ? acc[3] : acc[2]) + quad_xor<1>(odd ? acc[2] : acc[3]);
                own_sum = (hi ? w23 : w01) + quad_xor<2>(hi ? w01 : w23);
                own_sum += row_from_up<4>(own_sum);
            }
            float out_v = own_sum + D_u * code_byte_to_float(o.code, 0);
            if constexpr (HAS_Z) out_v *= gate;
            out_at[tq * 4 * Cfg::kOutPitch] = __float2half(out_v);
        }
    };

    // the tile's output rows: eight channels of one row a thread
    constexpr int kChunks = kCh / 8;
    const int out_t = tid / kChunks, ch8 = (tid % kChunks) * 8;
    __half* out_row = nullptr;
    bool out_mine = false, out_vec = false;
    if constexpr (OUT) {
        out_row = static_cast<__half*>(p.out) + b * p.out_batch_stride + (t_base + out_t) * p.out_l_stride + (c0 + ch8) * p.out_d_stride;
        out_mine = out_t < T && c0 + ch8 < p.dim;
        out_vec = vec_out && c0 + ch8 + 8 <= p.dim;
    }
    auto store = [&](int tile, int from) {
        if constexpr (OUT) {
            if (out_mine && tile * T + out_t < L) {
                if (out_vec) {
                    *reinterpret_cast<uint4*>(out_row) = *reinterpret_cast<const uint4*>(&sm.out[from][out_t][ch8]);
                } else {
                    for (int e = 0; e < 8; ++e) {
                        if (c0 + ch8 + e < p.dim) out_row[e * p.out_d_stride] = sm.out[from][out_t][ch8 + e];
                    }
                }
            }
            out_row += T * p.out_l_stride;
        }
    };

    if constexpr (HAS_Z && OUT) sm.gate_table[tid] = silu_gate(s_z * static_cast<float>(static_cast<int8_t>(tid)));
    if constexpr (DTK != 0) {
        __builtin_amdgcn_s_waitcnt(gemm::vmcnt_imm(0));
        __syncthreads();
    }
    stage(0, 0);
    __syncthreads();
    // Tile by tile, the shared tiles alternating between their two copies, one barrier each; the last one, which has nothing
    // to stage, on its own (as a branch inside the loop it leaves the compiler unsure which loads are in flight, and it waits
    // for the stores of the tile before)
    for (int tile = 0; tile + 1 < n_tiles; ++tile) {
        const int from = tile & 1;
        if (tile + 2 < n_tiles) load_x(tile + 2, from);
        issue_loads(tile + 1);
        compute(from);
        stage(tile + 1, from ^ 1);           // (every wave left that copy at the barrier of the tile before)
        if constexpr (DTK != 0) __builtin_amdgcn_s_waitcnt(gemm::vmcnt_imm(0));
        __syncthreads();                     // this tile's outputs, the next tile's B | C and x two tiles on are complete
        store(tile, from);
    }
    compute((n_tiles - 1) & 1);
    __syncthreads();
    store(n_tiles - 1, (n_tiles - 1) & 1);

    if constexpr (!OUT) {
        // the sum of the step sizes of each channel (the lanes of a quad of channels staged different steps), and its end
        // state, as fp32
        constexpr int kQuads = Cfg::kWaveCh / 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int m = 1; m < 16; m <<= 1) dt_sum4[e] += __shfl_xor(dt_sum4[e], m);
            if constexpr (kQuads <= 2) dt_sum4[e] += __shfl_xor(dt_sum4[e], 32);
            if (j == 0 && g == quad && c0 + lc4 < p.dim) p.dt_sum_out[static_cast<int64_t>(y) * p.dim + c0 + lc4 + e] = dt_sum4[e];
        }
        if (c_ok) {
            float* to = const_cast<float*>(p.carry_state) + (static_cast<int64_t>(y) * p.dim + c) * 16 + slice * NPL;
#pragma unroll
            for (int i = 0; i < NPL; ++i) to[i] = h[i];
        }
    } else if (c_ok && seg_i == segments - 1) {
        const int64_t base = (static_cast<int64_t>(b) * p.dim + c) * 16 + slice * NPL;
        const float s_state = p.last_state_i8 ? *p.scale_ssm_state : 1.0f;
#pragma unroll
        for (int i = 0; i < NPL; ++i) {
            if (p.last_state_f32) p.last_state_f32[base + i] = h[i];
            if (p.last_state_i8) p.last_state_i8[base + i] = sat8_half_away(h[i] / s_state);
        }
    }
}

template <int NSPLIT, bool HAS_Z, bool OUT, int DTK>
__global__ __launch_bounds__(kThreads, 3) void scan_tm_kernel(QaSScanParams p, SscanDtProj dtp, int vec_out) {
    __shared__ TmSmem<TmCfg<NSPLIT>, DTK> sm;
    scan_tm_body<NSPLIT, HAS_Z, OUT, DTK, NSPLIT == 4>(p, dtp, vec_out, blockIdx.x * TmCfg<NSPLIT>::kCh, blockIdx.y, sm);
}

// Two kinds of workgroup in one launch: the first `blocks_a` of a batch entry take 64 channels each with four lanes per
// channel, the others 32 with eight (see sscan_fwd_mixed_kernel in sscan.hip).
template <bool HAS_Z, int DTK>
__global__ __launch_bounds__(kThreads, 3) void scan_tm_mixed_kernel(QaSScanParams p, SscanDtProj dtp, int vec_out, int blocks_a) {
    __shared__ union Smem {
        TmSmem<TmCfg<4>, DTK> a;
        TmSmem<TmCfg<8>, DTK> b;
        __device__ Smem() {}
    } sm;
    const int bx = blockIdx.x;
    if (bx < blocks_a) scan_tm_body<4, HAS_Z, true, DTK, true>(p, dtp, vec_out, bx * 64, blockIdx.y, sm.a);
    else scan_tm_body<8, HAS_Z, true, DTK, true>(p, dtp, vec_out, blocks_a * 64 + (bx - blocks_a) * 32, blockIdx.y, sm.b);
}

// How a launch is laid out: lanes per channel (0: two kinds of workgroup, `blocks_a` of the first) and segments.
struct TmPlan {
    int lanes, blocks_a, segments, segment_len;
    int waves;                 // of a workgroup that cuts the time over them (sscan_waves.hip); 0: not so
};

// Nanoseconds per step of a launch of eight lanes per channel with so many waves on its busiest SIMD, as measured (a wave alone is
// bound by its own latencies; from about three on the vector units are), and the same without outputs.
int step_cost(bool out, int64_t waves) {
    static constexpr int kOut[4] = {63, 85, 117, 152}, kState[4] = {45, 60, 78, 100};
    return static_cast<int>(waves <= 4 ? (out ? kOut : kState)[waves - 1] : waves * (out ? 38 : 25));
}

TmPlan plan_of(const QaSScanParams& p) {
    TmPlan r = {4, 0, 1, p.seqlen, 0};
    const int cus = compute_units();
    const int64_t simds = 4LL * cus, rows = static_cast<int64_t>(p.batch) * p.dim;
    const int64_t waves4 = rows / 16, q = waves4 / simds, rest = waves4 % simds;
    auto cut = [&](int segments) {
        r.segment_len = ((p.seqlen + segments - 1) / segments + 31) / 32 * 32;
        r.segments = (p.seqlen + r.segment_len - 1) / r.segment_len;
    };
    if (p.mapping != 0) {
        r.lanes = (p.mapping >> 20) & 0xff;
        r.blocks_a = r.lanes == 0 ? p.mapping & 0xfffff : 0;
        if (r.lanes == kScanWavesMapping) {
            const ScanWavesPlan over_waves = scan_waves_plan(p, cus);
            r.lanes = over_waves.lanes;
            r.waves = over_waves.waves;
        } else if (r.lanes >= kScanWavesNamed && r.lanes < kScanWavesNamed + 64) {
            r.waves = r.lanes % 32 + 1;
            r.lanes = r.lanes < kScanWavesNamed + 32 ? 4 : 8;
        }
        if (r.lanes == 8 && r.waves == 0 && p.segments > 1) cut(p.segments);
    } else if (2 * waves4 <= 3 * simds) {
        // Up to one and a half waves of four lanes per SIMD eight lanes are the faster ones (8 x 512 x 3072 channels 63 us against
        // 72; 13 x 512 x 2048 78 against 71), and with fewer the time over the waves of a workgroup, while all workgroups are on the
        // chip at once (rule and measurements: scan_waves_plan).  Few channels of a long sequence are cut into segments of 64 steps
        // and more, which take a second launch, their state loads and a chain of end states: about 6.5 us, and 1.3 times the steps'
        // own cost in both launches (512 channels x 2048 steps 21.6 us, and 30.9 over the waves; 512 x 777 17.5 and 16.6, 1536 x
        // 4096 68 and 64).
        const int64_t wave_rows8 = (p.dim + 31) / 32 * 4;
        auto per_simd = [&](int64_t waves) { return (waves + simds - 1) / simds; };
        int64_t best = static_cast<int64_t>(p.seqlen) * step_cost(true, per_simd(wave_rows8 * p.batch));
        r.lanes = 8;
        TmPlan chosen = r;
        const ScanWavesPlan over_waves = scan_waves_plan(p, cus);
        if (p.segments == 0 && over_waves.ns < kScanWavesNever) {
            // one pass of eight lanes, in tiles of 32 steps, with one, two or three waves to a SIMD (within 5 % of it in 200 sizes of 16 ... 220
            // steps): the shorter one for a tile or less (2 x 31 x 3072 5.6 us and 7.2, 1 x 31 x 5120 6.2 and 7.5) and behind a tile's
            // beginning where the workgroups of the other are two or three to a CU (2 x 150 x 3072 13.4 and 14.4, 8 x 80 x 1536 12.7 and 14.4)
            static constexpr int kStart[3] = {3450, 4150, 4800}, kTile[3] = {1950, 2850, 4400};
            const int64_t w = std::min<int64_t>(per_simd(wave_rows8 * p.batch), 3) - 1;
            best = kStart[w] + static_cast<int64_t>((p.seqlen + 31) / 32) * kTile[w];
            if (over_waves.ns < best) {
                best = over_waves.ns;
                chosen.lanes = over_waves.lanes;
                chosen.waves = over_waves.waves;
            }
        }
        for (int n = 2; n <= 32 && 64 * n <= p.seqlen; ++n) {
            cut(n);
            const int64_t w = wave_rows8 * p.batch;
            const int64_t steps = r.segment_len * static_cast<int64_t>(step_cost(true, per_simd(w * r.segments)) + step_cost(false, per_simd(w * (r.segments - 1))));
            const int64_t cost = 6500 + steps * 13 / 10;
            if (r.segments > 1 && (p.segments == 0 ? cost < best : n == p.segments)) {
                best = cost;
                chosen = r;
            }
        }
        r = chosen;
    } else if (q >= 1 && rest > 0 && 2 * rest <= simds && p.dim % 64 == 0) {
        // between whole numbers of four-lane waves per SIMD the last channels go to the eight-lane kind
        const int64_t short_channels = rest * 16 / p.batch, blocks_a = (p.dim - short_channels) / 64;
        if (short_channels % 32 == 0 && (p.dim - short_channels) % 64 == 0 && blocks_a > 0 && blocks_a <= 0xfffff) {
            r.lanes = 0;
            r.blocks_a = static_cast<int>(blocks_a);
        }
    }
    return r;
}

int64_t segment_bytes(const QaSScanParams& p, const TmPlan& r) { return static_cast<int64_t>(p.batch) * (r.segments - 1) * p.dim * 17 * 4; }

template <bool HAS_Z, int DTK>
int launch(const QaSScanParams& p_in, const SscanDtProj& dtp, hipStream_t stream) {
    QaSScanParams p = p_in;
    TmPlan plan = plan_of(p);
    const int vec_out = p.out_d_stride == 1 && aligned16(p.out) && p.out_batch_stride % 8 == 0 && p.out_l_stride % 8 == 0;
    if (plan.segments > 1 && (!p.workspace || p.workspace_bytes < segment_bytes(p, plan))) {
        p.mapping = 0x40000000 | kScanWavesMapping << 20;       // one segment
        p.segments = 0;
        plan = plan_of(p);
    }
    p.segments = plan.segments;
    p.segment_len = plan.segments > 1 ? plan.segment_len : 0;
    if (static_cast<int64_t>(p.batch) * plan.segments > 65535) return QA_ERR_SHAPE;
    auto grid = [&](int channels, int entries) { return dim3((p.dim + channels - 1) / channels, static_cast<unsigned>(entries)); };
    if (plan.segments > 1) {
        const int entries = p.batch * (plan.segments - 1);
        p.dt_sum_out = static_cast<float*>(p.workspace);
        p.carry_dt_sum = p.dt_sum_out;
        p.carry_state = p.dt_sum_out + static_cast<int64_t>(entries) * p.dim;
        hipLaunchKernelGGL((scan_tm_kernel<8, false, false, DTK>), grid(32, entries), dim3(kThreads), 0, stream, p, dtp, vec_out);
    }
    if (plan.waves > 0) return sscan_waves_fwd(p, DTK != 0 ? &dtp : nullptr, plan.lanes, plan.waves, stream);
    const int entries = p.batch * plan.segments;
    switch (plan.lanes) {
        case 0:
            hipLaunchKernelGGL((scan_tm_mixed_kernel<HAS_Z, DTK>), dim3(plan.blocks_a + (p.dim - 64 * plan.blocks_a + 31) / 32, p.batch), dim3(kThreads), 0, stream, p, dtp, vec_out, plan.blocks_a);
            break;
        case 4: hipLaunchKernelGGL((scan_tm_kernel<4, HAS_Z, true, DTK>), grid(64, entries), dim3(kThreads), 0, stream, p, dtp, vec_out); break;
        case 8: hipLaunchKernelGGL((scan_tm_kernel<8, HAS_Z, true, DTK>), grid(32, entries), dim3(kThreads), 0, stream, p, dtp, vec_out); break;
        default: return QA_ERR_UNSUPPORTED;
    }
    return check_launch();
}

}  // namespace

int sscan_token_major_check(const QaSScanParams& p, const SscanDtProj* dt) {
    const auto mult4 = [](int64_t v) { return v % 4 == 0; };
    if (p.dstate != 16 || p.n_groups != 1 || p.dim < 4 || !mult4(p.dim) || p.carry_state || p.dt_sum_out || p.segments < 0) return QA_ERR_UNSUPPORTED;
    if (p.mapping != 0 && ((p.mapping & ~0x0fffffff) != 0x40000000 || (((p.mapping >> 20) & 0xff) == 0 && 64LL * (p.mapping & 0xfffff) > p.dim))) return QA_ERR_UNSUPPORTED;
    if (p.u_d_stride != 1 || (!dt && p.delta_d_stride != 1) || (p.z && p.z_d_stride != 1) || p.B_dstate_stride != 1 || p.C_dstate_stride != 1) return QA_ERR_STRIDE;
    if (!aligned4(p.u) || (!dt && !aligned4(p.delta)) || !aligned4(p.z) || !aligned4(p.B) || !aligned4(p.C)) return QA_ERR_STRIDE;
    for (const int64_t v : {p.u_batch_stride, p.u_l_stride, dt ? 0 : p.delta_batch_stride, dt ? 0 : p.delta_l_stride, p.z ? p.z_batch_stride : 0,
                            p.z ? p.z_l_stride : 0, p.B_batch_stride, p.B_l_stride, p.C_batch_stride, p.C_l_stride})
        if (!mult4(v) || v < 0) return QA_ERR_STRIDE;
    for (const int64_t v : {p.u_l_stride, dt ? dt->x_l_stride : p.delta_l_stride, p.z ? p.z_l_stride : 0, p.B_l_stride, p.C_l_stride})
        if (v >= 1 << 24) return QA_ERR_STRIDE;                        // a tile is addressed with 32-bit offsets
    if (!p.u || (!dt && !p.delta) || !p.A_log || !p.B || !p.C || !p.out) return QA_ERR_NULL;
    if (!p.scale_u || !p.scale_delta || !p.scale_A || !p.scale_B || !p.scale_C) return QA_ERR_NULL;
    if ((p.D && !p.scale_D) || (p.delta_bias && !p.scale_delta_bias) || (p.z && !p.scale_z) || (p.last_state_i8 && !p.scale_ssm_state)) return QA_ERR_NULL;
    if (!dt) return QA_OK;
    if (!dt->w || !dt->x || !dt->row_scale || !dt->col_scale) return QA_ERR_NULL;
    if (!p.z || dt->rank < 16 || dt->rank % 16 != 0 || dt->rank > kSscanDtRank) return QA_ERR_UNSUPPORTED;
    if (static_cast<int64_t>(p.seqlen) * dt->x_l_stride >= 1 << 30) return QA_ERR_UNSUPPORTED;       // 32-bit buffer offsets
    if (!aligned16(dt->w) || !aligned16(dt->x) || dt->x_l_stride % 16 != 0 || dt->x_batch_stride % 16 != 0) return QA_ERR_STRIDE;
    return QA_OK;
}

int sscan_token_major_fwd(const QaSScanParams& p, const SscanDtProj* dt, hipStream_t stream) {
    const int st = sscan_token_major_check(p, dt);
    if (st != QA_OK) return st;
    const SscanDtProj none = {};
    if (!dt) return p.z ? launch<true, 0>(p, none, stream) : launch<false, 0>(p, none, stream);
    if (dt->rank <= 64) return launch<true, 1>(p, *dt, stream);
    if (dt->rank <= 128) return launch<true, 2>(p, *dt, stream);
    return launch<true, 3>(p, *dt, stream);
}

int64_t sscan_token_major_workspace(const QaSScanParams& p) {
    const TmPlan plan = plan_of(p);
    return plan.segments > 1 ? segment_bytes(p, plan) : 0;
}

}  // namespace qa
