// One decode step of a Mamba1 layer's recurrence with dt_proj in front of it: sixteen states per channel, one head, per-tensor
// scales, everything back to back.  Arithmetic as in ssm_update_body (sscan.hip; reference
// quamba/triton/selective_state_update.py:83-126), with the same expressions for the states; only the order of a row's output
// sum differs.
//
// A wave takes sixteen channels of up to four batch entries, on its own: no barrier.  Four lanes share a channel, four states
// each, so that the sixteen channels of an entry are one run in memory (1 KB in fp32).  What belongs to a (batch entry,
// channel) alone - step size, input, skip term, gate - is made once, by the lane of the four whose number the entry has, and
// broadcast from there; the decay rates are made once for all entries.
//
// The step sizes are a product of the entries' rows of x_proj's output with the weights of the wave's channels on the matrix
// cores.  Both come as whole runs of memory and turn into fragments by way of LDS (read from memory as fragments, sixteen rows
// side by side, they are slow work for a CU's memory path).
//
// Bound by the state (64 entries x 5120 channels in fp32: 42 MB, 8.4 us at the rate of a copy) and, in int8, by vector issue.
// Against the product (3.7) and the update (11.1) as two launches: 64 x 5120 fp32 12.2 us, 128 x 5120 int8 4.0 + 15.6 -> 16.7, 100 x
// 3072 int8 12.8 -> 10.1; against a dot product per lane, which ended at sixteen entries: 1 x 1536 4.7 -> 4.5, 16 x 5120 int8 8.0 ->
// 6.3.  A workgroup of 64 channels and sixteen entries with one barrier instead: 13.7 at 64 x 5120, 18.0 at 128 x 5120.
#include "gemm_core.hpp"
#include "mixer_common.hpp"
#include "sscan_common.hpp"

namespace qa {
namespace {

using gemm::v4i;
using gemm::v4u;
constexpr int kWaves = 4, kThreads = 64 * kWaves, kWaveCh = 16;

// dt_proj's operands, rows of 16 * pieces codes back to back
template <int NB>
struct StepSmem {
    __attribute__((aligned(16))) int8_t w[kWaveCh * 16 * kSsmDtPieces], x[NB * 16 * kSsmDtPieces];
};

// what the kernel takes of QaSsmUpdateParams and SsmDtProj (a launch's arguments are host time, see gemv.hpp)
struct StepArgs {
    void* state;
    __half* out;
    const int8_t *x, *z, *A_log, *B, *C, *D, *dt_bias, *w, *dt_x;
    const float *x_scale, *dt_scale, *dt_bias_scale, *A_log_scale, *state_scale, *B_scale, *C_scale, *D_scale, *z_scale, *row_scale, *col_scale;
    int64_t state_batch_stride;
    int batch, dim, A_dim_stride, x_batch_stride, z_batch_stride, B_batch_stride, C_batch_stride, out_batch_stride, dt_x_batch_stride, pieces;
    float alpha;
    uint8_t softplus, use_alpha, one_col_scale;
};

template <int NB, bool FP32>
__global__ __launch_bounds__(kThreads) void mamba1_step_kernel(StepArgs p) {
    static_assert(NB == 1 || NB == 2 || NB == 4, "entries per wave");
    __shared__ StepSmem<NB> smem[kWaves];
    __shared__ __attribute__((aligned(16))) float bc_all[kWaves][NB][2][16];
    __shared__ __attribute__((aligned(16))) int8_t codes_all[kWaves][NB][kWaveCh];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c0 = (blockIdx.x * kWaves + wave) * kWaveCh, b0 = blockIdx.y * NB;
    if (c0 >= p.dim) return;
    const int slice = lane & 3, c = c0 + (lane >> 2);      // (dim is whole waves of channels)
    auto entry = [&](int b) { return static_cast<int64_t>(min(b0 + b, p.batch - 1)); };       // past the last: that one again, and nothing is stored
    StepSmem<NB>& sm = smem[wave];
    float(*const bc)[2][16] = bc_all[wave];

    // The states first - of many sequences most of the bytes, of few what comes from furthest away, the weights having passed through
    // the caches since - then the projection's operands, behind which everything else is needed.  With the states last a layer's step is
    // longer: 32 x 3072 fp32 by 0.3 of 23.7 us, 64 x 4096 by 0.6 of 29.9; one to eight sequences in a chain of 24 layers, int8 by 0.1 to 1.0
    // of 13 to 30 us (1 x 5120 21.2 -> 21.3, 3 x 1536 16.9 -> 17.2, 8 x 3072 23.9 -> 24.4), fp32 by -0.1 to 0.25 (1 x 1536 12.9 -> 13.1, 5 x 3072 23.8 as
    // well).  Of one layer called again and again, whose states the caches hold, 5 and 8 sequences of 1536 and 2048 channels in fp32 are 0.0 to
    // 0.2 of 16.2 us shorter that way.
    const int64_t at = static_cast<int64_t>(c) * 16 + 4 * slice;
    float4 st32[FP32 ? NB : 1];
    uint32_t st8[FP32 ? 1 : NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int64_t e = entry(b) * p.state_batch_stride + at;
        if constexpr (FP32) st32[b] = *reinterpret_cast<const float4*>(static_cast<const float*>(p.state) + e);
        else st8[b] = *reinterpret_cast<const uint32_t*>(static_cast<const int8_t*>(p.state) + e);
    }
    v4u rw[3], rx;
    const v4u* w = reinterpret_cast<const v4u*>(p.w + static_cast<int64_t>(c0) * (16 * p.pieces));
#pragma unroll
    for (int i = 0; i < 3; ++i) rw[i] = w[min(i * 64 + lane, kWaveCh * p.pieces - 1)];
    rx = *reinterpret_cast<const v4u*>(p.dt_x + entry(min(lane >> 4, NB - 1)) * p.dt_x_batch_stride + 16 * min(lane & 15, p.pieces - 1));
    // B | C: word lane % 8 of an entry's sixteen B and sixteen C codes
    const int bc_b = lane >> 3, bc_w = lane & 7;
    uint32_t bc_codes = 0;
    if (bc_b < NB) bc_codes = *reinterpret_cast<const uint32_t*>(bc_w < 4 ? p.B + entry(bc_b) * p.B_batch_stride + 4 * bc_w : p.C + entry(bc_b) * p.C_batch_stride + 4 * (bc_w - 4));
    // this lane's item: entry `slice`
    const int8_t* const standin = p.x + c;                 // (read where an optional operand is missing)
    const int64_t mine = entry(min(slice, NB - 1));
    const int8_t x_q = p.x[mine * p.x_batch_stride + c], z_q = *(p.z ? p.z + mine * p.z_batch_stride + c : standin);
    const int8_t D_q = *(p.D ? p.D + c : standin), bias_q = *(p.dt_bias ? p.dt_bias + c : standin);
    const uint32_t A_codes = *reinterpret_cast<const uint32_t*>(p.A_log + static_cast<int64_t>(c) * p.A_dim_stride + 4 * slice);
    const float dt_row = p.use_alpha ? p.alpha : *p.row_scale;
    const float dt_col = p.use_alpha ? 1.0f : p.col_scale[p.one_col_scale ? 0 : c0 + (lane & 15)];
    const float x_scale = *p.x_scale, dt_scale = *p.dt_scale, A_scale = *p.A_log_scale, B_scale = *p.B_scale, C_scale = *p.C_scale;
    const float bias_scale = p.dt_bias ? *p.dt_bias_scale : 0.0f, D_scale = p.D ? *p.D_scale : 0.0f, z_scale = p.z ? *p.z_scale : 0.0f;
    const float s_state = FP32 ? 0.0f : *p.state_scale;
    __builtin_amdgcn_sched_barrier(0);

    // (a wave writes and reads only its own part of LDS, where its operations complete in order)
    const int pieces = p.pieces;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int t = i * 64 + lane;
        if (t < kWaveCh * pieces) *reinterpret_cast<v4u*>(&sm.w[16 * t]) = rw[i];
    }
    if ((lane & 15) < pieces && (lane >> 4) < NB) *reinterpret_cast<v4u*>(&sm.x[16 * ((lane >> 4) * pieces + (lane & 15))]) = rx;
    gemm::wave_lds_sync();
    const int j = lane & 15, g = lane >> 4;
    v4i dots = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        v4i fw = {0, 0, 0, 0}, fx = {0, 0, 0, 0};
        if (4 * k + g < pieces) {
            fw = *reinterpret_cast<const v4i*>(&sm.w[16 * (j * pieces + 4 * k + g)]);
            fx = *reinterpret_cast<const v4i*>(&sm.x[16 * ((j & (NB - 1)) * pieces + 4 * k + g)]);
        }
        dots = __builtin_amdgcn_mfma_i32_16x16x64_i8(fx, fw, dots, 0, 0, 0);
    }
    // lane l: channel l % 16, entries 4 (l / 16) + 0 .. 3
    if (g == 0) {
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            float v = dt_col * static_cast<float>(dots[e]);
            asm volatile("" : "+v"(v));                // two products, each rounded (with alpha the first is by one)
            codes_all[wave][e][j] = sat8_rne(dt_row * v);
        }
    }
    if (bc_b < NB) {
        const float s = bc_w < 4 ? B_scale : C_scale;
        *reinterpret_cast<float4*>(&bc[bc_b][bc_w >> 2][4 * (bc_w & 3)]) =
            make_float4(s * code_byte_to_float(bc_codes, 0), s * code_byte_to_float(bc_codes, 1), s * code_byte_to_float(bc_codes, 2), s * code_byte_to_float(bc_codes, 3));
    }
    gemm::wave_lds_sync();
    const int8_t dt_q = codes_all[wave][min(slice, NB - 1)][lane >> 2];
    const float my_x = x_scale * static_cast<float>(x_q);
    float my_dt = dt_scale * static_cast<float>(dt_q), gate = 1.0f;
    my_dt += p.dt_bias ? bias_scale * static_cast<float>(bias_q) : 0.0f;
    if (p.softplus) my_dt = softplus20_flat(my_dt);
    if (p.z) {
        const float zv = z_scale * static_cast<float>(z_q);
        gate = zv * (1.0f / (1.0f + expf(-zv)));
    }
    float A[4], inv[4], sc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        A[e] = -__expf(A_scale * code_byte_to_float(A_codes, e));
        sc[e] = s_state;
        inv[e] = FP32 ? 0.0f : __builtin_amdgcn_rcpf(s_state * 1e2f);
    }

    float acc[4] = {};
    static_for<0, NB>([&](auto b_c) {
        constexpr int b = decltype(b_c)::value;
        const float dt = quad_bcast<4, b>(my_dt), xv = quad_bcast<4, b>(my_x);
        const float4 Bv = *reinterpret_cast<const float4*>(&bc[b][0][4 * slice]), Cv = *reinterpret_cast<const float4*>(&bc[b][1][4 * slice]);
        const float B[4] = {Bv.x, Bv.y, Bv.z, Bv.w}, C[4] = {Cv.x, Cv.y, Cv.z, Cv.w};
        float h[4];
        if constexpr (FP32) { h[0] = st32[b].x; h[1] = st32[b].y; h[2] = st32[b].z; h[3] = st32[b].w; }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (!FP32) h[e] = s_state * code_byte_to_float(st8[b], e);
            h[e] = h[e] * __expf(A[e] * dt) + (B[e] * dt) * xv;
            acc[b] += h[e] * C[e];
        }
        if (b0 + b < p.batch) {
            const int64_t e = (b0 + b) * p.state_batch_stride + at;
            if constexpr (FP32) *reinterpret_cast<float4*>(static_cast<float*>(p.state) + e) = make_float4(h[0], h[1], h[2], h[3]);
            else *reinterpret_cast<uint32_t*>(static_cast<int8_t*>(p.state) + e) = requantise4(h, sc, inv, 1e2f);
        }
    });
    // each lane of a quad completes the entry it owns
    const bool odd = slice & 1, hi = slice & 2;
    const float w01 = (odd ? acc[1] : acc[0]) + quad_xor<1>(odd ? acc[0] : acc[1]);
    const float w23 = (odd ? acc[3] : acc[2]) + quad_xor<1>(odd ? acc[2] : acc[3]);
    const float sum = (hi ? w23 : w01) + quad_xor<2>(hi ? w01 : w23);
    const float y = (sum + my_x * (D_scale * static_cast<float>(D_q))) * gate;
    if (slice < NB && b0 + slice < p.batch) p.out[static_cast<int64_t>(b0 + slice) * p.out_batch_stride + c] = __float2half(y);
}

template <bool FP32>
int launch(const StepArgs& a, hipStream_t stream) {
    const int64_t blocks = (a.dim / kWaveCh + kWaves - 1) / kWaves;
    auto go = [&](auto kernel, int nb) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks), static_cast<unsigned>((a.batch + nb - 1) / nb)), dim3(kThreads), 0, stream, a);
        return check_launch();
    };
    if (a.batch == 1) return go(mamba1_step_kernel<1, FP32>, 1);
    if (a.batch == 2) return go(mamba1_step_kernel<2, FP32>, 2);
    return go(mamba1_step_kernel<4, FP32>, 4);
}

}  // namespace

int mamba1_step(const QaSsmUpdateParams& p, const SsmDtProj& dt, hipStream_t stream) {
    const auto mult4 = [](int64_t v) { return v % 4 == 0; };
    if (p.dstate != 16 || p.nheads != 1 || p.ngroups != 1 || p.nhead_groups != 0 || p.dim % kWaveCh != 0 || p.batch > 65535) return QA_ERR_UNSUPPORTED;
    if (p.state_dstate_stride != 1 || p.state_dim_stride != 16 || !mult4(p.state_batch_stride) || !(p.state_is_fp32 ? aligned16(p.state) : aligned4(p.state))) return QA_ERR_UNSUPPORTED;
    if (p.A_dstate_stride != 1 || !mult4(p.A_dim_stride) || !aligned4(p.A_log) || p.out_dim_stride != 1 || p.x_dim_stride != 1 || (p.z && p.z_dim_stride != 1)) return QA_ERR_UNSUPPORTED;
    if (p.B_dstate_stride != 1 || p.C_dstate_stride != 1 || !mult4(p.B_batch_stride) || !mult4(p.C_batch_stride) || !aligned4(p.B) || !aligned4(p.C)) return QA_ERR_UNSUPPORTED;
    if ((p.D && p.D_dim_stride != 1) || (p.dt_bias && (p.dt_bias_is_fp16 || p.dt_bias_dim_stride != 1))) return QA_ERR_UNSUPPORTED;
    if (dt.pieces < 1 || dt.pieces > kSsmDtPieces || !aligned16(dt.w) || !aligned16(dt.x) || dt.x_batch_stride % 16 != 0) return QA_ERR_UNSUPPORTED;
    for (const int64_t v : {p.A_dim_stride, p.x_batch_stride, p.z ? p.z_batch_stride : 0, p.B_batch_stride, p.C_batch_stride, p.out_batch_stride, dt.x_batch_stride})
        if (v < 0 || v > 0x7fffffff) return QA_ERR_UNSUPPORTED;
    StepArgs a = {};
    a.state = p.state; a.out = static_cast<__half*>(p.out);
    a.x = p.x; a.z = p.z; a.A_log = p.A_log; a.B = p.B; a.C = p.C; a.D = p.D; a.dt_bias = static_cast<const int8_t*>(p.dt_bias); a.w = dt.w; a.dt_x = dt.x;
    a.x_scale = p.x_scale; a.dt_scale = p.dt_scale; a.dt_bias_scale = p.dt_bias_scale; a.A_log_scale = p.A_log_scale; a.state_scale = p.state_scale;
    a.B_scale = p.B_scale; a.C_scale = p.C_scale; a.D_scale = p.D_scale; a.z_scale = p.z_scale; a.row_scale = dt.row_scale; a.col_scale = dt.col_scale;
    a.state_batch_stride = p.state_batch_stride;
    a.batch = p.batch; a.dim = p.dim; a.A_dim_stride = static_cast<int>(p.A_dim_stride);
    a.x_batch_stride = static_cast<int>(p.x_batch_stride); a.z_batch_stride = static_cast<int>(p.z_batch_stride);
    a.B_batch_stride = static_cast<int>(p.B_batch_stride); a.C_batch_stride = static_cast<int>(p.C_batch_stride);
    a.out_batch_stride = static_cast<int>(p.out_batch_stride); a.dt_x_batch_stride = static_cast<int>(dt.x_batch_stride);
    a.pieces = dt.pieces; a.alpha = dt.alpha;
    a.softplus = p.dt_softplus != 0; a.use_alpha = dt.use_alpha != 0; a.one_col_scale = dt.col_numel == 1;
    return p.state_is_fp32 ? launch<true>(a, stream) : launch<false>(a, stream);
}

}  // namespace qa
