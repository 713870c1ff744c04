// Pieces shared by the selective-scan kernels (sscan.hip, sscan_tm.hip): the transcendental functions as they evaluate
// them, byte conversions, cross-lane moves.
#pragma once
#include "gemm_core.hpp"
#include "qa_common.hpp"

namespace qa {

constexpr float kLog2e = 1.44269504088896341f;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// float(int8 code in byte n of w) in one instruction (the sub-dword operand select converts the byte in place; the
// compiler, left to itself, shifts and sign-extends the byte out first)
__device__ __forceinline__ float code_byte_to_float(uint32_t w, int n) {
    float r;
    switch (n) {
        case 0: asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(r) : "v"(w)); break;
        case 1: asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(r) : "v"(w)); break;
        case 2: asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(r) : "v"(w)); break;
        default: asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(r) : "v"(w)); break;
    }
    return r;
}

// softplus with the reference's threshold; log1p evaluated so that small exp(x) keeps full
// relative accuracy (series below 2^-6, log2 above).
__device__ __forceinline__ float softplus20(float x) {
    if (x > 20.0f) return x;
    const float e = fast_exp2(x * kLog2e);
    const float series = e * __builtin_fmaf(e, __builtin_fmaf(e, __builtin_fmaf(e, -0.25f, 1.0f / 3.0f), -0.5f), 1.0f);
    const float big = fast_log2(1.0f + e) * 0.693147180559945309f;
    return e < 0.015625f ? series : big;
}

// The same function without a branch and with one rounding compensated instead of a series:
//   softplus(x) = max(x, 0) + log1p(e),  e = exp(-|x|) in (0, 1]
//   u = fl(1 + e) = 1 + e + r with r = (u - 1) - e exact, so log1p(e) = ln(u - r) = ln u - r / u + ..., and with
//   u in [1, 2] taking r for r / u is wrong by less than 2^-24 of the result.
// Above the threshold the second term is below half an ulp of x, so x comes back exactly, as the reference returns it.
__device__ __forceinline__ float softplus20_flat(float x) {
    const float e = fast_exp2(__builtin_fabsf(x) * -kLog2e);
    const float u = 1.0f + e;
    const float r = (u - 1.0f) - e;
    const float sp = __builtin_fmaf(fast_log2(u), 0.693147180559945309f, -r);
    float pos;                                        // max(x, 0): written out, because the builtins put a second
    asm("v_max_f32 %0, 0, %1" : "=v"(pos) : "v"(x));  // maximum of x with itself in front of it (quieting of NaNs)
    return pos + sp;
}

__device__ __forceinline__ float silu_gate(float z) {
    return z * fast_rcp(1.0f + fast_exp2(-z * kLog2e));
}

// Value of `v` in the lane of this quad that holds slice SRC of the same channel (NSPLIT lanes per
// channel, NSPLIT in {1,2,4}), as a DPP quad permutation that the compiler folds into the consumer.
template <int NSPLIT, int SRC>
__device__ __forceinline__ float quad_bcast(float v) {
    if (NSPLIT == 1) return v;
    constexpr int ctrl = NSPLIT == 4 ? (SRC | (SRC << 2) | (SRC << 4) | (SRC << 6))
                                     : (SRC | (SRC << 2) | ((2 + SRC) << 4) | ((2 + SRC) << 6));
    const int r = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xf, 0xf, false);
    return __builtin_bit_cast(float, r);
}
// Same with a source slice that is a constant only after loop unrolling.
template <int NSPLIT>
__device__ __forceinline__ float quad_bcast_sel(float v, int src) {
    switch (src) {
        case 0: return quad_bcast<NSPLIT, 0>(v);
        case 1: return quad_bcast<NSPLIT, 1>(v);
        case 2: return quad_bcast<NSPLIT, (NSPLIT > 2 ? 2 : 0)>(v);
        default: return quad_bcast<NSPLIT, (NSPLIT > 2 ? 3 : 1)>(v);
    }
}
// Value of `v` in lane (lane ^ M) of the quad, M in {1,2}.
template <int M>
__device__ __forceinline__ float quad_xor(float v) {
    constexpr int ctrl = M == 1 ? (1 | (0 << 2) | (3 << 4) | (2 << 6)) : (2 | (3 << 2) | (0 << 4) | (1 << 6));
    const int r = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xf, 0xf, false);
    return __builtin_bit_cast(float, r);
}

// Value of `v` in the lane UP above, inside a row of sixteen lanes (zero past its end).
template <int UP>
__device__ __forceinline__ float row_from_up(float v) {
    const int r = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x100 + UP, 0xf, 0xf, true);     // row_shl
    return __builtin_bit_cast(float, r);
}

__device__ __forceinline__ float i8_of(uint32_t word, int j) {
    return static_cast<float>(static_cast<int8_t>((word >> (8 * j)) & 0xffu));
}

// sat8_rne(fl(h k) / fl(s k)) of four states, packed.  The IEEE quotient is twelve instructions a state and was most of a
// lane's arithmetic; a product with the reciprocal is within 2^-21 of it, so the integers agree unless the product lies within
// 1e-4 of a rounding tie (values up to 128; beyond, both saturate), and only a wave that holds such a state divides.
// (inv: rcp of fl(s k))
__device__ __forceinline__ uint32_t requantise4(const float (&h)[4], const float (&s)[4], const float (&inv)[4], float k) {
    float t[4], num[4];
    bool tie = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        num[e] = h[e] * k;
        t[e] = num[e] * inv[e];
        tie |= !(__builtin_fabsf(t[e] - __builtin_rintf(t[e])) < 0.4999f);         // (NaN and infinities divide)
    }
    if (__builtin_amdgcn_ballot_w64(tie)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) t[e] = num[e] / (s[e] * k);
    }
    return gemm::pack4_rne_sat8(t[0], t[1], t[2], t[3]);
}

}  // namespace qa
