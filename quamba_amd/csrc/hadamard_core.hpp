// The Hadamard transform of one row in a workgroup's LDS: what the kernels that run it share (hadamard.hip, gemv.hip).
//
// The two fixed matrices are built here from their definitions instead of tables:
//   H_12: Paley's second construction for q = 5 (the symmetric conference matrix of order 6 with each
//         entry expanded to a 2x2 block);
//   H_40 = [[P, P], [P, -P]] with P the 20x20 Paley matrix for q = 19 (first row + - - ... -, first
//         column +, core delta(i,k) - chi(k - i)).
#pragma once
#include "qa_common.hpp"

#include <array>

namespace qa {

constexpr int legendre(int a, int q) {
    a %= q;
    if (a < 0) a += q;
    if (a == 0) return 0;
    for (int x = 1; x < q; ++x) {
        if ((x * x) % q == a) return 1;
    }
    return -1;
}

// sign bit masks, bit j of row i set = minus
constexpr std::array<uint64_t, 12> make_h12() {
    std::array<uint64_t, 12> rows{};
    for (int i = 0; i < 6; ++i) {
        for (int k = 0; k < 6; ++k) {
            const int c = (i == 0 || k == 0) ? (i == k ? 0 : 1) : legendre(k - i, 5);
            // 0 -> [[+,-],[-,-]], +1 -> [[+,+],[+,-]], -1 -> [[-,-],[-,+]]
            const int blk[2][2] = {{c == -1, c != 1}, {c != 1, c != -1}};
            for (int a = 0; a < 2; ++a) {
                for (int b = 0; b < 2; ++b) {
                    if (blk[a][b]) rows[2 * i + a] |= uint64_t(1) << (2 * k + b);
                }
            }
        }
    }
    return rows;
}

constexpr std::array<uint64_t, 40> make_h40() {
    std::array<uint64_t, 40> rows{};
    for (int i = 0; i < 40; ++i) {
        for (int k = 0; k < 40; ++k) {
            const int pi = i % 20, pk = k % 20;
            int s = 1;
            if (pi == 0) s = pk == 0 ? 1 : -1;
            else if (pk == 0) s = 1;
            else s = pi == pk ? 1 : -legendre(pk - pi, 19);
            if (i >= 20 && k >= 20) s = -s;
            if (s < 0) rows[i] |= uint64_t(1) << k;
        }
    }
    return rows;
}

constexpr auto kH12 = make_h12();
constexpr auto kH40 = make_h40();

// The rows in the order of their sign patterns, the first sign taken out: neighbours in it begin with the same signed sum, up to
// the sign of the whole, and a lane that makes a few neighbours adds up their common beginning once.
template <size_t S>
constexpr std::array<int, S> rows_by_pattern(const std::array<uint64_t, S>& rows) {
    auto pattern = [&](int i) {                                    // the first column in the highest bit
        uint64_t v = 0;
        for (size_t k = 0; k < S; ++k) v = v << 1 | (((rows[i] >> k) ^ rows[i]) & 1);
        return v;
    };
    std::array<int, S> order{};
    for (size_t i = 0; i < S; ++i) {
        size_t at = i;
        for (; at > 0 && pattern(order[at - 1]) > pattern(static_cast<int>(i)); --at) order[at] = order[at - 1];
        order[at] = static_cast<int>(i);
    }
    return order;
}
constexpr auto kOrder12 = rows_by_pattern(kH12);
constexpr auto kOrder40 = rows_by_pattern(kH40);

template <int S>
__device__ __forceinline__ bool minus_at(int i, int j) {
    if constexpr (S == 12) return (kH12[i] >> j) & 1;
    else return (kH40[i] >> j) & 1;
}

// one pad word per 32 keeps both the contiguous first pass and the strided later passes conflict free
__device__ __forceinline__ int phys(int e) { return e + (e >> 5); }

template <typename T>
__device__ __forceinline__ float load_as_float(const T* p) { return static_cast<float>(*p); }
template <>
__device__ __forceinline__ float load_as_float<__half>(const __half* p) { return __half2float(*p); }

// 2^B contiguous inputs starting at x + e0 (16-byte loads when `vec`)
template <int B, typename T>
__device__ __forceinline__ void load_run(const T* x, int e0, bool vec, float (&v)[1 << B]) {
    constexpr int R = 1 << B;
    constexpr int kPer16 = 16 / static_cast<int>(sizeof(T));
    if constexpr (R >= kPer16) {
        if (vec) {
#pragma unroll
            for (int q = 0; q < R / kPer16; ++q) {
                const uint4 raw = *reinterpret_cast<const uint4*>(x + e0 + q * kPer16);
                const T* t = reinterpret_cast<const T*>(&raw);
#pragma unroll
                for (int j = 0; j < kPer16; ++j) v[q * kPer16 + j] = load_as_float(t + j);
            }
            return;
        }
    }
#pragma unroll
    for (int j = 0; j < R; ++j) v[j] = load_as_float(x + e0 + j);
}

// Butterflies over index bits [bit0, bit0 + B): every lane takes groups of 2^B elements that differ in
// exactly those bits, lowest bit first.  The first pass (bit0 == 0) reads the input row x, later passes (and the first
// without x) LDS.
template <int B, int NT, typename T>
__device__ __forceinline__ void fwht_pass(float* buf, const T* x, int dim, int bit0, bool vec, int tid) {
    constexpr int R = 1 << B;
    const int groups = dim >> B;
    for (int g = tid; g < groups; g += NT) {
        const int lo = g & ((1 << bit0) - 1), hi = g >> bit0;
        const int base = ((hi << B) << bit0) | lo;
        float v[R];
        if (bit0 == 0 && x) {
            load_run<B, T>(x, base, vec, v);
        } else {
#pragma unroll
            for (int j = 0; j < R; ++j) v[j] = buf[phys(base + (j << bit0))];
        }
#pragma unroll
        for (int s = 0; s < B; ++s) {
#pragma unroll
            for (int j = 0; j < R; ++j) {
                if ((j & (1 << s)) == 0) {
                    const float a = v[j], c = v[j | (1 << s)];
                    v[j] = a + c;
                    v[j | (1 << s)] = a - c;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < R; ++j) buf[phys(base + (j << bit0))] = v[j];
    }
}

// The index bits of the row (2^log_m per column block) from `first` on, in passes of at most five bits, sizes as even as
// possible (7 -> 4+3, 13 -> 5+4+4).  Ends with a barrier.
template <int NT, typename T>
__device__ __forceinline__ void fwht_passes(float* buf, const T* x, int dim, int log_m, bool vec, int tid, int first = 0) {
    const int bits = log_m - first, n_pass = (bits + 4) / 5;
    for (int pass = 0, bit0 = first; pass < n_pass; ++pass) {
        const int b = bits / n_pass + (pass < bits % n_pass ? 1 : 0);
        switch (b) {
            case 1: fwht_pass<1, NT, T>(buf, x, dim, bit0, vec, tid); break;
            case 2: fwht_pass<2, NT, T>(buf, x, dim, bit0, vec, tid); break;
            case 3: fwht_pass<3, NT, T>(buf, x, dim, bit0, vec, tid); break;
            case 4: fwht_pass<4, NT, T>(buf, x, dim, bit0, vec, tid); break;
            default: fwht_pass<5, NT, T>(buf, x, dim, bit0, vec, tid); break;
        }
        bit0 += b;
        __syncthreads();
    }
}

// The S point transform of every column of the row in buf, quantised: PARTS lanes share the S outputs of a column, neighbours
// by pattern each (in four parts 283 additions a lane for S = 40, with neighbouring rows 373).
template <int S, int NT, int PARTS>
__device__ __forceinline__ void s_point_quantised(const float* buf, int8_t* out, int log_m, float scale, int tid) {
    constexpr int kPer = (S + PARTS - 1) / PARTS;
    const int M = 1 << log_m;
    for (int w = tid; w < M * PARTS; w += NT) {
        const int m = w & (M - 1), part = w >> log_m;
        float v[S];
#pragma unroll
        for (int c = 0; c < S; ++c) v[c] = buf[phys(c * M + m)];
        static_for<0, PARTS>([&](auto part_c) {
            constexpr int kPart = decltype(part_c)::value;
            if (part == kPart) {
#pragma unroll
                for (int o = kPart * kPer; o < (kPart + 1) * kPer && o < S; ++o) {
                    const int i = S == 12 ? kOrder12[o % 12] : kOrder40[o];
                    float acc = minus_at<S>(i, 0) ? -v[0] : v[0];
#pragma unroll
                    for (int j = 1; j < S; ++j) acc = minus_at<S>(i, j) ? acc - v[j] : acc + v[j];
                    out[i * M + m] = sat8_half_away(acc * scale);
                }
            }
        });
    }
}

// dim = S * 2^log_m with S = 12, 40 or 1 (in this order of preference); S = 0: no such form
struct HadamardShape {
    int s, log_m;
};
inline HadamardShape hadamard_shape(int dim) {
    int special = 1, rest = dim;
    if (rest % 12 == 0) { special = 12; rest /= 12; }
    else if (rest % 40 == 0) { special = 40; rest /= 40; }
    if (rest < 1 || (rest & (rest - 1)) != 0) return {0, 0};
    int log_m = 0;
    while ((1 << log_m) < rest) ++log_m;
    return {special, log_m};
}

}  // namespace qa
