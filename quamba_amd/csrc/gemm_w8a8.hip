// W8A8 GEMM on the int8 matrix cores with a fused scale epilogue.
//
//   acc[m,n] = sum_k a[m,k] * w[n,k]            (int32, exact)
//   d[m,n]   = cast( s_a[m|0] * ( s_w[n|0] * float(acc) ) )     cast: fp16 RN, or int8 saturating with
//                                                               round-half-even (or half-away for the GEMV rule)
// Reference arithmetic: csrc/linear/quant_linear_fwd_kernel.cuh:63-130 (epilogue :85-109),
// csrc/linear/quant_linear_fwd_gemv_kernel.cuh:56-60 (roundf variant).
// The tiling, LDS layout and epilogue are in gemm_core.hpp.
#include "gemm_core.hpp"
#include "gemv.hpp"

// Built with -DQA_GEMM_CLK (bench.py --gemm-phase-clocks, never the product library) thread 0 of every workgroup of
// the tiled kernel records the shader clock and the constant 100 MHz clock at four points - start, first fragments
// in registers, end of the main loop, end of the epilogue - and qa_gemm_clk_read copies the table out.
#ifdef QA_GEMM_CLK
__device__ unsigned long long g_gemm_clk[8192][8];
extern "C" int qa_gemm_clk_read(void* dst, int64_t bytes) {     // copies the table out and clears it
    if (bytes != static_cast<int64_t>(sizeof(g_gemm_clk))) return QA_ERR_SHAPE;
    void* table = nullptr;
    if (hipMemcpyFromSymbol(dst, HIP_SYMBOL(g_gemm_clk), sizeof(g_gemm_clk)) != hipSuccess) return QA_ERR_LAUNCH;
    if (hipGetSymbolAddress(&table, HIP_SYMBOL(g_gemm_clk)) != hipSuccess) return QA_ERR_LAUNCH;
    return hipMemset(table, 0, sizeof(g_gemm_clk)) == hipSuccess ? QA_OK : QA_ERR_LAUNCH;
}
#define CLK_MARK(i)                                                 \
    do {                                                            \
        if (threadIdx.x == 0 && blockIdx.x < 8192) {                \
            g_gemm_clk[blockIdx.x][2 * (i)] = clock64();            \
            g_gemm_clk[blockIdx.x][2 * (i) + 1] = wall_clock64();   \
        }                                                           \
    } while (0)
#else
#define CLK_MARK(i)
#endif

namespace qa {
namespace {

using namespace gemm;

template <int TM, int TN, int WGM, int WGN, int STAGES, int OUT, bool FLEX, bool COL_OUTER>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_w8a8_kernel(QaGemmW8A8Params p) {
    using C = Cfg<TM, TN, WGM, WGN, STAGES>;
    constexpr int BM = C::kBM, BN = C::kBN, WAVES = C::kWaves;
    static_assert(epilogue_lds_bytes<TM, TN, WAVES>() <= C::kLdsBytes, "epilogue staging does not fit");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WGM, wn = wave / WGM;
    const int tiles_m = (p.m + BM - 1) / BM, tiles_n = (p.n + BN - 1) / BN;
    int tile_m, tile_n;
    tile_of_workgroup<BM, BN>(blockIdx.x, tiles_m, tiles_n, tile_m, tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN;

    const v4i rsrc_a = make_rsrc(p.a, static_cast<int>((static_cast<int64_t>(p.m) - 1) * p.lda + p.k));
    const v4i rsrc_w = make_rsrc(p.w, static_cast<int>((static_cast<int64_t>(p.n) - 1) * p.ldw + p.k));
    const uint32_t lds_base = lds_offset_of(lds);

    using Scales = TileScales<BM, BN, WAVES>;
    if (!p.use_alpha) Scales::request(lds_base + C::kLdsBytes, p.a_scale, p.a_scale_numel, p.m, m0, p.w_scale, p.w_scale_numel, p.n, n0, wave, lane);
    TileLoader<C::kAInstr> load_a;
    TileLoader<C::kWInstr> load_w;
    load_a.template init<WAVES>(m0, p.m, p.lda, wave, lane);
    load_w.template init<WAVES>(n0, p.n, p.ldw, wave, lane);

    const int k_tiles = (p.k + kBK - 1) / kBK;
    Epilogue e;
    e.use_alpha = p.use_alpha; e.alpha = p.alpha; e.round_mode = p.round_mode; e.col_outer = p.scale_order;
    e.ldd = p.ldd; e.d = p.d;
    auto finish = [&](auto& acc) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        __syncthreads();
        CLK_MARK(2);
        epilogue<TM, TN, OUT, FLEX, false, COL_OUTER>(e, acc, lds, p.m, p.n, m0 + wm * TM * 32, n0 + wn * TN * 32, wave, lane,
                                                      reinterpret_cast<const float*>(lds + C::kLdsBytes), BN + wm * TM * 32, wn * TN * 32);
        CLK_MARK(3);
    };
    CLK_MARK(0);
    if constexpr (TM * TN > 1) {
        // The requests for a tile go out one at a time, one per kPace multiplications counted from the barrier (RotatedMma): those
        // that fit behind it, whose stage it has just freed, for tile t + STAGES, the rest during the next tile.  Past the
        // end of K every lane is out of range and stores zeros.
        // (Workgroups that go from one output tile to the next without a pause, the next one's first k tile requested
        // during the last ones of this one, gained nothing: the clock falls by what the matrix cores are busier.)
        // 128 x 256 tiles, three stages, against 32x32x32 with block fetches (us): 3063 x 2560 x 5120 42.8 -> 40.8, 3063 x
        // 1536 x 3072 20.6 -> 18.6, 16384 x 1536 x 3072 77.6 -> 68.2.
        using Mma = RotatedMma<TM, TN>;
        constexpr int kReq = C::kAInstr + C::kWInstr, kPace = kReq <= Mma::kPerTile / 4 ? 4 : Mma::kPerTile / kReq;
        constexpr int kEarly = Mma::kBehindBarrier / kPace < kReq ? Mma::kBehindBarrier / kPace : kReq;
        auto request = [&](int r, int tile, uint32_t stage) {
            if (r < C::kAInstr) load_a.template issue_one<WAVES>(r, rsrc_a, tile * kBK, p.k, lds_base + stage, wave);
            else if (r < kReq) load_w.template issue_one<WAVES>(r - C::kAInstr, rsrc_w, tile * kBK, p.k, lds_base + stage + BM * kBK, wave);
        };
        auto request_whole = [&](int r, int tile, uint32_t stage) {
            if (r < C::kAInstr) load_a.template issue_whole<WAVES>(r, rsrc_a, tile * kBK, lds_base + stage, wave);
            else if (r < kReq) load_w.template issue_whole<WAVES>(r - C::kAInstr, rsrc_w, tile * kBK, lds_base + stage + BM * kBK, wave);
        };
#pragma unroll
        for (int t = 0; t < STAGES - 1; ++t)
#pragma unroll
            for (int r = 0; r < kReq; ++r) request(r, t, t * C::kStageBytes);
#pragma unroll
        for (int r = 0; r < kEarly; ++r) request(r, STAGES - 1, (STAGES - 1) * C::kStageBytes);
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((STAGES - 2) * kReq + kEarly));
        __syncthreads();
        const uint8_t* my_a = lds + (wm * TM * 32) * kBK;
        const uint8_t* my_w = lds + BM * kBK + (wn * TN * 32) * kBK;
        Mma mma;
        mma.init(lane);
        mma.start(my_a, my_w);
        CLK_MARK(1);
        uint32_t cur = 0, late = (STAGES - 1) * C::kStageBytes;        // stages of this tile and of the tile STAGES - 1 further
        auto multiply = [&](int kt, auto&& req) {
            const uint32_t nxt = cur + C::kStageBytes == C::kLdsBytes ? 0 : cur + C::kStageBytes;
            mma.template tile<(STAGES - 2) * kReq>(my_a + cur, my_w + cur, my_a + nxt, my_w + nxt, [&](int idx) {
                if (idx % kPace != kPace - 1) return;
                const int r = idx / kPace;
                if (r < kEarly) req(r, kt + STAGES, cur);
                else req(r, kt + STAGES - 1, late);
            });
            late = cur;
            cur = nxt;
        };
        int kt = 0;
        for (const int whole = p.k / kBK - STAGES; kt < whole; ++kt) multiply(kt, request_whole);
        for (; kt < k_tiles; ++kt) multiply(kt, request);
        finish(mma.acc);
    } else {
    const int frow = lane & 31, fhalf = lane >> 5;
    v16i acc[1][1];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][0][r] = 0;
    auto issue = [&](int tile) {
        const uint32_t base = lds_base + (tile % STAGES) * C::kStageBytes;
        load_a.template issue<WAVES>(rsrc_a, tile * kBK, p.k, base, wave);
        load_w.template issue<WAVES>(rsrc_w, tile * kBK, p.k, base + BM * kBK, wave);
    };
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s) issue(s);

    for (int kt = 0; kt < k_tiles; ++kt) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((STAGES - 2) * (C::kAInstr + C::kWInstr)));
        __syncthreads();
        const uint8_t* stage = lds + (kt % STAGES) * C::kStageBytes;
        // the requests for the next tile go out one at a time between the multiplications of this one
        // (past the end of K every lane is out of range and stores zeros)
        const int nt = kt + STAGES - 1;
        const uint32_t nbase = lds_base + (nt % STAGES) * C::kStageBytes;
        static_assert(C::kAInstr + C::kWInstr <= 4, "a request behind each of four multiplications");
        mma_tile_paced(stage + wm * 32 * kBK, stage + BM * kBK + wn * 32 * kBK, frow, fhalf, acc[0][0], [&](int r) {
            if (r < C::kAInstr) load_a.template issue_one<WAVES>(r, rsrc_a, nt * kBK, p.k, nbase, wave);
            else if (r < C::kAInstr + C::kWInstr) load_w.template issue_one<WAVES>(r - C::kAInstr, rsrc_w, nt * kBK, p.k, nbase + BM * kBK, wave);
        });
    }
    finish(acc);
    }
}

template <int TM, int TN, int WGM, int WGN, int STAGES, int OUT, bool FLEX, bool COL_OUTER = false>
int launch_one(const QaGemmW8A8Params& p, hipStream_t stream) {
    using C = Cfg<TM, TN, WGM, WGN, STAGES>;
    if constexpr (!FLEX && !COL_OUTER) {
        if (p.scale_order == 1) return launch_one<TM, TN, WGM, WGN, STAGES, OUT, FLEX, true>(p, stream);
    }
    const int64_t tiles = static_cast<int64_t>((p.m + C::kBM - 1) / C::kBM) * ((p.n + C::kBN - 1) / C::kBN);
    if (tiles > 0x7fffffffLL) return QA_ERR_SHAPE;
    auto kernel = gemm_w8a8_kernel<TM, TN, WGM, WGN, STAGES, OUT, FLEX, COL_OUTER>;
    constexpr int kLds = C::kLdsBytes + TileScales<C::kBM, C::kBN, C::kWaves>::kBytes;
    if (kLds > 65536) {
        // allowing more than 64 KiB of dynamic LDS is a per-function attribute; setting it is idempotent
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                kLds) != hipSuccess) {
            return check_launch();
        }
    }
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(tiles)), dim3(C::kThreads), kLds, stream, p);
    return check_launch();
}

template <int TM, int TN, int WGM, int WGN, int STAGES, bool FLEX>
int launch_gemm(const QaGemmW8A8Params& p, hipStream_t stream) {
    if (p.out_type == QA_OUT_I8) return launch_one<TM, TN, WGM, WGN, STAGES, QA_OUT_I8, FLEX>(p, stream);
    if (p.out_type == QA_OUT_BF16) return launch_one<TM, TN, WGM, WGN, STAGES, QA_OUT_BF16, FLEX>(p, stream);
    return launch_one<TM, TN, WGM, WGN, STAGES, QA_OUT_F16, FLEX>(p, stream);
}

// ---------------------------------------------------------------------------------------------
// Few activation rows (M <= 64, the decode step): the product is a stream over the weight matrix
// and HBM-bound, so the shape of the launch is chosen for memory parallelism rather than reuse.
// A workgroup owns 32 output columns and all rows; its WAVES waves split K between them in
// interleaved 128-byte tiles.  A wave fetches its tiles with eight lanes per 128-byte row piece
// (whole cache lines; fetching MFMA fragments directly would touch 64 lines per instruction),
// DEPTH tiles in flight in registers, and turns a tile into fragments through a staging area in
// LDS that is private to the wave, so the main loop has no workgroup barrier.  The small
// activation matrix takes the same route and is served by the caches.  The partial sums of the
// waves are added in LDS (integers: the order does not matter), then every thread scales and
// writes four consecutive columns of one row.
// ---------------------------------------------------------------------------------------------
template <int TM, int WAVES, int DEPTH, int OUT, bool FLEX>
__global__ __launch_bounds__(64 * WAVES) void gemm_w8a8_skinny_kernel(QaGemmW8A8Params p) {
    constexpr int kThreads = 64 * WAVES;
    constexpr int kOob = 0x7ffffff0;                       // beyond any buffer: the load returns zeros
    constexpr int kTile = 32 * kBK;                        // one staged 32-row tile
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    int* red = reinterpret_cast<int*>(lds + WAVES * (1 + TM) * kTile);   // [row block][acc register][lane]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int frow = lane & 31, fhalf = lane >> 5;
    int m0, n0;
    skinny_tile_of_workgroup<TM>(blockIdx.x, p.m, p.n, m0, n0);
    for (int i = tid; i < TM * 16 * 64; i += kThreads) red[i] = 0;

    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(p.w), 0, static_cast<int>((static_cast<int64_t>(p.n) - 1) * p.ldw + p.k), kRsrcFlags);
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(p.a), 0, static_cast<int>((static_cast<int64_t>(p.m) - 1) * p.lda + p.k), kRsrcFlags);
    // fetch mapping: instruction i, lane l -> tile row 8i + l/8, 16-byte chunk l%8
    const int lrow = lane >> 3, lchunk = lane & 7;
    int w_off[4], a_off[TM][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = n0 + 8 * i + lrow;
        w_off[i] = row < p.n ? static_cast<int>(row * p.ldw) + lchunk * 16 : -1;
#pragma unroll
        for (int j = 0; j < TM; ++j) {
            const int arow = m0 + j * 32 + 8 * i + lrow;
            a_off[j][i] = arow < p.m ? static_cast<int>(arow * p.lda) + lchunk * 16 : -1;
        }
    }

    const int k_tiles = (p.k + kBK - 1) / kBK;
    const int my_tiles = (k_tiles - wave + WAVES - 1) / WAVES;      // tiles wave, wave + WAVES, ...
    v4u fw[DEPTH][4], fa[DEPTH][TM][4];
    auto load = [&](int i_tile, auto buf_c) {
        constexpr int buf = decltype(buf_c)::value;
        const int k0 = (wave + i_tile * WAVES) * kBK;
        const bool k_ok = k0 + lchunk * 16 < p.k;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            fw[buf][i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, (k_ok && w_off[i] >= 0) ? w_off[i] + k0 : kOob, 0, 0);
#pragma unroll
            for (int j = 0; j < TM; ++j) {
                fa[buf][j][i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, (k_ok && a_off[j][i] >= 0) ? a_off[j][i] + k0 : kOob, 0, 0);
            }
        }
    };

    v16i acc[TM];
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0;

    uint8_t* stage = lds + wave * ((1 + TM) * kTile);
    static_for<0, DEPTH - 1>([&](auto s) { load(decltype(s)::value, s); });
    for (int base = 0; base < my_tiles; base += DEPTH) {
        static_for<0, DEPTH>([&](auto s_c) {
            constexpr int s = decltype(s_c)::value;
            // tiles past this wave's share are outside K: their loads touch no memory
            load(base + s + DEPTH - 1, std::integral_constant<int, (s + DEPTH - 1) % DEPTH>{});
            if (base + s < my_tiles) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = 8 * i + lrow;
                    *reinterpret_cast<v4u*>(stage + row * kBK + swz(row, lchunk) * 16) = fw[s][i];
#pragma unroll
                    for (int j = 0; j < TM; ++j)
                        *reinterpret_cast<v4u*>(stage + (1 + j) * kTile + row * kBK + swz(row, lchunk) * 16) = fa[s][j][i];
                }
                wave_lds_sync();
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {
                    const int off = frow * kBK + swz(frow, kk * 2 + fhalf) * 16;
                    const v4i bw = *reinterpret_cast<const v4i*>(stage + off);
#pragma unroll
                    for (int j = 0; j < TM; ++j) {
                        const v4i ba = *reinterpret_cast<const v4i*>(stage + (1 + j) * kTile + off);
                        acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bw, ba, acc[j], 0, 0, 0);
                    }
                }
                wave_lds_sync();
            }
        });
    }

    Epilogue e;
    e.row_scale = p.a_scale; e.col_scale = p.w_scale;
    e.row_numel = p.a_scale_numel; e.col_numel = p.w_scale_numel;
    e.use_alpha = p.use_alpha; e.alpha = p.alpha; e.round_mode = p.round_mode; e.col_outer = p.scale_order;
    e.ldd = p.ldd; e.d = p.d;
    skinny_reduce_store<TM, OUT, FLEX, false>(e, acc, red, p.m, p.n, m0, n0, tid, kThreads);
}

template <int TM, int WAVES, int OUT, bool FLEX>
int launch_skinny_one(const QaGemmW8A8Params& p, hipStream_t stream) {
    constexpr int kLds = skinny_lds_bytes<TM, WAVES>();
    auto kernel = gemm_w8a8_skinny_kernel<TM, WAVES, 3, OUT, FLEX>;
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

template <int TM, int WAVES, bool FLEX>
int launch_skinny(const QaGemmW8A8Params& p, hipStream_t stream) {
    if (p.out_type == QA_OUT_I8) return launch_skinny_one<TM, WAVES, QA_OUT_I8, FLEX>(p, stream);
    if (p.out_type == QA_OUT_BF16) return launch_skinny_one<TM, WAVES, QA_OUT_BF16, FLEX>(p, stream);
    return launch_skinny_one<TM, WAVES, QA_OUT_F16, FLEX>(p, stream);
}

// ---------------------------------------------------------------------------------------------
// Products of so few outputs that even tiles of 32 x 32 leave most CUs idle (the step-size and B, C projection of a decode
// batch or a short prompt): 16 x 16 outputs per workgroup, K over sixteen waves.  What bounds them is latency - a CU fetches
// its operand rows at about 64 bytes a clock, and every trip to memory counts - so the outputs go to four times the CUs, a wave asks
// for all its fragments (16 rows x 64 bytes, straight into the operand registers of 16x16x64) before it multiplies, and the
// sixteen partial sums meet in LDS with one store and sixteen loads each.
// Against 32 x 32 with K over four waves (rows x outputs x K, us): 64 x 192 x 5120 7.5 -> 6.8, 64 x 80 x 1536 4.0 -> 3.2, 512 x 80
// x 1536 4.7 -> 3.8, 512 x 128 x 3072 5.7 -> 5.1, 16 x 2560 x 5120 9.4 -> 8.7, 16 x 3072 x 768 4.2 -> 3.2.
// ---------------------------------------------------------------------------------------------
template <int OUT>
__global__ __launch_bounds__(1024) void gemm_w8a8_narrow_kernel(QaGemmW8A8Params p) {
    constexpr int kWaves = 16, kUnits = 3;                 // units of 128 bytes of K at a time, all in flight
    __shared__ __align__(16) int red[kWaves][256];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int blocks_m = (p.m + 15) / 16;
    const int m0 = static_cast<int>(blockIdx.x) % blocks_m * 16, n0 = static_cast<int>(blockIdx.x) / blocks_m * 16;
    const int chunk = (lane >> 4) * 16;
    // rows outside repeat the last one: their outputs are not written
    const int8_t* a = p.a + static_cast<int64_t>(min(m0 + (lane & 15), p.m - 1)) * p.lda;
    const int8_t* w = p.w + static_cast<int64_t>(min(n0 + (lane & 15), p.n - 1)) * p.ldw;
    v4i acc = {0, 0, 0, 0};
    for (int k0 = wave * kBK; k0 < p.k; k0 += kUnits * kWaves * kBK) {
        v4i fa[2 * kUnits], fw[2 * kUnits];
#pragma unroll
        for (int s = 0; s < 2 * kUnits; ++s) {
            const int k = k0 + s / 2 * (kWaves * kBK) + s % 2 * 64 + chunk;
            fa[s] = fw[s] = v4i{0, 0, 0, 0};
            if (k < p.k) {
                fw[s] = *reinterpret_cast<const v4i*>(w + k);
                fa[s] = *reinterpret_cast<const v4i*>(a + k);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2 * kUnits; ++s) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw[s], fa[s], acc, 0, 0, 0);
    }
    *reinterpret_cast<v4i*>(&red[wave][lane * 4]) = acc;
    __syncthreads();
    if (threadIdx.x >= 256) return;
    // thread t: row (t >> 2) & 15, column 4 (t >> 6) + (t & 3)
    const int t = threadIdx.x, mm = m0 + ((t >> 2) & 15), nn = n0 + (t >> 6) * 4 + (t & 3);
    if (mm >= p.m || nn >= p.n) return;
    const float s_row = p.a_scale[p.a_scale_numel == 1 ? 0 : mm], s_col = p.w_scale[p.w_scale_numel == 1 ? 0 : nn];
    int sum = 0;
#pragma unroll
    for (int x = 0; x < kWaves; ++x) sum += red[x][t];
    const float accf = static_cast<float>(sum);
    float v = p.scale_order ? s_col * (s_row * accf) : s_row * (s_col * accf);
    asm volatile("" : "+v"(v));                            // the fp32 product is rounded on its own
    const int64_t at = static_cast<int64_t>(mm) * p.ldd + nn;
    if (OUT == QA_OUT_I8) static_cast<int8_t*>(p.d)[at] = static_cast<int8_t>(quant8(v, QA_ROUND_RNE));
    else static_cast<uint16_t*>(p.d)[at] = one_f16_or_bf16<OUT>(v);
}

int launch_narrow(const QaGemmW8A8Params& p, hipStream_t stream) {
    const int64_t blocks = static_cast<int64_t>((p.m + 15) / 16) * ((p.n + 15) / 16);
    auto kernel = p.out_type == QA_OUT_I8 ? gemm_w8a8_narrow_kernel<QA_OUT_I8> : p.out_type == QA_OUT_BF16 ? gemm_w8a8_narrow_kernel<QA_OUT_BF16> : gemm_w8a8_narrow_kernel<QA_OUT_F16>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(1024), 0, stream, p);
    return check_launch();
}

template <bool FLEX>
int dispatch_skinny(const QaGemmW8A8Params& p, hipStream_t stream) {
    return launch_skinny<1, 4, FLEX>(p, stream);
}

// Tile of a launch: the smallest whose tiles fit the part in one round.  With at most one tile per CU a launch takes a
// tile's own time - about 2.5 us and, per 128 bytes of K, 0.105 us (16 x 16, K split over the waves), 0.125 (32 x 32, the same), 0.20 (64 x 64), 0.31
// (128 x 64), 0.48 (128 x 128, four stages), 0.68 (128 x 256), 1.15 (256 x 256) - so smaller tiles win until a second round
// starts.  Measured at M 16 .. 16384 with ten of the projections' N and K: this choice is the fastest or
// within 8 % of it.  Against 128 x 128 tiles up to 192 tiles of 256 x 256 (rows x outputs x K, us): 512 x 80 x 1536 9.6 ->
// 4.1, 3063 x 192 x 5120 21.0 -> 11.7, 512 x 1536 x 3072 14.6 -> 7.7, 777 x 10240 x 2560 45 -> 38, 6144 x 1536 x 3072 47 -> 35.
// From 128 x 64 on a tile is divided over eight waves: a CU that holds one tile then has two waves per SIMD, and one issues
// while the other waits.  Four waves against eight (us): 1531 x 768 x 1536 6.9 -> 6.3, 1024 x 1536 x 3072 10.2 -> 9.8 with
// 128 x 64; 3063 x 768 x 1536 9.2 -> 7.8, 1531 x 1536 x 3072 14.0 -> 12.1, 1531 x 2560 x 5120 28.0 -> 27.8 with 128 x 128.
int dispatch_tiles(const QaGemmW8A8Params& p, hipStream_t stream) {
    const int cus = compute_units();
    auto tiles = [&](int64_t bm, int64_t bn) { return ((p.m + bm - 1) / bm) * ((p.n + bn - 1) / bn); };
    if (tiles(16, 16) <= cus) return launch_narrow(p, stream);                       // (two rounds of these: slower than one of 32 x 32)
    if (tiles(32, 32) <= cus) return dispatch_skinny<false>(p, stream);
    if (tiles(64, 64) <= cus) return launch_gemm<1, 1, 2, 2, 4, false>(p, stream);
    if (tiles(128, 64) <= cus) return launch_gemm<1, 1, 4, 2, 4, false>(p, stream);
    if (tiles(128, 128) <= cus) return launch_gemm<2, 1, 2, 4, 4, false>(p, stream);
    if (tiles(128, 256) <= cus) return launch_gemm<2, 2, 2, 4, 3, false>(p, stream);
    // More than a round: what counts is rounds times the tile's work, 128 x 256 at six fifths of its share and the 320-wide
    // ones at 24/25: they move a tenth less per product through the caches, which at the power limit is time (against
    // 256 x 256 at equal arithmetic 16384 x 10240 x 2560 321 -> 309 us, at 2 % more 16384 x 10576 x 2560 346 -> 339).
    auto cost = [&](int64_t bm, int64_t bn) { return ((tiles(bm, bn) + cus - 1) / cus) * bm * bn; };
    const int64_t c_sq = cost(256, 256), c_wide = cost(256, 320) * 24 / 25, c_tall = cost(320, 256) * 24 / 25, c_half = cost(128, 256) * 6 / 5;
    if (c_half < c_sq && c_half < c_wide && c_half < c_tall) return launch_gemm<2, 2, 2, 4, 3, false>(p, stream);
    if (c_wide <= c_sq && c_wide <= c_tall) return launch_gemm<2, 5, 4, 2, 2, false>(p, stream);
    if (c_tall <= c_sq) return launch_gemm<5, 2, 2, 4, 2, false>(p, stream);
    return launch_gemm<4, 2, 2, 4, 2, false>(p, stream);                             // 256x256 tile, 8 waves
}

}  // namespace
}  // namespace qa

extern "C" int qa_gemm_w8a8(const QaGemmW8A8Params* p, void* stream_) {
    using namespace qa;
    if (!p) return QA_ERR_NULL;
    if (p->m < 0 || p->n < 0 || p->k < 0) return QA_ERR_SHAPE;
    const bool empty = p->m == 0 || p->n == 0;                      // (an output without elements: tensors may be null)
    if (!empty && (!p->a || !p->w || !p->d)) return QA_ERR_NULL;
    if (!empty && !p->use_alpha && (!p->a_scale || !p->w_scale)) return QA_ERR_NULL;
    if (p->out_type != QA_OUT_I8 && p->out_type != QA_OUT_F16 && p->out_type != QA_OUT_BF16) return QA_ERR_UNSUPPORTED;
    if (p->scale_order != 0 && p->scale_order != 1) return QA_ERR_UNSUPPORTED;
    if (p->scale_order == 1 && (p->use_alpha || p->round_mode != QA_ROUND_RNE)) return QA_ERR_UNSUPPORTED;
    if (!p->use_alpha && p->a_scale_numel != 1 && p->a_scale_numel != p->m) return QA_ERR_SHAPE;
    if (!p->use_alpha && p->w_scale_numel != 1 && p->w_scale_numel != p->n) return QA_ERR_SHAPE;
    // 16-byte operand chunks: the same alignment the reference's tensor-core path demands
    if (p->k % 16 != 0 || p->lda % 16 != 0 || p->ldw % 16 != 0 || !aligned16(p->a) || !aligned16(p->w)) return QA_ERR_STRIDE;
    if (p->lda < p->k || p->ldw < p->k || p->ldd < p->n) return QA_ERR_STRIDE;
    if (p->m == 0 || p->n == 0) return QA_OK;
    // operands are addressed with 32-bit byte offsets inside a buffer descriptor
    if (static_cast<int64_t>(p->m) * p->lda >= 0x70000000LL || static_cast<int64_t>(p->n) * p->ldw >= 0x70000000LL) return QA_ERR_SHAPE;
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const bool flex = p->use_alpha || p->round_mode != QA_ROUND_RNE;
    if (p->m <= kGemvRows) {
        GemvParams g = {};
        g.m = p->m; g.n = p->n; g.k = p->k; g.bits = 8;
        g.out_type = p->out_type;
        g.rule = p->use_alpha ? kGemvAlpha : p->round_mode != QA_ROUND_RNE ? kGemvHalfAway : p->scale_order == 1 ? kGemvColOuter : kGemvRowOuter;
        g.alpha = p->alpha;
        g.half_away = p->round_mode != QA_ROUND_RNE;
        g.row_numel = p->a_scale_numel; g.col_numel = p->w_scale_numel;
        g.lda = p->lda; g.ldw = p->ldw; g.ldd = p->ldd;
        g.a = p->a; g.w = p->w; g.row_scale = p->a_scale; g.col_scale = p->w_scale; g.d = p->d;
        return gemv_launch(g, nullptr, stream);
    }
    // the single-row rules (host alpha, round-half-away) only ever come with tiny M
    if (flex) return p->m <= 64 ? dispatch_skinny<true>(*p, stream) : launch_gemm<2, 2, 2, 2, 2, true>(*p, stream);
    return dispatch_tiles(*p, stream);
}
