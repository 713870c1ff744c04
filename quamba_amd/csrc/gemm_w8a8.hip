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

#include <type_traits>

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

constexpr int kNarrow = 256;           // columns whose whole w a workgroup's XCD holds on to

template <int TM, int TN, int WGM, int WGN, int STAGES, int OUT, bool FLEX, bool COL_OUTER, bool TURN>
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
    // Where in K this workgroup's k tile `tile` lies (past the last one: outside K).  TURN: workgroups do not all start at K's
    // beginning.  In step, all of them ask for the same 128 bytes of rows that lie K bytes apart, which few of the memory's
    // channels hold; the order of the sum does not matter, it is exact.  The workgroups of an XCD, which share panels through
    // its L2, start together, an eighth of K from those of the next; with so few columns that w stays in every L2 each row block
    // by itself.
    const int turn = !TURN ? 0 : p.n <= kNarrow ? tile_m * 7 % k_tiles : static_cast<int>(blockIdx.x % 8) * k_tiles / 8;
    auto k_of = [&](int tile) {
        if constexpr (!TURN) return tile * kBK;
        const int t = tile + turn;
        return tile >= k_tiles ? k_tiles * kBK : (t >= k_tiles ? t - k_tiles : t) * kBK;
    };
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
        auto request = [&](int r, int k0, uint32_t stage) {
            if (r < C::kAInstr) load_a.template issue_one<WAVES>(r, rsrc_a, k0, p.k, lds_base + stage, wave);
            else if (r < kReq) load_w.template issue_one<WAVES>(r - C::kAInstr, rsrc_w, k0, p.k, lds_base + stage + BM * kBK, wave);
        };
        auto request_whole = [&](int r, int k0, uint32_t stage) {
            if (r < C::kAInstr) load_a.template issue_whole<WAVES>(r, rsrc_a, k0, lds_base + stage, wave);
            else if (r < kReq) load_w.template issue_whole<WAVES>(r - C::kAInstr, rsrc_w, k0, lds_base + stage + BM * kBK, wave);
        };
#pragma unroll
        for (int t = 0; t < STAGES - 1; ++t)
#pragma unroll
            for (int r = 0; r < kReq; ++r) request(r, k_of(t), t * C::kStageBytes);
        int k_late = k_of(STAGES - 1);                                 // of the tile STAGES - 1 further than the one at hand
#pragma unroll
        for (int r = 0; r < kEarly; ++r) request(r, k_late, (STAGES - 1) * C::kStageBytes);
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
            const int k_early = k_of(kt + STAGES);
            mma.template tile<(STAGES - 2) * kReq>(my_a + cur, my_w + cur, my_a + nxt, my_w + nxt, [&](int idx) {
                if (idx % kPace != kPace - 1) return;
                const int r = idx / kPace;
                if (r < kEarly) req(r, k_early, cur);
                else req(r, k_late, late);
            });
            k_late = k_early;
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
        load_a.template issue<WAVES>(rsrc_a, k_of(tile), p.k, base, wave);
        load_w.template issue<WAVES>(rsrc_w, k_of(tile), p.k, base + BM * kBK, wave);
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
        const int nk = k_of(nt);
        static_assert(C::kAInstr + C::kWInstr <= 4, "a request behind each of four multiplications");
        mma_tile_paced(stage + wm * 32 * kBK, stage + BM * kBK + wn * 32 * kBK, frow, fhalf, acc[0][0], [&](int r) {
            if (r < C::kAInstr) load_a.template issue_one<WAVES>(r, rsrc_a, nk, p.k, nbase, wave);
            else if (r < C::kAInstr + C::kWInstr) load_w.template issue_one<WAVES>(r - C::kAInstr, rsrc_w, nk, p.k, nbase + BM * kBK, wave);
        });
    }
    finish(acc);
    }
}

template <int TM, int TN, int WGM, int WGN, int STAGES, int OUT, bool FLEX, bool TURN, bool COL_OUTER = false>
int launch_one(const QaGemmW8A8Params& p, hipStream_t stream) {
    using C = Cfg<TM, TN, WGM, WGN, STAGES>;
    if constexpr (!FLEX && !COL_OUTER) {
        if (p.scale_order == 1) return launch_one<TM, TN, WGM, WGN, STAGES, OUT, FLEX, TURN, true>(p, stream);
    }
    const int64_t tiles = static_cast<int64_t>((p.m + C::kBM - 1) / C::kBM) * ((p.n + C::kBN - 1) / C::kBN);
    if (tiles > 0x7fffffffLL) return QA_ERR_SHAPE;
    auto kernel = gemm_w8a8_kernel<TM, TN, WGM, WGN, STAGES, OUT, FLEX, COL_OUTER, TURN>;
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

template <int TM, int TN, int WGM, int WGN, int STAGES, bool FLEX, bool TURN = false>
int launch_gemm(const QaGemmW8A8Params& p, hipStream_t stream) {
    if (p.out_type == QA_OUT_I8) return launch_one<TM, TN, WGM, WGN, STAGES, QA_OUT_I8, FLEX, TURN>(p, stream);
    if (p.out_type == QA_OUT_BF16) return launch_one<TM, TN, WGM, WGN, STAGES, QA_OUT_BF16, FLEX, TURN>(p, stream);
    return launch_one<TM, TN, WGM, WGN, STAGES, QA_OUT_F16, FLEX, TURN>(p, stream);
}

GemvParams as_gemv(const QaGemmW8A8Params& p) {
    GemvParams g = {};
    g.m = p.m; g.n = p.n; g.k = p.k; g.bits = 8;
    g.out_type = p.out_type;
    g.rule = p.use_alpha ? kGemvAlpha : p.round_mode != QA_ROUND_RNE ? kGemvHalfAway : p.scale_order == 1 ? kGemvColOuter : kGemvRowOuter;
    g.alpha = p.alpha;
    g.half_away = p.round_mode != QA_ROUND_RNE;
    g.row_numel = p.a_scale_numel; g.col_numel = p.w_scale_numel;
    g.lda = p.lda; g.ldw = p.ldw; g.ldd = p.ldd;
    g.a = p.a; g.w = p.w; g.row_scale = p.a_scale; g.col_scale = p.w_scale; g.d = p.d;
    return g;
}

// Tile of a launch: the smallest whose tiles fit the part in one round.  With at most one tile per CU a launch takes a
// tile's own time - about 2.5 us and, per 128 bytes of K, 0.20 us (64 x 64), 0.31 (128 x 64), 0.48 (128 x 128, four stages),
// 0.58 (192 x 128), 0.68 (128 x 256), 1.15 (256 x 256) - so smaller tiles win until a second round starts; below that K split over the waves
// (gemm_split.hpp) where its cost is the smaller one.  Measured at M 16 .. 16384 with ten of the projections' N and K: this choice is the fastest or
// within 8 % of it.  Against 128 x 128 tiles up to 192 tiles of 256 x 256 (rows x outputs x K, us): 512 x 1536 x 3072 14.6 ->
// 7.7, 777 x 10240 x 2560 45 -> 38, 6144 x 1536 x 3072 47 -> 35.
// From 128 x 64 on a tile is divided over eight waves: a CU that holds one tile then has two waves per SIMD, and one issues
// while the other waits.  Four waves against eight (us): 1531 x 768 x 1536 6.9 -> 6.3, 1024 x 1536 x 3072 10.2 -> 9.8 with
// 128 x 64; 3063 x 768 x 1536 9.2 -> 7.8, 1531 x 1536 x 3072 14.0 -> 12.1, 1531 x 2560 x 5120 28.0 -> 27.8 with 128 x 128.
int dispatch_tiles(const QaGemmW8A8Params& p, hipStream_t stream) {
    const int cus = compute_units();
    auto tiles = [&](int64_t bm, int64_t bn) { return ((p.m + bm - 1) / bm) * ((p.n + bn - 1) / bn); };
    if (tiles(128, 128) <= cus) {
        const SplitChoice split = split_choice(8, p.m, p.n, p.k, cus);
        // (64 rows and more columns than 256 times 64: what is wanted is the weights at the memory's rate, and 128 x 128 tiles, which
        // do not fetch the rows they lack, ask for them better: 64 x 18560 x 4096 17.9 us by 64 x 80, 15.4 in tiles, 48 x 17600 x 2048
        // 11.1 and 9.7, 33 x 16400 x 8192 24.7 and 25.7)
        // (a short K: what the tiles' estimate leaves out, their first trip to memory, is then most of it: 9 x 3072 x 96 4.6 us and 4.0 by
        // 16 x 16, 565 x 405 x 400 4.9 and 4.1 by 16 x 48, 65 x 3352 x 768 5.0 and 4.2 by 32 x 48; 512 x 1024 x 2048 5.7, 6.0 by 32 x 32)
        const float alone = p.k <= 1024 ? 0.6f : 0.0f;
        const bool streams = p.m <= 64 && kSplitShapes[split.shape].rows == 64;
        if (split.us < tiles_us_w8(p.m, p.n, p.k, cus) + alone && !streams) return split_launch_w8(as_gemv(p), split.shape, nullptr, stream);
    }
    if (tiles(64, 64) <= cus) return launch_gemm<1, 1, 2, 2, 4, false>(p, stream);
    if (tiles(128, 64) <= cus) return launch_gemm<1, 1, 4, 2, 4, false>(p, stream);
    if (tiles(128, 128) <= cus) {
        // (16384 x 192 x 5120 34.5 -> 26.2 us, 12000 x 160 x 4096 27.5 -> 19.5)
        if (p.n <= kNarrow && p.k >= 1024 && p.k % kBK == 0) return launch_gemm<2, 1, 2, 4, 4, false, true>(p, stream);
        return launch_gemm<2, 1, 2, 4, 4, false>(p, stream);
    }
    // (between the two a tile's time goes with its area, and a round of 192 x 128 is three quarters of one of 128 x 256: 1536 x 4096 x 1024
    // 10.3 -> 8.9 us, 777 x 6144 x 1536 15.9 -> 11.6, 768 x 8192 x 2048 19.7 -> 14.5, 2304 x 2560 x 5120 30 - 40 -> 27 - 34 with operands in the
    // last-level cache and from memory)
    if (tiles(192, 128) <= cus) return launch_gemm<3, 1, 2, 4, 3, false>(p, stream);
    if (tiles(128, 256) <= cus) return launch_gemm<2, 2, 2, 4, 3, false>(p, stream);
    // More than a round: what counts is rounds times the tile's work, 128 x 256 at six fifths of its share and the 320-wide
    // ones at 24/25: they move a tenth less per product through the caches, which at the power limit is time (against
    // 256 x 256 at equal arithmetic 16384 x 10240 x 2560 321 -> 309 us, at 2 % more 16384 x 10576 x 2560 346 -> 339).
    auto cost = [&](int64_t bm, int64_t bn) { return ((tiles(bm, bn) + cus - 1) / cus) * bm * bn; };
    const int64_t c_sq = cost(256, 256), c_wide = cost(256, 320) * 24 / 25, c_tall = cost(320, 256) * 24 / 25, c_half = cost(128, 256) * 6 / 5;
    if (c_half < c_sq && c_half < c_wide && c_half < c_tall) return launch_gemm<2, 2, 2, 4, 3, false>(p, stream);
    // Starting points in K of their own (us without and with): 16384 x 10240 x 2560 335 -> 313, 16384 x 10448 x 2560 364 -> 343,
    // 8192 x 2048 x 4096 56.6 -> 53.6, 16384 x 4096 x 8192 394 -> 387, 12000 x 1536 x 3072 51.0 -> 49.1.  A short K is over before they drift
    // together, and two rounds of tiles share less that way than in step: 12000 x 8192 x 2048 165 -> 170, 3000 x 10240 x 2560 63.5 -> 65.2.
    const bool turn = p.k % kBK == 0 && (p.k >= 3072 || (p.k >= 2560 && tiles(256, 256) > 2 * cus));
    auto go = [&](auto turn_c) {
        constexpr bool kTurn = decltype(turn_c)::value;
        if (c_wide <= c_sq && c_wide <= c_tall) return launch_gemm<2, 5, 4, 2, 2, false, kTurn>(p, stream);
        if (c_tall <= c_sq) return launch_gemm<5, 2, 2, 4, 2, false, kTurn>(p, stream);
        return launch_gemm<4, 2, 2, 4, 2, false, kTurn>(p, stream);                          // 256x256 tile, 8 waves
    };
    return turn ? go(std::true_type{}) : go(std::false_type{});
}

}  // namespace

float tiles_us_w8(int m, int n, int k, int cus) {
    auto fits = [&](int64_t bm, int64_t bn) { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn) <= cus; };
    return 2.5f + static_cast<float>((k + gemm::kBK - 1) / gemm::kBK) * (fits(64, 64) ? 0.20f : fits(128, 64) ? 0.31f : fits(128, 128) ? 0.48f : fits(192, 128) ? 0.58f : fits(128, 256) ? 0.68f : 1.15f);
}

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
    if (gemv_is_faster(8, p->m, p->n, p->k)) return gemv_launch(as_gemv(*p), nullptr, stream);
    // the single-row rules (host alpha, round-half-away) only ever come with tiny M
    if (flex && p->m <= 64) return split_launch_w8(as_gemv(*p), split_choice(8, p->m, p->n, p->k, compute_units()).shape, nullptr, stream);
    if (flex) return launch_gemm<2, 2, 2, 2, 2, true>(*p, stream);
    return dispatch_tiles(*p, stream);
}
