// Device entry points of the C ABI: validate on the host, then enqueue.
#include <algorithm>
#include <climits>
#include <cstdint>
#include <cmath>
#include <cstring>
#include <vector>

#include "nh_runtime.h"

using namespace nh;

namespace {

constexpr int64_t kMaxGrid = 0x7fffffff;

unsigned grid_for(int64_t items, int per_block) {
    int64_t g = (items + per_block - 1) / per_block;
    g = std::max<int64_t>(1, std::min<int64_t>(g, 1 << 20));
    return (unsigned)g;
}

// Whether [a, a + an) and [b, b + bn) share bytes.
bool overlap(const void* a, size_t an, const void* b, size_t bn) {
    return an != 0 && bn != 0 && (uintptr_t)a < (uintptr_t)b + bn && (uintptr_t)b < (uintptr_t)a + an;
}

// Waves per workgroup of the GEMV family: wave w owns K tiles w, w + W, ...,
// at most 16 of them per register slab; W = ceil(KT / 16) up to 8 waves
// (longer K is walked slab by slab).
int gemv_waves(int kt) { return std::max(1, std::min(8, (kt + 15) / 16)); }

// The linear entry point's M ranges: the fused decode unit (quantizer inside
// the GEMV, one launch) for up to 4 bf16 rows (K <= 8192) and for 3..16 bf16
// rows (K <= 4096, K % 512 == 0, the streaming form), and for one f32 or longer
// row that no output overlaps (long_row_ok); other bf16 rows up to 16 with K =
// 4048..8192 on a grid that the CUs take at once, or of weights enough to hide
// the rows, as the handoff launch (quantizer workgroups feeding the tiled-A
// GEMV's workgroups inside one launch); otherwise quantization into
// activation tiles + the tiled-A GEMV up to 16 rows, and the MFMA GEMMs beyond.
constexpr size_t kTiledActRows = 16;

// Fused decode unit: kernel, N tiles per workgroup, block size, LDS bytes.
struct DecodePlan {
    KernelId kid;
    int ntw, threads;
    size_t lds;
};

bool plan_decode(const nh_context* ctx, size_t m, size_t n, size_t k, DecodePlan* p) {
    if (m == 0 || m > 8 || k > 8192) return false;
    const int kt = (int)tiled_k_tiles(k);
    const int w = gemv_waves(kt);
    // one N tile per workgroup, the rows' codes in LDS (up to 4 rows)
    auto row_plan = [&]() {
        const size_t rows = m == 1 ? 1 : m <= 2 ? 2 : 4;
        const KernelId kid = m == 1 ? K_LINEAR_DECODE_M1 : m <= 2 ? K_LINEAR_DECODE_ROW2 : K_LINEAR_DECODE_ROW4;
        *p = DecodePlan{kid, 1, 64 * w, rows * ((size_t)w * 1024 + 16)};
        return p->lds <= ctx->max_shared_per_block;
    };
    if (m == 1) return row_plan();
    // several N tiles per workgroup: the widest (up to 16 waves) that still
    // gives every CU one; at one N tile the row kernel is faster up to 4 rows
    if (k % 512 == 0) {
        const int mm = m <= 2 ? 2 : m <= 4 ? 4 : 8;
        const int xr = mm == 2 ? 4 : 8;  // activation chunks each thread holds
        const KernelId kid = mm == 2 ? K_LINEAR_DECODE_M2 : mm == 4 ? K_LINEAR_DECODE : K_LINEAR_DECODE_M8;
        const size_t tiles = (n + 15) / 16;
        auto fits = [&](int ntw) {
            return m * (k / 8) <= (size_t)xr * 64 * w * ntw &&
                   (size_t)kt * 64 * mm + (size_t)w * ntw * 1024 + (size_t)mm * 4 <= ctx->max_shared_per_block;
        };
        auto wide = [&](int ntw) {
            *p = DecodePlan{kid, ntw, 64 * w * ntw, (size_t)kt * 64 * mm + (size_t)w * ntw * 1024 + (size_t)mm * 4};
            return true;
        };
        const size_t cu = (size_t)ctx->cu_count;
        for (int ntw = 16 / w; ntw >= 1; ntw /= 2) {
            // one wide workgroup per CU at a time: whole rounds only (a
            // partial second round costs a full one: 28.7 us at M = 8,
            // 4096 -> 21504, 336 workgroups, against ~20 us in two launches)
            const size_t wgs = (tiles + ntw - 1) / ntw;
            if (ntw > 1 && (wgs < cu || (wgs % cu != 0 && wgs < 4 * cu))) continue;
            if (ntw == 1 && m <= 4) break;
            if (fits(ntw)) return wide(ntw);
        }
        // (a wide workgroup on fewer CUs than the chip has loses to the
        // two-launch path: 20.0 vs ~15 us at M = 8, K = 8192, N = 4096)
    }
    return m <= 4 && row_plan();
}

// Streaming decode unit (3..16 bf16 rows, K % 512 == 0, K <= 4096, any N):
// G workgroups of 16 waves, each quantizing the rows once and walking a run
// of ceil(tiles / G) or one fewer N tiles; G is the CU count or, at the same
// number of rounds, as few workgroups as that many rounds need.  (At K = 8192
// each CU would load 128 KiB of activations, as much as its share of a
// 4096-wide output's weights: 16.4 us against 14.7 in two launches.)
bool plan_stream_grid(const nh_context* ctx, KernelId kid, size_t mm, size_t n, size_t k, DecodePlan* p, unsigned* grid) {
    const size_t tiles = (n + 15) / 16, cu = (size_t)ctx->cu_count;
    const size_t rounds = (tiles + cu - 1) / cu;
    if (rounds > 64) return false;  // a run's scales and bias: at most 1024 LDS floats each
    // codes [KT][4][MM][16], two sets of 16 partial tiles, the run's scales
    // and bias, row maxima, row scales and (W4) row code sums
    const size_t lds = (size_t)tiled_k_tiles(k) * 64 * mm + 2 * 16 * 64 * 16 + 2 * 1024 * 4 + 3 * mm * 4;
    if (lds > ctx->max_shared_per_block) return false;
    *p = DecodePlan{kid, 0, 1024, lds};
    *grid = (unsigned)((tiles + rounds - 1) / rounds);
    return true;
}

bool plan_stream(const nh_context* ctx, size_t m, size_t n, size_t k, DecodePlan* p, unsigned* grid) {
    if (m < 3 || m > 16 || k % 512 != 0 || k > 4096) return false;
    const size_t mm = m <= 4 ? 4 : m <= 8 ? 8 : 16;
    const KernelId kid =
        mm == 4 ? K_LINEAR_DECODE_STREAM_M4 : mm == 8 ? K_LINEAR_DECODE_STREAM_M8 : K_LINEAR_DECODE_STREAM_M16;
    return plan_stream_grid(ctx, kid, mm, n, k, p, grid);
}

// The INT4 form of 3..16 rows for the other K (multiples of 16): up to 4096,
// and up to 8 rows past that.  The one-tile unit quantizes 1..4 rows in every
// workgroup: at 3..4 it keeps short K, and the long form's narrow outputs (3
// rows, one-tile / this: K = 272 x 4096 5.4 us / 6.5, 1040 x 4096 6.8 / 6.9, 2064 x 4096 7.6 /
// 7.4, 4080 x 40960 26.8 / 17.5; 4640 x 8192 11.0 / 12.1, x 10000 17.4 / 14.4, x 40960 55.1 /
// 25.8); 2 rows are the same or slower here up to 24576 columns.
bool plan_stream_w4_any(const nh_context* ctx, size_t m, size_t n, size_t k, DecodePlan* p, unsigned* grid) {
    if (m > (k <= 4096 ? 16u : 8u) || k > 8192) return false;
    if (m <= 2 || (m <= 4 && (k <= 4096 ? k < 1024 : n <= 32 * (size_t)ctx->cu_count))) return false;
    const KernelId kid = k > 4096 ? K_LINEAR_DECODE_STREAM_W4_LONG_M8
                         : m <= 8 ? K_LINEAR_DECODE_STREAM_W4_ANY_M8
                                  : K_LINEAR_DECODE_STREAM_W4_ANY_M16;
    return plan_stream_grid(ctx, kid, m <= 8 ? 8 : 16, n, k, p, grid);
}

// The long-row decode unit takes one row of whole 16-byte chunks that its 512
// threads hold in registers.  Every workgroup quantizes the row, so where
// the CUs run several of them one after another that must be little next to
// their weights: K >= 8192 (1 x 12288 bf16 -> 16384 39.2 us against 42.0 in two
// launches), but 1 x 4096 f32 -> 12288 16.6 against 14.3.  They also read it while
// others already store, so no output may lie over the row (the two launches
// read it first, and take such calls).
bool long_row_ok(const nh_context* ctx, const void* x, nh_dtype dtype, size_t m, size_t n, size_t k, const void* out,
                 nh_dtype out_dtype, const int8_t* xq_out, const float* sx_out) {
    const size_t vpc = dtype == NH_BF16 ? 8 : 4, kt = (size_t)tiled_k_tiles(k), row = k * (16 / vpc);
    return m == 1 && k % 16 == 0 && aligned16(x) && ((uintptr_t)xq_out & (vpc - 1)) == 0 &&
           kt * 64 / vpc <= (size_t)kLongChunks && ((n + 15) / 16 <= (size_t)ctx->cu_count || kt >= 128) &&
           kt * 64 + 9 * 1024 <= ctx->max_shared_per_block &&
           !overlap(x, row, out, n * (out_dtype == NH_BF16 ? 2 : 4)) && !overlap(x, row, xq_out, xq_out ? k : 0) &&
           !overlap(x, row, sx_out, sx_out ? sizeof(float) : 0);
}

// Dynamic LDS of the GEMM kernels: a ring of `stages` stages of `ks` K tiles
// (BM rows x 64 ks bytes of A plus ks * BN/16 weight tiles of 1 KiB), then
// the tile's scales and bias (BM + 2 BN floats) for the epilogue.
size_t gemm_lds_bytes(int bm, int bn, int stages, int ks = 2) {
    const size_t ring = (size_t)stages * ((size_t)bm * 64 * ks + (size_t)ks * (size_t)(bn / 16) * 1024);
    return ring + (size_t)(bm + 2 * bn) * 4;
}

nh_status check_dtype(nh_dtype d, nh_error* err) {
    if (d != NH_F32 && d != NH_BF16) return set_error(err, NH_INVALID_PARAMS, "unknown dtype %d", (int)d);
    return NH_OK;
}

// Shared validation of the W8A8 GEMM family (GemmError::InvalidShape for a
// zero or overflowing dimension, gemm.rs:192-208; envelope for the rest).
nh_status check_w8a8_shape(size_t m, size_t n, size_t k, nh_error* err) {
    size_t t;
    if (m == 0 || n == 0 || k == 0 || !mul_ok(m, k, &t) || !mul_ok(n, k, &t) || !mul_ok(m, n, &t))
        return set_error(err, NH_INVALID_SHAPE, "invalid GEMM shape m=%zu n=%zu k=%zu", m, n, k);
    if (!nh_supports_gemm_w8a8(m, n, k))
        return set_error(err, NH_UNSUPPORTED, "shape m=%zu n=%zu k=%zu outside the gfx950 envelope (k %% 16 == 0, "
                         "k <= 131072, dims < 2^31)", m, n, k);
    return NH_OK;
}

// Row quantizer launch (Q1/Q2): codes row-major into q and/or into the
// activation tiles q_act (rows <= 16).  The vector path needs 16-byte aligned
// rows of whole 16-byte chunks and code stores aligned to a chunk's codes.
nh_status launch_quantize(nh_context* ctx, const void* x, nh_dtype dtype, size_t rows, size_t cols, int8_t* q,
                          float* scales, int32_t* row_status, int8_t* q_act, nh_stream stream, nh_error* err,
                          int act_p = 0, const int32_t* gather = nullptr, int gather_div = 1,
                          uint64_t* nonfinite = nullptr, int nonfinite_stage = 0) {
    const size_t esz = dtype == NH_BF16 ? 2 : 4;
    const size_t row_bytes = cols * esz;
    const bool vec = aligned16(x) && row_bytes % 16 == 0 && row_bytes < (1ull << 31) &&
                     ((uintptr_t)q % (16 / esz)) == 0 && aligned16(q_act);
    QuantizeRowsArgs a{x, q, scales, row_status, q_act, (int64_t)rows, (int64_t)cols, dtype, vec ? 1 : 0,
                       act_p > 0 ? act_p : (int)rows, gather_div, gather, nonfinite, nonfinite_stage, 0};
    // the GEMM's A tiles for rows of up to 512 chunks: 8 rows per workgroup,
    // whole 128-byte lines per store (M = 2048 linear layer, 4096 -> 4096:
    // 45.6-45.8 us against 46.1-46.7 with the wave kernel).  A few rows of more
    // than 1 KiB leave CUs idle that way, and a workgroup per row is faster
    // (profiles/quantizer_choice.csv, in calls with a 256-column product, tiles /
    // row: 288 x 64 f32 5.8 us / 6.2, 300 x 3072 bf16 0.6 more, 800 x 2048 f32
    // 13.9 / 15.1; 1298 x 3856 bf16, 31 KiB of codes per workgroup, 21.8 / 20.6).
    const size_t cus = (size_t)ctx->cu_count;
    const size_t tile_rows = row_bytes <= 1024 ? 0 : row_bytes <= 2048 ? cus : cols <= 2560 ? 2 * cus : 4 * cus;
    if (vec && q_act && act_p == 16 && !gather && rows >= tile_rows && row_bytes <= 512 * 16) {
        const size_t lds = 8 * 64 * tiled_k_tiles(cols);
        return launch(ctx, K_QUANTIZE_TILES, (unsigned)((rows + 7) / 8), 512, lds, stream, a, err);
    }
    // many rows of up to 512 16-byte chunks: one wave per row, no barrier
    // (3072 MoE routes: 299.6 vs 304 us per layer; a few decode rows keep a
    // workgroup each: 8 rows of 4096 on 2 workgroups cost the 52-layer stack
    // 2.26 vs 2.15 ms)
    if (vec && row_bytes <= 512 * 16 && rows >= 1024)
        return launch(ctx, K_QUANTIZE_ROWS_WAVE, (unsigned)((rows + 3) / 4), 256, 0, stream, a, err);
    // a few rows longer than a 256-thread workgroup holds in registers
    // (1024 chunks; 2816 in the form below): 1024 threads per row, one round
    // trip to memory; up to four rows per CU of more than 4608 chunks (500 x
    // 21504 f32 with its product 69.7 against 72.6 us, 1000 rows 83.5 / 86.7; but
    // 716 x 11776 f32 45.2 / 41.8, 899 x 15760 60.5 / 59.0)
    if (vec && row_bytes > 1024 * 16 && rows <= (row_bytes > 4608 * 16 ? 4 : 1) * cus)
        return launch(ctx, K_QUANTIZE_ROWS_LONG, (unsigned)rows, 1024, 0, stream, a, err);
    // many rows of 1025..2816 chunks: the whole row in a 256-thread workgroup's
    // registers, read once (2048 x 21504 bf16: 3 us less)
    if (vec && row_bytes > 1024 * 16 && row_bytes <= 2816 * 16)
        return launch(ctx, K_QUANTIZE_ROWS_R11, (unsigned)rows, 256, 0, stream, a, err);
    return launch(ctx, K_QUANTIZE_ROWS, (unsigned)rows, 256, 0, stream, a, err);
}

// Bytes of the activation tiles of m <= 16 rows of k codes.
size_t act_tiles_bytes(size_t m, size_t k) { return m * (size_t)tiled_k_tiles(k) * 64; }
size_t align256(size_t b) { return (b + 255) / 256 * 256; }

nh_status launch_gemv(nh_context* ctx, const int8_t* xq, const float* sx, const int8_t* wq, const float* sw,
                      const float* bias, int M, int N, int K, void* out, nh_dtype out_dtype, bool x_tiled,
                      nh_stream stream, nh_error* err, int relu2 = 0) {
    GemvW8A8Args a{};
    a.xq = xq;
    a.sx = sx;
    a.wq = wq;
    a.sw = sw;
    a.bias = bias;
    a.out = out;
    a.M = M;
    a.N = N;
    a.K = K;
    a.kt = (int)tiled_k_tiles(K);
    a.waves = gemv_waves(a.kt);
    a.out_dtype = out_dtype;
    a.x_tiled = x_tiled ? 1 : 0;
    a.relu2 = relu2;
    return launch(ctx, x_tiled ? K_GEMV_W8A8_XT : K_GEMV_W8A8, (unsigned)((N + 15) / 16), 64u * a.waves, 0, stream,
                  a, err);
}

// The persistent 256 x 224 GEMM (gemm_persistent.hip): whether its contract holds.
// Its LDS: two A slots of 2 x 16 tiles, three B slots of 2 x 14 tiles (the
// weights run a stage further ahead), three scale buffers, a spare KiB.
constexpr size_t kP224Lds = 2 * 8 * ((2 * 256 / 16 + 7) / 8) * 1024 + 3 * (2 * 224 / 16) * 1024 + 3 * 3 * 1024 + 1024;

bool persistent_224_ok(const nh_context* ctx, const void* xq, const float* sx, const float* sw, const float* bias,
                       int M, int N, int kt, const void* out, nh_dtype out_dtype) {
    const size_t esz = out_dtype == NH_BF16 ? 2 : 4;
    return kt % 2 == 0 && M % 4 == 0 && N % 4 == 0 && aligned16(xq) && aligned16(sx) && aligned16(sw) &&
           aligned16(bias) && aligned16(out) && (uint64_t)M * N * esz < (1ull << 31) &&
           kP224Lds <= ctx->max_shared_per_block;
}

// The LDS-tiled G3 kernels (gemm.hip) on tiled A, largest first.
struct GemmCfg {
    KernelId id;
    int bm, bn, threads;
    size_t lds;  // ring of stages + the tile's scales and bias
};

const GemmCfg kTiledCfgs[] = {{K_GEMM_TA_256, 256, 128, 1024, gemm_lds_bytes(256, 128, 3)},
                              {K_GEMM_TA_128, 128, 128, 512, gemm_lds_bytes(128, 128, 3)},
                              {K_GEMM_TA_64, 64, 128, 384, gemm_lds_bytes(64, 128, 3)},
                              {K_GEMM_TA_6464, 64, 64, 384, gemm_lds_bytes(64, 64, 3)}};

int64_t gemm_tiles(const GemmCfg& c, int M, int N) {
    return (int64_t)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
}

// What a GEMM on tiled A takes, in us: the kernels' choice is the least of
// these.  Coefficients fitted to the choice on 1600 shapes of 17..2048 rows,
// 64..131072 columns and K = 64..21504 with weights not in any cache, and 600
// with one matrix called over and over, each timed with all eight kernels (the
// times: profiles/gemm_choice.csv).  Over them and over 800 others the choice
// is within 1% of the best on average (2% in cache); a model of the LDS tiles
// alone, fitted from K = 1024 on, with the persistent kernel ahead of it, was
// 7% off, and up to 2.9 times (24 x 38400 x 80 13.9 us on the persistent kernel,
// 4.8 on 64 x 64 tiles; 64 x 33280 x 3440 43 / 23).
//
// A tile kernel: a launch; per whole round of workgroups an epilogue and what
// its stage loop takes per 64-deep K tile whatever the tile holds, more with
// more CUs busy (their clock) and with weights that come from HBM (`cold`,
// from 4 MB on); for each workgroup that shares a CU its own MFMAs.  Beside
// that runs the memory traffic, weights and outputs (f32 ones as much as 1 +
// out_f32 bf16 ones); the two overlap in part (root of the squares).
struct TileTime {
    double launch, round, kt, kt_fill, kt_cold, kt_each, hbm, out, out_f32;
};
constexpr TileTime kTileTime[] = {{1.90, 5.69, 0.148, 0.074, 0.034, 0.106, 9.0, 3.23, 0.19},  // kTiledCfgs[0..3]
                                  {3.02, 1.93, 0.151, 0.086, 0.041, 0.003, 7.9, 1.65, 0.24},
                                  {2.50, 1.53, 0.162, 0.018, 0.019, 0.000, 6.1, 4.39, 0.48},
                                  {2.95, 0.18, 0.082, -0.001, 0.003, 0.101, 9.0, 2.11, 0.12}};
constexpr TileTime kP224Time = {3.84, 6.34, 0.547, 0.022, 0.085, 0.0, 8.9, 2.58, 0.0};

// A GEMM's sizes as the models use them.
struct GemmSize {
    int M, N, kt;
    double weights, outputs;  // MB (outputs as bf16)
    bool f32_out;
};

GemmSize gemm_size(int M, int N, int kt, nh_dtype out_dtype) {
    return GemmSize{M, N, kt, (double)N * kt * 64e-6, (double)M * N * 2e-6, out_dtype == NH_F32};
}

double tile_us(const nh_context* ctx, const TileTime& c, int bm, int bn, const GemmSize& g) {
    const double cu = ctx->cu_count, t = (double)((g.M + bm - 1) / bm) * (double)((g.N + (int64_t)bn - 1) / bn);
    const double rounds = std::ceil(t / cu), each = std::max(1.0, t / cu), fill = std::min(1.0, t / cu);
    const double loop = rounds * (c.round + g.kt * (c.kt + c.kt_fill * fill + c.kt_cold * std::min(1.0, g.weights / 4))) +
                        each * g.kt * c.kt_each;
    const double mem = g.weights / c.hbm + g.outputs * (g.f32_out ? 1 + c.out_f32 : 1.0) / c.out;
    return c.launch + std::sqrt(loop * loop + mem * mem);
}

// The register-direct GEMM (gemm_direct.hip): its tile for a shape, and the
// time its launch takes, in us.
struct DirectPlan {
    KernelId id;
    int nr, groups;
    unsigned grid;
    double us;
};

// Its model: a launch, more with more CUs taking part; per round (or partly,
// INT4, per CU's share of one: two workgroups of a CU overlap there) an
// epilogue per fragment, and per K tile the fragments through the CU's load
// path (`a` us per KiB of activations, `b` of weights: 93 and 69 KiB per us), also, at
// `ahead` of the cost, for the loads past the end that a wave's `depth` K tiles
// in flight round up to; beside that the memory traffic and a wave's chain of dependent
// steps.  Against the LDS tiles, both measured at M x N x K: 17 x 2688 x 2688
// 5.5 / 11.8 us, 77 x 6144 x 4096 11.5 / 15.8, 400 x 2688 x 4096 15.5 / 20.9, 64 x
// 16384 x 1024 7.8 / 6.8, 512 x 16384 x 4096 49.2 / 36.2.
struct DirectTime {
    double whole, a, b, launch, round, frag, hbm, out, fill, out_f32, ahead, step;
};
constexpr DirectTime kDirectTime = {1.00, 0.0108, 0.0145, 2.50, 0.02, 0.042, 6.8, 1.81, 0.0, 0.33, 0.89, 0.78};
constexpr DirectTime kDirectTimeW4 = {0.83, 0.0131, 0.0288, 3.65, 0.36, 0.093, 8.9, 20.0, 0.0, 1.0, 0.68, 0.52};

// partial fragments of 4 waves, row and column scales, bias, INT4 row sums
constexpr size_t kDirectLds = 4 * 16 * 1024 + 3 * 128 * 4 + 4 * 128 * 4;
constexpr double kNoPlan = 1e30;

DirectPlan plan_direct(const nh_context* ctx, const GemmSize& g, bool w4) {
    DirectPlan best{};
    best.us = kNoPlan;
    if (kDirectLds > ctx->max_shared_per_block) return best;
    const DirectTime& c = w4 ? kDirectTimeW4 : kDirectTime;
    const int mtiles = (g.M + 15) / 16, steps = (g.kt + 3) / 4;
    const double cu = ctx->cu_count;
    const double mem = g.weights * (w4 ? 0.5 : 1.0) / c.hbm + g.outputs * (g.f32_out ? 1 + c.out_f32 : 1.0) / c.out;
    for (int nr : {1, 2, 4, 8}) {
        if (nr == 8 && !w4) break;
        const int maxr = nr == 8 ? 4 : 8;
        const int groups = (mtiles + maxr - 1) / maxr;
        const int mr = (mtiles + groups - 1) / groups;
        const int64_t tn = ((int64_t)g.N + 16 * nr - 1) / (16 * nr), wgs = tn * groups;
        const int64_t grid = (tn + 7) / 8 * 8 * groups;  // a column block's row groups are on one of 8 XCDs
        if (grid > kMaxGrid) continue;
        // (whole rounds are the fullest XCD's: 1309 x 640 x 2048 would be 220 workgroups
        // of 32 columns, 33 on some XCDs: 12.2 us, on 64 x 64 tiles 9.4)
        const double share = (double)wgs / cu;
        const double rounds = c.whole * std::ceil(w4 ? share : (double)grid / cu) + (1 - c.whole) * std::max(1.0, share);
        const int depth = direct_depth(mr, nr, w4);
        const int issued = 4 * (depth + (steps + depth - 1) / depth * depth);  // K tiles that the waves load
        const double tiles = g.kt + c.ahead * (issued - g.kt);
        // 128 columns of INT4: 6% less than their fragments
        const double load = rounds * tiles * (mr * c.a + (w4 ? 0.5 : 1.0) * nr * c.b) * (nr == 8 ? 0.94 : 1.0);
        const double chain = std::max(0.0, (double)steps / depth - 1) * c.step;
        const double us = c.launch + c.fill * std::min(1.0, share) + rounds * (c.round + c.frag * mr * nr) +
                          std::sqrt(load * load + mem * mem + chain * chain);
        if (us >= best.us) continue;
        const KernelId id8[] = {K_GEMM_DIRECT16, K_GEMM_DIRECT32, K_GEMM_DIRECT64, K_GEMM_DIRECT64};
        const KernelId id4[] = {K_GEMM_W4_DIRECT16, K_GEMM_W4_DIRECT32, K_GEMM_W4_DIRECT64, K_GEMM_W4_DIRECT128};
        const int at = nr == 1 ? 0 : nr == 2 ? 1 : nr == 4 ? 2 : 3;
        best = DirectPlan{w4 ? id4[at] : id8[at], nr, groups, (unsigned)grid, us};
    }
    return best;
}

// The int8 GEMM on tiled A: the fastest of all by those models.
struct GemmPlan {
    int tile;           // of kTiledCfgs, -1 for none
    bool persistent;    // 256 x 224
    DirectPlan direct;  // taken when neither
    double us;
};

GemmPlan plan_gemm(const nh_context* ctx, const GemmSize& g, bool persistent_ok) {
    GemmPlan p{-1, false, plan_direct(ctx, g, false), 0};
    p.us = p.direct.us;
    for (int at = 0; at < 4; ++at) {
        const GemmCfg& c = kTiledCfgs[at];
        if (c.lds > ctx->max_shared_per_block) continue;
        const double us = tile_us(ctx, kTileTime[at], c.bm, c.bn, g);
        if (us < p.us) p.tile = at, p.us = us;
    }
    if (persistent_ok) {
        const double us = tile_us(ctx, kP224Time, 256, 224, g);
        if (us < p.us) p.tile = -1, p.persistent = true, p.us = us;
    }
    return p;
}

// What W4A8 takes through the expanded form, without the rows' quantization: a
// pass that reads the INT4 tiles and writes int8 ones, then the int8 product
// (up to 16 rows the GEMV's; `fused`: one row, quantized there).  Fitted to 800
// shapes of 1..2048 rows that were timed all ways (profiles/w4a8_choice.csv).
double w4_expanded_us(const nh_context* ctx, const GemmSize& g, bool fused) {
    const double expand = 2.05 + g.weights * 1.5 / 3.6;
    if ((size_t)g.M <= kTiledActRows) return expand + 4.33 + 0.033 * g.kt + g.weights / 5.6 - (fused ? 1.5 : 0.0);
    return expand + 1.17 * plan_gemm(ctx, g, g.M % 4 == 0 && g.N % 4 == 0 && g.kt % 2 == 0).us;
}

nh_status launch_gemm_direct(nh_context* ctx, const DirectPlan& p, const GemmW8A8Args& g, int w4_zp, float w4_scale,
                             nh_stream stream, nh_error* err) {
    GemmDirectArgs d{g, p.groups, w4_zp, w4_scale, 0};
    d.g.tiles_n = (g.N + 16 * p.nr - 1) / (16 * p.nr);
    return launch(ctx, p.id, p.grid, 256u, kDirectLds, stream, d, err);
}

// G3 launch.  a_tiled: xq holds A in the weights' tiled layout (written by
// the row quantizer with 16 rows per tile), else row-major [M][K].
nh_status launch_gemm(nh_context* ctx, const int8_t* xq, const float* sx, const int8_t* wq, const float* sw,
                      const float* bias, int M, int N, int K, void* out, nh_dtype out_dtype, int relu2,
                      nh_stream stream, nh_error* err, bool a_tiled = false) {
    GemmW8A8Args a{};
    a.xq = xq;
    a.sx = sx;
    a.wq = wq;
    a.sw = sw;
    a.bias = bias;
    a.out = out;
    a.M = M;
    a.N = N;
    a.K = K;
    a.out_dtype = out_dtype;
    a.relu2 = relu2;
    a.kt = (int)tiled_k_tiles(K);
    a.ldo = N;
    // Tile choice.  Tiled A: by time (plan_gemm).  Row-major A: 256x128 unless
    // that leaves most CUs idle, then 128x128.
    const GemmCfg big = a_tiled ? kTiledCfgs[0] : GemmCfg{K_GEMM_W8A8, 256, 128, 1024, gemm_lds_bytes(256, 128, 3)};
    const GemmCfg small = a_tiled ? kTiledCfgs[1] : GemmCfg{K_GEMM_W8A8_128, 128, 128, 256, gemm_lds_bytes(128, 128, 3)};
    auto tiles = [&](const GemmCfg& c) { return gemm_tiles(c, M, N); };
    const GemmCfg* cfg = nullptr;
    if (a_tiled) {
        const GemmPlan p = plan_gemm(ctx, gemm_size(M, N, a.kt, out_dtype),
                                     persistent_224_ok(ctx, xq, sx, sw, bias, M, N, a.kt, out, out_dtype));
        if (p.persistent) {
            a.tiles_m = (M + 255) / 256;
            a.tiles_n = (N + 223) / 224;
            const int64_t n_tiles = (int64_t)a.tiles_m * a.tiles_n;
            const unsigned grid = (unsigned)std::min<int64_t>(n_tiles, ctx->cu_count);
            return launch(ctx, K_GEMM_P224, grid, 512u, kP224Lds, stream, a, err);
        }
        if (p.us >= kNoPlan) return set_error(err, NH_UNSUPPORTED, "LDS too small for the GEMM tiles");
        if (p.tile < 0) return launch_gemm_direct(ctx, p.direct, a, 0, 0.0f, stream, err);
        cfg = &kTiledCfgs[p.tile];
    } else if (tiles(big) >= ctx->cu_count / 4 && big.lds <= ctx->max_shared_per_block) {
        cfg = &big;
    } else if (small.lds <= ctx->max_shared_per_block) {
        cfg = &small;
    }
    if (!cfg) {
        // LDS too small for the MFMA tiles: 16-row GEMV passes (still exact)
        for (int m0 = 0; m0 < M; m0 += 16) {
            const int mm = std::min(16, M - m0);
            void* o = (char*)out + (size_t)m0 * N * (out_dtype == NH_BF16 ? 2 : 4);
            nh_status st = launch_gemv(ctx, xq + (size_t)m0 * K, sx + m0, wq, sw, bias, mm, N, K, o, out_dtype,
                                       false, stream, err, relu2);
            if (st) return st;
        }
        return NH_OK;
    }
    a.tiles_m = (M + cfg->bm - 1) / cfg->bm;
    a.tiles_n = (N + cfg->bn - 1) / cfg->bn;
    // Every workgroup runs in one of ceil(tiles / CUs) rounds.  When the last
    // round of 256x128 tiles would be at most half full, the columns of the
    // whole rounds take the big tiles and the rest takes 128x128 tiles (half
    // the work each, twice as many): 2048 x 21504 x 4096 is 5 rounds + about
    // half a round instead of 6.
    const int64_t cu = ctx->cu_count;
    const int64_t nbig = (int64_t)a.tiles_m * a.tiles_n;
    if (cfg->id == big.id && small.lds <= ctx->max_shared_per_block && nbig > cu && nbig % cu != 0 &&
        nbig % cu <= cu / 2) {
        const int tn_main = (int)(nbig / cu * cu / a.tiles_m);  // N tiles of whole rounds
        const int n_main = tn_main * big.bn;
        if (tn_main > 0 && n_main < N) {
            GemmW8A8Args r = a;
            a.N = n_main;
            a.tiles_n = tn_main;
            nh_status st =
                launch(ctx, big.id, (unsigned)(a.tiles_m * a.tiles_n), (unsigned)big.threads, big.lds, stream, a, err);
            if (st) return st;
            // columns n_main .. N: weights, scales, bias and outputs from there, rows still N apart
            const size_t esz = out_dtype == NH_BF16 ? 2 : 4;
            r.wq = wq + (size_t)(n_main / 16) * (size_t)r.kt * 1024;
            r.sw = sw + n_main;
            r.bias = bias ? bias + n_main : nullptr;
            r.out = (char*)out + (size_t)n_main * esz;
            r.N = N - n_main;
            r.tiles_m = (M + small.bm - 1) / small.bm;
            r.tiles_n = (r.N + small.bn - 1) / small.bn;
            return launch(ctx, small.id, (unsigned)(r.tiles_m * r.tiles_n), (unsigned)small.threads, small.lds, stream,
                          r, err);
        }
    }
    return launch(ctx, cfg->id, (unsigned)(a.tiles_m * a.tiles_n), (unsigned)cfg->threads, cfg->lds, stream, a, err);
}

}  // namespace

extern "C" {

int nh_supports_gemm_w8a8(size_t m, size_t n, size_t k) {
    // k <= 2^17 keeps the int32 accumulator exact: |acc| <= k * 127 * 127 < 2^31.
    // The kernels address the activations and each weight panel through
    // 32-bit buffer offsets: m * k < 2^31 (plus a tile's overshoot of at most
    // 255 rows) and the tiled weights below 2^40 bytes.
    return m > 0 && n > 0 && k > 0 && m < (1u << 31) && n < (1u << 31) && k <= (1u << 17) && (k % 16) == 0 &&
           (uint64_t)m * k < (1ull << 31) && (uint64_t)n * k < (1ull << 40);
}

nh_status nh_quantize_rows_i8(nh_context* ctx, const void* x, nh_dtype dtype, size_t rows, size_t cols, int8_t* q,
                              float* scales, int32_t* row_status, nh_stream stream, nh_error* err) {
    clear_error(err);
    nh_status st = check_dtype(dtype, err);
    if (st) return st;
    if (rows > (size_t)kMaxGrid || cols > (size_t)kMaxGrid)
        return set_error(err, NH_UNSUPPORTED, "rows/cols must be < 2^31");
    if ((st = bind_device(ctx, err))) return st;
    if (rows == 0 || cols == 0) return NH_OK;  // nothing to quantize (empty inputs are valid, quantize.rs:490-501)
    return launch_quantize(ctx, x, dtype, rows, cols, q, scales, row_status, nullptr, stream, err);
}

size_t nh_tiled_weights_bytes(size_t n, size_t k) {
    if (n == 0 || k == 0 || n > (1ull << 40) || k > (1ull << 40)) return 0;
    return (size_t)tiled_bytes(n, k);
}

nh_status nh_tile_weights_i8(nh_context* ctx, const int8_t* wq, size_t n, size_t k, int8_t* tiled, size_t tiled_len,
                             nh_stream stream, nh_error* err) {
    clear_error(err);
    if (n == 0 || k == 0) return set_error(err, NH_INVALID_SHAPE, "invalid weight shape n=%zu k=%zu", n, k);
    if (n >= (1u << 31) || k >= (1u << 31)) return set_error(err, NH_UNSUPPORTED, "n and k must be < 2^31");
    const size_t need = nh_tiled_weights_bytes(n, k);
    if (tiled_len != need) return mismatch(err, "tiled", need, tiled_len);
    if (!aligned16(tiled)) return set_error(err, NH_UNSUPPORTED, "tiled must be 16-byte aligned");
    nh_status st = bind_device(ctx, err);
    if (st) return st;
    TileWeightsArgs a{wq, tiled, (int64_t)n, (int64_t)k, (int64_t)(need / 16), (int)tiled_k_tiles(k), 0};
    return launch(ctx, K_TILE_WEIGHTS, grid_for(a.chunks, 256), 256, 0, stream, a, err);
}

size_t nh_tiled_int4_weights_bytes(size_t n, size_t k) {
    if (n == 0 || k == 0 || n > (1ull << 40) || k > (1ull << 40)) return 0;
    return (size_t)tiled_int4_bytes(n, k);
}

nh_status nh_tile_weights_int4(nh_context* ctx, const uint8_t* packed, size_t packed_len, size_t k, size_t n,
                               uint32_t zero_point, uint8_t* tiled, size_t tiled_len, nh_stream stream, nh_error* err) {
    clear_error(err);
    size_t kn;
    if (k == 0 || n == 0 || !mul_ok(k, n, &kn)) return set_error(err, NH_INVALID_SHAPE, "invalid INT4 weight shape");
    if (packed_len != nh_packed_int4_len(kn)) return mismatch(err, "packed_weights", nh_packed_int4_len(kn), packed_len);
    if (zero_point > 0x0F) return set_error(err, NH_INVALID_PARAMS, "zero_point %u > 15", zero_point);
    if (n >= (1u << 31) || k >= (1u << 31)) return set_error(err, NH_UNSUPPORTED, "n and k must be < 2^31");
    const size_t need = nh_tiled_int4_weights_bytes(n, k);
    if (tiled_len != need) return mismatch(err, "tiled", need, tiled_len);
    if (((uintptr_t)tiled & 7u) != 0) return set_error(err, NH_UNSUPPORTED, "tiled must be 8-byte aligned");
    nh_status st = bind_device(ctx, err);
    if (st) return st;
    TileInt4Args a{packed, tiled, (int64_t)n, (int64_t)k, (int64_t)(need / 8), (int)tiled_k_tiles(k), (int)zero_point};
    return launch(ctx, K_TILE_INT4, grid_for(a.lanes, 256), 256, 0, stream, a, err);
}

int nh_supports_linear_w4a8(size_t m, size_t n, size_t k) {
    // the fused decode unit: bf16 rows, K tiles of one slab per wave (k <= 8192), whole 16-byte chunks
    return m > 0 && m <= 16 && n > 0 && n < (1u << 31) && k > 0 && k <= 8192 && (k % 16) == 0;
}

size_t nh_linear_w4a8_workspace_size(size_t m, size_t n, size_t k) {
    if (m == 0 || n == 0 || k == 0 || m > (1ull << 31) || n > (1ull << 31) || k > (1ull << 31)) return 0;
    return align256((size_t)tiled_bytes(n, k)) + align256(n * sizeof(float)) + nh_linear_w8a8_workspace_size(m, k);
}

}  // extern "C"

namespace {
nh_status linear_w8a8(nh_context* ctx, const void* x, nh_dtype x_dtype, const int8_t* wq, const float* sw,
                      const float* bias, size_t m, size_t n, size_t k, void* out, nh_dtype out_dtype,
                      void* workspace, size_t workspace_bytes, int8_t* xq_out, float* sx_out, int relu2,
                      uint64_t* nonfinite, int nonfinite_stage, nh_stream stream, nh_error* err,
                      uint32_t* row_max = nullptr);
}  // namespace

namespace {

// nh_linear_w4a8 on the INT4 tiles themselves: the rows' codes as A tiles in the
// workspace, where the expanded weights would go (in the linear part of it
// when there are more row tiles than column tiles; that part holds A tiles
// then, as 16 rows or fewer are one row tile), then the register-direct GEMM.
nh_status linear_w4a8_direct(nh_context* ctx, const DirectPlan& p, const void* x, nh_dtype x_dtype,
                             const uint8_t* w4_tiled, float scale, uint32_t zero_point, const float* bias, size_t m,
                             size_t n, size_t k, void* out, nh_dtype out_dtype, void* workspace, uint64_t* nonfinite,
                             nh_stream stream, nh_error* err) {
    char* lin = (char*)workspace + align256((size_t)tiled_bytes(n, k)) + align256(n * sizeof(float));
    const size_t codes = (size_t)tiled_bytes(m, k);
    const bool in_w8 = codes <= (size_t)tiled_bytes(n, k);
    int8_t* atiles = (int8_t*)(in_w8 ? workspace : lin);
    float* sx = (float*)(in_w8 ? lin : lin + align256(codes));
    nh_status st = launch_quantize(ctx, x, x_dtype, m, k, nullptr, sx, nullptr, atiles, stream, err, 16, nullptr, 1,
                                   nonfinite, kStageInput);
    if (st) return st;
    GemmW8A8Args g{atiles, sx, (const int8_t*)w4_tiled, nullptr, bias, out, (int)m, (int)n, (int)k, 0, 0,
                   out_dtype, 0, (int)tiled_k_tiles(k), (int)n, 0};
    return launch_gemm_direct(ctx, p, g, (int)zero_point, scale, stream, err);
}

}  // namespace

extern "C" {

nh_status nh_linear_w4a8(nh_context* ctx, const void* x, nh_dtype x_dtype, const uint8_t* w4_tiled, float scale,
                         uint32_t zero_point, const float* bias, size_t m, size_t n, size_t k, void* out,
                         nh_dtype out_dtype, void* workspace, size_t workspace_bytes, uint64_t* nonfinite,
                         nh_stream stream, nh_error* err) {
    clear_error(err);
    nh_status st;
    // the checks of Int4LinearWeights::validate and project_into (linear.rs:113-124, 290-311)
    if (k == 0 || n == 0) return set_error(err, NH_INVALID_SHAPE, "invalid linear shape k=%zu n=%zu", k, n);
    if (!std::isfinite(scale) || scale <= 0.0f || zero_point > 0x0F)
        return set_error(err, NH_INVALID_PARAMS, "invalid INT4 params scale=%g zero_point=%u", (double)scale,
                         zero_point);
    if (m == 0) return set_error(err, NH_INVALID_ROW_COUNT, "row_count must be non-zero, got 0");
    if ((st = check_dtype(x_dtype, err)) || (st = check_dtype(out_dtype, err))) return st;
    if (((uintptr_t)w4_tiled & 7u) != 0) return set_error(err, NH_UNSUPPORTED, "w4_tiled must be 8-byte aligned");
    if (x_dtype != NH_BF16 || !nh_supports_linear_w4a8(m, n, k) || !aligned16(x)) {
        // any other shape, f32 or unaligned rows: the register-direct GEMM on the
        // INT4 tiles, or the weights expanded into int8 tiles of code - zp (the
        // layer's definition) and the W8A8 linear path on them, by their times
        if ((st = check_w8a8_shape(m, n, k, err))) return st;
        const size_t need = nh_linear_w4a8_workspace_size(m, n, k);
        if (!workspace || workspace_bytes < need) return mismatch(err, "workspace", need, workspace_bytes);
        if (!aligned16(workspace)) return set_error(err, NH_UNSUPPORTED, "workspace must be 16-byte aligned");
        if ((st = bind_device(ctx, err))) return st;
        int8_t* w8 = (int8_t*)workspace;
        float* sw = (float*)(w8 + align256((size_t)tiled_bytes(n, k)));
        void* lin = (char*)sw + align256(n * sizeof(float));
        const size_t lin_bytes = workspace_bytes - (size_t)((char*)lin - (char*)workspace);
        const GemmSize g = gemm_size((int)m, (int)n, (int)tiled_k_tiles(k), out_dtype);
        const DirectPlan p = plan_direct(ctx, g, true);
        if (p.us < w4_expanded_us(ctx, g, long_row_ok(ctx, x, x_dtype, m, n, k, out, out_dtype, nullptr, nullptr)))
            return linear_w4a8_direct(ctx, p, x, x_dtype, w4_tiled, scale, zero_point, bias, m, n, k, out, out_dtype,
                                      workspace, nonfinite, stream, err);
        ExpandInt4Args e{w4_tiled, w8, sw, (int64_t)(tiled_int4_bytes(n, k) / 8), (int64_t)n, scale,
                         (int32_t)zero_point};
        if ((st = launch(ctx, K_EXPAND_INT4, grid_for(e.lanes, 256), 256, 0, stream, e, err))) return st;
        return linear_w8a8(ctx, x, x_dtype, w8, sw, bias, m, n, k, out, out_dtype, lin, lin_bytes, nullptr, nullptr,
                           0, nonfinite, 0, stream, err);
    }
    if ((st = bind_device(ctx, err))) return st;
    const int kt = (int)tiled_k_tiles(k), w = gemv_waves(kt);
    const size_t esz = out_dtype == NH_BF16 ? 2 : 4;
    DecodePlan plan;
    unsigned grid = 0;
    if (plan_stream(ctx, m, n, k, &plan, &grid)) {
        // 3..16 rows: the streaming unit, the INT4 weights streamed once
        LinearDecodeArgs a{};
        a.x = x;
        a.wq = (const int8_t*)w4_tiled;
        a.bias = bias;
        a.out = out;
        a.M = (int)m;
        a.N = (int)n;
        a.K = (int)k;
        a.kt = kt;
        a.waves = 16;
        a.x_dtype = x_dtype;
        a.out_dtype = out_dtype;
        a.w4_zp = (int)zero_point;
        a.w4_scale = scale;
        a.nonfinite = nonfinite;
        const KernelId kid = m <= 4 ? K_LINEAR_DECODE_STREAM_W4_M4
                             : m <= 8 ? K_LINEAR_DECODE_STREAM_W4_M8
                                      : K_LINEAR_DECODE_STREAM_W4_M16;
        return launch(ctx, kid, grid, 1024u, plan.lds, stream, a, err);
    }
    // otherwise launches over groups of rows, each streaming the weights once:
    // all of up to 16 rows of K <= 4096, up to 8 past that, and small groups by the
    // one-tile units (plan_stream_w4_any).  No workspace: a call may share its buffer with others.
    for (size_t r0 = 0, rows; r0 < m; r0 += rows) {
        rows = std::min<size_t>(k <= 4096 ? 16 : 8, m - r0);
        const bool wide = plan_stream_w4_any(ctx, rows, n, k, &plan, &grid);
        if (!wide) rows = std::min<size_t>(4, rows);
        const size_t mm = rows == 1 ? 1 : rows <= 2 ? 2 : 4;
        const KernelId kid = mm == 1 ? K_LINEAR_DECODE_W4_M1 : mm == 2 ? K_LINEAR_DECODE_W4_ROW2 : K_LINEAR_DECODE_W4_ROW4;
        LinearDecodeArgs a{};
        a.x = (const uint16_t*)x + r0 * k;
        a.wq = (const int8_t*)w4_tiled;
        a.bias = bias;
        a.out = (char*)out + r0 * n * esz;
        a.M = (int)rows;
        a.N = (int)n;
        a.K = (int)k;
        a.kt = kt;
        a.waves = w;
        a.x_dtype = x_dtype;
        a.out_dtype = out_dtype;
        a.ntw = 1;
        a.w4_zp = (int)zero_point;
        a.w4_scale = scale;
        a.row0 = (int)r0;  // the group's first row: non-finite inputs are indexed in the whole x
        a.nonfinite = nonfinite;
        if (wide) {
            a.waves = 16;
            if ((st = launch(ctx, plan.kid, grid, 1024u, plan.lds, stream, a, err))) return st;
            continue;
        }
        const size_t lds = mm * ((size_t)w * 1024 + 16);
        if (lds > ctx->max_shared_per_block) return set_error(err, NH_UNSUPPORTED, "LDS too small");
        if ((st = launch(ctx, kid, (unsigned)((n + 15) / 16), (unsigned)(64 * w), lds, stream, a, err))) return st;
    }
    return NH_OK;
}

nh_status nh_dequantize_i8(nh_context* ctx, const int8_t* q, const float* scales, size_t rows, size_t cols,
                           float* out, nh_stream stream, nh_error* err) {
    clear_error(err);
    size_t total;
    if (!mul_ok(rows, cols, &total)) return set_error(err, NH_INVALID_SHAPE, "rows*cols overflows");
    nh_status st = bind_device(ctx, err);
    if (st) return st;
    if (total == 0) return NH_OK;
    DequantizeI8Args a{q, scales, out, (int64_t)rows, (int64_t)cols};
    // the kernel's 4-code chunks when the layout allows them (the same test)
    const bool vec = cols % 4 == 0 && ((uintptr_t)q & 3) == 0 && aligned16(out);
    return launch(ctx, K_DEQUANT_I8, grid_for((int64_t)(vec ? total / 4 : total), 256), 256, 0, stream, a, err);
}

nh_status nh_dequantize_int4(nh_context* ctx, const uint8_t* packed, size_t packed_len, size_t value_count,
                             float scale, uint32_t zero_point, float* out, size_t out_len, nh_stream stream,
                             nh_error* err) {
    clear_error(err);
    // same validation order as dequantize_int4_into_host (quantize.rs:156-178)
    if (!std::isfinite(scale) || scale <= 0.0f || zero_point > 0x0F)
        return set_error(err, NH_INVALID_PARAMS, "invalid INT4 params scale=%g zero_point=%u", (double)scale,
                         zero_point);
    if (out_len != value_count) return mismatch(err, "output", value_count, out_len);
    if (packed_len != nh_packed_int4_len(value_count))
        return mismatch(err, "packed", nh_packed_int4_len(value_count), packed_len);
    nh_status st = bind_device(ctx, err);
    if (st) return st;
    if (value_count == 0) return NH_OK;
    DequantizeInt4Args a{packed, out, (int64_t)value_count, scale, (float)zero_point};
    // the kernel's 4-code chunks when the layout allows them (the same test)
    const bool vec = value_count >= 4 && ((uintptr_t)packed & 1) == 0 && aligned16(out);
    return launch(ctx, K_DEQUANT_INT4, grid_for((int64_t)(vec ? value_count / 4 : value_count), 256), 256, 0,
                  stream, a, err);
}

int nh_supports_gemm_f32(size_t m, size_t k, size_t n) {
    // i32 shape bounds of the reference's device GEMM (gemm.rs:247-254), any
    // alignment; the grid holds ceil(m / 64) <= 65535 row tiles
    return m > 0 && k > 0 && n > 0 && m <= INT32_MAX && k <= INT32_MAX && n <= INT32_MAX && (m + 63) / 64 <= 65535;
}

// The exact f32 product's two kernels: 64 x 64 outputs per workgroup (16 per
// lane, f64 FMAs) while those tiles fill every CU, else 16 x 16 outputs per
// workgroup on the f64 matrix cores (v_mfma_f64_4x4x4f64 chains), so a narrow
// output such as the MoE router's 128 experts still spreads its k-ordered
// chains over the chip (512 x 2688 x 128: 19.4 us against 52.3 us for one
// output per lane on f64 FMAs; 2048 x 4096 x 128: 82 against 180 us;
// 512 x 4096 x 4096 stays on the 64 x 64 tiles: 531 us against 628 on the
// matrix cores).
static nh_status launch_gemm_f32(nh_context* ctx, const GemmF32Args& a, nh_stream stream, nh_error* err) {
    const int64_t big = ((a.M + 63) / 64) * ((a.N + 63) / 64);
    if (big >= ctx->cu_count)
        return launch(ctx, K_GEMM_F32, (unsigned)((a.N + 63) / 64), 256, 0, stream, a, err,
                      (unsigned)((a.M + 63) / 64));
    // fewer than cu_count 64 x 64 tiles: at most 16 x cu_count 16 x 16 tiles;
    // its buffer loads take 32-bit byte offsets into either operand
    const uint64_t lhs_bytes = (uint64_t)a.M * (uint64_t)a.K * (a.lhs_bf16 ? 2u : 4u);
    const uint64_t rhs_bytes = (uint64_t)a.K * (uint64_t)a.N * 4u;
    if (lhs_bytes >= 0x7ffffff0u || rhs_bytes >= 0x7ffffff0u)  // the kernels' out-of-range offset
        return launch(ctx, K_GEMM_F32, (unsigned)((a.N + 63) / 64), 256, 0, stream, a, err,
                      (unsigned)((a.M + 63) / 64));
    const bool vec = aligned16(a.lhs) && a.K % (a.lhs_bf16 ? 8 : 4) == 0;
    const bool brief = a.K <= kGemmF32Short;
    const KernelId id = !vec         ? brief ? K_GEMM_F32_MFMA_SHORT_ANY : K_GEMM_F32_MFMA_ANY
                        : a.lhs_bf16 ? brief ? K_GEMM_F32_MFMA_SHORT_BF16 : K_GEMM_F32_MFMA_BF16
                        : brief      ? K_GEMM_F32_MFMA_SHORT
                                     : K_GEMM_F32_MFMA;
    return launch(ctx, id, (unsigned)(((a.M + 15) / 16) * ((a.N + 15) / 16)), 512, (brief ? 2 : 3) * kGemmF32MfmaBuffer,
                  stream, a, err);
}

nh_status nh_gemm_f32(nh_context* ctx, const float* lhs, size_t lhs_len, const float* rhs, size_t rhs_len, size_t m,
                      size_t k, size_t n, float* out, size_t out_len, nh_stream stream, nh_error* err) {
    clear_error(err);
    // the validation of gemm_into (gemm.rs:341-363): shape, operand lengths, output length
    size_t ll, rl, ol;
    if (m == 0 || k == 0 || n == 0 || !mul_ok(m, k, &ll) || !mul_ok(k, n, &rl) || !mul_ok(m, n, &ol))
        return set_error(err, NH_INVALID_SHAPE, "invalid GEMM shape m=%zu k=%zu n=%zu", m, k, n);
    if (lhs_len != ll) return mismatch(err, "lhs", ll, lhs_len);
    if (rhs_len != rl) return mismatch(err, "rhs", rl, rhs_len);
    if (out_len != ol) return mismatch(err, "output", ol, out_len);
    if (!nh_supports_gemm_f32(m, k, n))
        return set_error(err, NH_UNSUPPORTED, "shape m=%zu k=%zu n=%zu outside the device envelope", m, k, n);
    if (!aligned16(out)) return set_error(err, NH_UNSUPPORTED, "out must be 16-byte aligned");
    nh_status st = bind_device(ctx, err);
    if (st) return st;
    GemmF32Args a{lhs, rhs, out, (int64_t)m, (int64_t)k, (int64_t)n, nullptr, 0, 0};
    return launch_gemm_f32(ctx, a, stream, err);
}

nh_status nh_gemm_w8a8(nh_context* ctx, const int8_t* xq, const float* sx, const int8_t* wq, const float* sw,
                       const float* bias, size_t m, size_t n, size_t k, void* out, nh_dtype out_dtype,
                       nh_stream stream, nh_error* err) {
    clear_error(err);
    nh_status st;
    if ((st = check_dtype(out_dtype, err)) || (st = check_w8a8_shape(m, n, k, err))) return st;
    if (!aligned16(xq) || !aligned16(wq))
        return set_error(err, NH_UNSUPPORTED, "xq and wq must be 16-byte aligned");
    if ((st = bind_device(ctx, err))) return st;
    if (m <= 16)
        return launch_gemv(ctx, xq, sx, wq, sw, bias, (int)m, (int)n, (int)k, out, out_dtype, false, stream, err);
    return launch_gemm(ctx, xq, sx, wq, sw, bias, (int)m, (int)n, (int)k, out, out_dtype, 0, stream, err);
}

nh_status nh_gemm_w8a8_ta(nh_context* ctx, const int8_t* xq_tiled, const float* sx, const int8_t* wq, const float* sw,
                          const float* bias, size_t m, size_t n, size_t k, void* out, nh_dtype out_dtype,
                          nh_stream stream, nh_error* err) {
    clear_error(err);
    nh_status st;
    if ((st = check_dtype(out_dtype, err)) || (st = check_w8a8_shape(m, n, k, err))) return st;
    if (!aligned16(xq_tiled) || !aligned16(wq))
        return set_error(err, NH_UNSUPPORTED, "xq_tiled and wq must be 16-byte aligned");
    if ((st = bind_device(ctx, err))) return st;
    return launch_gemm(ctx, xq_tiled, sx, wq, sw, bias, (int)m, (int)n, (int)k, out, out_dtype, 0, stream, err, true);
}

size_t nh_linear_w8a8_workspace_size(size_t m, size_t k) {
    if (m == 0 || k == 0 || m > (1ull << 31) || k > (1ull << 31)) return 0;
    if (m <= kTiledActRows) return align256(act_tiles_bytes(m, k)) + align256(m * sizeof(float));
    return align256(tiled_bytes(m, k)) + align256(m * sizeof(float));
}

}  // extern "C"

namespace {

// nh_linear_w8a8 with an optional ReLU^2 after the bias (the MLP's up
// projection, mlp.rs:205), validated by the caller up to the device binding.
nh_status linear_w8a8(nh_context* ctx, const void* x, nh_dtype x_dtype, const int8_t* wq, const float* sw,
                      const float* bias, size_t m, size_t n, size_t k, void* out, nh_dtype out_dtype,
                      void* workspace, size_t workspace_bytes, int8_t* xq_out, float* sx_out, int relu2,
                      uint64_t* nonfinite, int nonfinite_stage, nh_stream stream, nh_error* err,
                      uint32_t* row_max) {
    nh_status st;
    // bf16 rows: the fused decode unit when it fits (one launch, no workspace)
    DecodePlan plan;
    unsigned grid = 0;
    const bool streaming = plan_stream(ctx, m, n, k, &plan, &grid);
    if (x_dtype == NH_BF16 && aligned16(x) && ((uintptr_t)xq_out & 7u) == 0 &&
        (streaming || plan_decode(ctx, m, n, k, &plan))) {
        LinearDecodeArgs a{};
        a.x = x;
        a.wq = wq;
        a.sw = sw;
        a.bias = bias;
        a.out = out;
        a.xq_out = xq_out;
        a.sx_out = sx_out;
        a.M = (int)m;
        a.N = (int)n;
        a.K = (int)k;
        a.kt = (int)tiled_k_tiles(k);
        a.waves = gemv_waves(a.kt);
        a.x_dtype = x_dtype;
        a.out_dtype = out_dtype;
        a.ntw = plan.ntw;
        a.relu2 = relu2;
        a.nonfinite = nonfinite;  // the fused unit reads the caller's input only (stage 0)
        a.row_max = streaming ? row_max : nullptr;
        const size_t tiles = (n + 15) / 16;
        if (!streaming) grid = (unsigned)((tiles + plan.ntw - 1) / plan.ntw);
        return launch(ctx, plan.kid, grid, (unsigned)plan.threads, plan.lds, stream, a, err);
    }
    const size_t need = nh_linear_w8a8_workspace_size(m, k);
    if (m <= kTiledActRows) {
        // Q2 into activation tiles (and the caller's row-major xq_out), then
        // the GEMV reads each K tile's codes as M * 64 contiguous bytes
        if (!workspace || workspace_bytes < need) return mismatch(err, "workspace", need, workspace_bytes);
        if (!aligned16(workspace)) return set_error(err, NH_UNSUPPORTED, "workspace must be 16-byte aligned");
        int8_t* tiles = (int8_t*)workspace;
        float* sx = sx_out ? sx_out : (float*)((char*)workspace + align256(act_tiles_bytes(m, k)));
        // The quantizer's workgroups hand the rows to the GEMV's inside one
        // launch where that saves more than its wait costs.  Long rows with every
        // workgroup on a CU of its own (8 x 6144 -> 2048 9.8 us against 10.4 in
        // two launches, 8 x 7680 -> 355 8.9 / 10.7; but 5 x 2688 -> 4096 11.4 / 8.9);
        // or, for up to 8 rows on up to 1.5 CUs' worth of workgroups, so many
        // weights (126 K tiles per CU, 33 MB) that the rows are through before the
        // first slab is: 8 x 8192 -> 4096 13.4 / 13.8, 7168 -> 5120 16.0 / 16.3, 8192
        // -> 5120 17.1 / 17.8, 7680 -> 6144 17.5 / 17.8; but 7680 -> 4096 13.6 / 13.2,
        // 5120 -> 4096 12.8 / 10.4, 5 x 6144 -> 6144 15.5 / 14.9.
        const size_t tiles_n = (n + 15) / 16, cu = (size_t)ctx->cu_count, ktiles = (size_t)tiled_k_tiles(k);
        const bool handoff = (ktiles >= 64 && tiles_n + m <= cu) ||
                             (ktiles >= 108 && tiles_n * ktiles >= 126 * cu && 2 * tiles_n <= 3 * cu && m <= 8);
        if (handoff && x_dtype == NH_BF16 && aligned16(x) && k <= 8192 && ((uintptr_t)xq_out & 7u) == 0) {
            LinearHandoffArgs h{};
            h.q = QuantizeRowsArgs{x, xq_out, sx, nullptr, tiles, (int64_t)m, (int64_t)k, x_dtype, 1, (int)m, 1,
                                   nullptr, nonfinite, nonfinite_stage, 0};
            GemvW8A8Args& g = h.g;
            g.xq = tiles;
            g.sx = sx;
            g.wq = wq;
            g.sw = sw;
            g.bias = bias;
            g.out = out;
            g.M = (int)m;
            g.N = (int)n;
            g.K = (int)k;
            g.kt = (int)tiled_k_tiles(k);
            g.waves = gemv_waves(g.kt);
            g.out_dtype = out_dtype;
            g.x_tiled = 1;
            g.relu2 = relu2;
            h.consumers = (int)((n + 15) / 16);
            h.slot = ctx->handoff + (size_t)(ctx->handoff_next.fetch_add(1) % kHandoffSlots) * 16;
            return launch(ctx, K_LINEAR_HANDOFF, (unsigned)(m + h.consumers), 64u * (g.waves + 1), 0, stream, h, err);
        }
        if (long_row_ok(ctx, x, x_dtype, m, n, k, out, out_dtype, xq_out, sx_out)) {
            // one f32 or long row: quantized in the GEMV's workgroups
            LinearDecodeArgs a{};
            a.x = x;
            a.wq = wq;
            a.sw = sw;
            a.bias = bias;
            a.out = out;
            a.xq_out = xq_out;
            a.sx_out = sx_out;
            a.M = 1;
            a.N = (int)n;
            a.K = (int)k;
            a.kt = (int)tiled_k_tiles(k);
            a.x_dtype = x_dtype;
            a.out_dtype = out_dtype;
            a.relu2 = relu2;
            a.nonfinite = nonfinite;
            a.nonfinite_stage = nonfinite_stage;
            return launch(ctx, K_LINEAR_DECODE_LONG, (unsigned)((n + 15) / 16), kLongThreads, (size_t)a.kt * 64, stream,
                          a, err);
        }
        if ((st = launch_quantize(ctx, x, x_dtype, m, k, xq_out, sx, nullptr, tiles, stream, err, 0, nullptr, 1,
                                  nonfinite, nonfinite_stage)))
            return st;
        return launch_gemv(ctx, tiles, sx, wq, sw, bias, (int)m, (int)n, (int)k, out, out_dtype, true, stream, err,
                           relu2);
    }
    // two launches: Q2 into A tiles in the workspace (and the caller's
    // row-major xq_out), then G3 on the tiled A
    if (!workspace || workspace_bytes < need) return mismatch(err, "workspace", need, workspace_bytes);
    if (!aligned16(workspace)) return set_error(err, NH_UNSUPPORTED, "workspace must be 16-byte aligned");
    int8_t* atiles = (int8_t*)workspace;
    float* sx = sx_out ? sx_out : (float*)((char*)workspace + align256(tiled_bytes(m, k)));
    if ((st = launch_quantize(ctx, x, x_dtype, m, k, xq_out, sx, nullptr, atiles, stream, err, 16, nullptr, 1,
                              nonfinite, nonfinite_stage)))
        return st;
    return launch_gemm(ctx, atiles, sx, wq, sw, bias, (int)m, (int)n, (int)k, out, out_dtype, relu2, stream, err,
                       true);
}

}  // namespace

extern "C" {

nh_status nh_linear_w8a8(nh_context* ctx, const void* x, nh_dtype x_dtype, const int8_t* wq, const float* sw,
                         const float* bias, size_t m, size_t n, size_t k, void* out, nh_dtype out_dtype,
                         void* workspace, size_t workspace_bytes, int8_t* xq_out, float* sx_out, uint64_t* nonfinite,
                         nh_stream stream, nh_error* err) {
    clear_error(err);
    if (m == 0) return set_error(err, NH_INVALID_ROW_COUNT, "row_count must be non-zero, got 0");
    nh_status st;
    if ((st = check_dtype(x_dtype, err)) || (st = check_dtype(out_dtype, err)) ||
        (st = check_w8a8_shape(m, n, k, err)))
        return st;
    if (!aligned16(wq)) return set_error(err, NH_UNSUPPORTED, "wq must be 16-byte aligned");
    if ((st = bind_device(ctx, err))) return st;
    return linear_w8a8(ctx, x, x_dtype, wq, sw, bias, m, n, k, out, out_dtype, workspace, workspace_bytes, xq_out,
                       sx_out, 0, nonfinite, 0, stream, err);
}

// The MLP's workspace: the f32 intermediate h, the up projection's
// per-workgroup row maxima of h (streaming unit: at most kMaxStreamGroups
// workgroups x 8 rows), then the linear workspace of either projection.
constexpr size_t kMaxStreamGroups = 1024;

size_t nh_mlp_w8a8_workspace_size(size_t m, size_t hidden, size_t inter) {
    if (m == 0 || hidden == 0 || inter == 0 || m > (1ull << 31) || inter > (1ull << 31)) return 0;
    const size_t a = nh_linear_w8a8_workspace_size(m, hidden), b = nh_linear_w8a8_workspace_size(m, inter);
    return align256(m * inter * sizeof(float)) + align256(kMaxStreamGroups * 8 * sizeof(uint32_t)) + (a > b ? a : b);
}

}  // extern "C"

// nh_mlp_w8a8, its f32 intermediate reported at NonFiniteStage h_stage (the
// MoE layer's shared expert: kStageSharedIntermediate).
static nh_status mlp_w8a8(nh_context* ctx, const void* x, nh_dtype x_dtype, const int8_t* w_up, const float* s_up,
                          const float* b_up, const int8_t* w_down, const float* s_down, const float* b_down, size_t m,
                          size_t hidden, size_t inter, void* out, nh_dtype out_dtype, void* workspace,
                          size_t workspace_bytes, uint64_t* nonfinite, int h_stage, nh_stream stream, nh_error* err) {
    clear_error(err);
    if (hidden == 0 || inter == 0)
        return set_error(err, NH_INVALID_SHAPE, "mlp shape must be non-zero, got hidden_dim=%zu, intermediate_dim=%zu",
                         hidden, inter);
    if (m == 0) return set_error(err, NH_INVALID_ROW_COUNT, "row_count must be non-zero, got 0");
    nh_status st;
    if ((st = check_dtype(x_dtype, err)) || (st = check_dtype(out_dtype, err)) ||
        (st = check_w8a8_shape(m, inter, hidden, err)) || (st = check_w8a8_shape(m, hidden, inter, err)))
        return st;
    if (!aligned16(w_up) || !aligned16(w_down)) return set_error(err, NH_UNSUPPORTED, "weights must be 16-byte aligned");
    const size_t need = nh_mlp_w8a8_workspace_size(m, hidden, inter);
    if (!workspace || workspace_bytes < need) return mismatch(err, "workspace", need, workspace_bytes);
    if (!aligned16(workspace)) return set_error(err, NH_UNSUPPORTED, "workspace must be 16-byte aligned");
    if ((st = bind_device(ctx, err))) return st;
    // h = ReLU^2(x W_up^T + b_up) in f32 (the reference's intermediate), then
    // out = h W_down^T + b_down with h quantized per row
    float* h = (float*)workspace;
    uint32_t* hmax = (uint32_t*)((char*)workspace + align256(m * inter * sizeof(float)));
    void* lin_ws = (char*)hmax + align256(kMaxStreamGroups * 8 * sizeof(uint32_t));
    const size_t lin_bytes = workspace_bytes - (size_t)((char*)lin_ws - (char*)workspace);
    DecodePlan plan;
    unsigned groups = 0;
    if (x_dtype == NH_BF16 && aligned16(x) && inter % 4 == 0 && plan_stream(ctx, m, inter, hidden, &plan, &groups) &&
        (size_t)groups * m <= kMaxStreamGroups * 8) {
        // 3..16 rows: the streaming unit leaves each workgroup's row maxima of
        // h, so h's quantizer needs no reduction pass over the 4 * inter-byte
        // rows and spreads each row over many workgroups (K = 21504: 8.9 us
        // as one workgroup per row)
        if ((st = linear_w8a8(ctx, x, x_dtype, w_up, s_up, b_up, m, inter, hidden, h, NH_F32, lin_ws, lin_bytes,
                              nullptr, nullptr, 1, nonfinite, kStageInput, stream, err, hmax)))
            return st;
        int8_t* tiles = (int8_t*)lin_ws;
        float* sh = (float*)((char*)lin_ws + align256(act_tiles_bytes(m, inter)));
        QuantizePmaxArgs q{h, hmax, tiles, sh, nonfinite, (int)m, (int)inter, (int)groups, h_stage};
        if ((st = launch(ctx, K_QUANTIZE_ROWS_PMAX, (unsigned)((inter / 4 + 255) / 256), 256, 0, stream, q, err,
                         (unsigned)m)))
            return st;
        return launch_gemv(ctx, tiles, sh, w_down, s_down, b_down, (int)m, (int)hidden, (int)inter, out, out_dtype,
                           true, stream, err);
    }
    if ((st = linear_w8a8(ctx, x, x_dtype, w_up, s_up, b_up, m, inter, hidden, h, NH_F32, lin_ws, lin_bytes, nullptr,
                          nullptr, 1, nonfinite, kStageInput, stream, err)))
        return st;
    // h: the layer's intermediate (h_stage of the non-finite report)
    return linear_w8a8(ctx, h, NH_F32, w_down, s_down, b_down, m, hidden, inter, out, out_dtype, lin_ws, lin_bytes,
                       nullptr, nullptr, 0, nonfinite, h_stage, stream, err);
}

extern "C" {

nh_status nh_mlp_w8a8(nh_context* ctx, const void* x, nh_dtype x_dtype, const int8_t* w_up, const float* s_up,
                      const float* b_up, const int8_t* w_down, const float* s_down, const float* b_down, size_t m,
                      size_t hidden, size_t inter, void* out, nh_dtype out_dtype, void* workspace,
                      size_t workspace_bytes, uint64_t* nonfinite, nh_stream stream, nh_error* err) {
    return mlp_w8a8(ctx, x, x_dtype, w_up, s_up, b_up, w_down, s_down, b_down, m, hidden, inter, out, out_dtype,
                    workspace, workspace_bytes, nonfinite, kStageIntermediate, stream, err);
}

nh_status nh_gemv_w8a32(nh_context* ctx, const float* x, const int8_t* wq, const float* sw, size_t m, size_t n,
                        size_t k, float* y, nh_stream stream, nh_error* err) {
    clear_error(err);
    nh_status st;
    if ((st = check_w8a8_shape(m, n, k, err))) return st;
    if (!aligned16(x) || !aligned16(wq)) return set_error(err, NH_UNSUPPORTED, "x and wq must be 16-byte aligned");
    if ((st = bind_device(ctx, err))) return st;
    if ((m + 3) / 4 > 65535 || n >= (1u << 29))
        return set_error(err, NH_UNSUPPORTED, "device W8A32 GEMV needs m <= 262140 and n < 2^29");
    GemvW8A32Args a{x, wq, sw, y, (int)m, (int)n, (int)k, 0, 0, 0};
    a.kt = (int)tiled_k_tiles(k);
    a.waves = std::max(1, std::min(16, (a.kt + 3) / 4));  // 4 K tiles per wave and slab
    a.slabs = ((a.kt + a.waves - 1) / a.waves + 3) / 4;
    // one activation row per workgroup at m = 1, else 4
    const unsigned rows = m == 1 ? 1u : 4u;
    return launch(ctx, m == 1 ? K_GEMV_W8A32_M1 : K_GEMV_W8A32, (unsigned)((n + 15) / 16), 64u * a.waves, 0, stream,
                  a, err, (unsigned)((m + rows - 1) / rows));
}

// ---- MoE ------------------------------------------------------------------
nh_status nh_moe_route_sigmoid_topk(nh_context* ctx, const float* scores, size_t tokens, size_t experts,
                                    size_t top_k, int renormalize, float scaling, int32_t* indices, float* weights,
                                    nh_stream stream, nh_error* err) {
    clear_error(err);
    if (experts == 0 || top_k == 0 || top_k > experts)  // validate_shape, moe_routing.rs:261-267
        return set_error(err, NH_INVALID_SHAPE, "invalid routing shape tokens=%zu experts=%zu top_k=%zu", tokens,
                         experts, top_k);
    if (experts > 1024 || top_k > 64 || tokens > (size_t)kMaxGrid / 4)
        return set_error(err, NH_UNSUPPORTED, "device routing needs experts <= 1024 and top_k <= 64");
    nh_status st = bind_device(ctx, err);
    if (st) return st;
    if (tokens == 0) return NH_OK;
    RouteArgs a{scores, indices, weights, (int)tokens, (int)experts, (int)top_k, renormalize ? 1 : 0, scaling, 0,
                nullptr, nullptr, nullptr, nullptr, 0, 0, nullptr};
    return launch(ctx, K_ROUTE_SIGMOID, (unsigned)((tokens + 3) / 4), 256, 0, stream, a, err);
}

nh_status nh_moe_permute(nh_context* ctx, const int32_t* indices, size_t tokens, size_t top_k, size_t experts,
                         int32_t* offsets, int32_t* perm, int32_t* pos, nh_stream stream, nh_error* err) {
    clear_error(err);
    if (experts == 0 || top_k == 0) return set_error(err, NH_INVALID_SHAPE, "experts and top_k must be non-zero");
    size_t routes;
    if (!mul_ok(tokens, top_k, &routes) || routes > (size_t)kMaxGrid || experts > 4096)
        return set_error(err, NH_UNSUPPORTED, "device permutation needs routes < 2^31 and experts <= 4096");
    nh_status st = bind_device(ctx, err);
    if (st) return st;
    PermuteArgs a{indices, offsets, perm, pos, (int)routes, (int)experts};
    // one workgroup per expert while their reads of the ids stay small
    // (experts x routes <= 4M: 16 MiB of L2 reads; the 512-token top-6 layer
    // with 128 experts reads 1.5 MiB) and the ids are 16-byte aligned, else
    // the single-workgroup form
    if (experts * routes <= ((size_t)1 << 22) && aligned16(indices))
        return launch(ctx, K_PERMUTE_EXPERT, (unsigned)experts, 256, 0, stream, a, err);
    return launch(ctx, K_PERMUTE, 1, 1024, 2 * experts * sizeof(int), stream, a, err);
}

}  // extern "C"

constexpr int kExpertWaves = 8;

// Experts that evenly spread routes reach.
static double expected_experts(size_t experts, size_t routes) {
    return experts * (1.0 - std::pow(1.0 - 1.0 / (double)experts, (double)routes));
}

// Workgroups per expert: as many as give every CU one when the routes reach as
// many experts as evenly spread ones do, plus three standard deviations (their
// number's variance: E (q - (1 + R / E) q^2), q = e^(-R / E)); at least two, and no
// fewer than 4 N tiles each (8, one per wave, when segments are longer than a
// 16-row block: every part stages the whole segment).  A CU streams one part's
// weights at a time, so a few parts more than CUs cost a second round (8
// tokens over 128 experts top-6, ~40 reached, in 6 parts: 99 us per layer on
// some inputs and 120 on others; in 5 parts 99-102), while HBM is busy with
// 3/4 of the CUs streaming.  The up projection there in 2 / 6 / 11 / 16
// parts: 55.2 / 32.4 / 36.1 / 42.4 us; 16 tokens in 2 / 3 / 6: 61.4 / 53.1 / 57.8.
static int expert_parts(const nh_context* ctx, size_t experts, size_t routes, size_t max_rows, size_t n) {
    const double mean = expected_experts(experts, routes), load = (double)routes / (double)experts;
    const double q = std::exp(-load), var = (double)experts * (q - (1.0 + load) * q * q);
    const double active = std::min((double)experts, mean + 3.0 * std::sqrt(std::max(0.0, var)));
    const int64_t ntiles = (int64_t)((n + 15) / 16), least = max_rows <= 16 ? 4 : 8;
    int64_t parts = (int64_t)(ctx->cu_count / std::max(1.0, active));
    parts = std::min(parts, (ntiles + least - 1) / least);
    parts = std::min<int64_t>(parts, (int64_t)n / 4);  // the row maxima [R][parts] take the place of int8 codes [R][n]
    return (int)std::max<int64_t>(2, parts);
}

// The expert-block kernel (slot-ordered A, kernels/moe.hip) in one of its
// three forms; e carries the operands, this fills the launch shape.  `parts`
// workgroups per expert, each owning a range of its N tiles; a pass stages as
// many 16-row blocks (up to 4, and no more than the longest segment can have:
// max_rows) as the LDS holds next to the pass's row scales, 64 row maxima
// and the workgroup's weight scales: every pass re-streams the expert's
// weights.  NH_UNSUPPORTED when even one block does
// not fit (the caller takes the grouped kernel).
static nh_status launch_expert_gemm(nh_context* ctx, KernelId id, ExpertGemmArgs e, size_t experts, size_t n,
                                    size_t k, size_t routes, size_t max_rows, int parts, nh_stream stream, nh_error* err) {
    const int kt = (int)tiled_k_tiles(k);
    const int ntiles = (int)((n + 15) / 16);
    const int tiles_per_wg = (ntiles + parts - 1) / parts;
    // the weight scales arrive by 64-float direct-to-LDS rows (256 bytes
    // each, also past the workgroup's last column), so their region is a
    // whole number of rows
    // (and as many for the bias, when there is one)
    auto expert_lds = [&](int rb) {
        const size_t sws_floats = ((size_t)tiles_per_wg * 16 + 63) / 64 * 64;
        return (size_t)rb * kt * 1024 + (size_t)rb * 16 * 4 + 64 * 4 + sws_floats * 4 * (e.bias ? 2 : 1);
    };
    int row_blocks = (int)std::min<size_t>(4, (max_rows + 15) / 16);
    while (row_blocks > 1 && expert_lds(row_blocks) > ctx->max_shared_per_block) --row_blocks;
    const size_t lds = expert_lds(row_blocks);
    if (lds > ctx->max_shared_per_block) return set_error(err, NH_UNSUPPORTED, "expert tiles exceed the LDS");
    e.N = (int)n;
    e.K = (int)k;
    e.kt = kt;
    e.parts = parts;
    e.experts = (int)experts;
    e.streams = kExpertWaves;
    e.tiles_per_wg = tiles_per_wg;
    e.row_blocks = row_blocks;
    // Packed onto the experts with routes (a search of 0.2-0.6 us per launch)
    // where slots in natural order would give some CUs two live workgroups
    // and others none: as many slots as CUs and more, a tenth of the experts
    // without routes, and the live ones 0.4 of the CUs' worth or the slots three
    // per CU.  Natural order / packed, us per layer: 256 experts of 624 x 512 with 198
    // routes 55.3 / 41.5, 64 of 2048 x 1024 with 128 (4 slots each) 77.3 / 74.2, 1024
    // of 2048 x 96 with 684 168.2 / 143.2, 128 of 2688 x 1856 with 2 53.4 / 48.3; but
    // 64 of 960 x 1024 with 153 (nine in ten) 45.2 / 46.5, 60 of 336 x 512 with 2
    // 26.1 / 26.7.  On 800 layers of 16 to 1024 experts within 0.3% of the best
    // of both orders on average (packed wherever a tenth has none: 0.5%).
    // Past 1024 experts the search is long, and an empty workgroup leaves as
    // soon: packed up to three rounds (6297 of 416 x 64 with 1979 routes 82 / 145 us a launch,
    // 12302 of 16 x 64 with 1234 56.7 / 134; but 2457 of 16 x 3584 with 114 16.2 / 11.5).
    const double cu = ctx->cu_count, live = expected_experts(experts, routes), all = (double)parts * (double)experts;
    e.compact = all >= cu && live < 0.9 * (double)experts && (parts * live >= 0.4 * cu || all >= 3 * cu) &&
                (experts <= 1024 || parts * live <= 3 * cu);
    const size_t slots = e.compact ? std::min(experts, routes) : experts;
    return launch(ctx, id, (unsigned)parts, (unsigned)(64 * kExpertWaves), lds, stream, e, err, (unsigned)slots);
}

// Whether the MoE layer's two projections run as the fused expert-block
// pair: the envelope of nh_moe_grouped_gemm_w8a8 for both shapes, the f32
// intermediate within 32-bit buffer offsets, and a 16-row block of A tiles
// in the LDS for both (checked before anything is launched).
static bool expert_fused_ok(nh_context* ctx, size_t routes, size_t experts, size_t hidden, size_t inter,
                            const int8_t* w_up, const int8_t* w_down) {
    if (!nh_supports_gemm_w8a8(routes, inter, hidden) || !nh_supports_gemm_w8a8(routes, hidden, inter)) return false;
    if (experts > 65535 || hidden > 8192 || inter > 8192 || routes * inter * 4 >= (1ull << 31) ||
        routes * hidden >= (1ull << 31))
        return false;
    if (!aligned16(w_up) || !aligned16(w_down)) return false;
    // the down kernel stages each 16-row block as 4 K tiles per wave (8
    // waves): inter <= 2048
    if (tiled_k_tiles(inter) > 32) return false;
    auto fits = [&](size_t n, size_t k) {  // one row block, the weight scales and a bias
        const size_t tiles_per_wg = ((n + 15) / 16 + 1) / 2;
        const size_t sws_floats = (tiles_per_wg * 16 + 63) / 64 * 64;
        return tiled_k_tiles(k) * 1024 + 16 * 4 + 64 * 4 + 2 * sws_floats * 4 <= ctx->max_shared_per_block;
    };
    return fits(inter, hidden) && fits(hidden, inter);
}

// nh_moe_grouped_gemm_w8a8 with an optional per-expert bias [E][n], added
// before ReLU^2 (the experts' MlpLayer biases, mlp.rs:201-205).
static nh_status moe_grouped_gemm(nh_context* ctx, const int8_t* aq, const float* sa, int gather, size_t top_k,
                                  const int32_t* offsets, const int32_t* perm, size_t routes, size_t a_rows,
                                  size_t experts, const int8_t* w, const float* sw, const float* bias, size_t n,
                                  size_t k, int relu2, float* out, nh_stream stream, nh_error* err) {
    clear_error(err);
    if (experts == 0 || top_k == 0) return set_error(err, NH_INVALID_SHAPE, "experts and top_k must be non-zero");
    nh_status st;
    if ((st = check_w8a8_shape(routes ? routes : 1, n, k, err))) return st;
    if (!aligned16(aq) || !aligned16(w)) return set_error(err, NH_UNSUPPORTED, "aq and w must be 16-byte aligned");
    if (experts > 65535 || k > 8192 || a_rows * k >= (1ull << 31) || 16 * k >= (1ull << 31))
        return set_error(err, NH_UNSUPPORTED, "grouped GEMM envelope: experts <= 65535, k <= 8192, a_rows * k < 2^31");
    if ((st = bind_device(ctx, err))) return st;
    if (routes == 0) return NH_OK;
    if (!gather) {
        ExpertGemmArgs e{};
        e.aq = aq;
        e.sa = sa;
        e.offsets = offsets;
        e.w = w;
        e.sw = sw;
        e.bias = bias;
        e.out = out;
        e.a_rows = (int)a_rows;
        e.relu2 = relu2 ? 1 : 0;
        st = launch_expert_gemm(ctx, K_EXPERT_GEMM, e, experts, n, k, routes, routes, expert_parts(ctx, experts, routes, routes, n), stream,
                                err);
        if (st != NH_UNSUPPORTED) return st;
        clear_error(err);
    }
    GroupedGemmArgs a{};
    a.aq = aq;
    a.sa = sa;
    a.offsets = offsets;
    a.perm = perm;
    a.w = w;
    a.sw = sw;
    a.bias = bias;
    a.out = out;
    a.experts = (int)experts;
    a.N = (int)n;
    a.K = (int)k;
    a.top_k = (int)top_k;
    a.gather = gather ? 1 : 0;
    a.relu2 = relu2 ? 1 : 0;
    a.ntiles = (int)((n + 15) / 16);
    a.a_rows = (int)a_rows;
    a.kt = (int)tiled_k_tiles(k);
    a.waves = (a.kt + 15) / 16;  // k <= 8192: one 16-tile slab per wave
    return launch(ctx, K_GROUPED_GEMM, (unsigned)a.ntiles, 64u * a.waves, 0, stream, a, err, (unsigned)experts);
}

extern "C" {

nh_status nh_moe_grouped_gemm_w8a8(nh_context* ctx, const int8_t* aq, const float* sa, int gather, size_t top_k,
                                   const int32_t* offsets, const int32_t* perm, size_t routes, size_t a_rows,
                                   size_t experts, const int8_t* w, const float* sw, size_t n, size_t k, int relu2,
                                   float* out, nh_stream stream, nh_error* err) {
    return moe_grouped_gemm(ctx, aq, sa, gather, top_k, offsets, perm, routes, a_rows, experts, w, sw, nullptr, n, k,
                            relu2, out, stream, err);
}

nh_status nh_moe_combine(nh_context* ctx, const float* slot_out, const int32_t* pos, const float* weights,
                         size_t tokens, size_t top_k, size_t hidden, void* out, nh_dtype out_dtype, nh_stream stream,
                         nh_error* err) {
    return nh_moe_combine_shared(ctx, slot_out, pos, weights, nullptr, tokens, top_k, hidden, out, out_dtype, stream,
                                 err);
}

nh_status nh_moe_combine_shared(nh_context* ctx, const float* slot_out, const int32_t* pos, const float* weights,
                                const float* shared, size_t tokens, size_t top_k, size_t hidden, void* out,
                                nh_dtype out_dtype, nh_stream stream, nh_error* err) {
    clear_error(err);
    nh_status st;
    if ((st = check_dtype(out_dtype, err))) return st;
    if (tokens > (size_t)kMaxGrid || hidden > (size_t)kMaxGrid || top_k == 0)
        return set_error(err, NH_INVALID_SHAPE, "invalid combine shape");
    if ((st = bind_device(ctx, err))) return st;
    if (tokens == 0 || hidden == 0) return NH_OK;
    size_t routes;
    if (!mul_ok(tokens, top_k, &routes) || routes > (size_t)kMaxGrid)
        return set_error(err, NH_UNSUPPORTED, "tokens * top_k must be < 2^31");
    CombineArgs a{slot_out, pos, weights, out, shared, (int)tokens, (int)top_k, (int)hidden, out_dtype};
    // four columns per thread when every row starts 16-byte aligned (8 bytes for bf16 out)
    const bool vec4 = hidden % 4 == 0 && aligned16(slot_out) && aligned16(shared) &&
                      ((uintptr_t)out % (out_dtype == NH_BF16 ? 8 : 16)) == 0;
    if (vec4)
        return launch(ctx, K_COMBINE4, (unsigned)((hidden / 4 + 255) / 256), 256, 0, stream, a, err,
                      (unsigned)tokens);
    return launch(ctx, K_COMBINE, (unsigned)((hidden + 255) / 256), 256, 0, stream, a, err, (unsigned)tokens);
}

// Workspace of the fused MoE layer, 256-byte aligned fields.
static void moe_layout(size_t T, size_t H, size_t I, size_t E, size_t k, size_t off[12]) {
    const size_t R = T * k;
    size_t cur = 0;
    auto take = [&](size_t bytes) {
        size_t o = cur;
        cur += ((bytes + 255) / 256) * 256;
        return o;
    };
    off[0] = take(R * 4);        // indices
    off[1] = take(R * 4);        // weights
    off[2] = take((E + 1) * 4);  // offsets
    off[3] = take(R * 4);        // perm
    off[4] = take(R * 4);        // pos
    off[5] = take(R * H);        // xq, one row per route in expert order
    off[6] = take(R * 4);        // sx
    off[7] = take(R * I * 4);    // up output (f32, ReLU^2 applied; column-tile order on the fused path)
    off[8] = take(R * I);        // requantized up output
    off[9] = take(R * 4);        // its scales
    off[10] = take(R * H * 4);   // down output per slot (f32)
    off[11] = cur;               // total
}

size_t nh_moe_forward_w8a8_workspace_size(size_t tokens, size_t hidden, size_t inter, size_t experts,
                                          size_t top_k) {
    size_t off[12];
    moe_layout(tokens, hidden, inter, experts, top_k, off);
    return off[11];
}

void nh_moe_workspace_layout(size_t tokens, size_t hidden, size_t inter, size_t experts, size_t top_k,
                             size_t offsets_out[5]) {
    size_t off[12];
    moe_layout(tokens, hidden, inter, experts, top_k, off);
    for (int i = 0; i < 5; ++i) offsets_out[i] = off[i];
}

// The routed MoE layer, with the shared expert when w_up_sh is not null:
// shared = the int8 MLP of x (nh_mlp_w8a8, f32), added first by the combine.
// biases (optional) are the experts' and the shared expert's MlpLayer biases.
static nh_status moe_forward(nh_context* ctx, const void* x, nh_dtype x_dtype, const float* logits, size_t tokens,
                             size_t hidden, size_t inter, size_t experts, size_t top_k, int renormalize, float scaling,
                             const int8_t* w_up, const float* s_up, const int8_t* w_down, const float* s_down,
                             size_t inter_sh, const int8_t* w_up_sh, const float* s_up_sh, const int8_t* w_down_sh,
                             const float* s_down_sh, const nh_moe_biases* biases, void* out, nh_dtype out_dtype,
                             void* workspace, size_t workspace_bytes, uint64_t* nonfinite, nh_stream stream,
                             nh_error* err) {
    clear_error(err);
    if (tokens == 0) return set_error(err, NH_INVALID_ROW_COUNT, "row_count must be non-zero, got 0");
    if (hidden == 0 || experts == 0 || top_k == 0 || top_k > experts || inter == 0)
        return set_error(err, NH_INVALID_SHAPE, "invalid MoE shape");
    const bool has_shared = w_up_sh != nullptr;
    if (has_shared && (inter_sh == 0 || !s_up_sh || !w_down_sh || !s_down_sh))
        return set_error(err, NH_INVALID_SHAPE, "shared expert needs intermediate_dim > 0 and all four operands");
    const nh_moe_biases nob{nullptr, nullptr, nullptr, nullptr};
    const nh_moe_biases& b = biases ? *biases : nob;
    if (!has_shared && (b.shared_up || b.shared_down))
        return set_error(err, NH_INVALID_PARAMS, "shared expert biases given without a shared expert");
    size_t off[12];
    moe_layout(tokens, hidden, inter, experts, top_k, off);
    const size_t shared_at = off[11];
    const size_t shared_bytes = has_shared ? align256(tokens * hidden * sizeof(float)) : 0;
    const size_t need =
        off[11] + (has_shared ? shared_bytes + nh_mlp_w8a8_workspace_size(tokens, hidden, inter_sh) : 0);
    if (!workspace || workspace_bytes < need) return mismatch(err, "workspace", need, workspace_bytes);
    if (!aligned16(workspace)) return set_error(err, NH_UNSUPPORTED, "workspace must be 16-byte aligned");
    char* ws = (char*)workspace;
    int32_t* idx = (int32_t*)(ws + off[0]);
    float* wts = (float*)(ws + off[1]);
    int32_t* offsets = (int32_t*)(ws + off[2]);
    int32_t* perm = (int32_t*)(ws + off[3]);
    int32_t* pos = (int32_t*)(ws + off[4]);
    int8_t* xq = (int8_t*)(ws + off[5]);
    float* sx = (float*)(ws + off[6]);
    float* h = (float*)(ws + off[7]);
    int8_t* hq = (int8_t*)(ws + off[8]);
    float* sh = (float*)(ws + off[9]);
    float* d = (float*)(ws + off[10]);
    float* shared = has_shared ? (float*)(ws + shared_at) : nullptr;
    const size_t R = tokens * top_k;
    nh_status st;
    if ((st = check_dtype(x_dtype, err))) return st;
    const bool fused = expert_fused_ok(ctx, R, experts, hidden, inter, w_up, w_down);
    const size_t esz = x_dtype == NH_BF16 ? 2 : 4;
    // the routing wave of each token also quantizes its row (token-major)
    // when the row fits the wave quantizer; the up projection then gathers
    const bool route_q = fused && aligned16(x) && (hidden * esz) % 16 == 0 && hidden * esz <= 512 * 16 &&
                         experts <= 1024 && top_k <= 64 && tokens <= (size_t)kMaxGrid / 4;
    // The shared expert (an MLP over every token).  Past the GEMV's 16 rows
    // its up projection is a GEMM on A tiles of the same codes, so the
    // routing kernel writes them too (into the tiles of the MLP's workspace)
    // and the MLP's own quantization of x is skipped (512 tokens: 7.8 us).
    char* mlp_ws = ws + shared_at + shared_bytes;
    const size_t mlp_bytes = has_shared ? workspace_bytes - shared_at - shared_bytes : 0;
    const bool shared_tiles = has_shared && route_q && tokens > kTiledActRows && aligned16(w_up_sh) &&
                              aligned16(w_down_sh) && check_w8a8_shape(tokens, inter_sh, hidden, nullptr) == NH_OK &&
                              check_w8a8_shape(tokens, hidden, inter_sh, nullptr) == NH_OK;
    float* h_sh = (float*)mlp_ws;
    char* lin_sh = mlp_ws + align256(tokens * inter_sh * sizeof(float)) +
                   align256(kMaxStreamGroups * 8 * sizeof(uint32_t));  // nh_mlp_w8a8's layout
    // the shared expert's intermediate is reported ahead of the routed
    // experts' (the reference runs it first, moe.rs:197-219)
    if (has_shared && !shared_tiles &&
        (st = mlp_w8a8(ctx, x, x_dtype, w_up_sh, s_up_sh, b.shared_up, w_down_sh, s_down_sh, b.shared_down, tokens,
                       hidden, inter_sh, shared, NH_F32, mlp_ws, mlp_bytes, nonfinite, kStageSharedIntermediate, stream,
                       err)))
        return st;
    if (route_q) {
        if ((st = bind_device(ctx, err))) return st;
        RouteArgs ra{logits, idx, wts, (int)tokens, (int)experts, (int)top_k, renormalize ? 1 : 0, scaling, 0,
                     x, xq, sx, nonfinite, x_dtype == NH_BF16 ? DT_BF16 : DT_F32, (int)hidden,
                     shared_tiles ? (int8_t*)lin_sh : nullptr};
        // two tokens per workgroup: two waves route, two quantize
        if ((st = launch(ctx, K_ROUTE_SIGMOID, (unsigned)((tokens + 1) / 2), 256, 0, stream, ra, err))) return st;
    } else if ((st = nh_moe_route_sigmoid_topk(ctx, logits, tokens, experts, top_k, renormalize, scaling, idx, wts,
                                               stream, err))) {
        return st;
    }
    if (shared_tiles) {
        // nh_mlp_w8a8's steps from the tiles on: up (ReLU^2, f32 h), then the
        // linear path on h (its quantization: the layer's intermediate)
        if ((st = launch_gemm(ctx, (const int8_t*)lin_sh, sx, w_up_sh, s_up_sh, b.shared_up, (int)tokens,
                              (int)inter_sh, (int)hidden, h_sh, NH_F32, 1, stream, err, true)))
            return st;
        const size_t lin_bytes = mlp_bytes - (size_t)(lin_sh - mlp_ws);
        if ((st = linear_w8a8(ctx, h_sh, NH_F32, w_down_sh, s_down_sh, b.shared_down, tokens, hidden, inter_sh, shared,
                              NH_F32, lin_sh, lin_bytes, nullptr, nullptr, 0, nonfinite, kStageSharedIntermediate,
                              stream, err)))
            return st;
    }
    if ((st = nh_moe_permute(ctx, idx, tokens, top_k, experts, offsets, perm, pos, stream, err))) return st;
    // otherwise Q2 of each route's token, written in expert order (slot s =
    // token perm[s] / top_k): the up projection reads its rows contiguously
    if (!route_q && (st = launch_quantize(ctx, x, x_dtype, R, hidden, xq, sx, nullptr, nullptr, stream, err, 0, perm,
                                          (int)top_k, nonfinite, kStageInput)))
        return st;
    if (fused) {
        // up (+ bias) with ReLU^2, h in f32 plus each row's max finite |h|
        // per workgroup (non-finite h reported at kStageIntermediate: h is
        // the layer's intermediate); the down projection requantizes h per
        // row while it stages it (the codes and scales of
        // nh_quantize_rows_i8 on h), then adds its bias
        const int parts_up = expert_parts(ctx, experts, R, tokens, inter);
        uint32_t* hmax = (uint32_t*)(ws + off[8]);  // [R][parts_up]
        ExpertGemmArgs up{};
        up.aq = xq;
        up.sa = sx;
        if (route_q) {  // token-major codes: slot s reads token perm[s] / top_k
            up.perm = perm;
            up.gather_div = (int)top_k;
        }
        up.offsets = offsets;
        up.w = w_up;
        up.sw = s_up;
        up.bias = b.up;
        up.out = h;
        up.out_tcol = 1;  // h in column-tile order: 270.4-270.8 us per layer against 271.9-272.4 row-major
        up.out_rows = (int)R;
        up.a_rows = route_q ? (int)tokens : (int)R;
        up.relu2 = 1;
        up.omax = hmax;
        up.nonfinite = nonfinite;
        up.nonfinite_stage = kStageIntermediate;
        if ((st = launch_expert_gemm(ctx, K_EXPERT_GEMM_OMAX, up, experts, inter, hidden, R, tokens, parts_up, stream, err))) return st;
        ExpertGemmArgs down{};
        down.ah = h;
        down.ah_tcol = 1;
        down.ahmax = hmax;
        down.ah_parts = parts_up;
        down.offsets = offsets;
        down.w = w_down;
        down.sw = s_down;
        down.bias = b.down;
        down.out = d;
        down.a_rows = (int)R;
        if ((st = launch_expert_gemm(ctx, K_EXPERT_GEMM_QA, down, experts, hidden, inter, R, tokens,
                                     expert_parts(ctx, experts, R, tokens, hidden), stream, err))) return st;
    } else {
        if ((st = moe_grouped_gemm(ctx, xq, sx, 0, top_k, offsets, perm, R, R, experts, w_up, s_up, b.up, inter,
                                   hidden, 1, h, stream, err)))
            return st;
        // the up outputs per slot: the layer's intermediate
        if ((st = launch_quantize(ctx, h, NH_F32, R, inter, hq, sh, nullptr, nullptr, stream, err, 0, nullptr, 1,
                                  nonfinite, kStageIntermediate)))
            return st;
        if ((st = moe_grouped_gemm(ctx, hq, sh, 0, top_k, offsets, perm, R, R, experts, w_down, s_down, b.down,
                                   hidden, inter, 0, d, stream, err)))
            return st;
    }
    return nh_moe_combine_shared(ctx, d, pos, wts, shared, tokens, top_k, hidden, out, out_dtype, stream, err);
}

nh_status nh_moe_forward_w8a8(nh_context* ctx, const void* x, nh_dtype x_dtype, const float* logits, size_t tokens,
                              size_t hidden, size_t inter, size_t experts, size_t top_k, int renormalize,
                              float scaling, const int8_t* w_up, const float* s_up, const int8_t* w_down,
                              const float* s_down, const nh_moe_biases* biases, void* out, nh_dtype out_dtype,
                              void* workspace, size_t workspace_bytes, uint64_t* nonfinite, nh_stream stream,
                              nh_error* err) {
    return moe_forward(ctx, x, x_dtype, logits, tokens, hidden, inter, experts, top_k, renormalize, scaling, w_up,
                       s_up, w_down, s_down, 0, nullptr, nullptr, nullptr, nullptr, biases, out, out_dtype, workspace,
                       workspace_bytes, nonfinite, stream, err);
}

size_t nh_moe_forward_shared_w8a8_workspace_size(size_t tokens, size_t hidden, size_t inter, size_t experts,
                                                 size_t top_k, size_t shared_inter) {
    size_t off[12];
    moe_layout(tokens, hidden, inter, experts, top_k, off);
    return off[11] + align256(tokens * hidden * sizeof(float)) +
           nh_mlp_w8a8_workspace_size(tokens, hidden, shared_inter);
}

nh_status nh_moe_forward_shared_w8a8(nh_context* ctx, const void* x, nh_dtype x_dtype, const float* logits,
                                     size_t tokens, size_t hidden, size_t inter, size_t experts, size_t top_k,
                                     int renormalize, float scaling, const int8_t* w_up, const float* s_up,
                                     const int8_t* w_down, const float* s_down, size_t shared_inter,
                                     const int8_t* w_up_shared, const float* s_up_shared,
                                     const int8_t* w_down_shared, const float* s_down_shared,
                                     const nh_moe_biases* biases, void* out, nh_dtype out_dtype, void* workspace,
                                     size_t workspace_bytes, uint64_t* nonfinite, nh_stream stream, nh_error* err) {
    if (!w_up_shared) {
        clear_error(err);
        return set_error(err, NH_INVALID_PARAMS, "w_up_shared must not be null (nh_moe_forward_w8a8 has no shared expert)");
    }
    return moe_forward(ctx, x, x_dtype, logits, tokens, hidden, inter, experts, top_k, renormalize, scaling, w_up,
                       s_up, w_down, s_down, shared_inter, w_up_shared, s_up_shared, w_down_shared, s_down_shared,
                       biases, out, out_dtype, workspace, workspace_bytes, nonfinite, stream, err);
}

size_t nh_moe_layer_w8a8_workspace_size(size_t tokens, size_t hidden, size_t inter, size_t experts, size_t top_k,
                                        size_t shared_inter) {
    const size_t inner = shared_inter
                             ? nh_moe_forward_shared_w8a8_workspace_size(tokens, hidden, inter, experts, top_k,
                                                                         shared_inter)
                             : nh_moe_forward_w8a8_workspace_size(tokens, hidden, inter, experts, top_k);
    return align256(inner) + align256(tokens * experts * sizeof(float));
}

// MoeLayer::forward_into (moe.rs:154-249) from its input: the dense f32
// router (router.project, moe.rs:185-188) as the f64-accumulated device GEMM
// of gemm_into_host with the bias added after the rounding to f32, its
// logits after the inner layer's workspace (so nh_moe_workspace_layout's
// offsets still hold), then the routed layer (and the shared expert) on them.
nh_status nh_moe_layer_w8a8(nh_context* ctx, const void* x, nh_dtype x_dtype, const float* router_w,
                            const float* router_b, size_t tokens, size_t hidden, size_t inter, size_t experts,
                            size_t top_k, int renormalize, float scaling, const int8_t* w_up, const float* s_up,
                            const int8_t* w_down, const float* s_down, size_t shared_inter,
                            const int8_t* w_up_shared, const float* s_up_shared, const int8_t* w_down_shared,
                            const float* s_down_shared, const nh_moe_biases* biases, void* out, nh_dtype out_dtype,
                            void* workspace, size_t workspace_bytes, uint64_t* nonfinite, nh_stream stream,
                            nh_error* err) {
    clear_error(err);
    if (tokens == 0) return set_error(err, NH_INVALID_ROW_COUNT, "row_count must be non-zero, got 0");
    if (hidden == 0 || experts == 0 || top_k == 0 || top_k > experts || inter == 0)
        return set_error(err, NH_INVALID_SHAPE, "invalid MoE shape");
    if (!router_w) return set_error(err, NH_INVALID_PARAMS, "router_w must not be null");
    if ((shared_inter != 0) != (w_up_shared != nullptr))
        return set_error(err, NH_INVALID_SHAPE, "shared_inter and w_up_shared must be given together");
    nh_status st;
    if ((st = check_dtype(x_dtype, err))) return st;
    const size_t inner = shared_inter
                             ? nh_moe_forward_shared_w8a8_workspace_size(tokens, hidden, inter, experts, top_k,
                                                                         shared_inter)
                             : nh_moe_forward_w8a8_workspace_size(tokens, hidden, inter, experts, top_k);
    const size_t need = nh_moe_layer_w8a8_workspace_size(tokens, hidden, inter, experts, top_k, shared_inter);
    if (!workspace || workspace_bytes < need) return mismatch(err, "workspace", need, workspace_bytes);
    if (!aligned16(workspace)) return set_error(err, NH_UNSUPPORTED, "workspace must be 16-byte aligned");
    size_t t;
    if (!mul_ok(tokens, hidden, &t) || !nh_supports_gemm_f32(tokens, hidden, experts))
        return set_error(err, NH_UNSUPPORTED, "router shape tokens=%zu hidden=%zu experts=%zu outside the device "
                         "envelope", tokens, hidden, experts);
    if ((st = bind_device(ctx, err))) return st;
    float* logits = (float*)((char*)workspace + align256(inner));
    GemmF32Args a{x, router_w, logits, (int64_t)tokens, (int64_t)hidden, (int64_t)experts, router_b,
                  x_dtype == NH_BF16 ? 1 : 0, 0};
    if ((st = launch_gemm_f32(ctx, a, stream, err))) return st;
    return moe_forward(ctx, x, x_dtype, logits, tokens, hidden, inter, experts, top_k, renormalize, scaling, w_up,
                       s_up, w_down, s_down, shared_inter, w_up_shared, s_up_shared, w_down_shared, s_down_shared,
                       biases, out, out_dtype, workspace, align256(inner), nonfinite, stream, err);
}

}  // extern "C"

// One read of bytes from src (device memory, 16-byte aligned, a multiple of
// 16, < 2^31): 1024 workgroups of 256 threads, four 16-byte loads per thread
// in flight.  sink: 256 device ints, normally never written.
extern "C" nh_status nh_handoff_status(nh_context* ctx, uint32_t* timeouts, uint32_t* busy, nh_error* err) {
    clear_error(err);
    if (!timeouts || !busy) return set_error(err, NH_INVALID_PARAMS, "null output pointer");
    nh_status st = bind_device(ctx, err);
    if (st) return st;
    std::vector<uint32_t> ring((size_t)kHandoffSlots * 16);
    hipError_t e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(ring.data(), ctx->handoff, ring.size() * 4, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return device_error(err, e, "nh_handoff_status");
    *timeouts = *busy = 0;
    for (uint32_t i = 0; i < kHandoffSlots; ++i) {
        *timeouts += ring[i * 16 + 2] != 0;
        *busy += ring[i * 16] != 0 || ring[i * 16 + 1] != 0;
    }
    return NH_OK;
}

extern "C" nh_status nh_stream_read(nh_context* ctx, const void* src, size_t bytes, int32_t* sink, nh_stream stream,
                                    nh_error* err) {
    clear_error(err);
    if (bytes == 0 || bytes % 16 != 0 || bytes >= (1ull << 31))
        return set_error(err, NH_INVALID_SHAPE, "stream of %zu bytes: a multiple of 16 below 2^31", bytes);
    if (!aligned16(src)) return set_error(err, NH_UNSUPPORTED, "src must be 16-byte aligned");
    nh_status st = bind_device(ctx, err);
    if (st) return st;
    StreamReadArgs a{src, sink, (uint32_t)bytes, 0};
    const size_t chunks = bytes / 16;
    const unsigned grid = (unsigned)std::min<size_t>(1024, (chunks + 256 * 4 - 1) / (256 * 4));
    return launch(ctx, K_STREAM_READ, grid, 256, 0, stream, a, err);
}

extern "C" nh_status nh_take_nonfinite(nh_context* ctx, uint64_t* nonfinite, nh_stream stream, nh_error* err) {
    clear_error(err);
    if (!nonfinite) return set_error(err, NH_INVALID_PARAMS, "null non-finite word");
    nh_status st = bind_device(ctx, err);
    if (st) return st;
    hipError_t e = hipStreamSynchronize((hipStream_t)stream);
    if (e != hipSuccess) return device_error(err, e, "hipStreamSynchronize");
    uint64_t word = 0;
    e = hipMemcpy(&word, nonfinite, sizeof(word), hipMemcpyDeviceToHost);
    if (e != hipSuccess) return device_error(err, e, "hipMemcpy(DtoH)");
    if (word == 0) return NH_OK;
    const uint64_t zero = 0;  // cleared for the next call
    e = hipMemcpy(nonfinite, &zero, sizeof(zero), hipMemcpyHostToDevice);
    if (e != hipSuccess) return device_error(err, e, "hipMemcpy(HtoD)");
    // the key of report_nonfinite (nh_device.h): stage, 38-bit index, sign and mantissa
    const uint64_t key = ~word;
    const uint32_t stage = (uint32_t)(key >> 62);
    const char* what = stage == kStageInput                ? "input"
                       : stage == kStageSharedIntermediate ? "shared_intermediate"
                                                           : "intermediate";
    const uint64_t index = (key >> 24) & ((1ull << 38) - 1);
    const float value =
        f32_from_bits((uint32_t)(((key >> 23) & 1u) << 31) | 0x7f800000u | (uint32_t)(key & 0x7fffffu));
    if (err) {
        err->argument = what;
        err->index = index;
        err->value = value;
    }
    return set_error(err, NH_NON_FINITE_INPUT, "non-finite %s value %g at index %llu", what, (double)value,
                     (unsigned long long)index);
}

// nh_linear_w8a8 with the static device scratch (scratch.hip) as its
// workspace: no allocation, for callers that cannot allocate.  Validation as
// nh_linear_w8a8, then the workspace the shape needs is checked against the
// scratch before anything else touches the device.
extern "C" nh_status nh_linear_w8a8_noalloc(nh_context* ctx, const void* x, nh_dtype x_dtype, const int8_t* wq,
                                            const float* sw, const float* bias, size_t m, size_t n, size_t k,
                                            void* out, nh_dtype out_dtype, int8_t* xq_out, float* sx_out,
                                            uint64_t* nonfinite, nh_stream stream, nh_error* err) {
    clear_error(err);
    if (m == 0) return set_error(err, NH_INVALID_ROW_COUNT, "row_count must be non-zero, got 0");
    nh_status st;
    if ((st = check_dtype(x_dtype, err)) || (st = check_dtype(out_dtype, err)) ||
        (st = check_w8a8_shape(m, n, k, err)))
        return st;
    const size_t need = nh_linear_w8a8_workspace_size(m, k);
    if (need > kScratchBytes)
        return set_error(err, NH_UNSUPPORTED,
                         "m=%zu k=%zu needs a %zu-byte workspace, above the %zu-byte static scratch of "
                         "nh_linear_w8a8_noalloc (use nh_linear_w8a8 with a caller workspace)",
                         m, k, need, kScratchBytes);
    if (!aligned16(wq)) return set_error(err, NH_UNSUPPORTED, "wq must be 16-byte aligned");
    if ((st = bind_device(ctx, err))) return st;
    if (!ctx->scratch) return set_error(err, NH_DEVICE_ERROR, "static scratch unavailable: %s", ctx->scratch_error);
    return linear_w8a8(ctx, x, x_dtype, wq, sw, bias, m, n, k, out, out_dtype, ctx->scratch, kScratchBytes, xq_out,
                       sx_out, 0, nonfinite, 0, stream, err);
}
