// G0d: the reference's device f32 GEMM (gemm.rs:318-363) restated for gfx950.
// out[m][n] = sum_k lhs[m][k] * rhs[k][n] with lhs [M][K] and rhs [K][N]
// row-major f32, accumulated in f64 with k ascending for every output, then
// rounded to f32: the arithmetic and order of gemm_into_host (gemm.rs:99-109).
// Each f32 x f32 product is exact in f64, so the fused multiply-add rounds
// exactly like the reference's `acc += lhs as f64 * rhs as f64`, and the
// device result equals the host path bit for bit (no tolerance needed).
//
// A workgroup of 256 threads owns a 64 x 64 output tile, each thread a 4 x 4
// block; K advances 16 at a time through LDS (A transposed to [k][m] so both
// operand reads are 16-byte vectors).  The last K step accumulates only the
// positions that exist, so every output sees exactly K fused multiply-adds.
//
// For the MoE router (moe.rs:185-188, a dense f32 LinearProjection) the lhs
// may be bf16 (widened exactly to f32 on load) and a bias may follow the
// rounding to f32, as project_into adds it (linear.rs:330-336).
#include "nh_device.h"

using namespace nh;

extern "C" __global__ __launch_bounds__(256) void nh_gemm_f32_kernel(GemmF32Args a) {
    // operands widened to f64 once, as they are staged (each value is read by
    // 16 lanes), so the K loop is loads and fused multiply-adds only
    __shared__ __align__(16) double As[16][64 + 2];
    __shared__ __align__(16) double Bs[16][64 + 2];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int64_t M = a.M, K = a.K, N = a.N;
    const int64_t m0 = (int64_t)blockIdx.y * 64, n0 = (int64_t)blockIdx.x * 64;
    double acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.0;
    // one K step's values of this thread, loaded a step ahead of their use
    float ra[4], rb[4];
    auto fetch = [&](int64_t k0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = threadIdx.x + 256 * i;
            const int r = idx >> 4, kk = idx & 15;
            const int64_t gm = m0 + r, gk = k0 + kk;
            float v = 0.0f;
            if (gm < M && gk < K)
                v = a.lhs_bf16 ? f32_from_bits((uint32_t)((const uint16_t*)a.lhs)[gm * K + gk] << 16)
                               : ((const float*)a.lhs)[gm * K + gk];
            ra[i] = v;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = threadIdx.x + 256 * i;
            const int kk = idx >> 6, c = idx & 63;
            const int64_t gk = k0 + kk, gn = n0 + c;
            rb[i] = (gk < K && gn < N) ? a.rhs[gk * N + gn] : 0.0f;
        }
    };
    fetch(0);
    for (int64_t k0 = 0; k0 < K; k0 += 16) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = threadIdx.x + 256 * i;
            As[idx & 15][idx >> 4] = (double)ra[i];
            Bs[idx >> 6][idx & 63] = (double)rb[i];
        }
        __syncthreads();
        if (k0 + 16 < K) fetch(k0 + 16);  // uniform
        const int kmax = (int)(K - k0 < 16 ? K - k0 : 16);
        for (int kk = 0; kk < kmax; ++kk) {
            const double2 a01 = *(const double2*)&As[kk][ty * 4], a23 = *(const double2*)&As[kk][ty * 4 + 2];
            const double2 b01 = *(const double2*)&Bs[kk][tx * 4], b23 = *(const double2*)&Bs[kk][tx * 4 + 2];
            const double ad[4] = {a01.x, a01.y, a23.x, a23.y};
            const double bd[4] = {b01.x, b01.y, b23.x, b23.y};
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fma(ad[i], bd[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t gm = m0 + ty * 4 + i;
        if (gm >= M) break;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t gn = n0 + tx * 4 + j;
            if (gn < N) a.out[gm * N + gn] = a.bias ? (float)acc[i][j] + a.bias[gn] : (float)acc[i][j];
        }
    }
}

// The same product on the f64 matrix cores, for outputs too few to fill the
// CUs with 64 x 64 tiles (the MoE router: 512 tokens x 128 experts are 16 such
// tiles).  v_mfma_f64_4x4x4f64 computes, for each of its 64 outputs, four
// fused multiply-adds in k order onto the accumulator: on the device every
// output equals the chain fma(a3, b3, fma(a2, b2, fma(a1, b1, fma(a0, b0,
// c)))) bit for bit (12,800 outputs of random-exponent operands; the reversed
// order matched 61% of them), so a chain of these MFMAs is the reference's
// f64 accumulation in k order.  Operand roles (read off one-hot probes): A
// lane 16 k + 4 b + i holds A[i][k] of block b, B lane 16 k + 4 b + j holds
// B[k][j] of block b, D lane 16 i + 4 b + j holds D[i][j] of block b: four
// 4 x 4 blocks per wave.
//
// A workgroup owns 16 x 16 outputs and has two roles.  Chain wave w (0..3) runs
// the rows 4w..4w+3 with, as its blocks b, the columns 4b..4b+3: one chain of
// 64 outputs, 21 cycles per 4-k step (the MFMA's dependent latency; its issue
// rate is one per 16), and does nothing but operand reads and MFMAs.  Staging
// waves (4, 5: lhs, 6, 7: rhs) load the operands, widen them to f64 once and
// write them to LDS in the chain's order, two steps of a lane side by side, so
// a chain wave reads two steps' operands with two 16-byte reads.  With the
// loads and the widening in the chain waves a step took ~56 cycles.
// K advances in chunks of 64 through three LDS buffers (55 KiB: two workgroups
// per CU).  Barrier c says that chunk c is written; the chain waves pass it
// halfway through chunk c - 1 and read four step pairs ahead, so neither the
// barrier nor the LDS latency interrupts the chain.  The staging waves write
// chunk c + 1 after barrier c, into the buffer of chunk c - 2, which the chain
// waves have finished by then; their loads run six chunks ahead (a chunk is
// ~0.15 us of chain, a load from HBM over 1 us).
// k past K, rows past M and columns past N are zeros: an added fma(0, 0, acc)
// leaves acc unchanged, as acc starts at +0.0 and a k-ordered sum of products
// that starts there is never -0.0.
// Bound by the chain: 672 steps at K = 2688 are 6 us, the launch and the first
// loads ~6 more.  Measured: 8 x 2688 x 128 23.4 -> 14.2 us, 512 x 2688 x 128
// 25.0 -> 19.4, 100 x 4096 x 60 34.4 -> 24.0, 2048 x 4096 x 128 (four rounds, the
// MFMA pipes busy) 84.2 -> 82.0.  Chunks of 128 in 108 KiB were as fast on one
// round and 93 us on four.
// K of one or two chunks (SHORT) has two buffers and two chunks of loads, none
// ahead: with the third buffer's LDS two workgroups fit a CU and not four, and
// the loads past the end cost as much as the product.  1210 x 8 x 360 8.1 -> 5.9
// us, 546 x 107 x 101 4.6 -> 3.7, 2048 x 128 x 128 6.3 -> 5.2 (4.6 with one role
// per wave and 16-byte rhs loads, which one round of few workgroups loses by).
//
// Loads go through buffer resources over the whole operands (wave-uniform;
// the launch keeps both below 2^31 bytes), positions past the matrix sent out
// of range so they read zeros with no branch.  VEC (16-byte aligned lhs, K a
// multiple of 8 for bf16 or 4 for f32): 16-byte lhs loads; otherwise one load
// per value.
namespace {

constexpr int kF32Chunk = 64;                   // k per chunk: 8 pairs of 4-k steps
constexpr int kF32Ahead = 6;                     // chunks of operands in flight per staging thread
constexpr int kF32Pairs = kF32Chunk / 8;
constexpr int kF32APair = 320;                  // bytes of a step pair of 4 rows: 256, padded against bank conflicts
constexpr int kF32AGroup = kF32Pairs * kF32APair;
constexpr int kF32ABytes = 4 * kF32AGroup;
constexpr int kF32Buffer = kF32ABytes + kF32Pairs * 1024;  // A of the 4 row groups, then B
static_assert(kF32Buffer == kGemmF32MfmaBuffer, "the host's LDS size");

typedef double nh_v2d __attribute__((ext_vector_type(2)));

// One staging thread's operand (A: row t / 8, the step pair t % 8, i.e. 8
// consecutive k; B: column t % 16, the step pair t / 16), chunk by chunk.
// Offsets past the matrix get bit 31 (operands are below 2^31 bytes), by
// arithmetic: a select becomes a branch around the load, and then every wait
// a wait for all loads (23 us instead of 14 at 8 x 2688 x 128).
__device__ __forceinline__ uint32_t past_end(int v, int end) { return (uint32_t)((end - 1 - v) >> 31) & 0x80000000u; }

template <bool BF16, bool VEC>
struct StageA {
    static constexpr int kRegs = VEC && BF16 ? 4 : 8;
    static constexpr uint32_t esz = BF16 ? 2u : 4u;
    __amdgpu_buffer_rsrc_t r;
    uint32_t start;
    int k0, K, lds0;
    __device__ StageA(const GemmF32Args& a, int t, int64_t m0, int64_t)
        : r(make_rsrc(a.lhs, (uint32_t)a.M * (uint32_t)a.K * esz)), k0(8 * (t & 7)), K((int)a.K) {
        const int row = t >> 3, m = (int)m0 + row;
        start = ((uint32_t)m * (uint32_t)K + (uint32_t)k0) * esz | past_end(m, (int)a.M);
        lds0 = (row >> 2) * kF32AGroup + (t & 7) * kF32APair + (row & 3) * 16;
    }
    __device__ void fetch(int c, uint32_t (&v)[kRegs]) const {
        const uint32_t base = start + (uint32_t)(c * kF32Chunk) * esz;
        const int k = c * kF32Chunk + k0;
        if constexpr (VEC) {
#pragma unroll
            for (int h = 0; h < kRegs / 4; ++h) {
                const v4i x = buffer_load16(r, (int)((base + 16u * h) | past_end(k + 4 * h, K)));
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * h + e] = (uint32_t)x[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t off = (base + esz * e) | past_end(k + e, K);
                v[e] = BF16 ? (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0)
                            : (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
            }
        }
    }
    static __device__ double value(const uint32_t (&v)[kRegs], int e) {
        if constexpr (!BF16) return (double)f32_from_bits(v[e]);
        else if constexpr (VEC) return (double)f32_from_bits((e & 1) ? v[e >> 1] & 0xffff0000u : v[e >> 1] << 16);
        else return (double)f32_from_bits(v[e] << 16);
    }
    // k = 8 pair + 4 h + kk: step 2 pair + h, the MFMA's k index kk
    __device__ void store(int8_t* buf, const uint32_t (&v)[kRegs]) const {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) *(nh_v2d*)(buf + lds0 + kk * 64) = nh_v2d{value(v, kk), value(v, kk + 4)};
    }
};

struct StageB {
    static constexpr int kRegs = 8;
    __amdgpu_buffer_rsrc_t r;
    uint32_t start, step;
    int lds0;
    __device__ StageB(const GemmF32Args& a, int t, int64_t, int64_t n0)
        : r(make_rsrc(a.rhs, (uint32_t)a.K * (uint32_t)a.N * 4u)), step((uint32_t)a.N * 4u) {
        const int n = (int)n0 + (t & 15);
        start = (8u * (uint32_t)(t >> 4) * (uint32_t)a.N + (uint32_t)n) * 4u | past_end(n, (int)a.N);
        lds0 = kF32ABytes + (t >> 4) * 1024 + (t & 15) * 16;
    }
    __device__ void fetch(int c, uint32_t (&v)[kRegs]) const {  // (k past K: past the end of rhs)
        uint32_t off = start + (uint32_t)(c * kF32Chunk) * step;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
            off += step;
        }
    }
    __device__ void store(int8_t* buf, const uint32_t (&v)[kRegs]) const {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
            *(nh_v2d*)(buf + lds0 + kk * 256) =
                nh_v2d{(double)f32_from_bits(v[kk]), (double)f32_from_bits(v[kk + 4])};
    }
};

template <bool SHORT, class Stage>
__device__ __forceinline__ void gemm_f32_stage(const Stage& s, int8_t* lds, int nc) {
    constexpr int AHEAD = SHORT ? 2 : kF32Ahead;
    uint32_t v[AHEAD][Stage::kRegs];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {  // (chunks past the last: zeros)
        s.fetch(u, v[u]);
        __builtin_amdgcn_sched_barrier(0);
    }
    int buf = 0;
    for (int c = 0; c < nc; c += AHEAD) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            if (c + u >= nc) break;  // uniform
            s.store(lds + buf * kF32Buffer, v[u]);
            if constexpr (!SHORT) s.fetch(c + u + AHEAD, v[u]);
            lds_publish();  // barrier c + u
            buf = buf == 2 ? 0 : buf + 1;
        }
    }
}

template <bool SHORT>
__device__ __forceinline__ void gemm_f32_chain(const GemmF32Args& a, const int8_t* lds, int64_t m0, int64_t n0, int nc) {
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (m0 + 4 * w >= a.M) {  // no rows (uniform): the barriers only
        for (int c = 0; c < nc; ++c) lds_barrier();
        return;
    }
    // lane l: A[row l % 4][k l / 16], B[k l / 16][column l % 16]
    const int8_t* pa = lds + w * kF32AGroup + (lane >> 4) * 64 + (lane & 3) * 16;
    const int8_t* pb = lds + kF32ABytes + lane * 16;
    constexpr int AHEAD = 4;  // step pairs read ahead
    nh_v2d av[AHEAD], bv[AHEAD];
    auto read = [&](int buf, int p) {
        av[p % AHEAD] = *(const nh_v2d*)(pa + buf * kF32Buffer + p * kF32APair);
        bv[p % AHEAD] = *(const nh_v2d*)(pb + buf * kF32Buffer + p * 1024);
    };
    double acc = 0.0;
    lds_barrier();  // chunk 0
#pragma unroll
    for (int p = 0; p < AHEAD; ++p) read(0, p);
    int buf = 0;
    for (int c = 0; c < nc; ++c) {
        const int next = SHORT ? buf ^ 1 : buf == 2 ? 0 : buf + 1;
#pragma unroll
        for (int p = 0; p < kF32Pairs; ++p) {
            if (p == kF32Pairs / 2 && c + 1 < nc) lds_barrier();  // chunk c + 1
            const nh_v2d x = av[p % AHEAD], y = bv[p % AHEAD];
            acc = __builtin_amdgcn_mfma_f64_4x4x4f64(x[0], y[0], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f64_4x4x4f64(x[1], y[1], acc, 0, 0, 0);
            // (after the last chunk the reads are of an older one, and unused)
            if (p + AHEAD < kF32Pairs) read(buf, p + AHEAD);
            else read(next, p + AHEAD - kF32Pairs);
            __builtin_amdgcn_sched_barrier(0);
        }
        buf = next;
    }
    // D lane 16 i + 4 b + j: output (4w + i, 4b + j)
    const int64_t gm = m0 + 4 * w + (lane >> 4), gn = n0 + 4 * ((lane >> 2) & 3) + (lane & 3);
    if (gm < a.M && gn < a.N) a.out[gm * a.N + gn] = a.bias ? (float)acc + a.bias[gn] : (float)acc;
}

template <bool BF16, bool VEC, bool SHORT>
__device__ __forceinline__ void gemm_f32_mfma(const GemmF32Args& a, int8_t* lds) {
    const int64_t tiles_n = (a.N + 15) / 16;
    const int64_t m0 = (int64_t)(blockIdx.x / tiles_n) * 16, n0 = (int64_t)(blockIdx.x % tiles_n) * 16;
    const int nc = (int)((a.K + kF32Chunk - 1) / kF32Chunk);
    if (threadIdx.x < 256)
        gemm_f32_chain<SHORT>(a, lds, m0, n0, nc);
    else if (threadIdx.x < 384)
        gemm_f32_stage<SHORT>(StageA<BF16, VEC>(a, threadIdx.x - 256, m0, n0), lds, nc);
    else
        gemm_f32_stage<SHORT>(StageB(a, threadIdx.x - 384, m0, n0), lds, nc);
}

}  // namespace

// ANY: any alignment and K, one load per value.  SHORT: K <= 128.
#define NH_F32_MFMA_KERNEL(name, BF16, SHORT)                                      \
    extern "C" __global__ __launch_bounds__(512) void name(GemmF32Args a) {        \
        extern __shared__ __align__(1024) int8_t smem[];                           \
        gemm_f32_mfma<BF16, true, SHORT>(a, smem);                                 \
    }
#define NH_F32_MFMA_ANY_KERNEL(name, SHORT)                                        \
    extern "C" __global__ __launch_bounds__(512) void name(GemmF32Args a) {        \
        extern __shared__ __align__(1024) int8_t smem[];                           \
        if (a.lhs_bf16)                                                            \
            gemm_f32_mfma<true, false, SHORT>(a, smem);                            \
        else                                                                       \
            gemm_f32_mfma<false, false, SHORT>(a, smem);                           \
    }
NH_F32_MFMA_KERNEL(nh_gemm_f32_mfma_kernel, false, false)
NH_F32_MFMA_KERNEL(nh_gemm_f32_mfma_bf16_kernel, true, false)
NH_F32_MFMA_ANY_KERNEL(nh_gemm_f32_mfma_any_kernel, false)
NH_F32_MFMA_KERNEL(nh_gemm_f32_mfma_short_kernel, false, true)
NH_F32_MFMA_KERNEL(nh_gemm_f32_mfma_short_bf16_kernel, true, true)
NH_F32_MFMA_ANY_KERNEL(nh_gemm_f32_mfma_short_any_kernel, true)
