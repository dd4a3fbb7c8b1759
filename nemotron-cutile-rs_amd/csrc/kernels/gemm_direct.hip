// G3 for tens to a few hundred rows (batched decode, short prompts): a W8A8 or
// W4A8 GEMM whose waves load both MFMA operands straight into registers.
//
// With few rows the LDS-tiled kernels (gemm.hip) spend their time on the stage
// loop: a 64 x 64 tile takes ~0.21 us per 64-deep K tile whatever it holds
// (loads, a barrier, fragment reads and a few MFMAs in a chain), and few tiles
// leave CUs idle.  Here a workgroup owns 16 MR rows (MR <= 8) x 16 NR columns
// and its four waves split K: wave w takes K tiles w, w + 4, ...  Both operands
// are stored in MFMA operand order (tiled A, tiled weights), so every fragment
// is one contiguous 16-byte-per-lane load; the K loop has no LDS and no barrier,
// each wave keeps D K tiles in flight.  The four partial tiles meet in LDS once,
// at the end (int32 sums: exact in any order).
//
// What bounds it: the CU's vector-memory path, 65.7 KiB/us over the whole launch
// at 500 x 4096 x 21504 (256 workgroups of 336 K tiles of 12 KiB in 61.4 us).  A K
// tile costs MR + NR KiB there (MR + NR / 2 with INT4 weights); the tile shape, a
// function of the launch, keeps that small while filling the CUs (plan_direct).
// Workgroups are dealt so that the row groups of a column block run side by side
// on one XCD, whose L2 then reads the weights once.
//
// Measured against the LDS-tiled kernels (tiled A in, cold weights):
// 33 x 4096 x 8192 29.7 -> 13.0 us, 77 x 6144 x 4096 15.8 -> 11.5, 256 x 2688 x
// 8192 28.9 -> 22.6, 500 x 4096 x 21504 76.5 -> 61.4.
#include "nh_device.h"

using namespace nh;

namespace {

typedef float nh_v4f __attribute__((ext_vector_type(4)));

constexpr int kDirectWaves = 4;
constexpr int kDirectPhase = 16;  // fragments summed across the waves at a time (64 KiB of LDS)

// int8 B operand (codes 0..15, K order) from 8 bytes of tiled INT4 codes.
__device__ __forceinline__ v4i expand_int4_ordered(uint2 q) {
    v4i r;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t w = h ? q.y : q.x;
        const uint32_t even = w & 0x0F0F0F0Fu, odd = (w >> 4) & 0x0F0F0F0Fu;
        r[2 * h] = (int)__builtin_amdgcn_perm(odd, even, 0x05010400u);
        r[2 * h + 1] = (int)__builtin_amdgcn_perm(odd, even, 0x07030602u);
    }
    return r;
}

// One workgroup tile: M tiles mt0 .. mt0 + MR - 1 (all inside the matrix) by
// N tiles nt0 .. nt0 + NR - 1 (those past the matrix load zeros).  ST: the
// weights are read by this workgroup alone (one row group), with the
// non-temporal policy (64 x 16384 x 4096: 15.4 us against 17.1).
// W4: the MFMAs sum xq * code; the zero point comes off in the epilogue as
// zp * sum_k xq (integers: exact), the row sums from v_dot4 on the A fragments.
template <int MR, int NR, bool W4, bool ST>
__device__ __forceinline__ void direct_tile(const GemmDirectArgs& d, int8_t* lds, int mt0, int nt0) {
    constexpr int W = kDirectWaves, F = MR * NR;
    constexpr int kTile = W4 ? 512 : 1024;
    constexpr int D = direct_depth(MR, NR, W4);  // K tiles in flight per wave
    const GemmW8A8Args& a = d.g;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int KT = a.kt, M = a.M, N = a.N;
    const int m0 = mt0 * 16, n0 = nt0 * 16;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(a.xq + (int64_t)mt0 * KT * 1024, (uint32_t)(MR * KT) * 1024u);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc(a.wq + (int64_t)nt0 * KT * kTile,
                                                (uint32_t)(min(NR, (N + 15) / 16 - nt0) * KT) * (uint32_t)kTile);
    // the epilogue's operands, ahead of the stream (thread t: row m0 + t, column n0 + t)
    float sxv = 0.0f, swv = 0.0f, sbv = 0.0f;
    if (tid < MR * 16 && m0 + tid < M) sxv = a.sx[m0 + tid];
    if (tid < NR * 16 && n0 + tid < N) {
        swv = W4 ? d.w4_scale : a.sw[n0 + tid];
        if (a.bias) sbv = a.bias[n0 + tid];
    }
    const uint32_t la = (uint32_t)lane * 16u, lb = (uint32_t)lane * (kTile / 64);
    v4i fa[D][MR];
    v4i fb[W4 ? 1 : D][NR];
    uint2 fq[W4 ? D : 1][NR];
    // K tile wave + 4 s into slot u.  Past the last one every offset lies
    // beyond the operands (KT <= 2048: below 32 MiB), so the loads return
    // zeros without touching memory and all counts stay fixed.
    auto load = [&](int u, int s) {
        const int kt = wave + s * W;
        const uint32_t past = 0x78000000u;
        const uint32_t ob = (kt < KT ? (uint32_t)(kt * kTile) : past) + lb;
        const uint32_t oa = (kt < KT ? (uint32_t)kt * 1024u : past) + la;
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            const int off = (int)(ob + (uint32_t)(j * KT) * (uint32_t)kTile);
            if constexpr (W4)
                fq[u][j] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rb, off, 0, ST ? 2 : 0));
            else
                fb[u][j] = ST ? buffer_load16_stream(rb, off) : buffer_load16(rb, off);
        }
#pragma unroll
        for (int i = 0; i < MR; ++i) fa[u][i] = buffer_load16(ra, (int)(oa + (uint32_t)(i * KT) * 1024u));
        __builtin_amdgcn_sched_barrier(0);  // issue order = slot order: the waits below are exact counts
    };
    v4i acc[MR][NR];
    int rsum[MR];
#pragma unroll
    for (int i = 0; i < MR; ++i) {
        rsum[i] = 0;
#pragma unroll
        for (int j = 0; j < NR; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < D; ++s) load(s, s);
    const int steps = (KT + W - 1) / W;
    for (int s0 = 0; s0 < steps; s0 += D) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
            v4i b[NR];
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                if constexpr (W4) b[j] = expand_int4_ordered(fq[u][j]);
                else b[j] = fb[u][j];
            }
#pragma unroll
            for (int i = 0; i < MR; ++i) {
#pragma unroll
                for (int j = 0; j < NR; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b[j], fa[u][i], acc[i][j], 0, 0, 0);
                if constexpr (W4) {
#pragma unroll
                    for (int w = 0; w < 4; ++w) rsum[i] = __builtin_amdgcn_sdot4(fa[u][i][w], 0x01010101, rsum[i], false);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            load(u, s0 + u + D);
        }
    }
    // The waves' partial tiles summed through LDS, kDirectPhase fragments at a
    // time; wave w then finishes a quarter of them.  The MFMAs took the weight
    // fragment first: lane l holds row l % 16, columns 4 (l / 16) .. + 3 of a
    // fragment (one 8- or 16-byte store).
    v4i* red = (v4i*)lds;
    float* sx = (float*)(lds + W * kDirectPhase * 1024);  // [128]
    float* sw = sx + 128;                                 // [128]
    float* sb = sw + 128;                                 // [128]
    int* rs = (int*)(sb + 128);                           // [4 waves][128] INT4: row sums of the codes
    if (tid < 128) {
        sx[tid] = sxv;
        sw[tid] = swv;
        sb[tid] = sbv;
    }
    if constexpr (W4) {
#pragma unroll
        for (int i = 0; i < MR; ++i) {
            int v = rsum[i] + __shfl_xor(rsum[i], 16, kWave);
            v += __shfl_xor(v, 32, kWave);
            if (lane < 16) rs[wave * 128 + i * 16 + lane] = v;
        }
    }
    constexpr int PER = kDirectPhase / W;
    const int esz = a.out_dtype == DT_BF16 ? 2 : 4;
    const int64_t ldo = a.ldo;
#pragma unroll
    for (int p0 = 0; p0 < F; p0 += kDirectPhase) {
        if (p0) __syncthreads();
#pragma unroll
        for (int f = p0; f < F && f < p0 + kDirectPhase; ++f)
            red[(wave * kDirectPhase + f - p0) * 64 + lane] = acc[f / NR][f % NR];
        __syncthreads();
#pragma unroll 1
        for (int q = 0; q < PER; ++q) {
            const int fl = wave * PER + q, f = p0 + fl;
            if (f >= F) break;
            const int i = f / NR, j = f - i * NR;
            const int lm = i * 16 + (lane & 15), ln = j * 16 + 4 * (lane >> 4);
            const int m = m0 + lm, n = n0 + ln;
            v4i sum = red[fl * 64 + lane];
#pragma unroll
            for (int w = 1; w < W; ++w) sum += red[(w * kDirectPhase + fl) * 64 + lane];
            if constexpr (W4) {
                int v = 0;
#pragma unroll
                for (int w = 0; w < W; ++w) v += rs[w * 128 + lm];
                sum -= d.w4_zp * v;
            }
            const float sxm = sx[lm];
            const nh_v4f sw4 = *(const nh_v4f*)(sw + ln), sb4 = *(const nh_v4f*)(sb + ln);
            float y[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                y[r] = epilogue_w8a8(sum[r], sxm, sw4[r]);
                if (a.bias) y[r] = y[r] + sb4[r];
                if (a.relu2) y[r] = relu2(y[r]);
            }
            if (m >= M) continue;
            if (n + 3 < N) {
                store_cols4((int8_t*)a.out + ((int64_t)m * ldo + n) * esz, y, esz == 2);
            } else {  // the matrix edge
#pragma unroll 1
                for (int r = 0; r < 4 && n + r < N; ++r) {
                    store_out(a.out, (int64_t)m * ldo + n + r, y[0], a.out_dtype);
                    y[0] = y[1];
                    y[1] = y[2];
                    y[2] = y[3];
                }
            }
        }
    }
}

// Workgroup b: XCD b % 8 takes column blocks = b mod 8, the row groups of
// one block consecutive.  Row groups are balanced (sizes differ by one M
// tile), so with several groups none has fewer than MAXR / 2 tiles.
template <int NR, int MAXR, bool W4>
__device__ __forceinline__ void gemm_direct(const GemmDirectArgs& d, int8_t* lds) {
    const int i = (int)blockIdx.x >> 3, G = d.groups;
    const int g = i % G, tn = (i / G) * 8 + ((int)blockIdx.x & 7);
    if (tn >= d.g.tiles_n) return;  // uniform
    const int mtiles = (d.g.M + 15) / 16;
    const int mt0 = (int)((int64_t)g * mtiles / G), mr = (int)((int64_t)(g + 1) * mtiles / G) - mt0;
    const int nt0 = tn * NR;
#define NH_ROWS(r)                                                                          \
    case r:                                                                                 \
        if constexpr (r <= MAXR) {                                                          \
            if (G == 1) direct_tile<r, NR, W4, true>(d, lds, mt0, nt0);                     \
            else if constexpr (2 * r >= MAXR) direct_tile<r, NR, W4, false>(d, lds, mt0, nt0); \
        }                                                                                   \
        break;
    switch (mr) {
        NH_ROWS(1) NH_ROWS(2) NH_ROWS(3) NH_ROWS(4) NH_ROWS(5) NH_ROWS(6) NH_ROWS(7) NH_ROWS(8)
        default: break;
    }
#undef NH_ROWS
}

}  // namespace

#define NH_DIRECT_KERNEL(name, NR, MAXR, W4)                                                        \
    extern "C" __global__ __launch_bounds__(64 * kDirectWaves, 2) void name(GemmDirectArgs d) {     \
        extern __shared__ __align__(1024) int8_t smem[];                                            \
        gemm_direct<NR, MAXR, W4>(d, smem);                                                         \
    }
NH_DIRECT_KERNEL(nh_gemm_w8a8_direct16_kernel, 1, 8, false)   // 128 rows x 16 columns
NH_DIRECT_KERNEL(nh_gemm_w8a8_direct32_kernel, 2, 8, false)   // x 32
NH_DIRECT_KERNEL(nh_gemm_w8a8_direct64_kernel, 4, 8, false)   // x 64
NH_DIRECT_KERNEL(nh_gemm_w4a8_direct16_kernel, 1, 8, true)
NH_DIRECT_KERNEL(nh_gemm_w4a8_direct32_kernel, 2, 8, true)
NH_DIRECT_KERNEL(nh_gemm_w4a8_direct64_kernel, 4, 8, true)
NH_DIRECT_KERNEL(nh_gemm_w4a8_direct128_kernel, 8, 4, true)   // 64 rows x 128 columns
