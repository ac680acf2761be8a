// k_f16mm.hip — fp16 x fp16 -> fp16 matmul with the reference OP_MATMUL_F16 contract
// (oplist_exec.c:1709-1813): flags t0 (a stored [K,M]), t1 (w stored [N,K]), batched
// (Bn in flags >> 16), and the SPLIT column window [n0, n0+N) of an N_full-wide output.
//
//   M <= 4, t1:   GEMV, one wavefront per output column n streaming w's row n (the
//                 lm_head path); activations staged once per workgroup in LDS.
//   M <= 4, !t1:  GEMV over columns: 8 columns per lane, K split over a workgroup; for short
//                 K one column per thread.
//   otherwise:    MFMA 32x32x16 tiles (any shape, flags, alignment).
#include "dev_reduce.h"
#include "kernels.h"

#include <algorithm>
#include <type_traits>

namespace gehtp {

namespace {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef float f16x_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short s4_t __attribute__((ext_vector_type(4)));
// 16-byte load of fp16 rows at any element offset (an odd row length leaves rows 2-byte aligned)
typedef u32x4 u32x4_u __attribute__((aligned(2)));

// Reinterpret a 32-bit word as two halves. Takes the word BY VALUE: a bit cast applied
// directly to an ext_vector element (v[e]) miscompiles to always reading element 0.
__device__ __forceinline__ h2_t as_h2(uint32_t v) { return __builtin_bit_cast(h2_t, v); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// --- GEMV, w stored [N][K] ---------------------------------------------------
// 16 output columns per workgroup (4 per wave). vec: K % 8 == 0 and 16-byte alignment.
template <int MR>
__global__ __launch_bounds__(256) void gemv_nk_kernel(const __half* __restrict__ a,
                                                      const __half* __restrict__ w,
                                                      __half* __restrict__ y, uint32_t K,
                                                      uint32_t N_full, uint32_t n0, uint32_t N,
                                                      uint32_t M) {
    extern __shared__ u32x4 xs[];   // [MR][K/8]
    const uint32_t bb = blockIdx.y;
    const __half* ab = a + (size_t)bb * M * K;
    const __half* wb = w + (size_t)bb * N_full * K;
    __half* yb = y + (size_t)bb * M * N_full;
    const uint32_t kc = K / 8;
    for (uint32_t i = threadIdx.x; i < MR * kc; i += 256)
        xs[i] = reinterpret_cast<const u32x4*>(ab)[(i / kc) * kc + (i % kc)];
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (uint32_t r = 0; r < 4; ++r) {
        const uint32_t n = blockIdx.x * 16 + wave * 4 + r;
        if (n >= N) break;
        const u32x4* wr = reinterpret_cast<const u32x4*>(wb + (size_t)(n0 + n) * K);
        float acc[MR];
#pragma unroll
        for (int m = 0; m < MR; ++m) acc[m] = 0.0f;
        for (uint32_t c = lane; c < kc; c += 64) {
            const u32x4 wv = __builtin_nontemporal_load(&wr[c]);
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                const u32x4 xv = xs[m * kc + c];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    acc[m] = __builtin_amdgcn_fdot2(as_h2(wv[e]),
                                                    as_h2(xv[e]), acc[m], false);
            }
        }
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            const float s = wave_sum(acc[m]);
            if (lane == 0) yb[(size_t)m * N_full + n0 + n] = __float2half(s);
        }
    }
}

// The same GEMV for M = 1 when each lane owns NC = K / 512 16-byte chunks of a row (the
// lm_head: K = 2560, NC = 5): the activation chunks are requested first, then every
// weight chunk of the wave's 4 rows, and only then x is staged in LDS and the rows are
// computed, so a wave waits on one memory round trip instead of one per row. Each lane
// accumulates chunks lane, lane + 64, ... in the order of gemv_nk_kernel and the row sum
// is the same wave reduction: the same bits.
template <int NC>
__global__ __launch_bounds__(256) void gemv_nk_pre_kernel(const __half* __restrict__ a,
                                                          const __half* __restrict__ w,
                                                          __half* __restrict__ y, uint32_t K,
                                                          uint32_t N_full, uint32_t n0, uint32_t N) {
    constexpr uint32_t kc = 64 * NC, XC = (kc + 255) / 256;
    extern __shared__ u32x4 xs[];   // [K/8]
    const uint32_t bb = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const u32x4* ab = reinterpret_cast<const u32x4*>(a + (size_t)bb * K);
    const __half* wb = w + (size_t)bb * N_full * K;
    __half* yb = y + (size_t)bb * N_full;
    u32x4 xr[XC];
#pragma unroll
    for (uint32_t i = 0; i < XC; ++i) xr[i] = ab[min(tid + 256 * i, kc - 1)];
    const uint32_t nb = blockIdx.x * 16 + wave * 4;
    u32x4 wv[4][NC];
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
        const u32x4* wr = reinterpret_cast<const u32x4*>(wb + (size_t)(n0 + min(nb + r, N - 1)) * K);
#pragma unroll
        for (int j = 0; j < NC; ++j) wv[r][j] = __builtin_nontemporal_load(&wr[lane + 64 * j]);
    }
#pragma unroll
    for (uint32_t i = 0; i < XC; ++i)
        if (tid + 256 * i < kc) xs[tid + 256 * i] = xr[i];
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const u32x4 xv = xs[lane + 64 * j];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_fdot2(as_h2(wv[r][j][e]), as_h2(xv[e]), acc, false);
        }
        const float sum = wave_sum(acc);
        if (lane == 0 && nb + r < N) yb[n0 + nb + r] = __float2half(sum);
    }
}

// Tile of workgroup x of n when w is stored [K][N]: workgroups go to the 8 XCDs in turn,
// and tiles narrower than a 128-byte line share lines with their neighbours, so each XCD
// (one L2) takes a run of neighbouring tiles.
__device__ __forceinline__ uint32_t xcd_tile(uint32_t x, uint32_t n) {
    const uint32_t d = x & 7, per = n >> 3, rem = n & 7;
    return d * per + min(d, rem) + (x >> 3);
}

// --- GEMV, w stored [K][N_full] --------------------------------------------------
// Workgroup = 8 CW columns x all of K: a lane takes 8 columns (16 bytes) of rows
// k = (64 / CW) wave + lane / CW, so a load instruction covers 64 / CW rows, and every lane
// keeps 4 or 8 rows in flight (16 waves: 128 KiB per workgroup at 8); the k lanes' sums meet
// by DPP and row swaps, the waves' in LDS. Needs N >= 8 (the last chunk is moved back to
// end at column N; columns computed twice get the same value), so a window of fewer columns
// is computed in one of 8 and only columns [lo, lo + cnt) of it are stored. CW = 4 where that
// grid covers the CUs, else 2 (twice the workgroups; 1 x 2560 x 9728: 20 / 17.9 us).
// Bound: w's bytes; one thread per column walked K serially on N / 256 workgroups before
// (1 x 3072 x 1024: 131.9 -> 4.2 us a call; 1 x 2560 x 9728: 2.8 TB/s).
template <int MR, int CW>
__global__ __launch_bounds__(1024) void gemv_kn_kernel(const __half* __restrict__ a,
                                                       const __half* __restrict__ w,
                                                       __half* __restrict__ y, uint32_t K,
                                                       uint32_t N_full, uint32_t n0, uint32_t N, uint32_t lo,
                                                       uint32_t cnt, int t0) {
    constexpr int UMAX = MR <= 2 ? 8 : 4;              // rows in flight per lane
    constexpr uint32_t KR = 64 / CW, PASS = 16 * KR;   // k rows per wave and per workgroup pass
    __shared__ __align__(16) float red[16][MR][8 * CW];
    const uint32_t bb = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t c0 = xcd_tile(blockIdx.x, gridDim.x) * (8 * CW);
    const __half* ab = a + (size_t)bb * MR * K;
    const __half* wb = w + (size_t)bb * K * N_full + n0 + min(c0 + 8 * (lane % CW), N - 8);
    float acc[MR][8];
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[m][e] = 0.0f;
    const uint32_t as = t0 ? MR : 1u, am = t0 ? 1u : K;   // strides of a along k and m
    const uint32_t kl = wave * KR + lane / CW;
    auto passes = [&](uint32_t k0, auto count, auto edge) __attribute__((always_inline)) {   // U passes from k0 on
        constexpr int U = decltype(count)::value;
        u32x4 wv[U];
        _Float16 av[U][MR];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t k = decltype(edge)::value ? min(k0 + PASS * u, K - 1) : k0 + PASS * u;
            wv[u] = *reinterpret_cast<const u32x4_u*>(wb + (size_t)k * N_full);
#pragma unroll
            for (int m = 0; m < MR; ++m) av[u][m] = __builtin_bit_cast(_Float16, ab[(size_t)k * as + (size_t)m * am]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if constexpr (decltype(edge)::value) {   // rows past K count as zero (a branch would sink the loads into it)
                const bool in = k0 + PASS * u < K;
#pragma unroll
                for (int e = 0; e < 4; ++e) wv[u][e] = in ? wv[u][e] : 0u;
#pragma unroll
                for (int m = 0; m < MR; ++m) av[u][m] = in ? av[u][m] : (_Float16)0.0f;
            }
#pragma unroll
            for (int m = 0; m < MR; ++m)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const h2_t h = as_h2(wv[u][e]);
                    acc[m][2 * e] = __builtin_fmaf((float)av[u][m], (float)h[0], acc[m][2 * e]);
                    acc[m][2 * e + 1] = __builtin_fmaf((float)av[u][m], (float)h[1], acc[m][2 * e + 1]);
                }
        }
    };
    uint32_t kb = 0;
    using Four = std::integral_constant<int, 4>;
    for (; kb + PASS * UMAX <= K; kb += PASS * UMAX) passes(kb + kl, std::integral_constant<int, UMAX>{}, std::false_type{});
    if (UMAX > 4 && kb + PASS * 4 <= K) {
        passes(kb + kl, Four{}, std::false_type{});
        kb += PASS * 4;
    }
    if (kb < K) passes(kb + kl, Four{}, std::true_type{});
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int e = 0; e < 8; ++e) {   // lanes l, l + CW, ... of each 16 (row rotations), then the rows
            float v = acc[m][e];
            if constexpr (CW == 2) v += dev::dpp<0x122>(v);
            v += dev::dpp<0x124>(v);
            v += dev::dpp<0x128>(v);
            acc[m][e] = dev::cross_row_sum(v);
        }
    if (lane < CW)
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int e = 0; e < 8; ++e) red[wave][m][8 * lane + e] = acc[m][e];
    __syncthreads();
    if (tid < 8 * CW * MR) {
        const uint32_t m = tid / (8 * CW), j = tid % (8 * CW);
        float v = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) v += red[i][m][j];
        const uint32_t col = min(c0 + (j & ~7u), N - 8) + (j & 7);
        if (col - lo < cnt) y[((size_t)bb * MR + m) * N_full + n0 + col] = __float2half(v);
    }
}

// The same for short K: one column per thread, K in order.
template <int MR>
__global__ __launch_bounds__(256) void gemv_col_kernel(const __half* __restrict__ a, const __half* __restrict__ w,
                                                       __half* __restrict__ y, uint32_t K, uint32_t N_full, uint32_t n0,
                                                       uint32_t N, int t0) {
    const uint32_t bb = blockIdx.y, n = blockIdx.x * 256 + threadIdx.x;
    if (n >= N) return;
    const __half* ab = a + (size_t)bb * MR * K;
    const __half* wb = w + (size_t)bb * K * N_full + n0 + n;
    const uint32_t as = t0 ? MR : 1u, am = t0 ? 1u : K;   // strides of a along k and m
    float acc[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[m] = 0.0f;
#pragma unroll 8
    for (uint32_t k = 0; k < K; ++k) {
        const float wv = __half2float(wb[(size_t)k * N_full]);
#pragma unroll
        for (int m = 0; m < MR; ++m)
            acc[m] = __builtin_fmaf(__half2float(ab[(size_t)k * as + (size_t)m * am]), wv, acc[m]);
    }
#pragma unroll
    for (int m = 0; m < MR; ++m) y[((size_t)bb * MR + m) * N_full + n0 + n] = __float2half(acc[m]);
}

// --- MFMA GEMM ---------------------------------------------------------------------
// Workgroup tile BM x BN, K step BK; WM x WN waves over the tile, times KW that split the
// step's 16-deep sub-steps (small grids: more waves per output, summed in LDS at the end).
// An operand stored along k ([M,K], or w [N,K]) is staged row-major at a stride of BK + 8
// and read as 16-byte fragments; one stored across ([K,M], or w [K,N]) is staged in memory
// order and read through ds_read_b64_tr_b16, whose 16-lane groups each take 4 k rows x 16
// columns (row strides of 16 or 48 dwords mod 64: the 4 rows of a read fall in distinct
// banks). Loads are 16 bytes at any element alignment, PD steps ahead in registers,
// unconditional with clamped rows; across-stored chunks past the last column are moved
// back to end there (their columns are computed twice, with the same bits). Operands whose
// stored rows hold fewer than 8 elements go element by element, zero past the edge.
// Bound: below one round of the CUs the K loop's latency (0.27 us per step of 64 at 64 x 64),
// then LDS (512 x 3072 x 1024, 384 tiles of 64 x 64: 73 % of a busy CU's cycles, L1 42 %, MFMA
// 16 %, VALU 13 %), and on large grids LDS reads and MFMA (1024 x 4096 x 4096: 49 us, 700
// TFLOP/s). 512 x 3072 x 1024: 123.8 -> 11.0 us against 64 x 64 tiles filled by single elements
// with two barriers per 32.
__device__ __forceinline__ uint2 lds_read_tr16(const _Float16* p) {
    const s4_t r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s4_t*)(const_cast<_Float16*>(p)));
    return __builtin_bit_cast(uint2, r);
}

// One operand's tile: R rows (of A) or columns (of W) by BK, NTH threads.
template <int R, int BK, int NTH, bool KMAJ>
struct Tile {
    static constexpr int kStride = KMAJ ? BK + 8 : R == 32 ? 32 : R + 32;   // halves
    static constexpr int kSize = KMAJ ? R * kStride : BK * kStride;
    static constexpr int CH = R * BK / 8 / NTH;   // 16-byte chunks per thread
    static_assert(CH >= 1 && R * BK / 8 % NTH == 0, "whole chunks per thread");
    const __half* base;
    uint32_t r0, rows, ld, K;   // first row, row count, stride, K
    bool narrow;                // rows as stored hold fewer than 8 elements
    uint32_t tid;

    // Start of the chunk at tile row 8 c (across-stored): whole chunks inside [0, rows).
    __device__ __forceinline__ uint32_t chunk0(uint32_t c) const {
        return rows < 8 ? r0 + 8 * c : min(r0 + 8 * c, rows - 8);
    }
    // Row (column) that tile row j stands for.
    __device__ __forceinline__ uint32_t row_of(uint32_t j) const { return KMAJ ? r0 + j : chunk0(j >> 3) + (j & 7); }

    __device__ __forceinline__ void load(u32x4 (&v)[CH], uint32_t k0) const {
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const uint32_t id = tid + NTH * i;
            if constexpr (KMAJ)
                v[i] = *reinterpret_cast<const u32x4_u*>(base + (size_t)min(r0 + id / (BK / 8), rows - 1) * ld + k0 +
                                                         id % (BK / 8) * 8);
            else
                v[i] = *reinterpret_cast<const u32x4_u*>(base + (size_t)(k0 + id / (R / 8)) * ld + chunk0(id % (R / 8)));
        }
    }
    // The partial K step: a chunk along k that crosses K is loaded ending there and shifted
    // into place (by K % 8, the same for every row), zeros after it.
    __device__ __forceinline__ void load_tail(u32x4 (&v)[CH], uint32_t k0) const {
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const uint32_t id = tid + NTH * i;
            if constexpr (KMAJ) {
                const uint32_t k = k0 + id % (BK / 8) * 8;
                const u32x4 x = *reinterpret_cast<const u32x4_u*>(base + (size_t)min(r0 + id / (BK / 8), rows - 1) * ld +
                                                                  min(k, K - 8));
                const uint32_t sh = 8 - K % 8;   // 8: nothing crosses
                uint32_t t[8];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    t[e] = sh & 1 ? __builtin_amdgcn_alignbyte(e < 3 ? x[e + 1 < 4 ? e + 1 : 3] : 0u, x[e], 2) : x[e];
#pragma unroll
                for (int e = 4; e < 8; ++e) t[e] = 0u;
                if (sh & 2)
#pragma unroll
                    for (int e = 0; e < 7; ++e) t[e] = t[e + 1];
                if (sh & 4)
#pragma unroll
                    for (int e = 0; e < 6; ++e) t[e] = t[e + 2];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[i][e] = k + 8 <= K ? x[e] : k < K ? t[e] : 0u;
            } else {
                const uint32_t k = k0 + id / (R / 8);
                v[i] = *reinterpret_cast<const u32x4_u*>(base + (size_t)min(k, K - 1) * ld + chunk0(id % (R / 8)));
#pragma unroll
                for (int e = 0; e < 4; ++e) v[i][e] = k < K ? v[i][e] : 0u;
            }
        }
    }
    // The same element by element, for operands with fewer than 8 elements in a row.
    __device__ __forceinline__ void load_edge(u32x4 (&v)[CH], uint32_t k0) const {
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const uint32_t id = tid + NTH * i;
            uint16_t h[8];
#pragma unroll
            for (uint32_t e = 0; e < 8; ++e) {
                const uint32_t k = KMAJ ? k0 + id % (BK / 8) * 8 + e : k0 + id / (R / 8);
                const uint32_t r = KMAJ ? min(r0 + id / (BK / 8), rows - 1) : chunk0(id % (R / 8)) + e;
                const uint32_t kc = min(k, K - 1), rc = min(r, rows - 1);   // loaded in any case: no branch to wait at
                h[e] = __builtin_bit_cast(uint16_t, base[KMAJ ? (size_t)rc * ld + kc : (size_t)kc * ld + rc]);
                if (k >= K || r >= rows) h[e] = 0;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[i][e] = h[2 * e] | (uint32_t)h[2 * e + 1] << 16;
        }
    }
    __device__ __forceinline__ void store(const u32x4 (&v)[CH], _Float16* s) const {
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const uint32_t id = tid + NTH * i;
            const uint32_t o = KMAJ ? id / (BK / 8) * kStride + id % (BK / 8) * 8 : id / (R / 8) * kStride + id % (R / 8) * 8;
            *reinterpret_cast<u32x4*>(s + o) = v[i];
        }
    }
    // MFMA fragment: rows rb .. rb + 31, k = 16 kk + 8 (lane / 32) .. + 7.
    static __device__ __forceinline__ h8_t frag(const _Float16* s, uint32_t rb, uint32_t kk, uint32_t lane) {
        if constexpr (KMAJ) return *reinterpret_cast<const h8_t*>(s + (rb + (lane & 31)) * kStride + kk * 16 + 8 * (lane >> 5));
        const uint32_t g = lane >> 4, i = lane & 15;
        const _Float16* p = s + (kk * 16 + 8 * (g >> 1) + (i >> 2)) * kStride + rb + 16 * (g & 1) + 4 * (i & 3);
        const uint2 lo = lds_read_tr16(p), hi = lds_read_tr16(p + 4 * kStride);
        return __builtin_bit_cast(h8_t, u32x4{lo.x, lo.y, hi.x, hi.y});
    }
};

template <int BM, int BN, int WM, int WN, int KW, int BK, int PD, bool AK, bool BKM>
__global__ __launch_bounds__(64 * WM * WN * KW) void gemm_f16_kernel(const __half* __restrict__ a,
                                                                     const __half* __restrict__ w,
                                                                     __half* __restrict__ y, uint32_t M, uint32_t K,
                                                                     uint32_t N_full, uint32_t n0, uint32_t N) {
    constexpr int NTH = 64 * WM * WN * KW, WI = BM / 32 / WM, WJ = BN / 32 / WN, KS = BK / 16 / KW;
    using TA = Tile<BM, BK, NTH, AK>;
    using TB = Tile<BN, BK, NTH, BKM>;
    constexpr int kBuf = TA::kSize + TB::kSize;
    static_assert(KW == 1 || (size_t)NTH * WI * WJ * 64 <= (size_t)kBuf * 4, "sums fit the staging buffers");
    __shared__ __align__(16) _Float16 lds[2][kBuf];
    const uint32_t bb = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t kw = wave / (WM * WN), wm = wave % (WM * WN) / WN, wn = wave % WN;
    const __half* wb = w + (size_t)bb * K * N_full + (BKM ? (size_t)n0 * K : (size_t)n0);
    const TA ta{a + (size_t)bb * M * K, blockIdx.y * BM, M, AK ? K : M, K, (AK ? K : M) < 8, tid};
    const TB tb{wb, (BKM ? blockIdx.x : xcd_tile(blockIdx.x, gridDim.x)) * BN, N, BKM ? K : N_full, K, (BKM ? K : N) < 8, tid};

    f16x_t acc[WI][WJ];
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
        for (int j = 0; j < WJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    auto mfma = [&](int buf) __attribute__((always_inline)) {
        const _Float16 *sa = lds[buf], *sb = lds[buf] + TA::kSize;
#pragma unroll
        for (int q = 0; q < KS; ++q) {
            const uint32_t kk = kw * KS + q;
            h8_t af[WI], bf[WJ];
#pragma unroll
            for (int i = 0; i < WI; ++i) af[i] = TA::frag(sa, (wm * WI + i) * 32, kk, lane);
#pragma unroll
            for (int j = 0; j < WJ; ++j) bf[j] = TB::frag(sb, (wn * WJ + j) * 32, kk, lane);
#pragma unroll
            for (int i = 0; i < WI; ++i)
#pragma unroll
                for (int j = 0; j < WJ; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
    };

    const bool narrow = ta.narrow || tb.narrow;
    const uint32_t nfull = narrow ? 0u : K / BK;
    if (nfull) {
        u32x4 ra[PD][TA::CH], rb[PD][TB::CH];
        const uint32_t last = nfull - 1;
        auto load = [&](int st, uint32_t kb) __attribute__((always_inline)) {
            ta.load(ra[st], kb * BK);
            tb.load(rb[st], kb * BK);
        };
        auto stage = [&](int st, int buf) __attribute__((always_inline)) {
            ta.store(ra[st], lds[buf]);
            tb.store(rb[st], lds[buf] + TA::kSize);
        };
        // Step kb: MFMAs on buffer kb % 2 while step kb + PD loads into register stage kb % PD
        // (stored to LDS during step kb - 1) and stage kb + 1 goes to the other buffer. Past
        // the end the last step is loaded and stored again, unread.
        auto step = [&](int u, uint32_t kb) __attribute__((always_inline)) {
            load(u % PD, min(kb + PD, last));
            __builtin_amdgcn_sched_barrier(0);
            mfma(u % 2);
            stage((u + 1) % PD, (u + 1) % 2);
            __syncthreads();
        };
#pragma unroll
        for (int i = 0; i < PD; ++i) load(i, min((uint32_t)i, last));
        stage(0, 0);
        __syncthreads();
        uint32_t kb = 0;
#pragma unroll 1
        for (; kb + PD <= nfull; kb += PD) {
#pragma unroll
            for (int u = 0; u < PD; ++u) step(u, kb + u);
        }
#pragma unroll
        for (int u = 0; u < PD - 1; ++u)
            if (kb + u < nfull) step(u, kb + u);
    }
    for (uint32_t k0 = nfull * BK; k0 < K; k0 += BK) {
        u32x4 ra[TA::CH], rb[TB::CH];
        if (narrow) {
            ta.load_edge(ra, k0);
            tb.load_edge(rb, k0);
        } else {
            ta.load_tail(ra, k0);
            tb.load_tail(rb, k0);
        }
        ta.store(ra, lds[0]);
        tb.store(rb, lds[0] + TA::kSize);
        __syncthreads();
        mfma(0);
        __syncthreads();
    }

    // Accumulator layout (32x32): lane l, reg r -> col l%32, row 8*(r/4) + 4*(l/32) + r%4.
    __half* yb = y + (size_t)bb * M * N_full + n0;
    auto put = [&](int i, int j, int r4, const float (&v)[4]) __attribute__((always_inline)) {
        const uint32_t col = tb.row_of((wn * WJ + j) * 32 + (lane & 31));
        if (col >= N) return;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t row = ta.row_of((wm * WI + i) * 32 + 8 * r4 + 4 * (lane >> 5) + e);
            if (row < M) yb[(size_t)row * N_full + col] = __float2half(v[e]);
        }
    };
    if constexpr (KW == 1) {
#pragma unroll
        for (int i = 0; i < WI; ++i)
#pragma unroll
            for (int j = 0; j < WJ; ++j)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    const float v[4] = {acc[i][j][4 * r4], acc[i][j][4 * r4 + 1], acc[i][j][4 * r4 + 2], acc[i][j][4 * r4 + 3]};
                    put(i, j, r4, v);
                }
    } else {
        float* red = reinterpret_cast<float*>(&lds[0][0]);   // [wave][tile][quarter][lane][4]
        __syncthreads();
#pragma unroll
        for (int t = 0; t < WI * WJ; ++t)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                *reinterpret_cast<float4*>(&red[((wave * WI * WJ + t) * 4 + r4) * 256 + lane * 4]) =
                    make_float4(acc[t / WJ][t % WJ][4 * r4], acc[t / WJ][t % WJ][4 * r4 + 1], acc[t / WJ][t % WJ][4 * r4 + 2],
                                acc[t / WJ][t % WJ][4 * r4 + 3]);
        __syncthreads();
        for (uint32_t q = kw; q < WI * WJ * 4; q += KW) {
            float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < KW; ++k) {
                const float4 x = *reinterpret_cast<const float4*>(
                    &red[((k * WM * WN + wm * WN + wn) * WI * WJ * 4 + q) * 256 + lane * 4]);
                v[0] += x.x; v[1] += x.y; v[2] += x.z; v[3] += x.w;
            }
            put(q / 4 / WJ, q / 4 % WJ, q % 4, v);
        }
    }
}

template <bool AK, bool BKM>
hipError_t gemm_f16_launch(const __half* a, const __half* w, __half* y, uint32_t M, uint32_t K, uint32_t N_full,
                           uint32_t n0, uint32_t N, uint32_t Bn, hipStream_t st) {
    auto go = [&](auto kern, uint32_t bm, uint32_t bn, uint32_t nth) {
        hipLaunchKernelGGL(kern, dim3((N + bn - 1) / bn, (M + bm - 1) / bm, Bn), dim3(nth), 0, st, a, w, y, M, K, N_full,
                           n0, N);
        return hipGetLastError();
    };
    // K of one short step: the same order as the 64- and 128-square tiles, half their staging
    // (5 x 32768 x 4 with steps of 64: 4.1 us, now 3.4).
    if (K <= 32) return go(gemm_f16_kernel<64, 64, 2, 2, 1, 32, 2, AK, BKM>, 64, 64, 256);
    const size_t cus = (size_t)device_cu_count();
    // Tile by the grid's rounds. A round of one workgroup per CU took 2.4 / 4.2 / 11.5 us per
    // 1024 of K with 32 / 64 / 128-square tiles. Measured with the three, us (M x N x K):
    // 256 x 1024 x 1024 4.5 / 6.9 / 15.1; 512 x 3072 x 1024 17.0 / 11.0 / 15.7; 117 x 3760 x 3072
    // 31 / 15.7 / 36; 1024 x 4096 x 4096 194 / 64 / 49.
    // The 32-square tile sums K in another order than the other two, so whether it runs is the
    // whole product's choice and not a window's (128 x 1024 of 3072 x 1024: 4.8 us with it,
    // 7.3 without): a SPLIT chunk has the whole product's bits.
    auto cost = [&](size_t b, uint32_t n, double us) {
        return us * (double)(((M + b - 1) / b * ((n + b - 1) / b) * Bn + cus - 1) / cus);
    };
    if (cost(64, N_full, 4.2) < cost(32, N_full, 2.4) || cost(128, N_full, 11.5) < cost(32, N_full, 2.4)) {
        if (cost(128, N, 11.5) < cost(64, N, 4.2))
            return go(gemm_f16_kernel<128, 128, 2, 2, 1, 64, 2, AK, BKM>, 128, 128, 256);
        return go(gemm_f16_kernel<64, 64, 2, 2, 1, 64, 4, AK, BKM>, 64, 64, 256);
    }
    return go(gemm_f16_kernel<32, 32, 1, 1, 8, 128, 4, AK, BKM>, 32, 32, 512);
}

}  // namespace

hipError_t launch_matmul_f16(const __half* a, const __half* w, __half* y, uint32_t M, uint32_t K,
                             uint32_t N_full, uint32_t n0, uint32_t N, bool t0, bool t1,
                             uint32_t Bn, hipStream_t st) {
    if (!M || !N || !Bn) return hipSuccess;
    const bool batched = Bn > 1;
    const bool aligned = ((uintptr_t)a % 16 == 0) && ((uintptr_t)w % 16 == 0) && K % 8 == 0;
    if (M <= 4 && t1 && !t0 && aligned && (size_t)M * K * 2 <= 65536) {
        const size_t lds = (size_t)M * K * 2;
        dim3 grid((N + 15) / 16, Bn);
        if (M == 1 && K % 512 == 0 && K / 512 <= 8) {
            switch (K / 512) {
            case 1: hipLaunchKernelGGL(gemv_nk_pre_kernel<1>, grid, dim3(256), lds, st, a, w, y, K, N_full, n0, N); break;
            case 2: hipLaunchKernelGGL(gemv_nk_pre_kernel<2>, grid, dim3(256), lds, st, a, w, y, K, N_full, n0, N); break;
            case 3: hipLaunchKernelGGL(gemv_nk_pre_kernel<3>, grid, dim3(256), lds, st, a, w, y, K, N_full, n0, N); break;
            case 4: hipLaunchKernelGGL(gemv_nk_pre_kernel<4>, grid, dim3(256), lds, st, a, w, y, K, N_full, n0, N); break;
            case 5: hipLaunchKernelGGL(gemv_nk_pre_kernel<5>, grid, dim3(256), lds, st, a, w, y, K, N_full, n0, N); break;
            case 6: hipLaunchKernelGGL(gemv_nk_pre_kernel<6>, grid, dim3(256), lds, st, a, w, y, K, N_full, n0, N); break;
            case 7: hipLaunchKernelGGL(gemv_nk_pre_kernel<7>, grid, dim3(256), lds, st, a, w, y, K, N_full, n0, N); break;
            default: hipLaunchKernelGGL(gemv_nk_pre_kernel<8>, grid, dim3(256), lds, st, a, w, y, K, N_full, n0, N); break;
            }
            return hipGetLastError();
        }
        switch (M) {
        case 1: hipLaunchKernelGGL(gemv_nk_kernel<1>, grid, dim3(256), lds, st, a, w, y, K, N_full, n0, N, M); break;
        case 2: hipLaunchKernelGGL(gemv_nk_kernel<2>, grid, dim3(256), lds, st, a, w, y, K, N_full, n0, N, M); break;
        case 3: hipLaunchKernelGGL(gemv_nk_kernel<3>, grid, dim3(256), lds, st, a, w, y, K, N_full, n0, N, M); break;
        default: hipLaunchKernelGGL(gemv_nk_kernel<4>, grid, dim3(256), lds, st, a, w, y, K, N_full, n0, N, M); break;
        }
        return hipGetLastError();
    }
    const int ta = t0 && !batched;
    // Short K: a workgroup of the split form costs the same whatever K, a column per thread about
    // 0.1 us per k and row of a. Measured, us, split / one column per thread: 1 x 4096 x 8 3.1 /
    // 2.7, x 16 3.1 / 3.6; 4 x 4096 x 12 6.1 / 6.1; 1 x 32768 x 32 5.9 / 5.4, 4 x 32768 x 48 19.5 /
    // 18.7 (1, 2 and 4 split workgroups per CU).
    const uint64_t per_cu = ((uint64_t)(N_full + 31) / 32 * Bn + device_cu_count() - 1) / device_cu_count();
    if (M <= 4 && !t1 && K <= std::min<uint64_t>(128, 13 + (M % 2 ? 7 : 11) * (per_cu - 1))) {
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3((N + 255) / 256, Bn), dim3(256), 0, st, a, w, y, K, N_full, n0, N, ta);
            return hipGetLastError();
        };
        return M == 1 ? go(gemv_col_kernel<1>) : M == 2 ? go(gemv_col_kernel<2>) : M == 3 ? go(gemv_col_kernel<3>) : go(gemv_col_kernel<4>);
    }
    if (M <= 4 && !t1 && N_full >= 8) {
        const uint32_t nw = std::max(N, 8u), n0w = std::min(n0, N_full - nw);   // window computed
        auto go = [&](auto kern, uint32_t cols) {
            hipLaunchKernelGGL(kern, dim3((nw + cols - 1) / cols, Bn), dim3(1024), 0, st, a, w, y, K, N_full, n0w, nw,
                               n0 - n0w, N, ta);
            return hipGetLastError();
        };
        // 16-column workgroups where 32-column ones leave CUs idle and K fills their passes; rows
        // off 16-byte boundaries make 32-byte pieces cross lines, which only long K makes up for
        // (1 x 3073 x 1024: 4.8 us with 32 columns, 6.9 with 16; 1 x 2561 x 9728: 26.0 / 24.0;
        // 1 x 2560 x 9728: 20 / 18). The two order K differently, so the whole product decides
        // here too, not the window.
        const bool al = N_full % 8 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0;
        const bool wide = (size_t)((N_full + 31) / 32) * Bn >= (size_t)device_cu_count() || K < (al ? 1024u : 2048u);
        switch (M) {
        case 1: return wide ? go(gemv_kn_kernel<1, 4>, 32) : go(gemv_kn_kernel<1, 2>, 16);
        case 2: return wide ? go(gemv_kn_kernel<2, 4>, 32) : go(gemv_kn_kernel<2, 2>, 16);
        case 3: return wide ? go(gemv_kn_kernel<3, 4>, 32) : go(gemv_kn_kernel<3, 2>, 16);
        default: return wide ? go(gemv_kn_kernel<4, 4>, 32) : go(gemv_kn_kernel<4, 2>, 16);
        }
    }
    const bool ak = !(t0 && !batched);   // the reference's batched form ignores t0
    if (ak) return t1 ? gemm_f16_launch<true, true>(a, w, y, M, K, N_full, n0, N, Bn, st)
                      : gemm_f16_launch<true, false>(a, w, y, M, K, N_full, n0, N, Bn, st);
    return t1 ? gemm_f16_launch<false, true>(a, w, y, M, K, N_full, n0, N, Bn, st)
              : gemm_f16_launch<false, false>(a, w, y, M, K, N_full, n0, N, Bn, st);
}

}  // namespace gehtp
