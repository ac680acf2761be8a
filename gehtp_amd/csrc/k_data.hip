// k_data.hip — crouton16_row4 surfaces, OP_MATMUL_W4A16 (opcode 1), OP_RMSNORM_F16
// (opcode 2) and the runlist's data-movement / reduction ops, for gfx950.
//
// crouton16_row4 (kernels/src/runtime/gemm_dispatch.c:38-72): element (r, c) of a
// rows x cols u16 surface sits at
//   chunk = ((phase * n_kt + kt) * n_m32 + g) * 2 + rp,   pos = 64 * chunk + 2 * (c % 32) + (r & 1)
// with g = r / 32, phase = (r % 32) / 4, rp = (r % 4) / 2, kt = c / 32.
#include "kernels.h"

#include <cmath>

namespace gehtp {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ size_t crouton_pos(uint32_t r, uint32_t c, uint32_t n_m32, uint32_t n_kt) {
    const uint32_t rr = r & 31u;
    const size_t chunk = ((size_t)((rr >> 2) * n_kt + (c >> 5)) * n_m32 + (r >> 5)) * 2 + ((rr >> 1) & 1u);
    return chunk * 64 + 2 * (c & 31u) + (r & 1u);
}

// One thread per surface pair (two rows of one column): surface words are written in
// order, the linear side reads two rows.
__global__ void crouton_encode_kernel(const uint16_t* __restrict__ lin, uint32_t* __restrict__ surf,
                                      uint32_t rows, uint32_t cols) {
    const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t n_m32 = rows >> 5, n_kt = cols >> 5;
    if (q >= (size_t)rows * cols / 2) return;
    const uint32_t ci = (uint32_t)(q & 31u);
    size_t rest = q >> 5;
    const uint32_t rp = (uint32_t)(rest & 1u);
    rest >>= 1;
    const uint32_t g = (uint32_t)(rest % n_m32);
    rest /= n_m32;
    const uint32_t kt = (uint32_t)(rest % n_kt), phase = (uint32_t)(rest / n_kt);
    const uint32_t row0 = g * 32 + phase * 4 + rp * 2, c = kt * 32 + ci;
    surf[q] = (uint32_t)lin[(size_t)row0 * cols + c] | ((uint32_t)lin[(size_t)(row0 + 1) * cols + c] << 16);
}

__global__ void crouton_decode_kernel(const uint32_t* __restrict__ surf, uint16_t* __restrict__ lin,
                                      uint32_t rows, uint32_t cols) {
    const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t n_m32 = rows >> 5, n_kt = cols >> 5;
    if (q >= (size_t)rows * cols / 2) return;
    const uint32_t ci = (uint32_t)(q & 31u);
    size_t rest = q >> 5;
    const uint32_t rp = (uint32_t)(rest & 1u);
    rest >>= 1;
    const uint32_t g = (uint32_t)(rest % n_m32);
    rest /= n_m32;
    const uint32_t kt = (uint32_t)(rest % n_kt), phase = (uint32_t)(rest / n_kt);
    const uint32_t row0 = g * 32 + phase * 4 + rp * 2, c = kt * 32 + ci;
    const uint32_t v = surf[q];
    lin[(size_t)row0 * cols + c] = (uint16_t)(v & 0xFFFFu);
    lin[(size_t)(row0 + 1) * cols + c] = (uint16_t)(v >> 16);
}

// ---------------------------------------------------------------------------
// OP_MATMUL_W4A16: Y[m,n] = clip(nearest((sum_k (A[m,k]-32768) W[k,n]) / 7) + 32768), in
// whole numbers on the matrix cores (v_mfma_i32_32x32x32_i8). A u16 activation is two
// signed bytes once its bytes' top bits are flipped (word ^ 0x80808080): A - 32768 =
// 256 hi + lo + 128, so the sum is 256 sum(hi W) + sum(lo W) + 128 sum(W), the last from
// v_dot4 on the weight words. A stored nibble (q + 8) ^ 8 is q in two's complement; left in
// a byte's top half it is 16 q, so 8 weights unpack with a shift and two xor-ands (even k's
// in one word, odd ones in the other; A's columns are staged in that order), and the sums,
// all multiples of 16, are shifted down exactly.
// Workgroup tile 32 RT x 32 NT, its K steps (64 = two 32-column blocks of the surface)
// split over WV = 8 waves in contiguous ranges (one wave for short K on large grids): at
// M = 256, K = N = 2560 (160 tiles of 64 x 64) a serial K loop is latency. Each wave stages its own A block in LDS
// (256 RT-byte runs of the surface in, byte planes out), so its loop needs no barrier; W
// goes from memory to the B operand. The waves' sums meet in LDS. int32 holds the tile's
// whole sums up to 8064 columns (8064 * 32896 * 8 < 2^31); longer K runs in such chunks with
// int64 totals between them.
// Bound: no one unit. Counters at 1024 x 4096 x 4096 (64 x 64 tiles): VALU issue 51 % of the
// CU's cycles (the byte planes: 24 instructions per 16 u16 pairs), LDS 41 %, L1 55 %, MFMA
// 24 %. 256 x 2560 x 2560: 134.9 -> 12.5 us per call (the 64 x 64 v_dot2 tiles it replaces, one wave
// row per 16 columns and a barrier per 32 columns, against this).
constexpr uint32_t kWaChunk = 126;   // K steps of an int32 chunk: 8064 columns

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32_a2 __attribute__((aligned(2)));   // surfaces need only be u16-aligned on output

template <typename T>   // nearest of s / 7 (no ties), clipped to a u16 around the zero point
__device__ __forceinline__ uint32_t w4a16_out(T s) {
    const T y = (s >= 0 ? (s + 3) / 7 : -((-s + 3) / 7)) + 32768;
    return y < 0 ? 0u : y > 65535 ? 65535u : (uint32_t)y;
}

template <int RT, int NT, int MINW, uint32_t WV>
__global__ __launch_bounds__(64 * WV, MINW) void w4a16_gemm_kernel(const uint16_t* __restrict__ act,
                                                                   const uint8_t* __restrict__ w,
                                                                   uint16_t* __restrict__ out, uint32_t M,
                                                                   uint32_t K, uint32_t N) {
    // A staged plane: rows of 64 bytes at a stride of 80 (operand reads of 16 rows and
    // stores of every second row then spread over all banks), 128 bytes between row tiles.
    constexpr uint32_t RS = 80, TS = 32 * RS + 128, PLANE = RT * TS, NU = 2 * RT;
    constexpr uint32_t CS = 32 * RT + 4, TILE = 32 * CS;   // a wave's sums of one n tile: [column][row], padded
    constexpr uint32_t NQ = RT * 512 / (64 * WV);          // surface words per thread and n tile
    constexpr uint32_t WLDS = 2 * PLANE > TILE * 4 ? 2 * PLANE : TILE * 4;
    __shared__ __align__(16) uint8_t lds[WV * WLDS];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = lane >> 5, l32 = lane & 31;
    const uint32_t n_m32 = M >> 5, n_kt = K >> 5, nsteps = (n_kt + 1) / 2;
    const uint32_t nt = (N / 32 + NT - 1) / NT, g0 = (blockIdx.x / nt) * RT, n0 = (blockIdx.x % nt) * (32 * NT);
    uint8_t* st = lds + wave * WLDS;

    // A: a unit is 8 columns x one row pair (32 contiguous bytes); a phase's chunks of the
    // tile are 256 RT contiguous bytes per block. Unit 64 i + lane = (phase, kt, group,
    // pair, 8 columns).
    const uint32_t urp = (lane >> 2) & 1, uoct = lane & 3;
    const uint32_t ugl = RT == 2 ? (lane >> 3) & 1 : 0, ukt = RT == 2 ? (lane >> 4) & 1 : (lane >> 3) & 1;
    const uint32_t uph = RT == 2 ? lane >> 5 : lane >> 4;   // + (8 / NU) i
    const uint32_t ug = min(g0 + ugl, n_m32 - 1);           // rows past M repeat the last group (not stored)
    const size_t kt_bytes = (size_t)n_m32 * 256, ph_bytes = kt_bytes * n_kt;
    const uint8_t* abase = reinterpret_cast<const uint8_t*>(act) + uph * ph_bytes + (size_t)ug * 256 + urp * 128 + uoct * 32;
    uint8_t* sta = st + ugl * TS + (uph * 4 + urp * 2) * RS + ukt * 32 + uoct * 8;
    const uint8_t* wbase[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) wbase[j] = w + (size_t)min(n0 + 32 * j + l32, N - 1) * (K / 2);
    u32x4 ra[NU][2], rw[NT];
    auto load = [&](uint32_t s) __attribute__((always_inline)) {
        const uint32_t kw = min(2 * s + half, n_kt - 1);
#pragma unroll
        for (int j = 0; j < NT; ++j) rw[j] = *reinterpret_cast<const u32x4*>(wbase[j] + kw * 16);
        const uint8_t* p = abase + min(2 * s + ukt, n_kt - 1) * kt_bytes;
#pragma unroll
        for (uint32_t i = 0; i < NU; ++i) {
            const u32x4* q = reinterpret_cast<const u32x4*>(p + i * (8 / NU) * ph_bytes);
            ra[i][0] = q[0];
            ra[i][1] = q[1];
        }
    };

    int64_t tot[NT][NQ][2];   // [n tile][word][row of the pair]
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (uint32_t e = 0; e < 2 * NQ; ++e) tot[j][e >> 1][e & 1] = 0;

    for (uint32_t c0 = 0; c0 < nsteps; c0 += kWaChunk) {
        const uint32_t cn = min(kWaChunk, nsteps - c0), per = (cn + WV - 1) / WV;
        const uint32_t s0 = c0 + min(wave * per, cn), s1 = c0 + min((wave + 1) * per, cn);
        i32x16 acc[NT][2][RT];   // [n tile][plane][row tile]
        int wsum[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            wsum[j] = 0;
#pragma unroll
            for (int e = 0; e < 2 * RT; ++e)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[j][e / RT][e % RT][r] = 0;
        }
        load(min(s0, nsteps - 1));   // loads are unconditional: a branch would drain them at its join
#pragma unroll 1
        for (uint32_t s = s0; s < s1; ++s) {
            // byte planes of this step's block, and its weights, out of the load registers
#pragma unroll
            for (uint32_t i = 0; i < NU; ++i) {
                const u32x4 a = ra[i][0] ^ 0x80808080u, b = ra[i][1] ^ 0x80808080u;
                uint32_t pl[2][2][2];   // [plane][row][even / odd columns]
#pragma unroll
                for (int o = 0; o < 2; ++o) {
                    const uint32_t t0 = __builtin_amdgcn_perm(a[o + 2], a[o], 0x05010400u);
                    const uint32_t t1 = __builtin_amdgcn_perm(b[o + 2], b[o], 0x05010400u);
                    const uint32_t t2 = __builtin_amdgcn_perm(a[o + 2], a[o], 0x07030602u);
                    const uint32_t t3 = __builtin_amdgcn_perm(b[o + 2], b[o], 0x07030602u);
                    pl[0][0][o] = __builtin_amdgcn_perm(t1, t0, 0x05040100u);
                    pl[1][0][o] = __builtin_amdgcn_perm(t1, t0, 0x07060302u);
                    pl[0][1][o] = __builtin_amdgcn_perm(t3, t2, 0x05040100u);
                    pl[1][1][o] = __builtin_amdgcn_perm(t3, t2, 0x07060302u);
                }
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int b2 = 0; b2 < 2; ++b2)
                        *reinterpret_cast<uint64_t*>(sta + p * PLANE + (i * (32 / NU) + b2) * RS) =
                            (uint64_t)pl[p][b2][1] << 32 | pl[p][b2][0];
            }
            i32x4 bop[NT][2];
            // 0: past an odd block count, the last step's second block counts as zero weights
            const uint32_t nib = 2 * s + half < n_kt ? 0xF0F0F0F0u : 0u;
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t x = rw[j][e];
                    const int ev = (int)(((x << 4) ^ 0x80808080u) & nib), od = (int)((x ^ 0x80808080u) & nib);
                    bop[j][e >> 1][2 * (e & 1)] = ev;
                    bop[j][e >> 1][2 * (e & 1) + 1] = od;
                    wsum[j] = __builtin_amdgcn_sdot4(ev, 0x01010101, wsum[j], false);
                    wsum[j] = __builtin_amdgcn_sdot4(od, 0x01010101, wsum[j], false);
                }
            load(min(s + 1, nsteps - 1));
            __builtin_amdgcn_sched_barrier(0);
            // the wave's lanes read what other lanes of it wrote: DS operations of a wave
            // complete in order, the fences keep the compiler from moving them across
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int t = 0; t < RT; ++t) {
                        const i32x4 av =
                            *reinterpret_cast<const i32x4*>(st + p * PLANE + t * TS + l32 * RS + half * 32 + q * 16);
#pragma unroll
                        for (int j = 0; j < NT; ++j)
                            acc[j][p][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, bop[j][q], acc[j][p][t], 0, 0, 0);
                    }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        // Sums over the waves, one n tile at a time: [wave][column][row]. Thread t holds
        // surface words (row pair, column) = t, t + 64 WV, ...
        int* red = reinterpret_cast<int*>(lds);
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            __syncthreads();
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int r = 0; r < 16; r += 4) {   // 256 hi + lo, without the factor 16
                    i32x4 v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = acc[j][1][t][r + e] * 16 + (acc[j][0][t][r + e] >> 4);
                    *reinterpret_cast<i32x4*>(&red[wave * TILE + l32 * CS + t * 32 + 2 * r + 4 * half]) = v;
                }
            __syncthreads();
#pragma unroll
            for (uint32_t q = 0; q < NQ; ++q) {
                const uint32_t idx = tid + 64 * WV * q, col = idx & 31, pr = idx >> 5;
                int sum[2] = {0, 0};
#pragma unroll
                for (uint32_t v = 0; v < WV; ++v) {
                    const int2 x = *reinterpret_cast<const int2*>(&red[v * TILE + col * CS + 2 * pr]);
                    sum[0] += x.x;
                    sum[1] += x.y;
                }
                tot[j][q][0] += sum[0];
                tot[j][q][1] += sum[1];
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NT; ++j) red[(j * WV + wave) * 64 + lane] = wsum[j] >> 4;   // this lane's k half of column l32
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            int ws = 0;
#pragma unroll
            for (uint32_t v = 0; v < 2 * WV; ++v) ws += red[j * WV * 64 + v * 32 + (tid & 31)];
#pragma unroll
            for (uint32_t e = 0; e < 2 * NQ; ++e) tot[j][e >> 1][e & 1] += (int64_t)ws * 128;
        }
        __syncthreads();
    }

    const uint32_t on_kt = N >> 5;
    const bool small = nsteps <= kWaChunk;   // the whole sum fits int32
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (uint32_t q = 0; q < NQ; ++q) {
            const uint32_t idx = tid + 64 * WV * q, col = idx & 31, m = g0 * 32 + 2 * (idx >> 5), kt = (n0 >> 5) + j;
            if (m >= M || kt >= on_kt) continue;
            uint32_t v[2];
#pragma unroll
            for (int b = 0; b < 2; ++b) v[b] = small ? w4a16_out((int32_t)tot[j][q][b]) : w4a16_out(tot[j][q][b]);
            const uint32_t rr = m & 31u;
            const size_t chunk = ((size_t)((rr >> 2) * on_kt + kt) * n_m32 + (m >> 5)) * 2 + ((rr >> 1) & 1u);
            *reinterpret_cast<u32_a2*>(out + chunk * 64 + 2 * col) = v[0] | (v[1] << 16);
        }
}

// OP_RMSNORM_F16 (oplist_exec.c:559-591), one wavefront per row of the crouton surface:
// x = float(u16 - 32768), squares summed in double, rms = (float)sqrt(acc/n + 1e-6),
// y = f16((x / rms) * w) row-major.
__global__ __launch_bounds__(256) void rmsnorm_crouton_kernel(const uint16_t* __restrict__ x,
                                                              const __half* __restrict__ wt,
                                                              __half* __restrict__ y, uint32_t m,
                                                              uint32_t n) {
    const uint32_t lane = threadIdx.x & 63, r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= m) return;
    const uint32_t n_m32 = m >> 5, n_kt = n >> 5;
    double acc = 0.0;
    for (uint32_t c = lane; c < n; c += 64) {
        const float xf = (float)((int32_t)x[crouton_pos(r, c, n_m32, n_kt)] - 32768);
        acc += (double)xf * (double)xf;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    const float rms = (float)sqrt(acc / (double)n + 1e-6);
    for (uint32_t c = lane; c < n; c += 64) {
        const float xf = (float)((int32_t)x[crouton_pos(r, c, n_m32, n_kt)] - 32768);
        y[(size_t)r * n + c] = __float2half(__fmul_rn(__fdiv_rn(xf, rms), __half2float(wt[c])));
    }
}

// ---------------------------------------------------------------------------
// Data movement (bit copies of f16 words) and reductions.
struct Seg4 {
    const uint16_t* x[4];
    uint32_t size[4];
};

__global__ void concat_kernel(Seg4 s, uint16_t* __restrict__ y, uint32_t n_seg, uint32_t total, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t o = i / total;
    uint32_t c = i - o * total;
    for (uint32_t k = 0; k < n_seg; ++k) {
        if (c < s.size[k]) { y[i] = s.x[k][(size_t)o * s.size[k] + c]; return; }
        c -= s.size[k];
    }
}

__global__ void split_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ y, uint32_t total,
                             uint32_t off, uint32_t size, uint32_t n) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const uint32_t o = j / size, c = j - o * size;
    y[j] = x[(size_t)o * total + off + c];
}

__global__ void pad_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ y, uint32_t outer,
                           uint32_t in_inner, uint32_t out_inner, uint32_t before, uint16_t pv) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)outer * out_inner) return;
    const uint32_t r = (uint32_t)(i / out_inner), c = (uint32_t)(i - (size_t)r * out_inner);
    y[i] = (c >= before && c < before + in_inner) ? x[(size_t)r * in_inner + (c - before)] : pv;
}

// OP_REDUCE_F16 (oplist_exec.c:1258-1299): thread per output, the reference's order.
__global__ void reduce_kernel(const __half* __restrict__ x, __half* __restrict__ y, uint32_t outer,
                              uint32_t L, uint32_t inner, uint32_t subtype) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= outer * inner) return;
    const uint32_t o = t / inner, i = t - o * inner;
    const __half* base = x + ((size_t)o * L) * inner + i;
    float acc = subtype == 2 ? -3.0e38f : subtype == 3 ? 3.0e38f : 0.0f;
    for (uint32_t l = 0; l < L; ++l) {
        const float v = __half2float(base[(size_t)l * inner]);
        if (subtype == 2) acc = v > acc ? v : acc;
        else if (subtype == 3) acc = v < acc ? v : acc;
        else acc = __fadd_rn(acc, v);
    }
    if (subtype == 1) acc = __fdiv_rn(acc, (float)L);
    y[(size_t)o * inner + i] = __float2half(acc);
}

// OP_CUMSUM_F32 (oplist_exec.c:1320-1347): thread per row, sequential f32 sum.
__global__ void cumsum_kernel(const __half* __restrict__ x, __half* __restrict__ y, uint32_t rows,
                              uint32_t n, uint32_t exclusive, uint32_t reverse) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    float acc = 0.0f;
    for (uint32_t s = 0; s < n; ++s) {
        const size_t idx = (size_t)r * n + (reverse ? n - 1 - s : s);
        const float v = __half2float(x[idx]);
        y[idx] = __float2half(exclusive ? acc : __fadd_rn(acc, v));
        acc = __fadd_rn(acc, v);
    }
}

// OP_GATHER_F16 (oplist_exec.c:1378-1436), thread per output element.
struct GatherGeom {
    uint32_t axis, xrank, irank;
    uint32_t td[5], xd[5];
    uint64_t os[5], ts[5], xs[5];
};

__global__ void gather_kernel(const uint16_t* __restrict__ tbl, const int32_t* __restrict__ idx,
                              uint16_t* __restrict__ y, uint32_t n, GatherGeom G) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint64_t rem = i;
    uint32_t oc[5];
#pragma unroll
    for (int d = 0; d < 5; ++d) { oc[d] = (uint32_t)(rem / G.os[d]); rem %= G.os[d]; }
    uint64_t il = 0;
    for (uint32_t k = 0; k < G.xrank && k < 5; ++k) il += (uint64_t)(oc[G.axis + k] % G.xd[k]) * G.xs[k];
    int32_t r = idx[il];
    if (r < 0) r += (int32_t)G.td[G.axis];
    if (r < 0 || r >= (int32_t)G.td[G.axis]) { y[i] = 0; return; }
    uint64_t src = 0;
    for (uint32_t d = 0; d < G.axis && d < 5; ++d) src += (uint64_t)oc[d] * G.ts[d];
    src += (uint64_t)r * G.ts[G.axis];
    for (uint32_t d = G.axis + 1; d < G.irank && d < 5; ++d) {
        const uint32_t ocd = d + G.xrank - 1;
        src += (uint64_t)(ocd < 5 ? oc[ocd] : 0) * G.ts[d];
    }
    y[i] = tbl[src];
}

// OP_TRANSPOSE_F16 (oplist_exec.c:983-1011): (1, H, W, C) with perm[output axis] = input axis.
__global__ void transpose4_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ y, uint32_t Hh,
                                  uint32_t W, uint32_t Cc, uint32_t perm) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)Hh * W * Cc) return;
    const uint32_t dims[4] = {1, Hh, W, Cc};
    const uint32_t p[4] = {perm & 0xFF, (perm >> 8) & 0xFF, (perm >> 16) & 0xFF, (perm >> 24) & 0xFF};
    const uint64_t si[4] = {(uint64_t)Hh * W * Cc, (uint64_t)W * Cc, Cc, 1};
    uint64_t rem = i;
    uint32_t ic[4] = {0, 0, 0, 0};
    for (int ax = 3; ax >= 0; --ax) {
        const uint32_t d = dims[p[ax]];
        ic[p[ax]] = (uint32_t)(rem % d);
        rem /= d;
    }
    y[i] = x[ic[0] * si[0] + ic[1] * si[1] + ic[2] * si[2] + ic[3] * si[3]];
}

inline uint32_t nblk(size_t n, uint32_t bs) { return (uint32_t)((n + bs - 1) / bs); }

}  // namespace

hipError_t launch_crouton_encode(const uint16_t* lin, uint16_t* surf, uint32_t rows, uint32_t cols,
                                 hipStream_t st) {
    if (rows % 32 || cols % 32) return hipErrorInvalidValue;
    const size_t pairs = (size_t)rows * cols / 2;
    if (!pairs) return hipSuccess;
    hipLaunchKernelGGL(crouton_encode_kernel, dim3(nblk(pairs, 256)), dim3(256), 0, st, lin,
                       reinterpret_cast<uint32_t*>(surf), rows, cols);
    return hipGetLastError();
}

hipError_t launch_crouton_decode(const uint16_t* surf, uint16_t* lin, uint32_t rows, uint32_t cols,
                                 hipStream_t st) {
    if (rows % 32 || cols % 32) return hipErrorInvalidValue;
    const size_t pairs = (size_t)rows * cols / 2;
    if (!pairs) return hipSuccess;
    hipLaunchKernelGGL(crouton_decode_kernel, dim3(nblk(pairs, 256)), dim3(256), 0, st,
                       reinterpret_cast<const uint32_t*>(surf), lin, rows, cols);
    return hipGetLastError();
}

hipError_t launch_matmul_w4a16(const uint16_t* act, const uint8_t* w, uint16_t* out, uint32_t M, uint32_t K,
                               uint32_t N, hipStream_t st) {
    if (M % 32 || K % 32 || N % 32) return hipErrorInvalidValue;
    if (!M || !N || !K) return hipSuccess;
    // Tile by the time of the grid's rounds. A round (one workgroup on every CU) took 5.8 us
    // with 32 x 32 tiles (two fit a CU: 8.3 us a pair), 8.2 with 32 x 64 and 12 with 64 x 64
    // at K = 2560, in like proportion at other K. Measured with 32 x 32 / 32 x 64 / 64 x 64
    // tiles, us (M x N x K): 32 x 2560 x 2560 5.8 / 7.8 / 11.1; 256 x 2560 x 2560 14.7 / 16.5 /
    // 12.6; 512 x 2560 x 2560 22.5 / 24.6 / 23.5; 1024 x 512 x 4096 17.4 / 15.4 / 18.9;
    // 1024 x 4096 x 4096 91 / 82 / 62.
    const size_t cus = (size_t)device_cu_count();
    auto grid = [&](uint32_t rt, uint32_t nt) { return (size_t)((M / 32 + rt - 1) / rt) * ((N / 32 + nt - 1) / nt); };
    auto rounds = [&](size_t g) { return (double)((g + cus - 1) / cus); };
    const double r11 = rounds(grid(1, 1));
    const double t11 = 8.3 * std::floor(r11 / 2) + 5.8 * std::fmod(r11, 2.0);
    const double t12 = 8.2 * rounds(grid(1, 2)), t22 = 12.0 * rounds(grid(2, 2));
    auto go = [&](auto kern, uint32_t rt, uint32_t nt, uint32_t wv) {
        hipLaunchKernelGGL(kern, dim3((uint32_t)grid(rt, nt)), dim3(64 * wv), 0, st, act, w, out, M, K, N);
    };
    // One or two K steps leave most of 8 waves without work, so large grids run one wave per tile
    // (M x N x K, us, 8 waves / one): 2048 x 2560 x 32 26.5 / 12.7, x 128 26.6 / 13.8, 1024 x 1024
    // x 128 6.7 / 7.1.
    if (K <= 128 && grid(1, 2) > 2 * cus) go(w4a16_gemm_kernel<1, 2, 1, 1>, 1, 2, 1);
    else if (t22 < t11 && t22 < t12) go(w4a16_gemm_kernel<2, 2, 2, 8>, 2, 2, 8);
    else if (t12 < t11) go(w4a16_gemm_kernel<1, 2, 2, 8>, 1, 2, 8);
    else go(w4a16_gemm_kernel<1, 1, 4, 8>, 1, 1, 8);
    return hipGetLastError();
}

hipError_t launch_rmsnorm_crouton(const uint16_t* x, const __half* w, __half* y, uint32_t m, uint32_t n,
                                  hipStream_t st) {
    if (!m || m % 32 || n % 32) return hipErrorInvalidValue;
    hipLaunchKernelGGL(rmsnorm_crouton_kernel, dim3((m + 3) / 4), dim3(256), 0, st, x, w, y, m, n);
    return hipGetLastError();
}

hipError_t launch_concat(const uint16_t* const* xs, const uint32_t* sizes, uint32_t n_seg, uint16_t* y,
                         uint32_t n_elems, hipStream_t st) {
    Seg4 s{};
    uint32_t total = 0;
    for (uint32_t k = 0; k < n_seg && k < 4; ++k) {
        s.x[k] = xs[k];
        s.size[k] = sizes[k];
        total += sizes[k];
    }
    if (!total || n_elems % total) return hipErrorInvalidValue;
    if (!n_elems) return hipSuccess;
    hipLaunchKernelGGL(concat_kernel, dim3(nblk(n_elems, 256)), dim3(256), 0, st, s, y, n_seg < 4 ? n_seg : 4,
                       total, n_elems);
    return hipGetLastError();
}

hipError_t launch_split(const uint16_t* x, uint16_t* y, uint32_t outer, uint32_t total, uint32_t off,
                        uint32_t size, hipStream_t st) {
    const size_t n = (size_t)outer * size;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(split_kernel, dim3(nblk(n, 256)), dim3(256), 0, st, x, y, total, off, size, (uint32_t)n);
    return hipGetLastError();
}

hipError_t launch_pad(const uint16_t* x, uint16_t* y, uint32_t outer, uint32_t in_inner, uint32_t out_inner,
                      uint32_t before, uint16_t pv, hipStream_t st) {
    const size_t n = (size_t)outer * out_inner;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(pad_kernel, dim3(nblk(n, 256)), dim3(256), 0, st, x, y, outer, in_inner, out_inner,
                       before, pv);
    return hipGetLastError();
}

hipError_t launch_reduce(const __half* x, __half* y, uint32_t outer, uint32_t L, uint32_t inner,
                         uint32_t subtype, hipStream_t st) {
    const size_t n = (size_t)outer * inner;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(reduce_kernel, dim3(nblk(n, 256)), dim3(256), 0, st, x, y, outer, L, inner, subtype);
    return hipGetLastError();
}

hipError_t launch_cumsum(const __half* x, __half* y, uint32_t rows, uint32_t n, uint32_t exclusive,
                         uint32_t reverse, hipStream_t st) {
    if (!rows) return hipSuccess;
    hipLaunchKernelGGL(cumsum_kernel, dim3(nblk(rows, 64)), dim3(64), 0, st, x, y, rows, n, exclusive, reverse);
    return hipGetLastError();
}

hipError_t launch_gather(const uint16_t* tbl, const int32_t* idx, uint16_t* y, uint32_t n, uint32_t axis,
                         uint32_t xrank, uint32_t irank, const uint32_t* td, const uint32_t* xd,
                         hipStream_t st) {
    if (axis >= irank || irank > 5 || xrank > 5 || xrank == 0) return hipErrorInvalidValue;
    GatherGeom G{};
    G.axis = axis;
    G.xrank = xrank;
    G.irank = irank;
    for (int d = 0; d < 5; ++d) { G.td[d] = td[d]; G.xd[d] = xd[d]; }
    uint32_t od[5] = {1, 1, 1, 1, 1};
    for (uint32_t d = 0; d < axis && d < 5; ++d) od[d] = td[d];
    for (uint32_t k = 0; k < xrank && axis + k < 5; ++k) od[axis + k] = xd[k];
    for (uint32_t d = axis + 1; d < irank && d < 5; ++d)
        if (d + xrank - 1 < 5) od[d + xrank - 1] = td[d];
    for (int d = 0; d < 5; ++d) { G.os[d] = 1; G.ts[d] = 1; G.xs[d] = 1; }
    for (int d = 3; d >= 0; --d) {
        G.os[d] = G.os[d + 1] * od[d + 1];
        G.ts[d] = G.ts[d + 1] * td[d + 1];
        G.xs[d] = G.xs[d + 1] * xd[d + 1];
    }
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(gather_kernel, dim3(nblk(n, 256)), dim3(256), 0, st, tbl, idx, y, n, G);
    return hipGetLastError();
}

hipError_t launch_transpose4(const uint16_t* x, uint16_t* y, uint32_t Hh, uint32_t W, uint32_t Cc,
                             uint32_t perm, hipStream_t st) {
    for (int s = 0; s < 32; s += 8)
        if (((perm >> s) & 0xFF) > 3) return hipErrorInvalidValue;
    const size_t n = (size_t)Hh * W * Cc;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(transpose4_kernel, dim3(nblk(n, 256)), dim3(256), 0, st, x, y, Hh, W, Cc, perm);
    return hipGetLastError();
}

}  // namespace gehtp
