// gemm.hip -- nn_dense / nn_gemm on the matrix cores.
//
//   y[m,n] = alpha * sum_k a[m,k] * b[n,k]  (+ beta * c[n])          (transB = 1, the ResNet FC layer; transB = 0: b[k,n])
//
// Up to four rows go to gemv_nt_kernel, everything else to gemm_nt_staged_kernel / gemm_bf16x3_kernel (three-part fp32
// operands, bf16x3.h), k from 2^24 on to gemm_nt_long_kernel; tiny products that no vector load fits keep a
// one-thread-per-output kernel in the CPU loop's exact order.
#include <cstdlib>

#include "bf16x3.h"
#include "common.h"

using namespace kxc_hip;

namespace {

__device__ __forceinline__ float epilogue(float acc, float alpha, float beta, const float* c, int64_t j, int64_t c_len,
                                          bool scale_a, bool scale_c) {
    float v = acc;
    if (scale_a) v = __fmul_rn(v, alpha);
    if (c != nullptr) {
        float cb = c[c_len == 1 ? 0 : j];
        if (scale_c) cb = __fmul_rn(cb, beta);
        v = __fadd_rn(v, cb);
    }
    return v;
}

constexpr uint32_t kOob = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), 0x00020000);
}

// 16 bytes per lane from a buffer straight into LDS (lane l writes lds + 16*l; see qconv_c16_i8.hip)
typedef __attribute__((address_space(3))) void* lds_ptr_t;
__device__ __forceinline__ void load16_to_lds(__amdgpu_buffer_rsrc_t rsrc, char* lds, uint32_t voffset, uint32_t soffset) {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)lds, 16, voffset, soffset, 0, 0);
#endif
}

// The KS partial tiles of a workgroup meet in LDS: [wave][register quad][lane][16 bytes]; register g of a block is row
// 8*(g/4) + 4*half + g%4, column r.  Every wave finishes its share of the quads.
template <int RO, int RP, int KS, bool TB>
__device__ __forceinline__ void finish_tile(const f32x16 (&acc)[RO][RP], char* lds, int wave, int lane, const float* __restrict__ a, const float* __restrict__ b,
                                            const float* __restrict__ c, float* __restrict__ y, int32_t M, int32_t N, int32_t K, int m0, int n0,
                                            float alpha, float beta, int64_t c_len, int scale_a, int scale_c) {
    constexpr int NB = RO * RP;
    const int half = lane >> 5, r = lane & 31;
    auto at = [&](int w, int q) { return reinterpret_cast<f32x4*>(lds + ((w * NB * 4 + q) * 64 + lane) * 16); };
#pragma unroll
    for (int q = 0; q < NB * 4; ++q) {
        const f32x16& v = acc[q / 4 / RP][q / 4 % RP];
        *at(wave, q) = f32x4{v[4 * (q % 4)], v[4 * (q % 4) + 1], v[4 * (q % 4) + 2], v[4 * (q % 4) + 3]};
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < (NB * 4 + KS - 1) / KS; ++t) {
        const int q = t * KS + wave;
        if (q >= NB * 4) break;
        f32x4 v = *at(0, q);
#pragma unroll
        for (int w = 1; w < KS; ++w) {
            const f32x4 p = *at(w, q);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = __fadd_rn(v[e], p[e]);
        }
        const int n = n0 + (q / 4 % RP) * 32 + r;
        if (n >= N) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = m0 + (q / 4 / RP) * 32 + 8 * (q % 4) + 4 * half + e;
            if (m >= M) continue;
            float x = v[e];
            // a non-finite operand, or a sum next to the largest float (h h' alone may round past it): the fp32 loop decides
            if (__builtin_expect(!(__builtin_fabsf(x) <= 3.402823466e38f), 0)) {
                x = 0.0f;
                for (int k = 0; k < K; ++k)
                    x = fmaf(a[static_cast<int64_t>(m) * K + k], TB ? b[static_cast<int64_t>(n) * K + k] : b[static_cast<int64_t>(k) * N + n], x);
            }
            y[static_cast<int64_t>(m) * N + n] = epilogue(x, alpha, beta, c, n, c_len, scale_a != 0, scale_c != 0);
        }
    }
}

// A workgroup owns one tile of 32*RO rows of `a` by 32*RP columns of y; its KS waves split the k-steps of 16 (contiguous
// runs), read both operands straight into registers D steps ahead, split them into their three bf16 parts and multiply;
// the partial tiles meet in LDS and every wave finishes its share of the rows.  Lane (r, half) of a step holds eight
// consecutive k of row r: two 16-byte loads, or eight 4-byte loads of neighbouring columns when b is [k][n].
// What bounds it: the splitting (11 instructions per two values on the vector ALU) beside the matrix instructions of the
// other waves; before that, with few tiles, the chain launch - first load - last store.  No LDS staging: a tile's operands
// are read by one workgroup and the vector cache serves the two halves of a line.  Measured (us, one thread per output before):
// b = [k][n] 300 x 1000 x 2048 474 -> 23.5, 33 x 500 x 900 211 -> 7.5; k not a multiple of four 257 x 333 x 777 202 -> 9.6.
template <int RO, int RP, int KS, int D, bool TB>
__global__ void __launch_bounds__(64 * KS) __attribute__((amdgpu_waves_per_eu(2))) gemm_bf16x3_kernel(
    const float* __restrict__ a, const float* __restrict__ b, const float* __restrict__ c, float* __restrict__ y, int32_t M, int32_t N, int32_t K,
    int32_t m_tiles, int32_t tiles, int32_t tiles_per_xcd, float alpha, float beta, int64_t c_len, int scale_a, int scale_c) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63, half = lane >> 5, r = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    // an XCD (own L2) takes a contiguous run of tiles: all row tiles of a column tile before the next one
    const int tile = static_cast<int>(blockIdx.x & 7) * tiles_per_xcd + static_cast<int>(blockIdx.x >> 3);
    if (tile >= tiles || static_cast<int>(blockIdx.x >> 3) >= tiles_per_xcd) return;
    const int n_tile = tile / m_tiles, m0 = (tile - n_tile * m_tiles) * 32 * RO, n0 = n_tile * 32 * RP;

    // rows past the last one lie beyond the buffers and read as zero
    const __amdgpu_buffer_rsrc_t ar = make_rsrc(a + static_cast<int64_t>(m0) * K, static_cast<uint32_t>(min(32 * RO, M - m0)) * static_cast<uint32_t>(K) * 4u);
    const __amdgpu_buffer_rsrc_t br = TB ? make_rsrc(b + static_cast<int64_t>(n0) * K, static_cast<uint32_t>(min(32 * RP, N - n0)) * static_cast<uint32_t>(K) * 4u)
                                         : make_rsrc(b, static_cast<uint32_t>(K) * static_cast<uint32_t>(N) * 4u);
    uint32_t ao[RO], bo[RP];
#pragma unroll
    for (int i = 0; i < RO; ++i) ao[i] = m0 + i * 32 + r < M ? static_cast<uint32_t>((i * 32 + r) * K + 8 * half) * 4u : kOob;
#pragma unroll
    for (int j = 0; j < RP; ++j) {
        const int n = n0 + j * 32 + r;
        bo[j] = n >= N ? kOob : TB ? static_cast<uint32_t>((j * 32 + r) * K + 8 * half) * 4u : static_cast<uint32_t>(8 * half * N + n) * 4u;
    }
    const uint32_t row_bytes = static_cast<uint32_t>(N) * 4u;

    f32x16 acc[RO][RP];
#pragma unroll
    for (int i = 0; i < RO; ++i)
#pragma unroll
        for (int j = 0; j < RP; ++j)
#pragma unroll
            for (int g = 0; g < 16; ++g) acc[i][j][g] = 0.0f;

    float av[D][RO][8], bv[D][RP][8];
    auto load8 = [](float (&v)[8], __amdgpu_buffer_rsrc_t rs, uint32_t vo, uint32_t so) __attribute__((always_inline)) {
        const f32x4 lo = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, vo, so, 0));
        const f32x4 hi = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, vo + 16u, so, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) { v[e] = lo[e]; v[4 + e] = hi[e]; }
    };
    auto ldf = [](__amdgpu_buffer_rsrc_t rs, uint32_t vo, uint32_t so) __attribute__((always_inline)) {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, vo, so, 0));
    };
    auto load = [&](int step, int d) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RO; ++i) load8(av[d][i], ar, ao[i], static_cast<uint32_t>(step) * 64u);
#pragma unroll
        for (int j = 0; j < RP; ++j) {
            if constexpr (TB) {
                load8(bv[d][j], br, bo[j], static_cast<uint32_t>(step) * 64u);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) bv[d][j][e] = ldf(br, bo[j], static_cast<uint32_t>(step * 16 + e) * row_bytes);
            }
        }
    };
    auto multiply = [&](int d) __attribute__((always_inline)) {
        u32x4 af[RO][3], bf[RP][3];
#pragma unroll
        for (int i = 0; i < RO; ++i) { const Split8 p = split8(av[d][i]); af[i][0] = p.h; af[i][1] = p.m; af[i][2] = p.l; }
#pragma unroll
        for (int j = 0; j < RP; ++j) { const Split8 p = split8(bv[d][j]); bf[j][0] = p.h; bf[j][1] = p.m; bf[j][2] = p.l; }
        mfma6<RO, RP>(acc, af, bf);
    };
    const int steps = K >> 4;                                 // whole ones
    const int per = ((steps + KS - 1) / KS + 1) & ~1;         // (two steps share a 128-byte line)
    const int lo = min(steps, wave * per), hi = min(steps, lo + per);
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (lo + d < hi) load(lo + d, d);
    int s = lo;
    for (; s + 2 * D <= hi; s += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            multiply(d);
            load(s + D + d, d);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    for (; s < hi; s += D) {
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (s + d < hi) {
                multiply(d);
                if (s + D + d < hi) load(s + D + d, d);
                __builtin_amdgcn_sched_barrier(0);
            }
    }
    if ((K & 15) != 0 && wave == KS - 1) {                    // what is left of k, element by element
        const int k0 = steps << 4;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const bool in = k0 + 8 * half + e < K;
#pragma unroll
            for (int i = 0; i < RO; ++i) av[0][i][e] = ldf(ar, in ? ao[i] + 4u * e : kOob, static_cast<uint32_t>(k0) * 4u);
#pragma unroll
            for (int j = 0; j < RP; ++j)
                bv[0][j][e] = ldf(br, in ? bo[j] + (TB ? 4u * e : 0u) : kOob, TB ? static_cast<uint32_t>(k0) * 4u : static_cast<uint32_t>(k0 + e) * row_bytes);
        }
        multiply(0);
    }

    finish_tile<RO, RP, KS, TB>(acc, lds, wave, lane, a, b, c, y, M, N, K, m0, n0, alpha, beta, c_len, scale_a, scale_c);
}

// The same tiles where rows of both operands are whole 16-byte words (b = [n][k], k a multiple of four).  Lane (r, half)
// reading its own row touches 32 cache lines with every load, and the vector cache takes those one after the other:
// here a load covers eight rows by 128 bytes (eight lines) and goes straight into LDS, into a chunk of 32 k that belongs to
// the wave alone: no barrier, the wave waits for its own loads, moves the chunk into registers, requests the next one and
// multiplies (a ring of two or four chunks was slower or equal: fewer workgroups fit a compute unit).  Within a row the 16-byte words are stored in
// the order (word ^ row % 8), so the 32 rows that a fragment read takes at once hit all banks.
// Measured (us; before: fp32 matrix instructions on operands read row by row): 300 x 1000 x 2048 54.6 -> 18.4,
// 512 x 4096 x 4096 514 -> 113, 8 x 4096 x 4096 47.6 -> 20.0, 64 x 1000 x 512 7.6 -> 5.7; k = 1000 (no multiple of 32 before)
// 200 x 2000 x 1000 1667 -> 14.4.
template <int RO, int RP, int KS>
__global__ void __launch_bounds__(64 * KS) __attribute__((amdgpu_waves_per_eu(2))) gemm_nt_staged_kernel(
    const float* __restrict__ a, const float* __restrict__ b, const float* __restrict__ c, float* __restrict__ y, int32_t M, int32_t N, int32_t K,
    int32_t m_tiles, int32_t tiles, int32_t tiles_per_xcd, float alpha, float beta, int64_t c_len, int scale_a, int scale_c) {
    constexpr int L = 4 * (RO + RP);                          // loads of 1 KiB per chunk
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63, half = lane >> 5, r = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int tile = static_cast<int>(blockIdx.x & 7) * tiles_per_xcd + static_cast<int>(blockIdx.x >> 3);
    if (tile >= tiles || static_cast<int>(blockIdx.x >> 3) >= tiles_per_xcd) return;
    const int n_tile = tile / m_tiles, m0 = (tile - n_tile * m_tiles) * 32 * RO, n0 = n_tile * 32 * RP;

    // rows past the last one lie beyond the buffers and read as zero
    const __amdgpu_buffer_rsrc_t ar = make_rsrc(a + static_cast<int64_t>(m0) * K, static_cast<uint32_t>(min(32 * RO, M - m0)) * static_cast<uint32_t>(K) * 4u);
    const __amdgpu_buffer_rsrc_t br = make_rsrc(b + static_cast<int64_t>(n0) * K, static_cast<uint32_t>(min(32 * RP, N - n0)) * static_cast<uint32_t>(K) * 4u);
    char* const ring = lds + wave * (L * 1024);
    const int kword = (lane & 7) ^ (lane >> 3);               // the word of its row's chunk that a lane loads
    uint32_t vo[4 * (RO > RP ? RO : RP)];
#pragma unroll
    for (int i = 0; i < 4 * (RO > RP ? RO : RP); ++i) vo[i] = static_cast<uint32_t>((i * 8 + (lane >> 3)) * K + kword * 4) * 4u;
    const int chunks = (K + 31) >> 5, per = (chunks + KS - 1) / KS;
    const int lo = min(chunks, wave * per), hi = min(chunks, lo + per);
    auto issue = [&](int chunk) __attribute__((always_inline)) {
        const uint32_t mask = chunk * 32 + kword * 4 < K ? 0u : kOob;
#pragma unroll
        for (int i = 0; i < 4 * RO; ++i) load16_to_lds(ar, ring + i * 1024, vo[i] | mask, static_cast<uint32_t>(chunk) * 128u);
#pragma unroll
        for (int i = 0; i < 4 * RP; ++i) load16_to_lds(br, ring + (4 * RO + i) * 1024, vo[i] | mask, static_cast<uint32_t>(chunk) * 128u);
    };
    f32x16 acc[RO][RP];
#pragma unroll
    for (int i = 0; i < RO; ++i)
#pragma unroll
        for (int j = 0; j < RP; ++j)
#pragma unroll
            for (int g = 0; g < 16; ++g) acc[i][j][g] = 0.0f;
    if (lo < hi) {
        issue(lo);
        for (int chunk = lo; chunk < hi; ++chunk) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            float av[2][RO][8], bv[2][RP][8];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                auto read8 = [&](float (&v)[8], int row0) __attribute__((always_inline)) {
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const f32x4 w = *reinterpret_cast<const f32x4*>(ring + row0 * 128 + r * 128 + (((4 * s + 2 * half + q) ^ (r & 7)) << 4));
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[4 * q + e] = w[e];
                    }
                };
#pragma unroll
                for (int i = 0; i < RO; ++i) read8(av[s][i], i * 32);
#pragma unroll
                for (int j = 0; j < RP; ++j) read8(bv[s][j], (RO + j) * 32);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // read before it is filled again
            __builtin_amdgcn_sched_barrier(0);
            if (chunk + 1 < hi) issue(chunk + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                u32x4 af[RO][3], bf[RP][3];
#pragma unroll
                for (int i = 0; i < RO; ++i) { const Split8 p = split8(av[s][i]); af[i][0] = p.h; af[i][1] = p.m; af[i][2] = p.l; }
#pragma unroll
                for (int j = 0; j < RP; ++j) { const Split8 p = split8(bv[s][j]); bf[j][0] = p.h; bf[j][1] = p.m; bf[j][2] = p.l; }
                mfma6<RO, RP>(acc, af, bf);
            }
        }
    }
    __syncthreads();                                          // the chunks become the partial tiles
    finish_tile<RO, RP, KS, true>(acc, lds, wave, lane, a, b, c, y, M, N, K, m0, n0, alpha, beta, c_len, scale_a, scale_c);
}

// k from 2^24 on: row offsets of a tile no longer fit the 31 bits of a buffer offset, so the lanes walk their rows with 64-bit
// addresses, on the fp32 instructions: a workgroup of four waves owns 32 x 32 outputs, the waves split k four ways and
// the two half-waves of a wave two ways.  Bound by the latency of its loads (5 x 2 x 2^25:
// 235 ms; one thread per output, which this range fell to, 2.5 s and a single running sum).
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) gemm_nt_long_kernel(
    const float* __restrict__ a, const float* __restrict__ b, const float* __restrict__ c, float* __restrict__ y, int32_t M, int32_t N, int32_t K,
    float alpha, float beta, int64_t c_len, int scale_a, int scale_c) {
    __shared__ float part[4][32 * 33];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, half = lane >> 5, r = lane & 31;
    const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
    const int run = K / 8;                     // k values of a half-wave (a multiple of 4)
    // (rows past the last one are computed and never stored)
    const float* const ap = a + static_cast<int64_t>(min(m0 + r, M - 1)) * K + static_cast<int64_t>(wave * 2 + half) * run;
    const float* const bp = b + static_cast<int64_t>(min(n0 + r, N - 1)) * K + static_cast<int64_t>(wave * 2 + half) * run;
    f32x16 acc = {0};
    for (int k = 0; k < run; k += 4) {
        const f32x4 va = *reinterpret_cast<const f32x4*>(ap + k), vb = *reinterpret_cast<const f32x4*>(bp + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(va[e], vb[e], acc, 0, 0, 0);
    }
#pragma unroll
    for (int g = 0; g < 16; ++g) part[wave][(8 * (g / 4) + 4 * half + g % 4) * 33 + r] = acc[g];
    __syncthreads();
    for (int e = threadIdx.x; e < 1024; e += 256) {
        const int i = e >> 5, j = e & 31, m = m0 + i, n = n0 + j;
        float s = part[0][i * 33 + j];
#pragma unroll
        for (int w = 1; w < 4; ++w) s = __fadd_rn(s, part[w][i * 33 + j]);
        if (m < M && n < N) y[static_cast<int64_t>(m) * N + n] = epilogue(s, alpha, beta, c, n, c_len, scale_a != 0, scale_c != 0);
    }
}

// A handful of rows (batch 1-4 of a classifier layer): the matrix-core tile above would be 32 rows of which at
// most 4 are real, and its k loop is a chain of dependent load latencies.  Here a wave owns four output columns for
// every row; its lanes split k (a lane takes 4 consecutive floats of every 256), all loads of a 256-chunk are in
// flight together, and the lanes' sums are added across the wave at the end (a tree: not the CPU order, within the
// fp32 tolerance like the matrix-core kernel).  Measured on MI355X inside ResNet-18 (FC 512 -> 1000): batch 1
// 0.2068 -> 0.2040 ms per pass, batch 2 0.2511 -> 0.2480, batch 4 equal, batch 8 slower (0.4643 -> 0.4728).
constexpr int kGemvRows = 4;
constexpr int kGemvCols = 4;
template <int ROWS>
__global__ void __launch_bounds__(256) gemv_nt_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                      const float* __restrict__ c, float* __restrict__ y,
                                                      int32_t N, int32_t K, float alpha, float beta, int64_t c_len,
                                                      int scale_a, int scale_c) {
    const int lane = threadIdx.x & 63;
    const int n0 = (static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x >> 6)) * kGemvCols;
    if (n0 >= N) return;
    float acc[ROWS][kGemvCols];
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
#pragma unroll
        for (int j = 0; j < kGemvCols; ++j) acc[i][j] = 0.0f;
    for (int k0 = lane * 4; k0 < K; k0 += 256) {
        float4 vb[kGemvCols], va[ROWS];
#pragma unroll
        for (int j = 0; j < kGemvCols; ++j)
            vb[j] = *reinterpret_cast<const float4*>(b + static_cast<int64_t>(min(n0 + j, N - 1)) * K + k0);
#pragma unroll
        for (int i = 0; i < ROWS; ++i) va[i] = *reinterpret_cast<const float4*>(a + static_cast<int64_t>(i) * K + k0);
#pragma unroll
        for (int i = 0; i < ROWS; ++i)
#pragma unroll
            for (int j = 0; j < kGemvCols; ++j) {
                acc[i][j] = fmaf(va[i].x, vb[j].x, acc[i][j]);
                acc[i][j] = fmaf(va[i].y, vb[j].y, acc[i][j]);
                acc[i][j] = fmaf(va[i].z, vb[j].z, acc[i][j]);
                acc[i][j] = fmaf(va[i].w, vb[j].w, acc[i][j]);
            }
    }
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
#pragma unroll
        for (int j = 0; j < kGemvCols; ++j) {
            float v = acc[i][j];
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
            if (lane == 0 && n0 + j < N)
                y[static_cast<int64_t>(i) * N + n0 + j] = epilogue(v, alpha, beta, c, n0 + j, c_len, scale_a != 0, scale_c != 0);
        }
}

// Reference-order kernel: k ascending from 0.0f, multiply and add rounded separately.
template <bool TRANS_B>
__global__ void __launch_bounds__(256) gemm_direct_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                          const float* __restrict__ c, float* __restrict__ y,
                                                          int64_t M, int64_t N, int64_t K, float alpha, float beta,
                                                          int64_t c_len, int scale_a, int scale_c) {
    const int64_t total = M * N;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
    for (int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; e < total; e += stride) {
        const int64_t i = e / N, j = e - i * N;
        float acc = 0.0f;
        for (int64_t k = 0; k < K; ++k) {
            const float bv = TRANS_B ? b[j * K + k] : b[k * N + j];
            acc = __fadd_rn(acc, __fmul_rn(a[i * K + k], bv));
        }
        y[e] = epilogue(acc, alpha, beta, c, j, c_len, scale_a != 0, scale_c != 0);
    }
}

// int8 dense: acc int32 exact, y = (float)(acc + bias[n]) * mult[n].
__global__ void __launch_bounds__(256) qdense_kernel(const int8_t* __restrict__ a, const int8_t* __restrict__ b,
                                                     const int32_t* __restrict__ bias, const float* __restrict__ mult,
                                                     float* __restrict__ y, int64_t M, int64_t N, int64_t K) {
    const int64_t total = M * N;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
    for (int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; e < total; e += stride) {
        const int64_t i = e / N, j = e - i * N;
        const int8_t* ar = a + i * K;
        const int8_t* br = b + j * K;
        int32_t acc = 0;
        int64_t k = 0;
        if (((reinterpret_cast<uintptr_t>(ar) | reinterpret_cast<uintptr_t>(br)) & 3u) == 0) {
            for (; k + 4 <= K; k += 4) {
                const int32_t va = *reinterpret_cast<const int32_t*>(ar + k);
                const int32_t vb = *reinterpret_cast<const int32_t*>(br + k);
                acc = __builtin_amdgcn_sdot4(va, vb, acc, false);
            }
        }
        for (; k < K; ++k) acc += static_cast<int32_t>(ar[k]) * static_cast<int32_t>(br[k]);
        if (bias) acc += bias[j];
        y[e] = __fmul_rn(static_cast<float>(acc), mult[j]);
    }
}

// int8 dense, one wave per output column j and 64 rows at a time.  Lane l owns bytes [16l, 16l+16) of every
// 1 KiB slice of K: the weight row is read once, every activation row as one coalesced 16-byte load per lane,
// products go through the 4-way int8 dot instruction, and the 64 per-lane partial sums of the 64 rows are
// combined with a transposing butterfly (63 exchanges instead of 64 x 6) that leaves row r's total in lane r.
__global__ void __launch_bounds__(256) qdense_wave_kernel(const int8_t* __restrict__ a, const int8_t* __restrict__ b,
                                                          const int32_t* __restrict__ bias, const float* __restrict__ mult,
                                                          float* __restrict__ y, int32_t M, int32_t N, int32_t K) {
    const int lane = threadIdx.x & 63;
    const int j = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (j >= N) return;
    const int32_t bj = bias ? bias[j] : 0;
    const float mj = mult[j];
    for (int i0 = 0; i0 < M; i0 += 64) {
        int32_t acc[64];
#pragma unroll
        for (int r = 0; r < 64; ++r) acc[r] = 0;
        for (int k0 = 0; k0 < K; k0 += 1024) {
            const int kk = k0 + lane * 16;
            if (kk < K) {
                const int4 vb = *reinterpret_cast<const int4*>(b + static_cast<int64_t>(j) * K + kk);
#pragma unroll
                for (int r = 0; r < 64; ++r) {
                    if (i0 + r < M) {
                        const int4 va = *reinterpret_cast<const int4*>(a + static_cast<int64_t>(i0 + r) * K + kk);
                        int32_t t = acc[r];
                        t = __builtin_amdgcn_sdot4(va.x, vb.x, t, false);
                        t = __builtin_amdgcn_sdot4(va.y, vb.y, t, false);
                        t = __builtin_amdgcn_sdot4(va.z, vb.z, t, false);
                        t = __builtin_amdgcn_sdot4(va.w, vb.w, t, false);
                        acc[r] = t;
                    }
                }
            }
        }
#pragma unroll
        for (int s = 32; s >= 1; s >>= 1) {
            const bool upper = (lane & s) != 0;
#pragma unroll
            for (int t = 0; t < s; ++t) {
                const int32_t send = upper ? acc[t] : acc[t + s];
                const int32_t keep = upper ? acc[t + s] : acc[t];
                acc[t] = keep + __shfl_xor(send, s, 64);
            }
        }
        const int row = i0 + lane;
        if (row < M) y[static_cast<int64_t>(row) * N + j] = __fmul_rn(static_cast<float>(acc[0] + bj), mj);
    }
}

// int8 dense on the int8 matrix cores: one wave per 32x32 block of y, D[i][j] += A[i][k] * B[j][k].  Both
// operands are k-contiguous in memory, so a lane's 16-byte k-slice of the 32x32x32 instruction is one global
// load each (no LDS): lane (r, half) reads a[i0+r][32*step + 16*half ..] and b[j0+r][same].  Rows / columns
// past the end are clamped for the loads and skipped at the store.
typedef int intx4_t __attribute__((ext_vector_type(4)));
typedef int intx16_t __attribute__((ext_vector_type(16)));
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) qdense_mfma_kernel(const int8_t* __restrict__ a, const int8_t* __restrict__ b,
                                                         const int32_t* __restrict__ bias, const float* __restrict__ mult,
                                                         float* __restrict__ y, int32_t M, int32_t N, int32_t K,
                                                         int32_t col_blocks, FastDiv div_cols) {
    const int lane = threadIdx.x;
    const int r = lane & 31, half = lane >> 5;
    const int ib = fast_div(static_cast<int>(blockIdx.x), div_cols), jb = static_cast<int>(blockIdx.x) - ib * col_blocks;
    const int i0 = ib * 32, j0 = jb * 32;
    const int8_t* ap = a + static_cast<int64_t>(min(i0 + r, M - 1)) * K + 16 * half;
    const int8_t* bp = b + static_cast<int64_t>(min(j0 + r, N - 1)) * K + 16 * half;
    intx16_t acc;
#pragma unroll
    for (int g = 0; g < 16; ++g) acc[g] = 0;
    const int steps = K >> 5;
    int s = 0;
    for (; s + 4 <= steps; s += 4) {
        intx4_t av[4], bv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            av[u] = *reinterpret_cast<const intx4_t*>(ap + (s + u) * 32);
            bv[u] = *reinterpret_cast<const intx4_t*>(bp + (s + u) * 32);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[u], bv[u], acc, 0, 0, 0);
    }
    for (; s < steps; ++s) {
        const intx4_t av = *reinterpret_cast<const intx4_t*>(ap + s * 32);
        const intx4_t bv = *reinterpret_cast<const intx4_t*>(bp + s * 32);
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, bv, acc, 0, 0, 0);
    }
    const int j = j0 + r;
    if (j >= N) return;
    const int32_t bj = bias ? bias[j] : 0;
    const float mj = mult[j];
#pragma unroll
    for (int g = 0; g < 16; ++g) {
        const int i = i0 + 8 * (g / 4) + 4 * half + (g % 4);
        if (i < M) y[static_cast<int64_t>(i) * N + j] = __fmul_rn(static_cast<float>(acc[g] + bj), mj);
    }
}

}  // namespace

extern "C" {

int32_t kxc_hip_gemm_f32(const float* a, const float* b, const float* c, float* y, int64_t m, int64_t n, int64_t k,
                         float alpha, float beta, int32_t transB, int64_t c_len, void* stream) {
    KXC_HIP_REQUIRE(m >= 0 && n >= 0 && k >= 0, "kxc_hip_gemm_f32: negative dimension");
    if (m == 0 || n == 0) return KXC_HIP_OK;
    KXC_HIP_REQUIRE(a && b && y, "kxc_hip_gemm_f32: NULL pointer");
    KXC_HIP_REQUIRE(c == nullptr || c_len == n || c_len == 1, "kxc_hip_gemm_f32: bias length %lld is neither %lld nor 1",
                    static_cast<long long>(c_len), static_cast<long long>(n));
    hipStream_t s = ResolveStream(stream);
    const int scale_a = (static_cast<double>(alpha) != 1.0) ? 1 : 0;   // ScaleTensor, src/relay/op/nn/dense.cc:17-24
    const int scale_c = (static_cast<double>(beta) != 1.0) ? 1 : 0;
    const bool aligned = ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15u) == 0;
    // (rows of whole 16-byte words)
    if (transB && k > 0 && (k % 32) == 0 && aligned && m <= kGemvRows && n < (1 << 20) && k < (1 << 30)) {
        const unsigned grid = static_cast<unsigned>(CeilDiv(n, 4 * kGemvCols));
        const int32_t n32 = static_cast<int32_t>(n), k32 = static_cast<int32_t>(k);
#define KXC_GEMV(R) gemv_nt_kernel<R><<<NoteGrid(grid), NoteBlock(256), NoteLds(0), s>>>(a, b, c, y, n32, k32, alpha, beta, c_len, scale_a, scale_c)
        switch (m) {
            case 1: KXC_GEMV(1); break;
            case 2: KXC_GEMV(2); break;
            case 3: KXC_GEMV(3); break;
            default: KXC_GEMV(4); break;
        }
#undef KXC_GEMV
        return CheckLaunch("gemv_nt");
    }
    // (row offsets of a tile and, for b = [k][n], all of b are addressed with 31 bits; KXC_HIP_GEMM_BF16X3=0 keeps the fp32
    // instructions and the one-thread-per-output kernel, for operands below 2^-109: bf16x3.h)
    const bool small = m * n * k < (1 << 15);
    const char* const bx = std::getenv("KXC_HIP_GEMM_BF16X3");
    const bool three_part = !(bx && bx[0] == '0');
    if (three_part && k > 0 && (!small || (transB && k % 32 == 0)) && m < (1 << 20) && n < (1 << 20) && k < (1 << 24) && (transB || n * (k + 16) < (1 << 29))) {
        struct Tile { int ro, rp, ks; void (*kernel[3])(const float*, const float*, const float*, float*, int32_t, int32_t, int32_t, int32_t, int32_t, int32_t,
                                                        float, float, int64_t, int, int); };
#define KXC_GEMM(RO, RP, KS, D) {RO, RP, KS, {gemm_bf16x3_kernel<RO, RP, KS, D, false>, gemm_bf16x3_kernel<RO, RP, KS, D, true>, gemm_nt_staged_kernel<RO, RP, KS>}}
        static const Tile kTiles[] = {KXC_GEMM(1, 1, 8, 2), KXC_GEMM(2, 1, 8, 2), KXC_GEMM(2, 2, 4, 1)};
#undef KXC_GEMM
        // The largest tile (least splitting per product) that still leaves enough workgroups: 64 x 64 from 1024 blocks of
        // 32 x 32 on (512 x 4096 x 512: 21.5 us, 27.5 with 64 x 32, 28.3 with 32 x 32); 32 x 32 up to one per compute unit
        // (512 x 512 x 4096, 256 blocks: 22.8 against 30.7 with 64 x 32), 64 x 32 between (300 x 1000 x 2048, 320: 18.4
        // against 19.6 with 32 x 32)
        const int64_t blocks = CeilDiv(m, 32) * CeilDiv(n, 32);
        const Tile& t = kTiles[blocks <= 256 || k >= (1 << 22) ? 0 : blocks < 1024 ? 1 : 2];
        const int64_t m_tiles = CeilDiv(m, 32 * t.ro), tiles = m_tiles * CeilDiv(n, 32 * t.rp);
        KXC_HIP_REQUIRE(tiles < (1 << 28), "kxc_hip_gemm_f32: too many tiles");
        const int32_t per_xcd = static_cast<int32_t>(CeilDiv(tiles, 8));
        const bool staged = transB && k % 4 == 0 && aligned;
        const size_t lds = static_cast<size_t>(t.ks) * (staged ? t.ro + t.rp : t.ro * t.rp) * 4096;      // (a chunk is never smaller than a partial tile)
        const auto kernel = t.kernel[staged ? 2 : transB ? 1 : 0];
        if (lds > 64 * 1024)
            if (int32_t rc = GrantLds(reinterpret_cast<const void*>(kernel))) return rc;
        kernel<<<NoteGrid(static_cast<int>(per_xcd * 8)), NoteBlock(64 * t.ks), NoteLds(lds), s>>>(
            a, b, c, y, static_cast<int32_t>(m), static_cast<int32_t>(n), static_cast<int32_t>(k), static_cast<int32_t>(m_tiles),
            static_cast<int32_t>(tiles), per_xcd, alpha, beta, c_len, scale_a, scale_c);
        return CheckLaunch("gemm_bf16x3");
    }
    if (transB && k >= (three_part ? 1 << 24 : 1) && (k % 32) == 0 && aligned && m < (1 << 20) && n < (1 << 20) && k < (1 << 30)) {
        const dim3 grid(static_cast<unsigned>(CeilDiv(n, 32)), static_cast<unsigned>(CeilDiv(m, 32)));
        gemm_nt_long_kernel<<<NoteGrid(grid), NoteBlock(256), NoteLds(0), s>>>(a, b, c, y, static_cast<int32_t>(m), static_cast<int32_t>(n),
                                                                               static_cast<int32_t>(k), alpha, beta, c_len, scale_a, scale_c);
        return CheckLaunch("gemm_nt_long");
    }
    int64_t g = CeilDiv(m * n, 256);
    if (g > 256 * 32) g = 256 * 32;
    if (transB) gemm_direct_kernel<true><<<NoteGrid(static_cast<int>(g)), NoteBlock(256), NoteLds(0), s>>>(a, b, c, y, m, n, k, alpha, beta, c_len, scale_a, scale_c);
    else gemm_direct_kernel<false><<<NoteGrid(static_cast<int>(g)), NoteBlock(256), NoteLds(0), s>>>(a, b, c, y, m, n, k, alpha, beta, c_len, scale_a, scale_c);
    return CheckLaunch("gemm_direct");
}

int32_t kxc_hip_qdense_i8(const int8_t* a, const int8_t* b, const int32_t* bias, const float* mult, float* y,
                          int64_t m, int64_t n, int64_t k, void* stream) {
    KXC_HIP_REQUIRE(m >= 0 && n >= 0 && k >= 0, "kxc_hip_qdense_i8: negative dimension");
    if (m == 0 || n == 0) return KXC_HIP_OK;
    KXC_HIP_REQUIRE(a && b && mult && y, "kxc_hip_qdense_i8: NULL pointer");
    KXC_HIP_REQUIRE(k <= 2147483647LL / (128 * 128), "kxc_hip_qdense_i8: k too large for int32 accumulation");
    const bool aligned16 = ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15u) == 0;
    if (k % 32 == 0 && k > 0 && aligned16 && m < (1LL << 30) && n < (1LL << 30) &&
        CeilDiv(m, 32) * CeilDiv(n, 32) <= kMaxGridX) {
        const int32_t col_blocks = static_cast<int32_t>(CeilDiv(n, 32));
        qdense_mfma_kernel<<<NoteGrid(static_cast<int>(CeilDiv(m, 32) * col_blocks)), NoteBlock(64), NoteLds(0),
                             ResolveStream(stream)>>>(a, b, bias, mult, y, static_cast<int32_t>(m),
                                                      static_cast<int32_t>(n), static_cast<int32_t>(k), col_blocks, MakeFastDiv(col_blocks));
        return CheckLaunch("qdense_mfma");
    }
    if (k % 16 == 0 && m < (1LL << 31) && n < (1LL << 31) && CeilDiv(n, 4) <= kMaxGridX &&
        ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15u) == 0) {
        qdense_wave_kernel<<<NoteGrid(static_cast<int>(CeilDiv(n, 4))), NoteBlock(256), NoteLds(0), ResolveStream(stream)>>>(
            a, b, bias, mult, y, static_cast<int32_t>(m), static_cast<int32_t>(n), static_cast<int32_t>(k));
        return CheckLaunch("qdense_wave");
    }
    int64_t g = CeilDiv(m * n, 256);
    if (g > 256 * 32) g = 256 * 32;
    qdense_kernel<<<NoteGrid(static_cast<int>(g)), NoteBlock(256), NoteLds(0), ResolveStream(stream)>>>(a, b, bias, mult, y, m, n, k);
    return CheckLaunch("qdense");
}

}  // extern "C"
