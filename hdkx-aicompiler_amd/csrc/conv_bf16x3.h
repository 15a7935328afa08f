// conv_bf16x3.h -- convolutions of 1x1 to 7x7 filters with stride 1 and 2 as an implicit GEMM on the bf16 matrix cores with
// three-part operands (bf16x3.h); included by conv2d_bf16x3.hip (selection, launch) and conv2d_wino_f32.hip (the filters of a
// plan are packed by one launch).
//
// D[o][pixel] += W[o][tap, c] X[tap, c][pixel], pixels flattened over (n, oh, ow).  A workgroup owns 128 output channels x 64 pixels and
// walks the input channels 16 at a time, with stride 2 in two halves: the input rows of even, then of odd padded position (a
// 3x3 filter's rows 0 and 2, then 1).  Two LDS buffers; a 1x1 filter takes 64 channels at a time and no rows, only the tile's pixels.
//  * Two producer waves load the rows in pieces of four columns x eight channels, split every value into its three parts once,
//    and leave them in LDS as the 16-byte fragments that the matrix instructions take: [part][channels c .. c + 7][row][column
//    parity][column], so that neighbouring pixels of a tap are neighbouring fragments.  They load one half ahead of the one that
//    they split, which is one ahead of the one that is multiplied.
//  * Four consumer waves, 32 channels x 64 pixels each, do nothing but read fragments (X from LDS, W as packed once per weight
//    tensor and read from the L2 one tap ahead) and multiply: 12 matrix instructions per 6 LDS reads and 3 loads.
//  * Kept apart, the memory latency and the splits of the one run beside the matrix instructions of the other; with 168
//    registers a compute unit holds two workgroups, whose barriers do not meet.  (The same product with every wave splitting and
//    multiplying in turn took 4.7 us per 8 channels; here a step of 16 takes 2.9.)
//  * The large products h h' and the five small ones have accumulators of their own, added at the end: one chain of six
//    per 16 channels loses more than the fp32 instructions do (relative error against float64, 2304 terms: 6.7e-7, 1.6e-7 here,
//    v_mfma_f32_32x32x2_f32 split two ways 2.8e-7).  The second output has no registers for that; its small products of a
//    step borrow the first output's accumulators, which are added up before and begin at zero after (1.7e-7 in one chain, 0.8e-7
//    here, 1.1e-7 on the fp32 instructions at 256 terms).
//
// Measured with both outputs, 64 images, against the fp32-instruction kernel, us: 64 -> 128 channels at 56 x 56 97 -> 60, 128 -> 256 at 28 x 28
// 94 -> 54, 256 -> 512 at 14 x 14 104 -> 52 (950 TFLOP/s of bf16 products; a loop of nothing else reaches 1750 on the whole GPU
// and these 196 workgroups leave a quarter of it idle).  What is left, from timing-only builds: 46 to 51 us without any memory
// access; the input 5 to 13, the stores 6 to 14, of 5 to 7 per workgroup before the first matrix instruction and behind the last.
#pragma once

#include <algorithm>

#include "bf16x3.h"
#include "common.h"

namespace kxc_hip {
namespace conv_bx {

constexpr int kOut = 128, kPix = 64, kStep = 16;      // output channels and pixels of a workgroup; channels per step
constexpr int kConsumers = 4, kProducers = 2;         // waves
constexpr int kThreads = 64 * (kConsumers + kProducers);
constexpr int kPlane = 384;                           // positions of an LDS plane (16 bytes: eight channels of one part)
constexpr int kUnits = 2;                             // (channel half, row, four columns) pieces per producer lane
// Row phases of a filter (two halves of a step as described above, or the step as a whole), steps of 16 channels between two
// barriers (a 1x1 filter has one tap for each: four of them), bytes of an LDS buffer.
constexpr int Phases(int K, int S) { return S == 2 && K > 1 ? 2 : 1; }
constexpr int ChannelSteps(int K) { return K == 1 ? 4 : 1; }
constexpr int Plane(int K) { return K == 1 ? kPix : kPlane; }
constexpr int BufBytes(int K) { return 3 * 2 * ChannelSteps(K) * Plane(K) * 16; }
inline size_t LdsBytes(int K) { return 2 * static_cast<size_t>(BufBytes(K)); }

// Steps of the packed filter between two barriers (per row phase pair): the taps in the order the kernel takes them, the second output's filter
// behind the tap that it shares its operand with.
constexpr int Steps(int K, bool second) { return K == 1 ? ChannelSteps(K) : K * K + (second ? 1 : 0); }
// Taps of row phase rho: rows rh = rho, rho + S, ...
constexpr int PhaseTaps(int K, int S, int rho) { return (K - rho + S - 1) / S * K; }
constexpr int PhaseFirst(int K, int S, int rho) { return rho == 0 ? 0 : PhaseTaps(K, S, 0); }
// Tap rh * K + rw of the t-th tap of a phase.
constexpr int TapOf(int K, int S, int rho, int t) { return (rho + t / K * S) * K + t % K; }

inline size_t FilterBytes(int64_t O, int64_t C, int K, bool second) {
    return static_cast<size_t>(CeilDiv(O, 32) * CeilDiv(C, kStep * ChannelSteps(K))) * Steps(K, second) * 3 * 1024;
}
inline int64_t PackBlocks(int64_t O, int64_t C, int K) { return CeilDiv(O, 32) * 4 * CeilDiv(C, kStep * ChannelSteps(K)); }
constexpr int PackFloats(int K) { return 8 * (kStep * ChannelSteps(K) * K * K + 1); }

// How far `pix` neighbouring pixels (flattened over n, oh, ow) that start at a multiple of pix reach at most: `row` for every step to
// the next output row and `image` for every step to the next image.  Within an image, where tiles start in a row repeats after
// at most OW tiles; where the border of two images lies in a tile repeats after at most pix images.
inline int32_t TileReach(int32_t N, int32_t OHW, int32_t OW, int32_t pix, int32_t row, int32_t image) {
    const uint32_t p = static_cast<uint32_t>(pix), ow = static_cast<uint32_t>(OW), ohw = static_cast<uint32_t>(OHW), M = static_cast<uint32_t>(N) * ohw;
    uint32_t best = 0;
    auto tile = [&](uint32_t m0) {
        const uint32_t last = std::min(p, M - m0) - 1;
        best = std::max(best, (m0 % ow + last) / ow * static_cast<uint32_t>(row) + (m0 % ohw + last) / ohw * static_cast<uint32_t>(image));
    };
    for (uint32_t t = 0; t < ow && t * p < M; ++t) tile(t * p);
    for (uint32_t n = 1; n < static_cast<uint32_t>(N) && n <= p; ++n) tile(n * ohw / p * p);
    return static_cast<int32_t>(best);
}

struct Args {
    const float* x;
    const char* u;
    const float* bias;
    const float* res;
    float* y;
    const float* bias2;
    float* y2;
    float* partial;
    const float* w;                     // the filters as they were given, for outputs that are not finite
    const float* w2;
    int32_t N, C, H, W, O, OH, OW, M, OHW, HW, ph, pw;
    int32_t Hq, pitch, hp;              // rows per image in a row phase; LDS row pitch; positions of the even columns
    int32_t w4;                         // pieces of four columns per row
    int32_t csteps, cps, gsplit;        // channel steps (of 16 * ChannelSteps), per part, parts
    int32_t tail, quads;                // the last step is short of channels; K = 1: four pixels are 16 bytes of one channel
    int32_t p_tiles, o_tiles, num_units, units_per_xcd, o_fastest;
    uint32_t x_bytes, u_bytes, flags;
    FastDiv div_ohw, div_ow, div_hq, div_w4, div_tiles, div_gsplit;
};

#if defined(__HIPCC__)

constexpr uint32_t kOob = 0x80000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), 0x00020000);
}
__device__ __forceinline__ float relu_sel(float v) { return (v > 0.0f) ? v : 0.0f; }

template <int K, int S, bool SECOND>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3, 3))) conv_bf16x3_kernel(const Args a) {
    static_assert(!SECOND || (S == 2 && K == 3), "the second output reads the middle tap of the second phase");
    constexpr int NS = Steps(K, SECOND), PH = Phases(K, S), CS = ChannelSteps(K), PLANE = Plane(K), PART = 2 * CS * PLANE * 16, BUF = BufBytes(K);
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, half = lane >> 5, r = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slot = (blockIdx.x & 7) * a.units_per_xcd + (blockIdx.x >> 3);
    if (slot >= a.num_units * a.gsplit || static_cast<int>(blockIdx.x >> 3) >= a.units_per_xcd) return;
    const int unit = a.gsplit > 1 ? fast_div(slot, a.div_gsplit) : slot;
    const int split = slot - unit * a.gsplit;
    const int major = fast_div(unit, a.div_tiles);
    const int minor = unit - major * (a.o_fastest ? a.o_tiles : a.p_tiles);
    const int p_tile = a.o_fastest ? major : minor, o_tile = a.o_fastest ? minor : major;
    const int m0 = p_tile * kPix;
    const int c_lo = split * a.cps, c_hi = min(c_lo + a.cps, a.csteps);

    int qmin, rows;
    {
        const int n0 = fast_div(m0, a.div_ohw);
        qmin = n0 * a.Hq + fast_div(m0 - n0 * a.OHW, a.div_ow);
        const int ml = min(m0 + kPix, a.M) - 1, n1 = fast_div(ml, a.div_ohw);
        rows = n1 * a.Hq + fast_div(ml - n1 * a.OHW, a.div_ow) + (K - 1) / S - qmin + 1;
    }
    // borders, and rows and columns outside the image, stay zero
    auto clear = [&]() __attribute__((always_inline)) {
        if (K > 1)
            for (int i = tid; i < 2 * BUF / 16; i += kThreads) *reinterpret_cast<u32x4*>(lds + i * 16) = u32x4{0, 0, 0, 0};
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };

    if (wave >= kConsumers) {
        // ---- producers: pieces of four columns x eight channels, split into their three parts once per workgroup
        const int ptid = tid - 64 * kConsumers, per_half = rows * a.w4;
        constexpr int U = K == 1 ? 1 : kUnits;
        uint32_t goff[K == 1 ? 4 : PH][U];           // K = 1: of the four pixels
        int lpos[U], left[U], ch[U];                 // position of the first column's unit; columns that exist; first channel
        if constexpr (K == 1) {
            // (the positions are the tile's pixels)
            const int oct = ptid >> 4, q = ptid & 15;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = m0 + q * 4 + i, n = fast_div(m, a.div_ohw), rem = m - n * a.OHW, oh = fast_div(rem, a.div_ow);
                const int ih = oh * S - a.ph, iw = (rem - oh * a.OW) * S - a.pw;
                const bool ok = m < a.M && ih >= 0 && ih < a.H && iw >= 0 && iw < a.W;
                goff[i][0] = ok ? static_cast<uint32_t>(((n * a.C + oct * 8) * a.H + ih) * a.W + iw) * 4u : kOob;
            }
            ch[0] = oct * 8;
            lpos[0] = oct * PLANE + q * 4;
            left[0] = 4;
        } else {
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const int u = ptid + 64 * kProducers * k;
                const int h = u >= per_half ? 1 : 0, e = u - h * per_half;
                const int row = fast_div(e, a.div_w4), p4 = e - row * a.w4;
                const int Q = qmin + row, n = fast_div(Q, a.div_hq), idx = Q - n * a.Hq;
                const bool ok = u < 2 * per_half && n < a.N;
#pragma unroll
                for (int rho = 0; rho < PH; ++rho) {
                    const int ih = idx * S + rho - a.ph;
                    goff[rho][k] = ok && ih >= 0 && ih < a.H ? static_cast<uint32_t>(((n * a.C + h * 8) * a.H + ih) * a.W + p4 * 4) * 4u : kOob;
                }
                ch[k] = h * 8;
                lpos[k] = h * PLANE + row * a.pitch + p4 * (4 / S);
                left[k] = ok ? a.W - p4 * 4 : 0;
            }
        }
        f32x4 v[2][U][8];          // the next pieces are on their way while the ones before them are split
        auto load = [&](int q, auto set_c) __attribute__((always_inline)) {
            constexpr int SET = decltype(set_c)::value, RHO = PH == 2 ? SET : 0;
            const int c = (c_lo + q / PH) * kStep * CS;
#pragma unroll
            for (int k = 0; k < U; ++k) {
                if (k > 0 && 2 * per_half <= 64 * kProducers * k) break;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t skip = min(static_cast<uint32_t>(c + j) * static_cast<uint32_t>(a.HW) * 4u, a.x_bytes);
                    const __amdgpu_buffer_rsrc_t xr = rsrc(reinterpret_cast<const char*>(a.x) + skip, a.x_bytes - skip);
                    const bool absent = a.tail && c + ch[k] + j >= a.C;
                    if (K > 1 || a.quads) {
                        v[SET][k][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, absent ? kOob : goff[RHO][k], 0, 0));
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            v[SET][k][j][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, absent ? kOob : goff[K == 1 ? i : 0][k], 0, 0));
                    }
                }
            }
        };
        auto store = [&](auto set_c) __attribute__((always_inline)) {
            constexpr int SET = decltype(set_c)::value;
#pragma unroll
            for (int k = 0; k < U; ++k) {
                if (k > 0 && 2 * per_half <= 64 * kProducers * k) break;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float t[8];
#pragma unroll
                    for (int c = 0; c < 8; ++c) t[c] = __fmul_rn(v[SET][k][c][j], kOperandScale);
                    const Split8 s = split8(t);
                    if (j < left[k]) {
                        const int at = K == 1 ? j : ((j + a.pw) % S) * a.hp + (j + a.pw) / S;
                        char* const dst = lds + SET * BUF + (lpos[k] + at) * 16;
                        *reinterpret_cast<u32x4*>(dst) = s.h;
                        *reinterpret_cast<u32x4*>(dst + PART) = s.m;
                        *reinterpret_cast<u32x4*>(dst + 2 * PART) = s.l;
                    }
                }
            }
        };
        using S0 = std::integral_constant<int, 0>;
        using S1 = std::integral_constant<int, 1>;
        const int count = (c_hi - c_lo) * PH;        // buffers full
        load(0, S0{});
        if (count > 1) load(1, S1{});
        clear();
        store(S0{});
        if (count > 2) load(2, S0{});
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        for (int q = 0; q < count; q += 2) {
            // consumers read buffer 0
            if (q + 1 < count) store(S1{});
            if (q + 3 < count) load(q + 3, S1{});
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (q + 1 == count) break;
            // ... buffer 1
            if (q + 2 < count) store(S0{});
            if (q + 4 < count) load(q + 4, S0{});
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        return;
    }

    // ---- consumers: 32 output channels x 64 pixels each
    const int oblk = o_tile * (kOut / 32) + wave, o0 = oblk * 32;
    const __amdgpu_buffer_rsrc_t ur = rsrc(a.u, a.u_bytes);
    const uint32_t avo = o0 < a.O ? static_cast<uint32_t>(lane) * 16u : kOob;
    const uint32_t a_base = o0 < a.O ? static_cast<uint32_t>(oblk * a.csteps) * (NS * 3072u) : 0u;
    uint32_t a_so = a_base + static_cast<uint32_t>(c_lo) * (NS * 3072u);
    const uint32_t a_last = a_base + static_cast<uint32_t>(c_hi) * (NS * 3072u) - 3072u;
    int lbase[2], ybase[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int m = m0 + j * 32 + r, mc = min(m, a.M - 1);
        const int n = fast_div(mc, a.div_ohw), rem = mc - n * a.OHW;
        const int oh = fast_div(rem, a.div_ow), ow = rem - oh * a.OW;
        lbase[j] = (half * PLANE + (K == 1 ? j * 32 + r : (n * a.Hq + oh - qmin) * a.pitch + ow)) * 16;
        ybase[j] = m < a.M ? n * a.O * a.OHW + rem : -1;
    }
    f32x16 big[2], small[2], acc2[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int g = 0; g < 16; ++g) { big[j][g] = 0.0f; small[j][g] = 0.0f; acc2[j][g] = 0.0f; }

    u32x4 ua[2][3], vb[2][3];
    auto load_a = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 3; ++p)
            ua[b][p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ur, avo, a_so + static_cast<uint32_t>(p) * 1024u, 0));
        a_so = min(a_so + 3072u, a_last);
    };
    // parts: 0 = h, 1 = m, 2 = l
    auto read_b = [&](int toff, int p) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            vb[j][p] = *reinterpret_cast<const u32x4*>(lds + p * PART + lbase[j] + toff);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mul = [&](f32x16 (&acc)[2], int b, int pa, int pb) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = mfma_bf16(ua[b][pa], vb[j][pb], acc[j]);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mul0 = [&](f32x16 (&acc)[2], int b, int pa, int pb) __attribute__((always_inline)) {
        f32x16 zero;
#pragma unroll
        for (int g = 0; g < 16; ++g) zero[g] = 0.0f;
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = mfma_bf16(ua[b][pa], vb[j][pb], zero);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto fold = [&](f32x16 (&acc)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int g = 0; g < 16; ++g) acc[j][g] = __fadd_rn(acc[j][g], small[j][g]);
        __builtin_amdgcn_sched_barrier(0);
    };
    // offset of the t-th operand of a row phase in its buffer
    auto operand = [&](int rho, int t) {
        if (K == 1) return t * 2 * PLANE * 16;
        const int tap = TapOf(K, PH, rho, t);
        return ((tap / K / S) * a.pitch + ((tap % K) % S) * a.hp + (tap % K) / S) * 16;
    };
    auto phase = [&](auto rho_c, int buf) __attribute__((always_inline)) {
        constexpr int RHO = decltype(rho_c)::value;
        constexpr int T = K == 1 ? CS : PhaseTaps(K, PH, RHO);
        constexpr int CENTRE = SECOND && RHO == 1 ? 1 : -1;
        constexpr int FIRST = K == 1 ? 0 : PhaseFirst(K, PH, RHO);
        {
            const int t0 = buf + operand(RHO, 0);
            read_b(t0, 2);
            read_b(t0, 1);
            read_b(t0, 0);
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int step = FIRST + t + (CENTRE >= 0 && t > CENTRE ? 1 : 0), b = step & 1;
            const int next = buf + operand(RHO, t + 1 < T ? t + 1 : t);
            load_a(b ^ 1);
            if (SECOND && RHO == 1 && t == CENTRE + 1) mul0(small, b, 0, 2);
            else mul(small, b, 0, 2);
            if (t == CENTRE) {
                // (the same operand: its parts are read again only behind both outputs' products)
                mul(small, b, 1, 1); mul(small, b, 0, 1);
                mul(small, b, 2, 0); mul(small, b, 1, 0); mul(big, b, 0, 0);
                load_a(b);
                mul(acc2, b ^ 1, 0, 0);
                fold(big);
                mul0(small, b ^ 1, 0, 2);
                read_b(next, 2);
                mul(small, b ^ 1, 1, 1); mul(small, b ^ 1, 0, 1);
                read_b(next, 1);
                mul(small, b ^ 1, 2, 0); mul(small, b ^ 1, 1, 0);
                read_b(next, 0);
                fold(acc2);
                continue;
            }
            if (t + 1 < T) read_b(next, 2);
            mul(small, b, 1, 1); mul(small, b, 0, 1);
            if (t + 1 < T) read_b(next, 1);
            mul(small, b, 2, 0); mul(small, b, 1, 0); mul(big, b, 0, 0);
            if (t + 1 < T) read_b(next, 0);
        }
    };
    load_a(0);
    clear();
    asm volatile("s_barrier" ::: "memory");
    for (int c = c_lo; c < c_hi; ++c) {
        phase(std::integral_constant<int, 0>{}, PH == 1 && ((c - c_lo) & 1) ? BUF : 0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if constexpr (PH == 2) {
            phase(std::integral_constant<int, 1>{}, BUF);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        if constexpr (NS & 1) {
#pragma unroll
            for (int p = 0; p < 3; ++p) { const u32x4 t = ua[0][p]; ua[0][p] = ua[1][p]; ua[1][p] = t; }
        }
    }

    // ---- epilogue: lane = pixel, register g = channel 8 (g / 4) + 4 half + g % 4 of the block
    const uint32_t plane = static_cast<uint32_t>(a.OHW) * 4u;
    const uint32_t y_elems = static_cast<uint32_t>(a.M) * static_cast<uint32_t>(a.O), y_bytes = y_elems * 4u;
    const bool raw = a.gsplit > 1;
    uint32_t yb[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) yb[j] = ybase[j] >= 0 ? static_cast<uint32_t>(ybase[j]) * 4u + static_cast<uint32_t>(4 * half) * plane : kOob;
    // (every load of four registers' rows is issued before their first store)
    auto finish = [&](const f32x16 (&acc)[2], const float* bias, const float* res, bool do_relu, float* y) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t yr = rsrc(y, y_bytes), rr = rsrc(res ? res : y, res ? y_bytes : 0u);
        const __amdgpu_buffer_rsrc_t br = rsrc(bias ? bias : y, bias ? static_cast<uint32_t>(a.O) * 4u : 0u);
        uint32_t odd = 0;             // bit 2 * register + pixel block
#pragma unroll
        for (int gq = 0; gq < 4; ++gq) {
            float q[4][2], bv[4];
            uint32_t off[4][2];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int o = o0 + 8 * gq + 4 * half + e;
                bv[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(br, o < a.O ? static_cast<uint32_t>(o) * 4u : kOob, 0, 0));
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    off[e][j] = o < a.O && yb[j] != kOob ? yb[j] + static_cast<uint32_t>(o0 + 8 * gq + e) * plane : kOob;
                    if (res) q[e][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rr, off[e][j], 0, 0));
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    float v = acc[j][gq * 4 + e];
                    if (!(__builtin_fabsf(v) < __builtin_inff()) && off[e][j] != kOob) {
                        odd |= 1u << (2 * (gq * 4 + e) + j);
                        off[e][j] = kOob;
                    }
                    if (bias) v = __fadd_rn(v, bv[e]);
                    if (res) v = __fadd_rn(v, q[e][j]);
                    if (do_relu) v = relu_sel(v);
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), yr, off[e][j], 0, 0);
                }
        }
        return odd;
    };
    const bool has_bias = !raw && (a.flags & KXC_HIP_CONV_BIAS) != 0, has_res = !raw && (a.flags & KXC_HIP_CONV_RESIDUAL) != 0;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int g = 0; g < 16; ++g) {
            big[j][g] = __fmul_rn(__fadd_rn(big[j][g], small[j][g]), kSumScale);
            if constexpr (SECOND) acc2[j][g] = __fmul_rn(acc2[j][g], kSumScale);
        }
    const float* const bias = has_bias ? a.bias : nullptr;
    const float* const res = has_res ? a.res : nullptr;
    const float* const bias2 = raw ? nullptr : a.bias2;
    const bool do_relu = !raw && (a.flags & KXC_HIP_CONV_RELU) != 0;
    float* const y = raw ? a.partial + static_cast<int64_t>(split) * y_elems : a.y;
    float* const y2 = raw ? a.partial + static_cast<int64_t>(a.gsplit + split) * y_elems : a.y2;
    const uint32_t odd = finish(big, bias, res, do_relu, y);
    uint32_t odd2 = 0;
    if constexpr (SECOND) odd2 = finish(acc2, bias2, nullptr, false, y2);
    // Splitting turns an infinite operand into NaN, and so does it to one of 2^112 and more, and sums (times 2^32 here) overflow
    // from 2^96 on: a sum that is not finite is formed again by the operator's definition, over the channels of
    // this part.  Nothing is stored before (the residual may be the output's own buffer).
    if ((odd | odd2) == 0) return;
    auto again = [&](uint32_t mask, const float* w, bool one_tap, const float* bias, const float* res, bool do_relu, float* out) __attribute__((always_inline)) {
#pragma unroll 1
        for (int k = 0; k < 32; ++k) {
            if (!((mask >> k) & 1u)) continue;
            const int o = o0 + 8 * (k >> 3) + 4 * half + (k >> 1 & 3);
            const int m = m0 + (k & 1) * 32 + r, n = fast_div(m, a.div_ohw), rem = m - n * a.OHW, oh = fast_div(rem, a.div_ow), ow = rem - oh * a.OW;
            const int64_t at = static_cast<int64_t>(n * a.O + o) * a.OHW + rem;
            float s = 0.0f;
#pragma unroll 1
            for (int c = c_lo * kStep * CS; c < min(c_hi * kStep * CS, a.C); ++c) {
                const float* const xc = a.x + static_cast<int64_t>(n * a.C + c) * a.HW;
                if (one_tap) {
                    s = __fadd_rn(s, __fmul_rn(xc[oh * S * a.W + ow * S], w[static_cast<int64_t>(o) * a.C + c]));
                    continue;
                }
#pragma unroll 1
                for (int t = 0; t < K * K; ++t) {
                    const int ih = oh * S + t / K - a.ph, iw = ow * S + t % K - a.pw;
                    const bool in = ih >= 0 && ih < a.H && iw >= 0 && iw < a.W;
                    s = __fadd_rn(s, __fmul_rn(in ? xc[ih * a.W + iw] : 0.0f, w[(static_cast<int64_t>(o) * a.C + c) * K * K + t]));
                }
            }
            if (bias) s = __fadd_rn(s, bias[o]);
            if (res) s = __fadd_rn(s, res[at]);
            out[at] = do_relu ? relu_sel(s) : s;
        }
    };
    again(odd, a.w, false, bias, res, do_relu, y);
    if constexpr (SECOND) again(odd2, a.w2, true, bias2, nullptr, false, y2);
}

// ------------------------------------------------------------------------------------------
// The packed filter: [o / 32][c / 16 (64 for 1x1 filters)][step][part][lane][16 bytes], lane = o % 32 + 32 * (c / 8 % 2).  A
// workgroup of 256 threads takes 8 output channels of one [c]: their filters pass through LDS (PackFloats(K) floats), so that they
// are read as they lie in memory.
// ------------------------------------------------------------------------------------------
template <int K, int S>
__device__ __forceinline__ void pack_block(const float* __restrict__ w, const float* __restrict__ w2, char* __restrict__ u, int32_t O, int32_t C,
                                           int block, float* raw) {
    constexpr int KK = K * K, CH = kStep * ChannelSteps(K), RUN = CH * KK, PH = Phases(K, S);
    const bool second = w2 != nullptr;
    const int ns = Steps(K, second), csteps = (C + CH - 1) / CH;
    const int og = block / csteps, cs = block - og * csteps, c0 = cs * CH, run = min(CH, C - c0) * KK;
    const int tid = static_cast<int>(threadIdx.x);
    float t[(8 * RUN + 255) / 256];
#pragma unroll
    for (int k = 0; k < (8 * RUN + 255) / 256; ++k) {
        const int i = k * 256 + tid, ol = i / RUN, r = i - ol * RUN;
        const bool ok = ol < 8 && og * 8 + ol < O && r < run;
        const float x = w[ok ? (static_cast<int64_t>(og * 8 + ol) * C + c0) * KK + r : 0];
        t[k] = ok ? x : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < (8 * RUN + 255) / 256; ++k) {
        const int i = k * 256 + tid, ol = i / RUN;
        if (ol < 8) raw[ol * (RUN + 1) + i - ol * RUN] = t[k];
    }
    __syncthreads();
    const int n0 = PhaseTaps(K, PH, 0), centre = n0 + 1;            // (second: K = 3, S = 2, tap (1, 1))
    for (int i = tid; i < ns * 16; i += 256) {
        const int ol = i & 7, half = (i >> 3) & 1, step = i >> 4, o = og * 8 + ol;
        const bool is2 = second && step == centre + 1;
        const int tt = second && step > centre ? step - 1 : step;
        const int tap = K == 1 ? 0 : tt < n0 ? TapOf(K, PH, 0, tt) : TapOf(K, PH, 1, tt - n0), first = (K == 1 ? step * kStep : 0) + half * 8;
        float v[8];
#pragma unroll
        for (int c = 0; c < 8; ++c)
            v[c] = kOperandScale * (is2 ? (o < O && c0 + half * 8 + c < C ? w2[static_cast<int64_t>(o) * C + c0 + half * 8 + c] : 0.0f) : raw[ol * (RUN + 1) + (first + c) * KK + tap]);
        const Split8 s = split8(v);
        char* const dst = u + ((static_cast<int64_t>(o / 32) * csteps + cs) * ns + step) * 3072 + (half * 32 + o % 32) * 16;
        *reinterpret_cast<u32x4*>(dst) = s.h;
        *reinterpret_cast<u32x4*>(dst + 1024) = s.m;
        *reinterpret_cast<u32x4*>(dst + 2048) = s.l;
    }
}

#endif  // __HIPCC__

}  // namespace conv_bx
}  // namespace kxc_hip
