// conv_slice.h -- 3x3 convolutions of launches too small for the large-tile kernels, on the bf16 matrix cores with three-part operands
// (bf16x3.h) and a packed filter (conv_bf16x3.h's layout); included by conv2d_slice.hip (selection, launch).
//
// D[o][pixel] += W[o][tap, c] X[tap, c][pixel].  A workgroup owns 32 RO output channels x 32 pixels (neighbours, flattened over n, oh,
// ow) and its KS waves split the input channels: wave w takes the steps w, w + KS, ... of 16 channels, each by itself and with LDS of
// its own, so that nothing waits for another wave until the KS partial tiles meet at the end.  One launch, no scratch, no adding kernel.
//  * X: the input under the tile, eight loads of 16 bytes a lane and step (four columns x eight channels), split into three parts once
//    and left in LDS as the 16-byte fragments that the matrix instructions take: [part][channels c .. c + 7][position].  The next
//    step's loads are in flight while this one multiplies.  Positions are either whole input rows, shared by the output rows above and
//    below (narrow maps), or the columns under each output row of the tile, side by side (`seg`).
//  * W: fragments straight from memory into registers, D filter steps ahead.
//  * Large and small products have accumulators of their own (conv_bf16x3.h says why).  Relative error against float64 (2-norm), 64
//    channels at 49 x 49, batch 6 / 256 at 14 x 14, batch 2 / 512 at 7 x 7, batch 4: 0.5e-7 / 0.6e-7 / 0.7e-7, the fp32
//    instructions in the kernels that took these layers before 1.7e-7 / 1.7e-7 / 1.1e-7.
//
// What bounds it: a wave's 54 matrix instructions of a step take 1840 cycles when nothing else is needed, and 27 KiB of W and
// 8 of X a step come at 64 bytes a clock and compute unit, 8700 cycles of the 16 200 that 256 channels at 13 x 13, batch 6 take (10.6
// us; 6900 of matrix instructions).  Two blocks of output channels (RO = 2) share a patch, not W.  Around that, in cycles: 1500 until
// the first load of X (2200 before all arguments were requested at once), 3500 until it is split, 2000 at the barrier and 500 behind
// it.  Loads issued in a row stall a wave on the address unit (W all at once ahead of the split: 11.8 us), so they stand between
// other instructions.
// Measured in a plan, residual and ReLU, us, the kernel that took the layer before and here: 64 channels at 49 x 49, batch 3 / 6 12.3 / 16.2 and
// 7.0 / 10.0; 128 at 25 x 25 11.0 / 18.0 and 7.3 / 9.5; 256 at 13 x 13 10.6 / 22.6 and 9.2 / 10.6; 512 at 7 x 7 16.7 / 22.4 and 15.0
// both; batch 8, 128 at 28 x 28 21.1 and 13.8, 256 at 14 x 14 22.5 and 14.7.  Blocks of 64 pixels were slower at all but a few sizes.
#pragma once

#include "bf16x3.h"
#include "common.h"
#include "conv_bf16x3.h"

namespace kxc_hip {
namespace conv_sl {

constexpr int kStep = conv_bx::kStep;
constexpr int kK = 3, kPix = 32;          // filter extent; pixels of a workgroup
// Loads of a lane and channel (of 32 pieces of four columns each); positions of an LDS plane.
constexpr int Passes(int S) { return S; }
constexpr int Plane(int S) { return S == 2 ? 212 : 128; }
constexpr int WaveBytes(int S) { return 6 * Plane(S) * 16; }

struct Args {
    const float* x;
    const char* u;
    const float* bias;
    const float* res;
    float* y;
    const float* bias2;
    float* y2;
    const float* w;                     // the filters as they were given, for outputs that are not finite
    const float* w2;
    int32_t N, C, H, W, O, OH, OW, M, OHW, HW, ph, pw;
    int32_t seg;                        // 1: the columns under each output row, 0: whole rows
    int32_t Hq, w4, full4;              // rows per image and pieces per row (whole rows); pieces under a whole output row (seg)
    int32_t pitch, hp;                  // positions of a patch row; stride 2: of its even columns
    int32_t csteps, tail;
    int32_t p_tiles, o_tiles, num_tiles, tiles_per_xcd, o_fastest;
    uint32_t x_bytes, u_bytes, flags;
    FastDiv div_ohw, div_ow, div_oh, div_hq, div_w4, div_full4, div_tiles;
};

#if defined(__HIPCC__)

using conv_bx::kOob;
using conv_bx::relu_sel;
using conv_bx::rsrc;

template <int S, int RO, int KS, bool DS>
__global__ void __launch_bounds__(64 * KS) __attribute__((amdgpu_waves_per_eu(2))) conv_slice_kernel(const Args a) {
    static_assert(!DS || S == 2, "the second output's filter lies behind the centre tap of the second phase");
    constexpr int K = kK, KK = K * K, E = (K - 1) / S, NP = Passes(S), PL = Plane(S), PART = 2 * PL * 16;
    constexpr int TP = kPix, NB = RO * (DS ? 2 : 1);
    constexpr int NS = conv_bx::Steps(K, DS);
    // filter steps in registers: all of a step of channels where one tap's products are few
    constexpr int D = RO > 1 ? (DS ? 5 : 3) : (DS ? 5 : 9);
    static_assert(NS % D == 0, "a filter step stays in its slot");
    static_assert(WaveBytes(S) >= NB * 4096, "the partial tiles take the patch's place");
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, half = lane >> 5, r = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // (every line of the arguments is requested at once: one by one, as they are needed, each is a round trip to memory)
    asm volatile("" ::"s"(a.num_tiles), "s"(a.x), "s"(a.u), "s"(a.N), "s"(a.C), "s"(a.H), "s"(a.W), "s"(a.OH), "s"(a.OW), "s"(a.M), "s"(a.seg), "s"(a.Hq), "s"(a.w4),
                 "s"(a.pitch), "s"(a.csteps), "s"(a.x_bytes), "s"(a.div_ohw.mul), "s"(a.div_ow.mul), "s"(a.div_oh.mul), "s"(a.div_hq.mul), "s"(a.div_w4.mul), "s"(a.div_tiles.mul));
    const int tile = static_cast<int>(blockIdx.x & 7) * a.tiles_per_xcd + static_cast<int>(blockIdx.x >> 3);
    if (tile >= a.num_tiles || static_cast<int>(blockIdx.x >> 3) >= a.tiles_per_xcd) return;
    const int hi = fast_div(tile, a.div_tiles), lo = tile - hi * (a.o_fastest ? a.o_tiles : a.p_tiles);
    const int o0 = (a.o_fastest ? lo : hi) * 32 * RO, m0 = (a.o_fastest ? hi : lo) * TP;
    char* const mine = lds + wave * WaveBytes(S);

    // ---- filter fragments: [o / 32][step of channels][filter step][part] runs of 1 KiB
    const __amdgpu_buffer_rsrc_t ur = rsrc(a.u, a.u_bytes);
    u32x4 ua[D][RO][3];
    auto load_w = [&](int step, int fs, int i, int p) __attribute__((always_inline)) {
        const int ob = o0 / 32 + i;
        const uint32_t so = (static_cast<uint32_t>(ob * a.csteps + step) * NS + static_cast<uint32_t>(fs)) * 3072u + static_cast<uint32_t>(p) * 1024u;
        // (the range check does not see the scalar offset: absent channel blocks are masked in the vector offset)
        ua[fs % D][i][p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ur, ob * 32 < a.O ? static_cast<uint32_t>(lane) * 16u : kOob, so, 0));
    };
    // The address unit takes 16 cycles a load for all waves of a compute unit: a few go out before the geometry is worked out, the others
    // behind the patch's, one by one between the instructions that split it.
    constexpr int kWLoads = D * RO * 3, kEarly = 6;
    auto first_w = [&](int from, int to) __attribute__((always_inline)) {
#pragma unroll
        for (int e = from; e < to; ++e) load_w(wave, e / (3 * RO), e % (3 * RO) / 3, e % 3);
        __builtin_amdgcn_sched_barrier(0);
    };
    if (wave < a.csteps) first_w(0, kEarly);

    // ---- the patch: a lane's pieces of four columns (goff: of channel 0 of its half; left: columns that are written; lpos: position of
    // the first one, odd: of the second one with stride 2)
    const int ml = min(m0 + TP, a.M) - 1;
    const int R0 = fast_div(m0, a.div_ow), R1 = fast_div(ml, a.div_ow);              // output rows, over all images
    const int n0 = fast_div(m0, a.div_ohw);
    const int qmin = n0 * a.Hq + (R0 - n0 * a.OH) * S;
    uint32_t goff[NP];
    int left[NP], lpos[NP], lodd[NP];
    {
        const int ow0 = m0 - R0 * a.OW;
        auto pieces = [&](int from, int to) {      // under output columns from .. to: first input column and pieces
            const int f = max(from * S - a.pw, 0), e = min(to * S - a.pw + K, a.W);
            return (e - f + 3) >> 2;
        };
        const int last = ml - R1 * a.OW;
        const int first4 = pieces(ow0, R1 > R0 ? a.OW - 1 : last);
        const int row4 = first4 + (R1 > R0 ? (R1 - R0 - 1) * a.full4 + pieces(0, last) : 0);
        const int rows = fast_div(ml, a.div_ohw) * a.Hq + (R1 - fast_div(ml, a.div_ohw) * a.OH) * S + K - qmin;
#pragma unroll
        for (int k = 0; k < NP; ++k) {
            const int u = r + 32 * k;
            int n, ih, col, lc, at, odd;
            bool ok;
            if (a.seg) {
                const int kh = (u >= row4 ? 1 : 0) + (u >= 2 * row4 ? 1 : 0), v = u - kh * row4;
                const int past = max(v - first4, 0), s = v < first4 ? 0 : 1 + fast_div(past, a.div_full4);
                const int piece = v < first4 ? v : past - (s - 1) * a.full4;
                const int R = R0 + s, from = s == 0 ? ow0 : 0, to = R == R1 ? last : a.OW - 1;
                n = fast_div(R, a.div_oh);
                ih = (R - n * a.OH) * S - a.ph + kh;
                const int cs = from * S - a.pw;
                col = max(cs, 0) + 4 * piece;
                lc = col - cs;
                left[k] = min(to * S - a.pw + K, a.W) - col;
                const int first = s == 0 ? 0 : s * a.OW - ow0;        // of the row's pixels in the tile
                at = kh * a.pitch + first + s * E;
                odd = kh * a.pitch + a.hp + first;
                ok = u < 3 * row4;
            } else {
                const int row = fast_div(u, a.div_w4), Q = qmin + row;
                n = fast_div(Q, a.div_hq);
                ih = Q - n * a.Hq - a.ph;
                col = 4 * (u - row * a.w4);
                lc = col + a.pw;
                left[k] = a.W - col;
                at = row * a.pitch;
                odd = at + a.hp;
                ok = row < rows && n < a.N;
            }
            ok = ok && ih >= 0 && ih < a.H;
            goff[k] = ok ? static_cast<uint32_t>(((n * a.C + half * 8) * a.H + ih) * a.W + col) * 4u : kOob;
            if (!ok) left[k] = 0;
            if constexpr (S == 1) {
                lpos[k] = (half * PL + at + lc) * 16;
                lodd[k] = 0;
            } else {
                lpos[k] = (half * PL + ((lc & 1) ? odd : at) + (lc >> 1)) * 16;
                lodd[k] = (half * PL + ((lc & 1) ? at : odd) + ((lc + 1) >> 1)) * 16;
            }
        }
    }
    f32x4 xv[NP][8];
    const uint32_t plane_in = static_cast<uint32_t>(a.HW) * 4u;
    // (the step is part of the base, so that the range check ends the last piece of a row at the end of the tensor)
    auto patch_of = [&](int step) __attribute__((always_inline)) {
        const uint32_t skip = static_cast<uint32_t>(step * kStep) * plane_in;
        return rsrc(reinterpret_cast<const char*>(a.x) + skip, a.x_bytes - skip);
    };
    auto load_x = [&](__amdgpu_buffer_rsrc_t xr, int step, int e) __attribute__((always_inline)) {
        const int k = e >> 3, j = e & 7;
        const bool absent = a.tail && step * kStep + half * 8 + j >= a.C;
        xv[k][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, absent ? kOob : goff[k] + static_cast<uint32_t>(j) * plane_in, 0, 0));
    };
    auto store_x = [&](auto first_c) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < NP; ++k)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (decltype(first_c)::value) {
                    constexpr int kParts = NP * 4, kLate = kWLoads - kEarly;
                    first_w(kEarly + kLate * (k * 4 + j) / kParts, kEarly + kLate * (k * 4 + j + 1) / kParts);
                }
                float t[8];
#pragma unroll
                for (int c = 0; c < 8; ++c) t[c] = __fmul_rn(xv[k][c][j], kOperandScale);
                const Split8 s = split8(t);
                if (j < left[k]) {
                    char* const dst = mine + (S == 1 ? lpos[k] + j * 16 : ((j & 1) ? lodd[k] : lpos[k]) + (j >> 1) * 16);
                    *reinterpret_cast<u32x4*>(dst) = s.h;
                    *reinterpret_cast<u32x4*>(dst + PART) = s.m;
                    *reinterpret_cast<u32x4*>(dst + 2 * PART) = s.l;
                }
            }
    };

    if (wave < a.csteps) {
        const __amdgpu_buffer_rsrc_t xr = patch_of(wave);
#pragma unroll
        for (int e = 0; e < NP * 8; ++e) load_x(xr, wave, e);
    }
    __builtin_amdgcn_sched_barrier(0);
    // borders, and rows and columns outside the image, stay zero
#pragma unroll
    for (int i = 0; i < (WaveBytes(S) + 1023) / 1024; ++i)
        if ((i + 1) * 1024 <= WaveBytes(S) || i * 1024 + lane * 16 < WaveBytes(S)) *reinterpret_cast<u32x4*>(mine + i * 1024 + lane * 16) = u32x4{0, 0, 0, 0};

    // ---- where this lane's pixel is in the patch
    int rd, rd_odd;
    {
        const int m = min(m0 + r, a.M - 1), R = fast_div(m, a.div_ow);
        if (a.seg) {
            rd = m - m0 + (R - R0) * E;
            rd_odd = S == 2 ? m - m0 : 0;
        } else {
            const int n = fast_div(m, a.div_ohw);
            rd = (n * a.Hq + (R - n * a.OH) * S - qmin) * a.pitch + m - R * a.OW;
            rd_odd = rd;
        }
        rd = (half * PL + rd) * 16;
        rd_odd = (half * PL + rd_odd + a.hp) * 16;
    }
    __builtin_amdgcn_sched_barrier(0);

    f32x16 big[NB], small[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int g = 0; g < 16; ++g) { big[b][g] = 0.0f; small[b][g] = 0.0f; }
    u32x4 vb[3];
    // tap of a filter step, and whether it belongs to the second output
    constexpr int PH = conv_bx::Phases(K, S), kFirst = conv_bx::PhaseTaps(K, PH, 0), kSecond = DS ? kFirst + 2 : -1;
    auto tap_of = [](int fs) constexpr {
        const int t = DS && fs >= kSecond ? fs - 1 : fs;
        return t < kFirst ? conv_bx::TapOf(K, PH, 0, t) : conv_bx::TapOf(K, PH, 1, t - kFirst);
    };
    auto read_b = [&](int fs, int p) __attribute__((always_inline)) {
        const int tap = tap_of(fs), kh = tap / K, kw = tap % K;
        vb[p] = *reinterpret_cast<const u32x4*>(mine + (kw % S ? rd_odd : rd) + (kh * a.pitch + kw / S) * 16 + p * PART);
        __builtin_amdgcn_sched_barrier(0);
    };
    // One step of 16 channels; `more`: the wave's next step, whose loads are issued one by one between the products.
    auto multiply = [&](int step, auto more_c) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(more_c)::value;
        constexpr int PA[6] = {0, 1, 0, 2, 1, 0}, PB[6] = {2, 1, 1, 0, 0, 0};
        const __amdgpu_buffer_rsrc_t xr = patch_of(MORE ? step + KS : step);
        read_b(0, 2);
        read_b(0, 1);
        read_b(0, 0);
#pragma unroll
        for (int fs = 0; fs < NS; ++fs) {
            const bool second = fs == kSecond, next = fs + 1 < NS && fs + 1 != kSecond;
#pragma unroll
            for (int p = 0; p < 6; ++p) {
#pragma unroll
                for (int i = 0; i < RO; ++i) {
                    f32x16& acc = p == 5 ? big[(second ? RO : 0) + i] : small[(second ? RO : 0) + i];
                    acc = mfma_bf16(ua[fs % D][i][PA[p]], vb[PB[p]], acc);
                }
                __builtin_amdgcn_sched_barrier(0);
                // (a part is read again, or loaded again, behind the last product that takes it)
                if (next && p == 0) read_b(fs + 1, 2);
                if (next && p == 2) read_b(fs + 1, 1);
                if (next && p == 5) read_b(fs + 1, 0);
                if (p >= 3) {
                    const int part = 5 - p;      // 2, 1, 0
#pragma unroll
                    for (int i = 0; i < RO; ++i) {
                        if (fs + D < NS) load_w(step, fs + D, i, part);
                        else if (MORE) load_w(step + KS, fs + D - NS, i, part);
                    }
                } else if (MORE && fs * 3 + p < NP * 8) {
                    load_x(xr, step + KS, fs * 3 + p);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // ---- the outputs that this thread finishes: their bias and residual are on their way while the last products are formed
    constexpr int kTasks = NB * 256, T = 64 * KS, kRounds = (kTasks + T - 1) / T;
    const uint32_t plane = static_cast<uint32_t>(a.OHW) * 4u, y_bytes = static_cast<uint32_t>(a.M) * static_cast<uint32_t>(a.O) * 4u;
    const bool has_bias = (a.flags & KXC_HIP_CONV_BIAS) != 0, has_res = (a.flags & KXC_HIP_CONV_RESIDUAL) != 0, do_relu = (a.flags & KXC_HIP_CONV_RELU) != 0;
    const bool has_bias2 = DS && a.bias2 != nullptr;
    f32x4 bv[kRounds], qv[kRounds];
    uint32_t off[kRounds];                        // of the first of four channels
    // A wave's share of a round: four channels of 32 pixels for either half, of one block.
    auto block_of = [&](int t) __attribute__((always_inline)) { return (t * T + wave * 64) >> 8; };
    auto channel_of = [&](int t) __attribute__((always_inline)) {
        const int b = block_of(t);
        return o0 + (DS && b >= RO ? b - RO : b) * 32 + 8 * ((t * KS + wave) & 3) + 4 * half;
    };
    auto epilogue_loads = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < kRounds; ++t) {
            const int b = block_of(t), o = channel_of(t), m = m0 + r, n = fast_div(m, a.div_ohw);
            const bool second = DS && b >= RO, ok = b < NB && m < a.M;
            off[t] = ok ? static_cast<uint32_t>((n * a.O + o) * a.OHW + m - n * a.OHW) * 4u : kOob;
            const float* const bias = second ? (has_bias2 ? a.bias2 : nullptr) : has_bias ? a.bias : nullptr;
            const __amdgpu_buffer_rsrc_t br = rsrc(bias ? bias : a.y, bias ? static_cast<uint32_t>(a.O) * 4u : 0u);
            const __amdgpu_buffer_rsrc_t rr = rsrc(has_res && !second ? a.res : a.y, has_res && !second ? y_bytes : 0u);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool there = ok && o + e < a.O;
                bv[t][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(br, there ? static_cast<uint32_t>(o + e) * 4u : kOob, 0, 0));
                qv[t][e] = 0.0f;
                if (has_res && !second) qv[t][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rr, there ? off[t] + static_cast<uint32_t>(e) * plane : kOob, 0, 0));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    if (wave < a.csteps) {
        int step = wave;
        store_x(std::true_type{});
        for (; step + KS < a.csteps; step += KS) {
            multiply(step, std::true_type{});
            store_x(std::false_type{});
        }
        epilogue_loads();
        multiply(step, std::false_type{});
    } else {
        epilogue_loads();
    }

    // ---- partial tiles into the wave's own LDS: [block][four rows][lane][16 bytes], lane = pixel, register g = channel 8 (g / 4) + 4 half
    // + g % 4 of the block; then every thread adds and finishes some of them
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = __fmul_rn(__fadd_rn(big[b][4 * q + e], small[b][4 * q + e]), kSumScale);
            *reinterpret_cast<f32x4*>(mine + ((b * 4 + q) * 64 + lane) * 16) = v;
        }
    __syncthreads();
    uint32_t odd = 0;
#pragma unroll
    for (int t = 0; t < kRounds; ++t) {
        const int b = block_of(t), o = channel_of(t), at = (t * T + tid) * 16;
        if (b >= NB) break;
        const bool second = DS && b >= RO;
        f32x4 v = *reinterpret_cast<const f32x4*>(lds + at);
#pragma unroll
        for (int w = 1; w < KS; ++w) {
            const f32x4 p = *reinterpret_cast<const f32x4*>(lds + w * WaveBytes(S) + at);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = __fadd_rn(v[e], p[e]);
        }
        const __amdgpu_buffer_rsrc_t yr = rsrc(second ? a.y2 : a.y, y_bytes);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            bool store = off[t] != kOob && o + e < a.O;
            if (store && !(__builtin_fabsf(v[e]) < __builtin_inff())) {
                odd |= 1u << (4 * t + e);
                store = false;
            }
            float z = v[e];
            if (second ? has_bias2 : has_bias) z = __fadd_rn(z, bv[t][e]);
            if (!second) {
                if (has_res) z = __fadd_rn(z, qv[t][e]);
                if (do_relu) z = relu_sel(z);
            }
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, z), yr, store ? off[t] + static_cast<uint32_t>(e) * plane : kOob, 0, 0);
        }
    }
    // Sums that are not finite are formed again by the operator's definition (conv_bf16x3.h says when that happens).
    if (odd == 0) return;
#pragma unroll 1
    for (int k = 0; k < 4 * kRounds; ++k) {
        if (!((odd >> k) & 1u)) continue;
        const int b = block_of(k >> 2), o = channel_of(k >> 2) + (k & 3);
        const bool second = DS && b >= RO;
        const int m = m0 + r, n = fast_div(m, a.div_ohw), rem = m - n * a.OHW, oh = fast_div(rem, a.div_ow), ow = rem - oh * a.OW;
        const int64_t at = static_cast<int64_t>(n * a.O + o) * a.OHW + rem;
        float s = 0.0f;
#pragma unroll 1
        for (int c = 0; c < a.C; ++c) {
            const float* const xc = a.x + static_cast<int64_t>(n * a.C + c) * a.HW;
            if (second) {
                s = __fadd_rn(s, __fmul_rn(xc[oh * S * a.W + ow * S], a.w2[static_cast<int64_t>(o) * a.C + c]));
                continue;
            }
#pragma unroll 1
            for (int q = 0; q < KK; ++q) {
                const int ih = oh * S + q / K - a.ph, iw = ow * S + q % K - a.pw;
                const bool in = ih >= 0 && ih < a.H && iw >= 0 && iw < a.W;
                s = __fadd_rn(s, __fmul_rn(in ? xc[ih * a.W + iw] : 0.0f, a.w[(static_cast<int64_t>(o) * a.C + c) * KK + q]));
            }
        }
        if (second) {
            if (has_bias2) s = __fadd_rn(s, a.bias2[o]);
            a.y2[at] = s;
        } else {
            if (has_bias) s = __fadd_rn(s, a.bias[o]);
            if (has_res) s = __fadd_rn(s, a.res[at]);
            a.y[at] = do_relu ? relu_sel(s) : s;
        }
    }
}

#endif  // __HIPCC__

}  // namespace conv_sl
}  // namespace kxc_hip
