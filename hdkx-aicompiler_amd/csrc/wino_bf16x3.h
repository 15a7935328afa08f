// wino_bf16x3.h -- Winograd F(2x2, 3x3) on the bf16 matrix cores with three-part operands (bf16x3.h); included by
// conv2d_wino_f32.hip, which holds the fp32-instruction kernel for small launches, the selection and the entry points.
//
// A workgroup of eight waves owns 64 output channels x 64 tiles (2x2 outputs each) x all 16 positions f = (i, j) of the
// transform domain.  Wave (i, jp) computes f = (i, 2 jp) and (i, 2 jp + 1) for the whole 64 x 64 block: 128 accumulator
// registers, two waves per SIMD.  Why it is split this way and what bounds it:
//  * every U fragment and every V element is used by exactly one wave, so neither passes through LDS: U streams from
//    memory in the order the lanes read it (packed once per weight tensor, 96 bytes per (o, c)), and a wave transforms
//    the input it needs straight into matrix operands.  The L2 traffic of U sets the 64 x 64 block: half as many tiles
//    would double it to 64 bytes per clock and compute unit, the L2's limit.
//  * LDS holds only the raw input patches of 16 channels (filled by LDS-direct loads, three in flight).  A load occupies the
//    address unit for 16 cycles however wide it is, and with 4-byte loads the patches took half of every step there (with
//    three of four left out, timing only, 64 images: 82 -> 65, 63 -> 52, 52 -> 46, 68 -> 53 us for the layers below), so rows
//    come in pieces of 16 bytes wherever the padding allows it (WIDE).
//  * A wave's vector instructions do not run beside its own matrix instructions, only beside the other wave's of its
//    SIMD (measured: four vector instructions between two v_mfma_f32_32x32x16_bf16 of one wave add 15 cycles, issued by
//    another wave nothing), so the two waves of a SIMD work in opposite phases.  Per step of 16 channels a SIMD has 3072
//    cycles of matrix instructions, 1.8 us at the rate that a loop of nothing else reaches; a step takes about 2.2 us
//    (2.5-2.7 with 4-byte patch loads).  Loads issued in a row stall a wave on the address unit, so they stand one by one
//    between matrix instructions.
// The output transform needs all 16 f of one (o, tile): every wave applies the column half to its own two positions and
// leaves two values per (o, tile) in LDS, 32 x 32 outputs at a time; the row half sums over the eight waves.
//
// Measured (64 images, against 4-byte patch loads and the fp32-instruction kernel, us): 64 channels at 56 x 56 71 / 83 / 99,
// 128 at 28 x 28 54 / 64 / 90, 256 at 14 x 14 48 / 52 / 87, 512 at 7 x 7 62 / 67 / 88; 32 images 35 / 41 / 51, 28 / 33 / 47,
// 35 / 38 / 55, 39 / 42 / 55.  Relative error against
// float64 (2-norm): 1.0e-7 to 1.4e-7, the fp32-instruction kernel 1.3e-7 to 1.7e-7.
#pragma once

#include <algorithm>

#include "bf16x3.h"

namespace kxc_hip {
namespace wino_bx {

constexpr int kTiles = 64, kOut = 64, kStep = 16;        // tiles, output channels per workgroup; channels per step
constexpr int kThreads = 512;
// Floats per channel of the patch in LDS (template parameter): even columns in the first half, odd ones in the second, so
// that neighbouring tiles, two columns apart, read neighbouring words.
constexpr int kPlanes[2] = {512, 768};
constexpr size_t kLdsBytes = 3u * kStep * 768 * sizeof(float);       // 144 KiB: three patches, or the epilogue's two exchange areas

// Bytes of the packed three-part filter: [o / 32][c / 16][f][part][lane][16 bytes], lane = o % 32 + 32 * (c / 8 % 2).
inline size_t WeightBytes(int64_t O, int64_t C) { return static_cast<size_t>(CeilDiv(O, 32) * CeilDiv(C, kStep)) * 16 * 3 * 1024; }

// How the patch gets into LDS (template parameter).  kNarrow: 4-byte loads, even and odd columns in half planes of their own;
// any padding.  kWide, for a padding of one column: rows as they are in memory in pieces of 16 bytes behind one piece that
// reads as zero, which is the left border of its row and the right border of the row before.  kWideEdge: the same where the
// rows are no multiple of four floats; their last piece ends in floats of the next row, which the reader replaces by zeros.
enum PatchLoads { kNarrow = 0, kWide = 1, kWideEdge = 2 };

// Row pitch of a half plane (at least TW + 1): the smallest that puts 32 neighbouring tiles into different LDS banks, or the
// best one that fits `limit`.  The rows of a tile row are two pitches apart: at 14 x 14 outputs (7 tiles a row) a pitch of 8
// puts every second tile row into the same banks (measured: 3072 of 8300 cycles per step lost to conflicts).
inline int32_t RowPitch(int64_t TW, int64_t rows, int64_t limit) {
    int32_t best = static_cast<int32_t>(TW + 1);
    int best_worst = 1 << 30;
    for (int64_t pitch = TW + 1; pitch <= TW + 32 && 2 * rows * pitch <= limit; ++pitch) {
        int count[32] = {0}, worst = 0;
        for (int t = 0; t < 32; ++t) {
            const int c = ++count[(t / TW * 2 * pitch + t % TW) % 32];
            if (c > worst) worst = c;
        }
        if (worst < best_worst) { best_worst = worst; best = static_cast<int32_t>(pitch); }
        if (worst == 1) break;
    }
    return best;
}

// Row pitch of a kWide plane: a zero piece and the row, and more zero pieces where that spreads 32 neighbouring tiles better
// over the banks (a lane reads 8 bytes; the rows of a tile row are two pitches apart).
inline int32_t WideRowPitch(int64_t W, int64_t TW, int64_t rows, int64_t limit) {
    const int64_t least = 4 + CeilDiv(W, 4) * 4;
    int32_t best = static_cast<int32_t>(least);
    int best_worst = 1 << 30;
    for (int64_t pitch = least; pitch <= least + 28 && rows * pitch + 4 <= limit; pitch += 4) {
        int count[32] = {0}, worst = 0;
        for (int t = 0; t < 32; ++t) worst = std::max(worst, ++count[(t / TW * pitch + t % TW) % 32]);
        if (worst < best_worst) { best_worst = worst; best = static_cast<int32_t>(pitch); }
        if (worst == 1) break;
    }
    return best;
}

// Rows of the patch that a workgroup's tiles touch at most, in the row space Q = image * (2 TH + 2) + padded row of TH * TW = TI
// tiles per image: tiles t0 .. t1 take two rows per tile row and image border between them and four more.  Where a group
// starts within an image repeats after TI / gcd(TI, 64) groups, and a partial last group takes no more than a full one
// there (an eager call pays for this walk: 49 groups at 56 x 56 and 112 x 112, any batch).
inline int64_t MaxPatchRows(int64_t NT, int64_t TI, int64_t TW) {
    int64_t rem = TI, gcd = kTiles;
    while (rem != 0) { const int64_t r = gcd % rem; gcd = rem; rem = r; }
    const int64_t groups = std::min(CeilDiv(NT, kTiles), TI / gcd);
    const int64_t step_image = kTiles % TI, step_row = kTiles % TW;
    int64_t best = 0, in_image = 0, in_row = 0;
    for (int64_t g = 0; g < groups; ++g) {
        const int64_t last = std::min<int64_t>(kTiles, NT - g * kTiles) - 1;
        best = std::max(best, (in_row + last) / TW + (in_image + last) / TI);
        in_image += step_image;
        if (in_image >= TI) in_image -= TI;
        in_row += step_row;
        if (in_row >= TW) in_row -= TW;
    }
    return 2 * best + 4;
}

struct Args {
    const float* x;
    const char* u;
    const float* bias;
    const float* res;
    float* y;
    float* partial;
    const float* w;                    // RECHECK: OIHW weights
    int32_t N, C, H, W, O, OH, OW, ph, pw;
    int32_t TW, TI, NT, Hq, pitch;      // tiles per row, per image, in total; rows per image of the patch, row pitch of a (half) plane
    int32_t HW, OHW, ksteps;
    int32_t t_groups, k_groups, num_units, units_per_xcd, k_fastest;
    uint32_t x_bytes, u_bytes, flags;
    int32_t gsplit, steps_per_split;
    FastDiv div_ti, div_tw, div_kgroups, div_tgroups, div_gsplit, div_pitch, div_hq;
};

#if defined(__HIPCC__)

typedef __attribute__((address_space(3))) void* lds_void_t;

// ------------------------------------------------------------------------------------------
// Filter transform into the packed three-part form.  A workgroup takes 32 output channels x 16 input channels; thread
// (i, half, o) makes row i of U = G g G^T for eight channels and stores its four positions' fragments: the 32 lanes of a
// half-wave write 512 contiguous bytes.  PARTS: workgroups that share a tile's four columns of U.
// ------------------------------------------------------------------------------------------
template <int PARTS>
__device__ __forceinline__ void weight_tile(const float* __restrict__ w, char* __restrict__ u, int32_t O, int32_t C, int tile, int part,
                                            float* raw) {
    constexpr int RS = kStep * 9 + 1;
    const int ksteps = (C + kStep - 1) / kStep;
    const int ob = tile / ksteps, ks = tile - ob * ksteps;
    const int o0 = ob * 32, c0 = ks * kStep;
    const int cn = min(kStep, C - c0);
    const int tid = threadIdx.x;
    stage_filters<kStep>(w, O, C, o0, c0, cn, raw);
    __syncthreads();
    const int ol = tid & 31, half = (tid >> 5) & 1, i = tid >> 6;
    float v[4][8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const float* g = raw + ol * RS + (half * 8 + c) * 9;
        float t[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const float g0 = g[j], g1 = g[3 + j], g2 = g[6 + j];
            t[j] = i == 0 ? g0 : i == 1 ? 0.5f * ((g0 + g2) + g1) : i == 2 ? 0.5f * ((g0 + g2) - g1) : g2;
        }
        v[0][c] = t[0];
        v[1][c] = 0.5f * ((t[0] + t[2]) + t[1]);
        v[2][c] = 0.5f * ((t[0] + t[2]) - t[1]);
        v[3][c] = t[2];
    }
    char* const dst = u + (static_cast<int64_t>(tile) * 16 + i * 4) * 3072 + (half * 32 + ol) * 16;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (j / (4 / PARTS) != part) continue;
        const Split8 s = split8(v[j]);
        *reinterpret_cast<u32x4*>(dst + j * 3072) = s.h;
        *reinterpret_cast<u32x4*>(dst + j * 3072 + 1024) = s.m;
        *reinterpret_cast<u32x4*>(dst + j * 3072 + 2048) = s.l;
    }
}
inline int64_t WeightTiles(int64_t O, int64_t C) { return CeilDiv(O, 32) * CeilDiv(C, kStep); }

// RECHECK (the single operator): the transforms spread an Inf or NaN over the whole 2x2 tile, and so do sums beyond the
// largest float; a thread that finds such a tile evaluates its outputs by the loop of the operator's definition.
template <int kPlane, int LOADS, bool RECHECK>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) wino_bf16x3_kernel(const Args a) {
    constexpr int kHalf = kPlane / 2, kSegs = kPlane / 64;
    constexpr bool kIsWide = LOADS != kNarrow;
    constexpr int kPieces = kPlane / 256;                 // kWide: loads (64 pieces of 16 bytes) of a channel
    constexpr int NP = kIsWide ? 2 * kPieces : kSegs * kStep / 8;      // patch loads of a wave per step
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, half = lane >> 5, r = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wi = wave & 3, jp = wave >> 2;      // (waves w and w + 4 share a SIMD: one of each jp)
    // Consecutive workgroups go to the 8 XCDs round-robin; each XCD (own L2) takes a contiguous run of units.
    const int slot = (blockIdx.x & 7) * a.units_per_xcd + (blockIdx.x >> 3);
    if (slot >= a.num_units * a.gsplit || static_cast<int>(blockIdx.x >> 3) >= a.units_per_xcd) return;
    const int unit = a.gsplit > 1 ? fast_div(slot, a.div_gsplit) : slot;
    const int split = slot - unit * a.gsplit;
    int kg, tg;
    if (a.k_fastest) { tg = fast_div(unit, a.div_kgroups); kg = unit - tg * a.k_groups; }
    else { kg = fast_div(unit, a.div_tgroups); tg = unit - kg * a.t_groups; }
    const int t0 = tg * kTiles;
    const int s_lo = split * a.steps_per_split, s_hi = min(s_lo + a.steps_per_split, a.ksteps), s_last = s_hi - 1;
    const __amdgpu_buffer_rsrc_t ur = make_rsrc(a.u, a.u_bytes);

    // ---- geometry of the patch in padded row space
    int qmin, P;
    {
        const int tl = min(t0 + kTiles, a.NT) - 1;
        const int n0 = fast_div(t0, a.div_ti), n1 = fast_div(tl, a.div_ti);
        qmin = n0 * a.Hq + 2 * fast_div(t0 - n0 * a.TI, a.div_tw);
        const int qlast = n1 * a.Hq + 2 * fast_div(tl - n1 * a.TI, a.div_tw) + 3;
        P = (qlast - qmin + 1) * a.pitch;
    }
    // segments of 64 floats: wave w loads segment w of all 16 channels and, of a plane of 768, segment 8 + w % 4 of eight
    // (kWide: wave w loads channels 2 w and 2 w + 1, every lane pieces lane + 64 k)
    constexpr int kSecond = !kIsWide && NP > kStep ? 1 : 0;
    const int seg2 = 8 + (wave & 3), c2 = (wave >> 2) * 8;
    uint32_t goff[kIsWide ? kPieces : 1 + kSecond];
    if constexpr (kIsWide) {
#pragma unroll
        for (int k = 0; k < kPieces; ++k) {
            const int pos = (k * 64 + lane) * 4, q = fast_div(pos, a.div_pitch), iw = pos - q * a.pitch - 4;
            const int Q = qmin + q, n = fast_div(Q, a.div_hq), ih = Q - n * a.Hq - a.ph;
            const bool ok = pos < P && n < a.N && ih >= 0 && ih < a.H && iw >= 0 && iw < a.W;
            goff[k] = ok ? static_cast<uint32_t>((n * a.C * a.H + ih) * a.W + iw) * 4u : kOob;
        }
    } else {
#pragma unroll
        for (int k = 0; k < 1 + kSecond; ++k) {
            const int at = (k ? seg2 : wave) * 64 + lane, odd = at >= kHalf ? 1 : 0, pos = at - odd * kHalf;
            const int q = fast_div(pos, a.div_pitch), iw = 2 * (pos - q * a.pitch) + odd - a.pw;
            const int Q = qmin + q, n = fast_div(Q, a.div_hq), ih = Q - n * a.Hq - a.ph;
            const bool ok = pos < P && n < a.N && ih >= 0 && ih < a.H && iw >= 0 && iw < a.W;
            goff[k] = ok ? static_cast<uint32_t>((n * a.C * a.H + ih) * a.W + iw) * 4u : kOob;
        }
    }
    const uint32_t plane_bytes = static_cast<uint32_t>(a.HW) * 4u;
    // Always NP loads, so that every wait knows how many are younger: positions past the patch, and channels past the last
    // one or steps past the end (an empty descriptor), read as zero without touching memory.
    auto load_patch_one = [&](int s, float* buf, int e) __attribute__((always_inline)) {
        if constexpr (kIsWide) {
            // (the channel is part of the base, so that the range check ends the last piece of a row at the end of the tensor)
            const int cl = wave * 2 + e / kPieces, c = s * kStep + cl;
            const uint32_t skip = s < s_hi && c < a.C ? static_cast<uint32_t>(c) * plane_bytes : a.x_bytes;
            const __amdgpu_buffer_rsrc_t xr = make_rsrc(reinterpret_cast<const char*>(a.x) + skip, a.x_bytes - skip);
            load16_to_lds(xr, (lds_void_t)(buf + cl * kPlane + (e % kPieces) * 256), goff[e % kPieces], 0);
            return;
        }
        const bool second = e >= kStep;
        const int c = second ? c2 + e - kStep : e, seg = second ? seg2 : wave;
        const __amdgpu_buffer_rsrc_t xr = make_rsrc(a.x, s < s_hi && c < a.C - s * kStep ? a.x_bytes : 0u);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void_t)(buf + c * kPlane + seg * 64), 4, goff[second ? kSecond : 0],
                                                 static_cast<uint32_t>(s * kStep + c) * plane_bytes, 0, 0);
    };
    auto load_patch = [&](int s, float* buf) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < NP; ++e) load_patch_one(s, buf, e);
        __builtin_amdgcn_sched_barrier(0);
    };
    float* const buf0 = lds;
    float* const buf1 = lds + kStep * kPlane;
    float* const buf2 = lds + 2 * kStep * kPlane;
    load_patch(s_lo, buf0);

    // ---- U fragments: [o block][step][f][part] runs of 1 KiB
    u32x4 uf[2][2][3];      // [position][o block][part]
    auto load_u_one = [&](int s, int q, int e) __attribute__((always_inline)) {
        const int i = e / 3, p = e % 3;
        const uint32_t so = (static_cast<uint32_t>(kg * 2 + i) * static_cast<uint32_t>(a.ksteps) + static_cast<uint32_t>(s)) * 49152u +
                            static_cast<uint32_t>(wi * 4 + jp * 2 + q) * 3072u + static_cast<uint32_t>(p) * 1024u;
        // (the range check does not see the scalar offset: absent channel blocks are masked in the vector offset)
        const uint32_t vo = (kg * 2 + i) * 32 < a.O ? static_cast<uint32_t>(lane) * 16u : kOob;
        uf[q][i][p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ur, vo, so, 0));
    };
    auto load_u = [&](int s, int q) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 6; ++e) load_u_one(s, q, e);
        __builtin_amdgcn_sched_barrier(0);
    };
    load_u(s_lo, 0);
    load_patch(s_lo + 1, buf1);

    // ---- where this wave's operands come from: rows (ra, rb) of the 4x4 patch combine to t = ra + sr * rb,
    //   i = 0: d0 - d2, 1: d1 + d2, 2: d2 - d1, 3: d1 - d3,   and columns to t0 - t2, t1 + t2 (jp = 0) or t2 - t1, t1 - t3 (jp = 1)
    const int rowa = wi == 0 ? 0 : wi == 2 ? 2 : 1, rowb = wi == 0 ? 2 : wi == 1 ? 2 : wi == 2 ? 1 : 3;
    const float sr = wi == 1 ? 1.0f : -1.0f;
    bool in2[2], in3[2];                           // kWideEdge: the patch's third and fourth column lie in the image
    int base[2];                                   // (the second row's base is one addition away: registers are what is short here)
    const int drow = (rowb - rowa) * a.pitch;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int tile = min(t0 + j * 32 + r, a.NT - 1);
        const int n = fast_div(tile, a.div_ti), rem = tile - n * a.TI;
        const int ty = fast_div(rem, a.div_tw), tx = rem - ty * a.TW;
        base[j] = (n * a.Hq + 2 * ty + rowa - qmin) * a.pitch + (kIsWide ? 2 * tx + 3 : tx) + half * 8 * kPlane;
        if constexpr (LOADS == kWideEdge) { in2[j] = 2 * tx + 1 < a.W; in3[j] = 2 * tx + 2 < a.W; }
    }

    f32x16 acc[2][2][2];      // [position][o block][tile block]
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int g = 0; g < 16; ++g) acc[q][i][j][g] = 0.0f;

    u32x4 vf[2][3];           // V fragments of one tile block [position][part]
    // `between(k)` runs behind the k-th of four pieces / twelve matrix instructions: loads are issued one at a time there,
    // because a wave that issues several in a row waits for the address unit with everything that follows them
    auto nothing = [](int) {};
    auto transform = [&](auto jp_c, const float* buf, int j, auto between) __attribute__((always_inline)) {
        constexpr int JP = decltype(jp_c)::value;
        const float* const pa = buf + base[j];
        const float* const pb = pa + drow;
        // columns (u, w) give V of the wave's first position as t_u - t_w, (x, w) of its second
        constexpr int U = JP == 0 ? 0 : 1, X = JP == 0 ? kHalf : kHalf + 1, W_ = JP == 0 ? 1 : kHalf;
        // two channels at a time, read one pair ahead of their arithmetic
        float d[2][2][6];
        auto read = [&](int k) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int o = (2 * k + c) * kPlane;
                if constexpr (kIsWide) {
                    // columns 1 and 2 of the patch are 8 aligned bytes (the row's columns 2 tx and 2 tx + 1)
                    const f32x2 ma = *reinterpret_cast<const f32x2*>(pa + o + 1), mb = *reinterpret_cast<const f32x2*>(pb + o + 1);
                    constexpr int SIDE = JP == 0 ? 0 : 3;
                    d[k & 1][c][JP == 0 ? 0 : 1] = pa[o + SIDE]; d[k & 1][c][JP == 0 ? 1 : 2] = ma[0]; d[k & 1][c][JP == 0 ? 2 : 0] = ma[1];
                    d[k & 1][c][JP == 0 ? 3 : 4] = pb[o + SIDE]; d[k & 1][c][JP == 0 ? 4 : 5] = mb[0]; d[k & 1][c][JP == 0 ? 5 : 3] = mb[1];
                    continue;
                }
                d[k & 1][c][0] = pa[o + U]; d[k & 1][c][1] = pa[o + X]; d[k & 1][c][2] = pa[o + W_];
                d[k & 1][c][3] = pb[o + U]; d[k & 1][c][4] = pb[o + X]; d[k & 1][c][5] = pb[o + W_];
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto make = [&](int k) __attribute__((always_inline)) {
            float v0[2], v1[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const float* const e = d[k & 1][c];
                float tu = __builtin_fmaf(sr, e[3], e[0]), tx = __builtin_fmaf(sr, e[4], e[1]), tw = __builtin_fmaf(sr, e[5], e[2]);
                if constexpr (LOADS == kWideEdge) {
                    if (JP == 0) {
                        tw = in2[j] ? tw : 0.0f;
                    } else {
                        tu = in2[j] ? tu : 0.0f;
                        tx = in3[j] ? tx : 0.0f;
                    }
                }
                v0[c] = __fsub_rn(tu, tw);
                v1[c] = JP == 0 ? __fadd_rn(tx, tw) : __fsub_rn(tw, tx);
            }
            uint32_t h, m, l;
            split_pair(v0[0], v0[1], h, m, l);
            vf[0][0][k] = h; vf[0][1][k] = m; vf[0][2][k] = l;
            split_pair(v1[0], v1[1], h, m, l);
            vf[1][0][k] = h; vf[1][1][k] = m; vf[1][2][k] = l;
            __builtin_amdgcn_sched_barrier(0);
        };
        auto pause = [&](int k) __attribute__((always_inline)) { between(k); __builtin_amdgcn_sched_barrier(0); };
        read(0);
        read(1);
        make(0);
        pause(0);
        read(2);
        make(1);
        pause(1);
        read(3);
        make(2);
        pause(2);
        make(3);
        pause(3);
    };
    auto multiply = [&](int q, int j, auto between) __attribute__((always_inline)) {
        constexpr int PA[6] = {1, 0, 2, 0, 1, 0}, PB[6] = {1, 2, 0, 1, 0, 0};
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int e = 0; e < 12; ++e) {
            const int p = e >> 1, i = e & 1;
            acc[q][i][j] = mfma_bf16(uf[q][i][PA[p]], vf[q][PB[p]], acc[q][i][j]);
            between(e);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
    };
    // A wave's vector instructions do not run beside its own matrix instructions, only beside the other wave's of its
    // SIMD, so the two work in opposite phases: between two barriers, while the patch of step s is in LDS, the waves with
    // jp = 0 run T0 M0 T1 M1 of step s (T: transform a tile block, M: multiply it) and those with jp = 1 run M1 of step
    // s - 1 and then T0 M0 T1 of step s.  The filter fragments of the next step are requested as soon as their last use is
    // issued.  Loads complete in order: the patch of step s + 2 is requested where a wait for fragments does not wait for it
    // before it had a whole step to arrive, and the barrier at the end of step s waits for that of s + 1 only.
    float *cur = buf0, *nxt = buf1, *far = buf2;
    auto rotate = [&]() __attribute__((always_inline)) { float* const t = cur; cur = nxt; nxt = far; far = t; };
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(6 + NP) : "memory");      // the first patch
    auto first_u = [&](int s, int q) { return [&, s, q](int e) __attribute__((always_inline)) { if (e & 1) load_u_one(s, q, e >> 1); }; };
    auto patch_part = [&](int s, float* buf, int part) {
        return [&, s, buf, part](int e) __attribute__((always_inline)) { if (part * 12 + e < NP) load_patch_one(s, buf, part * 12 + e); };
    };
    auto second_u = [&](int s) {
        return [&, s](int k) __attribute__((always_inline)) {
            load_u_one(s, 1, k);
            if (k < 2) load_u_one(s, 1, 4 + k);
        };
    };
    if (jp == 0) {
        using JP = std::integral_constant<int, 0>;
        for (int s = s_lo; s < s_hi; ++s) {
            transform(JP{}, cur, 0, second_u(s));
            multiply(0, 0, patch_part(s + 2, far, 0));
            multiply(1, 0, patch_part(s + 2, far, 1));
            transform(JP{}, cur, 1, nothing);
            multiply(0, 1, nothing);
            multiply(1, 1, first_u(min(s + 1, s_last), 0));
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(6 + NP) : "memory");
            rotate();
        }
    } else {
        using JP = std::integral_constant<int, 1>;
        for (int s = s_lo; s < s_hi; ++s) {
            if (s > s_lo) {
                multiply(0, 1, nothing);
                multiply(1, 1, first_u(s, 0));
            }
            transform(JP{}, cur, 0, second_u(s));
            multiply(0, 0, patch_part(s + 2, far, 0));
            multiply(1, 0, patch_part(s + 2, far, 1));
            transform(JP{}, cur, 1, nothing);
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NP) : "memory");
            rotate();
        }
        multiply(0, 1, nothing);
        multiply(1, 1, nothing);
    }
    // (patches of steps past the end may still be on their way into LDS)
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");

    // ---- output transform and epilogue, 32 output channels x 32 tiles at a time.  ex[jp][i][p][o][tile]: p0 / p1 = the
    // wave's share of output column 0 / 1 of row i.  Two areas, so that one barrier per block is enough.
    const bool raw_part = a.gsplit > 1;
    const bool has_bias = !raw_part && (a.flags & KXC_HIP_CONV_BIAS) != 0;
    const bool has_res = !raw_part && (a.flags & KXC_HIP_CONV_RESIDUAL) != 0;
    const bool do_relu = !raw_part && (a.flags & KXC_HIP_CONV_RELU) != 0;
    const uint32_t y_bytes = static_cast<uint32_t>(a.N) * static_cast<uint32_t>(a.O) * static_cast<uint32_t>(a.OHW) * 4u;
    float* const yp = raw_part ? a.partial + static_cast<int64_t>(split) * (y_bytes / 4u) : a.y;
    const __amdgpu_buffer_rsrc_t yr = make_rsrc(yp, y_bytes);
    const __amdgpu_buffer_rsrc_t rr = make_rsrc(has_res ? a.res : yp, has_res ? y_bytes : 0u);
    const __amdgpu_buffer_rsrc_t br = make_rsrc(has_bias ? a.bias : yp, has_bias ? static_cast<uint32_t>(a.O) * 4u : 0u);
    const bool even = (a.OW & 1) == 0, wide = (a.TW & 1) == 0 && (a.OW & 3) == 0;      // wide: a pair of tiles is 16 aligned bytes of one row
    const int tp = tid & 15, ol = tid >> 4;                   // this thread finishes tiles 2 tp, 2 tp + 1 of channel ol of a block
    const uint32_t rowb_bytes = static_cast<uint32_t>(a.OW) * 4u, o_bytes = static_cast<uint32_t>(a.OHW) * 4u;
    constexpr int kArea = 8 * 2 * 1024;
    auto bits = [](float v) { return __builtin_bit_cast(uint32_t, v); };
    uint32_t again = 0;               // RECHECK: bit 2 j + i = this thread's outputs of the block
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        uint32_t off[2][2], cm[2];      // [tile][row] byte offset within channel 0 of a block; mask of the second column
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int tile = t0 + j * 32 + 2 * tp + e;
            const int tc = min(tile, a.NT - 1);
            const int n = fast_div(tc, a.div_ti), rem = tc - n * a.TI;
            const int ty = fast_div(rem, a.div_tw), tx = rem - ty * a.TW;
            const uint32_t at = static_cast<uint32_t>(((n * a.O + ol) * a.OH + 2 * ty) * a.OW + 2 * tx) * 4u;
            off[e][0] = tile < a.NT ? at : kOob;
            off[e][1] = tile < a.NT && 2 * ty + 1 < a.OH ? at + rowb_bytes : kOob;
            cm[e] = 2 * tx + 1 < a.OW ? 0u : kOob;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float* const ex = lds + i * kArea;
            float* const w0 = ex + wave * 2048 + 4 * half * 32 + r;
            if (jp == 0) {
#pragma unroll
                for (int g = 0; g < 16; ++g) {
                    w0[(8 * (g / 4) + g % 4) * 32] = __fadd_rn(acc[0][i][j][g], acc[1][i][j][g]);
                    w0[1024 + (8 * (g / 4) + g % 4) * 32] = acc[1][i][j][g];
                }
            } else {
#pragma unroll
                for (int g = 0; g < 16; ++g) {
                    w0[(8 * (g / 4) + g % 4) * 32] = acc[0][i][j][g];
                    w0[1024 + (8 * (g / 4) + g % 4) * 32] = -__fadd_rn(acc[0][i][j][g], acc[1][i][j][g]);
                }
            }
            const int ob = kg * kOut + i * 32;                                   // uniform: the block's first channel
            uint32_t om = ob + ol < a.O ? 0u : kOob;
            const uint32_t so = ob < a.O ? static_cast<uint32_t>(ob) * o_bytes : 0u;      // (the mask decides about absent channels)
            const float bv = load_f32(br, (static_cast<uint32_t>(ob + ol) * 4u) | om, 0);
            auto ld = [&](uint32_t o) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rr, o, so, 0)); };
            float q[2][2][2];               // residual [tile][row][column]
            if (has_res) {
                if (wide) {
#pragma unroll
                    for (int row = 0; row < 2; ++row) {
                        const f32x4 v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rr, off[0][row] | om, so, 0));
                        q[0][row][0] = v[0]; q[0][row][1] = v[1]; q[1][row][0] = v[2]; q[1][row][1] = v[3];
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int row = 0; row < 2; ++row) {
                            q[e][row][0] = ld(off[e][row] | om);
                            q[e][row][1] = ld((off[e][row] + 4u) | cm[e] | om);
                        }
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            float out[2][2][2];             // [tile][row][column]
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                f32x2 row[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const f32x2 e0 = *reinterpret_cast<const f32x2*>(ex + k * 2048 + p * 1024 + ol * 32 + 2 * tp);
                    const f32x2 e1 = *reinterpret_cast<const f32x2*>(ex + (k + 4) * 2048 + p * 1024 + ol * 32 + 2 * tp);
                    row[k][0] = __fadd_rn(e0[0], e1[0]); row[k][1] = __fadd_rn(e0[1], e1[1]);
                }
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    out[e][0][p] = __fadd_rn(__fadd_rn(row[0][e], row[1][e]), row[2][e]);
                    out[e][1][p] = __fsub_rn(__fsub_rn(row[1][e], row[2][e]), row[3][e]);
                }
            }
            if constexpr (RECHECK) {
                float odd = 0.0f;
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int row = 0; row < 2; ++row) odd = __builtin_fmaf(out[e][row][0], 0.0f, __builtin_fmaf(out[e][row][1], 0.0f, odd));
                if (!(odd == 0.0f) && om == 0) {
                    again |= 1u << (2 * j + i);
                    om = kOob;                  // (nothing is stored now: the residual may be the output's own buffer)
                }
            }
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int row = 0; row < 2; ++row)
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        float v = out[e][row][p];
                        if (has_bias) v = __fadd_rn(v, bv);
                        if (has_res) v = __fadd_rn(v, q[e][row][p]);
                        if (do_relu) v = relu_sel(v);
                        out[e][row][p] = v;
                    }
            if (wide) {
                // (no scalar offset on a 16-byte store: with one, the compiler lets the next vector instruction overwrite the
                // first data register, which on gfx950 the store has not read yet)
#pragma unroll
                for (int row = 0; row < 2; ++row)
                    __builtin_amdgcn_raw_buffer_store_b128(u32x4{bits(out[0][row][0]), bits(out[0][row][1]), bits(out[1][row][0]), bits(out[1][row][1])},
                                                           yr, (off[0][row] | om) == off[0][row] && off[0][row] != kOob ? off[0][row] + so : kOob, 0, 0);
            } else if (even) {
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int row = 0; row < 2; ++row)
                        __builtin_amdgcn_raw_buffer_store_b64(u32x2{bits(out[e][row][0]), bits(out[e][row][1])}, yr, off[e][row] | om, so, 0);
            } else {
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int row = 0; row < 2; ++row) {
                        __builtin_amdgcn_raw_buffer_store_b32(bits(out[e][row][0]), yr, off[e][row] | om, so, 0);
                        __builtin_amdgcn_raw_buffer_store_b32(bits(out[e][row][1]), yr, (off[e][row] + 4u) | cm[e] | om, so, 0);
                    }
            }
        }
    }
    if constexpr (RECHECK) {
        if (again == 0) return;
#pragma unroll 1
        for (int k = 0; k < 32; ++k) {
            const int block = k >> 3, e = (k >> 2) & 1, row = (k >> 1) & 1, p = k & 1;
            const int tile = t0 + (block >> 1) * 32 + 2 * tp + e, o = kg * kOut + (block & 1) * 32 + ol;
            if (!((again >> block) & 1u) || tile >= a.NT) continue;
            const int n = fast_div(tile, a.div_ti), rem = tile - n * a.TI;
            const int ty = fast_div(rem, a.div_tw), oh = 2 * ty + row, ow = 2 * (rem - ty * a.TW) + p;
            if (oh >= a.OH || ow >= a.OW) continue;
            float s = 0.0f;
#pragma unroll 1
            for (int c = 0; c < a.C; ++c) {
                const float* const xc = a.x + static_cast<int64_t>(n * a.C + c) * a.HW;
                const float* const wc = a.w + (static_cast<int64_t>(o) * a.C + c) * 9;
#pragma unroll 1
                for (int q = 0; q < 9; ++q) {
                    const int ih = oh + q / 3 - a.ph, iw = ow + q % 3 - a.pw;
                    const bool in = ih >= 0 && ih < a.H && iw >= 0 && iw < a.W;
                    s = __fadd_rn(s, __fmul_rn(in ? xc[ih * a.W + iw] : 0.0f, wc[q]));
                }
            }
            const int64_t at = (static_cast<int64_t>(n * a.O + o) * a.OH + oh) * a.OW + ow;
            if (has_bias) s = __fadd_rn(s, a.bias[o]);
            if (has_res) s = __fadd_rn(s, a.res[at]);
            a.y[at] = do_relu ? relu_sel(s) : s;
        }
    }
}

#endif  // __HIPCC__

}  // namespace wino_bx
}  // namespace kxc_hip
