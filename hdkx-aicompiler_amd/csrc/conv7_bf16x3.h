// conv7_bf16x3.h -- the 7x7 stride-2 convolution of three-channel images (a network's first layer) on the bf16 matrix cores
// with three-part operands (bf16x3.h); included by conv2d_bf16x3.hip (selection, launch) and conv2d_wino_f32.hip (the filters
// of a plan are packed by one launch).
//
// D[o][pixel] += W[o][c, rh, rw] X[c, rh, rw][pixel]: 147 products, taken as 21 rows (c, rh) of seven columns and a zero, two rows to a
// matrix instruction, 11 steps of 16 (176).  A wave owns 32 output channels x up to seven blocks of 32 pixels; a workgroup is two waves, 64
// channels, or, where the result is not pooled, two such pairs that share the tile.
//  * The whole reduction's input fits LDS (nine rows of a 224-wide image: 38 KiB): loaded, split into its three parts and stored
//    once, [channel][row][part][column].  The eight columns of a pixel's window are four words there, one word behind its left
//    neighbour's: two ds_read2_b32, whose reach (255 words) holds the three parts of a row.
//  * A tile is 224 pixels or, where those reach over too many rows for four workgroups on a compute unit, whole rows of one image: two of 97 pixels, say.
//  * One accumulator per block takes the small products of the whole reduction first and the large ones behind them (the h parts
//    are read twice for that): 11 roundings at the sum's full size.  Relative error against float64 0.6e-7, 1.8e-7 on the fp32 instructions.
//  * Nothing inside a workgroup overlaps its loads, its products and its stores; the others on a compute unit do.  An instruction is
//    four cycles of a wave, so what is around the 18 thousand cycles of products is kept short: a row's place in memory is formed once, by the lane
//    of its number (27 chains of scalar divisions before: 9.5 thousand cycles for the patch, 4.7 now), and a value of the result takes four
//    instructions (13.8 thousand cycles for a wave's 112, 3.1 now).
//
// Measured, 3 -> 64 channels at 224 x 224 with the pooling epilogue, 64 images, alone: 107 us (120 with the longer ends, 169 on the fp32 instructions;
// batch 32 57 and 64, batch 2 15 and 18); not pooled, 193 x 193, batch 16 30 (45 on the fp32 instructions), 189 x 189, batch 47 57 (107), 216 x 216, batch 36
// 60 (2312).  Two pairs to a tile against one of five to seven blocks a wave, with the filter's packing: batch 6 at 193 x 193 22 and 28, batch
// 47 at 189 x 189 61 and 66, batch 58 at 150 x 150 57 and 57.  62 us is what the first's products take at the rate of a loop of nothing else, 30 the bytes.  The
// address unit takes 16 cycles per load or store.  Both blocks of channels on four or three blocks of pixels per wave, with half as many LDS
// reads: 118 against 115.
#pragma once

#include "bf16x3.h"
#include "common.h"

namespace kxc_hip {
namespace conv7_bx {

constexpr int kK = 7, kC = 3, kOut = 64, kPix = 224, kThreads = 128;
// A step of 16 products is two groups (channel, filter row) of seven columns and a zero: group 2 s and, for the upper lanes, 2 s + 1.
constexpr int kGroups = kC * kK, kSteps = (kGroups + 1) / 2;

inline size_t FilterBytes(int64_t O) { return static_cast<size_t>(CeilDiv(O, 32)) * kSteps * 3 * 1024; }
// LDS: [channel][row][part][kPitch words], a word = two neighbouring columns of the padded row.
inline size_t LdsBytes(int64_t rows, int pitch) { return static_cast<size_t>(kC) * rows * 3 * pitch * 4; }
// What the epilogues and the sums that are not finite need of it, of each wave.  (Half-waves four channels apart write to different banks.)
constexpr int kTurnPitch = 40;
constexpr size_t kMinLdsBytes = 2 * 2 * 32 * kTurnPitch * 4;

struct Args {
    const float* x;
    const char* u;
    const float* bias;
    const float* res;
    float* y;
    const float* w;                     // the filter as it was given, for sums that are not finite
    int32_t N, H, W, O, OH, OW, M, OHW, HW, ph, pw, Hp, PW;
    int32_t tile_pix, span, tiles;      // pixels of a tile, of a run of tiles (all, or an image where tiles are whole rows), tiles of a run
    int32_t row_max;                    // rows of the patch in LDS
    int32_t o_tiles, num_units, units_per_xcd;
    uint32_t x_bytes, y_bytes, u_bytes, flags;
    FastDiv div_ohw, div_ow, div_hp, div_otiles, div_tiles;
};

#if defined(__HIPCC__)

constexpr uint32_t kOob = 0x80000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), 0x00020000);
}
__device__ __forceinline__ float relu_sel(float v) { return (v > 0.0f) ? v : 0.0f; }
__device__ __forceinline__ float load_f32(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

// HP: the result leaves the kernel max-pooled along W (KXC_HIP_CONV_HPOOL; window 3, stride 2, one column of padding on the left);
// the host guarantees ReLU, no residual, O % 8 == 0, an even OW that divides kPix, and full tiles.
// PARTS: pairs of waves that share the tile's pixels.
template <int kPitch, bool HP, int kBlocks, int PARTS>
__global__ void __launch_bounds__(PARTS * kThreads) __attribute__((amdgpu_waves_per_eu(PARTS + 1))) conv7_bf16x3_kernel(const Args a) {
    request_args(a);
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, half = lane >> 5, r = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int unit = (blockIdx.x & 7) * a.units_per_xcd + (blockIdx.x >> 3);
    if (unit >= a.num_units || static_cast<int>(blockIdx.x >> 3) >= a.units_per_xcd) return;
    const int p_tile = fast_div(unit, a.div_otiles), o_tile = unit - p_tile * a.o_tiles;
    const int run = fast_div(p_tile, a.div_tiles), m0 = run * a.span + (p_tile - run * a.tiles) * a.tile_pix;
    const int m_end = min(m0 + a.tile_pix, (run + 1) * a.span);
    const int part = wave >> 1, oblk = o_tile * 2 + (wave & 1), o0 = oblk * 32, mw = m0 + part * kBlocks * 32;

    int qmin, rows;
    {
        const int n0 = fast_div(m0, a.div_ohw);
        qmin = n0 * a.Hp + 2 * fast_div(m0 - n0 * a.OHW, a.div_ow);
        const int ml = m_end - 1, n1 = fast_div(ml, a.div_ohw);
        rows = n1 * a.Hp + 2 * fast_div(ml - n1 * a.OHW, a.div_ow) + kK - qmin;
    }
    // ---- filter fragments
    const __amdgpu_buffer_rsrc_t ur = rsrc(a.u, a.u_bytes);
    const uint32_t avo = o0 < a.O ? static_cast<uint32_t>(lane) * 16u : kOob;
    const uint32_t a_base = o0 < a.O ? static_cast<uint32_t>(oblk) * (kSteps * 3072u) : 0u;
    u32x4 ua[2][3];
    auto load_a = [&](int b, int s, int p) __attribute__((always_inline)) {
        ua[b][p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ur, avo, a_base + static_cast<uint32_t>(s * 3 + p) * 1024u, 0));
    };
#pragma unroll
    for (int p = 0; p < 3; ++p) load_a(0, 0, p);

    // ---- the patch: a thread owns one word of a row; what lies outside the image reads as zero.  The rows of a tile two maps' rows high
    // are in flight together.  Lane k forms the place of row k once (rows times channels times scalar divisions were half of the phase).
    {
        constexpr bool kNarrow = kPitch <= 64;
        constexpr int kPar = kNarrow ? 2 * PARTS : PARTS, kBatch = PARTS == 1 ? 9 : 5;      // rows side by side; rows of a batch
        const int d = kNarrow ? lane : tid & (kThreads - 1), iw = 2 * d - a.pw, at = min(max(iw, 0), a.W - 2);
        const uint32_t vo = static_cast<uint32_t>(at) * 4u, plane = static_cast<uint32_t>(a.HW) * 4u;
        const bool in0 = iw >= 0 && iw < a.W, in1 = iw >= -1 && iw + 1 < a.W, high0 = iw != at, high1 = iw == at;
        const __amdgpu_buffer_rsrc_t xr = rsrc(a.x, a.x_bytes);
        uint32_t row_at;
        {
            const int Q = qmin + lane, n = fast_div(Q, a.div_hp), ih = Q - n * a.Hp - a.ph;
            row_at = lane < rows && n < a.N && ih >= 0 && ih < a.H ? static_cast<uint32_t>((n * kC * a.H + ih) * a.W) * 4u : kOob;
        }
#pragma unroll 1
        for (int r0 = kNarrow ? wave : part; r0 < rows; r0 += kBatch * kPar) {
            u32x2 v[kBatch][kC];
#pragma unroll
            for (int k = 0; k < kBatch; ++k) {
                const uint32_t o = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(row_at), min(r0 + k * kPar, 63))) + vo;
#pragma unroll
                for (int c = 0; c < kC; ++c) v[k][c] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(xr, o, static_cast<uint32_t>(c) * plane, 0));
            }
            __builtin_amdgcn_sched_barrier(0);
            if (d < kPitch) {
                uint32_t* dst = lds + r0 * 3 * kPitch + d;
#pragma unroll
                for (int k = 0; k < kBatch; ++k, dst += kPar * 3 * kPitch) {
                    if (r0 + k * kPar >= rows) continue;
#pragma unroll
                    for (int c = 0; c < kC; ++c) {
                        const f32x2 x = __builtin_bit_cast(f32x2, v[k][c]);
                        const float x0 = x.x, x1 = x.y;
                        uint32_t h, m, l;
                        split_pair(__fmul_rn(in0 ? (high0 ? x1 : x0) : 0.0f, kOperandScale), __fmul_rn(in1 ? (high1 ? x1 : x0) : 0.0f, kOperandScale), h, m, l);
                        uint32_t* const to = dst + c * a.row_max * 3 * kPitch;
                        to[0] = h;
                        to[kPitch] = m;
                        to[2 * kPitch] = l;
                    }
                }
            }
        }
    }
    int base[kBlocks];
#pragma unroll
    for (int j = 0; j < kBlocks; ++j) {
        const int m = min(mw + j * 32 + r, m_end - 1);
        const int n = fast_div(m, a.div_ohw), rem = m - n * a.OHW, oh = fast_div(rem, a.div_ow);
        base[j] = (n * a.Hp + 2 * oh - qmin) * 3 * kPitch + rem - oh * a.OW;
    }
    f32x16 acc[kBlocks];
#pragma unroll
    for (int j = 0; j < kBlocks; ++j)
#pragma unroll
        for (int g = 0; g < 16; ++g) acc[j][g] = 0.0f;
    __syncthreads();

    // ---- the small products of the whole reduction first, then the large ones: 11 roundings at the sum's full size
    const int row_words = 3 * kPitch, ch_words = a.row_max * row_words;
    auto group_at = [&](int g) { return g / kK * ch_words + g % kK * row_words; };
    auto step_at = [&](int s) {
        const int lo = group_at(2 * s), hi = group_at(2 * s + 1 < kGroups ? 2 * s + 1 : 2 * s);      // (the last group's filter is zero)
        return half ? hi : lo;
    };
    auto read_b = [&](u32x4& f, int at) __attribute__((always_inline)) { f = u32x4{lds[at], lds[at + 1], lds[at + 2], lds[at + 3]}; };
    {
        u32x4 vb[2][3];
        int at = step_at(0);
#pragma unroll
        for (int p = 2; p >= 0; --p) read_b(vb[0][p], base[0] + at + p * kPitch);
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            const int b = s & 1, next = step_at(s + 1 < kSteps ? s + 1 : s);
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) {
                constexpr int odd = kBlocks & 1;
                const int vbi = (s * odd + j) & 1, word = j + 1 < kBlocks ? base[j + 1] + at : base[0] + next;
                if (j < 3 && s + 1 < kSteps) load_a(b ^ 1, s + 1, 2 - j);
#pragma unroll
                for (int p = 2; p >= 0; --p) read_b(vb[vbi ^ 1][p], word + p * kPitch);
                __builtin_amdgcn_sched_barrier(0);
                acc[j] = mfma_bf16(ua[b][0], vb[vbi][2], acc[j]);
                acc[j] = mfma_bf16(ua[b][1], vb[vbi][1], acc[j]);
                acc[j] = mfma_bf16(ua[b][0], vb[vbi][1], acc[j]);
                acc[j] = mfma_bf16(ua[b][2], vb[vbi][0], acc[j]);
                acc[j] = mfma_bf16(ua[b][1], vb[vbi][0], acc[j]);
                __builtin_amdgcn_sched_barrier(0);
            }
            at = next;
        }
    }
    const bool has_bias = (a.flags & KXC_HIP_CONV_BIAS) != 0;
    const __amdgpu_buffer_rsrc_t br = rsrc(has_bias ? a.bias : a.y, has_bias ? static_cast<uint32_t>(a.O) * 4u : 0u);
    float bv[16];
#pragma unroll
    for (int g = 0; g < 16; ++g) {
        const int o = o0 + 8 * (g / 4) + 4 * half + g % 4;
        bv[g] = load_f32(br, o < a.O ? static_cast<uint32_t>(o) * 4u : kOob);
    }
    {
        u32x4 vb[2];
        int at = step_at(0);
        load_a(0, 0, 0);
        read_b(vb[0], base[0] + at);
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            const int b = s & 1, next = step_at(s + 1 < kSteps ? s + 1 : s);
            if (s + 1 < kSteps) load_a(b ^ 1, s + 1, 0);
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) {
                const int vbi = (s * (kBlocks & 1) + j) & 1;
                read_b(vb[vbi ^ 1], j + 1 < kBlocks ? base[j + 1] + at : base[0] + next);
                __builtin_amdgcn_sched_barrier(0);
                acc[j] = mfma_bf16(ua[b][0], vb[vbi], acc[j]);
            }
            at = next;
        }
    }
    __syncthreads();          // (the patch is dead)

    // ---- Splitting turns an infinite operand into NaN, and so does it to one of 2^112 and more, and sums (times 2^32 here) overflow
    // from 2^96 on: a sum that is not finite is formed again by the operator's definition.
    float* const area = reinterpret_cast<float*>(lds) + wave * (HP ? 2 * 32 * kTurnPitch : 16 * 64);
    float scale[kBlocks];                  // what is left to do to a block's sums
#pragma unroll
    for (int j = 0; j < kBlocks; ++j) {
        float odd = 0.0f;
        scale[j] = kSumScale;
#pragma unroll
        for (int g = 0; g < 16; ++g) odd = __builtin_fmaf(acc[j][g], 0.0f, odd);
        if (__builtin_amdgcn_ballot_w64(!(odd == 0.0f)) == 0) continue;
        scale[j] = 1.0f;
#pragma unroll
        for (int g = 0; g < 16; ++g) area[g * 64 + lane] = __fmul_rn(acc[j][g], kSumScale);
        const int m = mw + j * 32 + r, n = fast_div(m, a.div_ohw), rem = m - n * a.OHW, oh = fast_div(rem, a.div_ow), ow = rem - oh * a.OW;
#pragma unroll 1
        for (int g = 0; g < 16; ++g) {
            const int o = o0 + 8 * (g / 4) + 4 * half + g % 4;
            if (__builtin_fabsf(area[g * 64 + lane]) < __builtin_inff() || m >= m_end || o >= a.O) continue;
            float s = 0.0f;
#pragma unroll 1
            for (int q = 0; q < kC * kK * kK; ++q) {
                const int c = q / (kK * kK), t = q - c * kK * kK, ih = 2 * oh + t / kK - a.ph, iw = 2 * ow + t % kK - a.pw;
                const bool in = ih >= 0 && ih < a.H && iw >= 0 && iw < a.W;
                s = __fadd_rn(s, __fmul_rn(in ? a.x[static_cast<int64_t>(n * kC + c) * a.HW + ih * a.W + iw] : 0.0f, a.w[o * kC * kK * kK + q]));
            }
            area[g * 64 + lane] = s;
        }
#pragma unroll
        for (int g = 0; g < 16; ++g) acc[j][g] = area[g * 64 + lane];
    }

    // ---- epilogue: register g of a block = channel 8 (g / 4) + 4 half + g % 4, lane r = pixel
    const __amdgpu_buffer_rsrc_t yr = rsrc(a.y, a.y_bytes);
    if (!has_bias) {
#pragma unroll
        for (int g = 0; g < 16; ++g) bv[g] = -0.0f;        // (x + -0 = x)
    }
    auto sum = [&](int j, int g) __attribute__((always_inline)) { return __builtin_fmaf(acc[j][g], scale[j], bv[g]); };
    if constexpr (HP) {
        // Turned through LDS, one block of 32 columns behind the other in two places: a lane owns the window of columns 2 p and 2 p + 1,
        // p = lane % 16, and the one to their left, in channels 4 i + lane / 16; a row's first column is its own left neighbour.  The
        // values are ReLU results (>= +0, never NaN), so no order matters.
        const uint32_t plane = static_cast<uint32_t>(a.OH * a.PW) * 4u;
        const int p = lane & 15, ch = lane >> 4;
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) {
            float* const to = area + (j & 1) * 32 * kTurnPitch;
            const float* const other = area + (~j & 1) * 32 * kTurnPitch;
#pragma unroll
            for (int g = 0; g < 16; ++g) to[(8 * (g / 4) + 4 * half + g % 4) * kTurnPitch + r] = __builtin_fmaxf(sum(j, g), 0.0f);
            const int m = mw + j * 32 + 2 * p, n = fast_div(m, a.div_ohw), rem = m - n * a.OHW, oh = fast_div(rem, a.div_ow), ow = rem - oh * a.OW;
            const uint32_t yb = static_cast<uint32_t>((n * a.O * a.OH + oh) * a.PW + (ow >> 1)) * 4u + static_cast<uint32_t>(ch) * plane;
            const float* const own = to + ch * kTurnPitch + 2 * p;
            const float* const left = ow == 0 ? own : p == 0 ? other + ch * kTurnPitch + 31 : own - 1;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const f32x2 v = *reinterpret_cast<const f32x2*>(own + 4 * i * kTurnPitch);
                const float pooled = fmaxf(fmaxf(left[4 * i * kTurnPitch], v.x), v.y);
                const int c = o0 + 4 * i;                          // uniform; its channels are c .. c + 3 (O % 8 == 0)
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, pooled), yr, c < a.O ? yb : kOob, c < a.O ? static_cast<uint32_t>(c) * plane : 0u, 0);
            }
        }
        return;
    }
    const bool has_res = (a.flags & KXC_HIP_CONV_RESIDUAL) != 0, do_relu = (a.flags & KXC_HIP_CONV_RELU) != 0;
    const __amdgpu_buffer_rsrc_t rr = rsrc(has_res ? a.res : a.y, has_res ? a.y_bytes : 0u);
    const uint32_t plane = static_cast<uint32_t>(a.OHW) * 4u;
    if (!has_res && do_relu && o0 + 32 <= a.O) {          // (what a network's first layer is: four instructions a value)
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) {
            const int m = mw + j * 32 + r, n = fast_div(min(m, m_end - 1), a.div_ohw), rem = m - n * a.OHW;
            const uint32_t yb = m < m_end ? static_cast<uint32_t>(n * a.O * a.OHW + rem) * 4u + static_cast<uint32_t>(4 * half) * plane : kOob;
#pragma unroll
            for (int g = 0; g < 16; ++g)
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, __builtin_fmaxf(sum(j, g), 0.0f)), yr, yb,
                                                      static_cast<uint32_t>(o0 + 8 * (g / 4) + g % 4) * plane, 0);
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < kBlocks; ++j) {
        const int m = mw + j * 32 + r, n = fast_div(min(m, m_end - 1), a.div_ohw), rem = m - n * a.OHW;
        const uint32_t yb = m < m_end ? static_cast<uint32_t>(n * a.O * a.OHW + rem) * 4u : kOob;
        uint32_t off[16];
        float q[16];
#pragma unroll
        for (int g = 0; g < 16; ++g) {
            const int o = o0 + 8 * (g / 4) + 4 * half + g % 4;
            off[g] = yb != kOob && o < a.O ? yb + static_cast<uint32_t>(o) * plane : kOob;
            if (has_res) q[g] = load_f32(rr, off[g]);
        }
#pragma unroll
        for (int g = 0; g < 16; ++g) {
            float v = sum(j, g);
            if (has_res) v = __fadd_rn(v, q[g]);
            if (do_relu) v = relu_sel(v);
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), yr, off[g], 0, 0);
        }
    }
}

// ------------------------------------------------------------------------------------------
// The packed filter: [o / 32][step][part][lane][16 bytes], lane = o % 32 + 32 * (group % 2).  256 threads, 32 output channels.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ void pack_tile(const float* __restrict__ w, char* __restrict__ u, int32_t O, int tile) {
    for (int i = static_cast<int>(threadIdx.x); i < kSteps * 64; i += 256) {
        const int s = i >> 6, lane = i & 63, o = tile * 32 + (lane & 31), g = 2 * s + (lane >> 5);
        float v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) v[t] = t < kK && g < kGroups && o < O ? kOperandScale * w[(static_cast<int64_t>(o) * kGroups + g) * kK + t] : 0.0f;
        const Split8 p = split8(v);
        char* const dst = u + (static_cast<int64_t>(tile) * kSteps + s) * 3072 + lane * 16;
        *reinterpret_cast<u32x4*>(dst) = p.h;
        *reinterpret_cast<u32x4*>(dst + 1024) = p.m;
        *reinterpret_cast<u32x4*>(dst + 2048) = p.l;
    }
}

#endif  // __HIPCC__

}  // namespace conv7_bx
}  // namespace kxc_hip
