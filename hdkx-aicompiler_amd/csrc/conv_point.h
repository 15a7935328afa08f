// conv_point.h -- 1x1 convolutions of at most 128 input channels on the bf16 matrix cores with three-part operands (bf16x3.h);
// included by conv2d_bf16x3.hip (selection, launch).
//
// Few input channels make such a call as many bytes as products: what a workgroup does before its first product and behind its last one
// decides.  So a workgroup keeps its 64 pixels: all their channels are loaded, split once and left in LDS as fragments ([part][step
// of 16 channels][channel half][pixel] of 16 bytes), and its four waves walk blocks of 32 output channels over them, one after the other.
//  * A block's filter fragments replace the block's before it register by register, behind the products that read those, and its residual
//    is requested ahead of the stores of the block before it: loads and stores complete in order, and a load behind a store waits for it.
//  * Large and small products have accumulators of their own (conv_bf16x3.h says why, and what happens to sums that are not finite).
//
// Bound by loading, splitting and storing around the products: 128 -> 512 channels at 28 x 28, batch 32, with a residual moves 116 MB and takes 34 us,
// 3.4 TB/s (the kernel of conv_bf16x3.h, which splits the pixels again for each 128 output channels, 46; the fp32 instructions 57); 64 -> 256 at
// 56 x 56, batch 64, with a residual 102 us, 4.5 TB/s (139 and 158); 64 -> 64 there 39 us (57 and 88); all with the filter's packing, and the first
// 40 (51) where each call finds other operands in the caches.  Small ones are
// a chain of loads, a split and two launches: 128 -> 256 at 20 x 24, batch 2 10.1 us (11.3 and 7.2), and keep the fp32 kernels.
#pragma once

#include "bf16x3.h"
#include "common.h"
#include "conv_bf16x3.h"

namespace kxc_hip {
namespace conv_pt {

constexpr int kPix = 64, kWaves = 4, kThreads = 64 * kWaves;
constexpr int kMaxSteps = 8;                           // of 16 channels
constexpr int64_t kMaxBlocks = 64;                     // of 32 output channels, of a workgroup
// Floats per channel of the area through which a wave turns 32 channels x 32 pixels (two half-waves, four channels apart, then write to
// different banks; rows of whole 16 bytes).
constexpr int kTurnPitch = 40;
inline size_t LdsBytes(int steps, int blocks) { return static_cast<size_t>(steps) * 6 * kPix * 16 + kWaves * 32 * kTurnPitch * 4 + static_cast<size_t>(blocks) * 128; }

struct Args {
    const float* x;
    const char* u;
    const float* bias;
    const float* res;
    float* y;
    const float* w;                     // the filter as it was given, for sums that are not finite
    int32_t C, O, HW, M;
    int32_t csteps;                     // steps of 64 channels of the packed filter
    int32_t blocks, groups;             // blocks of 32 output channels of a workgroup; workgroups that share their pixels
    int32_t num_units, units_per_xcd;
    uint32_t x_bytes, y_bytes, u_bytes, flags;
    FastDiv div_hw, div_groups;
};

#if defined(__HIPCC__)

using conv_bx::kOob;
using conv_bx::relu_sel;
using conv_bx::rsrc;

// CS: steps of 16 channels (the filter is packed in fours)
template <int CS>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) conv_point_kernel(const Args a) {
    request_args(a);
    constexpr int STEP = 2 * kPix * 16, PART = CS * STEP;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, half = lane >> 5, r = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float* const turn = reinterpret_cast<float*>(lds + 3 * PART) + wave * 32 * kTurnPitch;
    float* const bias_lds = reinterpret_cast<float*>(lds + 3 * PART) + kWaves * 32 * kTurnPitch;
    const int unit = static_cast<int>(blockIdx.x & 7) * a.units_per_xcd + static_cast<int>(blockIdx.x >> 3);
    if (unit >= a.num_units || static_cast<int>(blockIdx.x >> 3) >= a.units_per_xcd) return;
    const int p_tile = fast_div(unit, a.div_groups), group = unit - p_tile * a.groups;
    const int m0 = p_tile * kPix, first = group * a.blocks;
    const int blocks = min(a.blocks, (a.O + 31) / 32 - first);

    // ---- the pixels: a thread takes four of them (of one image: HW is a multiple of four) in eight channels
    const uint32_t plane = static_cast<uint32_t>(a.HW) * 4u;
    const __amdgpu_buffer_rsrc_t xr = rsrc(a.x, a.x_bytes);
    constexpr int kUnits = CS * 32, U = (kUnits + kThreads - 1) / kThreads;
    f32x4 xv[U][8];
#pragma unroll
    for (int k = 0; k < U; ++k) {
        const int u = tid + k * kThreads, c = (u >> 4) * 8, m = m0 + (u & 15) * 4, n = fast_div(min(m, a.M - 1), a.div_hw);
        const uint32_t at = static_cast<uint32_t>(n * a.C * a.HW + m - n * a.HW) * 4u + static_cast<uint32_t>(c) * plane;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            xv[k][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, u < kUnits && m < a.M && c + j < a.C ? at + static_cast<uint32_t>(j) * plane : kOob, 0, 0));
    }

    // ---- filter fragments of a block: [block][step][part] runs of 1 KiB
    const __amdgpu_buffer_rsrc_t ur = rsrc(a.u, a.u_bytes);
    const uint32_t block_bytes = static_cast<uint32_t>(a.csteps) * (4 * 3072u);
    u32x4 ua[CS][3];
    auto load_a = [&](int block, int s, int p) __attribute__((always_inline)) {
        ua[s][p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ur, static_cast<uint32_t>(lane) * 16u, static_cast<uint32_t>(block) * block_bytes + static_cast<uint32_t>(s) * 3072u + static_cast<uint32_t>(p) * 1024u, 0));
    };
    if (wave < blocks) {
#pragma unroll
        for (int s = 0; s < CS; ++s)
#pragma unroll
            for (int p = 2; p >= 0; --p) load_a(first + wave, s, p);
    }

    // ---- this lane's pixels, their residual
    const bool has_bias = (a.flags & KXC_HIP_CONV_BIAS) != 0, has_res = (a.flags & KXC_HIP_CONV_RESIDUAL) != 0, do_relu = (a.flags & KXC_HIP_CONV_RELU) != 0;
    const __amdgpu_buffer_rsrc_t yr = rsrc(a.y, a.y_bytes), rr = rsrc(has_res ? a.res : a.y, has_res ? a.y_bytes : 0u);
    // (a lane finishes four neighbouring pixels of channel 8 t + lane / 8, t = 0 .. 3, of either pixel block)
    const int oc = lane >> 3, quad = lane & 7;
    uint32_t yb[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int m = m0 + j * 32 + quad * 4, n = fast_div(min(m, a.M - 1), a.div_hw);
        yb[j] = m < a.M ? static_cast<uint32_t>(n * a.O * a.HW + m - n * a.HW) * 4u + static_cast<uint32_t>(oc) * plane : kOob;
    }
    auto offset = [&](int block, int t, int j) __attribute__((always_inline)) {
        const int o = block * 32 + 8 * t;
        return o + oc < a.O && yb[j] != kOob ? yb[j] + static_cast<uint32_t>(o) * plane : kOob;
    };
    f32x4 qv[4][2];
    auto load_res = [&](int block) __attribute__((always_inline)) {
        if (has_res) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int t = 0; t < 4; ++t) qv[t][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rr, offset(block, t, j), 0, 0));
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    if (wave < blocks) load_res(first + wave);
    for (int i = tid; i < blocks * 32; i += kThreads) bias_lds[i] = has_bias && first * 32 + i < a.O ? a.bias[first * 32 + i] : 0.0f;

    // ---- split into three parts once
#pragma unroll
    for (int k = 0; k < U; ++k) {
        const int u = tid + k * kThreads;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float t[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) t[c] = __fmul_rn(xv[k][c][j], kOperandScale);
            const Split8 s = split8(t);
            if (u < kUnits) {
                char* const dst = lds + ((u >> 4) * kPix + (u & 15) * 4 + j) * 16;
                *reinterpret_cast<u32x4*>(dst) = s.h;
                *reinterpret_cast<u32x4*>(dst + PART) = s.m;
                *reinterpret_cast<u32x4*>(dst + 2 * PART) = s.l;
            }
        }
    }
    __syncthreads();

    const char* const mine = lds + (half * kPix + r) * 16;
    u32x4 vb[2][3];
    auto read_b = [&](int s, int p) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j) vb[j][p] = *reinterpret_cast<const u32x4*>(mine + p * PART + s * STEP + j * 512);
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int b = wave; b < blocks; b += kWaves) {
        const int block = first + b;
        const bool more = b + kWaves < blocks;
        f32x16 big[2], small[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int g = 0; g < 16; ++g) { big[j][g] = 0.0f; small[j][g] = 0.0f; }
        constexpr int PA[6] = {0, 1, 0, 2, 1, 0}, PB[6] = {2, 1, 1, 0, 0, 0};
        read_b(0, 2);
        read_b(0, 1);
        read_b(0, 0);
#pragma unroll
        for (int s = 0; s < CS; ++s) {
#pragma unroll
            for (int p = 0; p < 6; ++p) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    f32x16& acc = p == 5 ? big[j] : small[j];
                    acc = mfma_bf16(ua[s][PA[p]], vb[j][PB[p]], acc);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (s + 1 < CS && p == 0) read_b(s + 1, 2);
                if (s + 1 < CS && p == 2) read_b(s + 1, 1);
                if (s + 1 < CS && p == 5) read_b(s + 1, 0);
                if (p >= 3 && more) load_a(block + kWaves, s, 5 - p);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // register g = channel 8 (g / 4) + 4 half + g % 4, lane = pixel: turned through LDS, so that a lane stores 16 bytes
        uint32_t odd = 0;                 // bit 16 * pixel block + 4 * t + pixel: not finite, formed again below
        f32x4 out[4][2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int g = 0; g < 16; ++g)
                turn[(8 * (g / 4) + 4 * half + g % 4) * kTurnPitch + r] = __fmul_rn(__fadd_rn(big[j][g], small[j][g]), kSumScale);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(turn + (8 * t + oc) * kTurnPitch + quad * 4);
                const float bv = bias_lds[b * 32 + 8 * t + oc];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float z = v[e];
                    if (!(__builtin_fabsf(z) < __builtin_inff())) odd |= 1u << (16 * j + 4 * t + e);
                    if (has_bias) z = __fadd_rn(z, bv);
                    if (has_res) z = __fadd_rn(z, qv[t][j][e]);
                    out[t][j][e] = do_relu ? relu_sel(z) : z;
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // (the residual may be the output's own buffer: a wave reads what it stores itself, and an odd quadruple is not stored yet)
        if (more) load_res(block + kWaves);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                // (no scalar offset on a 16-byte store: wino_bf16x3.h)
                const uint32_t at = (odd >> (16 * j + 4 * t)) & 15u ? kOob : offset(block, t, j);
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, out[t][j]), yr, at, 0, 0);
            }
        __builtin_amdgcn_sched_barrier(0);
        if (odd == 0) continue;
#pragma unroll 1
        for (int k = 0; k < 32; ++k) {
            const int o = block * 32 + 8 * (k >> 2 & 3) + oc, m = m0 + (k >> 4) * 32 + quad * 4 + (k & 3);
            if (((odd >> (k & ~3)) & 15u) == 0 || o >= a.O || m >= a.M) continue;      // (the whole quadruple)
            const int n = fast_div(m, a.div_hw), rem = m - n * a.HW;
            const int64_t at = static_cast<int64_t>(n * a.O + o) * a.HW + rem;
            float s = 0.0f;
#pragma unroll 1
            for (int c = 0; c < a.C; ++c) s = __fadd_rn(s, __fmul_rn(a.x[static_cast<int64_t>(n * a.C + c) * a.HW + rem], a.w[static_cast<int64_t>(o) * a.C + c]));
            if (has_bias) s = __fadd_rn(s, a.bias[o]);
            if (has_res) s = __fadd_rn(s, a.res[at]);
            a.y[at] = do_relu ? relu_sel(s) : s;
        }
    }
}

#endif  // __HIPCC__

}  // namespace conv_pt
}  // namespace kxc_hip
