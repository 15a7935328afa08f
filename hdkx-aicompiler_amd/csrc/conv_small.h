// conv_small.h -- convolution of small launches in ONE kernel: tiles of 16 output channels x 16 pixels whose reduction is
// split over the waves of a workgroup (v_mfma_f32_16x16x4_f32, fp32 operands as they are, no prepared weights).
//
// A small launch (batch 1, deep layers) has little to do and few places to do it: 512 -> 512 channels at 7 x 7 is 116 M
// products in 49 x 512 outputs.  Large tiles leave compute units idle, and splitting the reduction over workgroups takes
// a second launch to add the parts.  16 x 16 tiles give 128 to 800 workgroups, and KS waves share a tile's channels: wave
// w takes the chunks w, w + KS, ... of 4 * CPG channels, lane group g = lane / 16 the channels g * CPG .. of a chunk (a
// matrix instruction takes one k from each group; which k those are does not matter as long as both operands agree).
//   W  the 16 rows' weights of a chunk are contiguous runs of 4 * CPG * KH * KW floats: LDS-direct loads of 1 KiB bring them
//      in whole cache lines (a lane reading its own row would touch 64 lines a load), and every lane moves its
//      CPG * KH * KW values into registers with 16-byte reads.  The LDS belongs to the wave alone: no barrier.
//   X  XI = 0: straight from memory, one 4-byte load per matrix instruction (16 neighbouring pixels of four channels), E ahead; a
//      buffer offset per filter tap, out of range at the zero padding, the channel in the scalar offset.  The address unit
//      takes 16 cycles an instruction for a whole compute unit, which bounds this form once four waves are at it.
//      ROWS: one 12-byte load for the three values of a filter row, 12 loads a chunk instead of 36 (us, with a wave's last chunk
//      requesting nothing behind it: 64 channels at 56 x 56 7.9 -> 7.1, 64 -> 128 with stride 2 and the second output 8.8 -> 6.1, 128 ->
//      256 7.2 -> 5.4, at batch 3 11.1 -> 8.2).
//      XI > 0: the whole input rows that a tile touches, one contiguous run per channel, in XI loads of 1 KiB staged like W
//      (tiles then never cross images); a chunk's operands move into registers at its start.  Fewer loads but more
//      instructions: better for narrow maps, where few rows hold a tile and few tiles hide nothing.
// The KS partial tiles meet in LDS at the end.  What bounds it: loads (above) and the fp32 matrix instructions of the busiest
// compute unit, behind the chain launch - first loads - last store.  Measured, us, batch 1, residual and ReLU, against the
// Winograd kernel with its adding launch: 64 channels at 56 x 56 10.2 -> 8.6, 128 at 28 x 28 10.8 -> 7.8, 256 at 14 x 14
// 10.8 -> 7.6, 512 at 7 x 7 12.3 -> 11.1; against the implicit GEMM with two outputs: 64 -> 128 with stride 2 12.7 -> 8.7,
// 128 -> 256 13.4 -> 7.2, 256 -> 512 14.0 -> 8.6.  1x1, 256 -> 512 at 14 x 14: 9.3 -> 4.2.
#pragma once

#include "common.h"

namespace kxc_hip {
namespace conv_small {

struct Args {
    const float* x;
    const float* w;
    const float* bias;
    const float* res;
    float* y;
    const float* w2;                   // second output: a 1x1 convolution with the same strides on the same input
    const float* bias2;
    float* y2;
    int32_t N, C, H, W, O, OH, OW, sh, sw, ph, pw, dh, dw;
    int32_t M, OHW, nchunks;
    int32_t words;                     // 16-byte words of a channel's staged rows
    int32_t delta;                     // values between the 16-byte boundary below x and x
    int32_t image_tiles, p_tiles, o_tiles, num_tiles, tiles_per_xcd, o_fastest;
    uint32_t x_bytes, w_bytes, w2_bytes, flags;
    FastDiv div_ohw, div_ow, div_tiles, div_image, div_words;
};

#if defined(__HIPCC__)

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f3 __attribute__((ext_vector_type(3)));
typedef __attribute__((address_space(3))) void* lds_p;
constexpr uint32_t kOutside = 0x80000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), 0x00020000);
}
__device__ __forceinline__ void to_lds16(__amdgpu_buffer_rsrc_t rs, char* lds, uint32_t voffset, uint32_t soffset) {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_p)lds, 16, voffset, soffset, 0, 0);
#endif
}

// ROWS (XI = 0, 3x3 filters without dilation along a row, one column of padding at most, rows of three values at least): the three
// values that a filter row touches by one 12-byte load, moved to the row's end where it would reach across it.
template <int KH, int KW, int CPG, int XI, int RO, int KS, bool DS = false, bool ROWS = false>
__global__ void __launch_bounds__(64 * KS) __attribute__((amdgpu_waves_per_eu(2))) conv_small_kernel(const Args a) {
    request_args(a);
    constexpr bool STAGED = XI > 0;
    constexpr int KHW = KH * KW, E = CPG * KHW, WI = RO * E / 4, NB = DS ? 2 * RO : RO;
    static_assert(E % 4 == 0 && E <= 36 && (!DS || CPG == 4), "chunk layout");      // (36 loads of X in flight: vmcnt holds 63)
    constexpr int WAVE_LDS = (WI + XI) * 1024 + (STAGED ? 32 : 0);
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int tile = static_cast<int>(blockIdx.x & 7) * a.tiles_per_xcd + static_cast<int>(blockIdx.x >> 3);
    if (tile >= a.num_tiles || static_cast<int>(blockIdx.x >> 3) >= a.tiles_per_xcd) return;
    const int hi = fast_div(tile, a.div_tiles), lo = tile - hi * (a.o_fastest ? a.o_tiles : a.p_tiles);
    const int o0 = (a.o_fastest ? lo : hi) * 16 * RO, pt = a.o_fastest ? hi : lo;

    // ---- weights of a chunk: RO * 16 runs of 4 * E values
    const __amdgpu_buffer_rsrc_t wr = rsrc(a.w, a.w_bytes);
    char* const mine = lds + wave * WAVE_LDS;
    const uint32_t row_bytes = static_cast<uint32_t>(a.C) * (KHW * 4u);
    uint32_t wo[WI];
#pragma unroll
    for (int i = 0; i < WI; ++i) {
        const int word = i * 64 + lane, row = word / E;
        wo[i] = o0 + row < a.O ? static_cast<uint32_t>(o0 + row) * row_bytes + static_cast<uint32_t>(word - row * E) * 16u : kOutside;
    }
    auto load_w = [&](int chunk) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WI; ++i) to_lds16(wr, mine + i * 1024, wo[i], static_cast<uint32_t>(chunk) * (E * 16u));
    };
    float wf[RO][E];
    auto read_w = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RO; ++i)
#pragma unroll
            for (int q = 0; q < E / 4; ++q) {
                const f4 v = *reinterpret_cast<const f4*>(mine + ((i * 16 + r) * E + g * (E / 4) + q) * 16);
#pragma unroll
                for (int e = 0; e < 4; ++e) wf[i][4 * q + e] = v[e];
            }
    };
    if (wave < a.nchunks) load_w(wave);
    const __amdgpu_buffer_rsrc_t wr2 = rsrc(DS ? a.w2 : a.w, DS ? a.w2_bytes : 0u);
    uint32_t wo2[DS ? RO : 1];
    f4 wf2[DS ? RO : 1];
    if constexpr (DS) {
#pragma unroll
        for (int i = 0; i < RO; ++i)
            wo2[i] = o0 + i * 16 + r < a.O ? static_cast<uint32_t>((o0 + i * 16 + r) * a.C + g * 4) * 4u : kOutside;
    }
    auto load_w2 = [&](int chunk) __attribute__((always_inline)) {
        if constexpr (DS) {
#pragma unroll
            for (int i = 0; i < RO; ++i)
                wf2[i] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(wr2, wo2[i], static_cast<uint32_t>(chunk) * 64u, 0));
        }
    };

    // ---- pixels of the tile, and the one of this lane
    const int HW = a.H * a.W;
    const uint32_t plane = static_cast<uint32_t>(HW) * 4u;
    int n, q0, q;                      // image, first pixel (only used when tiles stay within an image), this lane's pixel
    bool in;
    if constexpr (STAGED) {
        n = fast_div(pt, a.div_image);
        q0 = (pt - n * a.image_tiles) * 16;
        q = q0 + r;
        in = q < a.OHW;
    } else {
        const int m = pt * 16 + r;
        n = fast_div(m, a.div_ohw);
        q = m - n * a.OHW;
        q0 = 0;
        in = m < a.M;
    }
    const int oh = fast_div(q, a.div_ow), ow = q - oh * a.OW;
    const int ih = oh * a.sh - a.ph, iw = ow * a.sw - a.pw;
    auto valid = [&](int t) __attribute__((always_inline)) {
        const int y = ih + t / KW * a.dh, x = iw + t % KW * a.dw;
        return in && static_cast<uint32_t>(y) < static_cast<uint32_t>(a.H) && static_cast<uint32_t>(x) < static_cast<uint32_t>(a.W);
    };

    f4 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](int j, float x) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RO; ++i) {
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i][j], x, acc[i], 0, 0, 0);
            if constexpr (DS) {
                if (j % KHW == KHW / 2) acc[RO + i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf2[i][j / KHW], x, acc[RO + i], 0, 0, 0);
            }
        }
    };

    if constexpr (STAGED) {
        const __amdgpu_buffer_rsrc_t xr = rsrc(a.x - a.delta, a.x_bytes);
        const uint32_t xs = static_cast<uint32_t>(wave * WAVE_LDS + WI * 1024);
        // rows r0 .. r1 of every channel; runs are loaded from the 16-byte boundary below them
        const int q1 = min(q0 + 16, a.OHW) - 1;
        const int r0 = min(max(fast_div(q0, a.div_ow) * a.sh - a.ph, 0), a.H - 1);
        const int r1 = max(min(fast_div(q1, a.div_ow) * a.sh - a.ph + (KH - 1) * a.dh, a.H - 1), r0);
        const int run = (r1 - r0 + 1) * a.W, first = n * a.C * HW + r0 * a.W + a.delta;
        uint32_t xo[XI > 0 ? XI : 1];
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const int word = i * 64 + lane, c = fast_div(word, a.div_words), k = word - c * a.words;
            const int at = first + c * HW;
            xo[i] = c < 4 * CPG && k * 4 < run + (at & 3) ? static_cast<uint32_t>((at & ~3) + k * 4) * 4u : kOutside;
        }
        auto load_x = [&](int chunk) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < XI; ++i)
                if (i * 64 < a.words * 4 * CPG) to_lds16(xr, lds + xs + i * 1024, xo[i], static_cast<uint32_t>(chunk * 4 * CPG) * plane);
        };
        if (wave < a.nchunks) load_x(wave);
        // channel g * CPG + jc, filter row rh; the column rides in the instruction
        uint32_t xa[CPG][KH];
        bool ok[KHW];
#pragma unroll
        for (int t = 0; t < KHW; ++t) ok[t] = valid(t);
#pragma unroll
        for (int jc = 0; jc < CPG; ++jc) {
            const int c = g * CPG + jc, mis = (first + c * HW) & 3;
#pragma unroll
            for (int rh = 0; rh < KH; ++rh) {
                // (a row or column that is not staged is never used: any address nearby will do)
                const int y = min(max(ih + rh * a.dh, r0), r1) - r0;
                xa[jc][rh] = xs + static_cast<uint32_t>(c * a.words * 16 + (mis + y * a.W + max(min(iw, a.W - 1), 1 - KW)) * 4);
            }
        }
        for (int chunk = wave; chunk < a.nchunks; chunk += KS) {
            float xf[E];
            load_w2(chunk);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            read_w();
#pragma unroll
            for (int j = 0; j < E; ++j) xf[j] = *reinterpret_cast<const float*>(lds + xa[j / KHW][j % KHW / KW] + j % KW * 4);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // read before they are written again
            __builtin_amdgcn_sched_barrier(0);
            if (chunk + KS < a.nchunks) {
                load_w(chunk + KS);
                load_x(chunk + KS);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < E; ++j) multiply(j, ok[j % KHW] ? xf[j] : 0.0f);
        }
    } else {
        const __amdgpu_buffer_rsrc_t xr = rsrc(a.x, a.x_bytes);
        static_assert(!ROWS || KW == 3, "rows of three");
        constexpr int PER = ROWS ? 3 : 1, XL = E / PER;            // values per load; loads of a chunk
        uint32_t xo[KHW / PER];
        const int xs = ROWS ? min(max(iw, 0), a.W - 3) : iw, shift = iw - xs;       // (-1, 0, 1)
        const bool first = iw >= 0, last = iw + 2 < a.W;
#pragma unroll
        for (int t = 0; t < KHW / PER; ++t) {
            const int y = ih + t * PER / KW * a.dh;
            const bool there = ROWS ? in && static_cast<uint32_t>(y) < static_cast<uint32_t>(a.H) : valid(t);
            xo[t] = there ? static_cast<uint32_t>(n * a.C + g * CPG) * plane + static_cast<uint32_t>(y * a.W + (ROWS ? xs : iw + t % KW * a.dw)) * 4u : kOutside;
        }
        float xf[E];
        auto load_x = [&](int chunk, int j) __attribute__((always_inline)) {
            const uint32_t so = static_cast<uint32_t>(chunk * 4 * CPG + j * PER / KHW) * plane;
            if constexpr (ROWS) {
                const f3 v = __builtin_bit_cast(f3, __builtin_amdgcn_raw_buffer_load_b96(xr, xo[j % (KHW / PER)], so, 0));
#pragma unroll
                for (int e = 0; e < 3; ++e) xf[3 * j + e] = v[e];
            } else {
                xf[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, xo[j % KHW], so, 0));
            }
        };
        if (wave < a.nchunks) {
#pragma unroll
            for (int j = 0; j < XL; ++j) {
                load_x(wave, j);
                __builtin_amdgcn_sched_barrier(0);                 // in this order: the waits of the loop count on it
            }
            // (a wave's last chunk requests nothing: with one or two chunks per wave a chunk more would be a third to half of all loads)
            auto step = [&](int chunk, auto more) __attribute__((always_inline)) {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(XL) : "memory");     // all but the loads of X behind the weights
                load_w2(chunk);
                read_w();
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // read before they are written again
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (decltype(more)::value) load_w(chunk + KS);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < XL; ++j) {
                    if constexpr (ROWS) {
                        const float v0 = xf[3 * j], v1 = xf[3 * j + 1], v2 = xf[3 * j + 2];
                        multiply(3 * j, first ? (shift > 0 ? v1 : v0) : 0.0f);
                        multiply(3 * j + 1, shift == 0 ? v1 : shift > 0 ? v2 : v0);
                        multiply(3 * j + 2, last ? (shift < 0 ? v1 : v2) : 0.0f);
                    } else {
                        multiply(j, xf[j]);
                    }
                    if constexpr (decltype(more)::value) load_x(chunk + KS, j);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            int chunk = wave;
            for (; chunk + KS < a.nchunks; chunk += KS) step(chunk, std::true_type{});
            step(chunk, std::false_type{});
        }
    }
    __syncthreads();
    // partial sums [block][wave][lane][16 bytes]: register e of a lane is row 4*g + e, column r
#pragma unroll
    for (int b = 0; b < NB; ++b) *reinterpret_cast<f4*>(lds + ((b * KS + wave) * 64 + lane) * 16) = acc[b];
    __syncthreads();
    // a thread finishes one output at a time: 16 neighbouring threads, 16 neighbouring pixels
    const int tid = static_cast<int>(threadIdx.x);
#pragma unroll
    for (int t = 0; t < (NB * 256 + 64 * KS - 1) / (64 * KS); ++t) {
        const int e = tid + t * 64 * KS, b = e >> 8, row = (e >> 4) & 15, col = e & 15;
        if (e >= NB * 256) break;
        const float* const p = reinterpret_cast<const float*>(lds) + (b * KS * 64 + (row >> 2) * 16 + col) * 4 + (row & 3);
        float v = p[0];
#pragma unroll
        for (int w = 1; w < KS; ++w) v = __fadd_rn(v, p[w * 256]);
        const int o = o0 + b % RO * 16 + row;
        int nn = n, at = q0 + col;
        bool store = o < a.O;
        if constexpr (STAGED) {
            store = store && at < a.OHW;
        } else {
            const int m = pt * 16 + col;
            nn = fast_div(m, a.div_ohw);
            at = m - nn * a.OHW;
            store = store && m < a.M;
        }
        if (!store) continue;
        at += (nn * a.O + o) * a.OHW;
        if (DS && b >= RO) {
            if (a.bias2) v = __fadd_rn(v, a.bias2[o]);
            a.y2[at] = v;
        } else {
            if (a.flags & KXC_HIP_CONV_BIAS) v = __fadd_rn(v, a.bias[o]);
            if (a.flags & KXC_HIP_CONV_RESIDUAL) v = __fadd_rn(v, a.res[at]);
            if (a.flags & KXC_HIP_CONV_RELU) v = v > 0.0f ? v : 0.0f;
            a.y[at] = v;
        }
    }
}

#endif  // __HIPCC__

}  // namespace conv_small
}  // namespace kxc_hip
