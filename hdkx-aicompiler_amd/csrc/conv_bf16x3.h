// conv_bf16x3.h -- implicit-GEMM convolution (NCHW data, OIHW weights, fp32, any filter, stride and dilation) on the bf16
// matrix cores with three-part operands (bf16x3.h); included by conv2d_f32.hip, which holds the fp32-instruction kernels,
// the selection and the entry points.
//
// D[o][pixel] += W[o][k] X[k][pixel].  A lane of v_mfma_f32_32x32x16_bf16 holds eight consecutive k of one row or column;
// here those are eight channels of one filter tap, so LDS keeps both operands as 16-byte words of eight channels, one
// word per part:
//   X  [part][channel block][position of the patch]   the raw input rows the tile touches, zero padding materialised; a
//                                                     filter tap is the same patch read at a shifted address
//   W  [part][q][output channel]                      q = tap * CB + channel block, the two lane halves of a k-step
//                                                     take q = 2 step and 2 step + 1
// A stage is a chunk of CB channel blocks and a group of its k-steps.  Its raw floats are requested into registers while the
// stage before it is multiplied, then split (11 instructions per two values) and written; every input value is split once
// per workgroup and used by all its output channels and taps.  What bounds it: the matrix cores where two workgroups share
// a compute unit (one stages while the other multiplies), otherwise the staging; a 64 x 64 block per wave reads 64 bytes
// of LDS per clock and compute unit at the full matrix rate, half of what LDS delivers.
//
// C4: images of at most four channels.  Eight channels per word would leave five eighths of the matrix work on zeros; the
// word is two neighbouring columns of four channels instead (positions of 8 bytes, q = (filter row, column pair)).
//
// DS: a second output, the 1x1 convolution with the same strides whose operand is tap ds_tap of this one's window (see
// ConvArgs): CB more q per chunk read that tap against a second weight tensor, into accumulators of their own.
//
// KS: the waves of a workgroup form KS groups that take every KS-th k-step of a stage and add their sums through LDS at
// the end, for launches with too few tiles to fill the GPU.
//
// A non-finite operand makes a sum NaN (bf16x3.h); a wave that finds one among its sums evaluates its outputs again with
// the fp32 loop, so Inf and NaN spread as in the other kernels.
#pragma once

#include "bf16x3.h"

namespace kxc_hip {
namespace conv_bx {

struct Args {
    const float* x;
    const float* w;
    const float* bias;
    const float* res;
    float* y;
    const float* w2;
    const float* bias2;
    float* y2;
    float* partial;
    int32_t N, C, H, W, O, OH, OW, KH, KW;
    int32_t sh, sw, ph, pw, dh, dw;
    int32_t Hp, Wp, Hv, row_step;      // padded extent; rows the kernel sees and their distance in input rows (ConvArgs)
    int32_t M, OHW;
    int32_t chs;                       // positions per channel block of the patch in LDS
    int32_t cb, nq, nq_main;           // channel blocks per chunk; q of a chunk (even), of which the main output's (even)
    int32_t group_steps, ngroups;      // k-steps per stage, stages per chunk
    int32_t nchunks, gsplit, cps;
    int32_t ds_off;                    // position offset of the second output's tap
    int32_t p_tiles, o_tiles, num_tiles, tiles_per_xcd, o_fastest;
    uint32_t x_bytes, w_bytes, w2_bytes, flags;
    int64_t out_elems;
    FastDiv div_wp, div_hp, div_ohw, div_ow, div_otiles, div_ptiles, div_gsplit, div_chs, div_gq, div_cb, div_kw;
};

constexpr int kMaxQ = 128;             // entries of the tap table

#if defined(__HIPCC__)

// One output summed like the direct kernel does, over input channels [c_lo, c_hi).
__device__ __noinline__ float direct_sum(const float* x, const float* w, int32_t C, int32_t H, int32_t W, int32_t KH, int32_t KW, int32_t c_lo,
                                         int32_t c_hi, int32_t ih0, int32_t iw0, int32_t dh, int32_t dw) {
    float s = 0.0f;
    for (int32_t c = c_lo; c < c_hi; ++c)
        for (int32_t rh = 0; rh < KH; ++rh)
            for (int32_t rw = 0; rw < KW; ++rw) {
                const int32_t ih = ih0 + rh * dh, iw = iw0 + rw * dw;
                const float v = ih >= 0 && ih < H && iw >= 0 && iw < W ? x[(static_cast<int64_t>(c) * H + ih) * W + iw] : 0.0f;
                s = __fadd_rn(s, __fmul_rn(v, w[(static_cast<int64_t>(c) * KH + rh) * KW + rw]));
            }
    return s;
}

template <int RO, int RP, int WO, int WP, int KS, int IX, int IW, bool C4, bool DS>
__global__ void __launch_bounds__(64 * WO * WP * KS) __attribute__((amdgpu_waves_per_eu(2))) conv_bf16x3_kernel(const Args a) {
    constexpr int NW = WO * WP, NT = 64 * NW * KS;
    constexpr int TO = 32 * RO * WO, TP = 32 * RP * WP;
    constexpr int XB = C4 ? 8 : 16;                           // bytes of a position in one part
    constexpr int WROW = (TO + 1) * 16;                       // bytes of one q of the weight tile (one word of skew per q)
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, half = lane >> 5, r = lane & 31;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kgroup = wave_all / NW, wave = wave_all - kgroup * NW;
    const int wave_o = wave / WP, wave_p = wave - wave_o * WP;
    // consecutive workgroups go to the 8 XCDs round-robin; each XCD (own L2) takes a contiguous run of units
    const int unit = (blockIdx.x & 7) * a.tiles_per_xcd + (blockIdx.x >> 3);
    if (unit >= a.num_tiles * a.gsplit || static_cast<int>(blockIdx.x >> 3) >= a.tiles_per_xcd) return;
    const int tile = a.gsplit > 1 ? fast_div(unit, a.div_gsplit) : unit;
    const int split = unit - tile * a.gsplit;
    int p_tile, o_tile;
    if (a.o_fastest) { p_tile = fast_div(tile, a.div_otiles); o_tile = tile - p_tile * a.o_tiles; }
    else { o_tile = fast_div(tile, a.div_ptiles); p_tile = tile - o_tile * a.p_tiles; }
    const int m0 = p_tile * TP, o0 = o_tile * TO;
    const int c_lo = split * a.cps, c_hi = min(a.nchunks, c_lo + a.cps);

    int* const ktab = reinterpret_cast<int*>(lds);            // q -> byte offset of its positions inside a part of X
    char* const xs = lds + kMaxQ * 4;
    const int xpart = (C4 ? 1 : a.cb) * a.chs * XB;
    char* const ws = xs + 3 * xpart;
    const int gq = 2 * a.group_steps, wpart = gq * WROW;

    for (int q = tid; q < a.nq; q += NT) {
        int off = 0;
        if (C4) {
            const int ncp = (a.KW + 1) >> 1, rh = q / ncp, cp = q - rh * ncp;
            if (rh < a.KH) off = (rh * a.dh * a.Wp + 2 * cp) * XB;
        } else if (q < a.KH * a.KW * a.cb) {
            const int tap = fast_div(q, a.div_cb), cb = q - tap * a.cb, rh = fast_div(tap, a.div_kw), rw = tap - rh * a.KW;
            off = (cb * a.chs + rh * a.dh * a.Wp + rw * a.dw) * XB;
        } else if (DS && q >= a.nq_main && q < a.nq_main + a.cb) {
            off = ((q - a.nq_main) * a.chs + a.ds_off) * XB;
        }
        ktab[q] = off;
    }

    // ---- geometry of this tile in padded row space
    const int m_last = min(m0 + TP, a.M) - 1;
    int qmin, P;
    {
        const int n = fast_div(m0, a.div_ohw), rem = m0 - n * a.OHW;
        qmin = n * a.Hp + fast_div(rem, a.div_ow) * a.sh;
        const int n2 = fast_div(m_last, a.div_ohw), rem2 = m_last - n2 * a.OHW;
        P = (n2 * a.Hp + fast_div(rem2, a.div_ow) * a.sh + (a.KH - 1) * a.dh - qmin + 1) * a.Wp;
    }
    const uint32_t plane_bytes = static_cast<uint32_t>(a.H * a.W) * 4u;
    const int KHW = a.KH * a.KW;
    uint32_t goff[IX];           // byte offset of channel 0 of the item's block; item i of a thread is word i * NT + tid of X
    int xleft[IX];               // channels of the item's block before the chunk's first (tail chunks)
#pragma unroll
    for (int i = 0; i < IX; ++i) {
        const int item = i * NT + tid;
        const int cb = C4 ? 0 : fast_div(item, a.div_chs), pos = item - cb * a.chs;
        const int q = fast_div(pos, a.div_wp), iw = pos - q * a.Wp - a.pw;
        const int Q = qmin + q, n = fast_div(Q, a.div_hp), ih = Q - n * a.Hp - a.ph;
        const bool ok = (C4 ? pos < a.chs : cb < a.cb) && pos < P && n < a.N && ih >= 0 && ih < a.Hv && iw >= 0 && iw < a.W;
        goff[i] = ok ? static_cast<uint32_t>(((n * a.C + cb * 8) * a.H + ih * a.row_step) * a.W + iw) * 4u : kOobOffset;
        xleft[i] = cb * 8;
    }
    const int x_items = (C4 ? 1 : a.cb) * a.chs;
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(a.x, a.x_bytes);
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(a.w, a.w_bytes);
    const __amdgpu_buffer_rsrc_t w2r = make_rsrc(DS ? a.w2 : a.w, DS ? a.w2_bytes : 0u);
    auto ldf = [](__amdgpu_buffer_rsrc_t rs, uint32_t vo, uint32_t so) __attribute__((always_inline)) {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, vo, so, 0));
    };

    // ---- raw floats of one stage in registers
    constexpr int XV = C4 ? 4 : 8;
    float xv[IX][XV], wv[IW][8];
    auto load_x = [&](int chunk) __attribute__((always_inline)) {
        const int c0 = chunk * a.cb * 8;
#pragma unroll
        for (int i = 0; i < IX; ++i) {
            if (i * NT >= x_items) break;
            if (C4) {
#pragma unroll
                for (int j = 0; j < XV; ++j) xv[i][j] = j < a.C ? ldf(xr, goff[i], static_cast<uint32_t>(j) * plane_bytes) : 0.0f;
            } else if (c0 + a.cb * 8 <= a.C) {
#pragma unroll
                for (int j = 0; j < XV; ++j) xv[i][j] = ldf(xr, goff[i], static_cast<uint32_t>(c0 + j) * plane_bytes);
            } else {
#pragma unroll
                for (int j = 0; j < XV; ++j)
                    xv[i][j] = ldf(xr, c0 + xleft[i] + j < a.C ? goff[i] : kOobOffset, static_cast<uint32_t>(c0 + j) * plane_bytes);
            }
        }
    };
    auto load_w = [&](int chunk, int group) __attribute__((always_inline)) {
        const int c0 = chunk * a.cb * 8;
#pragma unroll
        for (int i = 0; i < IW; ++i) {
            if (i * NT >= TO * gq) break;
            const int item = i * NT + tid;
            const int o = fast_div(item, a.div_gq), q = item - o * gq + group * gq;
            const bool row = o < TO && o0 + o < a.O;
            if (C4) {
                const int ncp = (a.KW + 1) >> 1, rh = q / ncp, cp = q - rh * ncp;
                const uint32_t at = static_cast<uint32_t>((o0 + o) * a.C * KHW + rh * a.KW + 2 * cp) * 4u;
                const uint32_t first = row && rh < a.KH ? at : kOobOffset, second = row && rh < a.KH && 2 * cp + 1 < a.KW ? at + 4u : kOobOffset;
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    wv[i][j] = (j & 3) < a.C ? ldf(wr, j < 4 ? first : second, static_cast<uint32_t>((j & 3) * KHW) * 4u) : 0.0f;
            } else {
                const int tap = fast_div(q, a.div_cb), cb = q - tap * a.cb;
                const bool main = q < KHW * a.cb;
                const bool second = DS && q >= a.nq_main && q < a.nq_main + a.cb;
                const int cb2 = q - a.nq_main;
                // (one descriptor per load: the wave's lanes hold items of both tensors, the other one's read as zero)
                const uint32_t v1 = row && main ? static_cast<uint32_t>(((o0 + o) * a.C + cb * 8) * KHW + tap) * 4u : kOobOffset;
                const uint32_t v2 = row && second ? static_cast<uint32_t>((o0 + o) * a.C + cb2 * 8) * 4u : kOobOffset;
                const int left = a.C - c0 - (second ? cb2 : cb) * 8;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float v = ldf(wr, j < left ? v1 : kOobOffset, static_cast<uint32_t>((c0 + j) * KHW) * 4u);
                    if constexpr (DS) v = second ? ldf(w2r, j < left ? v2 : kOobOffset, static_cast<uint32_t>(c0 + j) * 4u) : v;
                    wv[i][j] = v;
                }
            }
        }
    };
    auto store_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < IX; ++i) {
            if (i * NT >= x_items) break;
            const int item = i * NT + tid;
            if (item < x_items) {
                char* const dst = xs + item * XB;
                if constexpr (C4) {
                    u32x2 h, m, l;
                    uint32_t t0, t1, t2;
                    split_pair(xv[i][0], xv[i][1], t0, t1, t2); h[0] = t0; m[0] = t1; l[0] = t2;
                    split_pair(xv[i][2], xv[i][3], t0, t1, t2); h[1] = t0; m[1] = t1; l[1] = t2;
                    *reinterpret_cast<u32x2*>(dst) = h; *reinterpret_cast<u32x2*>(dst + xpart) = m; *reinterpret_cast<u32x2*>(dst + 2 * xpart) = l;
                } else {
                    const Split8 s = split8(xv[i]);
                    *reinterpret_cast<u32x4*>(dst) = s.h; *reinterpret_cast<u32x4*>(dst + xpart) = s.m; *reinterpret_cast<u32x4*>(dst + 2 * xpart) = s.l;
                }
            }
        }
    };
    auto store_w = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < IW; ++i) {
            if (i * NT >= TO * gq) break;
            const int item = i * NT + tid;
            const int o = fast_div(item, a.div_gq), ql = item - o * gq;
            if (o < TO) {
                char* const dst = ws + ql * WROW + o * 16;
                const Split8 s = split8(wv[i]);
                *reinterpret_cast<u32x4*>(dst) = s.h; *reinterpret_cast<u32x4*>(dst + wpart) = s.m; *reinterpret_cast<u32x4*>(dst + 2 * wpart) = s.l;
            }
        }
    };

    // ---- per-lane operand bases
    int xbase[RP], ybase[RP];    // byte offset of the pixel's window in X; offset of (n, o = 0, oh, ow) in y or -1
#pragma unroll
    for (int j = 0; j < RP; ++j) {
        const int m = m0 + (wave_p * RP + j) * 32 + r;
        const int mc = min(m, a.M - 1);
        const int n = fast_div(mc, a.div_ohw), rem = mc - n * a.OHW;
        const int oh = fast_div(rem, a.div_ow), ow = rem - oh * a.OW;
        xbase[j] = ((n * a.Hp + oh * a.sh - qmin) * a.Wp + ow * a.sw) * XB;
        ybase[j] = m < a.M ? n * a.O * a.OHW + rem : -1;
    }
    const int wbase = half * WROW + (wave_o * RO * 32 + r) * 16;

    f32x16 acc[RO][RP];
    f32x16 acc2[DS ? RO : 1][DS ? RP : 1];
#pragma unroll
    for (int i = 0; i < RO; ++i)
#pragma unroll
        for (int j = 0; j < RP; ++j)
#pragma unroll
            for (int g = 0; g < 16; ++g) {
                acc[i][j][g] = 0.0f;
                if constexpr (DS) acc2[i][j][g] = 0.0f;
            }

    load_x(c_lo);
    load_w(c_lo, 0);
    store_x();
    store_w();
    __syncthreads();
    int chunk = c_lo, group = 0;
    while (true) {
        const bool last_group = group + 1 >= a.ngroups;
        const int nchunk = last_group ? chunk + 1 : chunk, ngroup = last_group ? 0 : group + 1;
        const bool has_next = nchunk < c_hi;
        if (has_next) {
            if (last_group) load_x(nchunk);
            load_w(nchunk, ngroup);
        }
        __builtin_amdgcn_sched_barrier(0);
        // ---- this stage's k-steps; operands are read one step ahead
        const int first = group * a.group_steps, steps = min(a.group_steps, a.nq / 2 - first);
        u32x4 af[2][RO][3], bf[2][RP][3];
        auto fetch = [&](int s, int set) __attribute__((always_inline)) {
            const int xo = ktab[2 * (first + s) + half];
#pragma unroll
            for (int j = 0; j < RP; ++j)
#pragma unroll
                for (int p = 0; p < 3; ++p) {
                    const char* const at = xs + xbase[j] + xo + p * xpart;
                    if constexpr (C4) {
                        const u32x2 lo = *reinterpret_cast<const u32x2*>(at), hi = *reinterpret_cast<const u32x2*>(at + 8);
                        bf[set][j][p] = u32x4{lo[0], lo[1], hi[0], hi[1]};
                    } else {
                        bf[set][j][p] = *reinterpret_cast<const u32x4*>(at);
                    }
                }
            const char* const wt = ws + wbase + 2 * s * WROW;
#pragma unroll
            for (int i = 0; i < RO; ++i)
#pragma unroll
                for (int p = 0; p < 3; ++p) af[set][i][p] = *reinterpret_cast<const u32x4*>(wt + i * 512 + p * wpart);
        };
        auto multiply = [&](int s, int set) __attribute__((always_inline)) {
            if constexpr (DS) {
                if (first + s >= a.nq_main / 2) { mfma6<RO, RP>(acc2, af[set], bf[set]); return; }
            }
            mfma6<RO, RP>(acc, af[set], bf[set]);
        };
        if (kgroup < steps) {
            fetch(kgroup, 0);
            int s = kgroup;
            while (true) {
                if (s + KS < steps) fetch(s + KS, 1);
                __builtin_amdgcn_sched_barrier(0);
                multiply(s, 0);
                __builtin_amdgcn_sched_barrier(0);
                s += KS;
                if (s >= steps) break;
                if (s + KS < steps) fetch(s + KS, 0);
                __builtin_amdgcn_sched_barrier(0);
                multiply(s, 1);
                __builtin_amdgcn_sched_barrier(0);
                s += KS;
                if (s >= steps) break;
            }
        }
        __syncthreads();
        if (!has_next) break;
        if (last_group) store_x();
        store_w();
        __syncthreads();
        chunk = nchunk;
        group = ngroup;
    }

    // ---- combine the groups of waves: all but the first park their sums in LDS (the tiles are dead), the first adds them
    if constexpr (KS > 1) {
        float* const red = reinterpret_cast<float*>(lds);
        auto combine = [&](auto& s) __attribute__((always_inline)) {
            if (kgroup > 0) {
#pragma unroll
                for (int i = 0; i < RO; ++i)
#pragma unroll
                    for (int j = 0; j < RP; ++j)
#pragma unroll
                        for (int g = 0; g < 16; ++g) red[((((kgroup - 1) * NW + wave) * RO * RP + i * RP + j) * 16 + g) * 64 + lane] = s[i][j][g];
            }
            __syncthreads();
            if (kgroup == 0) {
#pragma unroll
                for (int kg = 1; kg < KS; ++kg)
#pragma unroll
                    for (int i = 0; i < RO; ++i)
#pragma unroll
                        for (int j = 0; j < RP; ++j)
#pragma unroll
                            for (int g = 0; g < 16; ++g) s[i][j][g] += red[((((kg - 1) * NW + wave) * RO * RP + i * RP + j) * 16 + g) * 64 + lane];
            }
        };
        combine(acc);
        if constexpr (DS) {
            __syncthreads();
            combine(acc2);
        }
        if (kgroup > 0) return;
    }

    // ---- epilogue: accumulator register g of a block holds row 8*(g/4) + 4*half + g%4, column r
    auto channel = [&](int i, int g) { return o0 + (wave_o * RO + i) * 32 + 8 * (g / 4) + 4 * half + (g % 4); };
    const bool has_bias = (a.flags & KXC_HIP_CONV_BIAS) != 0, has_res = (a.flags & KXC_HIP_CONV_RESIDUAL) != 0;
    const bool do_relu = (a.flags & KXC_HIP_CONV_RELU) != 0;
    float* const part = a.partial + static_cast<int64_t>(split) * a.out_elems;
    float* const part2 = part + static_cast<int64_t>(a.gsplit) * a.out_elems;      // the parts of a second output follow those of the first
    float odd = 0.0f;                                                              // NaN when a sum is not finite
#pragma unroll
    for (int i = 0; i < RO; ++i)
#pragma unroll
        for (int j = 0; j < RP; ++j)
#pragma unroll
            for (int g = 0; g < 16; ++g) {
                odd = __builtin_fmaf(acc[i][j][g], 0.0f, odd);
                if constexpr (DS) odd = __builtin_fmaf(acc2[i][j][g], 0.0f, odd);
            }
    if (__builtin_expect(__any(odd != odd), 0)) {
        // (channels of this part of a split reduction)
        const int cl = c_lo * a.cb * 8, ch = min(c_hi * a.cb * 8, a.C);
#pragma unroll 1
        for (int e = 0; e < RO * RP * 16; ++e) {
            const int i = e / (RP * 16), j = (e / 16) % RP, g = e % 16;
            const int o = channel(i, g);
            const int m = m0 + (wave_p * RP + j) * 32 + r;
            if (o >= a.O || m >= a.M) continue;
            const int n = fast_div(m, a.div_ohw), rem = m - n * a.OHW;
            const int oh = fast_div(rem, a.div_ow), ow = rem - oh * a.OW;
            const int64_t at = (static_cast<int64_t>(n) * a.O + o) * a.OHW + rem;
            const float* const xn = a.x + static_cast<int64_t>(n) * a.C * a.H * a.W;
            // (a filter one row high sees every row_step-th input row: sh is 1 then)
            const int ih0 = (oh * a.sh - a.ph) * a.row_step, iw0 = ow * a.sw - a.pw;
            float v = direct_sum(xn, a.w + static_cast<int64_t>(o) * a.C * KHW, a.C, a.H, a.W, a.KH, a.KW, cl, ch, ih0, iw0, a.dh, a.dw);
            if (a.gsplit > 1) {
                part[at] = v;
            } else {
                if (has_bias) v = __fadd_rn(v, a.bias[o]);
                if (has_res) v = __fadd_rn(v, a.res[at]);
                if (do_relu) v = relu_sel(v);
                a.y[at] = v;
            }
            if constexpr (DS) {
                float v2 = direct_sum(xn, a.w2 + static_cast<int64_t>(o) * a.C, a.C, a.H, a.W, 1, 1, cl, ch, oh * a.sh, ow * a.sw, 1, 1);
                if (a.gsplit > 1) part2[at] = v2;
                else a.y2[at] = a.bias2 ? __fadd_rn(v2, a.bias2[o]) : v2;
            }
        }
        return;
    }
    if (a.gsplit > 1) {
#pragma unroll
        for (int i = 0; i < RO; ++i)
#pragma unroll
            for (int g = 0; g < 16; ++g) {
                const int o = channel(i, g);
                if (o >= a.O) continue;
#pragma unroll
                for (int j = 0; j < RP; ++j)
                    if (ybase[j] >= 0) {
                        part[ybase[j] + o * a.OHW] = acc[i][j][g];
                        if constexpr (DS) part2[ybase[j] + o * a.OHW] = acc2[i][j][g];
                    }
            }
        return;
    }
    // (as in conv_mfma_kernel: buffer descriptors mask absent channels and pixels, every load precedes the first store; a
    // channel's plane offset rides in the scalar offset, the lane half's four channels in the vector offset)
    const uint32_t y_bytes = static_cast<uint32_t>(a.out_elems) * 4u, plane = static_cast<uint32_t>(a.OHW) * 4u;
    auto finish = [&](auto& s, const float* bias, const float* res, bool relu, float* y) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t yr = make_rsrc(y, y_bytes);
        const __amdgpu_buffer_rsrc_t rr = make_rsrc(res ? res : y, res ? y_bytes : 0u);
        const __amdgpu_buffer_rsrc_t br = make_rsrc(bias ? bias : y, bias ? static_cast<uint32_t>(a.O) * 4u : 0u);
        float bv[RO][16];
#pragma unroll
        for (int i = 0; i < RO; ++i)
#pragma unroll
            for (int g = 0; g < 16; ++g) {
                const int o = channel(i, g);
                bv[i][g] = bias ? ldf(br, o < a.O ? static_cast<uint32_t>(o) * 4u : kOobOffset, 0) : 0.0f;
            }
#pragma unroll
        for (int i = 0; i < RO; ++i) {
            const int ob = o0 + (wave_o * RO + i) * 32;                 // uniform
            const bool whole = ob + 32 <= a.O;
#pragma unroll
            for (int j = 0; j < RP; ++j) {
                const uint32_t yb = ybase[j] >= 0 ? (static_cast<uint32_t>(ybase[j]) + static_cast<uint32_t>(4 * half * a.OHW)) * 4u : kOobOffset;
                auto off = [&](int g) __attribute__((always_inline)) { return whole || channel(i, g) < a.O ? yb : kOobOffset; };
                auto so = [&](int g) __attribute__((always_inline)) { return static_cast<uint32_t>(ob + 8 * (g / 4) + g % 4) * plane; };
                float q[16];
                if (res) {
#pragma unroll
                    for (int g = 0; g < 16; ++g) q[g] = ldf(rr, off(g), so(g));
                }
#pragma unroll
                for (int g = 0; g < 16; ++g) {
                    float v = s[i][j][g];
                    if (bias) v = __fadd_rn(v, bv[i][g]);
                    if (res) v = __fadd_rn(v, q[g]);
                    if (relu) v = relu_sel(v);
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), yr, off(g), so(g), 0);
                }
            }
        }
    };
    finish(acc, has_bias ? a.bias : nullptr, has_res ? a.res : nullptr, do_relu, a.y);
    if constexpr (DS) finish(acc2, a.bias2, nullptr, false, a.y2);
}

#endif  // __HIPCC__

}  // namespace conv_bx
}  // namespace kxc_hip
