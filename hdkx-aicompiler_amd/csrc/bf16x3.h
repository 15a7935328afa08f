// bf16x3.h -- fp32 contractions on the bf16 matrix cores of gfx950 without giving up fp32's precision.
//
// The three-term split of Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations" (ARITH 2019).  An fp32 number has 24 significant bits, a bf16 number 8 and the same exponent
// range, so x = h + m + l with h = bf16(x), m = bf16(x - h), l = bf16(x - h - m): both subtractions are exact,
// |m| <= 2^-8 |x|, |l| <= 2^-17 |x|, and from |x| = 2^-109 on the three parts hold all 24 bits of x.  Below, the last bits lie
// under bf16's smallest step, 2^-133 (the matrix instructions take subnormal parts as they are), and h + m + l is off by
// at most 2^-134, which is all of an x of that size.  Multiplying operands by 2^16 while they are split, and sums by 2^-32,
// keeps those bits as well (every float times 2^16 is a whole number of such steps): the convolutions on a packed filter do it
// (conv_bf16x3.h, conv7_bf16x3.h), whose sums that are not finite, from 2^96 on, are formed again.  Not taken in products: 300 x
// 1000 x 2048 15.4 -> 16.6 us, 64 x 1000 x 512 4.7 -> 5.0 (with v_dot2_f32_bf16 in the place of each unpacking and subtraction,
// which is exact, 16.8 and 4.9), nor in a plan's Winograd layers, which have no second way to form a sum; KXC_HIP_GEMM_BF16X3=0
// and KXC_HIP_WINOGRAD_BF16X3=0 keep the fp32 instructions for callers whose operands are that small.
// A product of two such numbers is nine bf16 products, each exact in fp32; the three that are left out (m*l', l*m', l*l')
// add up to at most 2^-24 |x x'|, what rounding the product to fp32 may lose as well.  The six others are accumulated in
// fp32 by v_mfma_f32_32x32x16_bf16, smallest first.  Measured on random dot products of 64, 576 and 4608 terms against a
// float64 evaluation (relative error in the 2-norm): 1.1e-7 / 3.6e-7 / 1.1e-6, v_mfma_f32_32x32x2_f32 on the same data
// 1.4e-7 / 4.3e-7 / 1.2e-6; all nine products change nothing (what is left is the fp32 accumulation).
//
// Why: a bf16 matrix instruction does 16x the work of an fp32 one per cycle and runs beside the vector ALU (the fp32
// one shares its datapath), so six of them cost 6/16 of the fp32 instruction.  Measured in a loop of independent
// instructions on random data: 1 750 TFLOP/s = 290 TFLOP/s of fp32 products; the fp32 matrix peak is 157.
//
// An infinite or NaN operand gives NaN (inf - inf in the split), and so does one above 3.39e38 that rounds to an
// infinite bf16.  A kernel that has to spread them like the fp32 loop re-evaluates outputs that come out as NaN.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace kxc_hip {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

#if defined(__HIPCC__)

constexpr float kOperandScale = 65536.0f, kSumScale = 1.0f / (65536.0f * 65536.0f);      // for operands below 2^-109 (see above)

// Two floats -> two packed bf16, round to nearest even (one instruction on gfx950).
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ float bf16_lo(uint32_t p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t p) { return __builtin_bit_cast(float, p & 0xffff0000u); }

// The three parts of two floats, packed pairwise: 11 instructions for two values.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = pack_bf16(a, b);
    const float ra = __fsub_rn(a, bf16_lo(h)), rb = __fsub_rn(b, bf16_hi(h));
    m = pack_bf16(ra, rb);
    l = pack_bf16(__fsub_rn(ra, bf16_lo(m)), __fsub_rn(rb, bf16_hi(m)));
}

// Eight consecutive k values of one row or column as the three operand fragments a lane feeds to the matrix instruction.
struct Split8 {
    u32x4 h, m, l;
};
__device__ __forceinline__ Split8 split8(const float (&v)[8]) {
    Split8 s;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t h, m, l;
        split_pair(v[2 * q], v[2 * q + 1], h, m, l);
        s.h[q] = h; s.m[q] = m; s.l[q] = l;
    }
    return s;
}

__device__ __forceinline__ f32x16 mfma_bf16(u32x4 a, u32x4 b, f32x16 c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
#else
    return c;
#endif
}

// acc[i][j] += A_i B_j for RO x RP blocks of 32 x 32 over 16 k values; parts 0 / 1 / 2 = h / m / l.  The six products of
// a block are issued RO * RP instructions apart, so none waits for the one before it.
template <int RO, int RP>
__device__ __forceinline__ void mfma6(f32x16 (&acc)[RO][RP], const u32x4 (&a)[RO][3], const u32x4 (&b)[RP][3]) {
    constexpr int PA[6] = {1, 0, 2, 0, 1, 0}, PB[6] = {1, 2, 0, 1, 0, 0};
#pragma unroll
    for (int p = 0; p < 6; ++p)
#pragma unroll
        for (int i = 0; i < RO; ++i)
#pragma unroll
            for (int j = 0; j < RP; ++j) acc[i][j] = mfma_bf16(a[i][PA[p]], b[j][PB[p]], acc[i][j]);
}

// The 3x3 filters of 32 output channels x CHANNELS input channels (cn of them present) into LDS, rows of 9 * CHANNELS + 1
// floats, by 256 threads.  Every thread's loads are in flight together: a launch of few workgroups is one memory round trip
// (90 -> 150 channels: 11.7 us one load behind the other, 7.4 here; the thirteen layers of ResNet-18, which write 95 MB: 21.2, 20.1).
template <int CHANNELS>
__device__ __forceinline__ void stage_filters(const float* __restrict__ w, int32_t O, int32_t C, int o0, int c0, int cn, float* raw) {
    constexpr int RUN = CHANNELS * 9, N = 32 * RUN / 256;
    float v[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const int idx = k * 256 + static_cast<int>(threadIdx.x), ol = idx / RUN, r = idx - ol * RUN;
        const bool ok = o0 + ol < O && r < cn * 9;
        const float x = w[ok ? (static_cast<int64_t>(o0 + ol) * C + c0) * 9 + r : 0];
        v[k] = ok ? x : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const int idx = k * 256 + static_cast<int>(threadIdx.x), ol = idx / RUN;
        raw[ol * (RUN + 1) + idx - ol * RUN] = v[k];
    }
}

#endif  // __HIPCC__

}  // namespace kxc_hip
