// conv2d_bf16x3.hip -- a launch plan's 3x3 stride-2 convolutions, with or without the second (1x1) output, its 7x7 stride-2
// convolution of three-channel images, and large single calls of 1x1 to 7x7 filters on the bf16 matrix cores: which launches take
// the kernels of conv_bf16x3.h and conv7_bf16x3.h, and their launch.  The filter is read in packed form, written by the
// plan's filter launch (conv2d_wino_f32.hip) or by the call.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <memory>

#include "conv7_bf16x3.h"
#include "conv_bf16x3.h"
#include "conv_point.h"

using namespace kxc_hip;

namespace {

struct PackedLaunch {
    conv_bx::Args a;
    void (*kernel)(const conv_bx::Args) = nullptr;
    void (*pack)(const float*, char*, int32_t, int32_t) = nullptr;
    conv7_bx::Args a7;                                    // kernel7
    void (*kernel7)(const conv7_bx::Args) = nullptr;
    int threads7 = 0;
    bool whole7 = false;                                  // kernel7: tiles are whole rows of an image
    conv_pt::Args ap;                                     // kernel1
    void (*kernel1)(const conv_pt::Args) = nullptr;
    size_t lds_bytes = 0, filter_bytes = 0;
    double gflop = 0;
    const char* name = "";
    bool second = false;
    size_t scratch_bytes = 0;
};

// Parts of a reduction, while all of them together are at most one workgroup per compute unit: what gives the shortest of
// 0.29 us per tap and 16 channels + the adding launch (5 us and the parts' way to memory and back at 4.5 TB/s).  us, 1 / 2 / 4 / 8
// parts without the adding launch: 64 -> 128 channels at 49 x 49, batch 6 (59 workgroups) 19.9 / 14.8 / 12.9; 128 -> 256 at 25 x
// 25, batch 5 (28) 24.7 / 17.0 / 13.4 / 12.2; 256 -> 512 at 14 x 14, batch 32 (100) 47.5 / 30.8 / 34.2 / 41.9, batch 64 (196)
// 54.1 / 57.3 / 66.3; with it 64 -> 128 at 56 x 56, batch 8 (98) 22 and 28.
int Split(int64_t units, int csteps, int steps, int64_t out_bytes) {
    int best = 1;
    const double step_us = 0.29 * steps;
    double best_us = step_us * csteps;
    for (int s = 2; s <= 8 && units * s <= 256 && s <= csteps && out_bytes * s <= (16LL << 20); s *= 2) {
        const double us = step_us * static_cast<double>(CeilDiv(csteps, s)) + 5 + 2.0 * s * static_cast<double>(out_bytes) / 4.5e6;
        if (us < best_us) { best_us = us; best = s; }
    }
    return best;
}

struct FilterKernels {
    int k, s;
    void (*conv)(const conv_bx::Args);
    void (*pack)(const float*, char*, int32_t, int32_t);
    const char* name;
};
template <int K, int S>
__global__ void __launch_bounds__(256) pack_filter_kernel(const float* w, char* u, int32_t O, int32_t C) {
    __shared__ float raw[conv_bx::PackFloats(K)];
    conv_bx::pack_block<K, S>(w, nullptr, u, O, C, static_cast<int>(blockIdx.x), raw);
}
#define KXC_PACKED(K, S) {K, S, conv_bx::conv_bf16x3_kernel<K, S, false>, pack_filter_kernel<K, S>, "mfma_k" #K "x" #K "s" #S "_bf16x3"}
const FilterKernels kFilters[] = {KXC_PACKED(1, 1), KXC_PACKED(1, 2), KXC_PACKED(3, 1), KXC_PACKED(3, 2), KXC_PACKED(5, 1), KXC_PACKED(5, 2), KXC_PACKED(7, 1), KXC_PACKED(7, 2)};

// Whether the kernel covers a launch (`L` is filled if so).
bool Resolve(const kxc_hip_conv2d_desc* d, bool second, PackedLaunch* L) {
    using namespace conv_bx;
    if (!d || d->n <= 0 || d->c <= 0 || d->h <= 0 || d->w <= 0 || d->o <= 0 || d->kh != d->kw || d->stride_h != d->stride_w) return false;
    const int K = d->kh, S = d->stride_h;
    const FilterKernels* kernels = nullptr;
    for (const FilterKernels& k : kFilters)
        if (k.k == K && k.s == S) kernels = &k;
    if (!kernels || d->dil_h != 1 || d->dil_w != 1 || d->pad_h < 0 || d->pad_w < 0 || d->pad_h > 64 || d->pad_w > 64) return false;
    if (second && (K != 3 || S != 2 || d->pad_h != 1 || d->pad_w != 1)) return false;
    if (d->flags & (KXC_HIP_CONV_FORCE_DIRECT | KXC_HIP_CONV_HPOOL)) return false;
    const int64_t Hp = static_cast<int64_t>(d->h) + 2 * d->pad_h, Wp = static_cast<int64_t>(d->w) + 2 * d->pad_w;
    if (Hp < K || Wp < K) return false;
    const int64_t OH = (Hp - K) / S + 1, OW = (Wp - K) / S + 1;
    const int64_t x_bytes = 4LL * d->n * d->c * d->h * d->w, y_elems = static_cast<int64_t>(d->n) * d->o * OH * OW;
    const int64_t u_bytes = static_cast<int64_t>(FilterBytes(d->o, d->c, K, second));
    if (x_bytes >= (1LL << 31) || y_elems >= (1LL << 29) || u_bytes >= (1LL << 31) || (d->n + 1LL) * (OH + K) >= (1LL << 30)) return false;
    Args& a = L->a;
    std::memset(&a, 0, sizeof(a));
    a.N = d->n; a.C = d->c; a.H = d->h; a.W = d->w; a.O = d->o;
    a.OH = static_cast<int32_t>(OH); a.OW = static_cast<int32_t>(OW); a.OHW = a.OH * a.OW; a.HW = a.H * a.W;
    a.M = a.N * a.OHW;
    a.ph = d->pad_h; a.pw = d->pad_w;
    a.Hq = a.OH + (K - 1) / S;
    a.w4 = (a.W + 3) / 4;
    if (K > 1) {
        // (every call whose cost asks for the kernel comes here: wide maps go before the tiles are walked)
        if (a.W > 4 * kPlane || ((K - 1) / S + 1) * (a.OW + K - 1) > kPlane) return false;
        const int64_t rows = TileReach(a.N, a.OHW, a.OW, kPix, 1, a.Hq - a.OH) + (K - 1) / S + 1;
        if (2 * rows * a.w4 > 64 * kProducers * kUnits) return false;
        // Stride 2: even columns, odd ones behind them.  Where it fits, a row pitch that continues the banks of a row's last pixel
        // with the next row's first one (a lane reads 16 bytes: 16 positions go through all banks).
        a.hp = std::max(a.OW + (K - 1) / 2, (a.W - 1 + a.pw) / 2 + 1);
        a.pitch = S == 2 ? 2 * a.hp : std::max(a.OW + K - 1, a.W + a.pw);
        if (rows * a.pitch > kPlane) return false;
        const int32_t least = a.pitch;
        for (int32_t pitch = least; pitch < least + 16 && rows * pitch <= kPlane; ++pitch)
            if ((pitch - a.OW) % 16 == 0) { a.pitch = pitch; break; }
    }
    const int channels = kStep * ChannelSteps(K);
    a.csteps = static_cast<int32_t>(CeilDiv(a.C, channels));
    a.tail = a.C % channels != 0 ? 1 : 0;
    a.quads = S == 1 && a.ph == 0 && a.pw == 0 && a.HW % 4 == 0 ? 1 : 0;
    a.p_tiles = static_cast<int32_t>(CeilDiv(a.M, kPix));
    a.o_tiles = static_cast<int32_t>(CeilDiv(a.O, kOut));
    const int64_t units = static_cast<int64_t>(a.p_tiles) * a.o_tiles;
    if (units >= (1LL << 27)) return false;
    a.num_units = static_cast<int32_t>(units);
    a.x_bytes = static_cast<uint32_t>(x_bytes);
    a.u_bytes = static_cast<uint32_t>(u_bytes);
    a.flags = d->flags;
    const int64_t out_bytes = y_elems * 4 * (second ? 2 : 1);
    const int split = Split(units * SelectLanes(), a.csteps, Steps(K, second), out_bytes);
    a.cps = static_cast<int32_t>(CeilDiv(a.csteps, split));
    a.gsplit = static_cast<int32_t>(CeilDiv(a.csteps, a.cps));      // no empty part
    if (a.gsplit > 1) L->scratch_bytes = static_cast<size_t>(a.gsplit) * out_bytes;
    a.units_per_xcd = static_cast<int32_t>(CeilDiv(units * a.gsplit, 8));
    a.o_fastest = u_bytes <= (2 << 20) ? 1 : 0;      // an XCD's run of workgroups shares its input while the filters stay in the L2
    a.div_ohw = MakeFastDiv(a.OHW); a.div_ow = MakeFastDiv(a.OW); a.div_hq = MakeFastDiv(a.Hq); a.div_w4 = MakeFastDiv(a.w4);
    a.div_tiles = MakeFastDiv(a.o_fastest ? a.o_tiles : a.p_tiles); a.div_gsplit = MakeFastDiv(a.gsplit);
    L->second = second;
    L->filter_bytes = a.u_bytes;
    L->lds_bytes = LdsBytes(K);
    L->gflop = 2e-9 * a.M * a.O * a.C * (K * K + (second ? 1 : 0));
    L->kernel = second ? conv_bf16x3_kernel<3, 2, true> : kernels->conv;
    L->pack = kernels->pack;
    L->name = second ? "mfma_k3x3s2_bf16x3_ds" : kernels->name;
    return true;
}

// The same for the 7x7 kernel.  LDS for two workgroups (four waves) per compute unit at least.
bool Resolve7(const kxc_hip_conv2d_desc* d, PackedLaunch* L) {
    using namespace conv7_bx;
    if (!d || d->n <= 0 || d->c != kC || d->h <= 0 || d->w <= 0 || d->o <= 0) return false;
    if (d->kh != kK || d->kw != kK || d->stride_h != 2 || d->stride_w != 2 || d->dil_h != 1 || d->dil_w != 1) return false;
    if (d->pad_h < 0 || d->pad_w < 0 || d->pad_h >= kK || d->pad_w >= kK || d->w < 2 || (d->flags & KXC_HIP_CONV_FORCE_DIRECT)) return false;
    const int64_t Hp = static_cast<int64_t>(d->h) + 2 * d->pad_h, Wp = static_cast<int64_t>(d->w) + 2 * d->pad_w;
    if (Hp < kK || Wp < kK) return false;
    const int64_t OH = (Hp - kK) / 2 + 1, OW = (Wp - kK) / 2 + 1;
    const bool hpool = (d->flags & KXC_HIP_CONV_HPOOL) != 0;
    const int64_t M = d->n * OH * OW, y_elems = static_cast<int64_t>(d->n) * d->o * OH * (hpool ? OW / 2 : OW);
    if (4LL * d->n * kC * d->h * d->w >= (1LL << 31) || static_cast<int64_t>(d->n) * d->o * OH * OW >= (1LL << 29) || d->o > (1 << 16)) return false;
    if ((d->n + 1) * Hp >= (1LL << 30)) return false;
    if (hpool && (!(d->flags & KXC_HIP_CONV_RELU) || (d->flags & KXC_HIP_CONV_RESIDUAL) || d->o % 8 != 0 || (OW & 1) || kPix % OW != 0 || M % kPix != 0)) return false;
    Args& a = L->a7;
    std::memset(&a, 0, sizeof(a));
    a.N = d->n; a.H = d->h; a.W = d->w; a.O = d->o; a.OH = static_cast<int32_t>(OH); a.OW = static_cast<int32_t>(OW);
    a.OHW = a.OH * a.OW; a.HW = a.H * a.W; a.M = static_cast<int32_t>(M); a.ph = d->pad_h; a.pw = d->pad_w;
    a.Hp = static_cast<int32_t>(Hp); a.PW = a.OW / 2;
    const int pitch = OW + 3 <= 64 ? 64 : 120;      // (the last pixel's window takes four words; three parts within the reach of a ds_read2)
    if (OW + 3 > pitch) return false;
    int64_t rows = conv_bx::TileReach(a.N, a.OHW, a.OW, kPix, 2, a.Hp - 2 * a.OH) + kK, tiles = CeilDiv(M, kPix);
    a.tile_pix = kPix; a.span = a.M;
    if (!hpool && LdsBytes(rows, pitch) > kMaxLdsBytes / 4) {
        // Whole rows of an image: fewer rows of input, of which four workgroups find room in LDS.
        L->whole7 = true;
        int64_t high = std::min<int64_t>(kPix / OW, OH);
        while (high > 1 && LdsBytes(2 * high + kK - 2, pitch) > kMaxLdsBytes / 4) --high;
        tiles = CeilDiv(OH, high);
        high = CeilDiv(OH, tiles);
        rows = 2 * high + kK - 2;
        a.tile_pix = static_cast<int32_t>(high * OW); a.span = a.OHW;
    }
    a.tiles = static_cast<int32_t>(tiles);
    a.row_max = static_cast<int32_t>(rows);
    if (LdsBytes(rows, pitch) > kMaxLdsBytes / 2) return false;
    a.o_tiles = static_cast<int32_t>(CeilDiv(a.O, kOut));
    const int64_t units = tiles * (a.span == a.M ? 1 : a.N) * a.o_tiles;
    if (units >= (1LL << 30)) return false;
    a.num_units = static_cast<int32_t>(units);
    a.units_per_xcd = static_cast<int32_t>(CeilDiv(units, 8));
    a.x_bytes = static_cast<uint32_t>(4LL * d->n * kC * d->h * d->w);
    a.y_bytes = static_cast<uint32_t>(y_elems * 4);
    a.u_bytes = static_cast<uint32_t>(FilterBytes(a.O));
    a.flags = d->flags;
    a.div_ohw = MakeFastDiv(a.OHW); a.div_ow = MakeFastDiv(a.OW); a.div_hp = MakeFastDiv(a.Hp); a.div_otiles = MakeFastDiv(a.o_tiles);
    a.div_tiles = MakeFastDiv(a.tiles);
    L->filter_bytes = a.u_bytes;
    L->lds_bytes = std::max(LdsBytes(rows, pitch), kMinLdsBytes);
    L->gflop = 2e-9 * static_cast<double>(M) * a.O * kC * kK * kK;
    static void (*const kWhole[2][2])(const Args) = {{conv7_bf16x3_kernel<64, false, 3, 2>, conv7_bf16x3_kernel<64, false, 4, 2>},
                                                     {conv7_bf16x3_kernel<120, false, 3, 2>, conv7_bf16x3_kernel<120, false, 4, 2>}};
    L->kernel7 = hpool ? (pitch == 64 ? conv7_bf16x3_kernel<64, true, 7, 1> : conv7_bf16x3_kernel<120, true, 7, 1>) : kWhole[pitch != 64][a.tile_pix > 192];
    L->threads7 = hpool ? kThreads : 2 * kThreads;
    L->name = "mfma_k7x7s2_bf16x3";
    return true;
}

// conv_point.h: workgroups that share a tile of pixels.  As many as give 384 workgroups, each with a block for every wave (us, 1 / 2 / 4 groups:
// 128 -> 512 channels at 28 x 28, batch 32, 392 tiles, 34.1 / 37.3 / 39.8, batch 8, 98 tiles, 22.5 / 16.2 / 14.7; 128 -> 1024 at 14 x 14,
// batch 64, 196 tiles, 43.1 / 34.6 / 38.5), and at most 64 blocks to one: their biases lie in LDS, which two workgroups share.
int64_t PointGroups(int64_t tiles, int64_t all) {
    return std::max(CeilDiv(all, conv_pt::kMaxBlocks), std::min(CeilDiv(384, tiles), all / conv_pt::kWaves));
}

// The same for the 1x1 kernel that keeps a workgroup's pixels (after Resolve).
void ResolvePoint(const kxc_hip_conv2d_desc* d, PackedLaunch* L) {
    using namespace conv_pt;
    if (d->kh != 1 || d->stride_h != 1 || d->pad_h != 0 || d->pad_w != 0 || d->c > 16 * kMaxSteps || L->a.HW % 4 != 0) return;
    Args& a = L->ap;
    std::memset(&a, 0, sizeof(a));
    a.C = d->c; a.O = d->o; a.HW = L->a.HW; a.M = L->a.M;
    a.csteps = L->a.csteps;
    const int64_t all = CeilDiv(a.O, 32), tiles = CeilDiv(a.M, kPix);
    a.blocks = static_cast<int32_t>(CeilDiv(all, PointGroups(tiles, all)));
    a.groups = static_cast<int32_t>(CeilDiv(all, a.blocks));
    a.num_units = static_cast<int32_t>(tiles * a.groups);
    a.units_per_xcd = static_cast<int32_t>(CeilDiv(a.num_units, 8));
    a.x_bytes = L->a.x_bytes; a.u_bytes = L->a.u_bytes; a.flags = d->flags;
    a.y_bytes = static_cast<uint32_t>(a.M) * static_cast<uint32_t>(a.O) * 4u;
    a.div_hw = MakeFastDiv(a.HW); a.div_groups = MakeFastDiv(a.groups);
    const int steps = d->c <= 64 ? 4 : 8;
    L->kernel1 = steps == 4 ? conv_point_kernel<4> : conv_point_kernel<8>;
    L->lds_bytes = LdsBytes(steps, a.blocks);
    L->scratch_bytes = 0;
}

// Whether to take a kernel that the rule for its launch does or does not ask for.  KXC_HIP_CONV_BF16X3=1: wherever it covers the launch,
// =0: nowhere.  KXC_HIP_WINOGRAD_BF16X3=0 keeps every convolution on the fp32 instructions, as it did when no other kernel had
// three-part operands.
bool Switched(bool by_rule) {
    const char* e = std::getenv("KXC_HIP_CONV_BF16X3");
    if (e && (e[0] == '0' || e[0] == '1')) return e[0] == '1';
    if (!by_rule) return false;
    const char* w = std::getenv("KXC_HIP_WINOGRAD_BF16X3");
    return !(w && w[0] == '0');
}

// Switches that name one of the other kernels or say in how many parts it splits its reduction keep those.
bool OthersForced() {
    for (const char* name : {"KXC_HIP_CONV_VARIANT", "KXC_HIP_CONV_HPOOL_VARIANT"}) {
        const char* variant = std::getenv(name);
        if (variant && *variant) return true;
    }
    return std::getenv("KXC_HIP_CONV_GSPLIT") != nullptr;
}

// us of the launches but `fixed`: workgroups of `start` + `step` per step, `second` times that where two share a compute unit, and
// the adding launch.
double PackedUs(double fixed, double start, double step, double second, int64_t groups, int64_t steps, int split, double out_bytes) {
    const double load = groups <= 256 ? 1.0 : second * std::max(1.0, static_cast<double>(groups) / 512);
    return fixed + (start + step * static_cast<double>(steps)) * load + (split > 1 ? 5 + 2.0 * split * out_bytes / 4.5e6 : 0);
}

// GFLOP of the other kernels, whose blocks of outputs are `block` x `block`.
double BlockGflop(const kxc_hip_conv2d_desc* d, int64_t pixels, int taps, int block) {
    return 2e-9 * static_cast<double>(CeilDiv(pixels, block) * block) * static_cast<double>(CeilDiv(d->o, block) * block) * d->c * taps;
}

// Whether a plan's node should take it: with fewer than 64 channels from 0.12 GFLOP per step of 16 on, counting the launches
// expected side by side.  A workgroup takes 9 us and 2.9 per step however few there are, and the other kernels start with 16 x 16 tiles and
// split reductions inside a workgroup (us, theirs and here, both outputs): 64 -> 128 channels at 56 x 56, batch 2 (0.26 GFLOP)
// 12.3 and 16.4, batch 4 (0.51) 23.1 and 20.2, batch 8 32.4 and 20.9, batch 32 59 and 36, batch 64 97 and 60; 128 -> 256 at 28 x 28, batch 6
// (0.77) 20.5 and 22.1, batch 8 (1.03) 25.5 and 23.7, batch 16 39 and 31, batch 64 94 and 54; 256 -> 512 at 14 x 14, batch 8 (1.03)
// 21.8 and 22.8, batch 12 (1.54) 31 and 25, batch 32 71 and 37, batch 64 104 and 52; 512 -> 512 at 14 x 14, batch 5 (1.28) 21.5 and 22.6; 512 ->
// 1024 at 28 x 28, batch 2 68 and 36; 16 -> 32 at 56 x 56, batch 20 (0.16) 15.0 and 11.5.  From 64 channels on the small-launch
// kernel with one load per filter row is the other side, up to 2.3 million (16 x 16 tiles) * k (1.3 GFLOP): 64 -> 128 at 56 x 56, batch 6 / 8 / 10 15.7 /
// 19.0 / 22.9 and 22.8 / 23.1 / 23.3; 128 -> 256 at 28 x 28, batch 8 / 10 18.6 / 20.7 and 24.7 / 25.9; 256 -> 512 at 14 x 14 18.9 / 19.1 and 23.5 / 23.2.
// The 7x7 kernel, 3 -> 64 channels: pooled at 224 x 224, batch 16 / 32 / 64 51 / 100 / 169 and 29 / 50 / 93, at 64 x 64, batch 56 (1.1 GFLOP) 33 and
// 22.  Pooled, with a compute unit to each workgroup and tiles of many rows it loses to the others' tile of 224
// pixels (3 -> 64 at 30 x 56, batch 24 18.9 and 21.0; from 257 workgroups on 24 channels at 304 x 56, batch 17 29.6 and 27.8), not to the one of 448 that they
// take where it fits (31.5 and 20.5 at 56 x 56, batch 8).  Not pooled, on tiles that are whole rows: batch 1 / 6 / 16 at 193 x 193 10.7 / 21.4 / 45 and
// 10.3 / 17.5 / 30, batch 47 at 189 x 189 107 and 57, batch 8 at 99 x 99 13.1 and 10.7, and batch 36 at 216 x 216 2312 and 60: rows of 105, 108 or 113 to
// 117 pixels fit none of the others' tiles.  Of 420 such layers 392 are faster, of those from 48 channels on (1.4 times) three slower by more than 3 %, a tenth at most;
// up to 32 channels leave half of a workgroup's 64 empty and need wide rows and three workgroups to a compute unit (32 at 145 x 108, batch 16 13.5 and
// 16.8, 208 x 208, batch 12 21.5 and 23.1, batch 32 at 213 x 213 54.8 and 48.5).  Not pooled, on rows that fill tiles (224 x 224, batch 8 (1.9 GFLOP) 33 and
// 26, batch 64 184 and 103) it begins at 1.8 GFLOP.  That is no line of speed (batch 4 20.3 and 13): the tests of this selection name such nodes; up to 32 channels at 1800
// workgroups (32 at 144 x 112, batch 57 36.6 and 44.0, 224 x 224, batch 33 63.7 and 61.6).
// At 3x3 that must also be the shorter time by what either side takes, fitted within a tenth to 1000 shapes of 16 to 512 and 8 to 512 channels: here
// 2 us and a workgroup's 4 + 0.28 per tap and step, the others 10.5 and 12.7 per GFLOP of 32 x 32 blocks or, by the small-launch kernels, 4.9
// and 12.4 of 16 x 16 ones.  A workgroup has 128 output channels: no more than 48 of them (256 -> 8 at 60 x 38, batch 38 24.5 and 99.4, 384 ->
// 16 at 32 x 31, batch 43 34 and 61, 384 -> 48 at 21 x 45, batch 30 41.6 and 50.5) and a reduction of one step (16 -> 32 at 46 x 51, batch 59 15.3
// and 24.6, 16 -> 72 at 82 x 58, batch 15 12.9 and 14.8) are never worth it.  384 -> 64 at 13 x 56, batch 18 25.8 and 33.7, 512 -> 160 at 8 x
// 38, batch 14 23.9 and 36.2.  Of 237 of these shapes that are taken four are slower by more than 3 % (at most 16), of 322 by the first
// line alone 51 (up to four times).
bool Preferred(const kxc_hip_conv2d_desc* d, bool second, PackedLaunch* L) {
    if (OthersForced()) return false;
    if (!second && Resolve7(d, L)) {
        // Tiles that are few rows high: four workgroups to a compute unit, and one batch of loads.
        const bool pooled = (d->flags & KXC_HIP_CONV_HPOOL) != 0, low = L->lds_bytes <= kMaxLdsBytes / 4;
        const int64_t lanes = SelectLanes(), units = L->a7.num_units * lanes;
        const bool plain = L->whole7 ? d->o > 32 || (L->a7.OW > 61 && units >= 768) : L->gflop * lanes >= 1.8 && (d->o > 32 || units >= 1800);
        return Switched(pooled ? low || units > 256 || HpoolTilePixels(d) > conv7_bx::kPix : low && plain);
    }
    // (a plan's filter launch packs 3x3 stride-2 filters only)
    if (!d || d->kh != 3 || d->stride_h != 2 || d->pad_h != 1 || d->pad_w != 1 || d->c % conv_bx::kStep != 0 || !Resolve(d, second, L)) return false;
    auto rule = [&]() {
        const int64_t lanes = SelectLanes();
        if (d->o <= 48 || d->c <= conv_bx::kStep) return false;
        if (d->c >= 64 && d->w >= 3 ? CeilDiv(L->a.M, 16) * CeilDiv(d->o, 16) * lanes * d->c * 9 <= kSmallRowLoadsWork
                                    : L->gflop * lanes < std::min(0.12 * L->a.csteps, 1.4)) return false;
        const int taps = second ? 10 : 9;
        const double out_bytes = 4.0 * L->a.M * d->o * (second ? 2 : 1);
        const bool small = SmallConvTakes(d, second, true);
        const double others = small ? 4.9 + 12.4 * lanes * BlockGflop(d, L->a.M, taps, 16) : 10.5 + 12.7 * lanes * BlockGflop(d, L->a.M, taps, 32);
        return PackedUs(2, 4, 0.28, 2, lanes * L->a.num_units * L->a.gsplit, static_cast<int64_t>(taps) * L->a.cps, L->a.gsplit, out_bytes) < others;
    };
    return Switched(rule());
}

// `partials`: room for the partial outputs of a split reduction; nullptr: it is acquired here.
int32_t LaunchConv(const PackedLaunch& L, const float* x, const float* w, const void* u, const float* bias, const float* residual, float* y,
                   const float* w2, const float* bias2, float* y2, hipStream_t s, float* partials) {
    if (L.kernel1) {
        conv_pt::Args b = L.ap;
        b.x = x; b.w = w; b.u = static_cast<const char*>(u); b.bias = bias; b.res = residual; b.y = y;
        if (L.lds_bytes > 64 * 1024)
            if (int32_t rc = GrantLds(reinterpret_cast<const void*>(L.kernel1))) return rc;
        hipLaunchKernelGGL(L.kernel1, NoteGrid(dim3(static_cast<unsigned>(b.units_per_xcd * 8))), NoteBlock(dim3(conv_pt::kThreads)), NoteLds(L.lds_bytes), s, b);
        return CheckLaunch(L.name);
    }
    conv_bx::Args a = L.a;
    a.x = x; a.w = w; a.u = static_cast<const char*>(u); a.bias = bias; a.res = residual; a.y = y;
    a.w2 = w2; a.bias2 = bias2; a.y2 = y2;
    SplitScratchLease lease;      // held until the adding kernel is enqueued
    if (a.gsplit > 1) {
        bool split = partials != nullptr;
        a.partial = partials;
        if (!partials) {
            if (int32_t rc = AcquireSplitScratch(s, L.scratch_bytes, &lease, &split)) return rc;
            a.partial = lease.ptr;
        }
        if (!split) {             // no buffer to be had: the reduction in one piece
            a.gsplit = 1;
            a.cps = a.csteps;
            a.div_gsplit = MakeFastDiv(1);
            a.units_per_xcd = static_cast<int32_t>(CeilDiv(a.num_units, 8));
        }
    }
    if (L.lds_bytes > 64 * 1024)
        if (int32_t rc = GrantLds(reinterpret_cast<const void*>(L.kernel))) return rc;
    hipLaunchKernelGGL(L.kernel, NoteGrid(dim3(static_cast<unsigned>(a.units_per_xcd * 8))), NoteBlock(dim3(conv_bx::kThreads)),
                       NoteLds(L.lds_bytes), s, a);
    if (int32_t rc = CheckLaunch(L.name)) return rc;
    if (a.gsplit == 1) return KXC_HIP_OK;
    SplitReduceArgs r;
    r.partial = a.partial; r.bias = bias; r.res = residual; r.y = y;
    r.total = a.M * a.O; r.gsplit = a.gsplit; r.O = a.O; r.flags = a.flags; r.div_ohw = a.div_ohw;
    if (L.second) {
        r.partial2 = a.partial + static_cast<int64_t>(a.gsplit) * r.total;
        r.bias2 = bias2; r.y2 = y2; r.flags2 = bias2 ? KXC_HIP_CONV_BIAS : 0u;
    }
    return LaunchSplitReduce(s, r);
}

// Whether a 1x1 call of at most 128 channels should take conv_point.h: a twentieth shorter by the estimates, which are fitted to 420 calls of 0.01
// to 4 GFLOP within 8 % here, 9 % (small-launch kernel) and a quarter (the others: whole tiles of 128 channels; below 32 the direct kernel).
// 126 of them take it and run 1.37 times as fast, eight slower (23.3 us against 19.4 for 112 -> 48 at 53 x 96, batch 14, the furthest); 27
// others would have gained a tenth.
bool PointRule(const kxc_hip_conv2d_desc* d, int64_t pixels, int64_t lanes, double blocks, double memory) {
    const int64_t all = CeilDiv(d->o, 32), tiles = CeilDiv(pixels, conv_pt::kPix);
    const int64_t own = CeilDiv(all, PointGroups(tiles, all)), units = tiles * CeilDiv(all, own) * lanes;
    const double walk = 0.44 + (d->c <= 64 ? 1.86 : 2.77) * static_cast<double>(CeilDiv(own, conv_pt::kWaves));
    const double here = 6.5 + 0.71 * memory + walk * std::max(1.0, static_cast<double>(units) / 512), m = 2e-9 * static_cast<double>(lanes * pixels);
    const double others = SmallConvTakes(d, false, false) ? 3.3 + 8.5 * blocks + 1.06 * memory
                          : d->o < 32 ? 480 * m * d->o * d->c : 8.7 + 18.7 * m * (CeilDiv(d->o, 128) * 128) * (CeilDiv(d->c, 16) * 16) + 0.46 * memory;
    return here < 0.95 * others;
}

// Whether a single call, which packs its filter first, should take the kernel: a twentieth shorter than the others, by what both
// sides take, fitted to 500 calls of 0.05 to 4 GFLOP within 5 % here and a tenth there.  Here by filter: two launches, a workgroup's start and its steps
// (a 1x1 filter's few steps do not hide the bytes, from caches mostly).  The others: GFLOP of whole blocks, at 1x1 the bytes as well; the
// small-launch kernels take smaller blocks.  Of 1x1 calls 35 of 160 take it and none is slower by more than 3 %, 7x7 20 of 80 and none, 5x5 25 of
// 153 and one (11 -> 329 at 65 x 37, stride 2, batch 18 28.5 and 34.6), 3x3 11 of 107 and two (up to 9 %).  us, theirs and here: 5x5, 64 -> 96 channels at 27 x 27, batch 8 38.4 and 25.4; 7x7,
// 226 -> 161 at 26 x 33 72 and 44; 13 -> 356 at 64 x 12, batch 4 31.9 and 24.7; 3x3, 220 -> 260 at 9 x 10, batch 27 47.9 and 35.1; 1x1, 128 -> 512 at
// 28 x 28, batch 32 73.6 and 50.2.  Not taken: 5x5, 32 -> 32 at 19 x 12, batch 37 16.0 and 21.2; 6 -> 126 at 60 x 48, batch 11 18.4 and 26.6; 7x7, 64 ->
// 96 at 15 x 16 17.9 and 25.2; 3x3, 16 -> 144 at 90 x 9, batch 11 12.0 and 16.5; 32 -> 208 at 100 x 31, batch 3 18.2 and 22.4; 1x1, 120 -> 35 at 14 x 48,
// batch 2 6.4 and 10.8; 400 -> 448 at 22 x 78, batch 3 26.6 and 30.8; images of no whole 16 bytes, whose pixels come one by one, 160 ->
// 400 at 37 x 23, batch 7 17.5 and 29.6.
bool OperatorRule(const kxc_hip_conv2d_desc* d) {
    using namespace conv_bx;
    const int K = d->kh, S = d->stride_h;
    // (3x3, stride 2: single calls agree with the outputs of kxc_hip_conv2d_pair_nchw_f32, which packs nothing.  Stride 1: Winograd
    // takes large ones; half of a block of 128 output channels empty is no gain)
    if (K == 3 && (S == 2 || d->o < 96)) return false;
    const int64_t oh = (static_cast<int64_t>(d->h) + 2 * d->pad_h - K) / S + 1, ow = (static_cast<int64_t>(d->w) + 2 * d->pad_w - K) / S + 1;
    if (oh <= 0 || ow <= 0) return false;
    if (K == 1 && (S != 1 || d->pad_h != 0 || d->pad_w != 0 || static_cast<int64_t>(d->h) * d->w % 4 != 0)) return false;
    const double pixels_d = static_cast<double>(d->n) * oh * ow, out_bytes = 4.0 * pixels_d * d->o;
    if (pixels_d >= 1e9 || out_bytes >= 1e10) return false;
    const int64_t pixels = static_cast<int64_t>(pixels_d), lanes = SelectLanes();
    const double memory = lanes * (4.0 * d->n * d->c * d->h * d->w + out_bytes * ((d->flags & KXC_HIP_CONV_RESIDUAL) ? 2 : 1)) / 4.5e6;
    const double blocks = lanes * BlockGflop(d, pixels, K * K, 32);
    if (K == 1 && d->c <= 16 * conv_pt::kMaxSteps) return PointRule(d, pixels, lanes, blocks, memory);
    const int64_t units = CeilDiv(pixels, kPix) * CeilDiv(d->o, kOut);
    const int csteps = static_cast<int>(CeilDiv(d->c, kStep * ChannelSteps(K))), steps = Steps(K, false);
    const int split = Split(units * lanes, csteps, steps, static_cast<int64_t>(out_bytes));
    const int64_t groups = units * split * lanes, own = static_cast<int64_t>(steps) * CeilDiv(csteps, split);
    const double here = K == 1 ? PackedUs(6.7 + 0.35 * memory, 1.7, 0.29, 2.16, groups, own, split, out_bytes)
                        : K == 3 ? PackedUs(7, 2, 0.25, 2.6, groups, own, split, out_bytes)
                        : K == 5 ? PackedUs(4.6, 5.7, 0.205, 1.9, groups, own, split, out_bytes) : PackedUs(2.3, 8.8, 0.213, 1.9, groups, own, split, out_bytes);
    double others = K == 1 ? 9 + 17.5 * blocks + 0.33 * memory : K == 3 ? 7.5 + 10.5 * lanes * BlockGflop(d, pixels, 9, 16)
                    : K == 5 ? 10.5 + 10.9 * blocks : 12.5 + 11.5 * blocks;
    if (here >= 0.95 * others || K > 3 || !SmallConvTakes(d, false, false)) return here < 0.95 * others;
    others = K == 1 ? 3.3 + 7.7 * blocks + 0.96 * memory : 4.4 + 11.2 * lanes * BlockGflop(d, pixels, 9, 16);
    return here < 0.95 * others;
}

// (Every single call asks: from the shape alone first, then the environment, then whether the kernel covers it.)
bool OperatorPreferred(const kxc_hip_conv2d_desc* d, PackedLaunch* L) {
    const int K = d->kh, S = d->stride_h;
    if (K != d->kw || S != d->stride_w || d->n <= 0 || d->c <= 0 || d->o <= 0 || (S != 1 && S != 2) || K > 7) return false;
    if (!(Switched(OperatorRule(d)) && !OthersForced() && Resolve(d, false, L) && L->filter_bytes <= (32u << 20))) return false;      // (bounds the scratch kept per stream)
    ResolvePoint(d, L);
    return true;
}

}  // namespace

namespace kxc_hip {

const char* PackedOperatorName(const kxc_hip_conv2d_desc* desc) {
    PackedLaunch L;
    return desc && OperatorPreferred(desc, &L) ? L.name : nullptr;
}

int32_t RunPackedOperator(const kxc_hip_conv2d_desc* desc, const float* x, const float* w, const float* bias, const float* residual, float* y,
                          hipStream_t stream, bool* launched, bool* preferred) {
    const char* const who = "kxc_hip_conv2d_nchw_f32";
    *launched = false;
    PackedLaunch L;
    *preferred = OperatorPreferred(desc, &L);
    // (kernels meet in the scratch: one packs the filter, the convolution reads it, and its parts are added)
    if (!*preferred || !StreamOrdersScratch(stream)) return KXC_HIP_OK;
    KXC_HIP_REQUIRE(x && w && y, "%s: NULL pointer", who);
    KXC_HIP_REQUIRE(!(desc->flags & KXC_HIP_CONV_BIAS) || bias, "%s: bias flag without bias", who);
    KXC_HIP_REQUIRE(!(desc->flags & KXC_HIP_CONV_RESIDUAL) || residual, "%s: residual flag without residual", who);
    SplitScratchLease lease;      // held until the last kernel that reads the scratch is enqueued
    const size_t filter = (L.filter_bytes + 255) / 256 * 256;
    if (int32_t rc = AcquireSplitScratch(stream, filter + L.scratch_bytes, &lease, launched)) return rc;
    if (!*launched) return KXC_HIP_OK;
    // (the filter is packed by every call: the caller may have changed it)
    char* const u = reinterpret_cast<char*>(lease.ptr);
    hipLaunchKernelGGL(L.pack, NoteGrid(dim3(static_cast<unsigned>(conv_bx::PackBlocks(desc->o, desc->c, desc->kh)))), NoteBlock(dim3(256)), NoteLds(0), stream,
                       w, u, static_cast<int32_t>(desc->o), static_cast<int32_t>(desc->c));
    if (int32_t rc = CheckLaunch("pack_filter_kernel")) return rc;
    return LaunchConv(L, x, w, u, bias, residual, y, nullptr, nullptr, nullptr, stream, reinterpret_cast<float*>(u + filter));
}

// Fitted to 1320 shapes, within a tenth (packed kernel), 13 % (small-launch kernels) and 17 % (rms).
double PairNodeUs(const kxc_hip_conv2d_desc* d) {
    PackedLaunch L;
    const int64_t lanes = SelectLanes();
    if (d->c < 64 || d->kh != 3 || d->kw != 3 || d->stride_h != 2 || d->stride_w != 2) return 0;
    if (Preferred(d, true, &L)) {
        const double out_bytes = 8.0 * L.a.M * d->o;
        return 9.7 + 0.74 * PackedUs(2, 4, 0.28, 2, lanes * L.a.num_units * L.a.gsplit, 10LL * L.a.cps, L.a.gsplit, out_bytes);
    }
    const int64_t pixels = d->n * ((static_cast<int64_t>(d->h) + 2 * d->pad_h - 3) / 2 + 1) * ((static_cast<int64_t>(d->w) + 2 * d->pad_w - 3) / 2 + 1);
    if (pixels <= 0 || pixels >= (1LL << 31)) return 0;
    if (!SmallConvTakes(d, true, true)) return 10.5 + 12.7 * static_cast<double>(lanes) * BlockGflop(d, pixels, 10, 32);
    return SmallConvStagesRows(d, true) ? 0 : 4.9 + 13.4 * static_cast<double>(lanes) * BlockGflop(d, pixels, 10, 16);
}

struct PreparedPacked {
    PackedLaunch launch;
    PreparedSlicePtr slice;      // the launch, where it is set
};

size_t PackedFilterBytes(const kxc_hip_conv2d_desc* desc, bool second) {
    PackedLaunch L;
    if (const size_t bytes = desc && desc->stride_h == 2 ? SliceFilterBytes(desc, second) : 0) return bytes;
    return Preferred(desc, second, &L) ? L.filter_bytes : 0;
}

void PreparePacked(const kxc_hip_conv2d_desc* desc, bool second, size_t u_bytes, PreparedPacked** out) {
    std::unique_ptr<PreparedPacked> p(new PreparedPacked);
    if (desc->stride_h == 2) p->slice.reset(PrepareSlice(desc, second, u_bytes));
    if (p->slice) {
        *out = p.release();
        return;
    }
    *out = Preferred(desc, second, &p->launch) && u_bytes >= p->launch.filter_bytes ? p.release() : nullptr;
}

const char* PreparedPackedName(const PreparedPacked* p) { return p->slice ? PreparedSliceName(p->slice.get()) : p->launch.name; }
void FreePreparedPacked(PreparedPacked* p) { delete p; }

int32_t LaunchPreparedPacked(const PreparedPacked* p, const float* x, const float* w, const void* u, const float* bias, const float* residual,
                             float* y, const float* w2, const float* bias2, float* y2, hipStream_t s) {
    if (p->slice) return LaunchPreparedSlice(p->slice.get(), x, w, u, bias, residual, y, w2, bias2, y2, s);
    const PackedLaunch& L = p->launch;
    const uint32_t flags = L.kernel7 ? L.a7.flags : L.a.flags;
    KXC_HIP_REQUIRE(x && w && u && y && (!L.second || (w2 && y2)), "%s: NULL pointer", L.name);
    KXC_HIP_REQUIRE(!(flags & KXC_HIP_CONV_BIAS) || bias, "%s: bias flag without bias", L.name);
    KXC_HIP_REQUIRE(!(flags & KXC_HIP_CONV_RESIDUAL) || residual, "%s: residual flag without residual", L.name);
    if (L.kernel7) {
        conv7_bx::Args b = L.a7;
        b.x = x; b.w = w; b.u = static_cast<const char*>(u); b.bias = bias; b.res = residual; b.y = y;
        if (L.lds_bytes > 64 * 1024)
            if (int32_t rc = GrantLds(reinterpret_cast<const void*>(L.kernel7))) return rc;
        hipLaunchKernelGGL(L.kernel7, NoteGrid(dim3(static_cast<unsigned>(b.units_per_xcd * 8))), NoteBlock(dim3(static_cast<unsigned>(L.threads7))),
                           NoteLds(L.lds_bytes), s, b);
        return CheckLaunch(L.name);
    }
    return LaunchConv(L, x, w, u, bias, residual, y, w2, bias2, y2, s, nullptr);
}

}  // namespace kxc_hip

extern "C" int32_t kxc_hip_conv2d_node_filter_bytes(const kxc_hip_conv2d_desc* desc, int32_t second_output, size_t* out_bytes) {
    KXC_HIP_REQUIRE(desc && out_bytes, "kxc_hip_conv2d_node_filter_bytes: NULL argument");
    *out_bytes = PackedFilterBytes(desc, second_output != 0);
    return KXC_HIP_OK;
}
