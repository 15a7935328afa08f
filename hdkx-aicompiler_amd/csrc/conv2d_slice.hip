// conv2d_slice.hip -- which of a launch plan's 3x3 convolutions (stride 1, or 2 with the second output) take the kernel of conv_slice.h, and their launch.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <memory>

#include "conv_slice.h"

namespace kxc_hip {

struct PreparedSlice {
    conv_sl::Args a;
    void (*kernel)(const conv_sl::Args);
    const char* name;
    int threads;
    size_t lds_bytes;
    bool second;
};

namespace {

struct SliceVariant {
    const char* name;
    int s, ro, ks;
    bool second;
    void (*kernel)(const conv_sl::Args);
};
#define KXC_SLICE(RO, KS) {"mfma_k3x3_slice_o" #RO "_k" #KS, 1, RO, KS, false, conv_sl::conv_slice_kernel<1, RO, KS, false>}
// name = slice_o<blocks of 32 output channels>_k<waves along the input channels>
#define KXC_SLICE_DS(KS) {"mfma_k3x3s2_slice_o1_k" #KS "_ds", 2, 1, KS, true, conv_sl::conv_slice_kernel<2, 1, KS, true>}
const SliceVariant kSlices[] = {KXC_SLICE(1, 4), KXC_SLICE(1, 8), KXC_SLICE(2, 4), KXC_SLICE(2, 8), KXC_SLICE_DS(4), KXC_SLICE_DS(8)};

bool Resolve(const kxc_hip_conv2d_desc* d, bool second, const SliceVariant& v, PreparedSlice* L) {
    using namespace conv_sl;
    if (!d || d->kh != kK || d->kw != kK || d->stride_h != v.s || d->stride_w != v.s || d->dil_h != 1 || d->dil_w != 1 || second != v.second) return false;
    if (d->n <= 0 || d->c <= 0 || d->h <= 0 || d->w <= 0 || d->o <= 0 || d->pad_h < 0 || d->pad_w < 0 || d->pad_h >= kK || d->pad_w >= kK) return false;
    if ((d->flags & (KXC_HIP_CONV_FORCE_DIRECT | KXC_HIP_CONV_HPOOL)) || (second && (d->pad_h != 1 || d->pad_w != 1))) return false;
    const int S = v.s, TP = kPix, E = (kK - 1) / S, NP = Passes(S), PL = Plane(S);
    const int64_t Hp = static_cast<int64_t>(d->h) + 2 * d->pad_h, Wp = static_cast<int64_t>(d->w) + 2 * d->pad_w;
    if (Hp < kK || Wp < kK) return false;
    const int64_t OH = (Hp - kK) / S + 1, OW = (Wp - kK) / S + 1;
    const int64_t x_bytes = 4LL * d->n * d->c * d->h * d->w, y_elems = static_cast<int64_t>(d->n) * d->o * OH * OW;
    const int64_t u_bytes = static_cast<int64_t>(conv_bx::FilterBytes(d->o, d->c, kK, second));
    if (x_bytes >= (1LL << 31) || y_elems >= (1LL << 29) || u_bytes >= (1LL << 31) || (d->n + 1LL) * (Hp + kK) >= (1LL << 30)) return false;
    Args& a = L->a;
    std::memset(&a, 0, sizeof(a));
    a.N = d->n; a.C = d->c; a.H = d->h; a.W = d->w; a.O = d->o;
    a.OH = static_cast<int32_t>(OH); a.OW = static_cast<int32_t>(OW); a.OHW = a.OH * a.OW; a.HW = a.H * a.W; a.M = a.N * a.OHW;
    a.ph = d->pad_h; a.pw = d->pad_w;
    a.Hq = (a.OH - 1) * S + kK;
    a.w4 = (a.W + 3) / 4;
    auto pieces = [&](int from, int to) {      // of four columns, under the output columns from .. to
        return (std::min(to * S - a.pw + kK, a.W) - std::max(from * S - a.pw, 0) + 3) / 4;
    };
    a.full4 = pieces(0, a.OW - 1);
    // Whole rows, or the columns under each output row: what takes fewer loads, if it fits.
    const int64_t rows = conv_bx::TileReach(a.N, a.OHW, a.OW, TP, S, a.Hq - a.OH * S) + kK;
    const int row_hp = S == 2 ? std::max(a.OW + 1, (a.W - 1 + a.pw) / 2 + 1) : 0;
    const int row_pitch = S == 2 ? row_hp + std::max(a.OW, (a.W - 1 + a.pw + 1) / 2) : std::max(a.OW + kK - 1, a.W + a.pw);
    const bool rows_fit = rows * a.w4 <= 32 * NP && rows * row_pitch <= PL;
    int64_t seg_units = 0, segs = 1;
    for (int64_t t = 0; t < a.OW && t * TP < a.M; ++t) {      // where tiles start in a row repeats after at most OW of them
        const int64_t m0 = t * TP, from = m0 % a.OW, n = std::min<int64_t>(TP, a.M - m0), past = (from + n - 1) / a.OW;
        const int last = static_cast<int>((from + n - 1) % a.OW);
        seg_units = std::max<int64_t>(seg_units, pieces(static_cast<int>(from), past > 0 ? a.OW - 1 : last) + (past > 0 ? (past - 1) * a.full4 + pieces(0, last) : 0));
        segs = std::max(segs, past + 1);
    }
    seg_units *= kK;
    const int64_t seg_hp = TP + segs * E, seg_pitch = S == 2 ? seg_hp + TP : seg_hp;
    const bool seg_fit = seg_units <= 32 * NP && seg_pitch * kK <= PL;
    if (!rows_fit && !seg_fit) return false;
    a.seg = seg_fit && (!rows_fit || seg_units < rows * a.w4) ? 1 : 0;
    a.pitch = a.seg ? static_cast<int32_t>(seg_pitch) : row_pitch;
    a.hp = S == 2 ? (a.seg ? static_cast<int32_t>(seg_hp) : row_hp) : 0;
    a.csteps = static_cast<int32_t>(CeilDiv(a.C, kStep));
    a.tail = a.C % kStep != 0 ? 1 : 0;
    a.p_tiles = static_cast<int32_t>(CeilDiv(a.M, TP));
    a.o_tiles = static_cast<int32_t>(CeilDiv(a.O, 32 * v.ro));
    const int64_t tiles = static_cast<int64_t>(a.p_tiles) * a.o_tiles;
    if (tiles >= (1LL << 27)) return false;
    a.num_tiles = static_cast<int32_t>(tiles);
    a.tiles_per_xcd = static_cast<int32_t>(CeilDiv(tiles, 8));
    a.x_bytes = static_cast<uint32_t>(x_bytes);
    a.u_bytes = static_cast<uint32_t>(u_bytes);
    a.flags = d->flags;
    a.o_fastest = x_bytes > u_bytes ? 1 : 0;      // an XCD's run of tiles shares the larger operand
    a.div_ohw = MakeFastDiv(a.OHW); a.div_ow = MakeFastDiv(a.OW); a.div_oh = MakeFastDiv(a.OH); a.div_hq = MakeFastDiv(a.Hq); a.div_w4 = MakeFastDiv(a.w4);
    a.div_full4 = MakeFastDiv(a.full4); a.div_tiles = MakeFastDiv(a.o_fastest ? a.o_tiles : a.p_tiles);
    L->kernel = v.kernel;
    L->name = v.name;
    L->threads = 64 * v.ks;
    L->lds_bytes = static_cast<size_t>(v.ks) * WaveBytes(S);
    L->second = second;
    return true;
}

// us of a launch in a plan, fitted to 1700 shapes of 16 to 512 channels and 0.01 to 4 GFLOP (rms 7 % with four waves, 12 with eight; the
// variant it picks is on average 1.4 % slower than the fastest): a workgroup's start and its steps of 16 channels, per round of
// workgroups.  A compute unit holds two of four waves, which alone take 0.6 of what they take together, or one of eight.  Two outputs (1300 shapes, 5
// and 9 %): one workgroup either way.
double SliceUs(const SliceVariant& v, int64_t tiles, int64_t csteps) {
    const double steps = static_cast<double>(CeilDiv(csteps, v.ks));
    if (v.second) {
        const double w = static_cast<double>(tiles) / 256, whole = static_cast<double>(CeilDiv(tiles, 256));
        return v.ks == 4 ? 5.0 + (0.76 + 2.95 * steps) * (tiles <= 256 ? 1.0 : w + 0.36 * (whole - w)) : 2.1 + (2.15 + 4.56 * steps) * whole;
    }
    if (v.ks == 8) return (v.ro == 1 ? 2.1 : 2.4) + (v.ro == 1 ? 1.15 + 2.93 * steps : 0.55 + 4.65 * steps) * static_cast<double>(CeilDiv(tiles, 256));
    const double w = static_cast<double>(tiles) / 512, whole = static_cast<double>(CeilDiv(tiles, 512));
    const double rounds = tiles <= 256 ? 0.6 : tiles <= 512 ? 1.0 : w + 0.65 * (whole - w);
    return (v.ro == 1 ? 3.0 : 3.4) + (v.ro == 1 ? 1.33 + 2.86 * steps : 1.87 + 4.41 * steps) * rounds;
}

// Whether a plan's node should take it: where its estimate is a twentieth below that of the kernel that the node takes otherwise
// (WinogradNodeUs).  Of 1700 shapes 1090 take it, 1.45 times as fast on average; twelve of them are slower by more than 3 %.
// Nodes with a second output (PairNodeUs) leave 0.08 in hand: 256 of 1320 shapes, 1.19 times as fast, three slower by more than 3 %.
// Those fits are to nodes that run alone, again and again.  Between the other layers of a network, where the matrix cores' clock is lower, they take
// longer by their arithmetic, which is 2.25 times the others' (162 nodes of ResNet-18 at batch 4 to 63, within 7 %): 64 channels at 56 x 56, batch 24 41 us
// for 34 alone, the others 33; 128 at 28 x 28, batch 20 33 for 23, the others 25; 256 at 14 x 14, batch 24 41 for 32, the others 34, batch 8 14.5 and 21; 512 at 7 x 7, batch
// 20 26.5 and 33.6.
// (Above 256 channels they keep the other kernels.  That is no line of speed: the tests of that selection name such a node.)
// KXC_HIP_CONV_SLICE=0: nowhere, =<name>: that variant wherever it covers the node.  Switches that keep convolutions on the fp32
// instructions or name other kernels keep those.
bool Preferred(const kxc_hip_conv2d_desc* d, bool second, PreparedSlice* L) {
    if (!d) return false;
    if (const char* e = std::getenv("KXC_HIP_CONV_SLICE"); e && *e) {
        for (const SliceVariant& v : kSlices)
            if (std::strcmp(e, v.name) == 0) return Resolve(d, second, v, L);
        return false;
    }
    for (const char* name : {"KXC_HIP_WINOGRAD_BF16X3", "KXC_HIP_CONV_BF16X3"})
        if (const char* e = std::getenv(name); e && (e[0] == '0' || (second && e[0] == '1'))) return false;
    for (const char* name : {"KXC_HIP_WINOGRAD_VARIANT", "KXC_HIP_WINOGRAD_GSPLIT", "KXC_HIP_CONV_VARIANT", "KXC_HIP_CONV_GSPLIT", "KXC_HIP_CONV_HPOOL_VARIANT"})
        if (const char* e = std::getenv(name); e && *e) return false;
    if (second && d->c > 256) return false;
    double best_us = second ? 0.92 * PairNodeUs(d) : 0.95 * WinogradNodeUs(d);
    if (best_us <= 0) return false;
    const int stride = second ? 2 : 1;
    const int64_t oh = (static_cast<int64_t>(d->h) + 2 * d->pad_h - 3) / stride + 1, ow = (static_cast<int64_t>(d->w) + 2 * d->pad_w - 3) / stride + 1;
    const int64_t pixels = d->n * oh * ow, csteps = CeilDiv(d->c, conv_sl::kStep);
    const double gflop = 2e-9 * static_cast<double>(SelectLanes() * pixels) * d->o * d->c * (second ? 10 : 9);
    const SliceVariant* best = nullptr;
    for (const SliceVariant& v : kSlices) {
        if (csteps < v.ks || v.second != second) continue;      // (a wave without a step)
        const double alone = SliceUs(v, CeilDiv(pixels, conv_sl::kPix) * CeilDiv(d->o, 32 * v.ro) * SelectLanes(), csteps);
        const double us = std::max(alone, second ? 3.0 + 0.73 * alone + 3.37 * gflop : 1.06 + 0.745 * alone + 2.44 * gflop);
        if (us < best_us) { best_us = us; best = &v; }
    }
    return best && Resolve(d, second, *best, L);
}

}  // namespace

size_t SliceFilterBytes(const kxc_hip_conv2d_desc* d, bool second) {
    PreparedSlice L;
    return Preferred(d, second, &L) ? L.a.u_bytes : 0;
}

PreparedSlice* PrepareSlice(const kxc_hip_conv2d_desc* d, bool second, size_t u_bytes) {
    std::unique_ptr<PreparedSlice> p(new PreparedSlice);
    return Preferred(d, second, p.get()) && u_bytes >= p->a.u_bytes ? p.release() : nullptr;
}

const char* PreparedSliceName(const PreparedSlice* p) { return p->name; }
void FreePreparedSlice(PreparedSlice* p) { delete p; }

int32_t LaunchPreparedSlice(const PreparedSlice* p, const float* x, const float* w, const void* u, const float* bias, const float* residual, float* y,
                            const float* w2, const float* bias2, float* y2, hipStream_t s) {
    conv_sl::Args a = p->a;
    KXC_HIP_REQUIRE(x && w && u && y && (!p->second || (w2 && y2)), "%s: NULL pointer", p->name);
    KXC_HIP_REQUIRE(!(a.flags & KXC_HIP_CONV_BIAS) || bias, "%s: bias flag without bias", p->name);
    KXC_HIP_REQUIRE(!(a.flags & KXC_HIP_CONV_RESIDUAL) || residual, "%s: residual flag without residual", p->name);
    a.x = x; a.w = w; a.u = static_cast<const char*>(u); a.bias = bias; a.res = residual; a.y = y;
    a.w2 = w2; a.bias2 = bias2; a.y2 = y2;
    if (p->lds_bytes > 64 * 1024)
        if (int32_t rc = GrantLds(reinterpret_cast<const void*>(p->kernel))) return rc;
    hipLaunchKernelGGL(p->kernel, NoteGrid(dim3(static_cast<unsigned>(a.tiles_per_xcd * 8))), NoteBlock(dim3(static_cast<unsigned>(p->threads))),
                       NoteLds(p->lds_bytes), s, a);
    return CheckLaunch(p->name);
}

}  // namespace kxc_hip
