// common.h -- shared host-side helpers of libkxc_hip.so (error reporting, stream resolution).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>

#include "kxc_hip.h"

namespace kxc_hip {

// Per-thread message of the last failure (returned by kxc_hip_last_error).
std::string& LastError();
// Per-thread current stream (DeviceAPI::SetStream semantics: thread local).
hipStream_t& CurrentStream();
// Counts every device allocation the library makes (kxc_hip_debug_device_allocations): call next to each hipMalloc.
void NoteDeviceAllocation();

inline int32_t Fail(int32_t code, const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    LastError() = buf;
    return code;
}

inline hipStream_t ResolveStream(void* stream) {
    return stream ? reinterpret_cast<hipStream_t>(stream) : CurrentStream();
}

// Launch-error check: hipGetLastError after a triple-chevron launch.
inline int32_t CheckLaunch(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return Fail(KXC_HIP_ERR_RUNTIME, "%s launch failed: %s", what, hipGetErrorString(e));
    return KXC_HIP_OK;
}

// Geometry of the calling thread's most recent kernel launch, for the profiled plan run: the launch sites
// pass their grid, block and dynamic-LDS arguments through these.
struct LaunchNote {
    uint32_t grid[3] = {0, 0, 0};
    uint32_t block[3] = {0, 0, 0};
    uint32_t dynamic_lds = 0;
};
LaunchNote& LastLaunch();
inline dim3 NoteGrid(dim3 g) { LaunchNote& n = LastLaunch(); n.grid[0] = g.x; n.grid[1] = g.y; n.grid[2] = g.z; return g; }
inline dim3 NoteBlock(dim3 b) { LaunchNote& n = LastLaunch(); n.block[0] = b.x; n.block[1] = b.y; n.block[2] = b.z; return b; }
inline size_t NoteLds(size_t bytes) { LastLaunch().dynamic_lds = static_cast<uint32_t>(bytes); return bytes; }

// floor(x / d) for 0 <= x < 2^31 as a multiply and a shift: shift = 31 + ceil(log2 d), mul = floor(2^shift / d) + 1.
// The kernels' tile set-up divides by launch-invariant values about twenty times; an integer division without
// hardware support costs ~35 instructions, this costs three.
struct FastDiv {
    uint32_t mul, shift;
};
inline FastDiv MakeFastDiv(int32_t d) {
    FastDiv f{1u << 31, 31};
    if (d <= 0) return f;
    uint32_t s = 0;
    while ((1LL << s) < d) ++s;
    f.shift = 31 + s;
    f.mul = static_cast<uint32_t>((1ULL << f.shift) / static_cast<uint64_t>(d) + 1);
    return f;
}
__device__ __forceinline__ int fast_div(int x, FastDiv f) {
    return static_cast<int>((static_cast<uint64_t>(static_cast<uint32_t>(x)) * f.mul) >> f.shift);
}

// Requests the whole argument struct of a kernel at once, at its start.  Left alone the compiler loads members as they are needed, three
// to five times in a row behind one another, each a round trip to memory that a launch of a few microseconds feels (conv_slice.h: 2200 ->
// 1500 cycles until the first load of its input).
#if defined(__HIPCC__)
template <typename Args>
__device__ __forceinline__ void request_args(const Args& a) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int n = static_cast<int>(sizeof(Args) / 8);
    const uint64_t* const q = reinterpret_cast<const uint64_t*>(&a);
    auto at = [&](int i) __attribute__((always_inline)) { return q[i < n ? i : n - 1]; };
    asm volatile("" ::"s"(at(0)), "s"(at(1)), "s"(at(2)), "s"(at(3)), "s"(at(4)), "s"(at(5)), "s"(at(6)), "s"(at(7)), "s"(at(8)), "s"(at(9)), "s"(at(10)), "s"(at(11)),
                 "s"(at(12)), "s"(at(13)), "s"(at(14)), "s"(at(15)), "s"(at(16)), "s"(at(17)), "s"(at(18)), "s"(at(19)), "s"(at(20)), "s"(at(21)), "s"(at(22)), "s"(at(23)),
                 "s"(at(24)), "s"(at(25)), "s"(at(26)), "s"(at(27)), "s"(at(28)), "s"(at(29)));
#endif
}
// The same for kernels that have no scalar registers to hold them all: one word of every 64 bytes, which brings the rest near.
template <typename Args>
__device__ __forceinline__ void request_lines(const Args& a) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int n = static_cast<int>(sizeof(Args) / 4);
    const uint32_t* const q = reinterpret_cast<const uint32_t*>(&a);
    auto at = [&](int i) __attribute__((always_inline)) { return q[i < n ? i : n - 1]; };
    asm volatile("" ::"s"(at(0)), "s"(at(16)), "s"(at(32)), "s"(at(48)), "s"(at(64)), "s"(at(80)), "s"(at(96)));
#endif
}
#endif

// Reductions split over workgroups (both convolution kernels): every part writes raw partial outputs to
// partial[split][total]; SplitReduce adds them in split order (deterministic) and applies the layer's epilogue,
// y = relu(((p0 + p1) + ...) + bias[channel] + residual).
struct SplitReduceArgs {
    const float* partial;
    const float* bias;
    const float* res;
    float* y;
    int32_t gsplit, total, O;
    uint32_t flags;            // KXC_HIP_CONV_BIAS | _RESIDUAL | _RELU
    FastDiv div_ohw;
    // second output of a two-output launch (same shape; y2 == nullptr: none): its parts, bias and flags
    const float* partial2 = nullptr;
    const float* bias2 = nullptr;
    float* y2 = nullptr;
    uint32_t flags2 = 0;
};
// Scratch for the partial outputs: one grow-only buffer per (device, stream), so that launches on different
// streams never share one.  In steady state no call allocates.  The lease keeps other host threads that enqueue
// on the same stream out until the adding kernel has been enqueued behind the parts (release it after that).
struct SplitScratchLease {
    float* ptr = nullptr;
    uint32_t* counters = nullptr;      // kSplitCounters arrival counters, all zero between launches
    std::unique_lock<std::mutex> lock;
};
// A buffer that would have to grow while the stream is being captured (no allocation is allowed there), or that cannot be
// allocated (KXC_HIP_SCRATCH_MAX bytes per buffer at most, where set), is not an error: *available tells, and the caller
// takes a launch that needs none.
int32_t AcquireSplitScratch(hipStream_t stream, size_t bytes, SplitScratchLease* lease, bool* available);
// Whether launches enqueued on a stream run one behind the other for as long as they live, so that they can share the
// buffer of its handle: not while it is being captured (the graph may be replayed on another stream, beside calls on this
// one or beside a second graph captured on it), and not hipStreamPerThread (one handle, a stream for every thread).
bool StreamOrdersScratch(hipStream_t stream);
int32_t LaunchSplitReduce(hipStream_t stream, const SplitReduceArgs& a);

constexpr size_t kMaxLdsBytes = 160 * 1024;  // LDS of one gfx950 compute unit
// Above the default 64 KiB the dynamic LDS size has to be granted per kernel and device (once; device_api.hip).
int32_t GrantLds(const void* kernel);

// A split reduction without the adding kernel: every part stores its raw partial outputs as before, then counts
// itself in at its tile's arrival counter; the part that arrives last adds all parts in split order (the same
// order, hence the same bits, as the adding kernel) and applies the epilogue.  The counters sit in front of the
// partial outputs, start at zero and are set back to zero by the last arrival, so a launch (or the replay of a
// captured one) leaves them as it found them.  Launches that share a scratch buffer are ordered by their stream.
constexpr int32_t kSplitCounters = 16384;
constexpr size_t kSplitCounterBytes = static_cast<size_t>(kSplitCounters) * sizeof(uint32_t);
// Largest number of parts the last arrival finishes itself (0: the adding kernel always does; see split_reduce.hip).
int32_t SplitFuseMaxParts();
// Number of equal launches expected to run beside this one on other streams (1: the launch has the GPU to itself).
// Variant selection sizes its fill rules for that many times the launch's workgroups.
int32_t SelectLanes();

#if defined(__HIPCC__)
// Cache policy of the parts' stores and of the last part's loads of partial outputs: device scope (sc1), i.e.
// written through to and read from the level all XCDs share.  With it no cache-wide write-back or invalidate is
// needed around the counter (a release fence at device scope writes back the whole L2 of the XCD: measured at about
// 20 us per launch of 200 workgroups).
constexpr int kDeviceScopeAux = 0x10;
// True for the workgroup that arrives last of `parts` at `counter`.  Every thread of the workgroup calls it after
// its device-scope stores of partial outputs; `flag` is a word of LDS nobody else uses until the call returns.
// The counter is bumped by a vector memory atomic at device scope once every wave's stores have been acknowledged.
__device__ __forceinline__ bool split_arrive_last(uint32_t* counter, int32_t parts, uint32_t* flag) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t prev = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = prev + 1u == static_cast<uint32_t>(parts);
        if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = last ? 1u : 0u;
    }
    __syncthreads();
    return *flag != 0u;
}
#endif

// A convolution launch resolved ahead of time (a launch plan's node): kernel, tile shape, grid, the split of the
// reduction and every environment switch are decided once, from the descriptor; a launch combines them with the
// operand pointers and the stream.  conv2d_f32.hip (implicit GEMM, one or two outputs) and conv2d_wino_f32.hip.
struct PreparedConv;
int32_t PrepareConv2d(const kxc_hip_conv2d_desc* desc, bool second_output, PreparedConv** out);
int32_t LaunchPreparedConv2d(const PreparedConv* p, const float* x, const float* w, const float* bias, const float* residual,
                             float* y, const float* w2, const float* bias2, float* y2, hipStream_t stream);
const char* PreparedConvName(const PreparedConv* p);
constexpr int64_t kSmallRowLoadsWork = 2300000;      // (16 x 16 tiles) * channels * 9 up to which small 3x3 launches win (conv2d_f32.hip)
bool SmallConvTakes(const kxc_hip_conv2d_desc* desc, bool second_output, bool in_plan);      // ... or a small-launch kernel at all
int32_t HpoolTilePixels(const kxc_hip_conv2d_desc* desc);      // pixels of a tile of the fp32 kernel that takes a pooled launch (0: none does)
bool SmallConvBeatsWinograd(const kxc_hip_conv2d_desc* desc);      // a plan's Winograd node is better launched as PreparedConv
bool SmallConvStagesRows(const kxc_hip_conv2d_desc* desc, bool second_output);      // ... by the kernel that stages whole rows
void FreePreparedConv(PreparedConv* p);
struct PreparedWinograd;
// A node whose filter buffer has u_bytes, holding the one form that the launch reads.  *out = nullptr: no form fits.
int32_t PrepareWinograd(const kxc_hip_conv2d_desc* desc, size_t u_bytes, PreparedWinograd** out, bool may_slice = true);
const char* PreparedWinogradName(const PreparedWinograd* p);
size_t WinogradF32FilterBytes(const kxc_hip_conv2d_desc* desc);
double PairNodeUs(const kxc_hip_conv2d_desc* desc);          // us of a plan's two-output node without the kernel of conv_slice.h (0: never take that)
double WinogradNodeUs(const kxc_hip_conv2d_desc* desc);      // us of a plan's Winograd node without the kernel of conv_slice.h (0: never take that)
int32_t LaunchPreparedWinograd(const PreparedWinograd* p, const float* x, const float* w, const float* u, const float* bias,
                               const float* residual, float* y, hipStream_t stream);
void FreePreparedWinograd(PreparedWinograd* p);

// A convolution on a packed filter (conv2d_bf16x3.hip): bytes of the filter that a plan's node of this shape reads (0: it reads
// its weights as they are), and the launch; *out = nullptr: no such launch, or u_bytes do not hold the filter.
struct PreparedPacked;
size_t PackedFilterBytes(const kxc_hip_conv2d_desc* desc, bool second_output);
void PreparePacked(const kxc_hip_conv2d_desc* desc, bool second_output, size_t u_bytes, PreparedPacked** out);
const char* PreparedPackedName(const PreparedPacked* p);
int32_t LaunchPreparedPacked(const PreparedPacked* p, const float* x, const float* w, const void* u, const float* bias, const float* residual,
                             float* y, const float* w2, const float* bias2, float* y2, hipStream_t stream);
void FreePreparedPacked(PreparedPacked* p);
// The same for small launches (conv2d_slice.hip), 3x3 with stride 1 or, with the second output, 2.
struct PreparedSlice;
size_t SliceFilterBytes(const kxc_hip_conv2d_desc* desc, bool second_output);
PreparedSlice* PrepareSlice(const kxc_hip_conv2d_desc* desc, bool second_output, size_t u_bytes);
const char* PreparedSliceName(const PreparedSlice* p);
int32_t LaunchPreparedSlice(const PreparedSlice* p, const float* x, const float* w, const void* u, const float* bias, const float* residual, float* y,
                            const float* w2, const float* bias2, float* y2, hipStream_t stream);
void FreePreparedSlice(PreparedSlice* p);
struct PreparedSliceDelete {
    void operator()(PreparedSlice* p) const { FreePreparedSlice(p); }
};
using PreparedSlicePtr = std::unique_ptr<PreparedSlice, PreparedSliceDelete>;
// A single nn_conv2d by one of these kernels, its filter packed first: the kernel's name (nullptr: not for this shape), and the
// call.  *launched = false, nothing enqueued: not for this shape (*preferred says), no scratch for the filter, or the stream does
// not order it.
const char* PackedOperatorName(const kxc_hip_conv2d_desc* desc);
int32_t RunPackedOperator(const kxc_hip_conv2d_desc* desc, const float* x, const float* w, const float* bias, const float* residual, float* y,
                          hipStream_t stream, bool* launched, bool* preferred);

// A single nn_conv2d by the three-part Winograd kernel, filter transform included (conv2d_wino_f32.hip): which shapes it is
// for, and the call.  *launched = false, nothing enqueued: there is no scratch for the filter, or the stream does not order it.
bool WinogradOperatorPreferred(const kxc_hip_conv2d_desc* desc);
int32_t RunWinogradOperator(const kxc_hip_conv2d_desc* desc, const float* x, const float* w, const float* bias, const float* residual,
                            float* y, hipStream_t stream, bool* launched);
extern const char* const kWinogradOperatorName;

// The filter transforms of several Winograd layers, and the packed filters of other convolutions, in one launch
// (conv2d_wino_f32.hip).
constexpr uint32_t kWinoFormF32 = 1, kWinoFormThreePart = 2, kFormPacked = 4, kFormSlice = 8;
struct WinoWeightJob {
    const kxc_hip_conv2d_desc* desc;
    const float* w;      // OIHW weights
    float* u;            // where they go, the fp32 form first
    uint32_t forms;      // kWinoForm*: the forms of the filter to write (PreparedWinogradForms: what a node's launch reads), kFormPacked or kFormSlice
    const float* w2;     // kFormPacked: the second output's weights, or nullptr
};
uint32_t PreparedWinogradForms(const PreparedWinograd* p);
int32_t LaunchWinogradWeightTransforms(const WinoWeightJob* jobs, int32_t count, hipStream_t stream);

// The int8 weight tensors of several convolutions packed by one launch (qconv_c16_i8.hip); kind = KXC_HIP_QPACK_*.
struct QPackJob {
    int32_t kind;
    const kxc_hip_qconv2d_desc* desc;
    const int8_t* w;     // OIHW
    int8_t* wp;          // QPackedBytes(job) bytes
};
int32_t QPackedBytes(const QPackJob& job, size_t* out_bytes);
int32_t LaunchQWeightPacks(const QPackJob* jobs, int32_t count, hipStream_t stream);

// Activity recording (activity.hip).  ApiScope times one HIP runtime call on the host; DeviceScope brackets the
// copy / fill / kernel that call enqueues with two HIP events on its stream.  Both do nothing while recording is off.
bool ActivityOn();
struct ActivitySuppress {      // the calling thread records nothing while one of these lives (a profiled plan run
    ActivitySuppress();        // times its launches itself)
    ~ActivitySuppress();
};
class ApiScope {
public:
    explicit ApiScope(const char* name);
    ~ApiScope();
    void SetResult(hipError_t e) { result_ = static_cast<int32_t>(e); }
    uint64_t correlation() const { return correlation_; }
private:
    bool on_;
    const char* name_;
    uint64_t correlation_ = 0;
    int64_t start_ns_ = 0;
    int32_t result_ = 0;
};
class DeviceScope {
public:
    DeviceScope(int32_t kind, const char* name, hipStream_t stream, uint64_t correlation);
    ~DeviceScope();
    int64_t bytes = 0;
    int32_t value = 0, copy_kind = 0;
    uint32_t grid[3] = {0, 0, 0}, block[3] = {0, 0, 0}, dynamic_shared_memory = 0;
private:
    bool on_;
    int32_t kind_;
    const char* name_;
    hipStream_t stream_;
    uint64_t correlation_;
    int64_t host_start_ns_ = 0;
    hipEvent_t start_ = nullptr, stop_ = nullptr;
};

constexpr int64_t kMaxGridX = 2147483647LL;

inline int64_t CeilDiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

}  // namespace kxc_hip

#define KXC_HIP_CALL(expr, what)                                                              \
    do {                                                                                      \
        hipError_t _e = (expr);                                                               \
        if (_e != hipSuccess)                                                                 \
            return ::kxc_hip::Fail(KXC_HIP_ERR_RUNTIME, "%s failed: %s", what, hipGetErrorString(_e)); \
    } while (0)

#define KXC_HIP_REQUIRE(cond, ...)                                              \
    do {                                                                        \
        if (!(cond)) return ::kxc_hip::Fail(KXC_HIP_ERR_INVALID, __VA_ARGS__);  \
    } while (0)
