// Shared plumbing of the HIP device layer: error reporting and a few device helpers.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <vector>

#include "dr_hip.h"

namespace drhip {

// Per-thread message of the last failure, returned by drhip_last_error().
char* error_slot();

inline int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(error_slot(), 512, fmt, ap);
    va_end(ap);
    return code;
}

inline int check(hipError_t e, const char* what) {
    if (e == hipSuccess) return DRHIP_OK;
    return fail(DRHIP_EDEVICE, "%s: %s", what, hipGetErrorString(e));
}

// Reports a launch-time error (bad configuration) right after a kernel launch.
inline int launched(const char* kernel) { return check(hipGetLastError(), kernel); }

inline hipStream_t as_stream(void* s) { return (hipStream_t)s; }

constexpr int kWave = 64;   // CDNA wavefront width
constexpr unsigned kBufferFlags = 0x00020000u;      // dword 3 of a gfx9 raw buffer resource (32-bit data format)
constexpr unsigned kOutOfRange = 0x80000000u;       // byte offset no resource of at most 2 GiB contains

// Per-thread record of kernel execution times (drhip_timing_begin / drhip_timing_end).  While it is
// on, every launch carries its own start and stop event (hipExtLaunchKernelGGL attaches them to the
// dispatch packet), so the span is the kernel alone -- no extra packets between the kernels, which
// is what events recorded between launches would put there.
struct LaunchTimer {
    bool on = false;
    size_t used = 0;                   // events handed out since drhip_timing_begin
    std::vector<hipEvent_t> events;    // [2*i] start, [2*i+1] stop of launch i
};
LaunchTimer& launch_timer();

// Every kernel of this library is launched through here.
template <typename Kernel, typename... Args>
inline void launch(Kernel kernel, dim3 grid, dim3 block, size_t ldsBytes, hipStream_t stream, Args... args) {
    LaunchTimer& t = launch_timer();
    if (!t.on) {
        hipLaunchKernelGGL(kernel, grid, block, ldsBytes, stream, args...);
        return;
    }
    while (t.events.size() < t.used + 2) {
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess) { hipLaunchKernelGGL(kernel, grid, block, ldsBytes, stream, args...); return; }
        t.events.push_back(e);
    }
    hipExtLaunchKernelGGL(kernel, grid, block, ldsBytes, stream, t.events[t.used], t.events[t.used + 1], 0, args...);
    t.used += 2;
}

// More than 64 KiB of dynamic LDS has to be asked for once per kernel and device (the attribute belongs to the kernel's
// code object on ONE device); `asked` is the kernel's own memory of that, one bit per device.  Graphs may be prepared
// and applied from several host threads.
constexpr int kMaxDynamicLds = 159 * 1024;           // (of 160 KiB: what a kernel declares statically comes on top)
inline int allow_lds(const void* kernel, size_t bytes, std::atomic<unsigned long long>& asked) {
    if (bytes <= 65536) return DRHIP_OK;
    int device = 0;
    if (int rc = check(hipGetDevice(&device), "hipGetDevice")) return rc;
    const unsigned long long bit = device >= 0 && device < 64 ? 1ull << device : 0;
    if (asked.load(std::memory_order_acquire) & bit) return DRHIP_OK;
    if (int rc = check(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxDynamicLds), "hipFuncSetAttribute(max dynamic LDS)")) return rc;
    asked.fetch_or(bit, std::memory_order_acq_rel);
    return DRHIP_OK;
}

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// Division by a number known at launch time, as a multiplication (Granlund & Montgomery): with
// l = ceil(log2 d) and mul = floor(2^32 (2^l - d) / d) + 1, n / d = (mulhi(n, mul) + n) >> l for every n < 2^31.
// A hardware integer division is some 30 dependent instructions, and in the short kernels of a batch-1 pass
// those in front of a workgroup's first loads are part of every layer's latency (~0.1 us per kernel).
struct FastDiv { unsigned d, mul, shift; };
inline FastDiv make_fastdiv(int d) {                 // d >= 1
    unsigned l = 0;
    while ((1ull << l) < (unsigned long long)d) ++l;
    const unsigned long long m = ((1ull << 32) * ((1ull << l) - (unsigned long long)d)) / (unsigned long long)d + 1;
    return FastDiv{(unsigned)d, (unsigned)m, l};
}
__device__ inline int fast_div(int n, const FastDiv& f) { return (int)((__umulhi((unsigned)n, f.mul) + (unsigned)n) >> f.shift); }

// A layer's results are stored written through (system-scope store: sc0 sc1) instead of being left dirty in the
// XCD's L2: the reader is the next kernel, whose workgroups mostly sit on other XCDs and read from memory anyway,
// and what has been written during the kernel need not be written back when it ends (0.15-0.45 us per launch on
// the 14x14 layers, 1.5 us on a 12.8 MB output).
__device__ inline void store_through(float* p, float v) {
    __hip_atomic_store((unsigned*)p, __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A value for the host (drhip_push), and, by every lane of the workgroup behind its last one, the flag that tells it of them.
__device__ inline void push_value(const drhip_push& p, unsigned at, float v) {
    __hip_atomic_store((unsigned*)p.host + at, __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ inline void push_flag(const drhip_push& p) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // this lane's stores have been accepted
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(p.flag, p.value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Element `row` of an activation vector that a split GEMV left as partial sums: slices added in
// order, then bias and ReLU -- bit for bit what the GEMV's finishing kernel stores.
__device__ inline float deferred_element(const drhip_deferred_vec& d, int row) {
    const float* pp = d.partials + row;
    float s = 0.0f;
    int sl = 0;
    // 32, 16, then 8 independent loads in flight, always summed in slice order: the partial sums come
    // from other XCDs' workgroups, so every round of loads costs a trip to memory
    for (; sl + 32 <= d.slices; sl += 32) {
        float v[32];
#pragma unroll
        for (int u = 0; u < 32; ++u) v[u] = pp[(size_t)(sl + u) * d.n];
#pragma unroll
        for (int u = 0; u < 32; ++u) s += v[u];
    }
    if (sl + 16 == d.slices) {                      // (a GEMV that fills the chip leaves 16 slices: one round, not two)
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = pp[(size_t)(sl + u) * d.n];
#pragma unroll
        for (int u = 0; u < 16; ++u) s += v[u];
        sl += 16;
    }
    if (d.slices - sl > 8) {                        // the ragged end in one round as well: clamped loads, zeros by select
        float v[32];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = pp[(size_t)min(sl + u, d.slices - 1) * d.n];
        if (d.slices - sl > 16) {
#pragma unroll
            for (int u = 16; u < 32; ++u) v[u] = pp[(size_t)min(sl + u, d.slices - 1) * d.n];
        }
#pragma unroll
        for (int u = 0; u < 32; ++u) s = (sl + u < d.slices) ? s + v[u] : s;
        sl = d.slices;
    }
    for (; sl < d.slices; sl += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = pp[(size_t)min(sl + u, d.slices - 1) * d.n];
#pragma unroll
        for (int u = 0; u < 8; ++u) s = (sl + u < d.slices) ? s + v[u] : s;
    }
    if (d.bias) s += d.bias[row];
    if (d.relu) s = fmaxf(s, 0.0f);
    if (d.divisor != 0.0f) s = s / d.divisor;
    return s;
}

// Number of compute units of the active device (cached by drhip_init; 256 on MI355X).
int num_cu();

// Per-device set-up of the fully-connected kernels' built-in scratch (k_fc.hip); `device` must be current.
int fc_static_scratch_setup(int device);

}  // namespace drhip

#define DRHIP_REQUIRE(cond, ...)                                   \
    do {                                                           \
        if (!(cond)) return drhip::fail(DRHIP_EINVAL, __VA_ARGS__); \
    } while (0)
