// Softmax over a flat fp32 vector in ONE workgroup of sixteen waves: reductions within a wave in registers, one
// small LDS exchange between the waves for the maximum and one for the sum, behind barriers that wait for LDS only: the
// logits on their way to memory or the host stay under way (0.45 us a pass less than with butterflies and full barriers).
// Vectors of up to 2048 elements are read once and kept in registers.  (Sixteen waves, not four: a lane then
// finishes one or two logits of a deferred input, and each of them is a round of dependent loads -- 1000 logits
// behind 16 slices: 4.0 against 8.8 us.)
//
// The reference computes exp(x) on the device, downloads the vector, sums it sequentially on the
// host and launches a scale kernel (src/dR_nodes_math.c:620-678).  Mathematically this kernel is
// the same function, exp(x_i)/sum_j exp(x_j); it subtracts max(x) first so that large logits do
// not overflow, and the whole node stays on the device and asynchronous.
#include "drhip_common.hpp"

#include <cfloat>
#include <type_traits>

namespace drhip {

constexpr int kSoftmaxThreads = 1024;
constexpr int kSoftmaxRegs = 2;     // vectors of up to 2048 elements live in registers: one read of x

// Maximum / sum over a wave, in registers: within rows of sixteen lanes, across two rows, across four; the last lane has it.  (A
// butterfly through LDS is six dependent trips of 100 clocks.)
template <bool MAX>
__device__ inline float wave_reduce(float v) {
    constexpr float none = MAX ? -FLT_MAX : 0.0f;
    auto with = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
    auto from = [none](float a, auto ctrl, auto rows) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, none), __builtin_bit_cast(int, a), decltype(ctrl)::value, decltype(rows)::value, 0xf, false));
    };
    using std::integral_constant;
    v = with(v, from(v, integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{}));      // row_shr:1
    v = with(v, from(v, integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{}));
    v = with(v, from(v, integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{}));
    v = with(v, from(v, integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{}));
    v = with(v, from(v, integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{}));      // row_bcast:15
    v = with(v, from(v, integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{}));      // row_bcast:31
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// LDS only: what has been stored for other kernels or the host stays under way.
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Workgroup-wide maximum / sum; the result is valid in every lane.  `red` has one slot per wave, and is of this reduction alone.
template <bool MAX>
__device__ inline float block_reduce(float v, float* red) {
    constexpr int nwaves = kSoftmaxThreads / kWave;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    v = wave_reduce<MAX>(v);
    if (lane == 0) red[wave] = v;
    lds_barrier();
    float r = red[0];
#pragma unroll
    for (int w = 1; w < nwaves; ++w) r = MAX ? fmaxf(r, red[w]) : r + red[w];
    return r;
}

// xdef.partials != NULL: the logits arrive as the partial sums of the GEMV in front (slices added
// in order, then its bias and ReLU); they are finished first (and stored to xdef.finished when the
// caller wants to read the logits too).
template <bool SMALL>
__global__ void __launch_bounds__(kSoftmaxThreads)
softmax_kernel(const float* x, float* y, int n, drhip_deferred_vec xdef, drhip_push push) {    // no __restrict__: x may become y
    __shared__ __attribute__((aligned(16))) float red[2][kSoftmaxThreads / kWave];
    const int tid = threadIdx.x;
    if (SMALL) {                                    // n <= kSoftmaxThreads * kSoftmaxRegs
        float v[kSoftmaxRegs];
#pragma unroll
        for (int u = 0; u < kSoftmaxRegs; ++u) {
            const int i = tid + u * kSoftmaxThreads;
            v[u] = -FLT_MAX;
            if (i < n) v[u] = xdef.partials ? deferred_element(xdef, i) : x[i];
        }
        if (xdef.partials && xdef.finished) {       // (behind all the loads: a store in between would order them)
#pragma unroll
            for (int u = 0; u < kSoftmaxRegs; ++u) {
                const int i = tid + u * kSoftmaxThreads;
                if (i < n) xdef.finished[i] = v[u];
            }
        }
        if (push.host && push.atInput != 0xffffffffu) {
#pragma unroll
            for (int u = 0; u < kSoftmaxRegs; ++u)
                if (tid + u * kSoftmaxThreads < n) push_value(push, push.atInput + tid + u * kSoftmaxThreads, v[u]);
        }
        float m = -FLT_MAX;
#pragma unroll
        for (int u = 0; u < kSoftmaxRegs; ++u) m = fmaxf(m, v[u]);
        m = block_reduce<true>(m, red[0]);
        float s = 0.0f;
#pragma unroll
        for (int u = 0; u < kSoftmaxRegs; ++u) {
            v[u] = (tid + u * kSoftmaxThreads < n) ? expf(v[u] - m) : 0.0f;
            s += v[u];
        }
        const float inv = 1.0f / block_reduce<false>(s, red[1]);
#pragma unroll
        for (int u = 0; u < kSoftmaxRegs; ++u) {
            const int i = tid + u * kSoftmaxThreads;
            if (i < n) store_through(y + i, v[u] * inv);
            if (push.host && i < n) push_value(push, push.at + i, v[u] * inv);
        }
        if (push.host) push_flag(push);
        return;
    }
    if (xdef.partials) {
        for (int i = tid; i < n; i += kSoftmaxThreads) {
            const float s = deferred_element(xdef, i);
            y[i] = s;                           // every lane re-reads only the elements it wrote itself
            if (xdef.finished) xdef.finished[i] = s;
        }
        x = y;
    }
    float m = -FLT_MAX;
    for (int i = tid; i < n; i += kSoftmaxThreads) m = fmaxf(m, x[i]);
    m = block_reduce<true>(m, red[0]);
    float s = 0.0f;
    for (int i = tid; i < n; i += kSoftmaxThreads) s += expf(x[i] - m);
    const float inv = 1.0f / block_reduce<false>(s, red[1]);
    for (int i = tid; i < n; i += kSoftmaxThreads) store_through(y + i, expf(x[i] - m) * inv);
}

// A small layer and the softmax behind it.  As a launch of its own such a layer is one or two workgroups that wait for one trip to
// memory; here the waves that wait for the logits do it.  A thread has column n and every T-th row, so that neighbouring
// threads read neighbouring weights, and the T sums of a column are added in order.
// (128 -> 10 behind 25 slices: 2.8 + 2.8 us as two launches; a thumbnail classifier's call 44 -> 40 us, and 36 with its outputs on
// their way to the host from here.  Loads of rows that do not exist left out and the sums of a column read at once: 7.2 -> 5.9 us, 28.8 -> 28.1 a call.)
constexpr int kFcSoftmaxRows = 16;                  // rows of a thread under way
constexpr int kFcSoftmaxGroups = 32;                // T at most
__global__ void __launch_bounds__(kSoftmaxThreads)
fc_softmax_kernel(const float* __restrict__ Wt, const float* x, const float* __restrict__ bias, float* z, float* y, int K, int N, int T, unsigned mulN, unsigned shN, int relu,
                  drhip_deferred_vec xdef, drhip_push push) {
    __shared__ float xs[1024], part[kSoftmaxThreads];
    __shared__ __attribute__((aligned(16))) float red[2][kSoftmaxThreads / kWave];
    const int tid = threadIdx.x;
    const FastDiv nd = {(unsigned)N, mulN, shN};
    const int g = fast_div(tid, nd), n = tid - g * N;
    float w[kFcSoftmaxRows];
    const float* column = Wt + n;
    const bool works = (tid & ~63) < T * N;             // (the same for a wave; the address unit takes a load of a wave every 8 clocks)
#pragma unroll
    for (int u = 0; u < kFcSoftmaxRows; ++u) w[u] = works && u * T < K ? column[(size_t)min(g + u * T, K - 1) * N] : 0.0f;
    const float b = bias && tid < N ? bias[tid] : 0.0f;
    const float xv = tid < K ? (xdef.partials ? deferred_element(xdef, tid) : x[tid]) : 0.0f;
    if (tid < K) xs[tid] = xv;
    lds_barrier();
    float s = 0.0f;
    for (int k0 = g; k0 < K; k0 += kFcSoftmaxRows * T) {
#pragma unroll
        for (int u = 0; u < kFcSoftmaxRows; ++u) s = k0 + u * T < K ? fmaf(w[u], xs[min(k0 + u * T, K - 1)], s) : s;
        if (k0 + kFcSoftmaxRows * T < K) {
#pragma unroll
            for (int u = 0; u < kFcSoftmaxRows; ++u) w[u] = column[(size_t)min(k0 + (kFcSoftmaxRows + u) * T, K - 1) * N];
        }
    }
    if (g < T) part[g * N + n] = s;
    lds_barrier();
    float v = -FLT_MAX;
    if (tid < N) {
        float p[kFcSoftmaxGroups];                      // (all read before the first is added)
#pragma unroll
        for (int k = 0; k < kFcSoftmaxGroups; ++k) p[k] = part[min(k, T - 1) * N + tid];
        v = p[0];
#pragma unroll
        for (int k = 1; k < kFcSoftmaxGroups; ++k) v = k < T ? v + p[k] : v;
        v += b;
        if (relu) v = fmaxf(v, 0.0f);
        if (z) z[tid] = v;
        if (push.host && push.atInput != 0xffffffffu) push_value(push, push.atInput + tid, v);
    }
    if (xdef.partials && xdef.finished && tid < K) xdef.finished[tid] = xv;
    const float m = block_reduce<true>(v, red[0]);
    const float e = tid < N ? expf(v - m) : 0.0f;
    const float inv = 1.0f / block_reduce<false>(e, red[1]);
    if (tid < N) {
        store_through(y + tid, e * inv);
        if (push.host) push_value(push, push.at + tid, e * inv);
    }
    if (push.host) push_flag(push);
}

}  // namespace drhip

using namespace drhip;

extern "C" int drhip_fc_softmax_usable(int K, int N) { return K >= 1 && N >= 1 && K <= 1024 && N <= 1024 && K * N <= 32768; }

extern "C" int drhip_fc_softmax_f32(const float* x, const drhip_deferred_vec* xdef, const float* Wt, const float* bias, float* z, float* y, int K, int N, int relu,
                                    const drhip_push* push, void* stream) {
    DRHIP_REQUIRE((x || xdef) && Wt && y && y != z, "drhip_fc_softmax_f32: NULL tensor");
    DRHIP_REQUIRE(drhip_fc_softmax_usable(K, N), "drhip_fc_softmax_f32: %d -> %d is not covered", K, N);
    DRHIP_REQUIRE(!xdef || (xdef->partials && xdef->slices > 0 && xdef->n == K), "drhip_fc_softmax_f32: deferred input must carry partial sums of a vector of length %d", K);
    const drhip_deferred_vec none = {nullptr, nullptr, 0, 0, 0, nullptr, 0.0f};
    const drhip_push nowhere = {nullptr, 0, 0, nullptr, 0};
    const FastDiv nd = make_fastdiv(N);
    const int most = kSoftmaxThreads / N, T = most < kFcSoftmaxGroups ? most : kFcSoftmaxGroups;
    launch(fc_softmax_kernel, dim3(1), dim3(kSoftmaxThreads), 0, as_stream(stream), Wt, x, bias, z, y, K, N, T, nd.mul, nd.shift, relu, xdef ? *xdef : none, push ? *push : nowhere);
    return launched("fc_softmax_kernel");
}

extern "C" int drhip_softmax_ex_f32(const float* x, const drhip_deferred_vec* xdef, float* y, int n, void* stream) {
    return drhip_softmax_push_f32(x, xdef, y, n, nullptr, stream);
}

extern "C" int drhip_softmax_push_f32(const float* x, const drhip_deferred_vec* xdef, float* y, int n, const drhip_push* push, void* stream) {
    DRHIP_REQUIRE((x || xdef) && y, "drhip_softmax_f32: NULL tensor");
    DRHIP_REQUIRE(n > 0, "drhip_softmax_f32: n = %d", n);
    DRHIP_REQUIRE(!xdef || (xdef->partials && xdef->slices > 0 && xdef->n == n), "drhip_softmax_f32: deferred input must carry partial sums of a vector of length %d", n);
    DRHIP_REQUIRE(!xdef || xdef->finished != y, "drhip_softmax_f32: the finished logits and the probabilities need separate arrays");
    DRHIP_REQUIRE(!push || n <= kSoftmaxThreads * kSoftmaxRegs, "drhip_softmax_push_f32: %d values are too many", n);
    const drhip_deferred_vec none = {nullptr, nullptr, 0, 0, 0, nullptr, 0.0f};
    const drhip_push nowhere = {nullptr, 0, 0, nullptr, 0};
    if (n <= kSoftmaxThreads * kSoftmaxRegs)
        launch(softmax_kernel<true>, dim3(1), dim3(kSoftmaxThreads), 0, as_stream(stream), x, y, n, xdef ? *xdef : none, push ? *push : nowhere);
    else
        launch(softmax_kernel<false>, dim3(1), dim3(kSoftmaxThreads), 0, as_stream(stream), x, y, n, xdef ? *xdef : none, nowhere);
    return launched("softmax_kernel");
}

extern "C" int drhip_softmax_f32(const float* x, float* y, int n, void* stream) {
    DRHIP_REQUIRE(x, "drhip_softmax_f32: NULL tensor");
    return drhip_softmax_ex_f32(x, nullptr, y, n, stream);
}
