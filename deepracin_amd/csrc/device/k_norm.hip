// Normalization of a whole tensor to a target mean and/or standard deviation:
//
//   mean = sum(x) / n,   dev = sqrt(sum((x - mean)^2) / n)      over all n = W*H*C elements
//   type 0 (mean):      y = x + (targetMean - mean)
//   type 1 (dev):       y = x * (targetDev / dev)
//   type 2 (mean, dev): y = (x + (targetMean - mean)) * (targetDev / dev)
//
// Reference: src/dR_nodes_misc.c:1163-1446 -- tree reductions in 16x8 work-groups per channel
// (`getAvg`, `getSumDev`, Kernels/dR_helper.cl:315-471), repeated until one value per channel is left,
// a blocking download and a host loop over the channels after each of the two reductions, then
// `addScalar` / `mulScalar` / `addMulScalar` (Kernels/dR_math.cl:100-144).  The deviation is taken
// about the mean for type 1 as well (the reference computes the average for all three types).
//
// Here the node stays on the device and asynchronous (HBM-bound, 4n bytes read for both sums, 8n up to where a workgroup's
// elements do not fit its registers, plus 8n for the last sweep): a grid of at most 1024 workgroups leaves its two sums each, and the
// kernel that needs the totals adds those up itself, every workgroup in the same fixed order,
// so no host round trip, no atomics and no device-scope fence are needed and the result is
// reproducible run to run.  The summation order differs from the reference's trees (~1e-7 relative).
#include "drhip_common.hpp"

namespace drhip {

constexpr int kNormThreads = 256;
constexpr int kNormMaxBlocks = 1024;

typedef float nf32x4 __attribute__((ext_vector_type(4)));

__device__ inline float norm_wave_sum(float v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Sum over the workgroup; the result is valid in every lane.
__device__ inline float norm_block_sum(float v, float* red) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    v = norm_wave_sum(v);
    __syncthreads();                    // red may still be read from a previous call
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float s = 0.0f;
#pragma unroll
    for (int w = 0; w < kNormThreads / kWave; ++w) s += red[w];
    return s;
}

// Total of the `count` per-workgroup partials, added in index order by every caller alike.
__device__ inline float norm_total(const float* __restrict__ partials, int count, float* red) {
    float v = 0.0f;
    for (int i = threadIdx.x; i < count; i += kNormThreads) v += partials[i];
    return norm_block_sum(v, red);
}

// Elements of workgroup b of `blocks`: vectors of four in turns of the whole grid, what is left over in workgroup 0.
__device__ inline size_t norm_count(size_t n, int blocks, int b) {
    const size_t n4 = n / 4, turn = (size_t)blocks * kNormThreads, rest = n4 % turn, before = (size_t)b * kNormThreads;
    const size_t mine = rest > before ? (rest - before < kNormThreads ? rest - before : kNormThreads) : 0;
    return 4 * (n4 / turn * kNormThreads + mine) + (b == 0 ? n & 3 : 0);
}

// sums[block] = sum over the workgroup's elements, devs[block] (DEV) = sum of their squared distances from THEIR OWN mean: that
// makes one launch of what the two reductions would be (451x299x3: 4.8 + 4.8 us -> 4.9).
template <bool DEV>
__global__ void __launch_bounds__(kNormThreads)
norm_partial_kernel(const float* __restrict__ x, float* __restrict__ sums, float* __restrict__ devs, size_t n, int blocks) {
    __shared__ float red[kNormThreads / kWave];
    constexpr int R = 4;                                // turns whose elements stay in registers for the second look at them
    const size_t n4 = n / 4, turn = (size_t)blocks * kNormThreads, i0 = (size_t)blockIdx.x * kNormThreads + threadIdx.x;
    const nf32x4* x4 = (const nf32x4*)x;
    nf32x4 keep[R];
    float s = 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const size_t i = i0 + r * turn;
        keep[r] = i < n4 ? x4[i] : nf32x4{0.f, 0.f, 0.f, 0.f};
    }
    const bool last = blockIdx.x == 0 && threadIdx.x < (n & 3);
    const float tail = last ? x[n4 * 4 + threadIdx.x] : 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int k = 0; k < 4; ++k) s += keep[r][k];
    for (size_t i = i0 + R * turn; i < n4; i += turn) {
        const nf32x4 v = x4[i];
#pragma unroll
        for (int k = 0; k < 4; ++k) s += v[k];
    }
    s += tail;
    s = norm_block_sum(s, red);
    if (threadIdx.x == 0) sums[blockIdx.x] = s;
    if constexpr (DEV) {
        const float mean = s / (float)norm_count(n, blocks, blockIdx.x);
        float q = 0.0f;
        auto add = [&](nf32x4 v) {
#pragma unroll
            for (int k = 0; k < 4; ++k) { const float d = v[k] - mean; q += d * d; }
        };
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (i0 + r * turn < n4) add(keep[r]);
        for (size_t i = i0 + R * turn; i < n4; i += turn) add(x4[i]);
        if (last) { const float d = tail - mean; q += d * d; }
        q = norm_block_sum(q, red);
        if (threadIdx.x == 0) devs[blockIdx.x] = q;
    }
}

__global__ void __launch_bounds__(kNormThreads)
norm_apply_kernel(const float* __restrict__ x, float* __restrict__ y, const float* __restrict__ sums,
                  const float* __restrict__ devs, size_t n, int blocks, int type, float targetMean, float targetDev) {
    __shared__ float red[kNormThreads / kWave];
    const float mean = norm_total(sums, blocks, red) / (float)n;
    float add = 0.0f, mul = 1.0f;
    if (type != 1) add = -(mean - targetMean);
    if (type != 0) {
        // about the mean of all: each workgroup's sum about its own, and the distance of that from the other, once per element
        float q = 0.0f;
        for (int b = threadIdx.x; b < blocks; b += kNormThreads) {
            const float count = (float)norm_count(n, blocks, b), d = sums[b] / count - mean;
            q += devs[b] + count * (d * d);
        }
        const float dev = sqrtf(norm_block_sum(q, red) / (float)n);
        mul = 1.0f / (dev / targetDev);
    }
    const size_t n4 = n / 4;
    for (size_t i = (size_t)blockIdx.x * kNormThreads + threadIdx.x; i < n4; i += (size_t)gridDim.x * kNormThreads) {
        nf32x4 v = ((const nf32x4*)x)[i];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = (v[k] + add) * mul;
        ((nf32x4*)y)[i] = v;
    }
    if (blockIdx.x == 0)
        for (size_t i = n4 * 4 + threadIdx.x; i < n; i += kNormThreads) y[i] = (x[i] + add) * mul;
}

static int norm_blocks(size_t n) {
    size_t b = (n / 4 + kNormThreads - 1) / kNormThreads;
    if (b < 1) b = 1;
    return (int)(b > (size_t)kNormMaxBlocks ? kNormMaxBlocks : b);
}

}  // namespace drhip

using namespace drhip;

extern "C" size_t drhip_normalize_scratch_floats(size_t n) { return n ? 2 * (size_t)norm_blocks(n) : 0; }

extern "C" int drhip_normalize_f32(const float* x, float* y, size_t n, int type, float targetMean, float targetDev,
                                   float* scratch, void* stream) {
    DRHIP_REQUIRE(x && y && scratch, "drhip_normalize_f32: NULL pointer");
    DRHIP_REQUIRE(n > 0, "drhip_normalize_f32: empty tensor");
    DRHIP_REQUIRE(type >= 0 && type <= 2, "drhip_normalize_f32: unknown normalization type %d (0 mean, 1 deviation, 2 both)", type);
    DRHIP_REQUIRE((((size_t)x | (size_t)y) & 15) == 0, "drhip_normalize_f32: tensors must be 16-byte aligned");
    const int blocks = norm_blocks(n);
    float* sums = scratch;
    float* devs = scratch + blocks;
    hipStream_t s = as_stream(stream);
    if (type == 0) launch((norm_partial_kernel<false>), dim3(blocks), dim3(kNormThreads), 0, s, x, sums, devs, n, blocks);
    else launch((norm_partial_kernel<true>), dim3(blocks), dim3(kNormThreads), 0, s, x, sums, devs, n, blocks);
    if (int rc = launched("norm_partial_kernel")) return rc;
    launch(norm_apply_kernel, dim3(blocks), dim3(kNormThreads), 0, s, x, y, (const float*)sums, (const float*)devs, n, blocks,
           type, targetMean, targetDev);
    return launched("norm_apply_kernel");
}
