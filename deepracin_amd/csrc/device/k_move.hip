// Box copy between [C][H][W] tensors and element-wise scalar ops (bandwidth-bound helpers).
//
// copy3d serves the Concat node when its producers could not be planned straight into the concat
// buffer (the reference always launches a generated copy kernel, src/dR_nodes_transform.c:468-553)
// and the Slice node (`extractSlice`, Kernels/dR_transform.cl:5-24).
#include "drhip_common.hpp"

namespace drhip {

__global__ void __launch_bounds__(256)
copy3d_kernel(const float* __restrict__ src, int sW, int sH, int sx0, int sy0, int sz0,
              float* __restrict__ dst, int dW, int dH, int dx0, int dy0, int dz0, int w, int h, int c) {
    const int total = w * h * c;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
        const int x = i % w, y = (i / w) % h, z = i / (w * h);
        dst[((size_t)(z + dz0) * dH + (y + dy0)) * dW + (x + dx0)] =
            src[((size_t)(z + sz0) * sH + (y + sy0)) * sW + (x + sx0)];
    }
}

// Up to four tensors into one: a picture whose channels have a mean of their own each is three of them, and took three slices and
// three of these, 14 us of launches in a row (one: 2.4).
struct ScalarOps { const float* x[4]; size_t n[4], at[4]; int op[4]; float s[4]; };

__global__ void __launch_bounds__(256)
scalar_op_kernel(ScalarOps ops, float* __restrict__ y) {
    const int k = blockIdx.y, op = ops.op[k];
    const float* __restrict__ x = ops.x[k];
    const float s = ops.s[k];
    float* const d = y + ops.at[k];
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < ops.n[k]; i += (size_t)gridDim.x * 256) {
        const float v = x[i];
        float r;
        switch (op) {
            case 0: r = v + s; break;
            case 1: r = v - s; break;
            case 2: r = v * s; break;
            case 3: r = v / s; break;
            case 4: r = logf(v); break;
            case 5: r = expf(v); break;
            case 6: r = sqrtf(v); break;
            case 7: r = s; break;
            default: r = powf(v, s); break;
        }
        d[i] = r;
    }
}

}  // namespace drhip

using namespace drhip;

extern "C" int drhip_copy3d_f32(const float* src, int sW, int sH, int sx0, int sy0, int sz0,
                                float* dst, int dW, int dH, int dx0, int dy0, int dz0,
                                int w, int h, int c, void* stream) {
    DRHIP_REQUIRE(src && dst, "drhip_copy3d_f32: NULL tensor");
    DRHIP_REQUIRE(w > 0 && h > 0 && c > 0, "drhip_copy3d_f32: empty box %dx%dx%d", w, h, c);
    DRHIP_REQUIRE(sx0 >= 0 && sy0 >= 0 && sz0 >= 0 && dx0 >= 0 && dy0 >= 0 && dz0 >= 0, "drhip_copy3d_f32: negative origin");
    DRHIP_REQUIRE(sx0 + w <= sW && sy0 + h <= sH, "drhip_copy3d_f32: box leaves the source plane (%d+%d>%d or %d+%d>%d)", sx0, w, sW, sy0, h, sH);
    DRHIP_REQUIRE(dx0 + w <= dW && dy0 + h <= dH, "drhip_copy3d_f32: box leaves the destination plane");
    DRHIP_REQUIRE((long long)w * h * c < (1ll << 31), "drhip_copy3d_f32: box too large");
    const int total = w * h * c, block = 256;
    int blocks = ceil_div(total, block);
    if (blocks > 16 * num_cu()) blocks = 16 * num_cu();
    launch(copy3d_kernel, dim3(blocks), dim3(block), 0, as_stream(stream),
                       src, sW, sH, sx0, sy0, sz0, dst, dW, dH, dx0, dy0, dz0, w, h, c);
    return launched("copy3d_kernel");
}

extern "C" int drhip_scalar_ops_f32(int count, const float* const* x, const size_t* n, const int* op, const float* s, float* y, void* stream) {
    DRHIP_REQUIRE(count >= 1 && count <= 4 && x && n && op && s && y, "drhip_scalar_ops_f32: %d operations", count);
    ScalarOps ops = {};
    size_t at = 0, most = 0;
    for (int k = 0; k < count; ++k) {
        DRHIP_REQUIRE(x[k], "drhip_scalar_op_f32: NULL tensor");
        DRHIP_REQUIRE(op[k] >= 0 && op[k] <= 8, "drhip_scalar_op_f32: unknown op %d", op[k]);
        ops.x[k] = x[k]; ops.n[k] = n[k]; ops.at[k] = at; ops.op[k] = op[k]; ops.s[k] = s[k];
        at += n[k];
        most = n[k] > most ? n[k] : most;
    }
    if (most == 0) return DRHIP_OK;
    size_t blocks = (most + 255) / 256;
    if (blocks > (size_t)16 * num_cu()) blocks = (size_t)16 * num_cu();
    launch(scalar_op_kernel, dim3((unsigned)blocks, count), dim3(256), 0, as_stream(stream), ops, y);
    return launched("scalar_op_kernel");
}

extern "C" int drhip_scalar_op_f32(const float* x, float* y, size_t n, int op, float s, void* stream) {
    DRHIP_REQUIRE(x && y, "drhip_scalar_op_f32: NULL tensor");
    return drhip_scalar_ops_f32(1, &x, &n, &op, &s, y, stream);
}
