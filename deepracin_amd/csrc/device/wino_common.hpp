// What the Winograd kernels share: the filter transform, buffer-access constants and stores of 2x2 output tiles.
#pragma once

#include "drhip_common.hpp"

namespace drhip {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kXcds = 8;            // L2 domains of MI355X

// u = G g G^T for one 3x3 filter g, row by row.
__device__ inline void wino_filter_transform(const float* __restrict__ g, float (&u)[16]) {
    float t[4][3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const float g0 = g[j], g1 = g[3 + j], g2 = g[6 + j];
        t[0][j] = g0;
        t[1][j] = 0.5f * g0 + 0.5f * g1 + 0.5f * g2;
        t[2][j] = 0.5f * g0 - 0.5f * g1 + 0.5f * g2;
        t[3][j] = g2;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float a = t[r][0], b = t[r][1], cc = t[r][2];
        u[4 * r + 0] = a;
        u[4 * r + 1] = 0.5f * a + 0.5f * b + 0.5f * cc;
        u[4 * r + 2] = 0.5f * a - 0.5f * b + 0.5f * cc;
        u[4 * r + 3] = cc;
    }
}

// Output stores are written through (system-scope store: sc0 sc1) instead of being left dirty in this XCD's L2:
// the consumer is the next kernel, whose workgroups mostly sit on other XCDs and read from memory anyway, and
// what is written during the kernel need not be written back when it ends (224x224x64: 23.5 vs 25.0 us).
__device__ inline void store1_through(float* p, float a) {
    __hip_atomic_store((unsigned*)p, __float_as_uint(a), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ inline void store2_through(float* p, float a, float b) {
    const f32x2 v = {a, b};
    __hip_atomic_store((unsigned long long*)p, __builtin_bit_cast(unsigned long long, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// 2x2 store with edge guards; vec2: W even and the base 8-byte aligned.
__device__ inline void wino_store_tile(float* po, int W, int H, int ox, int oy, int vec2,
                                       float y00, float y01, float y10, float y11) {
    if (vec2) {
        store2_through(po, y00, y01);
        if (oy + 1 < H) store2_through(po + W, y10, y11);
    } else {
        po[0] = y00;
        if (ox + 1 < W) po[1] = y01;
        if (oy + 1 < H) {
            po[W] = y10;
            if (ox + 1 < W) po[W + 1] = y11;
        }
    }
}

// Joined splits: the splits of a panel add their partial tiles up inside the one launch.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
constexpr unsigned kWinoEmpty = 0xffa5c3e1u;        // a signalling NaN: marks a workspace slot whose partial tile has not arrived
constexpr int kAuxThrough = 1 | 16;                 // cache policy of a buffer access: sc0 sc1, written through to memory
constexpr int kAuxDeviceVolatile = 16 | (int)0x80000000u;   // sc1 and volatile, which comes out as sc0 sc1: not served from a cache, reloaded every time
int ws_join_timeouts(unsigned* count);              // of the split-operand kernel
int wino_join_spins();                              // bound on the wait for a partner's partial tile
int wino_halvings(int W, int H, int I, int O);      // of the input channels where the fp32 kernel neither joins nor helps; -1: its 16-tile form
int wino_donated(int W, int H, int I, int O);       // stages of 8 channels that helpers take off each of its panels where it has helpers (0x2c01)

// Nothing of a launch may lie in its workspace when the launch has ended: the next one would take a partial tile that came too
// late for its own panel.  Whoever gives a tile up adds to the kernel's counter first and looks once more behind that; whoever has stored
// tiles reads the counter once they have arrived.  So either the last look finds the tile, or its writer finds the counter not zero.
// From then on (the counter never goes back) writers see their tiles off: they wait until the reader has put the marker back and
// do it themselves where it does not.  (Both sides are on one XCD.  The counter is a trip to memory at the end of the launch: 40x30 512->512 in
// pieces 27.5 / 27.7 us repeated by itself, 30.2 / 30.9 between other layers.)
__device__ inline void wino_gives_up(unsigned* counter) {
    atomicAdd(counter, 1u);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}
__device__ inline unsigned wino_given_up(unsigned* counter) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    // (the caller's tiles have arrived)
    return __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline bool wino_slot_full(u32x4 v) { return v[0] != kWinoEmpty && v[1] != kWinoEmpty && v[2] != kWinoEmpty && v[3] != kWinoEmpty; }
// (spins: for all slots of the caller together)
__device__ inline void wino_see_off(__amdgpu_buffer_rsrc_t r, int at, int& spins) {
    for (; spins > 0; --spins) {
        asm volatile("" ::: "memory");
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, kAuxDeviceVolatile);
        if (v[0] == kWinoEmpty && v[1] == kWinoEmpty && v[2] == kWinoEmpty && v[3] == kWinoEmpty) return;
    }
    __builtin_amdgcn_raw_buffer_store_b128(u32x4{kWinoEmpty, kWinoEmpty, kWinoEmpty, kWinoEmpty}, r, at, 0, kAuxThrough);
}

constexpr int kEpiRelu = DRHIP_EPILOGUE_RELU, kEpiMaxPool2 = DRHIP_EPILOGUE_MAXPOOL2;   // bits of the `relu` argument

// Bias, ReLU and store of one 2x2 tile of channel o, or of its maximum (a following 2x2/2 max pooling; W and H even).
// scale: a power of two that the sums are to be multiplied by.
__device__ inline void wino_finish(float* out, f32x4 y, float bias, int flags, int o, int plane, int W, int H, int ox, int oy, int vec2, float scale = 1.0f) {
#pragma unroll
    for (int k = 0; k < 4; ++k) y[k] = fmaf(y[k], scale, bias);
    if (flags & kEpiRelu) { y[0] = fmaxf(y[0], 0.f); y[1] = fmaxf(y[1], 0.f); y[2] = fmaxf(y[2], 0.f); y[3] = fmaxf(y[3], 0.f); }
    if (flags & kEpiMaxPool2)
        store1_through(out + (size_t)o * (plane >> 2) + (size_t)(oy >> 1) * (W >> 1) + (ox >> 1), fmaxf(fmaxf(y[0], y[1]), fmaxf(y[2], y[3])));
    else
        wino_store_tile(out + (size_t)o * plane + (size_t)oy * W + ox, W, H, ox, oy, vec2, y[0], y[1], y[2], y[3]);
}

}  // namespace drhip
