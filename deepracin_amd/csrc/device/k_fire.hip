// Fire modules in a chain: the expand layers of one module and the squeeze layer of the next in one launch.
//
// A fire module is a 1x1 "squeeze" layer to S channels and two "expand" layers of E channels each on its output, one 1x1 and one
// 3x3, whose outputs are concatenated; what reads them is the squeeze layer of the next module, sometimes behind a 3x3 / stride-2
// max pooling.  A squeeze layer needs nothing but the pixel itself, so a workgroup that holds expand outputs of some pixels can
// multiply them with its part of the next squeeze layer's filters right away: the 2E-channel tensor never exists, and a module
// is one launch instead of two.
//
// What bounds it: nothing but the launch.  A layer of such a network is a few MFLOP, and a launch that waits for the one in front of it
// takes 3 to 4 us whatever it does (start, one trip to memory, the stores).  So the work is cut for latency:
//   * A workgroup owns a block of output pixels, mostly at most 16 (an MFMA column each), and a slice of 16*Q channels of either
//     expand layer.  Slices make enough workgroups of 14x14 maps; each leaves its part of the next squeeze layer's sums,
//     [slice][pixel][channel], and the next launch adds the slices (in order: the results do not depend on timing), bias and ReLU
//     while it loads them.
//   * Every load of a workgroup is issued at its start: the input, the filters (16 bytes per lane are four k-steps, see below)
//     and the next layer's; of the filters 20 packs, for behind other layers a pack is a trip to memory (12 / 16 / 20 / 24 packs: SqueezeNet at
//     224x224 57.8 / 57.3 / 57.4 / 57.5 us a pass, at 451x299 84.7 / 83.9 / 83.1 / 82.8).
//   * Four waves, one per SIMD, and few instructions: what a wave does once is paid per wave, 4 clocks an instruction.  A first form with
//     eight waves and shapes known at run time issued its first loads a microsecond after its start and took 430 clocks for
//     the four MFMAs of an item.  So the item loop is unrolled over constants (S/16 is a template parameter, rows of the patch lie 12
//     pixels apart in LDS: an operand is one read at an immediate offset), the grid has three dimensions instead of
//     divisions, loads carry what is common to a wave in a scalar register and return zeros beside the map, and the arguments of
//     the first loads arrive with the wave.
//   * With Q = 4 every wave has a sixteen of channels for itself; otherwise the waves of a sixteen share the k-steps of each item, and
//     their sums meet in LDS.
// Measured: SqueezeNet v1.1's eight modules at 224x224, two launches each / one, 79.2 / 60.7 us a pass (56x56 module and
// the next squeeze layer 7.5 / 3.2 us, 28x28 8.1 / 4.4, 14x14 9.2 to 9.7 / 5.0 to 5.6; with a pooling between them 8.9 and 9.9 / 4.4
// and 4.9).  A photograph of 451x299 through the same network 190 / 163 us with its feed and download.
// The arithmetic is plain fp32 (v_mfma_f32_16x16x4_f32): a slice is 320*S/16*Q clocks of it, less than the trips to memory, and
// direct sums need no care about infinities and are closer to the exact result than Winograd's.
//
// Replaces for such modules conv2d1x1 (Kernels/dR_conv2d1x1.cl), the Winograd kernel (Kernels/dR_winograd2.cl) and the generated
// pooling kernel (src/dR_nodes_pooling.c:277-401), which the reference runs one after the other.
#include "drhip_common.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace drhip {

typedef float f32x4f __attribute__((ext_vector_type(4)));
typedef float f32x2f __attribute__((ext_vector_type(2)));
typedef unsigned u32x4f __attribute__((ext_vector_type(4)));
constexpr int kAuxThrough16 = 1 | 16;           // sc0 sc1: written through to memory
constexpr int kFireThreads = 256;
constexpr int kFireAhead = 20;                  // packs of filters a wave has under way at most
constexpr int kFireSlices = 8;                  // slices of a quad of the patch that are under way together
constexpr int kFireRow = 12;                    // pixels from row to row of the patch in LDS

// n / d by multiplication for small numbers: n * d < 2^20
constexpr unsigned small_mul(int d) { return (1u << 20) / (unsigned)d + 1; }
__device__ inline int small_div(int n, unsigned mul) { return (int)((unsigned)n * mul >> 20); }

// An item is a tap and 16 input channels of the 3x3 layer (9*S16 of them, channels fastest), or 16 input channels of the 1x1 layer (S16).
// A fragment of an item, for 16 output channels: lane l holds output channel l%16 and input channels 4*(l/16) .. +3; the MFMA of
// k-step s contracts channels s, 4+s, 8+s and 12+s, one from each sixteen lanes.  The G = 4/Q waves of a sixteen take 4/G k-steps
// each, so 16 bytes per lane are a pack of G items.
// Bank, slice by slice: packs [pack][wave][lane][4]; the next squeeze layer's fragments [2Q sixteens of expand channels, 1x1 layer's
// first][MB][lane][4]; the expand layers' biases [1x1, 3x3][16*Q].
constexpr int fire_packs(int S16, int Q) { return (10 * S16 + 4 / Q - 1) / (4 / Q); }
constexpr int fire_slice_bytes(int S16, int Q, int MB) { return fire_packs(S16, Q) * 4096 + 2 * Q * MB * 1024 + 128 * Q; }
// LDS, in floats: sums of waves that share something; expand outputs, and pooled; the patch
constexpr int fire_columns(bool pool) { return pool ? 3 : 1; }          // columns of 16 expand pixels of a workgroup
constexpr int fire_sums(int Q, bool pool) { return 256 * std::max((4 / Q - 1) * Q * 2 * fire_columns(pool), 3); }
constexpr int fire_outs(int Q, bool pool) { return (16 * fire_columns(pool) + (pool ? 16 : 0)) * (32 * Q + 4); }

// quads of the patch that a thread has under way: patches of up to 32 pixels without a pooling, 77 with one, go over at once
constexpr int fire_quads(int S16, bool pool) { return pool ? (S16 > 1 ? 3 : 2) : (S16 > 1 ? 2 : 1); }

// Q: sixteens of channels of either layer per slice.  STORE: the expand outputs themselves are
// stored, 1x1 layer first, [2E][H][W] or, with bit 31 of outWh, [H][W][2E].  PLAIN: the input is a tensor [S][H][W].  Grid: slices x blocks across x blocks down (eight slices: one per XCD and its L2).
// wh: W | H << 16.  block: bw | bh << 8 (output pixels of a workgroup) | ew << 16 | epx << 24 (expand pixels under them: columns, number).
// misc: patch pixels | S << 8 | slices of the input << 16 | ReLU of the input << 24 | ReLU << 25 | MB << 26 |
// log2(waves of different mb) << 29.  outWh: map of what is stored, Wo | Ho << 16 (STORE: E).
template <int S16, int Q, bool POOL, bool STORE, bool PLAIN>
__global__ void __launch_bounds__(kFireThreads, 2)
fire_kernel(const float* __restrict__ in, const float* __restrict__ bank, unsigned wh, unsigned block, unsigned misc, unsigned mulHw,
            const float* __restrict__ inBias, unsigned mulHpx, unsigned mulEw, unsigned mulBw, unsigned outWh, float* __restrict__ out) {
    constexpr int NCW = fire_columns(POOL), G = 4 / Q, KS = 4 / G;        // waves that share a sixteen; k-steps of an item each takes
    constexpr int NI = 10 * S16, N9 = 9 * S16, NP = fire_packs(S16, Q), D = NP < kFireAhead ? NP : kFireAhead;
    constexpr int SP = 16 * S16, PITCH = SP + 4, QUADS = SP / 4;        // channels; floats from pixel to pixel of the patch
    constexpr int RP = 32 * Q + 4;              // the same of the expand outputs
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float* const outs = lds + fire_sums(Q, POOL);
    float* const patch = outs + (STORE ? 0 : fire_outs(Q, POOL));
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lk = lane >> 4, q = wave / G, g = wave % G;
    const int W = wh & 0xffff, H = wh >> 16, plane = W * H;
    const int bw = block & 255, bh = block >> 8 & 255, ew = block >> 16 & 255, hw = ew + 2;
    const int hpx = misc & 255, S = misc >> 8 & 255, slicesIn = misc >> 16 & 255;
    const int ox0 = blockIdx.y * bw, oy0 = blockIdx.z * bh, ex0 = POOL ? 2 * ox0 : ox0, ey0 = POOL ? 2 * oy0 : oy0;
    const int items = hpx * QUADS;

    // ---- loads ---------------------------------------------------------------------------------------------------------
    auto load16 = [](const __amdgpu_buffer_rsrc_t& r, int v, int sOff) { return __builtin_bit_cast(f32x4f, __builtin_amdgcn_raw_buffer_load_b128(r, v, sOff, 0)); };
    const int MB = misc >> 26 & 7, mbBits = misc >> 29, KP = 4 >> mbBits;       // (MB = 0: nothing behind)
    const int mb = wave & ((1 << mbBits) - 1), kp = wave >> mbBits;             // this wave's part of the next squeeze layer
    const __amdgpu_buffer_rsrc_t rBank = __builtin_amdgcn_make_buffer_rsrc((void*)bank, 0, 0x7ffffff0, kBufferFlags);
    const int bank0 = blockIdx.x * (NP * 4096 + 2 * Q * 1024 * MB + 128 * Q), bank2 = bank0 + NP * 4096, bank3 = bank2 + 2 * Q * 1024 * MB;
    f32x4f a[D], a2[2 * Q], biasE[2];
    auto load_a = [&](int p) { a[p % D] = load16(rBank, 16 * lane, bank0 + p * 4096 + wave * 1024); };
    auto everything_else = [&] {
        asm volatile("" ::: "memory");
#pragma unroll
        for (int p = 0; p < D; ++p) load_a(p);
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (G == 1 || k == 0) biasE[k] = load16(rBank, 16 * lk, bank3 + 64 * Q * (G == 1 ? k : g & 1) + 64 * q);
        if (!STORE && mb < MB) {
#pragma unroll
            for (int u = 0; u < 2 * Q; ++u)
                if (u * KP < 2 * Q) a2[u] = load16(rBank, 16 * lane, bank2 + (min(kp + u * KP, 2 * Q - 1) * MB + mb) * 1024);
        }
        asm volatile("" ::: "memory");
    };
    constexpr int U = fire_quads(S16, POOL);    // quads of the patch a thread has under way
    const int stride = plane * SP * 4;          // bytes of a slice
    const __amdgpu_buffer_rsrc_t rIn = __builtin_amdgcn_make_buffer_rsrc((void*)in, 0, PLAIN ? S * plane * 4 : slicesIn * stride, kBufferFlags);
    const __amdgpu_buffer_rsrc_t rBias = __builtin_amdgcn_make_buffer_rsrc((void*)inBias, 0, inBias ? SP * 4 : 0, kBufferFlags);
    auto fill = [&](int base, bool first) {
        f32x4f v[U][PLAIN ? 1 : kFireSlices], biasIn[U];
        int at[U], qd[U];
        unsigned vo[U], away[U];                // (the sign bit: out of every range)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = base + u * kFireThreads + tid;
            qd[u] = PLAIN ? small_div(i, mulHpx) : i % QUADS;                   // (plain: neighbouring lanes, neighbouring addresses)
            const int px = PLAIN ? i - qd[u] * hpx : i / QUADS;
            const int hy = small_div(px, mulHw), hx = px - hy * hw, x = ex0 - 1 + hx, y = ey0 - 1 + hy;
            away[u] = (unsigned)x < (unsigned)W && (unsigned)y < (unsigned)H && i < items ? 0u : kOutOfRange;
            at[u] = (hy * kFireRow + hx) * PITCH + 4 * qd[u];
            const unsigned place = (unsigned)(y * W + x);
            if constexpr (PLAIN) {              // (the range check does not see the scalar offset, and the last quad may be a part of one)
                vo[u] = 4u * ((unsigned)(4 * qd[u] * plane) + place);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[u][0][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rIn, (int)((vo[u] + 4u * e * plane) | away[u]), 0, 0));
            } else {
                vo[u] = (4u * (place * SP + 4u * qd[u])) | away[u];
                v[u][0] = load16(rIn, (int)vo[u], 0);
            }
        }
        if constexpr (!PLAIN) {
#pragma unroll
            for (int j = 1; j < kFireSlices; ++j)
                if (j < slicesIn) {
#pragma unroll
                    for (int u = 0; u < U; ++u) v[u][j] = load16(rIn, (int)vo[u], j * stride);
                }
#pragma unroll
            for (int u = 0; u < U; ++u) biasIn[u] = load16(rBias, (int)(16u * qd[u] | away[u]), 0);             // (zeros beside the map)
        }
        if (first) everything_else();
        if constexpr (!PLAIN) {
#pragma unroll
            for (int j = 1; j < kFireSlices; ++j)
                if (j < slicesIn) {
#pragma unroll
                    for (int u = 0; u < U; ++u) v[u][0] += v[u][j];
                }
            if (__builtin_expect(slicesIn > kFireSlices, 0))
                for (int j = kFireSlices; j < slicesIn; ++j)
#pragma unroll
                    for (int u = 0; u < U; ++u) v[u][0] += load16(rIn, (int)vo[u], j * stride);
#pragma unroll
            for (int u = 0; u < U; ++u) v[u][0] += biasIn[u];
            if (misc & 1u << 24) {
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[u][0][e] = fmaxf(v[u][0][e], 0.0f);
            }
            if (__builtin_expect(S != SP, 0)) { // channels that do not exist: zeros also behind infinities
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[u][0][e] = 4 * qd[u] + e < S ? v[u][0][e] : 0.0f;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (base + u * kFireThreads + tid < items) *(f32x4f*)(patch + at[u]) = v[u][0];
    };
    fill(0, true);
    if (__builtin_expect(items > U * kFireThreads, 0))
        for (int base = U * kFireThreads; base < items; base += U * kFireThreads) fill(base, false);
    auto barrier = [&] {                        // (LDS only: loads stay under way)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    // ---- expand: D of the MFMA: lane -> pixel lane%16, register r -> channel 4*(lane/16) + r -----------------------------
    f32x4f acc[2][NCW];                         // 1x1 layer, 3x3 layer
    const float* here[NCW];
    bool inMap[NCW];
    int place[NCW];
#pragma unroll
    for (int c = 0; c < NCW; ++c) {
        acc[0][c] = acc[1][c] = f32x4f{0.f, 0.f, 0.f, 0.f};
        const int e = 16 * c + l16, p = e < (int)(block >> 24) ? e : 0;         // (columns without a pixel repeat the first)
        const int ey = small_div(p, mulEw), ex = p - ey * ew;
        here[c] = patch + (ey * kFireRow + ex) * PITCH + 4 * lk + g * KS;
        inMap[c] = e < (int)(block >> 24) && ex0 + ex < W && ey0 + ey < H;
        place[c] = (ey0 + ey) * W + ex0 + ex;
    }
    barrier();
    f32x4f b[2][NCW];                           // (the patch's samples of the next item are read in front of the products of this one)
    auto read_b = [&](int i) {
        const int tap = i < N9 ? i / S16 : 4, c16 = i < N9 ? i % S16 : i - N9, off = (tap / 3 * kFireRow + tap % 3) * PITCH + 16 * c16;
#pragma unroll
        for (int c = 0; c < NCW; ++c) {
            if (KS == 4) b[i & 1][c] = *(const f32x4f*)(here[c] + off);
            else if (KS == 2) { const f32x2f v = *(const f32x2f*)(here[c] + off); b[i & 1][c][0] = v[0]; b[i & 1][c][1] = v[1]; }
            else b[i & 1][c][0] = here[c][off];
        }
    };
    read_b(0);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        if (i + 1 < NI) read_b(i + 1);
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
            for (int c = 0; c < NCW; ++c)
                acc[i < N9][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i / G % D][i % G * KS + k], b[i & 1][c][k], acc[i < N9][c], 0, 0, 0);
        if (i % G == G - 1 && i / G + D < NP) load_a(i / G + D);
    }

    // ---- sums of the waves that share a sixteen; bias and ReLU ----------------------------------------------------------------
    // (one of them finishes the 1x1 layer's and another the 3x3 layer's, so that both are finished at once)
    auto finish = [&](f32x4f (&sum)[NCW], int k, const f32x4f& bias) {
        if (misc & 1u << 25) {
#pragma unroll
            for (int c = 0; c < NCW; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) sum[c][r] = fmaxf(sum[c][r] + bias[r], 0.0f);
        } else {
#pragma unroll
            for (int c = 0; c < NCW; ++c) sum[c] += bias;
        }
#pragma unroll
        for (int c = 0; c < NCW; ++c) {
            if constexpr (STORE) {
                const int E = outWh & 0x7fffffff, o = k * E + blockIdx.x * 16 * Q + 16 * q + 4 * lk;
                if (outWh >> 31) {
                    const __amdgpu_buffer_rsrc_t rOut = __builtin_amdgcn_make_buffer_rsrc((void*)out, 0, 0x7ffffff0, kBufferFlags);
                    if (inMap[c]) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4f, sum[c]), rOut, 4 * (place[c] * 2 * E + o), 0, kAuxThrough16);
                } else if (inMap[c]) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) store_through(out + (size_t)(o + r) * plane + place[c], sum[c][r]);
                }
            } else {
                if (POOL && !inMap[c]) sum[c] = f32x4f{0.f, 0.f, 0.f, 0.f};     // (samples beside the map count as 0.0)
                *(f32x4f*)(outs + (16 * c + l16) * RP + 16 * (k * Q + q) + 4 * lk) = sum[c];
            }
        }
    };
    if constexpr (G == 1) {
#pragma unroll
        for (int k = 0; k < 2; ++k) finish(acc[k], k, biasE[k]);
    } else {
        float* sums = lds + 4 * lane;           // [layer][other waves, in order][q][column]
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            if (g == k) continue;
            const int other = g < k ? g : g - 1;
#pragma unroll
            for (int c = 0; c < NCW; ++c) *(f32x4f*)(sums + (((k * (G - 1) + other) * Q + q) * NCW + c) * 256) = acc[k][c];
        }
        barrier();
        if (g < 2) {
            f32x4f sum[NCW];
#pragma unroll
            for (int c = 0; c < NCW; ++c) {
                const f32x4f* others = (const f32x4f*)(sums + ((g * (G - 1) * Q + q) * NCW + c) * 256);
                sum[c] = g == 0 ? acc[0][c] : acc[1][c];
#pragma unroll
                for (int o = 0; o < G - 1; ++o) sum[c] += others[o * Q * NCW * 64];
            }
            finish(sum, g, biasE[0]);
        }
    }
    if constexpr (!STORE) {
        barrier();
        const float* es = outs;                 // [output pixel][32*Q]
        if constexpr (POOL) {
            float* pooled = outs + 16 * NCW * RP;
            constexpr int CQ = 8 * Q;
#pragma unroll
            for (int i0 = 0; i0 < 16 * CQ; i0 += kFireThreads) {
                const int i = i0 + tid, px = i / CQ, c = i % CQ, p = px < bw * bh ? px : 0;
                if (16 * CQ < kFireThreads && px >= 16) break;
                const int py = small_div(p, mulBw);
                const float* from = outs + (2 * py * ew + 2 * (p - py * bw)) * RP + 4 * c;
                f32x4f m = {-3.402823466e+38f, -3.402823466e+38f, -3.402823466e+38f, -3.402823466e+38f};
#pragma unroll
                for (int dy = 0; dy < 3; ++dy)
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx) {
                        const f32x4f v = *(const f32x4f*)(from + (dy * ew + dx) * RP);
#pragma unroll
                        for (int k = 0; k < 4; ++k) m[k] = fmaxf(m[k], v[k]);
                    }
                *(f32x4f*)(pooled + px * RP + 4 * c) = m;
            }
            barrier();
            es = pooled;
        }
        // ---- squeeze: KP waves share the 2Q sixteens of expand channels of a sixteen of its own --------------------------
        f32x4f sq = {0.f, 0.f, 0.f, 0.f};
        const float* mine = es + l16 * RP + 16 * kp + 4 * lk;
        if (mb < MB && kp < 2 * Q) {
#pragma unroll
            for (int u = 0; u < 2 * Q; ++u) {
                if (u * KP >= 2 * Q) break;
                const f32x4f v = *(const f32x4f*)(mine + 16 * u * KP);
#pragma unroll
                for (int k = 0; k < 4; ++k) sq = __builtin_amdgcn_mfma_f32_16x16x4f32(a2[u][k], v[k], sq, 0, 0, 0);
            }
        }
        const int Wo = outWh & 0xffff, Ho = outWh >> 16, oy = small_div(l16, mulBw), ox = l16 - oy * bw;
        const int to = 4 * (((blockIdx.x * Ho + oy0 + oy) * Wo + ox0 + ox) * 16 * MB + 16 * mb + 4 * lk);
        const bool mineToStore = l16 < bw * bh && ox0 + ox < Wo && oy0 + oy < Ho;
        if (KP > 1) {
            float* sums = lds + 4 * lane;
            if (kp > 0 && mb < MB) *(f32x4f*)(sums + ((kp - 1) * MB + mb) * 256) = sq;
            barrier();
            if (kp == 0)
                for (int k = 0; k < KP - 1; ++k) sq += *(const f32x4f*)(sums + (k * MB + mb) * 256);
        }
        if (kp > 0 || mb >= MB) return;
        const __amdgpu_buffer_rsrc_t rOut = __builtin_amdgcn_make_buffer_rsrc((void*)out, 0, 0x7ffffff0, kBufferFlags);
        if (mineToStore) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4f, sq), rOut, to, 0, kAuxThrough16);
    }
}

struct FirePlan {
    int Q, bw, bh, ew, eh, hpx, nbx, nby, slices, S16, MB;
    size_t lds;
    int Wo, Ho;
    double clocks;
};

// The shape of a launch: the block of output pixels and the channels of a slice that take the fewest clocks.  A workgroup takes
// some 2500 clocks that do not depend on its shape; its matrix work, its filters and its patch (48 bytes a clock) add up, once for
// every workgroup on a CU, the first again when there are more of those than registers for them (4 of 16 squeeze channels,
// otherwise 2); and the reader loads every slice.  That picks among the shapes that measure best or within 4 % (us): 56x56 16->2x64->16
// 3.1 (Q = 4; 196 workgroups), 56x56 16->2x64->32 behind a pooling 4.4 (Q = 2; Q = 1 4.6), 28x28 32->2x128->48 behind one 4.9 (Q = 1,
// 8 slices; Q = 2 5.9), 14x14 64->2x256->64 5.5 (Q = 2, 8 slices; Q = 4 6.2), 29x19 64->2x256->64 6.1 (Q = 4), 128x128 16->2x64->16 5.6
// (1024 workgroups of 16 pixels; 256 of 64 pixels, which load a filter once for four columns, 6.3).
//
// rows: the expand outputs are stored in rows of a map.  Then a block's rows count too: each is a piece of a line for every channel, written through, some 7
// clocks each where there are many (85x96 12->2x128 stored from blocks of 1x16 pixels 36 us, from 8x2 8 us, and so the Winograd kernel behind
// a squeeze layer 10 us).  Only the block is chosen by that, the channels of a slice are those of the bank.
static bool fire_plan(int W, int H, int S, int E, int Sn, int pool, FirePlan* best, bool rows = false) {
    if (W < 1 || H < 1 || S < 1 || S > 64 || E < 32 || E % 32 != 0 || E > 2048 || Sn < 0 || Sn > 64 || (pool && Sn == 0)) return false;
    if (W > 16384 || H > 16384 || (long long)W * H * 64 >= (1ll << 26)) return false;
    const int S16 = ceil_div(S, 16), SP = 16 * S16, MB = ceil_div(Sn, 16), Wo = pool ? (W + 1) / 2 : W, Ho = pool ? (H + 1) / 2 : H;
    const int columns = fire_columns(pool), atOnce = kFireThreads * fire_quads(S16, pool), resident = S16 == 1 ? 4 : 2;
    auto search = [&](int firstQ, int lastQ, double clocksPerRow) {
        double least = 0;
        for (int Q = firstQ; Q <= lastQ; Q *= 2) {
            const int slices = E / 16 / Q;
            if (slices * 16 * Q != E || slices > 32 || (long long)Wo * Ho * 16 * std::max(MB, 1) * slices >= (1ll << 28)) continue;
            for (int bw = 1; bw <= (pool ? (kFireRow - 3) / 2 : kFireRow - 2); ++bw)
                for (int bh = 1; bw * bh <= 16; ++bh) {
                    const int ew = pool ? 2 * bw + 1 : bw, eh = pool ? 2 * bh + 1 : bh, hpx = (ew + 2) * (eh + 2), nbx = ceil_div(Wo, bw), nby = ceil_div(Ho, bh);
                    if (ew * eh > 16 * columns) break;
                    if (nbx > 65535 || nby > 65535) continue;
                    const double perCu = std::ceil((double)nbx * nby * slices / num_cu()), filters = (10 * S16 + 2 * MB) * Q * 1024 / 48.0;
                    // (the last two: smaller patches, and longer runs of addresses, where nothing else decides)
                    const double work = 320.0 * S16 * Q * columns + filters + ceil_div(hpx * SP / 4, atOnce) * atOnce * 64 / 48.0 + hpx * SP / 48.0 + 300.0 / bw + 32 * Q * bh * clocksPerRow;
                    const double cost = std::ceil(perCu / resident) * 2500 + perCu * work + slices * 36 * 16 * MB * 4 / 48.0 + std::max(0, slices - kFireSlices) * 900.0;
                    if (least != 0 && cost >= least) continue;
                    const size_t lds = (size_t)(fire_sums(Q, pool) + (Sn > 0 ? fire_outs(Q, pool) : 0) + (eh + 2) * kFireRow * (SP + 4)) * sizeof(float);
                    least = cost;
                    *best = FirePlan{Q, bw, bh, ew, eh, hpx, nbx, nby, slices, S16, MB, lds, Wo, Ho, cost};
                }
        }
        return least != 0;
    };
    return search(pool ? 1 : 2, 4, 0.0) && (!rows || search(best->Q, best->Q, 7.0));
}

struct FireCall { const float *in, *bank, *inBias; float* out; unsigned wh, block, misc, outWh; hipStream_t st; };

template <int S16, int Q, bool POOL, bool STORE, bool PLAIN>
static int launch_fire(const FirePlan& p, const FireCall& c) {
    static std::atomic<unsigned long long> asked{0};
    if (int rc = allow_lds((const void*)fire_kernel<S16, Q, POOL, STORE, PLAIN>, p.lds, asked)) return rc;
    launch((fire_kernel<S16, Q, POOL, STORE, PLAIN>), dim3(p.slices, p.nbx, p.nby), dim3(kFireThreads), p.lds, c.st, c.in, c.bank, c.wh, c.block, c.misc,
           small_mul(p.ew + 2), c.inBias, small_mul(p.hpx), small_mul(p.ew), small_mul(p.bw), c.outWh, c.out);
    return launched("fire_kernel");
}
template <int S16>
static int launch_fire_s(const FirePlan& p, const FireCall& c, bool pool, bool store, bool plain) {
    if (pool)
        return p.Q == 1 ? launch_fire<S16, 1, true, false, false>(p, c) : p.Q == 2 ? launch_fire<S16, 2, true, false, false>(p, c) : launch_fire<S16, 4, true, false, false>(p, c);
    if (store) return p.Q == 2 ? launch_fire<S16, 2, false, true, false>(p, c) : launch_fire<S16, 4, false, true, false>(p, c);
    if (plain) return p.Q == 2 ? launch_fire<S16, 2, false, false, true>(p, c) : launch_fire<S16, 4, false, false, true>(p, c);
    return p.Q == 2 ? launch_fire<S16, 2, false, false, false>(p, c) : launch_fire<S16, 4, false, false, false>(p, c);
}

}  // namespace drhip

using namespace drhip;

extern "C" int drhip_fire_slices(int W, int H, int S, int E, int Sn, int pool) {
    FirePlan p;
    return fire_plan(W, H, S, E, Sn, pool, &p) ? p.slices : 0;
}

// What the launches of a module take in a pass, us, for the choice between them: the launch above from the clocks of its plan, the others from the
// products they do and the numbers they move (the Winograd kernels store maps of odd width less well).  Fitted to 330 shapes, maps of 13x13 to 320x320, 16 to 64
// channels to 2x32 to 2x1024: half of them come out within 6 %, nine of ten within 17 %.  The launch above is put 3 % lower, which lost least.
// On 450 random networks of one to six modules the choice is 0.8 % slower than the better side on average and 14 % at most, always taking the next layer
// along 0.8 and 19 %, never doing so 19 and 94 %; runs of four alike modules, us apart / chosen / always along: 112x112 64->2x256 214 / 214 / 249, 80x80
// 32->2x1024 242 / 240 / 382, 56x56 64->2x256 83 / 82 / 90, 28x28 64->2x256 46 / 38 / 38; left on the slower side: 64x64 64->2x256 87 / 95 / 95.
extern "C" float drhip_fire_us(int W, int H, int S, int E, int Sn, int pool, int slicesIn) {
    FirePlan p;
    if (!fire_plan(W, H, S, E, Sn, pool, &p)) return 0.0f;
    const int perCu = ceil_div(p.nbx * p.nby * p.slices, num_cu());
    const double us = p.clocks / 2400;
    // (every workgroup adds up all slices of its patch: with sixteen of them 10 to 30 us of 50 to 100 on large maps)
    const double patches = std::max(0.0, 16.0 * p.S16 * 4 / 48 / 2400 * p.hpx * slicesIn * perCu - 2);
    return 0.97f * (float)(pool ? 1.6 + 1.12 * us + patches : Sn > 0 ? 2.1 + (0.73 + 0.06 * p.S16) * us + 1.8 * patches : 1.95 + 0.89 * us + 1.8 * patches);
}
// (An expand pair apart is a launch in three bf16 parts or in fp32: with a 1x1 layer riding along it never is one in two f16 parts.)
extern "C" float drhip_fire_expand_us(int W, int H, int S, int E) {
    const double mpxE = 1e-6 * W * H * E;
    if (drhip_conv3x3_winograd_split_pick_variant(W, H, S, 2 * E)) return (float)(5.4 + (W & 1 ? 5.4 : 2.9) * mpxE + 0.094 * mpxE * S + 0.000009 * E * S);
    const int variant = drhip_conv3x3_winograd_pick_variant(W, H, S, 2 * E);
    const double second = (variant & 0xf0) != 0 && (variant & 0x800) == 0 ? 3.5 : 0.0;          // (a kernel that adds up splits)
    return (float)(3.7 + second + (W & 1 ? 4.6 : 1.7) * mpxE + 0.186 * mpxE * S + 0.00001 * E * S);
}
extern "C" float drhip_fire_squeeze_us(int W, int H, int C, int Sn, int pool) {
    const double mpx = 1e-6 * W * H;
    return (float)(pool ? 2.5 + 0.89 * mpx * C + 0.035 * mpx * C * Sn + 0.000114 * C * Sn : 2.8 + 0.63 * mpx * C + 0.026 * mpx * C * Sn + 0.000024 * C * Sn);
}

extern "C" size_t drhip_fire_bank_floats(int W, int H, int S, int E, int Sn, int pool) {
    FirePlan p;
    return fire_plan(W, H, S, E, Sn, pool, &p) ? (size_t)p.slices * fire_slice_bytes(p.S16, p.Q, p.MB) / 4 : 0;
}

extern "C" size_t drhip_fire_partials_floats(int W, int H, int S, int E, int Sn, int pool) {
    FirePlan p;
    return fire_plan(W, H, S, E, Sn, pool, &p) && Sn > 0 ? (size_t)p.slices * p.Wo * p.Ho * 16 * p.MB : 0;
}

// On the host: the banks of a network are some hundred thousand numbers, laid out once.
extern "C" int drhip_fire_layout_f32(const float* w1, const float* w3, const float* b1, const float* b3, const float* wn, float* bank,
                                     int W, int H, int S, int E, int Sn, int pool) {
    DRHIP_REQUIRE(w1 && w3 && bank && (wn || Sn == 0), "drhip_fire_layout_f32: NULL array");
    FirePlan p;
    DRHIP_REQUIRE(fire_plan(W, H, S, E, Sn, pool, &p), "drhip_fire_layout_f32: %dx%d, %d -> 2 x %d -> %d is not covered", W, H, S, E, Sn);
    // By rows of the filters: nine taps in a row, whose places in a slice are those of the items plus one for the channel and the output.
    const int Q = p.Q, G = 4 / Q, KS = 4 / G, S16 = p.S16, MB = p.MB, sliceFloats = fire_slice_bytes(S16, Q, MB) / 4;
    memset(bank, 0, (size_t)p.slices * sliceFloats * sizeof(float));
    int item[40];
    for (int i = 0; i < 10 * S16; ++i) item[i] = i / G * 1024 + i % G * KS;
    for (int c = 0; c < S; ++c) {
        const int in16 = c / 16, at0 = c % 4 / KS * 256 + c % 16 / 4 * 64 + c % 4 % KS;
        for (int o = 0; o < E; ++o) {
            const float* f = w3 + ((size_t)c * E + o) * 9;
            float* d = bank + (size_t)(o / (16 * Q)) * sliceFloats + at0 + o / 16 % Q * G * 256 + o % 16 * 4;
            for (int tap = 0; tap < 9; ++tap) d[item[tap * S16 + in16]] = f[tap];
            d[item[9 * S16 + in16]] = w1[(size_t)c * E + o];
        }
    }
    const int packs = fire_packs(S16, Q) * 1024;
    for (int row = 0; row < (Sn > 0 ? 2 * E : 0); ++row) {
        const int c = row % E, e = row / E * Q + c / 16 % Q;
        float* d = bank + (size_t)(c / (16 * Q)) * sliceFloats + packs + (size_t)e * MB * 256 + c % 16 / 4 * 64 + c % 4;
        for (int o = 0; o < Sn; ++o) d[o / 16 * 256 + o % 16 * 4] = wn[(size_t)row * Sn + o];
    }
    for (int c = 0; c < E; ++c) {
        float* d = bank + (size_t)(c / (16 * Q)) * sliceFloats + packs + 2 * Q * MB * 256 + c % (16 * Q);
        if (b1) d[0] = b1[c];
        if (b3) d[16 * Q] = b3[c];
    }
    return DRHIP_OK;
}

extern "C" int drhip_fire_f32(const float* in, int slicesIn, const float* inBias, int inRelu, const float* bank, float* out,
                              int W, int H, int S, int E, int Sn, int pool, int relu, int pixels, void* stream) {
    DRHIP_REQUIRE(in && bank && out, "drhip_fire_f32: NULL tensor");
    DRHIP_REQUIRE(slicesIn >= 0 && slicesIn <= 32, "drhip_fire_f32: %d slices", slicesIn);
    DRHIP_REQUIRE(slicesIn > 0 || (Sn > 0 && !pool), "drhip_fire_f32: a plain input is not covered where the expand outputs are stored or pooled");
    DRHIP_REQUIRE(!pixels || (Sn == 0 && (long long)W * H * 2 * E < (1ll << 28)), "drhip_fire_f32: [H][W][2E] is for expand outputs of less than 1 GiB");
    DRHIP_REQUIRE((((size_t)bank | (size_t)(slicesIn > 0 ? in : nullptr) | (size_t)(slicesIn > 0 ? inBias : nullptr) | (size_t)(Sn > 0 || pixels ? out : nullptr)) & 15) == 0,
                  "drhip_fire_f32: banks, partial sums, their bias and outputs by pixel need 16-byte alignment");
    FirePlan p;
    DRHIP_REQUIRE(fire_plan(W, H, S, E, Sn, pool, &p, Sn == 0 && !pixels), "drhip_fire_f32: %dx%d, %d -> 2 x %d -> %d is not covered", W, H, S, E, Sn);
    DRHIP_REQUIRE((long long)slicesIn * W * H * 16 * p.S16 < (1ll << 29), "drhip_fire_f32: %d slices of %dx%dx%d are too large", slicesIn, W, H, S);
    FireCall c = {in, bank, inBias, out, 0, 0, 0, 0, as_stream(stream)};
    c.wh = (unsigned)(W | H << 16);
    c.block = (unsigned)(p.bw | p.bh << 8 | p.ew << 16) | (unsigned)(p.ew * p.eh) << 24;
    c.misc = (unsigned)(p.hpx | S << 8 | slicesIn << 16) | (inRelu ? 1u << 24 : 0u) | (relu ? 1u << 25 : 0u) | (unsigned)p.MB << 26 | (p.MB > 2 ? 2u : p.MB > 1 ? 1u : 0u) << 29;
    c.outWh = Sn > 0 ? (unsigned)(p.Wo | p.Ho << 16) : (unsigned)E | (pixels ? 1u << 31 : 0u);
    switch (p.S16) {
        case 1: return launch_fire_s<1>(p, c, pool != 0, Sn == 0, slicesIn == 0);
        case 2: return launch_fire_s<2>(p, c, pool != 0, Sn == 0, slicesIn == 0);
        case 3: return launch_fire_s<3>(p, c, pool != 0, Sn == 0, slicesIn == 0);
        default: return launch_fire_s<4>(p, c, pool != 0, Sn == 0, slicesIn == 0);
    }
}
