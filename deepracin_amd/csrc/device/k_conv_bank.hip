// Convolution with any odd filter and any stride as an implicit GEMM on the bf16 matrix cores, at fp32 accuracy (see
// bf16x3.hpp): everything that is neither 3x3/stride 1 (Winograd) nor 1x1 (GEMM), such as 7x7/2 first layers and 5x5
// layers.
//
//   out[o][p] = act(b[o] + sum over k-steps of F[k][o] . in[k][pixel p shifted by the step's tap])
//
// What bounds it: the matrix cores on large layers (2 * 6 * Ho*Wo * I*O*kh*kw FLOP of bf16 MFMA), one workgroup's chain
// of staging, matrix steps and store on small ones; figures stand at the choice of the tile.
//
// A workgroup owns a tile of 32*MT output pixels and 32*WO output channels:
//   * The input patch under the tile is staged in LDS, 16 to 128 channels at a time, zero padding included, ALREADY SPLIT into
//     its three bf16 parts and with the eight channels an MFMA lane wants next to each other: inside the tap loop a
//     B operand is one 16-byte LDS read whatever the tap (a tap is an address offset), and there is no vector arithmetic at all.
//     Reading the samples from global memory per tap would cost a dword gather and a split per sample and tap, 25 times
//     for a 5x5 filter.  The next stage's are fetched into registers while the taps run and go to the other half of LDS.
//   * The filters come from a bank laid out and split once, when the layer is prepared, so that an A operand is one 16-byte
//     buffer load per lane and 1 KiB in a row per wave.  Every wave reads only its own 32 channels, several steps ahead.
//   * Two, four or eight waves share the k-steps of a stage and 32 output channels round-robin and meet in LDS at the end, in wave order: layers with
//     few tiles fill the chip that way without a second kernel.
//   * A 2x2/2 max pooling behind the layer is taken from these sums: a pooled pixel a lane.  (28x28 with 5x5 filters and poolings, 16
//     and 32 channels, its image from the host and its results back: 36.4 -> 32.2 us, two launches less.)
//   * So is a 3x3/2 max pooling (P3): the pixels of a workgroup are then the 9x7 or 9x9 under 4x3 or 4x4 pooled ones, in two or three
//     blocks of 32, so that 1.33 or 1.5 times the products are done, and one launch less and a quarter of the outputs stored.  (Figures stand at the choice of the variant.)
//   * Outputs that do not come out finite are worked out again in fp32, at the end.
// Layers with at most four input channels (images) put four neighbouring pixels x four channels into one step of 16 k
// (CP = 4) instead of 16 channels of one pixel, most of which would be zero: a 7x7 filter over RGB is 14 steps, not 49.
#include "bf16x3.hpp"

#include <algorithm>
#include <cfloat>
#include <type_traits>

namespace drhip {

constexpr int kBankThreads = 512;                       // eight waves: two per SIMD, one reads and counts while the other multiplies
// P3: 4 x 3 (two blocks) or 4 x 4 (three) pooled pixels of a workgroup, 9 columns of pixels under them, and what lgBW says then
constexpr int kP3X = 4, kP3W = 2 * kP3X + 1, kP3Tile = 6;
constexpr int p3_rows(int mt) { return mt + 1; }

struct BankShape {                                      // everything but the pointers; by value to the kernel
    int W, H, I, O, Wo, Ho;
    int kw, sx, sy, padX, padY;
    int lgBW;                                           // 32 pixels of one MFMA = 2^lgBW columns x the rest rows (kP3Tile: see there)
    int pw, patchN;                                     // patch width, patch pixels
    int spr, steps, nChunks, oBlocks;                   // k-steps per filter row, per chunk; chunks; 32-channel blocks in the bank
    int group, nStages;                                 // chunks that are staged together; stages
    unsigned pwMul, pwShift, patchMul, patchShift;      // division by pw and patchN
    unsigned sprMul, stepsMul;                          // j = tap * sprMul >> 16, chunk of a stage = step * stepsMul >> 16
    int relu, pool;                                     // pool: a 2x2/2 (with P3: 3x3/2) max pooling stands behind the layer, `out` is its tensor
};

__device__ inline u32x4b bank_load4(__amdgpu_buffer_rsrc_t r, unsigned voffset, unsigned soffset) {
    return __builtin_bit_cast(u32x4b, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voffset, (int)soffset, 0));
}

// F[chunk][step][part][o/32][lane][8] (bf16) from w[c][o][kh][kw]: lane l of a wave holds output channel o = l%32 and
// the values k = 8*(l/32) .. +7 of the step.  CP = 16: k is the channel within the chunk, the step a tap.  CP = 4: k is
// (pixel within a group of four, channel).  What does not exist is zero.
__global__ void __launch_bounds__(256)
conv_bank_layout_kernel(const float* __restrict__ w, unsigned short* __restrict__ F, int I, int O, int kw, int kh, int cp, int spr, int steps, int nChunks, int oBlocks) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;          // (chunk, step, oblock, lane, e)
    const size_t total = (size_t)nChunks * steps * oBlocks * 512;
    if (idx >= total) return;
    const int e = (int)(idx & 7), lane = (int)((idx >> 3) & 63);
    const size_t rest = idx >> 9;
    const int ob = (int)(rest % oBlocks);
    const int step = (int)(rest / oBlocks % steps), chunk = (int)(rest / oBlocks / steps);
    const int k = 8 * (lane >> 5) + e, o = 32 * ob + (lane & 31);
    const int j = step / spr;
    const int c = cp == 16 ? 16 * chunk + k : (k & 3), i = cp == 16 ? step % spr : 4 * (step % spr) + (k >> 2);
    const float v = (c < I && o < O && i < kw) ? w[(((size_t)c * O + o) * kh + j) * kw + i] : 0.0f;
    unsigned short part[3];
    split_one(v, part);
#pragma unroll
    for (int q = 0; q < 3; ++q) F[((((size_t)chunk * steps + step) * 3 + q) * oBlocks + ob) * 512 + lane * 8 + e] = part[q];
}

// PF: staging rounds (512 units each) of the next stage that are kept in registers.
template <int CP, int MT, int WO, int WK, int PF, bool P3>
__global__ void __launch_bounds__(kBankThreads)
conv_bank_mfma_kernel(const float* __restrict__ in, const unsigned short* __restrict__ F, const float* __restrict__ bias,
                      float* __restrict__ out, BankShape s) {
    static_assert(WO * WK * 64 == kBankThreads, "eight waves");
    static_assert(CP == 4 || CP == 16, "channels of one pixel in a k-step");
    constexpr int kP3Y = p3_rows(MT), kP3H = 2 * kP3Y + 1;
    static_assert(!P3 || (MT >= 2 && kP3W * kP3H <= 32 * MT), "the pixels under a tile of pooled ones");
    constexpr int kGroups = CP == 16 ? 2 : 1;           // staging units per pixel, 8 (4) channels each
    constexpr int kUnitBytes = CP == 16 ? 16 : 8;
    __shared__ float biasT[32 * WO];                    // (a load in the epilogue would wait for the stores in front of it)
    constexpr int kDepth = 4;                           // k-steps whose filters are in flight (even: two operand buffers alternate)
    extern __shared__ __attribute__((aligned(16))) char lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wo = wave % WO, wk = wave / WO;
    const int l32 = lane & 31, half = lane >> 5;
    const int BW = 1 << s.lgBW, BH = 32 >> s.lgBW;
    const int x0 = P3 ? blockIdx.x * (2 * kP3X) : blockIdx.x << s.lgBW, y0 = blockIdx.y * (P3 ? 2 * kP3Y : BH * MT);
    const int ob = blockIdx.z * WO + wo;                // this wave's 32 output channels
    const int bx = l32 & (BW - 1), by = l32 >> s.lgBW;
    const int plane = s.H * s.W;

    // ---- staging: unit u -> (channel group, patch pixel); a unit is 8 (4) channels of one pixel, split ----------------
    const int units = s.patchN * kGroups * s.group;
    const int rounds = (units + kBankThreads - 1) / kBankThreads;
    const int partBytes = (units * kUnitBytes + 15) & ~15;
    const int bufBytes = 3 * partBytes;
    const FastDiv pwd = {(unsigned)s.pw, s.pwMul, s.pwShift}, patchd = {(unsigned)s.patchN, s.patchMul, s.patchShift};
    const int px0 = x0 * s.sx - s.padX, py0 = y0 * s.sy - s.padY;
    constexpr int kUC = CP == 16 ? 8 : 4;               // channels of a unit
    auto unit_offset = [&](int u, unsigned& off) {
        const int grp = kGroups == 2 ? fast_div(u, patchd) : 0, q = u - grp * s.patchN;
        const int py = fast_div(q, pwd), px = q - py * s.pw;
        const int ix = px0 + px, iy = py0 + py;
        const bool ok = u < units && ix >= 0 && ix < s.W && iy >= 0 && iy < s.H;
        off = ok ? 4u * (unsigned)(grp * 8 * plane + iy * s.W + ix) : kOutOfRange;
    };
    auto load_unit = [&](float (&v)[kUC], unsigned off, int stage) {
#pragma unroll
        for (int q = 0; q < kUC; ++q) {                 // (channels past the last one: a resource that ends in front of them)
            const int c = stage * s.group * 16 + q, left = max(s.I - c, 0);
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)(in + (size_t)min(c, s.I) * plane), 0, left * plane * 4, kBufferFlags);
            v[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
        }
    };
    auto store_unit = [&](char* buf, const float (&v)[kUC], int u) {
        if (u >= units) return;
        Bf16Pair3 p[kUC / 2];
#pragma unroll
        for (int q = 0; q < kUC / 2; ++q) p[q] = split_pair(kSplitScale * v[2 * q], kSplitScale * v[2 * q + 1]);
        char* d = buf + u * kUnitBytes;
        if constexpr (CP == 16) {
            *(u32x4b*)d = u32x4b{p[0].hi, p[1].hi, p[2].hi, p[3].hi};
            *(u32x4b*)(d + partBytes) = u32x4b{p[0].mid, p[1].mid, p[2].mid, p[3].mid};
            *(u32x4b*)(d + 2 * partBytes) = u32x4b{p[0].lo, p[1].lo, p[2].lo, p[3].lo};
        } else {
            *(u32x2b*)d = u32x2b{p[0].hi, p[1].hi};
            *(u32x2b*)(d + partBytes) = u32x2b{p[0].mid, p[1].mid};
            *(u32x2b*)(d + 2 * partBytes) = u32x2b{p[0].lo, p[1].lo};
        }
    };

    // ---- filters: the steps of this wave, wk, wk + WK, ..., -------------------------------------
    const int allSteps = s.nChunks * s.steps;
    const int bankBytes = allSteps * 3 * s.oBlocks * 1024;
    const __amdgpu_buffer_rsrc_t rF = __builtin_amdgcn_make_buffer_rsrc((void*)F, 0, bankBytes, kBufferFlags);
    const unsigned fLane = ob < s.oBlocks ? (unsigned)(ob * 1024 + lane * 16) : kOutOfRange;    // (a wave without channels multiplies zeros)
    auto load_filters = [&](u32x4b (&f)[3], int step) {     // (of the whole layer)
#pragma unroll
        for (int q = 0; q < 3; ++q) f[q] = bank_load4(rF, fLane, (unsigned)((min(step, allSteps - 1) * 3 + q) * s.oBlocks) * 1024u);
    };
    u32x4b f[kDepth][3];
#pragma unroll
    for (int g = 0; g < kDepth; ++g) load_filters(f[g], wk + g * WK);

    unsigned off[PF];
    float raw[PF][kUC];
#pragma unroll
    for (int r = 0; r < PF; ++r) {
        unit_offset(tid + kBankThreads * r, off[r]);
        load_unit(raw[r], off[r], 0);
    }
    if (tid < 32 * WO) biasT[tid] = bias ? bias[min((int)blockIdx.z * 32 * WO + tid, s.O - 1)] : 0.0f;
    // what of the patch does not fit the prefetch registers is loaded when it is stored
    auto stage = [&](char* buf, int n) {
#pragma unroll
        for (int r = 0; r < PF; ++r) store_unit(buf, raw[r], tid + kBankThreads * r);
        for (int r = PF; r < rounds; ++r) {
            unsigned o;
            float v[kUC];
            unit_offset(tid + kBankThreads * r, o);
            load_unit(v, o, n);
            store_unit(buf, v, tid + kBankThreads * r);
        }
    };

    // MT = 1 keeps three accumulators, so that the MFMAs of a step do not wait for each other
    constexpr int NA = MT == 1 ? 3 : 1;
    f32x16b acc[MT][NA];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[m][a][r] = 0.0f;

    // byte offset of this lane's operand for tap (0, 0), per 32-pixel block
    int bBase[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int p3 = min(32 * m + l32, kP3W * kP3H - 1);
        const int q = P3 ? (p3 / kP3W) * s.sy * s.pw + (p3 % kP3W) * s.sx : (by + BH * m) * s.sy * s.pw + bx * s.sx;
        bBase[m] = CP == 16 ? (half * s.patchN + q) * 16 : q * 8 + half * 16;
    }

    stage(lds, 0);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");

    auto read_operands = [&](const char* buf, u32x4b (&b)[MT][3], int step) {
        const int c = CP == 16 ? (int)(((unsigned)step * s.stepsMul) >> 16) : 0, tap = step - c * s.steps;
        const int j = (int)(((unsigned)tap * s.sprMul) >> 16), i = tap - j * s.spr;
        const char* at = buf + (CP == 16 ? (2 * c * s.patchN + j * s.pw + i) * 16 : (j * s.pw + 4 * i) * 8);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const char* p = at + q * partBytes + bBase[m];
                if constexpr (CP == 16) b[m][q] = *(const u32x4b*)p;
                else {
                    const u32x2b lo = *(const u32x2b*)p, hi = *(const u32x2b*)(p + 8);
                    b[m][q] = u32x4b{lo[0], lo[1], hi[0], hi[1]};
                }
            }
    };
    auto multiply = [&](const u32x4b (&fs)[3], const u32x4b (&b)[MT][3]) {
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m][q % NA] = mfma_bf16(fs[kProdA[q]], b[m][kProdB[q]], acc[m][q % NA]);
    };

    for (int n0 = 0; n0 < s.nStages; ++n0) {
        const char* buf = lds + (n0 & 1) * bufBytes;
        const bool more = n0 + 1 < s.nStages;
        const int first = n0 * s.group * s.steps, steps = min(s.group * s.steps, allSteps - first), mySteps = wk < steps ? (steps - wk + WK - 1) / WK : 0;
        if (more) {
#pragma unroll
            for (int r = 0; r < PF; ++r) load_unit(raw[r], off[r], n0 + 1);
        }
        // A step's operands are read from LDS while the step in front of it multiplies (a wave is often alone on its SIMD, and
        // a trip to LDS is as long as six MFMAs); its filters were requested kDepth steps ago.  The loads of a group go
        // out whether or not the steps exist, so that the number of loads in flight is known where it is waited for.
        u32x4b b[2][MT][3];
        read_operands(buf, b[0], min(wk, steps - 1));                   // (a wave may have no step at all)
        for (int n = 0; n < mySteps; n += kDepth) {
#pragma unroll
            for (int g = 0; g < kDepth; ++g) {
                const int t = n + g;
                if (t < mySteps) {
                    read_operands(buf, b[(g + 1) & 1], wk + min(t + 1, mySteps - 1) * WK);
                    multiply(f[g], b[g & 1]);
                }
                // the step that takes this slot next: kDepth on, or the slot's first one in the next stage
                load_filters(f[g], first + wk + (t + kDepth < mySteps ? (t + kDepth) * WK : s.group * s.steps + g * WK));
            }
        }
        if (more) {
            stage(lds + ((n0 + 1) & 1) * bufBytes, n0 + 1);             // (read last before the barrier in front of this stage)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        }
    }

    // D of the 32x32 MFMA: lane -> pixel lane%32; register r -> channel 8*(r/4) + 4*(lane/32) + r%4
    const int P = s.Wo * s.Ho;
    if constexpr (NA > 1) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[m][0][r] = (acc[m][0][r] + acc[m][1][r]) + acc[m][2][r];
    }
    constexpr int kPitch = 33;
    float* part = (float*)lds;                          // [WK][32*WO channels][MT][33]
    auto barrier = [] {                                 // (LDS only)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    __syncthreads();                                    // the patch has been read for the last time
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            part[((wk * 32 * WO + 32 * wo + 8 * (r / 4) + 4 * half + r % 4) * MT + m) * kPitch + l32] = acc[m][0][r];
    __syncthreads();
    unsigned again = 0;                                 // turns whose output did not come out finite
    auto finish = [&](float v, float scale, float b) {
        v = fmaf(v, scale, b);
        return s.relu ? fmaxf(v, 0.0f) : v;
    };
    // The sum at pixel (x, y) of the map for channel oc of the workgroup: CH channels side by side, 64 / CH lanes for each.
    // (kh by the caller, once: the division is not for every output)
    auto once_more = [&](auto channels, int kh, int x, int y, int oc) {
        constexpr int CH = decltype(channels)::value;
        const int o = blockIdx.z * (32 * WO) + oc;
        const unsigned fAgain = (unsigned)(min(o >> 5, s.oBlocks - 1) * 1024 + (o & 31) * 16);
        const int left = x * s.sx - s.padX, top = y * s.sy - s.padY;
        for (int j = 0; j < kh; ++j) {
            bool nan = false;
            const float* row = in + (size_t)min(max(top + j, 0), s.H - 1) * s.W;        // (a row beside the map stands for one that is in the window)
            for (int c = lane; c < s.I; c += 64)
                for (int i = 0; i < s.kw; ++i) {
                    const float v = row[(size_t)c * plane + min(max(left + i, 0), s.W - 1)];
                    nan = nan || v != v;
                }
            if (__builtin_amdgcn_ballot_w64(nan) != 0) return __builtin_nanf("");
        }
        // (its instructions bound this, not its loads: one offset for the samples of a position, and channels that do not exist end the resource)
        const __amdgpu_buffer_rsrc_t rAll = __builtin_amdgcn_make_buffer_rsrc((void*)in, 0, s.I * plane * 4, kBufferFlags);
        float v = 0.0f;
        for (int chunk = 0; chunk < s.nChunks; ++chunk)
            for (int u = lane / CH; u < 2 * s.steps; u += 64 / CH) {            // half a k-step: eight values of k
                const int step = u >> 1, h = u & 1, j = (int)(((unsigned)step * s.sprMul) >> 16), i0 = step - j * s.spr;
                const unsigned f = fAgain + (unsigned)((chunk * s.steps + step) * 3 * s.oBlocks * 1024 + 512 * h), partF = (unsigned)s.oBlocks * 1024u;
                const u32x4b hi = bank_load4(rF, f, 0), mid = bank_load4(rF, f + partF, 0), lo = bank_load4(rF, f + 2 * partF, 0);
                constexpr int G = CP == 16 ? 1 : 2;     // positions of eight values
                bool ok[G];
                float sample[8];
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const int i = CP == 16 ? i0 : 4 * i0 + 2 * h + g, ix = left + i, iy = top + j;
                    ok[g] = i < s.kw && ix >= 0 && ix < s.W && iy >= 0 && iy < s.H;
                    const int at = 4 * ((CP == 16 ? (16 * chunk + 8 * h) * plane : 0) + iy * s.W + ix);
#pragma unroll
                    for (int e = 0; e < 8 / G; ++e) sample[8 / G * g + e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rAll, (ok[g] ? at : 0) + 4 * e * plane, 0, 0));
                }
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    float w = v;
#pragma unroll
                    for (int e = 8 / G * g; e < 8 / G * (g + 1); ++e) {
                        auto of = [&](u32x4b q) { return e & 1 ? q[e / 2] >> 16 : q[e / 2] & 0xffffu; };
                        w = fmaf(whole(of(hi), of(mid), of(lo)), sample[e], w);
                    }
                    v = ok[g] ? w : v;
                }
            }
#pragma unroll
        for (int k = CH; k < 64; k *= 2) v += __shfl_xor(v, k);
        return v;
    };
    if constexpr (P3) {
        // Outputs first, each in the place of its first sum, zeros beside the map; then the pooling, by its own kernel's rules.  (A turn is 16
        // channels of one block: no division.)
        constexpr int NT = 2 * WO * MT;
        float* const mine = part + (tid >> 5) * MT * kPitch + l32;
        auto block_of = [](int n) { return n / (2 * WO); };
        auto first_of = [](int n) { return 16 * (n % (2 * WO)); };         // channel, less tid / 32
        float v[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            v[n] = 0.0f;
#pragma unroll
            for (int k = 0; k < WK; ++k) v[n] += mine[((k * 32 * WO + first_of(n)) * MT + block_of(n)) * kPitch];
            again |= fabsf(v[n]) < __builtin_inff() ? 0u : 1u << n;
            v[n] = finish(v[n], kSplitUnscale, biasT[first_of(n) + (tid >> 5)]);
        }
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(again != 0u) != 0, 0)) {       // (as below, output by output)
            const int kh = s.steps / s.spr;
#pragma unroll
            for (int n = 0; n < NT; ++n)
                for (unsigned long long bad = __builtin_amdgcn_ballot_w64((again >> n & 1u) != 0); bad != 0; bad &= bad - 1) {
                    const int src = __builtin_ctzll(bad), oc = first_of(n) + ((tid & ~63) + src) / 32, pl = 32 * block_of(n) + (src & 31);
                    const int x = x0 + pl % kP3W, y = y0 + pl / kP3W;
                    if (pl >= kP3W * kP3H || x >= s.Wo || y >= s.Ho) continue;
                    const float once = finish(once_more(std::integral_constant<int, 1>{}, kh, x, y, oc), 1.0f, biasT[oc]);
                    v[n] = lane == src ? once : v[n];
                }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int pl = 32 * m + l32;
            const bool inMap = x0 + pl % kP3W < s.Wo && y0 + pl / kP3W < s.Ho;
#pragma unroll
            for (int n = 2 * WO * m; n < 2 * WO * (m + 1); ++n) mine[(first_of(n) * MT + m) * kPitch] = inMap ? v[n] : 0.0f;
        }
        barrier();
        const int Wp = (s.Wo + 1) >> 1, Hp = (s.Ho + 1) >> 1;
#pragma unroll
        for (int i0 = 0; i0 < 32 * WO * kP3X * kP3Y; i0 += kBankThreads) {
            const int i = i0 + tid, oc = i / (kP3X * kP3Y), pp = i % (kP3X * kP3Y), ppy = pp / kP3X, ppx = pp % kP3X;
            if (32 * WO * kP3X * kP3Y < i0 + kBankThreads && oc >= 32 * WO) break;
            float best = -FLT_MAX;
#pragma unroll
            for (int d = 0; d < 9; ++d) {
                const int q = (2 * ppy + d / 3) * kP3W + 2 * ppx + d % 3;
                const float u = part[(oc * MT + (q >> 5)) * kPitch + (q & 31)];
                best = u > best ? u : best;
            }
            const int o = blockIdx.z * (32 * WO) + oc, px = (x0 >> 1) + ppx, py = (y0 >> 1) + ppy;
            if (o < s.O && px < Wp && py < Hp) store_through(out + ((size_t)o * Hp + py) * Wp + px, best);
        }
        return;
    }
    // Pooled: 512 lanes, 64 (channel, block) pairs of 8 pooled pixels a turn.  The maximum as the pooling's own kernel takes it: in scan
    // order from the lowest number on, what lies beside the map counts as 0.
    constexpr int kPooled = WO * MT / 2 > 0 ? WO * MT / 2 : 1;
    const int px2 = tid & ((BW >> 1) - 1), py2 = (tid & 7) >> (s.lgBW - 1), Wp = (s.Wo + 1) >> 1, Pp = Wp * ((s.Ho + 1) >> 1);
    auto pooled_of = [&](int n, int& oc, int& x, int& y) {
        const int pair = 64 * n + (tid >> 3), m = pair % MT;
        oc = pair / MT; x = x0 + 2 * px2; y = y0 + 2 * py2 + BH * m;
        return ((oc * MT) + m) * kPitch + 2 * py2 * BW + 2 * px2;
    };
    auto larger = [](float best, float v) { return v > best ? v : best; };
    if (s.pool) {
#pragma unroll
        for (int n = 0; n < kPooled; ++n) {
            int oc, x, y;
            const int at = pooled_of(n, oc, x, y);
            if (oc >= 32 * WO) break;                   // (a single block for half of the lanes)
            const int o = blockIdx.z * (32 * WO) + oc;
            float best = -FLT_MAX;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = 0.0f;
#pragma unroll
                for (int k = 0; k < WK; ++k) v += part[k * 32 * WO * MT * kPitch + at + (e & 1) + (e >> 1) * BW];
                again |= fabsf(v) < __builtin_inff() ? 0u : 1u << n;
                best = larger(best, x + (e & 1) < s.Wo && y + (e >> 1) < s.Ho ? finish(v, kSplitUnscale, biasT[oc]) : 0.0f);
            }
            if (o < s.O && x < s.Wo && y < s.Ho) store_through(out + (size_t)o * Pp + (size_t)(y >> 1) * Wp + (x >> 1), best);
        }
    } else
#pragma unroll
    for (int n = 0; n < 2 * WO * MT; ++n) {             // 512 lanes: 16 (channel, block) pairs of 32 pixels a turn
        const int pair = 16 * n + (tid >> 5), m = pair % MT, oc = pair / MT, pl = tid & 31;
        float v = 0.0f;
#pragma unroll
        for (int k = 0; k < WK; ++k) v += part[((k * 32 * WO + oc) * MT + m) * kPitch + pl];
        again |= fabsf(v) < __builtin_inff() ? 0u : 1u << n;
        const int o = blockIdx.z * (32 * WO) + oc;
        const int x = x0 + (pl & (BW - 1)), y = y0 + (pl >> s.lgBW) + BH * m;
        v = finish(v, kSplitUnscale, biasT[oc]);
        if (o < s.O && x < s.Wo && y < s.Ho) store_through(out + (size_t)o * P + (size_t)y * s.Wo + x, v);
    }

    // ---- outputs that did not come out finite ------------------------------------------------------------------------------
    // An infinite sample (or one that is infinite once it is scaled) has no three-part form and leaves NaN behind, and so do the parts of
    // ordinary samples times an infinite weight: such outputs are worked out again in fp32 from the samples and the filters put
    // together.  Every wave for itself, pixel by pixel: its output channels side by side, the lanes left over share the k-steps.  A
    // pixel with a NaN in its window stays one.  (56x56 64->96 5x5, us: 11.1, with a NaN and an infinity among the samples 289 - 441
    // with a 64-bit address and a check for every sample - and all NaN 113; by one lane each the second took 2000.)
    const unsigned long long any = __builtin_amdgcn_ballot_w64(again != 0u);
    if (__builtin_expect(any == 0, 1)) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    // (what is stored below lies where other lanes have stored)
    const int kh = s.steps / s.spr;
    if (s.pool) {                                       // output by output, the four of its window by the whole wave
        for (int n = 0; n < kPooled; ++n)
            for (unsigned long long bad = __builtin_amdgcn_ballot_w64((again >> n & 1u) != 0); bad != 0; bad &= bad - 1) {
                const int src = __builtin_ctzll(bad);
                int oc, x, y;
                pooled_of(n, oc, x, y);
                oc = __shfl(oc, src); x = __shfl(x, src); y = __shfl(y, src);
                const int o = blockIdx.z * (32 * WO) + oc;
                if (o >= s.O || x >= s.Wo || y >= s.Ho) continue;
                float best = -FLT_MAX;
                for (int e = 0; e < 4; ++e) {
                    const int xe = x + (e & 1), ye = y + (e >> 1);
                    best = larger(best, xe < s.Wo && ye < s.Ho ? finish(once_more(std::integral_constant<int, 1>{}, kh, xe, ye, oc), 1.0f, biasT[oc]) : 0.0f);
                }
                if (lane == src) store_through(out + (size_t)o * Pp + (size_t)(y >> 1) * Wp + (x >> 1), best);
            }
        return;
    }
    constexpr int CH = 4 * WO;                          // channels of this wave
    const int ci = lane % CH, oc = MT == 1 ? 16 * (ci >> 1) + 2 * wave + (ci & 1) : 8 * ci + wave, o = blockIdx.z * (32 * WO) + oc;
    for (unsigned long long bad = MT == 1 ? (any | any >> 32) & 0xffffffffull : any; bad != 0; bad &= bad - 1) {
        const int px = __builtin_ctzll(bad), pl = px & 31, m = px >> 5;
        const int x = x0 + (pl & (BW - 1)), y = y0 + (pl >> s.lgBW) + BH * m;
        if (x >= s.Wo || y >= s.Ho) continue;
        const float v = finish(once_more(std::integral_constant<int, CH>{}, kh, x, y, oc), 1.0f, biasT[oc]);
        const unsigned noted = (unsigned)__shfl((int)again, MT == 1 ? 32 * (ci & 1) + pl : px) >> (MT == 1 ? ci >> 1 : ci);
        if (lane < CH && (noted & 1u) && o < s.O) store_through(out + (size_t)o * P + (size_t)y * s.Wo + x, v);
    }
}

struct BankPlan { int cp, mt, wo, wk, pf, tilesX, tilesY; BankShape s; size_t lds; double clocks; };

static bool bank_shape(int W, int H, int I, int O, int kw, int kh, int sx, int sy, int mt, int wo, int wk, int lgBW, BankPlan* p) {
    p->cp = I <= 4 ? 4 : 16;
    p->mt = mt; p->wo = wo; p->wk = wk;
    BankShape& s = p->s;
    s.W = W; s.H = H; s.I = I; s.O = O; s.Wo = W / sx; s.Ho = H / sy;
    s.kw = kw; s.sx = sx; s.sy = sy; s.padX = kw / 2; s.padY = kh / 2;
    s.lgBW = lgBW;
    const bool p3 = lgBW >= kP3Tile;
    const int BW = p3 ? kP3W : 1 << lgBW, BH = p3 ? 2 * p3_rows(mt) + 1 : (32 >> lgBW) * mt, stepX = p3 ? BW - 1 : BW, stepY = p3 ? BH - 1 : BH;
    s.spr = p->cp == 16 ? kw : ceil_div(kw, 4);
    s.steps = s.spr * kh;
    s.pw = (BW - 1) * sx + (p->cp == 16 ? kw : 4 * s.spr);
    s.patchN = s.pw * ((BH - 1) * sy + kh);
    s.nChunks = p->cp == 16 ? ceil_div(I, 16) : 1;
    s.oBlocks = ceil_div(O, 32);
    const FastDiv d = make_fastdiv(s.pw), dp = make_fastdiv(s.patchN);
    s.pwMul = d.mul; s.pwShift = d.shift;
    s.patchMul = dp.mul; s.patchShift = dp.shift;
    s.sprMul = (unsigned)(65536 / s.spr + 1);
    const size_t sums = (size_t)wk * 32 * wo * mt * 33 * sizeof(float);
    p->tilesX = ceil_div(s.Wo, stepX); p->tilesY = ceil_div(s.Ho, stepY);
    const long long wgs = (long long)p->tilesX * p->tilesY * ceil_div(s.oBlocks, wo);
    // As few stages as LDS allows (half of it where a CU is to hold two workgroups), of the same number of chunks: the loads of a stage are
    // one trip to memory, and every stage leaves waves without a last step.  56x56 64->96 5x5 12.9 us by single chunks, 11.4 in one stage of
    // four; 28x28 128->128 5x5 14.5 and 11.7 in two of four.
    s.nStages = 0;
    do {
        s.group = ceil_div(s.nChunks, ++s.nStages);
        const int units = s.patchN * (p->cp == 16 ? 2 : 1) * s.group;
        const size_t partBytes = ((size_t)units * (p->cp == 16 ? 16 : 8) + 15) & ~(size_t)15;
        p->pf = std::min(ceil_div(units, kBankThreads), p->cp == 16 ? 4 : 2);
        p->lds = std::max(3 * partBytes * (s.nStages > 1 ? 2 : 1), sums);
        if (s.group <= 8 && units <= 4 * kBankThreads && p->lds <= (wgs > num_cu() ? kMaxDynamicLds / 2 : kMaxDynamicLds) && s.group * s.steps * s.steps < 65536) break;
    } while (s.group > 1);
    s.nStages = ceil_div(s.nChunks, s.group);
    s.stepsMul = s.group > 1 ? (unsigned)(65536 / s.steps + 1) : 0;         // (exact by the last condition)
    return p->lds <= kMaxDynamicLds && s.steps * s.spr < 65536;      // (the kernel's division of a step number by spr)
}

// The tile that finishes first, by a count of what the busiest CU does, in clocks: per workgroup a fixed 1500 for the store, per stage 1200
// for the trip to memory and 1200 per round of staging (the address unit takes one dword gather every 8 to 16 clocks), and the MFMAs of
// one of its four SIMDs at 42 clocks or, if that is more, the filters at 42 bytes a clock, and 2 clocks for every row of outputs of
// a channel in a block, a piece of a line each (8 or 16 columns: 384x384 3->96 7x7/2 22.4 / 20.8 us, 224x224 3->64 7x7/2 6.2 / 5.9).  Pixel tiles wider than the map or
// hanging over its edge count in full, which picks the tile shape as well.  Measured, us per layer, this choice / the
// other tiles: 56x56 64->96 5x5 11.4 / 11.5 to 25, 224x224 3->64 7x7/2 6.1 / 7.7 to 13.7, 96x70 50->75 5x5 17.7 / 19.5 to 25, 28x28 128->128 5x5
// 11.7 / 16 to 47, 112x112 64->128 3x3/2 9.2 / 10.1 to 15.5, 14x14 16->32 5x5 4.3 / 5 to 9.
// pool: 0, 1 (2x2/2 behind the layer) or 2 (3x3/2: lgBW is kP3Tile or one more, and mt 2 or 3; never with waves for four blocks of channels,
// whose sums and pooling take longer than they save).
static bool bank_plan(int W, int H, int I, int O, int kw, int kh, int sx, int sy, int variant, int pool, BankPlan* best) {
    bool found = false;
    const int firstBW = pool == 2 ? kP3Tile : 3, lastBW = pool == 2 ? kP3Tile + 1 : pool ? 4 : 5;       // (2x2: two rows of a window in one block)
    auto blocks = [&](int lgM, int lgBW) { return pool == 2 ? 2 + lgBW - kP3Tile : 1 << lgM; };
    if (variant >> 12) {                                // everything chosen beforehand
        const int wsel = variant >> 4 & 3, lgBW = variant >> 12;
        return (variant & 0xfce) == 0x100 && wsel < 3 && lgBW >= firstBW && lgBW <= lastBW && (pool != 2 || ((variant & 1) && wsel > 0)) &&
               bank_shape(W, H, I, O, kw, kh, sx, sy, blocks(variant & 1, lgBW), 4 >> wsel, 2 << wsel, lgBW, best);
    }
    for (int wsel = pool == 2 ? 1 : 0; wsel < 3; ++wsel)
        for (int lgM = pool == 2 ? 1 : 0; lgM < 2; ++lgM) {
            const int wo = 4 >> wsel, wk = 2 << wsel;
            if (variant && variant != (0x100 | wsel << 4 | lgM)) continue;
            for (int lgBW = firstBW; lgBW <= lastBW; ++lgBW) {
                const int mt = blocks(lgM, lgBW);
                BankPlan p;
                if (!bank_shape(W, H, I, O, kw, kh, sx, sy, mt, wo, wk, lgBW, &p)) continue;
                const BankShape& s = p.s;
                const double wgs = (double)p.tilesX * p.tilesY * ceil_div(s.oBlocks, wo);
                const double waveSteps = (s.nStages - 1.0) * ceil_div(s.group * s.steps, wk) + ceil_div((s.nChunks - (s.nStages - 1) * s.group) * s.steps, wk);
                const double staging = s.nStages * 1200.0 * (1 + ceil_div(s.patchN * (p.cp == 16 ? 2 : 1) * s.group, kBankThreads));
                const double work = std::max(1.3 * waveSteps * 2 * 6 * 32 * mt, (double)s.nChunks * s.steps * wo * 3072 / 42);
                const double rows = pool == 2 ? 800.0 + 1000.0 * wo : pool ? 0.0 : 2.0 * 32 * wo * mt * (32 >> lgBW);
                p.clocks = 6000 + std::ceil(wgs / num_cu()) * (1500 + staging + work + rows);
                if (!found || p.clocks < best->clocks) { found = true; *best = p; }
            }
        }
    return found;
}

template <int CP, int MT, int WO, int WK, int PF, bool P3>
static int launch_bank_pf(const float* in, const unsigned short* F, const float* bias, float* out, const BankPlan& p, hipStream_t st) {
    const dim3 grid(p.tilesX, p.tilesY, ceil_div(p.s.oBlocks, WO));
    static std::atomic<unsigned long long> asked{0};
    if (int rc = allow_lds((const void*)conv_bank_mfma_kernel<CP, MT, WO, WK, PF, P3>, p.lds, asked)) return rc;
    launch((conv_bank_mfma_kernel<CP, MT, WO, WK, PF, P3>), grid, dim3(kBankThreads), p.lds, st, in, F, bias, out, p.s);
    return launched("conv_bank_mfma_kernel");
}

template <int CP, int MT, int WO, int WK, bool P3>
static int launch_bank(const float* in, const unsigned short* F, const float* bias, float* out, const BankPlan& p, hipStream_t st) {
    if constexpr (CP == 16) {
        if (p.pf == 4) return launch_bank_pf<CP, MT, WO, WK, 4, P3>(in, F, bias, out, p, st);
        if (p.pf == 3) return launch_bank_pf<CP, MT, WO, WK, 3, P3>(in, F, bias, out, p, st);
    }
    return p.pf == 1 ? launch_bank_pf<CP, MT, WO, WK, 1, P3>(in, F, bias, out, p, st) : launch_bank_pf<CP, MT, WO, WK, 2, P3>(in, F, bias, out, p, st);
}

template <int CP, int MT, bool P3>
static int launch_bank_w(const float* in, const unsigned short* F, const float* bias, float* out, const BankPlan& p, hipStream_t st) {
    if constexpr (!P3)
        if (p.wk == 2) return launch_bank<CP, MT, 4, 2, P3>(in, F, bias, out, p, st);
    if (p.wk == 4) return launch_bank<CP, MT, 2, 4, P3>(in, F, bias, out, p, st);
    return launch_bank<CP, MT, 1, 8, P3>(in, F, bias, out, p, st);
}

template <int CP>
static int launch_bank_m(const float* in, const unsigned short* F, const float* bias, float* out, const BankPlan& p, hipStream_t st) {
    if (p.s.lgBW >= kP3Tile) return p.mt == 2 ? launch_bank_w<CP, 2, true>(in, F, bias, out, p, st) : launch_bank_w<CP, 3, true>(in, F, bias, out, p, st);
    if (p.mt == 1) return launch_bank_w<CP, 1, false>(in, F, bias, out, p, st);
    return launch_bank_w<CP, 2, false>(in, F, bias, out, p, st);
}

}  // namespace drhip

using namespace drhip;

static size_t bank_blocks(int I, int O, int kw, int kh) {      // KiB of the bank per part
    const size_t steps = (size_t)kh * (I <= 4 ? ceil_div(kw, 4) : kw), chunks = I <= 4 ? 1 : ceil_div(I, 16);
    return steps * chunks * ceil_div(O, 32);
}

extern "C" size_t drhip_conv_bank_floats(int I, int O, int kw, int kh) {
    if (I <= 0 || O <= 0 || kw <= 0 || kh <= 0) return 0;
    return bank_blocks(I, O, kw, kh) * 3 * 256;
}

static bool bank_limits(int W, int H, int I, int O, int kw, int kh, int strideX, int strideY) {
    if (W <= 0 || H <= 0 || I <= 0 || O <= 0 || kw <= 0 || kh <= 0 || !(kw & 1) || !(kh & 1) || strideX <= 0 || strideY <= 0) return false;
    if (W / strideX <= 0 || H / strideY <= 0) return false;
    // byte offsets into the input and the bank are 32-bit, and 0x80000000 must lie outside both
    if ((long long)W * H * (I + 15) >= (1ll << 29) || (long long)(W / strideX) * (H / strideY) * O >= (1ll << 31)) return false;
    if (bank_blocks(I, O, kw, kh) * 3 * 1024 >= (1ull << 31)) return false;
    return H / strideY <= 65535 && ceil_div(O, 32) <= 65535;
}

extern "C" int drhip_conv_bank_usable(int W, int H, int I, int O, int kw, int kh, int strideX, int strideY) {
    BankPlan p;
    return bank_limits(W, H, I, O, kw, kh, strideX, strideY) && bank_plan(W, H, I, O, kw, kh, strideX, strideY, 0, 0, &p) ? 1 : 0;
}

// (Choosing a tile costs the host a microsecond or two: once when a layer is scheduled, not at every launch.)
static int bank_variant(const BankPlan& p) { return 0x100 | (p.wk == 2 ? 0 : p.wk == 4 ? 0x10 : 0x20) | (p.mt > 1 ? 1 : 0) | p.s.lgBW << 12; }

extern "C" int drhip_conv_bank_pick_variant(int W, int H, int I, int O, int kw, int kh, int strideX, int strideY, int maxpool2) {
    BankPlan p;
    if (!bank_limits(W, H, I, O, kw, kh, strideX, strideY) || !bank_plan(W, H, I, O, kw, kh, strideX, strideY, 0, maxpool2 != 0, &p)) return 0;
    return bank_variant(p);
}

// A 3x3/2 pooling in the layer's launch, or apart: its own launch takes 3 us and its map's way to memory and back, 2500 bytes a clock; a 1x1 layer
// behind it that takes it on load 0.7 us and 0.6 a megabyte.  us, apart / in one launch: 224x224 3->64 7x7/2 10.6 / 8.5 (in
// tiles of 4x4; of 4x3, 266 workgroups on 256 CUs, 12.8), 200x200 3->64 9.9 / 7.3, 96x96 3->24 8.5 / 5.9; 384x384 3->96 26.4 / 27.1, 224x224 3->32
// 5x5 19.2 / 19.2, 56x56 64->64 5x5 10.9 / 10.8, which stay apart: 7 % are asked for, as the estimates are no better.  With a 1x1 layer, taken on load / in
// one launch: 300x300 3->64 20.4 / 17.8, 200x200 3->64 12.2 / 10.9, 224x224 3->64 11.3 / 11.5, 128x128 3->32 7.8 / 8.4.
extern "C" int drhip_conv_bank_maxpool3s2_pick_variant(int W, int H, int I, int O, int kw, int kh, int strideX, int strideY, int against) {
    BankPlan p, apart;
    if (!bank_limits(W, H, I, O, kw, kh, strideX, strideY) || !bank_plan(W, H, I, O, kw, kh, strideX, strideY, 0, 2, &p)) return 0;
    const double bytes = 4.0 * (W / strideX) * (H / strideY) * O, pooling = against == 1 ? 1600 + bytes / 714 : 7000 + 1.25 * bytes / 2500;
    return against != 2 && bank_plan(W, H, I, O, kw, kh, strideX, strideY, 0, 0, &apart) && 0.93 * (apart.clocks + pooling) < p.clocks ? 0 : bank_variant(p);
}

extern "C" int drhip_conv_bank_layout_f32(const float* w, float* F, int I, int O, int kw, int kh, void* stream) {
    DRHIP_REQUIRE(w && F, "drhip_conv_bank_layout_f32: NULL tensor");
    DRHIP_REQUIRE(I > 0 && O > 0 && kw > 0 && kh > 0 && bank_blocks(I, O, kw, kh) * 3 * 1024 < (1ull << 31), "drhip_conv_bank_layout_f32: bad shape I=%d O=%d %dx%d", I, O, kw, kh);
    const int cp = I <= 4 ? 4 : 16, spr = cp == 4 ? ceil_div(kw, 4) : kw, chunks = cp == 4 ? 1 : ceil_div(I, 16);
    launch(conv_bank_layout_kernel, dim3((unsigned)(bank_blocks(I, O, kw, kh) * 2)), dim3(256), 0, as_stream(stream), w, (unsigned short*)F, I, O, kw, kh, cp, spr,
           spr * kh, chunks, ceil_div(O, 32));
    return launched("conv_bank_layout_kernel");
}

static int conv_bank(const float* in, const float* F, const float* bias, float* out, int W, int H, int I, int O,
                     int kw, int kh, int strideX, int strideY, int relu, int pool, int variant, void* stream, const char* who) {
    DRHIP_REQUIRE(in && F && out, "%s: NULL tensor", who);
    DRHIP_REQUIRE(bank_limits(W, H, I, O, kw, kh, strideX, strideY), "%s: shape %dx%dx%d -> %d, %dx%d/%dx%d not covered", who, W, H, I, O, kw, kh, strideX, strideY);
    DRHIP_REQUIRE(((size_t)F & 15) == 0, "%s: the filter bank must be 16-byte aligned", who);
    BankPlan p;
    DRHIP_REQUIRE(bank_plan(W, H, I, O, kw, kh, strideX, strideY, variant, pool, &p), "%s: variant %#x does not fit this shape", who, variant);
    p.s.relu = relu ? 1 : 0;
    p.s.pool = pool;
    if (p.cp == 4) return launch_bank_m<4>(in, (const unsigned short*)F, bias, out, p, as_stream(stream));
    return launch_bank_m<16>(in, (const unsigned short*)F, bias, out, p, as_stream(stream));
}

extern "C" int drhip_conv_bank_f32(const float* in, const float* F, const float* bias, float* out, int W, int H, int I, int O,
                                   int kw, int kh, int strideX, int strideY, int relu, int variant, void* stream) {
    return conv_bank(in, F, bias, out, W, H, I, O, kw, kh, strideX, strideY, relu, 0, variant, stream, "drhip_conv_bank_f32");
}

extern "C" int drhip_conv_bank_maxpool2_f32(const float* in, const float* F, const float* bias, float* out, int W, int H, int I, int O,
                                            int kw, int kh, int strideX, int strideY, int relu, int variant, void* stream) {
    return conv_bank(in, F, bias, out, W, H, I, O, kw, kh, strideX, strideY, relu, 1, variant, stream, "drhip_conv_bank_maxpool2_f32");
}

extern "C" int drhip_conv_bank_maxpool3s2_f32(const float* in, const float* F, const float* bias, float* out, int W, int H, int I, int O,
                                              int kw, int kh, int strideX, int strideY, int relu, int variant, void* stream) {
    return conv_bank(in, F, bias, out, W, H, I, O, kw, kh, strideX, strideY, relu, 2, variant, stream, "drhip_conv_bank_maxpool3s2_f32");
}
