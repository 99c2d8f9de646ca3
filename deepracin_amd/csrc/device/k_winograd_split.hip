// Winograd F(2x2,3x3) on the bf16 matrix cores, at fp32 accuracy: the large layers of k_winograd.hip, with the same
// transforms, the same grouping into 16 products of filters and tiles and the same fusions, each product as six partial
// products of bf16 parts (bf16x3.hpp).  That is 2.67 times the matrix rate of fp32, and vector instructions run beside a
// bf16 MFMA where they exclude an fp32 one.
//
// What bounds it: the address unit of a CU.  Operands come as 16-byte loads per lane, 1 KiB each and 20 to 26 clocks; two
// workgroups on a CU need 192 of them for filters and 40 for samples per 16 channels.  Counted on 320x240 128->128, per 16
// channels of two workgroups with their share of the first loads and the stores: the CU busy for 7300 clocks, its address
// unit for 6000, the MFMAs of a SIMD 3070, LDS 2600 (1150 of them bank conflicts).  (A filter fragment serves two MFMAs here.  With two
// blocks of tiles per wave it would serve four, but then the transform and the split of the samples, which every wave does
// for its own row of the transform, take as long as the loads; splitting the positions of a row over two waves balances all
// four units on paper and measured 5750 to 6300 with nothing left to overlap the first loads and the stores with.)
// Measured per layer, normally distributed data, us, fp32 kernel / this one: 448x448 64->64 78 / 61, 224x224 64->64 22.8 / 18.6,
// 224x224 128->128 75 / 57, 320x240 128->128 90 / 72, 160x120 256->256 107 / 84, 112x112 128->128 21.1 / 17.7,
// 80x60 512->512 105 / 84, 56x56 512->512 73 / 52.
//
// A workgroup owns 32 consecutive tiles and 64 output channels; each of four waves owns one row of the 4x4 transform, 16
// input channels per step:
//   * The samples under the tiles go from global memory straight to LDS (buffer load with the LDS destination), two steps
//     ahead, raw and row by row: no registers, no instructions, any alignment, and what lies outside the map or beyond the
//     last channel arrives as zeros.
//   * A lane reads the two window rows of its tile that its row of the transform combines, transforms and splits them;
//     that work is cut into ticks and dealt out between the MFMAs of the position in front of it (without that the
//     compiler gathers it in front of the MFMAs, and the matrix cores wait).
//   * Filters are transformed and split once, when the layer is prepared, and come as 1 KiB fragments a step or half a step ahead.
//   * Tiles that do not come out finite are worked out again in fp32, at the end.
// With KW = 2 two such sets of four waves share the tiles and take alternate steps; their sums meet in LDS.  That is for
// launches that leave at most one workgroup per CU, where a single set is alone on its SIMDs and waits for its own loads.
// Launches whose panels do not fill the CUs evenly cut the input channels of all or of the last panels into pieces, which add their
// sums up inside the launch (the rule, and what it measured, stands at the choice of the variant).
//
// The second kernel of this file does the same with operands in two f16 parts (f16x2.hpp).
#include "f16x2.hpp"
#include "wino_common.hpp"

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <vector>

namespace drhip {

constexpr int kWsKC = 16;               // input channels per step
// WC: 16-byte pieces of a window row of one channel in LDS, 20 or (narrow maps) 24.  The rows of tiles whose samples fit:
// 2*31 + 3 floats, 4 more per row, 4 in front.
constexpr int ws_segments(int WC) { return (4 * WC - 72) / 4 + 1; }

struct WsShape {                            // everything but the pointers; by value to the kernel
    int W, H, I, O, tilesX, T, nTB, nBlocks, nC, nOB;   // tiles, panels of 32 tiles, panels of outputs; 16-channel chunks, 32-channel blocks of filters
    unsigned mulX, shX, mulTB, shTB;                    // division by tilesX and by nTB
    int flags, vec2, pairs;                             // pairs: rows of two neighbouring tiles' outputs are 16 bytes, on 8
    // The first nA output panels of an XCD are cut into sA splits of perA chunks (in nA * sA workgroups), the others into sB of
    // perB; mulA, mulB: division by sA and sB
    int wgsA, nA, sA, sB, perA, perB, mulA, mulB;
    int joinSpins;
};

__device__ unsigned g_ws_join_timeouts;     // partial tiles that never arrived, over the life of the process

// U[row][chunk][o/32][position in the row][part][lane][8] (bf16): lane l of a wave holds output channel o = l%32 and input
// channels 8*(l/32) .. +7 of the chunk's 16.  What does not exist is zero.
__global__ void __launch_bounds__(256)
wino_split_filter_kernel(const float* __restrict__ w, unsigned short* __restrict__ U, int I, int O, int nC, int nOB) {
    const int row = threadIdx.x >> 6, lane = threadIdx.x & 63, ob = blockIdx.x % nOB, chunk = blockIdx.x / nOB;
    const int c0 = chunk * 16 + 8 * (lane >> 5), o = ob * 32 + (lane & 31);
    float u[8][4];                                  // the row's four positions of eight channels
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float all[16] = {};
        if (c0 + e < I && o < O) wino_filter_transform(w + ((size_t)(c0 + e) * O + o) * 9, all);
#pragma unroll
        for (int x = 0; x < 4; ++x) u[e][x] = row == 0 ? all[x] : row == 1 ? all[4 + x] : row == 2 ? all[8 + x] : all[12 + x];
    }
    u32x4b* d = (u32x4b*)U + ((size_t)(row * nC + chunk) * nOB + ob) * 12 * 64 + lane;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        u32x4b part[3];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            unsigned short a[3], b[3];
            split_one(u[2 * p][x], a);
            split_one(u[2 * p + 1][x], b);
#pragma unroll
            for (int q = 0; q < 3; ++q) part[q][p] = a[q] | (unsigned)b[q] << 16;
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) d[(x * 3 + q) * 64] = part[q];
    }
}

// What a workgroup computes: a split of the input channels of a panel of 32 tiles and 64 output channels.
template <int KW>
struct WsPlace {
    int wave, set, nSp, split, inXcd, first, perSplit, steps, oBlock, o0, t0;      // (wave: the row of the transform, of both sets)
    bool ok;
    __device__ __forceinline__ explicit WsPlace(const WsShape& s) {
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3;
        set = KW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
        const FastDiv nTBd = {(unsigned)s.nTB, s.mulTB, s.shTB};
        const int perXcd = (s.nBlocks + kXcds - 1) / kXcds;
        const int slot = (int)(blockIdx.x >> 3), later = slot - s.wgsA;        // (an XCD works on neighbouring panels)
        nSp = later < 0 ? s.sA : s.sB;
        const int place = later < 0 ? slot : later, panel = nSp == 1 ? place : place * (later < 0 ? s.mulA : s.mulB) >> 16;
        split = nSp == 1 ? 0 : place - panel * nSp;
        inXcd = (later < 0 ? 0 : s.nA) + panel;
        const int logical = (int)(blockIdx.x & 7) * perXcd + inXcd;
        ok = !(inXcd >= perXcd || logical >= s.nBlocks);
        perSplit = later < 0 ? s.perA : s.perB;
        first = split * perSplit;
        steps = (perSplit + KW - 1) / KW;
        oBlock = fast_div(logical, nTBd);
        o0 = oBlock * 64;
        t0 = (logical - oBlock * s.nTB) * 32;
    }
};

// The samples of a workgroup's steps on their way from global memory to LDS, and where they lie there.
// A segment is the part of the panel's 32 tiles that lies in one row of tiles; its samples lie in a row in LDS, from a
// multiple of 16 bytes on: from column 2*tx-1 of its first tile, or from column 0 where that is left of the map (the sample
// in front of it is then whatever lies in front of it: it is multiplied by zero).
// TURNS: panels of an XCD begin at different channels (`turn`) and go round: the first to reach a fragment of the filters brings it
// from memory, the others find it in L2, and they take turns at that instead of all waiting for it together.  (A template parameter,
// because even its few instructions show on layers of three steps: 41x53 254->254 0.17 us.)
template <int KW, int WC, bool TURNS>
struct WsSamples {
    static constexpr int CHB = WC * 16, ROWB = kWsKC * CHB, BUFB = 4 * ROWB;    // bytes of a window row of one channel, of 16, of a step's samples
    static constexpr int NDMA = ROWB / 1024;        // loads of a wave for them: one window row each
    unsigned voff[NDMA];                            // (never below kOutOfRange where it started from that)
    unsigned stepB, ldsBase, toNext;
    int steps, fetching, left;                      // the step whose samples are fetched next; how many are to come
    __amdgpu_buffer_rsrc_t rIn;

    __device__ __forceinline__ static int segment_at(const WsShape& s, int off0, int k) { return k == 0 ? 4 : (2 * (k * s.tilesX - off0) + 4 * k + 6) & ~3; }     // in floats

    __device__ __forceinline__ WsSamples(const float* in, const char* lds, const WsShape& s, const WsPlace<KW>& at, int ty0, int off0, int turn) {
        const int lane = threadIdx.x & 63, W = s.W, H = s.H, plane = W * H;
        steps = at.steps;
        stepB = 64u * KW * (unsigned)plane;
        const int first16 = 16 * (at.first + at.set);
        // Segment by segment, for a wave's window row and the same in all lanes: where its samples lie in LDS, behind which of them the
        // row ends (not one of them, for a row beside the map), and the address that the first would have at the row's beginning.
        constexpr int SEG = ws_segments(WC);
        const unsigned plane4 = 4u * (unsigned)plane;
        int segAt[SEG], segEnd[SEG];
        unsigned segBase[SEG];
#pragma unroll
        for (int k = 0; k < SEG; ++k) {
            const int iy = 2 * (ty0 + k) - 1 + at.wave, skip = k == 0 && off0 > 0 ? 2 * off0 - 1 : 0;
            segAt[k] = segment_at(s, off0, k);
            segEnd[k] = iy >= 0 && iy < H ? W - skip + segAt[k] : 0;
            segBase[k] = 4u * (unsigned)(iy * W + skip - segAt[k]) + (unsigned)first16 * plane4;
        }
        auto offsets = [&](auto segments) {
            int piece = lane % WC;
            unsigned chOff = (unsigned)(lane / WC) * plane4;
#pragma unroll
            for (int i = 0; i < NDMA; ++i) {
                const int f = 4 * piece;
                int end = segEnd[0];
                unsigned base = segBase[0];
#pragma unroll
                for (int k = 1; k < decltype(segments)::value; ++k) {
                    end = f >= segAt[k] ? segEnd[k] : end;
                    base = f >= segAt[k] ? segBase[k] : base;
                }
                voff[i] = (f >= 4 && f < end ? base + 4u * (unsigned)f + chOff : kOutOfRange) + (unsigned)turn * stepB;
                const bool wrap = piece >= WC - 64 % WC;        // 64 pieces on
                piece += 64 % WC - (wrap ? WC : 0);
                chOff += (unsigned)(64 / WC) * plane4 + (wrap ? plane4 : 0u);
            }
        };
        if (WC == 20 && s.tilesX >= 31) offsets(std::integral_constant<int, 2>{});      // (no panel touches three rows of tiles)
        else offsets(std::integral_constant<int, SEG>{});
        rIn = __builtin_amdgcn_make_buffer_rsrc((void*)in, 0, min(s.I, 16 * (at.first + at.perSplit)) * plane * 4, kBufferFlags);    // (ends with the split)
        ldsBase = (unsigned)(size_t)(__attribute__((address_space(3))) char*)lds + (unsigned)(at.set * 3 * BUFB + at.wave * ROWB);
        fetching = turn;
        left = steps;
        toNext = 0;
    }
    // The i-th load of the next step into buffer `buf`: 16 bytes per lane, lane by lane, to LDS at M0.  The compiler does not count these
    // loads: where it waits for a filter it waits for a few more loads than it means to, and for the samples the kernels wait themselves.
    __device__ __forceinline__ void fetch(int buf, int i) {
        if (i == 0) {
            const bool last = TURNS && fetching == steps - 1;
            toNext = last ? stepB - (unsigned)steps * stepB : stepB;
            // (behind the last one out of the map: zeros that nobody uses cost no trip to memory)
            if (TURNS) toNext = left == 1 ? kOutOfRange : toNext;
            if (TURNS) toNext = left < 1 ? 0u : toNext;
            --left;
            if (TURNS) fetching = last ? 0 : fetching + 1;
        }
        const unsigned at = ldsBase + (unsigned)(buf * BUFB);
        unsigned m0;                                    // (put back: the compiler may keep a value there, and takes no clobber for it)
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds\n\ts_mov_b32 m0, %0"
                     : "=&s"(m0) : "v"(voff[i]), "s"(rIn), "s"(at + 1024u * i) : "memory");
        voff[i] += toNext;
    }
};

__device__ __forceinline__ void ws_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ int ws_lane() { return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

// The bank of three bf16 parts: its fragments of 32 output channels by 16 input channels in pieces of 16 bytes, and a weight out of its parts.
struct WsBf16x3 {
    static constexpr int PARTS = 3;
    __device__ __forceinline__ static float whole(const unsigned (&part)[PARTS], float) { return drhip::whole(part[0], part[1], part[2]); }
};

// The sums of a panel, rows of the transform (and the two wave sets) side by side in LDS as P[set][row][2][64][32], become outputs: joined with
// those of the other splits, checked, finished.  scaleT: by output channel, what the sums are to be multiplied by (none: kSplitUnscale).
template <int KW, class Bank>
__device__ __forceinline__ void ws_finish(const float* P, const float* biasT, const float* scaleT, const WsShape& s, const WsPlace<KW>& at, const float* in, const unsigned short* U, float* out, float* ws) {
    constexpr int NT = 2, OB = 32 * NT;
    using std::integral_constant;
    // (the lane is asked for once more: what lives through the loop would be spilled there)
    const int lane = ws_lane(), tid = 64 * (4 * at.set + at.wave) + lane, nSp = at.nSp, split = at.split, oBlock = at.oBlock, o0 = at.o0, t0 = at.t0;
    const int W = s.W, H = s.H, I = s.I, plane = W * H;
    const FastDiv tilesXd = {(unsigned)s.tilesX, s.mulX, s.shX};
    auto scale = [&](int ol) { return scaleT ? scaleT[ol] : kSplitUnscale; };
    constexpr int EO = 8 * KW, NP = OB / EO;        // output channels finished per pass, passes
    const int et = tid & 31, eo = tid >> 5;
    const int etg = t0 + et;
    const bool eOk = etg < s.T;
    const int eTy = eOk ? fast_div(etg, tilesXd) : 0;
    const int ox = eOk ? 2 * (etg - eTy * s.tilesX) : 0, oy = 2 * eTy;
    auto tile_of = [&](int ol) {
        float p[4][2];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                p[r][x] = P[((r * 2 + x) * OB + ol) * 32 + et];
                if (KW == 2) p[r][x] += P[(((4 + r) * 2 + x) * OB + ol) * 32 + et];
            }
        return f32x4{p[0][0] + p[1][0] + p[2][0], p[0][1] + p[1][1] + p[2][1], p[1][0] - p[2][0] + p[3][0], p[1][1] - p[2][1] + p[3][1]};
    };
    // An infinity, or a value that is one once it is scaled, has no three-part form and has left NaN behind, and so has the sample
    // beside the map that is multiplied by zero where it is one of those: what is not finite is noted, by pass, for the end.
    unsigned again = 0;
    auto note = [&](int q, f32x4 y) { again |= (fabsf(y[0]) + fabsf(y[1])) + (fabsf(y[2]) + fabsf(y[3])) < __builtin_inff() ? 0u : 1u << q; };
    if (nSp > 1) {
        // The splits of a panel add their partial tiles up as those of the fp32 kernel do: each finishes its share of the
        // passes, stores the others' shares and then looks for its own in the slots of the other splits, whose contents
        // say themselves whether they have arrived.  (Slots lie at a workgroup's place in the grid, whole panels in front left out, 8
        // apart within a panel.)
        const __amdgpu_buffer_rsrc_t rWs = __builtin_amdgcn_make_buffer_rsrc((void*)ws, 0, 0x7ffffff0, kBufferFlags);
        const unsigned group0 = blockIdx.x - (unsigned)(kXcds * (split + (s.sA == 1 ? s.wgsA : 0)));
        // The whole offset goes in the vector register.  With the region in the scalar one the compiler lets the next vector
        // instruction overwrite the data of a 16-byte store, and on gfx950 the store then now and then takes the new value.
        auto slot_of = [&](int u, int q) { return (int)((group0 + (unsigned)(kXcds * u)) * (unsigned)(OB * 32 * 16)) + 16 * ((eo + EO * q) * 32 + et); };
        auto join = [&](auto splitsConst) {
            constexpr int S = decltype(splitsConst)::value, C = (NP + S - 1) / S;       // C: passes of a split, at most
            const int q0 = (split * NP + S - 1) / S, count = ((split + 1) * NP + S - 1) / S - q0;
#pragma unroll
            for (int q = 0; q < NP; ++q)
                if (q < q0 || q >= q0 + count)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, tile_of(eo + EO * q)), rWs, slot_of(split, q), 0, kAuxThrough);
            const u32x4 empty = {kWinoEmpty, kWinoEmpty, kWinoEmpty, kWinoEmpty};
            f32x4 own[C];
            u32x4 part[C][S] = {};
#pragma unroll
            for (int i = 0; i < C; ++i) own[i] = tile_of(eo + EO * (q0 + min(i, count - 1)));
            bool ready = false;
            for (int spins = 0; spins <= s.joinSpins && !ready; ++spins) {
                if (spins == s.joinSpins) wino_gives_up(&g_ws_join_timeouts);
                asm volatile("" ::: "memory");          // (to the compiler these loads are invariant)
                ready = true;
#pragma unroll
                for (int i = 0; i < C; ++i)
#pragma unroll
                    for (int u = 0; u < S; ++u) if (u != split) part[i][u] = __builtin_amdgcn_raw_buffer_load_b128(rWs, slot_of(u, q0 + min(i, count - 1)), 0, kAuxDeviceVolatile);
#pragma unroll
                for (int i = 0; i < C; ++i)
#pragma unroll
                    for (int u = 0; u < S; ++u)
                        ready = ready && (u == split || wino_slot_full(part[i][u]));
            }
            const unsigned givenUp = wino_given_up(&g_ws_join_timeouts);    // (waits for nothing: the parts have come behind the own stores)
#pragma unroll
            for (int i = 0; i < C; ++i) {
                if (i >= count) continue;
                const int q = q0 + i, ol = eo + EO * q;
                f32x4 y = {0.f, 0.f, 0.f, 0.f};         // splits in order
#pragma unroll
                for (int u = 0; u < S; ++u) y += u == split ? own[i] : __builtin_bit_cast(f32x4, part[i][u]);
#pragma unroll
                for (int u = 0; u < S; ++u) if (u != split) __builtin_amdgcn_raw_buffer_store_b128(empty, rWs, slot_of(u, q), 0, kAuxThrough);
                note(q, y);
                if (!ready) {                           // a partner never delivered: it shows in the result, too
                    y = f32x4{__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf("")};
                    again &= ~(1u << q);
                }
                if (eOk && o0 + ol < s.O) wino_finish(out, y, biasT[ol], s.flags, o0 + ol, plane, W, H, ox, oy, s.vec2, scale(ol));
            }
            if (__builtin_expect(givenUp != 0, 0)) {
                int spins = s.joinSpins;
#pragma clang loop unroll(disable)
                for (int q = 0; q < NP; ++q)
                    if (q < q0 || q >= q0 + count) wino_see_off(rWs, slot_of(split, q), spins);
            }
        };
        constexpr bool kHalvesOnly = KW == 1 && Bank::PARTS == 3;
        if (kHalvesOnly || nSp == 2) join(integral_constant<int, 2>{});
        else if constexpr (!kHalvesOnly) {
            if (nSp == 3) join(integral_constant<int, 3>{});
            else join(integral_constant<int, 4>{});
        }
    } else if (s.pairs) {
        // Two neighbouring tiles a thread: half of the reads, and rows of 16 bytes to store, without branches between the stores: tiles, rows and output
        // channels that do not exist lie out of the range of the buffer.  A CU takes 16 bytes a clock of stores of 8 bytes a lane, and 20 to 25 of 16.
        // (640x480 64->64, clocks of a workgroup: sums 1360 -> 840, stores 4120 -> 2560 of 24800; the layer 69.2 -> 67.8 us, 320x240 64->128 37.0 -> 35.9.)
        constexpr int EP = 2 * EO, NQ = OB / EP;
        const int pt = 2 * (tid & 15), po = tid >> 4;
        const bool pOk = t0 + pt < s.T;
        const int pTy = pOk ? fast_div(t0 + pt, tilesXd) : 0, px = pOk ? 2 * (t0 + pt - pTy * s.tilesX) : 0;
        f32x4 rows[NQ][2];
        float sum = 0.0f;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int ol = po + EP * q;
            f32x2 p[4][2];
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    p[r][x] = *(const f32x2*)&P[((r * 2 + x) * OB + ol) * 32 + pt];
                    if (KW == 2) {
                        const f32x2 other = *(const f32x2*)&P[(((4 + r) * 2 + x) * OB + ol) * 32 + pt];
                        p[r][x] = f32x2{p[r][x][0] + other[0], p[r][x][1] + other[1]};
                    }
                }
            const float b = biasT[ol], f = scale(ol);
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const float top = p[0][x][t] + p[1][x][t] + p[2][x][t], bottom = p[1][x][t] - p[2][x][t] + p[3][x][t];
                    sum += fabsf(top) + fabsf(bottom);
                    rows[q][0][2 * t + x] = fmaf(top, f, b);
                    rows[q][1][2 * t + x] = fmaf(bottom, f, b);
                }
        }
        if (s.flags & kEpiRelu)
#pragma unroll
            for (int q = 0; q < NQ; ++q)
#pragma unroll
                for (int k = 0; k < 4; ++k) { rows[q][0][k] = fmaxf(rows[q][0][k], 0.f); rows[q][1][k] = fmaxf(rows[q][1][k], 0.f); }
        const bool pool = s.flags & kEpiMaxPool2;
        const int outPlane = pool ? plane >> 2 : plane;
        auto channels = [&](int q) {                    // (their buffer: the EP output channels of pass q)
            return __builtin_amdgcn_make_buffer_rsrc((void*)(out + (size_t)(o0 + EP * q) * outPlane), 0, max(min(s.O - o0 - EP * q, EP), 0) * outPlane * 4, kBufferFlags);
        };
        if (pool) {
            const int to = pOk ? 4 * (po * outPlane + pTy * (W >> 1) + (px >> 1)) : (int)kOutOfRange;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const f32x2 most = {fmaxf(fmaxf(rows[q][0][0], rows[q][0][1]), fmaxf(rows[q][1][0], rows[q][1][1])), fmaxf(fmaxf(rows[q][0][2], rows[q][0][3]), fmaxf(rows[q][1][2], rows[q][1][3]))};
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2b, most), channels(q), to, 0, kAuxThrough);
            }
        } else {
            const int to = pOk ? 4 * (po * plane + 2 * pTy * W + px) : (int)kOutOfRange, below = pOk && 2 * pTy + 1 < H ? to + 4 * W : (int)kOutOfRange;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const __amdgpu_buffer_rsrc_t r = channels(q);
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, rows[q][0]), r, to, 0, kAuxThrough);
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, rows[q][1]), r, below, 0, kAuxThrough);
            }
        }
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(pOk && !(sum < __builtin_inff())) != 0, 0)) {
#pragma clang loop unroll(disable)
            for (int n = 0; n < 2 * NQ; ++n) {          // bit 2 * pass + tile of the pair
                auto at = [&](int r, int x) { const float* row = &P[((r * 2 + x) * OB + po + EP * (n >> 1)) * 32 + pt + (n & 1)]; return KW == 2 ? row[0] + row[8 * OB * 32] : row[0]; };
                float all = 0.0f;
#pragma unroll
                for (int x = 0; x < 2; ++x) all += fabsf(at(0, x) + at(1, x) + at(2, x)) + fabsf(at(1, x) - at(2, x) + at(3, x));
                again |= pOk && !(all < __builtin_inff()) ? 1u << n : 0u;
            }
        }
    } else {
        f32x4 y[NP];                                    // (read in one go: with each store behind its own reads the notes cost the trunk
        float b[NP], f[NP];                             // 4.5 us)
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            y[q] = tile_of(eo + EO * q);
            b[q] = biasT[eo + EO * q];
            f[q] = scale(eo + EO * q);
            note(q, y[q]);
        }
#pragma unroll
        for (int q = 0; q < NP; ++q)
            if (eOk && o0 + eo + EO * q < s.O) wino_finish(out, y[q], b[q], s.flags, o0 + eo + EO * q, plane, W, H, ox, oy, s.vec2, f[q]);
    }

    // ---- tiles that did not come out finite --------------------------------------------------------------------------------
    // Once more in fp32, step by step as the fp32 kernel does it, and with the samples beside the map left out.  Every wave
    // for itself, tile by tile: its 2 * NP output channels side by side, the lanes left over share the input channels.  (Us, without
    // and with one NaN and one infinity among the samples: 56x56 512->512 58 / 241, 224x224 64->64 18 / 39; all NaN 68 and 30.)
    const bool pairs = nSp == 1 && s.pairs;
    const unsigned long long any = __builtin_amdgcn_ballot_w64((pairs || eOk) && again != 0u);
    if (__builtin_expect(any == 0, 1)) return;          // (expected: otherwise what follows lies between instructions that every launch
                                                        // fetches, and a trunk of 640x480 takes 713 us instead of 702)
    constexpr int C = 2 * NP, S = 64 / C;               // channels of this wave, lanes per channel
    constexpr int PARTS = Bank::PARTS, FRAG = 4 * PARTS * 64;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    // (what is stored below lies where other lanes have stored)
    const __amdgpu_buffer_rsrc_t rAll = __builtin_amdgcn_make_buffer_rsrc((void*)in, 0, I * plane * 4, kBufferFlags);
    // (the channels that this wave has stored: of 2 a pass, or, of pairs of tiles, of 4)
    const int part = lane / C, first = pairs ? lane & 3 : lane & 1, pass = pairs ? lane % C >> 2 : lane % C >> 1, ol = pairs ? 4 * (tid >> 6) + first + 2 * EO * pass : 2 * (tid >> 6) + first + EO * pass;
    const u32x4b* uLane = (const u32x4b*)U + (size_t)min(oBlock * NT + (ol >> 5), s.nOB - 1) * FRAG + (ol & 31);
    unsigned bad = (unsigned)any | (unsigned)(any >> 32);
    if (pairs) {                                        // lanes with pairs become tiles
        bad = 0;
#pragma clang loop unroll(disable)
        for (int x = 0; x < 2; ++x) {
            const unsigned long long odd = __builtin_amdgcn_ballot_w64((again & 0x55555555u << x) != 0u);
            unsigned m = (unsigned)(odd | odd >> 16 | odd >> 32 | odd >> 48) & 0xffffu;
            m = (m | m << 8) & 0x00ff00ffu; m = (m | m << 4) & 0x0f0f0f0fu; m = (m | m << 2) & 0x33333333u; m = (m | m << 1) & 0x55555555u;
            bad |= m << x;
        }
    }
    for (; bad != 0; bad &= bad - 1) {
        const int t = __builtin_ctz(bad), ty = fast_div(t0 + t, tilesXd), x0 = 2 * (t0 + t - ty * s.tilesX) - 1, y0 = 2 * ty - 1;
        // A NaN among the samples at the tile's own four pixels reaches all four outputs, whatever the others are.
        bool own = false;
        for (int c = 0; c < I && !own; c += 64) {
            const float* at = in + (size_t)min(c + lane, I - 1) * plane + x0 + 1;
            const int right = x0 + 2 < W ? 1 : 0, r0 = (y0 + 1) * W, r1 = min(y0 + 2, H - 1) * W;
            own = __builtin_amdgcn_ballot_w64(__builtin_isunordered(at[r0], at[r0 + right]) || __builtin_isunordered(at[r1], at[r1 + right])) != 0;
        }
        if (own) continue;
        const int shift = x0 < 0 ? 1 : 0;               // (the first column's tiles load from column 0)
        f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma clang loop unroll(disable)
        for (int r = 0; r < 4; ++r) {                   // a row of the transform
            const int ya = y0 + r, yb = y0 + (r < 2 ? 2 : 1);
            const float sign = r == 1 ? 1.0f : -1.0f;
            float m[4] = {0.f, 0.f, 0.f, 0.f};
#pragma clang loop unroll(disable)
            for (int c8 = part; c8 < 2 * s.nC; c8 += S) {       // eight channels, half of a chunk
                const u32x4b* u = uLane + (size_t)(r * s.nC + (c8 >> 1)) * s.nOB * FRAG + 32 * (c8 & 1);
                float v[8][4];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    auto row = [&](int iy) {
                        const unsigned at = iy >= 0 && iy < H ? 4u * (unsigned)((8 * c8 + j) * plane + iy * W + x0 + shift) : kOutOfRange;
                        const f32x4 e = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rAll, (int)at, 0, 0));
                        return shift ? f32x4{0.f, e[0], e[1], e[2]} : e;
                    };
                    const f32x4 a = row(ya), b = row(yb);
                    float d[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) d[c] = x0 + c < W ? fmaf(sign, b[c], a[c]) : 0.0f;
                    v[j][0] = d[0] - d[2]; v[j][1] = d[1] + d[2]; v[j][2] = d[2] - d[1]; v[j][3] = d[3] - d[1];
                }
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    u32x4b parts[PARTS];
#pragma unroll
                    for (int q = 0; q < PARTS; ++q) parts[q] = u[(PARTS * x + q) * 64];
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        unsigned of[PARTS];
#pragma unroll
                        for (int q = 0; q < PARTS; ++q) of[q] = j & 1 ? parts[q][j / 2] >> 16 : parts[q][j / 2] & 0xffffu;
                        m[x] = fmaf(Bank::whole(of, scale(ol)), v[j][x], m[x]);
                    }
                }
            }
            const float p0 = m[0] + m[1] + m[2], p1 = m[1] - m[2] + m[3], back = r == 2 ? -1.0f : 1.0f;
            if (r < 3) { y[0] += p0; y[1] += p1; }
            if (r > 0) { y[2] = fmaf(back, p0, y[2]); y[3] = fmaf(back, p1, y[3]); }
        }
#pragma unroll
        for (int k = C; k < 64; k *= 2)
#pragma unroll
            for (int c = 0; c < 4; ++c) y[c] += __shfl_xor(y[c], k);
        const unsigned noted = (unsigned)__shfl((int)again, pairs ? 16 * first + (t >> 1) : 32 * first + t);
        if (part == 0 && (noted >> (pairs ? 2 * pass + (t & 1) : pass) & 1u) && o0 + ol < s.O) wino_finish(out, y, biasT[ol], s.flags, o0 + ol, plane, W, H, x0 + 1, y0 + 1, s.vec2);
    }
}

template <int KW, int WC, bool TURNS>
__global__ void __launch_bounds__(256 * KW, 2)
winograd_f23_split_kernel(const float* __restrict__ in, const unsigned short* __restrict__ U, const float* __restrict__ bias,
                          float* __restrict__ out, WsShape s, float* __restrict__ ws) {
    constexpr int NT = 2, OB = 32 * NT;
    using Samples = WsSamples<KW, WC, TURNS>;
    constexpr int CHB = Samples::CHB, ROWB = Samples::ROWB, BUFB = Samples::BUFB, NDMA = Samples::NDMA;
    constexpr int kPA[6] = {0, 0, 0, 1, 1, 2}, kPB[6] = {2, 1, 0, 1, 0, 0}; // partial products: part of the filter, part of the sample
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ float biasT[OB];

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
    const WsPlace<KW> at(s);
    if (!at.ok) return;
    const int wave = at.wave, set = at.set, first = at.first, steps = at.steps, oBlock = at.oBlock, o0 = at.o0, W = s.W;
    const FastDiv tilesXd = {(unsigned)s.tilesX, s.mulX, s.shX};
    const int ty0 = fast_div(at.t0, tilesXd), off0 = at.t0 - ty0 * s.tilesX, turn = TURNS ? min(at.inXcd & 31, steps - 1) : 0;
    Samples fetched(in, lds, s, at, ty0, off0, turn);
    auto fetch_sample = [&](int buf, int i) { fetched.fetch(buf, i); };

    // ---- filters ---------------------------------------------------------------------------------------------------
    // The waits for samples count the filter loads issued behind them, so these must stay where they stand: an address whose
    // origin the compiler does not see keeps it from taking them for loads that no memory clobber concerns.
    const unsigned short* uHere = U;
    asm volatile("" : "+s"(uHere));
    const int uBytes = 16 * s.nC * 3 * s.nOB * 1024;
    const __amdgpu_buffer_rsrc_t rU = __builtin_amdgcn_make_buffer_rsrc((void*)uHere, 0, uBytes, kBufferFlags);
    unsigned uOb[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) uOb[nt] = (unsigned)((wave * s.nC * s.nOB + min(oBlock * NT + nt, s.nOB - 1)) * 12288);
    const unsigned uStep = (unsigned)s.nOB * 12288u;
    // (what the last step requests for one behind it comes from nowhere)
    __amdgpu_buffer_rsrc_t rNext = rU;
    // the first part of two positions and the others of one: no more registers are left
    u32x4b f0[2][NT], f12[NT][2];
    auto filter = [&](int e, int nt, int q) -> u32x4b& { return q == 0 ? f0[e & 1][nt] : f12[nt][q - 1]; };
    auto load_filter = [&](const __amdgpu_buffer_rsrc_t& from, int e, int nt, int q, int step) {
        filter(e, nt, q) = __builtin_bit_cast(u32x4b, __builtin_amdgcn_raw_buffer_load_b128(from, lane * 16 + q * 1024, (int)(uOb[nt] + (unsigned)min(step, s.nC - 1) * uStep + (unsigned)(e * 3072)), 0));
    };

    // ---- operands --------------------------------------------------------------------------------------------------
    const int rowA = wave, rowB = wave < 2 ? 2 : 1;
    const float sgn = wave == 1 ? 1.0f : -1.0f;
    const int lr = fast_div(l32 + off0, tilesXd), tx = l32 + off0 - lr * s.tilesX;
    const int firstTx = lr == 0 ? off0 : 0;
    const int rLds = half * 8 * CHB + 4 * (Samples::segment_at(s, off0, lr) + 2 * (tx - firstTx) - (firstTx == 0 ? 1 : 0));
    // the masks of the samples beside the map carry the scale of the split as well
    const float k0f = tx > 0 ? kSplitScale : 0.0f, k2f = 2 * tx + 1 < W ? kSplitScale : 0.0f, k3f = 2 * tx + 2 < W ? kSplitScale : 0.0f;
    float mm[8][4];                                 // combined window rows of this lane's tile, 8 channels
    float ra[4], rb[4];                             // a channel's rows on their way from LDS
    const char* samples = lds + set * 3 * BUFB;
    auto read_rows = [&](int buf, int j) {
        const float* a = (const float*)(samples + buf * BUFB + rowA * ROWB + rLds + j * CHB);
        const float* b = (const float*)(samples + buf * BUFB + rowB * ROWB + rLds + j * CHB);
#pragma unroll
        for (int c = 0; c < 4; ++c) { ra[c] = a[c]; rb[c] = b[c]; }
    };
    auto combine = [&](int j) {
#pragma unroll
        for (int c = 0; c < 4; ++c) mm[j][c] = fmaf(sgn, rb[c], ra[c]);
        mm[j][1] *= kSplitScale;                    // (the other two are multiplied where they are used)
        mm[j][2] *= k2f;
    };
    u32x4b B[2][3];                                 // [position parity][part]
    float va[2], vb[2], xa[2], xb[2];               // the two items being split
    auto vvalue = [&](int e, int c) {
        return e == 0 ? fmaf(k0f, mm[c][0], -mm[c][2]) : e == 1 ? mm[c][1] + mm[c][2] : e == 2 ? mm[c][2] - mm[c][1] : fmaf(k3f, mm[c][3], -mm[c][1]);
    };
    auto pack = [&](float a, float b) { return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2b{a, b}, bf16x2)); };
    // The operands of position e out of mm: 12 ticks for two items (an item is two channels), whose instructions
    // alternate: a vector instruction that needs the result of the one in front of it waits for it.
    auto split_tick = [&](int e, int tick) {
        const int u = tick / 12, k = tick % 12;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int p = 2 * u + x;
            u32x4b(&d)[3] = B[e & 1];
            if (k == 0) va[x] = vvalue(e, 2 * p);
            if (k == 1) vb[x] = vvalue(e, 2 * p + 1);
            if (k == 2 || k == 7 || k == 11) d[k == 2 ? 0 : k == 7 ? 1 : 2][p] = pack(va[x], vb[x]);
            if (k == 3 || k == 8) xa[x] = __builtin_bit_cast(float, d[k == 3 ? 0 : 1][p] << 16);
            if (k == 4 || k == 8) xb[x] = __builtin_bit_cast(float, d[k == 4 ? 0 : 1][p] & 0xffff0000u);
            if (k == 5 || k == 9) va[x] -= xa[x];
            if (k == 6 || k == 10) vb[x] -= xb[x];
        }
    };

    f32x16b acc[4][NT];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[e][nt][r] = 0.0f;

    // ---- prologue --------------------------------------------------------------------------------------------------
    float biasEarly = 0.0f;
    if (tid < OB && bias) biasEarly = bias[min(o0 + tid, s.O - 1)];
    asm volatile("" ::: "memory");
    // What the first products need comes first, the rest behind the barrier.
#pragma unroll
    for (int i = 0; i < (KW == 1 ? 2 : 1) * NDMA; ++i) fetch_sample(i / NDMA, i % NDMA);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int q = 0; q < 3; ++q) load_filter(rU, 0, nt, q, first + set + KW * turn);
    if (tid < OB) biasT[tid] = biasEarly;
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * NT + (KW == 1 ? NDMA : 0)) : "memory");
    ws_barrier();
#pragma unroll
    for (int i = 0; i < NDMA; ++i) if (KW == 2) fetch_sample(1, i);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) load_filter(rU, 1, nt, 0, first + set + KW * turn);
#pragma unroll
    for (int j = 0; j < 8; ++j) { read_rows(0, j); combine(j); }
#pragma unroll
    for (int t = 0; t < 24; ++t) split_tick(0, t);

    // ---- steps -----------------------------------------------------------------------------------------------------
    // A position is 12 MFMAs, one per slot; with each go two ticks of the next position's operands and what else is due.
    auto position = [&](auto ec, int step, int stepNext, int nxt, int nxt2) {
        constexpr int e = decltype(ec)::value;
#pragma unroll
        for (int i = 0; i < 6 * NT; ++i) {
            const int q = i / NT, nt = i % NT;
            acc[e][nt] = mfma_bf16(filter(e, nt, kPA[q]), B[e & 1][kPB[q]], acc[e][nt]);
            // a part's last product has been issued: its registers take the filters that come next
            if (q == 2 || q == 4 || q == 5) {
                const int by = q == 2 ? 2 : 1;
                load_filter(e + by >= 4 ? rNext : rU, (e + by) & 3, nt, kPA[q], e + by >= 4 ? stepNext : step);
            }
#pragma unroll
            for (int tk = 2 * i; tk < 2 * i + 2; ++tk) {
                split_tick((e + 1) & 3, tk);
                const int at = 24 * e + tk;         // 0..95 over the step
                if (at % 4 == 0 && at / 4 < NDMA) fetch_sample(nxt2, at / 4);
                // Rows of the next step, one channel after the other: read, and some ticks later combined, behind the last
                // use of what they replace and in front of their own first use.
                constexpr int kRead[8] = {46, 52, 57, 62, 67, 71, 76, 80}, kComb[8] = {51, 56, 61, 66, 70, 75, 79, 83};
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    if (at == kComb[j]) combine(j);
                    if (at == kRead[j]) read_rows(nxt, j);
                }
            }
            // The next step's samples, requested a step ago, have to be visible before they are read.  (Younger than them are this
            // step's fetch and at least the filters of a position: more than the count waited for.)
            if (24 * e + 2 * i + 2 == 36) {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NDMA + 4 * NT) : "memory");
                ws_barrier();
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    using std::integral_constant;
    int nxt = 1, nxt2 = 2;
    for (int n = 0, m = turn; n < steps; ++n) {
        const int step = first + set + KW * m;
        m = TURNS && m == steps - 1 ? 0 : m + 1;
        const int stepNext = first + set + KW * m;
        rNext = __builtin_amdgcn_make_buffer_rsrc((void*)uHere, 0, n + 1 < steps ? uBytes : 0, kBufferFlags);
        position(integral_constant<int, 0>{}, step, stepNext, nxt, nxt2);
        position(integral_constant<int, 1>{}, step, stepNext, nxt, nxt2);
        position(integral_constant<int, 2>{}, step, stepNext, nxt, nxt2);
        position(integral_constant<int, 3>{}, step, stepNext, nxt, nxt2);
        nxt = nxt2;
        nxt2 = nxt2 == 2 ? 0 : nxt2 + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // (fetches beyond the last step, of every wave: LDS is about to be used for
    ws_barrier();                                              // something else)

    // ---- epilogue --------------------------------------------------------------------------------------------------
    // D of the 32x32 MFMA: lane -> tile lane%32; register r -> channel 8*(r/4) + 4*(lane/32) + r%4.  Each wave reduces its row of the
    // transform to two columns, the rows (and the two sets) meet in LDS.
    float* P = (float*)lds;                         // [set][row][2][OB][32]
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float m0 = acc[0][nt][r], m1 = acc[1][nt][r], m2 = acc[2][nt][r], m3 = acc[3][nt][r];
            const int ol = 32 * nt + 8 * (r / 4) + 4 * half + (r % 4);
            P[(((set * 4 + wave) * 2 + 0) * OB + ol) * 32 + l32] = m0 + m1 + m2;
            P[(((set * 4 + wave) * 2 + 1) * OB + ol) * 32 + l32] = m1 - m2 + m3;
        }
    ws_barrier();
    ws_finish<KW, WsBf16x3>(P, biasT, nullptr, s, at, in, U, out, ws);
}

// ---- two f16 parts ---------------------------------------------------------------------------------------------------------

// The bank of two f16 parts: U[row][chunk][o/32][position in the row][part][lane][8], the filters of output channel o multiplied by a power of two;
// behind it, by output channel, what their sums are to be multiplied by.
struct WsF16x2 {
    static constexpr int PARTS = 2;
    __device__ __forceinline__ static float whole(const unsigned (&part)[PARTS], float scale) {
        return scale * (float)__builtin_bit_cast(f16x2h, part[0])[0] + scale * (float)__builtin_bit_cast(f16x2h, part[1])[0];
    }
};

// A bank's tail, in words: by output channel (rounded up to 32) what its sums are multiplied by; by 32 of them, how many the bank cannot hold; by
// 16-channel chunk and output channel the bits of the largest weight of the largest filter and of the smallest.
struct WsPairTail {
    float* scale;
    int *unfit, *largest, *least;
    __host__ __device__ WsPairTail(float* tail, int nC, int nOB) : scale(tail), unfit((int*)tail + 32 * nOB), largest(unfit + nOB), least(largest + 32 * nC * nOB) {}
    static __host__ __device__ size_t words(int nC, int nOB) { return (size_t)nOB * (33 + 64 * (size_t)nC); }
};
// Magnitudes by their bits, which are in the same order and put NaN last.  Where the largest weight of an output channel is in range and no filter's is below
// 2^-12 of it (why: drhip_winograd_pair_fits), two parts can hold the channel; one without any weight is exact.
__host__ __device__ inline bool ws_pair_holds(int largest, int least) {
    constexpr int low = (127 - 100) << 23, high = (127 + 100) << 23;        // the bits of 2^-100 and 2^100
    return largest == 0 || (largest >= low && largest <= high && least + (12 << 23) >= largest);
}

// On the device, where the weights are for the next kernel anyway: a pass over them on the host, 0.28 ns each, made dR_prepare of VGG16's convolutions over
// 640x480 8.4 ms (5.9 now, 5.4 with three parts) and that of three layers 56x56 128->256 0.99 (0.74, 0.76).
__global__ void __launch_bounds__(256)
wino_pair_range_kernel(const float* __restrict__ w, int* __restrict__ largest, int* __restrict__ least, int I, int O, int outputs) {
    __shared__ int part[2][4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, o = blockIdx.x * 64 + lane, chunk = blockIdx.y;
    int most = 0, fewest = 0x7fffffff;
    if (o < O)
        for (int c = 16 * chunk + wave; c < min(16 * chunk + 16, I); c += 4) {
            const float* f = w + ((size_t)c * O + o) * 9;
            int m = 0;
#pragma unroll
            for (int k = 0; k < 9; ++k) m = max(m, (int)(__float_as_uint(f[k]) & 0x7fffffffu));
            most = max(most, m);
            fewest = min(fewest, m);
        }
    part[0][wave][lane] = most;
    part[1][wave][lane] = fewest;
    __syncthreads();
    if (wave == 0 && o < outputs) {
        largest[(size_t)chunk * outputs + o] = max(max(part[0][0][lane], part[0][1][lane]), max(part[0][2][lane], part[0][3][lane]));
        least[(size_t)chunk * outputs + o] = min(min(part[1][0][lane], part[1][1][lane]), min(part[1][2][lane], part[1][3][lane]));
    }
}

// scale[o]: 2^-k, where 2^k brings the largest weight of output channel o to 2^13 .. 2^14.  Transformed filters are at most 2.25 times as large, and
// at least a quarter.
__global__ void __launch_bounds__(256)
wino_pair_filter_kernel(const float* __restrict__ w, unsigned short* __restrict__ U, float* tail, int I, int O, int nC, int nOB) {
    const WsPairTail t(tail, nC, nOB);
    __shared__ int range[2][8][32];
    __shared__ float upOf[32];
    const int row = threadIdx.x >> 6, lane = threadIdx.x & 63, ob = blockIdx.x % nOB, chunk = blockIdx.x / nOB;
    {
        const int ol = threadIdx.x & 31, eighth = threadIdx.x >> 5;
        int most = 0, fewest = 0x7fffffff;
        for (int c = eighth; c < nC; c += 8) {
            most = max(most, t.largest[(size_t)c * 32 * nOB + ob * 32 + ol]);
            fewest = min(fewest, t.least[(size_t)c * 32 * nOB + ob * 32 + ol]);
        }
        range[0][eighth][ol] = most;
        range[1][eighth][ol] = fewest;
    }
    __syncthreads();
    if (threadIdx.x < 32) {
        const int ol = threadIdx.x;
        int most = 0, fewest = 0x7fffffff;
        for (int k = 0; k < 8; ++k) { most = max(most, range[0][k][ol]); fewest = min(fewest, range[1][k][ol]); }
        const int e = (most >> 23) - 127;
        const float scale = most == 0 ? 1.0f : __uint_as_float((unsigned)(127 + max(min(e - 13, 114), -126)) << 23);
        upOf[ol] = __uint_as_float((254u << 23) - __float_as_uint(scale));
        if (chunk == 0) {
            t.scale[ob * 32 + ol] = scale;
            const unsigned long long unfit = __builtin_amdgcn_ballot_w64(!ws_pair_holds(most, fewest));
            if (ol == 0) t.unfit[ob] = __builtin_popcountll(unfit);
        }
    }
    __syncthreads();
    const int c0 = chunk * 16 + 8 * (lane >> 5), o = ob * 32 + (lane & 31);
    const float up = upOf[lane & 31];
    float u[8][4];                                  // the row's four positions of eight channels
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float all[16] = {};
        if (c0 + e < I && o < O) wino_filter_transform(w + ((size_t)(c0 + e) * O + o) * 9, all);
#pragma unroll
        for (int x = 0; x < 4; ++x) u[e][x] = up * (row == 0 ? all[x] : row == 1 ? all[4 + x] : row == 2 ? all[8 + x] : all[12 + x]);
    }
    u32x4b* d = (u32x4b*)U + ((size_t)(row * nC + chunk) * nOB + ob) * 8 * 64 + lane;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        u32x4b hi, lo;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            hi[p] = pack_f16(u[2 * p][x], u[2 * p + 1][x]);
            lo[p] = pack_f16(f16_rest(u[2 * p][x], hi[p], 0, -1.0f), f16_rest(u[2 * p + 1][x], hi[p], 1, -1.0f));
        }
        d[(2 * x) * 64] = hi;
        d[(2 * x + 1) * 64] = lo;
    }
}

// One word per lane, by byte offset, to consecutive words of LDS.
__device__ __forceinline__ void ws_word_to_lds(__amdgpu_buffer_rsrc_t from, int offset, const float* to) {
    const unsigned at = (unsigned)(size_t)(__attribute__((address_space(3))) const float*)to;
    unsigned m0;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(m0) : "v"(offset), "s"(from), "s"(at) : "memory");
}

// Winograd on the f16 matrix cores, operands in two parts (f16x2.hpp): the three-part kernel's panels, waves, steps and pieces, with 24 MFMAs a wave and
// step instead of 48, 16 KiB of filters instead of 24 and 176 vector instructions instead of 270.  Layers, us, three parts / two, with their errors
// against 64 bits (rms, 1e-7): 640x480 64->64 81.8 / 66.2 (1.82 / 1.62), 320x240 128->128 75.0 / 55.7 (2.40 / 2.01), 160x120 256->256 73.7 / 53.9
// (3.23 / 2.56), 112x112 128->128 16.9 / 13.4 (1.85 / 1.66), 40x30 512->512 29.2 / 22.9 (2.24 / 1.96), 80x60 512->512 76.4 / 54.0 (3.16 / 3.05).
// No value may go to scratch: a kernel that has any starts about 1 us later (the eight such layers of VGG16 293 -> 287 us a pass).
// What bounds it: two workgroups of a CU take 4480 clocks a step on 320x240, the fetches without the MFMAs 2630 (168 KB at 64 bytes a clock), MFMAs and vector
// instructions without fetches 1940: eight fragments of filters under way per wave do not cover the way to L2 while a CU's eight waves queue there.
template <int KW, int WC, bool TURNS>
__global__ void __launch_bounds__(256 * KW, 2)
winograd_f23_pair_kernel(const float* __restrict__ in, const unsigned short* __restrict__ U, const float* __restrict__ bias,
                         float* __restrict__ out, WsShape s, float* __restrict__ ws) {
    constexpr int NT = 2, OB = 32 * NT;
    using Samples = WsSamples<KW, WC, TURNS>;
    constexpr int CHB = Samples::CHB, ROWB = Samples::ROWB, BUFB = Samples::BUFB, NDMA = Samples::NDMA;
    constexpr int kPA[3] = {1, 0, 0}, kPB[3] = {0, 1, 0};   // partial products: part of the filter, part of the sample
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ float biasT[OB], scaleT[OB];

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, half = lane >> 5;
    const WsPlace<KW> at(s);
    if (!at.ok) return;
    const int wave = at.wave, set = at.set, first = at.first, steps = at.steps, oBlock = at.oBlock, o0 = at.o0, W = s.W;
    const FastDiv tilesXd = {(unsigned)s.tilesX, s.mulX, s.shX};
    const int ty0 = fast_div(at.t0, tilesXd), off0 = at.t0 - ty0 * s.tilesX, turn = TURNS ? min(at.inXcd & 31, steps - 1) : 0;
    Samples fetched(in, lds, s, at, ty0, off0, turn);

    // ---- filters ---------------------------------------------------------------------------------------------------
    // (an address whose origin the compiler does not see, for the reason that the three-part kernel has)
    const unsigned short* uHere = U;
    asm volatile("" : "+s"(uHere));
    const int uBytes = 16 * s.nC * 2 * s.nOB * 1024;
    const __amdgpu_buffer_rsrc_t rU = __builtin_amdgcn_make_buffer_rsrc((void*)uHere, 0, uBytes, kBufferFlags);
    unsigned uOb[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) uOb[nt] = (unsigned)((wave * s.nC * s.nOB + min(oBlock * NT + nt, s.nOB - 1)) * 8192);
    const unsigned uStep = (unsigned)s.nOB * 8192u;
    __amdgpu_buffer_rsrc_t rNext = rU;              // (what the last step requests for one behind it comes from nowhere)
    u32x4b f[2][NT][2];                             // of two positions
    int lane16 = lane * 16;                         // (told to the compiler anew in every step: the other part's offset goes in the instruction then)
    auto load_filter = [&](const __amdgpu_buffer_rsrc_t& from, int e, int nt, int q, int step) {
        f[e & 1][nt][q] = __builtin_bit_cast(u32x4b, __builtin_amdgcn_raw_buffer_load_b128(from, lane16 + q * 1024, (int)(uOb[nt] + (unsigned)min(step, s.nC - 1) * uStep + (unsigned)(e * 2048)), 0));
    };

    // ---- operands --------------------------------------------------------------------------------------------------
    // A column of tiles (a lane and the one 32 on) has its samples multiplied by a power of two of its own, `scale`, so that the largest that the wave
    // has met is below 2^14 once two rows of the window are combined, and was 2^11 or more when the scale was chosen.  A step that brings a larger one
    // lowers the scale, and what has been summed up with it, before its products begin.  As long as all samples are zero any scale will do.  A sample that the
    // scale takes beyond fp32 (2^64 behind nothing but zeros, 2^114 or more times as large as the ones in front of it) becomes an infinity, and its tile is worked out
    // again at the end.
    const int rowA = wave, rowB = wave < 2 ? 2 : 1;
    const float sgn = wave == 1 ? 1.0f : -1.0f;
    const int lr = fast_div(l32 + off0, tilesXd), tx = l32 + off0 - lr * s.tilesX;
    const int firstTx = lr == 0 ? off0 : 0;
    const int rLds = half * 8 * CHB + 4 * (Samples::segment_at(s, off0, lr) + 2 * (tx - firstTx) - (firstTx == 0 ? 1 : 0));
    float k[4] = {tx > 0 ? 1.0f : 0.0f, 1.0f, 2 * tx + 1 < W ? 1.0f : 0.0f, 2 * tx + 2 < W ? 1.0f : 0.0f};      // masks of the columns of the window, with the scale
    constexpr float kLimit = 0x1p14f;
    float most = 0.0f;                              // of the samples that come next
    unsigned long long noneYet = ~0ull;             // lanes that have met zeros only: any other sample sets their scale
    float minusOne;
    asm volatile("s_mov_b32 %0, 0xbf800000" : "=s"(minusOne));
    float mm[8][4];                                 // combined window rows of this lane's tile, 8 channels
    constexpr int RING = WC == 24 ? 2 : 3;
    float ra[RING][2], rb[RING][2];                 // two channels' samples of a column on their way from LDS, of three columns (two: registers)
    const char* samples = lds + set * 3 * BUFB;
    auto read_two = [&](int buf, int slot, int c, int j) {
        const float* a = (const float*)(samples + buf * BUFB + rowA * ROWB + rLds + j * CHB) + c;
        const float* b = (const float*)(samples + buf * BUFB + rowB * ROWB + rLds + j * CHB) + c;
#pragma unroll
        for (int x = 0; x < 2; ++x) { ra[slot][x] = a[x * (CHB / 4)]; rb[slot][x] = b[x * (CHB / 4)]; }
    };
    auto combine_two = [&](int slot, int c, int j) {
#pragma unroll
        for (int x = 0; x < 2; ++x) mm[j + x][c] = k[c] * fmaf(sgn, rb[slot][x], ra[slot][x]);
        most = fmaxf(fmaxf(fabsf(mm[j][c]), fabsf(mm[j + 1][c])), most);
    };
    u32x4b B[2][2];                                 // [position parity][part]
    float va[2], vb[2];                             // the two items being split
    auto vvalue = [&](int e, int c) {
        return e == 0 ? mm[c][0] - mm[c][2] : e == 1 ? mm[c][1] + mm[c][2] : e == 2 ? mm[c][2] - mm[c][1] : mm[c][3] - mm[c][1];
    };
    // The operands of position e out of mm: 6 ticks for two items (an item is two channels), whose instructions alternate.
    auto split_tick = [&](int e, int tick) {
        const int u = tick / 6, n = tick % 6;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int p = 2 * u + x;
            u32x4b(&d)[2] = B[e & 1];
            if (n == 0) va[x] = vvalue(e, 2 * p);
            if (n == 1) vb[x] = vvalue(e, 2 * p + 1);
            if (n == 2) d[0][p] = pack_f16(va[x], vb[x]);
            if (n == 3) va[x] = f16_rest(va[x], d[0][p], 0, minusOne);
            if (n == 4) vb[x] = f16_rest(vb[x], d[0][p], 1, minusOne);
            if (n == 5) d[1][p] = pack_f16(va[x], vb[x]);
        }
    };

    f32x16b acc[4][NT];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[e][nt][r] = 0.0f;

    // The scale that suits `most`, and everything that has been multiplied by the old one with it.
    auto rescale = [&](bool sums) {
        const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(most), __float_as_uint(most), false, false);
        const float largest = fmaxf(__uint_as_float(halves[0]), __uint_as_float(halves[1]));
        const int e = (int)(__float_as_uint(largest) >> 23) - 127, has = (int)(__float_as_uint(k[1]) >> 23) - 127;
        const bool lower = (largest >= kLimit || (largest != 0.0f && __builtin_amdgcn_inverse_ballot_w64(noneYet))) && e < 128;    // (an infinity stays one whatever the scale)
        const int by = lower ? min(11 - e, 126 - has) : 0;         // (-116 to 126: one factor)
        // Samples that no scale makes large enough, fp32 denormals, are left to the pass over what did not come out finite.
        const float factor = e + by < 1 && lower ? __builtin_nanf("") : __uint_as_float((unsigned)(127 + by) << 23);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            k[c] *= factor;
#pragma unroll
            for (int j = 0; j < 8; ++j) mm[j][c] *= factor;
        }
        noneYet &= ~__builtin_amdgcn_ballot_w64(lower);
        if (sums)
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[x][nt][r] *= factor;
#pragma unroll
        for (int t = 0; t < 12; ++t) split_tick(0, t);
    };

    // ---- prologue --------------------------------------------------------------------------------------------------
    if (wave == 0 && set == 0) {                    // to LDS as well; what does not exist, a missing bias among it, arrives as zeros
        const __amdgpu_buffer_rsrc_t rBias = __builtin_amdgcn_make_buffer_rsrc((void*)bias, 0, bias ? 4 * s.O : 0, kBufferFlags);
        const __amdgpu_buffer_rsrc_t rScale = __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)U + uBytes), 0, 128 * s.nOB, kBufferFlags);
        ws_word_to_lds(rBias, 4 * (o0 + lane), biasT);
        ws_word_to_lds(rScale, 4 * (o0 + lane), scaleT);
    }
    // What the first products need comes first, the rest behind the barrier.
#pragma unroll
    for (int i = 0; i < (KW == 1 ? 2 : 1) * NDMA; ++i) fetched.fetch(i / NDMA, i % NDMA);
#pragma unroll
    for (int q = 0; q < 2 * NT; ++q) load_filter(rU, 0, q & 1, kPA[q / 2], first + set + KW * turn);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NT + (KW == 1 ? NDMA : 0)) : "memory");
    ws_barrier();
#pragma unroll
    for (int i = 0; i < NDMA; ++i) if (KW == 2) fetched.fetch(1, i);
#pragma unroll
    for (int q = 0; q < 2 * NT; ++q) load_filter(rU, 1, q & 1, kPA[q / 2], first + set + KW * turn);
#pragma unroll
    for (int c = 0; c < 4; c += 2) {                // (eight reads under way: the sums' registers are still free)
        float pa[8][2], pb[8][2];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            read_two(0, 0, c + i / 4, 2 * (i % 4));
            pa[i][0] = ra[0][0]; pa[i][1] = ra[0][1]; pb[i][0] = rb[0][0]; pb[i][1] = rb[0][1];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            ra[0][0] = pa[i][0]; ra[0][1] = pa[i][1]; rb[0][0] = pb[i][0]; rb[0][1] = pb[i][1];
            combine_two(0, c + i / 4, 2 * (i % 4));
        }
    }
    {   // the first scale: for `most` where it is not zero
        rescale(false);
        if (__builtin_amdgcn_inverse_ballot_w64(noneYet)) {
#pragma unroll
            for (int c = 0; c < 4; ++c) k[c] *= 0x1p64f;
        }
        most = 0.0f;
    }

    // ---- steps -----------------------------------------------------------------------------------------------------
    // A position is 6 MFMAs, one per slot; with each go two ticks of the next position's operands and what else is due.
    auto position = [&](auto ec, int step, int stepNext, int nxt, int nxt2) {
        constexpr int e = decltype(ec)::value;
#pragma unroll
        for (int i = 0; i < 3 * NT; ++i) {
            const int q = i / NT, nt = i % NT, slot = 6 * e + i;        // slot: 0..23 over the step
            acc[e][nt] = mfma_f16(f[e & 1][nt][kPA[q]], B[e & 1][kPB[q]], acc[e][nt]);
            // a part's last product has been issued: its registers take the filters of the position after the next
            if (q != 1) load_filter(e >= 2 ? rNext : rU, (e + 2) & 3, nt, kPA[q], e >= 2 ? stepNext : step);
            split_tick((e + 1) & 3, 2 * i);
            split_tick((e + 1) & 3, 2 * i + 1);
            // The samples of the next step, two channels of a column at a time, read and two slots later combined, behind the last use of
            // what they replace: the first column is used by the first position alone, the third by the first three.
            if (slot >= 8) combine_two((slot - 8) % RING, (slot - 8) / 4 == 1 ? 2 : (slot - 8) / 4 == 2 ? 1 : (slot - 8) / 4, 2 * ((slot - 8) % 4));
            if (slot >= 6 && slot < 22) read_two(nxt, (slot - 6) % RING, (slot - 6) / 4 == 1 ? 2 : (slot - 6) / 4 == 2 ? 1 : (slot - 6) / 4, 2 * ((slot - 6) % 4));
            if (slot % 4 == 0 && slot / 4 < NDMA) fetched.fetch(nxt2, slot / 4);
            // The next step's samples, requested a step ago, have to be visible before they are read.  (Younger than them are filters behind
            // slot 16, or 20, of the step before, or of the prologue, those of this position and two loads for the step after.)
            if (slot == 5) {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NDMA == 5 ? 10 : 8) : "memory");
                ws_barrier();
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    using std::integral_constant;
    int nxt = 1, nxt2 = 2;
    for (int n = 0, m = turn; n < steps; ++n) {
        const int step = first + set + KW * m;
        m = TURNS && m == steps - 1 ? 0 : m + 1;
        const int stepNext = first + set + KW * m;
        rNext = __builtin_amdgcn_make_buffer_rsrc((void*)uHere, 0, n + 1 < steps ? uBytes : 0, kBufferFlags);
        if (__builtin_expect((__builtin_amdgcn_ballot_w64(most >= kLimit) | (__builtin_amdgcn_ballot_w64(most != 0.0f) & noneYet)) != 0, 0)) rescale(true);
        most = 0.0f;
        asm volatile("" : "+v"(lane16));
        position(integral_constant<int, 0>{}, step, stepNext, nxt, nxt2);
        position(integral_constant<int, 1>{}, step, stepNext, nxt, nxt2);
        position(integral_constant<int, 2>{}, step, stepNext, nxt, nxt2);
        position(integral_constant<int, 3>{}, step, stepNext, nxt, nxt2);
        nxt = nxt2;
        nxt2 = nxt2 == 2 ? 0 : nxt2 + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // (fetches beyond the last step, of every wave: LDS is about to be used for
    ws_barrier();                                           // something else)

    // ---- epilogue --------------------------------------------------------------------------------------------------
    float* P = (float*)lds;                         // [set][row][2][OB][32]
    const int at32 = ws_lane() & 31, atHalf = ws_lane() >> 5;
    const float back = __uint_as_float((254u << 23) - __float_as_uint(k[1]));
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float m0 = acc[0][nt][r], m1 = acc[1][nt][r], m2 = acc[2][nt][r], m3 = acc[3][nt][r];
            const int ol = 32 * nt + 8 * (r / 4) + 4 * atHalf + (r % 4);
            P[(((set * 4 + wave) * 2 + 0) * OB + ol) * 32 + at32] = back * (m0 + m1 + m2);
            P[(((set * 4 + wave) * 2 + 1) * OB + ol) * 32 + at32] = back * (m1 - m2 + m3);
        }
    ws_barrier();
    ws_finish<KW, WsF16x2>(P, biasT, scaleT, s, at, in, U, out, ws);
}

struct WsPlan { int kw, wc, perXcd; bool turns, pair; size_t lds; WsShape s; };

// Variant: 0x100 | wave sets - 1 | sA << 12 | sB << 16 | nA << 20, where the first nA output panels of every XCD are cut into
// sA splits (1 to 4, with one wave set 1 or 2) of their input channels and the others into sB; all zero: nothing is split.
static bool ws_plan(int W, int H, int I, int O, int variant, WsPlan* p) {
    if (variant < 0 || (variant & 0xdfe) != 0x100 || W < 1 || H < 1 || I < 1 || O < 1) return false;
    p->kw = 1 + (variant & 1);
    p->pair = (variant & 0x200) != 0;
    WsShape& s = p->s;
    s.W = W; s.H = H; s.I = I; s.O = O;
    s.tilesX = (W + 1) / 2;
    const int segments = (31 + s.tilesX - 1) / s.tilesX + 1;                // rows of tiles that a panel can touch
    p->wc = segments <= ws_segments(20) ? 20 : 24;
    if (segments > ws_segments(p->wc) || (p->wc == 24 && p->kw == 1)) return false;     // (one wave set never gained on narrow maps)
    // 32-bit byte offsets on the input (a set's last step may lie beyond the last channel) and on the filters
    if ((long long)W * H * (I + 31) >= (1ll << 29) || (long long)W * H * O >= (1ll << 31) ||
        (long long)ceil_div(I, kWsKC) * ceil_div(O, 32) * 12288 * 4 >= (1ll << 31)) return false;
    s.T = s.tilesX * ((H + 1) / 2);
    s.nC = ceil_div(I, kWsKC);
    s.nOB = ceil_div(O, 32);
    s.nTB = ceil_div(s.T, 32);
    s.nBlocks = s.nTB * ceil_div(O, 64);
    const FastDiv dx = make_fastdiv(s.tilesX), dt = make_fastdiv(s.nTB);
    s.mulX = dx.mul; s.shX = dx.shift; s.mulTB = dt.mul; s.shTB = dt.shift;
    p->lds = (size_t)p->kw * std::max<size_t>(3 * 4 * kWsKC * p->wc * 16, 8 * 64 * 32 * sizeof(float));
    const int panels = ceil_div(s.nBlocks, kXcds), cusPerXcd = num_cu() / kXcds;
    s.nA = variant >> 20; s.sA = variant >> 12 & 15; s.sB = variant >> 16 & 15;
    if (variant >> 12 == 0) { s.sA = s.sB = 1; s.nA = 0; }
    s.wgsA = s.nA * s.sA;
    p->perXcd = s.wgsA + (panels - s.nA) * s.sB;
    if (s.sA < 1 || s.sB < 1) return false;
    s.perA = ceil_div(s.nC, s.sA); s.perB = ceil_div(s.nC, s.sB);
    s.mulA = 65536 / s.sA + 1; s.mulB = 65536 / s.sB + 1;                   // (exact up to 8192 workgroups)
    // Beginning at different channels.  Measured with other filters and maps for every launch, us, all from the first channel
    // on / in 32 turns: two wave sets, 80x60 512->512 87.7 / 82.1, 80x60 256->512 51.4 / 46.2, 56x56 512->512 63.5 / 59.3, 40x30
    // 512->512 32.4 / 31.1; one set in one to two rounds, 160x120 256->256 84.1 / 78.4, 128->256 49.4 / 47.0.  With one set in
    // less than a round a CU's two workgroups read the same filters and lose that (80x60 512->512 93 / 100); over more rounds
    // the panels drift apart by themselves (320x240 128->128 87.0 / 87.7).
    // (Pieces of fewer than 8 chunks have no turns to take: 41x53 254->254 in thirds 0.1 us slower.)
    const int longest = s.nA > 0 ? s.perA : s.perB;
    p->turns = longest >= 8 && (p->kw == 2 || (panels > 2 * cusPerXcd && panels <= 4 * cusPerXcd));
    if (s.sA == 1 && s.sB == 1) return true;
    // A workgroup waits for the other splits of its panel, which are its neighbours in dispatch order on the same XCD: as long
    // as one XCD holds more workgroups than a panel has splits, they all get to run.
    auto allowed = [&](int n) { return n >= 1 && n <= (p->pair ? 4 : 2 * p->kw) && (n - 1) * ceil_div(s.nC, n) < s.nC; };
    return s.nA <= panels && allowed(s.sA) && allowed(s.sB) && std::max(s.sA, s.sB) < num_cu() / kXcds && p->perXcd < 8192 &&
           (long long)p->perXcd * kXcds * 32768 < (1ll << 31);
}

template <int KW, int WC, bool TURNS, bool PAIR>
static int launch_ws(const float* in, const unsigned short* U, const float* bias, float* out, float* ws, const WsPlan& p, hipStream_t st) {
    constexpr auto kernel = [] { if constexpr (PAIR) return winograd_f23_pair_kernel<KW, WC, TURNS>; else return winograd_f23_split_kernel<KW, WC, TURNS>; }();
    static std::atomic<unsigned long long> asked{0};
    if (int rc = allow_lds((const void*)kernel, p.lds, asked)) return rc;
    launch(kernel, dim3(p.perXcd * kXcds), dim3(256 * KW), p.lds, st, in, U, bias, out, p.s, ws);
    return launched(PAIR ? "winograd_f23_pair_kernel" : "winograd_f23_split_kernel");
}
template <bool PAIR>
static int launch_ws(const float* in, const unsigned short* U, const float* bias, float* out, float* ws, const WsPlan& p, hipStream_t st) {
    if (p.wc == 24) {
        if constexpr (!PAIR) { if (!p.turns) return launch_ws<2, 24, false, PAIR>(in, U, bias, out, ws, p, st); }
        return launch_ws<2, 24, true, PAIR>(in, U, bias, out, ws, p, st);       // (of the pair kernel always: without turns the compiler keeps a value in scratch)
    }
    if (p.kw == 2) return p.turns ? launch_ws<2, 20, true, PAIR>(in, U, bias, out, ws, p, st) : launch_ws<2, 20, false, PAIR>(in, U, bias, out, ws, p, st);
    return p.turns ? launch_ws<1, 20, true, PAIR>(in, U, bias, out, ws, p, st) : launch_ws<1, 20, false, PAIR>(in, U, bias, out, ws, p, st);
}

int ws_join_timeouts(unsigned* count) {
    return check(hipMemcpyFromSymbol(count, HIP_SYMBOL(g_ws_join_timeouts), sizeof(unsigned)), "hipMemcpyFromSymbol(join timeouts)");
}

}  // namespace drhip

using namespace drhip;

// Against the fp32 kernel this one gains with the work of a CU and loses with the time of its first loads and its stores, 6 us.
// Measured, ratio of the times: where every CU has more than one workgroup 0.65 to 0.93 with at least 64 input channels (4
// steps), 0.91 with 32 channels and 1.5 workgroups per CU and 1.08 to 1.4 with fewer, at best 0.93 with 16; with one
// workgroup for 0.6 to 1 of the CUs 0.71 to 0.92 from 128 channels on, 0.9 to 1.06 with 64, and with fewer workgroups 1.1 to 1.5
// (72x72 128->128 1.21, 56x56 256->256 1.26).
// Up to 32 output channels half of a workgroup would be padding.  Two wave sets where a CU gets one workgroup or none
// (112x112 128->128 17.7 us against 20.0, 56x56 512->512 52 against 61), one where it gets more (112x112 128->256 29.4 against 34.5).
//
// Splits even out what the panels leave uneven, and cost 2.6 us where they are joined (all times here: one layer launched over
// and over; between other layers the filters come from memory first).  n is the panels per XCD, of 32 CUs:
//   * n <= 16: all panels in 2 to 4 pieces, as many as leave one workgroup per CU.  That takes 2.75 us per pair of chunks and
//     10.6 more; the fp32 kernel takes 0.56 us per 8-channel stage of its busiest CU, 3 more and 1.5 for joining.  (40x30
//     512->512 27.9 us against 36.9; 56x56 256->256 20.8 against 20.7 and 28x28 512->512 21.4 against 21.6 stay there.)
//   * a few panels more than CUs: two wave sets, a round of whole panels and the rest in 3 or 4 pieces (80x60 512->512
//     74.4 us, 83.5 with one wave set unsplit; 256->512 43.8 and 45.4).  More than 10 of 32 left over, or below 384
//     channels more than 6: nothing gained (81x239 256->128, 7 over: 48.6 against 47.6).
//   * a few more than two per CU: the rest in halves (160x120 256->256 76.1 us against 84.3, 128->256 43.8 against 46.5).
//     After more rounds than one the workgroups do not end together any more (320x240 128->128, 2.3 rounds: 80 against 74).
//
// Two f16 parts take less (measured like that, 70 shapes drawn and VGG16's, with other filters each time, us fp32 kernel / this):
//   * pieces 7.8, 2 more per pair of chunks and 0.22 per MB of filters (56x56 256->256 20.3 / 16.4, 28x28 512->512 23.2 / 18.9, 61x75 320->140 23.3 / 19.8,
//     62x41 376->106 19.0 / 14.1, 51x41 191->384 18.0 / 15.5; 56x56 128->256 12.2 / 11.7, 28x28 256->512 14.0 / 14.4, 84x68 224->64 12.0 / 12.2 and fewer panels
//     stay there).  Where that kernel has helpers it takes 0.56 per stage that its own workgroups keep and 3.6 (39x152 198->68 13.6 / 15.2, 18x74 230->466
//     16.0 / 17.8 stay there).  300 drawn shapes of up to 16 panels: 0.90 to 1.003 times the fp32 kernel's time but for one, on a narrow map.
//     Those (six loads a step, each of more pieces of rows) take 6.5 around the pairs, 0.1 more for each workgroup of an XCD and 0.09 per MB, and the fp32 kernel's
//     time is taken for 0.4 less, or with a second launch for 1.5 more.  Of 20000 drawn shapes 32 stay in fp32 for it (21x148 232->79 12.9 / 14.2, 12x359 236->48
//     12.1 / 13.8, 17x236 237->55 12.0 / 13.5, 12x433 196->134 17.9 / 19.9; of the 32 half within 4 % of even, three 6 to 10 % slower in fp32).
//   * two thirds of a panel per CU at most, and fp32 panels for more than half of a round: from 19 chunks on all in thirds, with one wave set (73x28 400->476
//     32 / 28, 52x56 440->330 35.3 / 30.7; two wave sets unsplit 30.0 and 33.5; 80x60 512->256 33.6 against 35.8, 256->256 23.5 against 21.0).
//   * up to one and a half panels per CU: with one wave set, whole panels on seven CUs of eight and all others in halves, or, where there is room for
//     those at once as well, in thirds or quarters (whole / this: 88x64 512->512 65.2 / 58.7, 132x66 200->256 31.1 / 25.5, 122x93 128->256 21.7 / 20.7;
//     with fewer chunks than 8 no more than 4 %).  With more than one and a half panels per CU halves do not fit in beside them (100x78 400->400 56.0 / 61.8).
//   * Where three parts would have whole panels of two wave sets, whose sums are half as long, that would be less exact than they (by up to 3 %).  Up to
//     1/4 over, without padded outputs: half of the panels in halves, or, with 1/16 over, as many in quarters as leave two slots of the XCD empty (three parts /
//     seven of eight / this, and the errors against 64 bits, 1e-7: 80x60 512->512 76.4 / 52.9 / 54.0, 3.16 / 3.18 / 3.05; 80x60 256->512 43.7 / 30.7 / 31.2,
//     2.37 / 2.44 / 2.36; 71x119 256->256 42.8 / 28.8 / 29.5, 2.60 / 2.63 / 2.56; all slots taken 63 against 57 where 10 fewer are).  Otherwise two wave
//     sets here too (81x86 384->384 65.2 / 45.4 / 49.2, 2.79 / 2.89 / 2.30).  Over 100 drawn shapes the error is 0.62 to 0.998 times three parts'.
//   * no more than one in six CUs over two panels each: those in quarters (144x120 256->256 in halves 51.8, in quarters 48.5; 160x120, one in three, 53.8 and 57.4).
//   * one workgroup for more than half of the CUs from 4 chunks on (112x112 64->128 12.0 / 9.4, 48x56 64->448 12.0 / 9.4, 55x57 93->305 17.1 / 12.1), with
//     two wave sets from 8 (118x112 160->70 18.0 / 15.5, one set 16.2; 85x111 288->128 23.4 and 26.7), but none where the fp32 kernel's panels, of 32 outputs,
//     are a round (73x28 66->476 9.0 / 11.0, 34x159 140->141 12.9 / 16.2, 38x74 300->344 24.4 / 25.2).
static int ws_pick(int W, int H, int I, int O, bool pair) {
    WsPlan p;
    if (O <= 32 || !ws_plan(W, H, I, O, 0x101, &p)) return 0;
    const int blocks = p.s.nBlocks, nC = p.s.nC, cus = num_cu(), cusPerXcd = cus / kXcds, n = ceil_div(blocks, kXcds);
    const bool wide = p.wc == 20;                       // (narrower maps are taken only as pieces)
    static const bool joins = [] { const char* e = getenv("DR_WINO_JOIN"); return !(e && e[0] == '0'); }();
    auto split = [&](int base, int nA, int sA, int sB) {
        const int v = base | sA << 12 | sB << 16 | nA << 20;
        return ws_plan(W, H, I, O, v | (pair ? 0x200 : 0), &p) ? v : 0;
    };
    if (joins && 2 * n <= cusPerXcd) {
        // Against the fp32 kernel in equal splits and two launches, although its joined halves and helpers may be up to 1.2 times as fast as the
        // pieces: the pieces are more exact than those (error against 64 bits, 0.70 of joined halves' and 0.86 of helpers' over 15 shapes)
        // and stay where they gain on a form whose sums are as short.  And against what that kernel takes, where that is the slower one.
        const int S = std::min(4, cusPerXcd / n), halvings = wino_halvings(W, H, I, O), panels32 = p.s.nTB * ceil_div(O, 32);
        auto fp32 = [&](int lg) { return 0.56 * ceil_div(2 * nC, 1 << lg) * ceil_div(panels32 << lg, cus) + (lg > 0 ? 4.5 : 3); };
        const int pairs = ceil_div(ceil_div(nC, S), 2), picked = drhip_conv3x3_winograd_pick_variant(W, H, I, O);
        const double taken = fp32(picked >> 4 & 15);
        const double helped = picked & 0x2000 ? 0.56 * (ceil_div(I, 8) - wino_donated(W, H, I, O)) + 3.6 : taken, filterMB = 64e-6 * I * O;
        const double summed = (picked & 0xf00) == 0x400 && picked & 0xf0 ? 1.9 : 0;        // (two wave sets a panel, and a second launch)
        const bool gains = 2.0 * pairs + 7.8 + 0.22 * filterMB < 0.93 * helped && (wide || 2.0 * pairs + 6.9 + 0.105 * n * S + 0.09 * filterMB < helped + summed);
        if (halvings >= 0 &&                            // (layers of its 16-tile form are too small)
            (2.75 * pairs + 10.6 < 0.93 * std::max(fp32(halvings), taken) || (pair && gains)))
            if (const int v = split(0x101, 0, S, S)) return v;
    }
    if (!wide) return 0;
    const int over = n - cusPerXcd, over2 = n - 2 * cusPerXcd;
    const bool fewMore = joins && over > 0 && (nC >= 24 ? 3 * over <= cusPerXcd : nC >= 16 && 5 * over <= cusPerXcd);      // than one panel per CU
    if (pair && fewMore && O % 64 == 0 && 4 * over <= cusPerXcd) {
        const int k = 16 * over <= cusPerXcd ? 4 : 2, whole = k == 4 ? ceil_div(4 * n - 2 * cusPerXcd + 2, 3) : n / 2;
        if (const int v = split(0x100, whole, 1, k)) return v;
    }
    if (pair && joins && !fewMore && over > 0 && 2 * over <= cusPerXcd && nC >= 8) {
        const int whole = std::max(cusPerXcd * 7 / 8, 2 * over);
        for (int k = std::min(4, (2 * cusPerXcd - whole) / (n - whole)); k >= 2; --k)
            if (const int v = split(0x100, whole, 1, k)) return v;
    }
    if (fewMore)
        if (const int v = split(0x101, cusPerXcd, 1, 4 * over <= cusPerXcd ? 4 : 3)) return v;
    if (pair && joins && nC >= 8 && over2 > 0 && 6 * over2 <= cusPerXcd)
        if (const int v = split(0x100, 2 * cusPerXcd, 1, 4)) return v;
    if (joins && nC >= 8 && over2 > 0 && 2 * over2 <= cusPerXcd)
        if (const int v = split(0x100, 2 * cusPerXcd, 1, 2)) return v;
    if (pair && joins && over <= 0 && 3 * n <= 2 * cusPerXcd && 2 * n > cusPerXcd && nC >= 19)
        if (const int v = split(0x100, 0, 3, 3)) return v;
    if (pair && blocks <= cus) return p.s.nTB * ceil_div(O, 32) > cus && nC >= 4 ? (nC >= 8 ? 0x101 : 0x100) : 0;
    if (blocks <= cus) return nC >= 8 && 20 * blocks >= 11 * cus ? 0x101 : 0;
    return nC >= 4 || (nC >= 2 && 2 * blocks >= 3 * cus) ? 0x100 : 0;
}

extern "C" int drhip_conv3x3_winograd_split_pick_variant(int W, int H, int I, int O) { return ws_pick(W, H, I, O, false); }

// Two f16 parts from 64 input channels on: with fewer their sums are less exact than three bf16 parts' (16 channels 1.34 against 1.11e-7 rms, 32 channels
// 1.45 against 1.32).
extern "C" int drhip_conv3x3_winograd_pair_pick_variant(int W, int H, int I, int O) {
    const int v = I >= 64 ? ws_pick(W, H, I, O, true) : 0;
    return v ? v | 0x200 : 0;
}

extern "C" size_t drhip_conv3x3_winograd_split_filter_floats(int I, int O) {
    return I <= 0 || O <= 0 ? 0 : (size_t)ceil_div(I, kWsKC) * ceil_div(O, 32) * 12288;
}

extern "C" size_t drhip_conv3x3_winograd_split_workspace_floats(int W, int H, int I, int O, int variant) {
    WsPlan p;
    if (!ws_plan(W, H, I, O, variant, &p) || (p.s.sA == 1 && p.s.sB == 1)) return 0;
    const int slots = (p.s.sA > 1 ? p.s.wgsA : 0) + (p.s.sB > 1 ? p.perXcd - p.s.wgsA : 0);     // whole panels need none
    return (size_t)std::max(slots, 1) * kXcds * 8192;       // (never 0 for a variant with pieces: that means it is refused)
}

extern "C" int drhip_winograd_split_filter_transform_f32(const float* w, float* U, int I, int O, void* stream) {
    DRHIP_REQUIRE(w && U && I > 0 && O > 0, "drhip_winograd_split_filter_transform_f32: bad arguments");
    const long long fragments = (long long)ceil_div(I, kWsKC) * ceil_div(O, 32);
    DRHIP_REQUIRE(fragments * 12288 * 4 < (1ll << 31), "drhip_winograd_split_filter_transform_f32: %dx%d filters are too many", I, O);
    launch(wino_split_filter_kernel, dim3((unsigned)fragments), dim3(256), 0, as_stream(stream), w, (unsigned short*)U, I, O, ceil_div(I, kWsKC), ceil_div(O, 32));
    return launched("wino_split_filter_kernel");
}

extern "C" size_t drhip_conv3x3_winograd_pair_filter_floats(int I, int O) {
    return I <= 0 || O <= 0 ? 0 : (size_t)ceil_div(O, 32) * ceil_div(I, kWsKC) * 8192 + WsPairTail::words(ceil_div(I, kWsKC), ceil_div(O, 32));
}

// A filter next to the largest of its output channel.  This is about samples: those of a column of tiles share a scale that follows the largest, so each
// may lose 2^-36 of that.  With no filter below 2^-12 of the largest that loss is below 2^-24 of what the largest sample itself adds to the output (but for
// sums in which it cancels).  At a channel without any weight it adds nothing, however large it is: a filter of zeros, exact as it is, does not fit either
// (samples 2^24 times as large there, rms error of the outputs 6e-4; three parts 1.6e-7).  Filters of nine normally distributed weights are far from that line,
// single weights, as in 1x1 layers, are not.
extern "C" int drhip_winograd_pair_fits(const float* w, int I, int O, int taps) {
    if (!w || I <= 0 || O <= 0 || (taps != 1 && taps != 9)) return 0;
    std::vector<int> least((size_t)O, 0x7fffffff), largest((size_t)O, 0);
    for (int c = 0; c < I; ++c)
        for (int o = 0; o < O; ++o, w += taps) {
            int most = 0;
            for (int k = 0; k < taps; ++k) {
                int bits;
                memcpy(&bits, w + k, sizeof bits);
                most = std::max(most, bits & 0x7fffffff);
            }
            least[o] = std::min(least[o], most);
            largest[o] = std::max(largest[o], most);
        }
    for (int o = 0; o < O; ++o)
        if (!ws_pair_holds(largest[o], least[o])) return 0;
    return 1;
}

extern "C" int drhip_winograd_pair_filter_transform_f32(const float* w, float* U, int I, int O, void* stream) {
    DRHIP_REQUIRE(w && U && I > 0 && O > 0, "drhip_winograd_pair_filter_transform_f32: bad arguments");
    const int nC = ceil_div(I, kWsKC), nOB = ceil_div(O, 32);
    DRHIP_REQUIRE((long long)nC * nOB * 12288 * 4 < (1ll << 31), "drhip_winograd_pair_filter_transform_f32: %dx%d filters are too many", I, O);
    float* tail = U + (size_t)nC * nOB * 8192;
    const WsPairTail t(tail, nC, nOB);
    launch(wino_pair_range_kernel, dim3((32 * nOB + 63) / 64, nC), dim3(256), 0, as_stream(stream), w, t.largest, t.least, I, O, 32 * nOB);
    if (int rc = launched("wino_pair_range_kernel")) return rc;
    launch(wino_pair_filter_kernel, dim3((unsigned)(nC * nOB)), dim3(256), 0, as_stream(stream), w, (unsigned short*)U, tail, I, O, nC, nOB);
    return launched("wino_pair_filter_kernel");
}

extern "C" int drhip_winograd_pair_holds(const float* U, int I, int O, int* holds, void* stream) {
    DRHIP_REQUIRE(U && holds && I > 0 && O > 0, "drhip_winograd_pair_holds: bad arguments");
    const int nC = ceil_div(I, kWsKC), nOB = ceil_div(O, 32);
    std::vector<int> unfit((size_t)nOB);
    const WsPairTail t((float*)U + (size_t)nC * nOB * 8192, nC, nOB);
    if (int rc = drhip_download(unfit.data(), t.unfit, 0, unfit.size() * sizeof(int), stream)) return rc;
    *holds = std::all_of(unfit.begin(), unfit.end(), [](int n) { return n == 0; });
    return DRHIP_OK;
}

extern "C" int drhip_conv3x3_winograd_split_f32(const float* in, const float* U, const float* bias, float* out, int W, int H, int I, int O, int flags, int variant, float* workspace, void* stream) {
    DRHIP_REQUIRE(in && U && out, "drhip_conv3x3_winograd_split_f32: NULL tensor");
    DRHIP_REQUIRE((flags & ~(kEpiRelu | kEpiMaxPool2)) == 0, "drhip_conv3x3_winograd_split_f32: unknown epilogue flags %#x", flags);
    DRHIP_REQUIRE(!(flags & kEpiMaxPool2) || ((W | H) & 1) == 0, "drhip_conv3x3_winograd_split_f32: fused max pooling needs an even map, not %dx%d", W, H);
    WsPlan p;
    DRHIP_REQUIRE(ws_plan(W, H, I, O, variant, &p), "drhip_conv3x3_winograd_split_f32: variant %#x does not cover %dx%dx%d -> %d", variant, W, H, I, O);
    DRHIP_REQUIRE(workspace || (p.s.sA == 1 && p.s.sB == 1), "drhip_conv3x3_winograd_split_f32: variant %#x joins splits and needs a prepared workspace", variant);
    p.s.flags = flags;
    p.s.joinSpins = p.s.sA == 1 && p.s.sB == 1 ? 0 : wino_join_spins();
    p.s.vec2 = ((W & 1) == 0) && (((size_t)out & 7) == 0);
    p.s.pairs = (W & 3) == 0 && ((size_t)out & 7) == 0 && (long long)W * H * 32 * p.kw < (1ll << 31) / 2;
    const unsigned short* F = (const unsigned short*)U;
    hipStream_t st = as_stream(stream);
    return p.pair ? launch_ws<true>(in, F, bias, out, workspace, p, st) : launch_ws<false>(in, F, bias, out, workspace, p, st);
}
