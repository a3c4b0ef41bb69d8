// Coarse-to-fine pyramid kernels for CDNA4 (gfx950): 2x decimation,
// initial-disparity propagation, and the per-pixel-window cost, aggregation
// and WTA of the finer levels (ethan-li-coding/FasterStereoCuda:
// FasterStereoCuda.cpp:114-166, SgmStereoCuda/cusgm_cc.cu:14-21, 173-237,
// 294-360, cusgm_ca.cu:1181-1339, 3425-3512).
//
// A finer level searches LR (16 or 32) disparities t around a per-pixel base
// b(p): d = b(p) + t.  Its aggregation keeps one disparity per lane (a wave
// holds 64/LR scanlines) because the previous pixel's window is shifted by
// b - b' and the neighbour terms index L'[t + b - b' -+ 1] -- an arbitrary
// lane shift, fetched with ds_bpermute.  Arithmetic is uint32 with the
// reference's wrap-around after INVALID base pixels.
#include <algorithm>
#include <atomic>
#include <mutex>

#include "pyr_internal.h"

#pragma clang fp contract(off)

namespace fsgm {
namespace {

constexpr int kInvalidShort = -32768;

__device__ __forceinline__ uint32_t bperm(int src_lane, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute(src_lane << 2, (int)v);
}

// lanes whose source is outside the row read 0 (bound_ctrl), so the move
// needs no zeroed destination first
template <int CTRL>
__device__ __forceinline__ uint32_t dppu(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}

// minimum over each aligned group of LR lanes (LR = 16 or 32)
template <int LR>
__device__ __forceinline__ uint32_t group_min(uint32_t m, int lane) {
    m = min(m, dppu<0x128>(m));
    m = min(m, dppu<0x124>(m));
    m = min(m, dppu<0x122>(m));
    m = min(m, dppu<0x121>(m));
    if constexpr (LR == 32) m = min(m, bperm(lane ^ 16, m));
    return m;
}

__global__ __launch_bounds__(256) void zoom_kernel(PyrZoom z) {
    const int wd = z.w / 2, hd = z.h / 2;
    const int64_t n = (int64_t)wd * hd;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= 2 * n) return;
    const int v = i >= n;
    const int64_t k = v ? i - n : i;
    const int y = (int)(k / wd), x = (int)(k - (int64_t)y * wd);
    const uint8_t* src = v ? z.src_r : z.src_l;
    uint8_t* dst = v ? z.dst_r : z.dst_l;
    dst[k] = src[(int64_t)(2 * y) * z.w + 2 * x];
}

// FasterStereoCuda.cpp:138-166.  Row i takes its value from row
// src_row(i): odd rows copy the row above, and the last row (when even)
// copies the row above it, which copies the one above that.
__global__ __launch_bounds__(256) void init_next_kernel(PyrInit a) {
    const int64_t n = (int64_t)a.w * a.h;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int y = (int)(i / a.w), x = (int)(i - (int64_t)y * a.w);
    int r = y;
    if (r % 2 == 1) r -= 1;            // odd row: the even row above
    else if (r == a.h - 1) r -= 2;     // even last row: row above, itself a copy of y-2
    int16_t v = kInvalidShort;
    if (r >= 0) {
        const int wc = a.w >> 1;
        const float d = a.coarse[(int64_t)(r >> 1) * wc + min(x >> 1, wc - 1)];
        if (d != kInvalidDisp) v = (int16_t)(2 * d - (a.level_range >> 1));
    }
    a.next[i] = v;
}

__device__ __forceinline__ uint32_t cost_adjust(int t, int lr) {
    // (uint8)expf(k) for the integer exponent k = 4|t - LR/2| / (LR/2) in 0..4
    const int half = lr / 2;
    const int k = min(4 * abs(t - half) / half, 4);
    return k == 0 ? 1u : k == 1 ? 2u : k == 2 ? 7u : k == 3 ? 20u : 54u;
}

// cost with initial disparity, left view: xr = x - t - b;
// 0 < xr < W -> popc + CostAdjust(t); else 0xFF (9x7) or 127 (5x5)
template <int LR>
__global__ __launch_bounds__(256) void cost_init_kernel(PyrLevel a) {
    const int64_t n = (int64_t)a.w * a.h;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int y = (int)(i / a.w), x = (int)(i - (int64_t)y * a.w);
    const int b = a.init[i];
    const uint64_t cl = a.census_l[i];
    const uint64_t* cr = a.census_r + (int64_t)y * a.w;
    const uint32_t invalid = a.cs_type ? 0xFFu : 127u;
    uint32_t words[LR / 4];
#pragma unroll
    for (int k = 0; k < LR / 4; ++k) words[k] = 0u;
    if (x - b - (LR - 1) > 0 && x - b < a.w) {
        // every partner column of the window is inside the image (all but
        // the pixels near the borders and those with an invalid base)
        const uint64_t* crb = cr + (x - b);
#pragma unroll
        for (int t = 0; t < LR; ++t) {
            const uint32_t c = (uint32_t)__popcll(cl ^ crb[-t]) + cost_adjust(t, LR);
            words[t >> 2] |= (c & 0xFFu) << (8 * (t & 3));
        }
    } else {
#pragma unroll
        for (int t = 0; t < LR; ++t) {
            const int xr = x - t - b;
            uint32_t c = invalid;
            if (xr > 0 && xr < a.w) c = (uint32_t)__popcll(cl ^ cr[xr]) + cost_adjust(t, LR);
            words[t >> 2] |= (c & 0xFFu) << (8 * (t & 3));
        }
    }
    uint4* dst = reinterpret_cast<uint4*>(a.cost + i * LR);
#pragma unroll
    for (int q = 0; q < LR / 16; ++q)
        dst[q] = make_uint4(words[4 * q], words[4 * q + 1], words[4 * q + 2], words[4 * q + 3]);
}

// Aggregation over the per-pixel window (cusgm_ca.cu:1181-1339), one
// disparity per lane, SPW = 64 / LR scanlines per wave.  Step rules, with b
// and b' the window bases of this and the previous pixel: the neighbour
// terms read the previous L at window index t + b - 1 - b' and t + b + 1 - b'
// plus P1 (127 outside [0, LR)), the same-d term is L(t) unshifted, P2 is
// max(P1, P2 / max(1, |b' - b + 1|)), and a pixel with an invalid base keeps
// the previous L and b' and sets m' = 127.  The first pixel of a vertical
// scanline takes b' from row 0.  A scanline is walked in blocks of K = LR steps.  For the loads
// and stores lane j stands for pixel (line j / K, step j % K) of a block: it
// fetches that pixel's whole window (LR cost bytes) and base disparity one
// block ahead, and the block passes through a per-wave LDS area, from which
// every step reads its byte and base.  Each step's results are gathered
// there and leave as one LR-byte store per lane and block.  (Loading one
// byte per lane and step, and waiting for it, made the scanline walk
// latency-bound.)  Pixels whose base is invalid are never read by the WTA;
// they are written as 0.
template <int LR>
struct AggInitLds {
    uint8_t cost[64 * LR];   // [line][step][t]
    uint8_t out[64 * LR];
    int16_t init[64];        // [line][step]
    uint32_t pen2[256];      // max(P1, P2 / k), k = max(1, index)
};

template <int LR, bool PEN2_TABLE>
__device__ __forceinline__ void agg_init_lines(const PyrLevel& a, int dir, int group, int lane,
                                               AggInitLds<LR>& S) {
    constexpr int SPW = 64 / LR, K = LR, NV = LR / 16;
    const int sub = lane / LR, t = lane % LR;        // recurrence: line, disparity
    const int lsub = lane / K, lstep = lane % K;     // loads / stores: line, step
    const bool horiz = (dir == 1 || dir == 3);
    const bool fwd = (dir == 0 || dir == 1);
    const int W = a.w, H = a.h;
    const int nlines = horiz ? H : W;
    const int n = horiz ? W : H;
    // pixel of (line, step); lines past the last and steps past the end are
    // clamped (computed, never stored)
    auto pix_of = [&](int line, int step) -> int64_t {
        line = min(line, nlines - 1);
        step = min(step, n - 1);
        const int pos = fwd ? step : n - 1 - step;
        return horiz ? (int64_t)line * W + pos : (int64_t)pos * W + line;
    };
    const int line = min(group * SPW + sub, nlines - 1);
    const int lline = group * SPW + lsub;
    uint8_t* out = (dir == 0) ? a.path[0] : (dir == 1) ? a.path[1] : (dir == 2) ? a.path[2] : a.path[3];
    const uint32_t p1 = (uint32_t)a.p1;
    const int gbase = sub * LR;

    static_assert(NV == 1 || NV == 2, "windows of 16 or 32 bytes");
    uint4 nc0 = make_uint4(0u, 0u, 0u, 0u), nc1 = nc0;   // named, so they stay in registers
    int nb = 0;
    auto fetch = [&](int blk) __attribute__((always_inline)) {
        const int64_t p = pix_of(lline, blk * K + lstep);
        const uint4* src = reinterpret_cast<const uint4*>(a.cost + p * LR);
        nc0 = src[0];
        if constexpr (NV == 2) nc1 = src[1];
        nb = a.init[p];
    };
    auto stage = [&]() __attribute__((always_inline)) {
        uint4* dst = reinterpret_cast<uint4*>(S.cost + lane * LR);
        dst[0] = nc0;
        if constexpr (NV == 2) dst[1] = nc1;
        S.init[lane] = (int16_t)nb;
    };

    // P2 / max(1, |b' - b + 1|) by table (PEN2_TABLE, for P2 <= 254): every
    // divisor from 255 on gives P2 / k = 0, the same as entry 255, so the
    // table is exact.  A larger P2 divides (an integer division costs ~15
    // VALU per step).
    if constexpr (PEN2_TABLE) {
#pragma unroll
        for (int k = lane; k < 256; k += 64) S.pen2[k] = (uint32_t)max(a.p1, a.p2 / max(1, k));
    }

    uint32_t L = 0, m = 0;
    int last_b = 0;
    const int nblk = (n + K - 1) / K;
    fetch(0);
    stage();
    if (nblk > 1) fetch(1);
    for (int blk = 0; blk < nblk; ++blk) {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s = 0; s < K; ++s) {
            const uint32_t c = S.cost[(sub * K + s) * LR + t];
            const int b = S.init[sub * K + s];
            uint32_t o;
            if (s == 0 && blk == 0) {
                L = c;
                m = group_min<LR>(L, lane);
                // A11: vertical directions seed b' from row 0 whichever end they start at
                last_b = horiz ? b : a.init[line];
                o = L;
            } else {
                const bool valid = b != kInvalidShort;
                const int i1 = t + b - 1 - last_b, i2 = t + b + 1 - last_b;
                const uint32_t v1 = bperm(gbase + min(max(i1, 0), LR - 1), L);
                const uint32_t v2 = bperm(gbase + min(max(i2, 0), LR - 1), L);
                const uint32_t bm = (i1 >= 0 && i1 < LR) ? v1 + p1 : 127u;
                const uint32_t bp = (i2 >= 0 && i2 < LR) ? v2 + p1 : 127u;
                const int div = max(1, abs(last_b - b + 1));
                uint32_t pen2;
                if constexpr (PEN2_TABLE) pen2 = S.pen2[min(div, 255)];
                else pen2 = (uint32_t)max(a.p1, a.p2 / div);
                const uint32_t v = min(min(L, bm), min(bp, m + pen2));
                const uint32_t l = c + (v - m);
                const uint32_t mn = group_min<LR>(l, lane);
                o = valid ? l : 0u;
                L = valid ? l : L;
                m = valid ? mn : 127u;
                last_b = valid ? b : last_b;
            }
            S.out[(sub * K + s) * LR + t] = (uint8_t)o;
        }
        __builtin_amdgcn_wave_barrier();
        {   // this block's results, one window per lane
            const int step = blk * K + lstep;
            if (lline < nlines && step < n) {
                uint4* dst = reinterpret_cast<uint4*>(out + pix_of(lline, step) * LR);
                const uint4* src = reinterpret_cast<const uint4*>(S.out + lane * LR);
#pragma unroll
                for (int q = 0; q < NV; ++q) dst[q] = src[q];
            }
        }
        if (blk + 1 < nblk) {
            stage();
            if (blk + 2 < nblk) fetch(blk + 2);
        }
    }
}

template <int LR>
__global__ __launch_bounds__(64) void agg_init_kernel(PyrLevel a) {
    __shared__ __align__(16) AggInitLds<LR> lds;
    constexpr int SPW = 64 / LR;
    const int nh = (a.h + SPW - 1) / SPW, nv = (a.w + SPW - 1) / SPW;
    const int item = blockIdx.x;
    int dir, group;
    if (item < nh) { dir = 1; group = item; }
    else if (item < 2 * nh) { dir = 3; group = item - nh; }
    else if (item < 2 * nh + nv) { dir = 0; group = item - 2 * nh; }
    else { dir = 2; group = item - 2 * nh - nv; }
    if (a.p2 <= 254) agg_init_lines<LR, true>(a, dir, group, threadIdx.x, lds);
    else agg_init_lines<LR, false>(a, dir, group, threadIdx.x, lds);
}

// The same aggregation with NP packed u16 pairs per lane (2 NP disparities):
// LPL = LR / (2 NP) lanes per scanline, SPW = 64 / LPL scanlines per wave, a
// block of K = LR / 2 steps (NP pixels per lane), and every VALU instruction
// of a step works on two cells.  A step needs the neighbour pairs that start
// at f + q - 1, f + q + 1, .. (f: the lane's first disparity, q = b - b'); the
// middle one of NP = 2 serves both of its pairs.
//
// Where no line of the wave shifts its window by more than one disparity, the
// shifted pairs are this lane's and its neighbours' (DPP), picked by a byte
// selector.  The selector, the P2 term, the validity and the base of the last
// valid pixel before (a scan over the block's steps) are worked out per pixel
// by the lane that loads it, not per step by every lane of the scanline, and
// the steps where some line shifts by more are known to the wave, as bits of a
// scalar, before the block is walked.  In such a step each line's L + P1 is
// written as a row of overlapping pairs, C[e] = (L'[e - PAD], L'[e - PAD + 1])
// + P1, padded on both sides with 127, and a lane reads the pairs it needs,
// dword-aligned whatever the parity of q.  (Reading the u16 of a plain row is a
// misaligned LDS access, and its stalls took most of the time.)  A pad is
// exactly the 127 of a neighbour outside the window, so no range test remains.
// q is clamped to +-(LR + 1), past which every term is a pad, and, separately,
// to [-254, 256] to index a table of max(P1, P2 / max(1, |1 - q|)).
//
// A wave that is alone on its SIMD waits out every latency, so LDS is read a
// block ahead: while block i is walked, block i + 1 is staged and read into
// registers, and the results of block i - 1 are read back and stored.
//
// Exact when P1 <= 127 and P2 <= 254: the true (unbounded) values of the
// recurrence then lie in [-382, 763] (l <= c + P2 <= 509, and l >= 127 - m
// after a neighbour outside the window), so the minima of their u16
// representatives pick the same entries as those of their u32
// representatives, and the stored low bytes agree.  Other penalties take
// agg_init_kernel.
//
// What bounds it: the chain of a scanline's dependent steps at one or two waves
// per SIMD (20 instructions per step, 16 more for its share of the staging; a
// wide step waits for LDS).  Staging and streaming alone take 0.47 of 0.77 ms
// for 4800x3409 in quads.  Rows of unpadded LDS put all of an access's lanes
// on 8 banks (quads 0.87 -> 0.77 ms, window 32 0.77 -> 0.51 ms).  With that, the
// reads a block ahead and the per-pixel preparation, against the form that
// worked out every step's shift in the step: 4800x3409 window 16 0.79 -> 0.66
// ms, 7000x5000 1.44 -> 1.20, 2900x2200 window 32 0.64 -> 0.49, 850x600 window
// 32 0.27 -> 0.21, 1600x1200 window 16 0.20 -> 0.19, 800x600 0.094 -> 0.100.
typedef unsigned short pk16 __attribute__((ext_vector_type(2)));
typedef unsigned int pyr_u32x4 __attribute__((ext_vector_type(4)));

// A block's pixels as buffer accesses from a base that moves by a fixed step
// per block, each pixel at an offset from it fixed for the whole walk.  A
// pixel past the scanlines or the line's end gets an offset beyond the
// resource's range: it loads 0 and its store is dropped, so every block issues
// the same accesses with no branch around them, and the compiler counts the
// prefetch ring's outstanding loads exactly instead of draining them.  Block
// blk of scanline group l0 holds pixel (scanline l0 + ln, step blk K + j); the
// base is the lowest such pixel, offsets stay below (64 + K) W LR bytes.  In
// the reverse directions the base of a line's last, partial block (and of the
// blocks past it) lies before the volume: only pixels inside the line are in
// range, and their offsets land inside it.
template <int K>
struct BlockPixels {
    int64_t base0, step;   // base pixel at block 0, and its move per block
    __device__ BlockPixels(bool horiz, bool fwd, int W, int n, int l0) {
        base0 = horiz ? (int64_t)l0 * W + (fwd ? 0 : n - K) : (fwd ? 0 : (int64_t)(n - K) * W) + l0;
        step = (horiz ? 1 : (int64_t)W) * (fwd ? K : -K);
    }
    // pixels from the base to (ln, j)
    __device__ static uint32_t offset(bool horiz, bool fwd, int W, int ln, int j) {
        const int jj = fwd ? j : K - 1 - j;
        return (uint32_t)(horiz ? ln * W + jj : jj * W + ln);
    }
};
// Successive blocks of a volume of `bytes` per pixel.
struct BlockWalk {
    uintptr_t base, step;
    template <int K>
    __device__ BlockWalk(const BlockPixels<K>& px, const void* volume, int bytes, int blk)
        : base((uintptr_t)volume + (uintptr_t)((px.base0 + blk * px.step) * bytes)),
          step((uintptr_t)(px.step * bytes)) {}
    __device__ __amdgpu_buffer_rsrc_t next() {
        const uintptr_t b = base;
        base += step;
        return __builtin_amdgcn_make_buffer_rsrc((void*)b, (short)0, 0x7fffffff, 0x00020000);
    }
};

constexpr int kPkDeltaLo = -254, kPkDeltaHi = 256;   // table range of b - b'
// Blocks of cost loads in flight per wave, so that the HBM latency (1-2 us
// under load) is spread over that many blocks of steps.
template <int LR> constexpr int kPkAheadOf = LR == 16 ? 4 : 2;   // 32 steps

template <int LR, int NP>
struct AggInitPkLds {
    static constexpr int LPL = LR / (2 * NP), SPW = 64 / LPL, K = LR / 2;
    static constexpr int PAD = (LR + 2 + 3) / 4 * 4;         // a multiple of 4: aligned row stores
    static constexpr int ROW = (PAD + 2 * LR + 1 + 3) / 4 * 4;   // reads reach PAD + 2 LR
    // Strides that spread the lanes of an access over the 64 banks: staging
    // writes K steps of 64 / K lines per pair (a line stride of K more than a
    // multiple of 64 words), a step writes a word or half of one per lane.
    static constexpr int PAIR = K + 4, LINE = LR / 2 * PAIR + K, OUT = LR * (K + 1);
    uint32_t cost[SPW * LINE];               // [line][pair][step]: the pair's costs as u16
    uint32_t sel[64 * NP], pen[64 * NP];     // [line][step]: selector and P2 term of a shift of at most
                                             // one, or the shift itself
    uint8_t out[SPW * OUT];                  // [line][step][t]
    alignas(16) int16_t valid[64 * NP];      // [line][step]: 0 or all ones
    uint32_t pen2[kPkDeltaHi - kPkDeltaLo + 1];   // by b - b', both halves
    alignas(16) uint32_t win[SPW][ROW];      // overlapping pairs, see above
};

__device__ __forceinline__ uint32_t pk_bits(pk16 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ pk16 pk_of(uint32_t v) { return __builtin_bit_cast(pk16, v); }
__device__ __forceinline__ pk16 pk_min2(pk16 a, pk16 b) { return __builtin_elementwise_min(a, b); }

// v_perm selector of bytes 2 (q + 1) .. 2 (q + 1) + 3 of {hi, lo} for a
// window shift q in {-1, 0, 1}: the dword starting one disparity below, at,
// or one above the middle of the pair boundary.  Other q (pixels whose step
// is skipped) are clamped into that range; their result is not used.
// Three full-rate instructions: q clamped by v_med3, then 24-bit multiply-adds
// (written out: the compiler merges the steps into one quarter-rate 32-bit
// multiply).  The constants come in registers (no literals in VOP3).
__device__ __forceinline__ uint32_t shift_sel(int q, uint32_t k0202, uint32_t k10001, uint32_t kbase) {
    uint32_t t, u, sel;
    asm volatile(   // not moved into a branch
        "v_med3_i32 %0, %3, -1, 1\n\t"
        "v_mad_i32_i24 %1, %0, %4, %4\n\t"     // (q + 1) * 0x0202
        "v_mad_u32_u24 %2, %1, %5, %6"           // u * 0x10001 + 0x03020100
        : "=&v"(t), "=&v"(u), "=v"(sel)
        : "v"(q), "s"(k0202), "v"(k10001), "s"(kbase));
    return sel;
}

template <int LR, int NP>
__device__ __forceinline__ void agg_init_pk_lines(const PyrLevel& a, int dir, int group, int lane,
                                                  AggInitPkLds<LR, NP>& S) {
    using Lds = AggInitPkLds<LR, NP>;
    constexpr int LPL = Lds::LPL, SPW = Lds::SPW, K = Lds::K, PAD = Lds::PAD;
    constexpr int NV = LR / 16, kPkAhead = kPkAheadOf<LR>;
    constexpr uint32_t kPadPair = 127u * 0x10001u;
    static_assert(SPW * K == 64 * NP, "a block is NP pixels per lane");
    // The lanes of a scanline sit STRIDE = 16 / LPL apart in one DPP row, so a
    // neighbouring lane's pair is a row shift by STRIDE.  The line's first and
    // last lanes then read from outside the row, which leaves a move's old
    // value in place: the 127 pads stay in those lanes of two persistent
    // registers, with no select per step.
    constexpr int STRIDE = 16 / LPL;
    const int sub = (lane / 16) * STRIDE + lane % STRIDE;   // recurrence: line
    const int k = (lane % 16) / STRIDE;                     // lane of the line
    const bool horiz = (dir == 1 || dir == 3);
    const bool fwd = (dir == 0 || dir == 1);
    const int W = a.w, H = a.h;
    const int nlines = horiz ? H : W;
    const int n = horiz ? W : H;
    uint8_t* out = (dir == 0) ? a.path[0] : (dir == 1) ? a.path[1] : (dir == 2) ? a.path[2] : a.path[3];

    // loads and stores: lane j handles the block's pixels j, j + 64 in
    // [line][step] order
    const BlockPixels<K> px(horiz, fwd, W, n, group * SPW);
    const int lstep = lane % K;              // 64 is a multiple of K
    uint32_t off[NP];
    bool on_line[NP];
#pragma unroll
    for (int h = 0; h < NP; ++h) {
        const int ln = (lane + 64 * h) / K;
        off[h] = BlockPixels<K>::offset(horiz, fwd, W, ln, lstep);
        on_line[h] = group * SPW + ln < nlines;
    }
    auto inside = [&](int h, int blk) __attribute__((always_inline)) {
        return on_line[h] && lstep < n - blk * K;
    };
    // a ring of kPkAhead blocks of loads in flight (slot = block mod kPkAhead)
    pyr_u32x4 nc[kPkAhead][NP][NV];
    uint16_t nb[kPkAhead][NP];
    BlockWalk costs(px, a.cost, LR, 0), bases(px, a.init, 2, 0), outs(px, out, LR, -1);
    auto fetch = [&](int slot, int blk) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rc = costs.next(), rb = bases.next();
#pragma unroll
        for (int h = 0; h < NP; ++h) {
            const bool in = inside(h, blk);
#pragma unroll
            for (int v = 0; v < NV; ++v)
                nc[slot][h][v] = __builtin_amdgcn_raw_buffer_load_b128(
                    rc, (int)(in ? off[h] * LR + 16 * v : 0x80000000u), 0, 0);
            nb[slot][h] = __builtin_amdgcn_raw_buffer_load_b16(rb, (int)(in ? off[h] * 2 : 0x80000000u), 0, 0);
        }
    };

    for (int e = lane; e < SPW * Lds::ROW; e += 64) (&S.win[0][0])[e] = kPadPair;
    for (int e = lane; e <= kPkDeltaHi - kPkDeltaLo; e += 64) {
        const int q = e + kPkDeltaLo;
        const uint32_t v = (uint32_t)max(a.p1, a.p2 / max(1, abs(1 - q)));
        S.pen2[e] = v | (v << 16);
    }
    __builtin_amdgcn_wave_barrier();

    uint32_t* wrow = &S.win[sub][0];
    const uint32_t* wlane = wrow + (PAD - 1 + 2 * NP * k);     // + q: the first neighbour pair
    const bool last_k = k == LPL - 1;
    uint8_t* obase = S.out + sub * Lds::OUT + 2 * NP * k;
    const pk16 p1v = pk_of((uint32_t)a.p1 * 0x10001u);
    const pk16 m127 = pk_of(kPadPair);
    const uint32_t k10001 = 0x10001u;
    // P2 terms of the shifts -1, 0 and 1 (divisors 2, 1 and 1)
    const uint32_t pen2_m1 = S.pen2[-1 - kPkDeltaLo], pen2_01 = S.pen2[0 - kPkDeltaLo];
    auto small_pen = [=](int q) __attribute__((always_inline)) {
        const uint32_t neg = 0u - (uint32_t)(q < 0);
        return (pen2_m1 & neg) | (pen2_01 & ~neg);
    };

    // A11: vertical directions seed b' from row 0 whichever end they start at
    int seed[NP], pb[NP];                    // pb: last valid bases of the block before
#pragma unroll
    for (int h = 0; h < NP; ++h) {
        seed[h] = horiz ? 0 : a.init[min(group * SPW + (lane + 64 * h) / K, nlines - 1)];
        pb[h] = 0;
    }
    // A block into LDS: the costs transposed, so that a lane later reads the
    // cost pairs of all K steps of its line with wide loads (zero-extended to
    // u16), and what each pixel's step needs.  Returns the steps at which some
    // line shifts by more than one, as bits, and kInvalid if a pixel is invalid.
    constexpr uint32_t kInvalid = 1u << 16;
    auto stage = [&](int slot, int blk) __attribute__((always_inline)) -> uint32_t {
        int b[NP], q[NP];
        uint32_t kind = 0u;
#pragma unroll
        for (int h = 0; h < NP; ++h) {
            uint32_t wv[LR / 4];
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                wv[4 * v] = nc[slot][h][v].x; wv[4 * v + 1] = nc[slot][h][v].y;
                wv[4 * v + 2] = nc[slot][h][v].z; wv[4 * v + 3] = nc[slot][h][v].w;
            }
#pragma unroll
            for (int j = 0; j < LR / 2; ++j)
                S.cost[(lane + 64 * h) / K * Lds::LINE + j * Lds::PAIR + lstep] =
                    __builtin_amdgcn_perm(0u, wv[j / 2], (j & 1) ? 0x0c030c02u : 0x0c010c00u);
            b[h] = (int)(int16_t)nb[slot][h];
            // v: the base of the last valid pixel up to this one (none: the
            // marker, whose distance is past every window, as it should be)
            const int before = __builtin_amdgcn_mov_dpp(pb[h], 0x100 + K - 1, 0xF, 0xF, true);   // row_shl:K-1
            int v = b[h];
            if (lstep == 0) {
                if (blk == 0) v = horiz ? v : seed[h];
                else v = v == kInvalidShort ? before : v;
            }
            if (__builtin_amdgcn_ballot_w64(b[h] == kInvalidShort) != 0) {
                kind |= kInvalid;
                auto pull = [&](int d, int from) __attribute__((always_inline)) {
                    v = v == kInvalidShort && lstep >= d ? from : v;
                };
                pull(1, __builtin_amdgcn_mov_dpp(v, 0x111, 0xF, 0xF, true));   // row_shr:1, 2, 4, 8
                pull(2, __builtin_amdgcn_mov_dpp(v, 0x112, 0xF, 0xF, true));
                pull(4, __builtin_amdgcn_mov_dpp(v, 0x114, 0xF, 0xF, true));
                if constexpr (K == 16) pull(8, __builtin_amdgcn_mov_dpp(v, 0x118, 0xF, 0xF, true));
            }
            const int last = __builtin_amdgcn_mov_dpp(v, 0x111, 0xF, 0xF, true);
            q[h] = b[h] - (lstep == 0 ? before : last);
            pb[h] = v;
            const bool far = (uint32_t)(q[h] + 1) > 2u && b[h] != kInvalidShort && inside(h, blk) &&
                             (blk > 0 || lstep > 0);
            uint64_t f = __builtin_amdgcn_ballot_w64(far);
            f |= f >> 32;
            f |= f >> 16;
            if constexpr (K == 8) f |= f >> 8;
            kind |= (uint32_t)f & ((1u << K) - 1u);
        }
#pragma unroll
        for (int h = 0; h < NP; ++h) {
            const int idx = lane + 64 * h;
            S.valid[idx] = (int16_t)(b[h] == kInvalidShort ? 0 : -1);
            const uint32_t sel = shift_sel(q[h], 0x0202u, k10001, 0x03020100u);
            S.sel[idx] = (kind >> lstep) & 1u ? (uint32_t)q[h] : sel;
            S.pen[idx] = small_pen(q[h]);
        }
        return kind;
    };
    // a staged block as this lane walks it
    struct Block {
        uint32_t valid[K / 2], cost[NP][K], sel[K], pen[K];
    };
    auto wide = [](const void* src, int words, uint32_t* dst) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < words / 4; ++i) {
            const uint4 v = reinterpret_cast<const uint4*>(src)[i];
            dst[4 * i] = v.x; dst[4 * i + 1] = v.y; dst[4 * i + 2] = v.z; dst[4 * i + 3] = v.w;
        }
    };
    auto take = [&](Block& B) __attribute__((always_inline)) {
        wide(&S.valid[sub * K], K / 2, B.valid);
#pragma unroll
        for (int i = 0; i < NP; ++i) wide(&S.cost[sub * Lds::LINE + (NP * k + i) * Lds::PAIR], K, B.cost[i]);
        wide(&S.sel[sub * K], K, B.sel);
        wide(&S.pen[sub * K], K, B.pen);
    };

    // the window row from this lane's pairs of L + P1: the lane's pairs and
    // the ones between them, and C[PAD - 1] from the first lane
    auto put = [&](const uint32_t (&o)[NP]) __attribute__((always_inline)) {
        uint32_t nxt = dppu<0x100 + STRIDE>(o[0]);        // row_shl: the next lane's first pair
        nxt = last_k ? kPadPair : nxt;
        uint32_t* dst = wrow + PAD + 2 * NP * k;
        if constexpr (NP == 2)
            *reinterpret_cast<uint4*>(dst) =
                make_uint4(o[0], __builtin_amdgcn_alignbit(o[1], o[0], 16), o[1],
                           __builtin_amdgcn_alignbit(nxt, o[1], 16));
        else
            *reinterpret_cast<uint2*>(dst) = make_uint2(o[0], __builtin_amdgcn_alignbit(nxt, o[0], 16));
        if (k == 0) wrow[PAD - 1] = (o[0] << 16) | 127u;
    };
    // minimum over the scanline's lanes of both halves, in both halves
    auto line_min = [&](const pk16 (&v)[NP]) __attribute__((always_inline)) {
        pk16 w = v[0];
        if constexpr (NP == 2) w = pk_min2(w, v[1]);
        w = pk_min2(w, w.yx);
        uint32_t r = pk_bits(w);                          // equal halves: u32 order = u16 order
        r = min(r, dppu<0x120 + STRIDE>(r));              // row_ror by STRIDE, 2 STRIDE, ...
        if constexpr (2 * STRIDE < 16) r = min(r, dppu<0x120 + 2 * STRIDE>(r));
        if constexpr (4 * STRIDE < 16) r = min(r, dppu<0x120 + 4 * STRIDE>(r));
        if constexpr (8 * STRIDE < 16) r = min(r, dppu<0x120 + 8 * STRIDE>(r));
        return pk_of(r);
    };
    uint32_t nxt_r = kPadPair, prv_r = kPadPair;   // pads kept in the last / first lane of a line
    // neighbour pairs for a shift in {-1, 0, 1}: bytes 2 (q + 1) .. 2 (q + 1) + 3
    // of {first, the lane before's last}, ..., {the next lane's first, last}
    auto dpp_pairs = [&](const uint32_t (&o)[NP], uint32_t sel, uint32_t (&x)[NP + 1]) __attribute__((always_inline)) {
        nxt_r = (uint32_t)__builtin_amdgcn_update_dpp((int)nxt_r, (int)o[0], 0x100 + STRIDE, 0xF, 0xF, false);
        prv_r = (uint32_t)__builtin_amdgcn_update_dpp((int)prv_r, (int)o[NP - 1], 0x110 + STRIDE, 0xF, 0xF, false);
        x[0] = __builtin_amdgcn_perm(o[0], prv_r, sel);
        if constexpr (NP == 2) x[1] = __builtin_amdgcn_perm(o[1], o[0], sel);
        x[NP] = __builtin_amdgcn_perm(nxt_r, o[NP - 1], sel);
    };
    pk16 L[NP], m = pk_of(0u);
#pragma unroll
    for (int i = 0; i < NP; ++i) L[i] = pk_of(0u);
    // this step's L from the previous L, m and the neighbour pairs
    auto relax = [&](const Block& B, int s, const uint32_t (&x)[NP + 1], uint32_t pen, pk16 (&l)[NP])
        __attribute__((always_inline)) {
        const pk16 t = pk_min2(pk_of(x[1]), m + pk_of(pen));
        l[0] = pk_min2(pk_min2(L[0], pk_of(x[0])), t);
        if constexpr (NP == 2) l[1] = pk_min2(pk_min2(L[1], pk_of(x[2])), t);
#pragma unroll
        for (int i = 0; i < NP; ++i) l[i] = pk_of(B.cost[i][s]) - m + l[i];
    };
    // the low bytes of a step's results
    auto emit = [&](int s, const pk16 (&l)[NP], uint32_t mask) __attribute__((always_inline)) {
        if constexpr (NP == 2)
            *reinterpret_cast<uint32_t*>(obase + s * LR) =
                __builtin_amdgcn_perm(pk_bits(l[1]), pk_bits(l[0]), 0x06040200u) & mask;
        else
            *reinterpret_cast<uint16_t*>(obase + s * LR) =
                (uint16_t)(__builtin_amdgcn_perm(0u, pk_bits(l[0]), 0x0c0c0200u) & mask);
    };

    // a block with no invalid pixel and no wide step
    auto straight = [&](const Block& B) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < K; ++s) {
            uint32_t o[NP], x[NP + 1];
#pragma unroll
            for (int i = 0; i < NP; ++i) o[i] = pk_bits(L[i] + p1v);
            dpp_pairs(o, B.sel[s], x);
            pk16 l[NP];
            relax(B, s, x, B.pen[s], l);
            m = line_min(l);
#pragma unroll
            for (int i = 0; i < NP; ++i) L[i] = l[i];
            emit(s, l, ~0u);
        }
    };
    auto mixed = [&](const Block& B, uint32_t wide_steps, bool first) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < K; ++s) {
            if (s == 0 && first) {
#pragma unroll
                for (int i = 0; i < NP; ++i) L[i] = pk_of(B.cost[i][0]);
                m = line_min(L);
                emit(0, L, ~0u);
                continue;
            }
            uint32_t o[NP], x[NP + 1], pen;
#pragma unroll
            for (int i = 0; i < NP; ++i) o[i] = pk_bits(L[i] + p1v);
            if ((wide_steps >> s & 1u) == 0) {
                dpp_pairs(o, B.sel[s], x);
                pen = B.pen[s];
            } else {
                const int q = (int)B.sel[s];
                const int qw = min(max(q, -(LR + 1)), LR + 1);
                if constexpr (NP == 1) {
                    // the three pairs from disparity 2k + q - 1 (rounded down
                    // to even) on, straight from their lanes
                    const int e = 2 * k + qw - 1, j = e >> 1;
                    uint32_t p[3];
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        const uint32_t v = bperm(lane - k * STRIDE + (j + i) * STRIDE, o[0]);
                        p[i] = (uint32_t)(j + i) < (uint32_t)LPL ? v : kPadPair;
                    }
                    const uint32_t sel = e & 1 ? 0x05040302u : 0x03020100u;
                    x[0] = __builtin_amdgcn_perm(p[1], p[0], sel);
                    x[1] = __builtin_amdgcn_perm(p[2], p[1], sel);
                } else {
                    put(o);    // the window row holds L only when a step needs it
#pragma unroll
                    for (int i = 0; i <= NP; ++i) x[i] = wlane[qw + 2 * i];
                }
                pen = S.pen2[min(max(q, kPkDeltaLo), kPkDeltaHi) - kPkDeltaLo];
            }
            pk16 l[NP];
            relax(B, s, x, pen, l);
            const pk16 mn = line_min(l);
            // an invalid pixel keeps L, sets m to 127 and leaves 0; selects as
            // bit operations (v_bfi), so the step stays one block
            const uint32_t vm = (uint32_t)(int)(int16_t)(B.valid[s / 2] >> (16 * (s & 1)));
            emit(s, l, NP == 2 ? vm : vm & 0xFFFFu);
#pragma unroll
            for (int i = 0; i < NP; ++i) L[i] = pk_of((pk_bits(l[i]) & vm) | (pk_bits(L[i]) & ~vm));
            m = pk_of((pk_bits(mn) & vm) | (pk_bits(m127) & ~vm));
        }
    };

    const int nblk = (n + K - 1) / K;
    // a block's results, one window per pixel: read back, then stored
    auto results = [&](uint4 (&r)[NP][NV]) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < NP; ++h)
#pragma unroll
            for (int v = 0; v < NV; ++v)
                r[h][v] = reinterpret_cast<const uint4*>(S.out + (lane + 64 * h) / K * Lds::OUT + lstep * LR)[v];
    };
    auto store = [&](const uint4 (&r)[NP][NV], int blk) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rs = outs.next();
#pragma unroll
        for (int h = 0; h < NP; ++h) {
            const uint32_t o = inside(h, blk) && blk >= 0 ? off[h] * LR : 0x80000000u;
#pragma unroll
            for (int v = 0; v < NV; ++v)
                __builtin_amdgcn_raw_buffer_store_b128(pyr_u32x4{r[h][v].x, r[h][v].y, r[h][v].z, r[h][v].w}, rs,
                                                       (int)(o + 16 * v), 0, 0);
        }
    };

    // the prologue issues the ring's slots in the loop's order: the wait
    // counts at the loop head merge both paths
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kPkAhead; ++u) {
        fetch(u, u);
        __builtin_amdgcn_sched_barrier(0);
    }
    Block B[2];
    uint32_t kind = stage(0, 0);
    fetch(0, kPkAhead);
    __builtin_amdgcn_wave_barrier();
    take(B[0]);
    kind |= kInvalid;                        // the first pixel has a rule of its own
    int blk0 = 0;
    do {
#pragma unroll
        for (int u = 0; u < kPkAhead; ++u) {
            // blocks past the last one (at most kPkAhead - 1) hold nothing;
            // their stores are dropped
            const int blk = blk0 + u;
            uint4 r[NP][NV];
            __builtin_amdgcn_wave_barrier();
            results(r);                                          // block blk - 1
            const uint32_t next = stage((u + 1) % kPkAhead, blk + 1);
            __builtin_amdgcn_wave_barrier();
            take(B[(u + 1) % 2]);
            store(r, blk - 1);
            fetch((u + 1) % kPkAhead, blk + 1 + kPkAhead);
            __builtin_amdgcn_wave_barrier();
            if (__builtin_expect(kind == 0, 1)) straight(B[u % 2]);
            else mixed(B[u % 2], kind, blk == 0);
            kind = next;
        }
        blk0 += kPkAhead;
    } while (blk0 <= nblk);                  // one block further: the last one's results
}

template <int LR, int NP>
__global__ __launch_bounds__(64) void agg_init_pk_kernel(PyrLevel a) {
    __shared__ __align__(16) AggInitPkLds<LR, NP> lds;
    constexpr int SPW = AggInitPkLds<LR, NP>::SPW;
    const int nh = (a.h + SPW - 1) / SPW, nv = (a.w + SPW - 1) / SPW;
    const int item = blockIdx.x;
    int dir, group;
    if (item < nh) { dir = 1; group = item; }
    else if (item < 2 * nh) { dir = 3; group = item - nh; }
    else if (item < 2 * nh + nv) { dir = 0; group = item - 2 * nh; }
    else { dir = 2; group = item - 2 * nh - nv; }
    agg_init_pk_lines<LR, NP>(a, dir, group, threadIdx.x, lds);
}

// WTA with initial disparity (cusgm_ca.cu:3425-3512), one lane per pixel
template <int LR>
__global__ __launch_bounds__(256) void wta_init_kernel(PyrLevel a) {
    const int64_t n = (int64_t)a.w * a.h;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int y = (int)(i / a.w), x = (int)(i - (int64_t)y * a.w);
    const int W = a.w, H = a.h;
    float out = kInvalidDisp;
    const int b = a.init[i];
    if (y < 4 * (H / 4) && !(x > W - 5 || y > H - 5 || x < 5 || y < 5) && b != kInvalidShort) {
        uint32_t S[LR];
#pragma unroll
        for (int t = 0; t < LR; ++t) S[t] = 0u;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint8_t* pr = (r == 0) ? a.path[0] : (r == 1) ? a.path[1] : (r == 2) ? a.path[2] : a.path[3];
            const uint4* src = reinterpret_cast<const uint4*>(pr + i * LR);
#pragma unroll
            for (int q = 0; q < LR / 16; ++q) {
                const uint4 v = src[q];
                const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int k = 0; k < 16; ++k) S[q * 16 + k] += (w4[k >> 2] >> (8 * (k & 3))) & 0xFFu;
            }
        }
        uint32_t c2 = 0xFFFFFFFFu;
        int ds = 0;
#pragma unroll
        for (int t = 0; t < LR; ++t)
            if (S[t] < c2) { c2 = S[t]; ds = t; }
        if (ds > 1 && ds < LR - 1) {
            uint32_t s1 = 0, s3 = 0;
#pragma unroll
            for (int t = 0; t < LR; ++t) {
                s1 = (t == ds - 1) ? S[t] : s1;
                s3 = (t == ds + 1) ? S[t] : s3;
            }
            const float c1 = (float)s1, c2f = (float)c2, c3 = (float)s3;
            const float aa = c1 - c2f, bb = c3 - c2f;
            const float uniq = (aa < bb) ? aa : bb;
            if (!(uniq <= c2f * (1.0f - a.uniqueness))) {
                const float tt = c1 + c3 - 2.0f * c2f;
                const float den = (1.0f < tt) ? tt : 1.0f;
                const float bias = (float)((double)(c1 - c3 + den) / (double)(2.0f * den));
                out = (float)(ds + b) + bias;
            }
        }
    }
    a.disp[i] = out;
}

// cusgm_df.cu:188-218: INVALID interior pixels take their window maximum
__global__ __launch_bounds__(256) void dilation_kernel(const float* __restrict__ in,
                                                       float* __restrict__ out, int W, int H,
                                                       int wnd) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)W * H) return;
    const int y = (int)(i / W), x = (int)(i - (int64_t)y * W);
    const int r = (wnd - 1) / 2;
    float v = in[i];
    if (v == kInvalidDisp && x > r && x < W - r && y > r && y < H - r)
        for (int a = -r; a <= r; ++a)
            for (int b = -r; b <= r; ++b) v = fmaxf(v, in[(int64_t)(y + b) * W + x + a]);
    out[i] = v;
}

inline unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

hipError_t pyr_launch_zoom(const PyrZoom& z, hipStream_t s) {
    const int64_t n = 2 * (int64_t)(z.w / 2) * (z.h / 2);
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(zoom_kernel, dim3(blocks_for(n)), dim3(256), 0, s, z);
    return hipGetLastError();
}

hipError_t pyr_launch_dilation(const float* in, float* out, int w, int h, int wnd, hipStream_t s) {
    hipLaunchKernelGGL(dilation_kernel, dim3(blocks_for((int64_t)w * h)), dim3(256), 0, s, in, out,
                       w, h, wnd);
    return hipGetLastError();
}

hipError_t pyr_launch_init_next(const PyrInit& a, hipStream_t s) {
    hipLaunchKernelGGL(init_next_kernel, dim3(blocks_for((int64_t)a.w * a.h)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t pyr_launch_cost_init(const PyrLevel& a, hipStream_t s) {
    const dim3 g(blocks_for((int64_t)a.w * a.h)), b(256);
    if (a.level_range == 16) hipLaunchKernelGGL(cost_init_kernel<16>, g, b, 0, s, a);
    else hipLaunchKernelGGL(cost_init_kernel<32>, g, b, 0, s, a);
    return hipGetLastError();
}

// Whether the packed-u16 window aggregation is exact for these penalties.
static bool agg_init_packed_ok(const PyrLevel& a) { return a.p1 <= 127 && a.p2 <= 254; }

static std::atomic<int> g_window_form{SGM_WINDOW_AUTO};
int window_form() { return g_window_form.load(); }
void set_window_form(int form) { g_window_form.store(form); }

// SIMDs of the current device (4 per compute unit), looked up once per device
static int device_simds() {
    static std::mutex mu;
    static int simds[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 1024;
    std::lock_guard<std::mutex> lock(mu);
    if (!simds[dev]) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            cus <= 0)
            cus = 256;
        simds[dev] = 4 * cus;
    }
    return simds[dev];
}

hipError_t pyr_launch_aggregate_init(const PyrLevel& a, hipStream_t s) {
    auto items = [&](int spw) { return 2 * ((a.h + spw - 1) / spw) + 2 * ((a.w + spw - 1) / spw); };
    int form = window_form();
    if (!agg_init_packed_ok(a)) form = SGM_WINDOW_U32;
    // Quads issue fewer instructions per cell, pairs have twice the waves and
    // the shorter step.  Pairs / quads, us: window 16, 4800x3409 (1.0 quad waves
    // per SIMD) 661 / 785, 7000x5000 (1.5) 1195 / 1221, 9600x6800 (2.0) 2330 /
    // 2250; window 32, 1700x1200 (0.7) 205 / 271, 2900x2200 (1.2) 538 / 493.
    if (form == SGM_WINDOW_AUTO)
        form = items(256 / a.level_range) >= (a.level_range == 16 ? 2 : 1) * device_simds() ? SGM_WINDOW_QUADS
                                                                                           : SGM_WINDOW_PAIRS;
    if (form == SGM_WINDOW_QUADS) {
        const int n = items(256 / a.level_range);
        if (a.level_range == 16) hipLaunchKernelGGL((agg_init_pk_kernel<16, 2>), dim3(n), dim3(64), 0, s, a);
        else hipLaunchKernelGGL((agg_init_pk_kernel<32, 2>), dim3(n), dim3(64), 0, s, a);
        return hipGetLastError();
    }
    if (form == SGM_WINDOW_PAIRS) {
        const int n = items(128 / a.level_range);
        if (a.level_range == 16) hipLaunchKernelGGL((agg_init_pk_kernel<16, 1>), dim3(n), dim3(64), 0, s, a);
        else hipLaunchKernelGGL((agg_init_pk_kernel<32, 1>), dim3(n), dim3(64), 0, s, a);
        return hipGetLastError();
    }
    if (a.level_range == 16) {
        const int n = items(4);
        hipLaunchKernelGGL(agg_init_kernel<16>, dim3(n), dim3(64), 0, s, a);
    } else {
        const int n = items(2);
        hipLaunchKernelGGL(agg_init_kernel<32>, dim3(n), dim3(64), 0, s, a);
    }
    return hipGetLastError();
}

hipError_t pyr_launch_wta_init(const PyrLevel& a, hipStream_t s) {
    const dim3 g(blocks_for((int64_t)a.w * a.h)), b(256);
    if (a.level_range == 16) hipLaunchKernelGGL(wta_init_kernel<16>, g, b, 0, s, a);
    else hipLaunchKernelGGL(wta_init_kernel<32>, g, b, 0, s, a);
    return hipGetLastError();
}

}  // namespace fsgm
