// SGM aggregation with the matching cost computed from the census words on
// the fly (no stored cost volume), for D = 64, 128, 256 (gfx950, wave64).
//
// Same arithmetic as the stored-cost kernels in sgm_kernels.hip (the
// reference's cusgm_cc.cu:118-172 cost and cusgm_ca.cu:1480-1888 recurrence,
// WTA cusgm_ca.cu:3606-3809), so every volume and disparity is bit-identical;
// only where the cost comes from and how lanes are laid out differ:
//
//   * one scanline = D/DPL lanes ("a line"), DPL disparities per lane (16
//     unless FSGM_DPL_* lowers it) held as packed u16 pairs; a wave covers
//     64 DPL / D scanlines.  Neighbour terms
//     d-1 / d+1 across lanes come from row_shr:1 / row_shl:1 DPP moves, the
//     line minimum from quad_perm / mirror DPP reductions.
//   * horizontal directions keep each lane's 16 partner census words in a
//     register window: one step slides it by one disparity, so a lane takes
//     the word its left neighbour drops (one DPP move) and the line's first
//     lane loads the entering word.  The window slots rotate at compile time
//     over a 16-step unrolled block.  A direction whose window would slide the
//     other way runs with the disparity order reversed inside the lanes (the
//     recurrence is symmetric in d).
//   * vertical directions load the census words of the next PF steps into
//     registers (PF = FSGM_PF_V or FSGM_PF_F) and stage, per step, the wave's
//     own words and the D + lines - 1 partner words into one of two LDS
//     slots private to the (single-wave) workgroup; each lane reads its DPL
//     partners from there.
//   * cost(x, t) = popcount(own(x) ^ partner(x, t)): 2 v_xor + 2 v_bcnt, the
//     v_bcnt accumulating onto the step's packed -m'.
//
// The volumes these kernels hand each other are in an order of their own
// (wide_export_kernel undoes it for the stage entry point):
//   * top->bottom: [H][W][D]; left->right and right->left: row tiles, the
//     rows of one horizontal wave side by side per column
//     ([H / lines][W][lines][D], the last tile lower), so that a step of that
//     wave stores 1 KB in one piece instead of `lines` pieces of D bytes.  At
//     D = 64 the pieces are half a cache line, and 32 pairs of 1242x375 took
//     1.63 ms for the two directions against 1.27 ms (the bottom->top kernel,
//     which reads them column by column, went from 1.34 to 1.40 ms).
//   * a reversed direction stays reversed, and a word's bytes are in the order
//     d, d + 2, d + 1, d + 3 (pack_lane).
#include <algorithm>

#include "sgm_device.h"
#include "sgm_internal.h"
#include "sgm_line.h"

#pragma clang fp contract(off)

// prefetch depths (steps) of the top->bottom and fused kernels
#ifndef FSGM_PF_V
#define FSGM_PF_V 8
#endif
#ifndef FSGM_PF_F
#define FSGM_PF_F 4
#endif

namespace fsgm {
namespace {

using namespace dev;

__device__ __forceinline__ uint64_t g64(const uint64_t* p) { return gld(p); }

__device__ __forceinline__ int clampcol(int p, int W) { return (p >= 0 && p < W) ? p : 0; }

// ------------------------------------------------------------ horizontal ---
// Left->right or right->left over the wave's rows.  With t' the lane-local
// order (t' = t, or D-1-t when reversed), the partner column is
//   p(x, t') = a + x + st * t',   and   p(x + dx, t') = p(x, t' - 1),
// so every step the window moves up by one: lane q takes lane q-1's element
// t' = DPL q - 1 and the line's lane 0 loads p(x, 0) = a + x.
template <int D, bool BIG>
__device__ __forceinline__ void wide_horizontal(const SgmJob& J, int path, int group, int lane) {
    constexpr int DPL = wide_dpl(kWideH, D), NP = DPL / 2, LPL = D / DPL, LPW = 64 / LPL;
    const int q = lane % LPL, sub = lane / LPL;
    const bool first = q == 0, last = q == LPL - 1;
    const int W = J.W, H = J.H, roi_x = J.roi_x, min_d = J.min_d;
    int y = group * LPW + sub;
    const bool active = y < H;
    if (!active) y = H - 1;
    const bool fwd = path == kLR;
    const int n = W - roi_x;
    const int x0 = fwd ? roi_x : W - 1, dx = fwd ? 1 : -1;
    const bool right = J.is_right != 0;
    const bool rev = right != (path == kRL);
    const int a = right ? (rev ? min_d + D - 1 : min_d) : (rev ? -min_d - (D - 1) : -min_d);
    const int st = (right != rev) ? 1 : -1;
    const uint64_t* cb = J.census + (int64_t)y * J.cpitch;
    const uint64_t* cm = J.census_other + (int64_t)y * J.cpitch;
    const uint32_t P1v = (uint32_t)J.p1 * 0x10001u, P2v = (uint32_t)J.p2 * 0x10001u;
    const uint32_t sel = rev ? kSelRev : kSelFwd;
    uint8_t* const out_base = (path == kLR) ? J.path[kLR] : J.path[kRL];
    // row tile: the wave's rows side by side per column
    const int ty = group * LPW, trows = min(LPW, H - ty);
    uint8_t* const dst0 =
        out_base + ((int64_t)ty * W + (int64_t)x0 * trows + (y - ty)) * D + q * DPL;
    const int64_t dstep = (int64_t)dx * trows * D;

    // window: slot j holds element t' = DPL q + j at the start of a block
    uint64_t win[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) win[j] = g64(cm + clampcol(a + x0 + st * (DPL * q + j), W));
    Line<NP> s;
    {
        uint32_t c[NP];
        lane_costs<NP>(g64(cb + x0), 0u, [&](int j) { return win[j]; }, c);
        line_init<BIG, LPL>(s, c);
        uint32_t o[NP / 2];
        pack_lane(s, sel, o);
        if (active) store_words<NP / 2>(dst0, o);
    }

    // Census words of a block of DPL steps, fetched one block ahead: lane q
    // of a line loads the own and entering-partner words of steps
    // q + LPL k (k < E), and each step takes them from the line's lane
    // (step mod LPL) by a lane broadcast.  Few, early loads keep the census
    // traffic (many scattered 8-byte reads) off the step's critical path.
    // (Refilling each slot right after its last step instead saves 16
    // registers at D = 64 but waits for stores every LPL steps: 1.62 against
    // 1.27 ms for 32 pairs of 1242x375.)
    constexpr int E = DPL / LPL;
    static_assert(E * LPL == DPL, "a block's steps spread evenly over the line's lanes");
    uint64_t c_own[E], c_in[E], n_own[E], n_in[E];   // this block, next block
    auto xat = [&](int i) { return x0 + dx * min(i, n - 1); };
    auto load_block = [&](int i0, uint64_t (&o)[E], uint64_t (&in)[E]) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < E; ++k) {
            const int x = xat(i0 + q + LPL * k);
            o[k] = g64(cb + x);
            in[k] = g64(cm + clampcol(a + x, W));
        }
    };
    load_block(1, c_own, c_in);
    // blocks of DPL steps: the window slots rotate once per block
    for (int i0 = 1; i0 < n; i0 += DPL) {
        load_block(i0 + DPL, n_own, n_in);
#pragma unroll
        for (int sb = 0; sb < DPL; ++sb) {
            const int i = i0 + sb;
            const uint64_t own = line_bcast64<LPL>(c_own[sb / LPL], sb % LPL);
            const uint64_t in = line_bcast64<LPL>(c_in[sb / LPL], sb % LPL);
            // the slot of the leaving element t' = DPL q + DPL - 1 takes the
            // entering one; element j then sits in slot (e + j) mod DPL
            const int e = (DPL - 1 - sb) & (DPL - 1);
            const uint64_t lv = win[e];
            const uint32_t nlo = from_prev<LPL>((uint32_t)lv, (uint32_t)in, first);
            const uint32_t nhi = from_prev<LPL>((uint32_t)(lv >> 32), (uint32_t)(in >> 32), first);
            win[e] = ((uint64_t)nhi << 32) | nlo;
            uint32_t c[NP];
            lane_costs<NP>(own, 0u - s.m, [&](int j) { return win[(e + j) & (DPL - 1)]; }, c);
            line_step<BIG, LPL>(s, c, P1v, P2v, first, last);
            uint32_t o[NP / 2];
            pack_lane(s, sel, o);
            if (active && i < n) store_words<NP / 2>(dst0 + (int64_t)i * dstep, o);
        }
#pragma unroll
        for (int k = 0; k < E; ++k) {
            c_own[k] = n_own[k];
            c_in[k] = n_in[k];
        }
    }
}

// -------------------------------------------------------------- vertical ---
// Top->bottom (stored) or bottom->top fused with the WTA, over the wave's
// columns.  Per step the wave stages NV = LPW + D + LPW - 1 census words in
// LDS: [0, LPW) its own columns, then the partner columns pbase + k.
template <int D, int DPL>
struct VertGeom {
    static constexpr int LPL = D / DPL, LPW = 64 / LPL;
    static constexpr int NV = D + 2 * LPW - 1;
    static constexpr int NR = (NV + 63) / 64;   // words loaded per lane per step
};

template <int DMAX, int KIND>
struct VertLds {
    static constexpr int NV = (DMAX >= 256) ? VertGeom<256, wide_dpl(KIND, 256)>::NV
                            : (DMAX >= 128) ? VertGeom<128, wide_dpl(KIND, 128)>::NV
                                            : VertGeom<64, wide_dpl(KIND, 64)>::NV;
};

template <int D, bool FUSE, bool BIG>
__device__ __forceinline__ void wide_vertical(const SgmJob& J, int group, int lane, uint64_t* lds,
                                              uint16_t* sums /* FUSE: [lines][D] */) {
    constexpr int KIND = FUSE ? kWideF : kWideV;
    constexpr int DPL = wide_dpl(KIND, D), NP = DPL / 2, NW = NP / 2;
    using G = VertGeom<D, DPL>;
    constexpr int LPL = G::LPL, LPW = G::LPW, NV = G::NV, NR = G::NR;
    const int q = lane % LPL, sub = lane / LPL;
    const bool first = q == 0, last = q == LPL - 1;
    const int W = J.W, H = J.H, roi_x = J.roi_x, min_d = J.min_d;
    const int nlines = W - roi_x;
    const int line0 = group * LPW;
    int line = line0 + sub;
    const bool active = line < nlines;
    if (!active) line = nlines - 1;
    const int c0 = roi_x + line0, x = roi_x + line;
    const int y0 = FUSE ? H - 1 : 0, dy = FUSE ? -1 : 1;
    const bool right = J.is_right != 0;
    const int pbase = right ? c0 + min_d : c0 - min_d - (D - 1);
    // this lane's LDS indices: own word, then partner t = DPL q + j at
    // kp + j (right view) or kp - j (left view)
    const int kown = x - c0;
    const int kp = LPW + (right ? (x - c0) + DPL * q : (x - c0) + (D - 1) - DPL * q);
    const uint32_t P1v = (uint32_t)J.p1 * 0x10001u, P2v = (uint32_t)J.p2 * 0x10001u;
    // volume offsets: a wave-uniform row part and the lane's 32-bit part
    const int64_t ubase = ((int64_t)y0 * W + c0) * D;
    const uint32_t loff = (uint32_t)((x - c0) * D + q * DPL);
    const int64_t off0 = ubase + loff;
    const int64_t ostep = dy * (int64_t)W * D;
    uint8_t* const out_base = FUSE ? J.path[kDU] : J.path[kUD];

    // the other three directions' bytes of step i (FUSE): top->bottom by rows,
    // the horizontal pair in the row tiles of the horizontal kernel, one of
    // them (left->right of the right view, right->left of the left view) with
    // the disparity order reversed
    constexpr int TR = wide_lines(kWideH, D);
    const uint8_t* const src_fwd = right ? J.path[kRL] : J.path[kLR];
    const uint8_t* const src_rev = right ? J.path[kLR] : J.path[kRL];
    auto load_others = [&](int i, uint32_t (&w)[3][NW]) __attribute__((always_inline)) {
        const int y = y0 + dy * min(i, H - 1);
        const int ty = y & -TR, trows = min(TR, H - ty);
        load_words<NW>(J.path[kUD] + ((int64_t)y * W + c0) * D + loff, w[0]);
        const int64_t to = ((int64_t)ty * W + (int64_t)c0 * trows + (y - ty)) * D;
        const uint32_t tv = (uint32_t)((x - c0) * trows * D + q * DPL);
        const uint32_t tr = (uint32_t)((x - c0) * trows * D + (LPL - 1 - q) * DPL);
        load_words<NW>(src_fwd + to + tv, w[1]);
        load_words<NW>(src_rev + to + tr, w[2]);
    };
    // census words staged for step i: lane loads v = lane + 64 r
    auto load_step = [&](int i, uint64_t (&g)[NR]) __attribute__((always_inline)) {
        const int y = y0 + dy * min(i, H - 1);
        const uint64_t* cb = J.census + (int64_t)y * J.cpitch;
        const uint64_t* cm = J.census_other + (int64_t)y * J.cpitch;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int v = min(lane + 64 * r, NV - 1);
            g[r] = (v < LPW) ? g64(cb + min(c0 + v, W - 1)) : g64(cm + clampcol(pbase + v - LPW, W));
        }
    };
    auto stage = [&](int slot, const uint64_t (&g)[NR]) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int v = lane + 64 * r;
            if (v < NV) lds[slot * NV + v] = g[r];
        }
    };
    // The fused kernel up to D = 128 reads a step's words back from LDS beside
    // the arithmetic of the step before: 34 registers more, two waves per SIMD
    // instead of three, and still 1.42 -> 1.39 ms for 32 pairs of 1242x375 and
    // 3.86 -> 3.71 ms for a mixed batch.  At D = 256 (7.1 against 6.7 ms for
    // 4800x3409) and in the top->bottom kernel (10.0 -> 10.7 ms there with the
    // horizontal one, no change at D = 64) it does not pay.
    constexpr bool AHEAD = FUSE && D <= 128;
    uint64_t wo = 0, wp[AHEAD ? DPL : 1];
    auto fetch = [&](int slot) __attribute__((always_inline)) {
        if constexpr (AHEAD) {
            const uint64_t* b = lds + slot * NV;
            wo = b[kown];
#pragma unroll
            for (int j = 0; j < DPL; ++j) wp[j] = right ? b[kp + j] : b[kp - j];
        }
    };
    auto costs = [&](int slot, uint32_t base, uint32_t (&c)[NP]) __attribute__((always_inline)) {
        const uint64_t* b = lds + slot * NV;
        if constexpr (AHEAD) lane_costs<NP>(wo, base, [&](int j) { return wp[j]; }, c);
        else lane_costs<NP>(b[kown], base, [&](int j) { return right ? b[kp + j] : b[kp - j]; }, c);
    };

    // WTA (FUSE): lane q < 4 of a line keeps the integer result of step
    // i0 + q of the 4-step block i0 .. i0 + 3 (i0 = 1 + 4b); the block ends
    // with those lanes finishing their pixels with the float rules.
    const float uthr = 1.0f - J.uniqueness;
    uint32_t kb = 0u, kboth = 0u;
    uint16_t* const sline = sums + sub * D;   // this line's sums (FUSE)
    auto wta_flush = [&](int i0) __attribute__((always_inline)) {
        const int i = i0 + q;
        const int y = y0 - i;
        const int ds = (int)(kb & 0xFFFFu);
        const uint32_t c2 = kb >> 16;
        constexpr bool warp_rule = (D == 64 || D == 128);
        const int rows_cov = warp_rule ? 2 * (H / 2) : H;
        float outv = kInvalidDisp;
        if (y < rows_cov && !(x > W - 5 || y > H - 5 || x < 5 || y < 5) && ds > 0 &&
            (warp_rule || ds < D - 1)) {
            const float c1 = (float)(kboth >> 16);
            const float c2f = (float)c2;
            const float c3 = (ds == D - 1) ? (float)(D - 1) : (float)(kboth & 0xFFFFu);
            const float fa = c1 - c2f, fb = c3 - c2f;
            const float uniq = (fa < fb) ? fa : fb;
            if (!(uniq <= c2f * uthr)) {
                const float t = c1 + c3 - 2.0f * c2f;
                const float den = (1.0f < t) ? t : 1.0f;
                const float bias = (float)((double)(c1 - c3 + den) / (double)(2.0f * den));
                outv = (float)(ds + min_d) + bias;
            }
        }
        if (active && q < 4 && i < H) gst(J.disp + (int64_t)y * W + x, outv);
    };
    auto wta_step = [&](const Line<NP>& s, const uint32_t (&o3)[3][NW], int i) __attribute__((always_inline)) {
        uint32_t S[NP];
#pragma unroll
        for (int k = 0; k < NP; ++k) {
            const int w = k >> 1;
            const uint32_t a0 = word_pair(o3[0][w], k & 1), a1 = word_pair(o3[1][w], k & 1);
            const uint32_t a2 = word_pair(o3[2][NW - 1 - w], (k & 1) ^ 1);
            S[k] = a0 + a1 + a2 + (s.L[k] & 0x00FF00FFu);   // each half <= 1020
        }
        // argmin with the smallest d: inside the lane on u16 keys S * DPL + j
        // (one 32-bit v_lshl_or_b32 per pair shifts both halves without a carry
        // between them, and the keys are finite f16 patterns), then across the
        // line's lanes on (S << 16) | d
        static_assert(wta_key_max(DPL) < kF16Inf && (DPL & (DPL - 1)) == 0, "argmin keys S * DPL + j");
        constexpr int kLog = __builtin_ctz(DPL);
        uint32_t keys[NP];
#pragma unroll
        for (int k = 0; k < NP; ++k) {
            const uint32_t jk = (uint32_t)(2 * k) | ((uint32_t)(2 * k + 1) << 16);
            keys[k] = (S[k] << kLog) | jk;
        }
        const uint32_t key = pk_min_halves(pk_min_all<false>(keys)) & 0xFFFFu;
        uint32_t best = ((key / DPL) << 16) | (uint32_t)(DPL * q + key % DPL);
        best = line_min<LPL>(best);
        const int ds = (int)(best & 0xFFFFu);
        // S(ds - 1) and S(ds + 1): the lanes of a line hold consecutive
        // disparities, so their packed sums laid side by side in LDS are the
        // line's u16 S[d]; every lane then reads the two it needs.  Indices
        // are clamped: S(-1) and S(D) are never used (ds = 0 is invalid, and
        // ds = D - 1 takes c3 = D - 1).
        uint32_t* const mine = reinterpret_cast<uint32_t*>(sline + DPL * q);
#pragma unroll
        for (int k = 0; k < NP; ++k) mine[k] = S[k];
        __builtin_amdgcn_wave_barrier();
        const uint32_t c1 = sline[max(ds - 1, 0)], c3 = sline[min(ds + 1, D - 1)];
        __builtin_amdgcn_wave_barrier();
        if (q == ((i - 1) & 3)) { kb = best; kboth = (c1 << 16) | c3; }
    };

    // rings (PF steps ahead) of census words and, with FUSE, of the other
    // three directions' bytes; the loop body covers BLK steps (with FUSE one
    // 4-step WTA block).  The fused kernel at D = 256 looks 2 steps ahead: its
    // 5 census words per step and lane made 179 registers, two waves per SIMD
    // (4800x3409: 7.8 -> 6.7 ms at 139).
    constexpr int PF = FUSE ? (D == 256 ? 2 : FSGM_PF_F) : FSGM_PF_V;
    constexpr int BLK = (PF > 4) ? PF : 4;
    static_assert(BLK % PF == 0, "the loop body must hold whole ring turns");
    static_assert(!FUSE || BLK == 4, "the WTA finishes its pixels in 4-step blocks");
    uint64_t gr[PF][NR];
    uint32_t pr[FUSE ? PF : 1][3][NW];
    {
        uint64_t g0[NR];
        load_step(0, g0);
        stage(0, g0);
    }
    // the prologue issues the rings in the loop's own order (the wait counts
    // at the loop head merge both paths)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 0; p < PF; ++p) {
        load_step(1 + p, gr[p]);
        if constexpr (FUSE) load_others(1 + p, pr[p]);
        __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_wave_barrier();
    Line<NP> s;
    {
        uint32_t c[NP];
        fetch(0);
        costs(0, 0u, c);
        if constexpr (AHEAD) {
            stage(1, gr[0]);
            load_step(1 + PF, gr[0]);
            __builtin_amdgcn_wave_barrier();
            fetch(1);
        }
        line_init<BIG, LPL>(s, c);
        if constexpr (!FUSE) {
            uint32_t o[NW];
            pack_lane(s, kSelFwd, o);
            if (active) store_words<NW>(out_base + off0, o);
        } else {
            // row H - 1 is a border row of the WTA
            if (active && first) gst(J.disp + (int64_t)y0 * W + x, kInvalidDisp);
        }
    }
    // row offset of step i's store, advanced by a scalar add
    int64_t row_i = ubase + ostep;
    for (int i0 = 1; i0 < H; i0 += BLK) {
#pragma unroll
        for (int b = 0; b < BLK; ++b) {
            const int i = i0 + b, p = b % PF;
            // stage step i (slot i & 1), or with AHEAD step i + 1, whose words
            // replace those of step i once its costs are taken; the other slot
            // still holds the step before
            const int a = AHEAD ? 1 : 0, pa = (p + a) % PF;
            stage((i + a) & 1, gr[pa]);
            load_step(i + a + PF, gr[pa]);
            __builtin_amdgcn_wave_barrier();
            uint32_t c[NP];
            costs(i & 1, 0u - s.m, c);
            fetch((i + 1) & 1);
            line_step<BIG, LPL>(s, c, P1v, P2v, first, last);
            if constexpr (!FUSE) {
                uint32_t o[NW];
                pack_lane(s, kSelFwd, o);
                int64_t r = row_i;
                asm volatile("" : "+s"(r));   // keep it a scalar of its own
                if (active && i < H) store_words<NW>(out_base + r + loff, o);
            } else {
                // consume the slot, then refill it for step i + PF
                wta_step(s, pr[p], i);
                load_others(i + PF, pr[p]);
            }
            row_i += ostep;
        }
        if constexpr (FUSE) wta_flush(i0);
    }
}

// Kernels.  The horizontal (left->right, right->left) and vertical
// (top->bottom, or bottom->top fused with the WTA) scanline code run as
// separate kernels: each fits 4+ waves per SIMD on its own, together they
// would not.  Grid form: item `local` of a job is its scanline group
// (horizontal: left->right groups, then right->left groups).
template <int DMAX, bool BIG, bool ONLY>
__global__ __launch_bounds__(64) void wide_h_kernel(const SgmJob* __restrict__ jobs,
                                                    const int* __restrict__ offs, int njobs) {
    const int item = blockIdx.x;
    const int j = find_job(offs, njobs, item);
    const SgmJob& J = jobs[j];
    const int local = item - offs[j];
    const int lw = wide_lines(kWideH, J.D);
    const int nh = (J.H + lw - 1) / lw;
    const int path = local < nh ? kLR : kRL, group = local < nh ? local : local - nh;
    switch (J.D) {
        case 64: if constexpr (!ONLY || DMAX == 64) wide_horizontal<64, BIG>(J, path, group, threadIdx.x); break;
        case 128: if constexpr (ONLY ? DMAX == 128 : DMAX >= 128) wide_horizontal<128, BIG>(J, path, group, threadIdx.x); break;
        case 256: if constexpr (DMAX >= 256) wide_horizontal<256, BIG>(J, path, group, threadIdx.x); break;
        default: break;
    }
}

// sums of the fused WTA: 64 * DPL u16 per wave (lines x D), largest at DMAX
template <int DMAX>
constexpr int kSumsLen = 64 * wide_dpl(kWideF, DMAX);

template <int DMAX, bool FUSE, bool BIG, bool ONLY>
__global__ __launch_bounds__(64) void wide_v_kernel(const SgmJob* __restrict__ jobs,
                                                    const int* __restrict__ offs, int njobs) {
    __shared__ uint64_t lds[2 * VertLds<DMAX, FUSE ? kWideF : kWideV>::NV];
    __shared__ __align__(16) uint16_t sums[FUSE ? kSumsLen<DMAX> : 1];
    const int item = xcd_item(blockIdx.x, gridDim.x);
    const int j = find_job(offs, njobs, item);
    const SgmJob& J = jobs[j];
    const int group = item - offs[j];
    switch (J.D) {
        case 64: if constexpr (!ONLY || DMAX == 64) wide_vertical<64, FUSE, BIG>(J, group, threadIdx.x, lds, sums); break;
        case 128: if constexpr (ONLY ? DMAX == 128 : DMAX >= 128) wide_vertical<128, FUSE, BIG>(J, group, threadIdx.x, lds, sums); break;
        case 256: if constexpr (DMAX >= 256) wide_vertical<256, FUSE, BIG>(J, group, threadIdx.x, lds, sums); break;
        default: break;
    }
}

// Persistent forms: packed items (job << 16 | direction << 14 | group)
// pulled from a device counter by a fixed grid of resident waves; every wave
// leaves through the one test on the counter.
__device__ __forceinline__ bool next_item(const uint32_t* items, int n, uint32_t* counter, uint32_t* it) {
    uint32_t idx = 0;
    if (threadIdx.x == 0) idx = atomicAdd(counter, 1u);
    idx = (uint32_t)__builtin_amdgcn_readfirstlane((int)__shfl(idx, 0));
    if (idx >= (uint32_t)n) return false;
    *it = items[idx];
    return true;
}

template <int DMAX, bool BIG>
__global__ __launch_bounds__(64) void wide_h_persistent(const SgmJob* __restrict__ jobs,
                                                        const uint32_t* __restrict__ items, int n,
                                                        uint32_t* __restrict__ counter) {
    uint32_t it;
    while (next_item(items, n, counter, &it)) {
        const SgmJob& J = jobs[it >> 16];
        const int path = (int)((it >> 14) & 3u), group = (int)(it & 0x3FFFu);
        switch (J.D) {
            case 64: wide_horizontal<64, BIG>(J, path, group, threadIdx.x); break;
            case 128: if constexpr (DMAX >= 128) wide_horizontal<128, BIG>(J, path, group, threadIdx.x); break;
            case 256: if constexpr (DMAX >= 256) wide_horizontal<256, BIG>(J, path, group, threadIdx.x); break;
            default: break;
        }
    }
}

template <int DMAX, bool FUSE, bool BIG>
__global__ __launch_bounds__(64) void wide_v_persistent(const SgmJob* __restrict__ jobs,
                                                        const uint32_t* __restrict__ items, int n,
                                                        uint32_t* __restrict__ counter) {
    __shared__ uint64_t lds[2 * VertLds<DMAX, FUSE ? kWideF : kWideV>::NV];
    __shared__ __align__(16) uint16_t sums[FUSE ? kSumsLen<DMAX> : 1];
    uint32_t it;
    while (next_item(items, n, counter, &it)) {
        const SgmJob& J = jobs[it >> 16];
        const int group = (int)(it & 0x3FFFu);
        switch (J.D) {
            case 64: wide_vertical<64, FUSE, BIG>(J, group, threadIdx.x, lds, sums); break;
            case 128: if constexpr (DMAX >= 128) wide_vertical<128, FUSE, BIG>(J, group, threadIdx.x, lds, sums); break;
            case 256: if constexpr (DMAX >= 256) wide_vertical<256, FUSE, BIG>(J, group, threadIdx.x, lds, sums); break;
            default: break;
        }
    }
}

// A plan whose jobs all have one D runs the kernel of that D alone: the code
// of several ranges in one kernel takes the registers of the largest.
hipError_t launch_h(const StagePlan& p, hipStream_t s) {
    if (p.n_wh <= 0) return hipSuccess;
    const dim3 g(p.n_wh), b(64);
    auto go = [&](auto ker) { hipLaunchKernelGGL(ker, g, b, 0, s, p.jobs, p.offs_wh, p.njobs); };
    if (p.big) go(wide_h_kernel<256, true, false>);
    else if (p.dmax <= 64) go(wide_h_kernel<64, false, true>);
    else if (p.dmin == p.dmax) p.dmax == 128 ? go(wide_h_kernel<128, false, true>) : go(wide_h_kernel<256, false, true>);
    else p.dmax <= 128 ? go(wide_h_kernel<128, false, false>) : go(wide_h_kernel<256, false, false>);
    return hipGetLastError();
}

template <bool FUSE>
hipError_t launch_v(const StagePlan& p, hipStream_t s) {
    const int n = FUSE ? p.n_wf : p.n_wv;
    const int* offs = FUSE ? p.offs_wf : p.offs_wv;
    if (n <= 0) return hipSuccess;
    const dim3 g(n), b(64);
    auto go = [&](auto ker) { hipLaunchKernelGGL(ker, g, b, 0, s, p.jobs, offs, p.njobs); };
    if (p.big) go(wide_v_kernel<256, FUSE, true, false>);
    else if (p.dmax <= 64) go(wide_v_kernel<64, FUSE, false, true>);
    else if (p.dmin == p.dmax) p.dmax == 128 ? go(wide_v_kernel<128, FUSE, false, true>) : go(wide_v_kernel<256, FUSE, false, true>);
    else p.dmax <= 128 ? go(wide_v_kernel<128, FUSE, false, false>) : go(wide_v_kernel<256, FUSE, false, false>);
    return hipGetLastError();
}

hipError_t launch_h_persistent(const StagePlan& p, const uint32_t* items, int n, uint32_t* counter,
                               int grid, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const dim3 g(grid), b(64);
    auto go = [&](auto ker) { hipLaunchKernelGGL(ker, g, b, 0, s, p.jobs, items, n, counter); };
    if (p.big) go(wide_h_persistent<256, true>);
    else if (p.dmax <= 64) go(wide_h_persistent<64, false>);
    else p.dmax <= 128 ? go(wide_h_persistent<128, false>) : go(wide_h_persistent<256, false>);
    return hipGetLastError();
}

template <bool FUSE>
hipError_t launch_v_persistent(const StagePlan& p, const uint32_t* items, int n, uint32_t* counter,
                               int grid, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const dim3 g(grid), b(64);
    auto go = [&](auto ker) { hipLaunchKernelGGL(ker, g, b, 0, s, p.jobs, items, n, counter); };
    if (p.big) go(wide_v_persistent<256, FUSE, true>);
    else if (p.dmax <= 64) go(wide_v_persistent<64, FUSE, false>);
    else p.dmax <= 128 ? go(wide_v_persistent<128, FUSE, false>) : go(wide_v_persistent<256, FUSE, false>);
    return hipGetLastError();
}

// Internal direction volumes to plain [H][W][D] ones: a word's bytes back in
// order, and for the horizontal directions (`tiled`) the row tiles and the
// reversed disparity order of `rev` undone.
__global__ __launch_bounds__(256) void wide_export_kernel(const uint32_t* __restrict__ src,
                                                          uint32_t* __restrict__ dst, int W, int H,
                                                          int D, int roi_x, int tile, int rev) {
    const int nw = D / 4;
    const int64_t n = (int64_t)H * W * nw;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int k = (int)(i % nw);
        const int64_t pix = i / nw;
        const int x = (int)(pix % W), y = (int)(pix / W);
        if (x < roi_x) continue;   // not matched: left as it is
        const int ty = y / tile * tile, trows = min(tile, H - ty);
        const int64_t sp = (int64_t)ty * W + (int64_t)x * trows + (y - ty);
        const uint32_t w = src[sp * nw + (rev ? nw - 1 - k : k)];
        const uint32_t a = w & 0x00FF00FFu, b = (w >> 8) & 0x00FF00FFu;   // pairs (0, 1), (2, 3)
        dst[i] = rev ? pack4(b, a) : pack4(a, b);
    }
}

}  // namespace

// left->right + right->left, then top->bottom (one stream, in order)
hipError_t launch_wide3(const StagePlan& p, hipStream_t s) {
    const hipError_t e = launch_h(p, s);
    return e != hipSuccess ? e : launch_v<false>(p, s);
}

hipError_t launch_wide_wta(const StagePlan& p, hipStream_t s) { return launch_v<true>(p, s); }

// schedule: items3 = [horizontal items (n3h)][top->bottom items]; counters
// [0] horizontal, [1] bottom->top, [2] top->bottom
hipError_t launch_wide3_sched(const StagePlan& p, const AggSchedule& sc, hipStream_t s) {
    hipError_t e = launch_reset_counters(sc.counters, 3, s);
    if (e != hipSuccess) return e;
    if ((e = launch_h_persistent(p, sc.items3, sc.n3h, sc.counters, sc.grid, s)) != hipSuccess) return e;
    return launch_v_persistent<false>(p, sc.items3 + sc.n3h, sc.n3 - sc.n3h, sc.counters + 2, sc.grid, s);
}

hipError_t launch_wide_wta_sched(const StagePlan& p, const AggSchedule& sc, hipStream_t s) {
    return launch_v_persistent<true>(p, sc.items_dw, sc.ndw, sc.counters + 1, sc.grid, s);
}

hipError_t launch_wide_export(const SgmJob& j, const uint8_t* const (&src)[4],
                              uint8_t* const (&dst)[4], hipStream_t s) {
    const int64_t n = (int64_t)j.H * j.W * (j.D / 4);
    const unsigned blocks = (unsigned)std::min<int64_t>((n + 255) / 256, 65535);
    for (int r : {(int)kUD, (int)kLR, (int)kRL}) {
        const int tile = r == kUD ? 1 : wide_lines(kWideH, j.D);
        const int rev = r != kUD && (j.is_right != 0) != (r == kRL);
        hipLaunchKernelGGL(wide_export_kernel, dim3(blocks), dim3(256), 0, s,
                           reinterpret_cast<const uint32_t*>(src[r]),
                           reinterpret_cast<uint32_t*>(dst[r]), j.W, j.H, j.D, j.roi_x, tile, rev);
    }
    return hipGetLastError();
}

// resident waves per CU: the smallest over the three persistent kernels
hipError_t wide_occupancy(const StagePlan& p, int* per_cu) {
    int a = 0, b = 0, c = 0;
    hipError_t e;
    if (p.dmax <= 64) {
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, wide_h_persistent<64, false>, 64, 0);
        if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, wide_v_persistent<64, false, false>, 64, 0);
        if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&c, wide_v_persistent<64, true, false>, 64, 0);
    } else if (p.dmax <= 128) {
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, wide_h_persistent<128, false>, 64, 0);
        if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, wide_v_persistent<128, false, false>, 64, 0);
        if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&c, wide_v_persistent<128, true, false>, 64, 0);
    } else {
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, wide_h_persistent<256, false>, 64, 0);
        if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, wide_v_persistent<256, false, false>, 64, 0);
        if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&c, wide_v_persistent<256, true, false>, 64, 0);
    }
    if (e == hipSuccess) *per_cu = std::max(1, std::min(a, std::min(b, c)));
    return e;
}

}  // namespace fsgm
