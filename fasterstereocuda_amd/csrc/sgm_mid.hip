// SGM aggregation with the cost from the census words, for plans too small to
// fill the GPU with the waves of sgm_wide.hip (gfx950, wave64).
//
// Same arithmetic and results as sgm_wide.hip and the stored-cost kernels.  A
// wave is four 16-lane lines with D / 16 disparities per lane, so a plan has
// 4 (D = 64), 2 (D = 128) or as many waves (D = 256) and a lone wave's step is
// short: about one wave per SIMD, a step costs its instruction count.  Hence:
//   * census rows are padded with the word of column 0 (what a partner column
//     outside the image reads; column 0 is a border pixel, so the word is a
//     constant, which the census kernel writes): no clamps.  A vertical step's partner words go
//     through an LDS slot private to the wave, loaded PF steps
//     ahead, and are read back a step ahead;
//   * buffer accesses with a scalar offset per step; volumes are plain
//     [H][W][D] (32-bit offsets, see mid_ok), only their words' byte order is
//     that of sgm_wide.hip (pack_lane), and left->right of the right view and
//     right->left of the left view hold the disparities reversed;
//   * every step stores (a last group's lines past the region repeat its last
//     line), so the waits are exact;
//   * the horizontal and the top->bottom lines run in one launch, long ones
//     first; then bottom->top with the WTA.
// The 5x5 right view's skipped-pixel rule (cusgm_cc.cu:288: the last pixel of
// every D-pixel block has the left view's cost) makes its columns lines of
// their own in the vertical directions, computed as the left view's, and
// replaces the costs of their steps in the horizontal ones.
#include <algorithm>
#include <type_traits>

#include "sgm_device.h"
#include "sgm_internal.h"
#include "sgm_line.h"

#pragma clang fp contract(off)

namespace fsgm {
namespace {

using namespace dev;

// N consecutive census words (N a multiple of 4) in ascending address order
template <int N>
__device__ __forceinline__ void load_census(__amdgpu_buffer_rsrc_t r, uint32_t v, int s, uint64_t (&w)[N]) {
#pragma unroll
    for (int k = 0; k < N; k += 2) {
        const buf_u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(v + 8 * k), s, 0);
        w[k] = ((uint64_t)t.y << 32) | t.x;
        w[k + 1] = ((uint64_t)t.w << 32) | t.z;
    }
}
__device__ __forceinline__ uint64_t load_word(__amdgpu_buffer_rsrc_t r, uint32_t v, int s) {
    const buf_u32x2 t = __builtin_amdgcn_raw_buffer_load_b64(r, (int)v, s, 0);
    return ((uint64_t)t.y << 32) | t.x;
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_of(const SgmJob& J, const uint64_t* census) {
    return buf_at(reinterpret_cast<const uint8_t*>(census - J.cpad));
}

// ------------------------------------------------------------ horizontal ---
// As sgm_wide.hip's wide_horizontal: each lane keeps its partner words in a
// register window that slides by one disparity per step; blocks of 16 steps
// take the own and entering words their lanes loaded a block earlier.
template <int D, bool BIG, bool QUIRK>
__device__ __forceinline__ void mid_horizontal(const SgmJob& J, int path, int group, int lane) {
    constexpr int DPL = D / 16, NP = DPL / 2, NW = NP / 2;
    const int q = lane & 15, sub = lane >> 4;
    const int W = J.W, H = J.H, roi_x = J.roi_x, min_d = J.min_d;
    const int line0 = group * 4;
    const int y = min(line0 + sub, H - 1);
    const int n = W - roi_x;
    const bool fwd = path == kLR;
    const int x0 = fwd ? roi_x : W - 1, dx = fwd ? 1 : -1;
    const bool right = J.is_right != 0;
    const bool rev = right != (path == kRL);
    const int a = right ? (rev ? min_d + D - 1 : min_d) : (rev ? -min_d - (D - 1) : -min_d);
    const int st = (right != rev) ? 1 : -1;
    const uint32_t P1v = (uint32_t)J.p1 * 0x10001u, P2v = (uint32_t)J.p2 * 0x10001u;
    const uint32_t sel = rev ? kSelRev : kSelFwd;
    // census words: scalar row of the group's first line + the lane's rest
    const auto own_r = rows_of(J, J.census), oth_r = rows_of(J, J.census_other);
    const int rowb = J.cpitch * 8, srow = line0 * rowb;
    const uint32_t vrow = (uint32_t)((y - line0) * rowb + J.cpad * 8);
    auto word = [&](__amdgpu_buffer_rsrc_t r, int col) __attribute__((always_inline)) {
        return load_word(r, vrow + (uint32_t)(col * 8), srow);
    };
    const auto out = buf_at(path == kLR ? J.path[kLR] : J.path[kRL]);
    const uint32_t vout = (uint32_t)((y - line0) * W * D + q * DPL);
    const int sout0 = (line0 * W + x0) * D, dstep = dx * D;

    // the left view's cost of column x (skipped-pixel rule): its own word is
    // the other view's, its partners this view's columns x - min_d - t
    auto quirk_costs = [&](int i, uint32_t (&c)[NP]) __attribute__((always_inline)) {
        const int x = x0 + dx * i;
        const int p0 = x - min_d - (rev ? D - 1 : 0), sg = rev ? 1 : -1;
        uint64_t w[DPL];
#pragma unroll
        for (int j = 0; j < DPL; ++j) w[j] = word(own_r, p0 + sg * (DPL * q + j));
        lane_costs<NP>(word(oth_r, x), 0u, [&](int j) { return w[j]; }, c);
    };
    // the next such step at or after i: positions D - 1 mod D from roi_x, and
    // the last column (the last step left->right, step 0 right->left)
    auto quirk_step = [&](int i) {
        const int r = fwd ? (D - 1 - i % D + D) % D : ((n - i) % D + D) % D;
        return i + r;
    };

    uint64_t win[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) win[j] = word(oth_r, a + x0 + st * (DPL * q + j));
    Line<NP> s;
    {
        uint32_t c[NP];
        lane_costs<NP>(word(own_r, x0), 0u, [&](int j) { return win[j]; }, c);
        if constexpr (QUIRK)
            if (right && J.cs_type == 0 && (quirk_step(0) == 0 || !fwd || n == 1)) quirk_costs(0, c);
        line_init<BIG, 16>(s, c);
        uint32_t o[NW];
        pack_lane(s, sel, o);
        buf_store<NW>(out, vout, sout0, o);
    }
    uint64_t c_own, c_in, n_own, n_in;   // lane q: the words of the block's step q
    auto load_block = [&](int i0, uint64_t& o, uint64_t& in) __attribute__((always_inline)) {
        const int x = x0 + dx * min(i0 + q, n - 1);
        o = word(own_r, x);
        in = word(oth_r, a + x);
    };
    load_block(1, c_own, c_in);
    auto block = [&](int i0, auto full, auto quirk) __attribute__((always_inline)) {
        load_block(i0 + 16, n_own, n_in);
        int s1 = -1, s2 = -1;
        uint32_t q1[NP], q2[NP];
        if constexpr (quirk.value) {
            s1 = quirk_step(i0);
            s2 = fwd ? n - 1 : -1;
            if (s1 < n) quirk_costs(s1, q1);
            if (fwd) quirk_costs(n - 1, q2);
        }
        int so = sout0 + i0 * dstep;
#pragma unroll
        for (int sb = 0; sb < 16; ++sb) {
            const uint64_t own = line_bcast64<16>(c_own, sb), in = line_bcast64<16>(c_in, sb);
            // the slot of the leaving element t' = DPL q + DPL - 1 takes the
            // entering one; element j then sits in slot (e + j) mod DPL
            const int e = (15 - sb) & (DPL - 1);
            const uint64_t lv = win[e];
            const uint32_t nlo = dpp<kRowShr1>((uint32_t)in, (uint32_t)lv);
            const uint32_t nhi = dpp<kRowShr1>((uint32_t)(in >> 32), (uint32_t)(lv >> 32));
            win[e] = ((uint64_t)nhi << 32) | nlo;
            uint32_t c[NP];
            lane_costs<NP>(own, 0u - s.m, [&](int j) { return win[(e + j) & (DPL - 1)]; }, c);
            if constexpr (quirk.value) {
#pragma unroll
                for (int k = 0; k < NP; ++k)
                    c[k] = i0 + sb == s1 ? q1[k] - s.m : i0 + sb == s2 ? q2[k] - s.m : c[k];
            }
            line_step<BIG, 16>(s, c, P1v, P2v, false, false);
            uint32_t o[NW];
            pack_lane(s, sel, o);
            if (full.value || i0 + sb < n) buf_store<NW>(out, vout, so, o);
            so += dstep;
        }
        c_own = n_own;
        c_in = n_in;
    };
    const bool quirk_job = QUIRK && right && J.cs_type == 0;
    int i0 = 1;
    for (; i0 + 16 <= n; i0 += 16) {
        if constexpr (QUIRK) {
            if (quirk_job && (quirk_step(i0) < i0 + 16 || (fwd && n - 1 < i0 + 16))) {
                block(i0, std::true_type{}, std::true_type{});
                continue;
            }
        }
        block(i0, std::true_type{}, std::false_type{});
    }
    if (i0 < n) {
        if constexpr (QUIRK) {
            if (quirk_job) {
                block(i0, std::false_type{}, std::true_type{});
                return;
            }
        }
        block(i0, std::false_type{}, std::false_type{});
    }
}

// -------------------------------------------------------------- vertical ---
// Top->bottom (stored), or bottom->top with the WTA, over four columns.  A
// lane's partner columns are x + min_d + DPL q + j (right view) or
// x - min_d - (DPL q + j) (left view, and the special columns of a 5x5 right
// view with the two censuses exchanged).  The columns of a group lie within
// five, so a step stages KW = 128 NR >= D + 4 words; the special ones lie D
// apart and load their words themselves.
//
// Word v of a staged step sits at v ^ ((v >> 5 & 3) << 2): lanes DPL words
// apart would otherwise meet in a quarter (DPL = 8) or an eighth (DPL = 16) of
// the LDS banks.
__device__ __forceinline__ int lds_slot(int v) { return v ^ (((v >> 5) & 3) << 2); }
template <int D> constexpr int kStageLoads = (D + 4 + 127) / 128;
template <int D> constexpr int kStageWords = 128 * kStageLoads<D>;

struct MidColumns {
    int x, x0;       // this lane's column, the group's first
    bool active;
    bool special;    // wave-uniform
};
__device__ __forceinline__ MidColumns mid_columns(const SgmJob& J, int group, int sub) {
    const int D = J.D, n = J.W - J.roi_x, sp = mid_specials(J), normal = n - sp;
    const int ng = (normal + 3) / 4;
    MidColumns c;
    c.special = group >= ng;
    int line = (c.special ? group - ng : group) * 4 + sub;
    const int lines = c.special ? sp : normal;
    c.active = line < lines;
    line = min(line, lines - 1);
    // special columns: the last of every D-column block, and the last one
    int pos = line;
    if (c.special) pos = min((line + 1) * D - 1, n - 1);
    else if (sp > 0) pos = line + line / (D - 1);
    c.x = J.roi_x + pos;
    c.x0 = __builtin_amdgcn_readfirstlane(c.x);   // line 0's
    return c;
}

template <int D, bool FUSE, bool BIG, bool SPECIAL>
__device__ __forceinline__ void mid_vertical(const SgmJob& J, const MidColumns& col, int lane,
                                             uint64_t* lds, uint16_t* sums /* FUSE: [4][4][D] */) {
    constexpr int DPL = D / 16, NP = DPL / 2, NW = NP / 2;
    const int q = lane & 15, sub = lane >> 4;
    const int W = J.W, H = J.H, min_d = J.min_d, x = col.x;
    const bool right = J.is_right != 0;
    const auto own_r = rows_of(J, SPECIAL ? J.census_other : J.census);
    const auto oth_r = rows_of(J, SPECIAL ? J.census : J.census_other);
    constexpr int NR = kStageLoads<D>, KW = kStageWords<D>;
    // the first word this lane loads: its own partners in address order, or
    // its share of the group's
    const int g0 = right ? col.x0 + min_d : col.x0 - min_d - (D - 1);
    const int p0 = SPECIAL ? x - min_d - DPL * q - (DPL - 1) : g0 + 2 * lane;
    const uint32_t vown = (uint32_t)((x + J.cpad) * 8), voth = (uint32_t)((p0 + J.cpad) * 8);
    // where its partners sit in a staged step
    int at[SPECIAL ? 1 : DPL];
    if constexpr (!SPECIAL) {
#pragma unroll
        for (int j = 0; j < DPL; ++j)
            at[j] = lds_slot(x - col.x0 + (right ? DPL * q + j : D - 1 - (DPL * q + j)));
    }
    const int put = lds_slot(2 * lane);   // + 128 r: the swizzle has that period
    const uint32_t P1v = (uint32_t)J.p1 * 0x10001u, P2v = (uint32_t)J.p2 * 0x10001u;
    const uint32_t vvol = (uint32_t)(x * D + q * DPL), vrev = (uint32_t)(x * D + (15 - q) * DPL);
    const int y0 = FUSE ? H - 1 : 0;
    const int rowc = (FUSE ? -1 : 1) * J.cpitch * 8, rowv = (FUSE ? -1 : 1) * W * D;
    const auto ud_r = buf_at(J.path[kUD]);
    // the horizontal volumes in this lane's order and reversed
    const auto same_r = buf_at(right ? J.path[kRL] : J.path[kLR]);
    const auto rev_r = buf_at(right ? J.path[kLR] : J.path[kRL]);
    auto costs = [&](uint64_t own, const uint64_t (&p)[DPL], uint32_t base, uint32_t (&c)[NP])
        __attribute__((always_inline)) {
        lane_costs<NP>(own, base, [&](int j) { return p[SPECIAL ? DPL - 1 - j : j]; }, c);
    };

    // rings of PF steps: census words and, with FUSE, the other directions
    constexpr int PF = SPECIAL && D == 256 ? 2 : 4, BLK = 4;
    constexpr int NC = SPECIAL ? DPL : 2 * NR;
    uint64_t wo[PF], wp[PF][NC];
    uint32_t pr[FUSE ? PF : 1][3][NW];
    int sc = y0 * J.cpitch * 8, sv = y0 * W * D;   // offsets of the next step to load
    const int last_c = FUSE ? 0 : (H - 1) * J.cpitch * 8, last_v = FUSE ? 0 : (H - 1) * W * D;
    auto load_step_words = [&](uint64_t& o, uint64_t (&w)[NC]) __attribute__((always_inline)) {
        o = load_word(own_r, vown, sc);
        if constexpr (SPECIAL) {
            load_census<DPL>(oth_r, voth, sc, w);
        } else {
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                uint64_t t[2];
                load_census<2>(oth_r, voth + 1024 * r, sc, t);
                w[2 * r] = t[0]; w[2 * r + 1] = t[1];
            }
        }
    };
    auto load_volumes_at = [&](int p) __attribute__((always_inline)) {
        buf_load<NW>(ud_r, vvol, sv, pr[p][0]);
        buf_load<NW>(same_r, vvol, sv, pr[p][1]);
        buf_load<NW>(rev_r, vrev, sv, pr[p][2]);
    };
    auto next_row = [&]() __attribute__((always_inline)) {   // stays on the line's last row
        sc = FUSE ? max(sc + rowc, last_c) : min(sc + rowc, last_c);
        sv = FUSE ? max(sv + rowv, last_v) : min(sv + rowv, last_v);
    };
    uint64_t own = 0, w[DPL];   // the words of the step whose costs come next
    auto stage = [&](int slot, const uint64_t (&g)[NC]) __attribute__((always_inline)) {
        typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int r = 0; r < NR; ++r)
            *reinterpret_cast<u64x2*>(lds + slot * KW + 128 * r + put) = u64x2{g[2 * r], g[2 * r + 1]};
        __builtin_amdgcn_wave_barrier();
    };
    auto fetch = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < DPL; ++j) w[j] = lds[slot * KW + at[j]];
        __builtin_amdgcn_wave_barrier();
    };
    uint64_t o0, g0w[NC];
    load_step_words(o0, g0w);
    next_row();
    __builtin_amdgcn_sched_barrier(0);
    // the rings' slots in the loop's own order
#pragma unroll
    for (int p = 0; p < PF; ++p) {
        load_step_words(wo[p], wp[p]);
        if constexpr (FUSE) load_volumes_at(p);
        next_row();
        __builtin_amdgcn_sched_barrier(0);
    }
    Line<NP> s;
    {
        uint32_t c[NP];
        if constexpr (SPECIAL) {
            costs(o0, g0w, 0u, c);
        } else {
            stage(0, g0w);
            fetch(0);
            costs(o0, w, 0u, c);
            stage(1, wp[0]);
            own = wo[0];
            fetch(1);
        }
        line_init<BIG, 16>(s, c);
        if constexpr (!FUSE) {
            uint32_t o[NW];
            pack_lane(s, kSelFwd, o);
            buf_store<NW>(ud_r, vvol, y0 * W * D, o);
        } else {
            // row H - 1 is a border row of the WTA
            if (col.active && q == 0) gst(J.disp + (int64_t)y0 * W + x, kInvalidDisp);
        }
    }

    // WTA (FUSE): every lane of a line has each step's winner; lane q < 4 of a
    // line finishes step i0 + q of the 4-step block
    const float uthr = 1.0f - J.uniqueness;
    uint16_t* const sline = sums + sub * D;
    uint32_t wb[BLK], w1[BLK], w3[BLK];
    auto wta_step = [&](const uint32_t (&o3)[3][NW], int b) __attribute__((always_inline)) {
        constexpr int kLog = __builtin_ctz(DPL);
        static_assert(wta_key_max(DPL) < kF16Inf, "argmin keys S * DPL + j are finite f16 patterns");
        uint32_t S[NP], keys[NP];
#pragma unroll
        for (int k = 0; k < NP; ++k) {
            const int w = k >> 1, o = k & 1;
            S[k] = word_pair(o3[0][w], o) + word_pair(o3[1][w], o) + word_pair(o3[2][NW - 1 - w], o ^ 1) +
                   (s.L[k] & 0x00FF00FFu);   // each half <= 1020
            keys[k] = (S[k] << kLog) | (uint32_t)(2 * k) | ((uint32_t)(2 * k + 1) << 16);
        }
        const uint32_t key = pk_min_halves(pk_min_all<false>(keys)) & 0xFFFFu;
        uint32_t best = ((key / DPL) << 16) | (uint32_t)(DPL * q + key % DPL);
        best = line_min<16>(best);
        const int ds = (int)(best & 0xFFFFu);
        // the line's u16 sums side by side in LDS, a slot per step of the
        // block; the two beside the winner are used at the block's end.
        // Indices are clamped: S(-1) and S(D) are never used.
        uint32_t* const mine = reinterpret_cast<uint32_t*>(sline + b * 4 * D + DPL * q);
#pragma unroll
        for (int k = 0; k < NP; ++k) mine[k] = S[k];
        __builtin_amdgcn_wave_barrier();
        wb[b] = best;
        w1[b] = sline[b * 4 * D + max(ds - 1, 0)];
        w3[b] = sline[b * 4 * D + min(ds + 1, D - 1)];
        __builtin_amdgcn_wave_barrier();
    };
    auto wta_flush = [&](int i0) __attribute__((always_inline)) {
        const int i = i0 + q, y = y0 - i;
        auto pick = [&](const uint32_t (&v)[BLK]) {
            return q == 0 ? v[0] : q == 1 ? v[1] : q == 2 ? v[2] : v[3];
        };
        const uint32_t kb = pick(wb), k1 = pick(w1), k3 = pick(w3);
        const int ds = (int)(kb & 0xFFFFu);
        const uint32_t c2 = kb >> 16;
        constexpr bool warp_rule = (D == 64 || D == 128);
        const int rows_cov = warp_rule ? 2 * (H / 2) : H;
        float outv = kInvalidDisp;
        if (y < rows_cov && !(x > W - 5 || y > H - 5 || x < 5 || y < 5) && ds > 0 &&
            (warp_rule || ds < D - 1)) {
            const float c1 = (float)k1;
            const float c2f = (float)c2;
            const float c3 = (ds == D - 1) ? (float)(D - 1) : (float)k3;
            const float fa = c1 - c2f, fb = c3 - c2f;
            const float uniq = (fa < fb) ? fa : fb;
            if (!(uniq <= c2f * uthr)) {
                const float t = c1 + c3 - 2.0f * c2f;
                const float den = (1.0f < t) ? t : 1.0f;
                const float bias = (float)((double)(c1 - c3 + den) / (double)(2.0f * den));
                outv = (float)(ds + min_d) + bias;
            }
        }
        if (col.active && q < BLK && i < H) gst(J.disp + (int64_t)y * W + x, outv);
    };

    int st = (y0 + (FUSE ? -1 : 1)) * W * D;   // the store offset of step i (not FUSE)
    auto block = [&](int i0, auto full) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < BLK; ++b) {
            const int p = b % PF;
            uint32_t c[NP];
            if constexpr (SPECIAL) {
                costs(wo[p], wp[p], 0u - s.m, c);
            } else {
                // stage the next step, take this one's costs, read the next
                // one's words back beside the recurrence
                stage(b & 1, wp[(p + 1) % PF]);
                costs(own, w, 0u - s.m, c);
                own = wo[(p + 1) % PF];
                fetch(b & 1);
            }
            load_step_words(wo[p], wp[p]);
            line_step<BIG, 16>(s, c, P1v, P2v, false, false);
            if constexpr (!FUSE) {
                uint32_t o[NW];
                pack_lane(s, kSelFwd, o);
                if (full.value || i0 + b < H) buf_store<NW>(ud_r, vvol, st, o);
                st += rowv;
            } else {
                wta_step(pr[p], b);
                load_volumes_at(p);
            }
            next_row();
        }
        if constexpr (FUSE) wta_flush(i0);
    };
    int i0 = 1;
    for (; i0 + BLK <= H; i0 += BLK) block(i0, std::true_type{});
    if (i0 < H) block(i0, std::false_type{});
}

template <int D, bool FUSE, bool BIG, bool QUIRK>
__device__ __forceinline__ void mid_columns_run(const SgmJob& J, int group, int lane, uint64_t* lds,
                                                uint16_t* sums) {
    const MidColumns col = mid_columns(J, group, lane >> 4);
    if constexpr (QUIRK)
        if (col.special) return mid_vertical<D, FUSE, BIG, true>(J, col, lane, lds, sums);
    mid_vertical<D, FUSE, BIG, false>(J, col, lane, lds, sums);
}

// LDS of one wave (bytes): two staged steps, and the WTA's four steps of sums
template <int DMAX, bool FUSE>
constexpr int kMidLds = 16 * kStageWords<DMAX> + (FUSE ? 32 * DMAX : 0);

// Items of a job: left->right rows, right->left rows, then columns, those
// dealt so that each XCD has a contiguous run (neighbours share census words).
template <int DMAX, bool BIG, bool ONLY, bool QUIRK>
__global__ __launch_bounds__(256) void mid3_kernel(const SgmJob* __restrict__ jobs,
                                                   const int* __restrict__ offs, int njobs, int n) {
    extern __shared__ __align__(16) uint64_t mid_lds[];
    const int lane = threadIdx.x & 63, item = wave_item();
    if (item >= n) return;
    uint64_t* const lds = mid_lds + wave_in_group() * (kMidLds<DMAX, false> / 8);
    const int j = find_job(offs, njobs, item);
    const SgmJob& J = jobs[j];
    const int local = item - offs[j], nh = (J.H + 3) / 4;
    const bool horiz = local < 2 * nh;
    const int path = local < nh ? kLR : kRL, row = local < nh ? local : local - nh;
    const int col = horiz ? 0 : xcd_item(local - 2 * nh, offs[j + 1] - offs[j] - 2 * nh);
#define FSGM_MID_CASE(DD)                                                                   \
    case DD:                                                                                \
        if constexpr (ONLY ? DMAX == DD : DMAX >= DD) {                                     \
            if (horiz) mid_horizontal<DD, BIG, QUIRK>(J, path, row, lane);                  \
            else mid_columns_run<DD, false, BIG, QUIRK>(J, col, lane, lds, nullptr);        \
        }                                                                                   \
        break;
    switch (J.D) {
        FSGM_MID_CASE(64)
        FSGM_MID_CASE(128)
        FSGM_MID_CASE(256)
        default: break;
    }
#undef FSGM_MID_CASE
}

template <int DMAX, bool BIG, bool ONLY, bool QUIRK>
__global__ __launch_bounds__(256) void mid_wta_kernel(const SgmJob* __restrict__ jobs,
                                                      const int* __restrict__ offs, int njobs, int n) {
    extern __shared__ __align__(16) uint64_t mid_lds[];
    const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
    const int item = xcd_item(blockIdx.x, gridDim.x) * waves + wave_in_group();
    if (item >= n) return;
    uint64_t* const lds = mid_lds + wave_in_group() * (kMidLds<DMAX, true> / 8);
    uint16_t* const sums = reinterpret_cast<uint16_t*>(lds + 2 * kStageWords<DMAX>);
    const int j = find_job(offs, njobs, item);
    const SgmJob& J = jobs[j];
    const int group = item - offs[j];
    switch (J.D) {
        case 64: if constexpr (!ONLY || DMAX == 64) mid_columns_run<64, true, BIG, QUIRK>(J, group, lane, lds, sums); break;
        case 128: if constexpr (ONLY ? DMAX == 128 : DMAX >= 128) mid_columns_run<128, true, BIG, QUIRK>(J, group, lane, lds, sums); break;
        case 256: if constexpr (DMAX >= 256) mid_columns_run<256, true, BIG, QUIRK>(J, group, lane, lds, sums); break;
        default: break;
    }
}

}  // namespace

hipError_t launch_mid3(const StagePlan& p, hipStream_t s) {
    const int n = p.n_m3, wg = waves_per_group(n, 16);
    if (n <= 0) return hipSuccess;
    auto go = [&](auto ker, int lds) {
        hipLaunchKernelGGL(ker, dim3((n + wg - 1) / wg), dim3(64 * wg), wg * lds, s, p.jobs, p.offs_m3,
                           p.njobs, n);
    };
    constexpr int l64 = kMidLds<64, false>, l128 = kMidLds<128, false>, l256 = kMidLds<256, false>;
    if (p.big) go(mid3_kernel<256, true, false, true>, l256);
    else if (p.dmin != p.dmax) go(mid3_kernel<256, false, false, true>, l256);
    else if (p.dmax == 64) p.quirk ? go(mid3_kernel<64, false, true, true>, l64) : go(mid3_kernel<64, false, true, false>, l64);
    else if (p.dmax == 128) p.quirk ? go(mid3_kernel<128, false, true, true>, l128) : go(mid3_kernel<128, false, true, false>, l128);
    else p.quirk ? go(mid3_kernel<256, false, true, true>, l256) : go(mid3_kernel<256, false, true, false>, l256);
    return hipGetLastError();
}

hipError_t launch_mid_wta(const StagePlan& p, hipStream_t s) {
    const int n = p.n_mf, wg = waves_per_group(n, 4);
    if (n <= 0) return hipSuccess;
    auto go = [&](auto ker, int lds) {
        hipLaunchKernelGGL(ker, dim3((n + wg - 1) / wg), dim3(64 * wg), wg * lds, s, p.jobs, p.offs_mf,
                           p.njobs, n);
    };
    constexpr int l64 = kMidLds<64, true>, l128 = kMidLds<128, true>, l256 = kMidLds<256, true>;
    if (p.big) go(mid_wta_kernel<256, true, false, true>, l256);
    else if (p.dmin != p.dmax) go(mid_wta_kernel<256, false, false, true>, l256);
    else if (p.dmax == 64) p.quirk ? go(mid_wta_kernel<64, false, true, true>, l64) : go(mid_wta_kernel<64, false, true, false>, l64);
    else if (p.dmax == 128) p.quirk ? go(mid_wta_kernel<128, false, true, true>, l128) : go(mid_wta_kernel<128, false, true, false>, l128);
    else p.quirk ? go(mid_wta_kernel<256, false, true, true>, l256) : go(mid_wta_kernel<256, false, true, false>, l256);
    return hipGetLastError();
}

}  // namespace fsgm
