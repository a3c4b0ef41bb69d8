// Differentiable FP32 SGM for CDNA4 (gfx950): forward, soft-argmin and a
// hand-written backward.
//
// Definition (per image b of a batch; cost C[B][H][W][D], per-pixel penalty
// maps P1[B][H][W], P2[B][H][W], temperature T):
//   per direction r (0 top->bottom, 1 left->right, 2 bottom->top,
//   3 right->left) over the whole image
//     L(p0, d) = C(p0, d)
//     L(p, d)  = C(p, d) + min(L'(d), min(L'(d-1), L'(d+1)) + P1(p), m' + P2(p)) - m'
//     L'(-1) = L'(D) = +inf,  m' = min_d L'(d)
//   S = ((L_1 + L_3) + L_0) + L_2
//   disp(p) = sum_d d * softmax_d(-S(p, d) / T)
// Subgradients: the first min candidate in the order [L'(d), L'(d-1)+P1,
// L'(d+1)+P1, m'+P2] wins; m' = L'(k*) with k* the smallest argmin.
//
// Memory: S is built in place and no per-direction volume is kept.  The
// forward's first launch runs, per pair of rows, left->right and right->left
// at the same time in one wave: each pixel is reached by one direction in the
// first half of the walk, which stores its L, and by the other in the second
// half, which adds onto it (two-term sums commute, so S = L_1 + L_3 whichever
// came first).  Beside them the top->bottom groups write L_0 into the one
// workspace volume.  The second launch runs bottom->top, forms
// S = (S + L_0) + L_2 and the soft-argmin, and keeps the minimum of S
// and the softmax normaliser per pixel.  Every direction also saves, per
// step, the winner code of each disparity (2 bits) and k* of the previous
// step's L (one byte per pixel): 1 byte per cell over the four directions,
// a quarter of a volume, which is all the reverse recurrence needs of the
// forward.  The backward walks each scanline from its last step to its
// first, once:
//   G(s-1, d) = gS(s-1, d) + G(s, d)[w(s,d)=0] + G(s, d+1)[w(s,d+1)=1]
//             + G(s, d-1)[w(s,d-1)=2] - [d = k*(s-1)] sum_e G(s,e)[w(s,e)!=3]
// with gS = dLoss/dS formed from S, the kept minimum and normaliser, and
// emits dC_r(s, d) = G(s, d), dP1_r(s) = sum_d G(s,d)[w in {1,2}],
// dP2_r(s) = sum_d G(s,d)[w = 3].  Its launches mirror the forward's: dC,
// dP1 and dP2 are built in place by the horizontal pairs, the top->bottom
// terms go to the workspace, and bottom->top adds both in the same order as S.
//
// Layout per wave: four 16-lane DPP rows, one scanline per row (two rows in
// both directions, or four columns), D/16 disparities per lane.  Lanes past
// the image repeat its last line: same values, same addresses.
//
// Little work (pairs_ok) runs as one launch of all four directions, columns too
// as pairs walked from both ends into the workspace volume, and a pass that
// joins the sums: S = (L_1 + L_3) + (L_0 + L_2), and the gradients likewise.
//
// What bounds these passes: for one image or a few, the chain of a scanline's
// steps, max(H, W) + H forward and again backward, each 130-300 instructions
// of a wave that has its SIMD to itself; for many, the copy rate (93 bytes per
// cell).  Walking a row's directions one after the other made the chain
// 2 W + H: forward + backward of one image 1242x375 D = 128 3.24 -> 1.54 ms, D =
// 256 6.04 -> 3.27 ms, 4 images D = 64 3.13 -> 2.37 ms, 2 images 321x119 D = 64
// 0.57 -> 0.27 and, in one launch, 0.20 ms.
#include <algorithm>
#include <type_traits>

#include "dsgm_device.h"
#include "sgm_device.h"

#pragma clang fp contract(off)

namespace fsgm {
using namespace dsgm;
namespace {

// Steps of loads in flight: a wave that is alone on its SIMD would otherwise
// wait the memory latency at every step.  The inputs of step s + kAhead are
// issued right after step s has used its slot; steps past the end load the
// last pixel again and are not used.
// (Fewer at D = 256, where four would pass the 256 vector registers.)
template <int D, bool LAST> constexpr int kAhead = D < 256 ? 4 : LAST ? 2 : 3;

// Byte offsets from a wave-uniform base: 32 bits, which an access takes beside
// a scalar base, unless two rows of the image or two directions' codes pass
// 2^31 bytes (64-bit address arithmetic took a sixth of a D = 64 step).
template <bool WIDE> using Off = std::conditional_t<WIDE, int64_t, uint32_t>;

template <class T, class O>
__device__ __forceinline__ T* at(T* base, O bytes) {
    return (T*)((std::conditional_t<std::is_const_v<T>, const char, char>*)base + bytes);
}
// Winner codes are loaded as the dword that holds the lane's: the masking of a
// 1- or 2-byte load would wait at the top of the loop for the whole ring.
// (The codes of a pixel are D / 4 bytes, and the buffer starts on 8.)
template <int D> constexpr int kCodeBytes = D / 4;
template <int D> __device__ __forceinline__ uint32_t code_byte(int l) { return (uint32_t)l * (D / 64); }
__device__ __forceinline__ uint32_t load_codes(const uint8_t* p) {
    return *(const __attribute__((address_space(1))) uint32_t*)p;
}
template <int D>
__device__ __forceinline__ uint32_t shift_codes(uint32_t w, int l) { return w >> (8 * (code_byte<D>(l) & 3)); }
template <int D>
__device__ __forceinline__ void store_codes(uint8_t* p, uint32_t w) {
    *(__attribute__((address_space(1))) WinWord<D>*)p = (WinWord<D>)w;
}
__device__ __forceinline__ void storeb(uint8_t* p, int v) { *(__attribute__((address_space(1))) uint8_t*)p = (uint8_t)v; }
__device__ __forceinline__ int loadb(const uint8_t* p) { return *(const __attribute__((address_space(1))) uint8_t*)p; }
__device__ __forceinline__ void store1(float* p, float v) { *(g_f*)p = v; }

// Two scanlines of an image, walked from both ends at once: lanes 0-31 in the
// first direction (left->right, or top->bottom of columns), lanes 32-63 in the
// second (in the backward, each reversed).  At step t every lane is t pixels
// into its direction's walk.
template <bool VERT, bool WIDE>
struct LinePair {
    int n, n1, n2;             // steps; those that reach a pixel first; first step that reaches one second
    bool second;               // this lane walks the second direction
    Off<WIDE> pix0, step;      // pixel of step 0 from q0, and its move
    int64_t q0;                // the pair's first pixel in the batch
    __device__ LinePair(const DsgmArgs& A, int b, int g, int lane, bool reversed) {
        n = VERT ? A.H : A.W;
        n1 = n / 2;
        n2 = (n + 1) / 2;
        const int sub = lane >> 4, lines = VERT ? A.W : A.H;
        second = sub >= 2;
        const bool from_end = second != reversed;
        const int line = min(2 * g + (sub & 1), lines - 1) - 2 * g;
        const Off<WIDE> along = VERT ? (Off<WIDE>)A.W : 1, across = VERT ? 1 : (Off<WIDE>)A.W;
        pix0 = (Off<WIDE>)line * across + (Off<WIDE>)(from_end ? n - 1 : 0) * along;
        step = from_end ? 0 - along : along;
        q0 = (int64_t)b * A.H * A.W + (int64_t)2 * g * (VERT ? 1 : A.W);
    }
    __device__ Off<WIDE> pix(int t) const { return pix0 + step * (Off<WIDE>)t; }
    // a walk's next pixel, staying on the last one (t: the step moved to)
    __device__ Off<WIDE> move(Off<WIDE> p, int t) const { return t < n ? p + step : p; }
};
// the other direction's value of the same line
__device__ __forceinline__ float other_half(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __builtin_bit_cast(int, v)));
}

// Runs n steps with NA of them loaded ahead: whole blocks, then the remainder.
// (An exit from the middle of a block would join the loop's head, whose wait
// counts would then cover the shortest path: every block would wait for loads
// just issued.)
template <int NA, class Issue, class Step>
__device__ __forceinline__ void run_steps(int n, Issue issue, Step step) {
#pragma unroll
    for (int u = 0; u < NA; ++u) issue(u);
    int blocks = n / NA;
    const int rest = n - blocks * NA;
    if (blocks > 0) {
        do {
#pragma unroll
            for (int u = 0; u < NA; ++u) {
                step(u);
                issue(u);
            }
        } while (--blocks > 0);
    }
#pragma unroll
    for (int u = 0; u < NA - 1; ++u)
        if (u < rest) step(u);
}

// Three phases of a pair of walks: pixels reached first (STORE), a middle
// pixel reached by both at once when W is odd (both halves hold the sum), and
// pixels reached second (ADD).
enum PairPhase { kPairStore = 0, kPairMiddle = 1, kPairAdd = 2 };

// ------------------------------------------------------------- forward ---
template <int D, bool VERT, bool WIDE>
__device__ __forceinline__ void fwd_pair(const DsgmArgs& A, int b, int g, int lane) {
    constexpr int DPD = D / 16, NA = kAhead<D, false>;
    const float inf = __builtin_inff();
    const int l = lane & 15;
    const LinePair<VERT, WIDE> rp(A, b, g, lane, false);
    const int64_t npix = (int64_t)A.B * A.H * A.W;
    const float* cost = A.cost + rp.q0 * D;
    float* S = (VERT ? A.vol : A.S) + rp.q0 * D;   // where the pair's sum is built
    const float *p1 = A.p1 + rp.q0, *p2 = A.p2 + rp.q0;
    constexpr int P = VERT ? 0 : 1;                // the first direction; the second is two planes on
    uint8_t* wout = A.wins + (P * npix + rp.q0) * kCodeBytes<D>;
    uint8_t* kout = A.kstar + P * npix + rp.q0;
    const Off<WIDE> plane = rp.second ? (Off<WIDE>)(2 * npix) : 0;
    const Off<WIDE> lane_c = (Off<WIDE>)(l * DPD * 4), lane_w = plane * kCodeBytes<D> + code_byte<D>(l);

    float qc[NA][DPD], qp1[NA], qp2[NA], qs[NA][DPD];
    float L[DPD];
#pragma unroll
    for (int k = 0; k < DPD; ++k) L[k] = 0.f;   // with infinite penalties: L = C at the first step

    auto walk = [&](auto phase, int t0, int t1) __attribute__((always_inline)) {
        constexpr int PHASE = decltype(phase)::value;
        if (t0 >= t1) return;
        Off<WIDE> pi = rp.pix(t0), ps = pi;      // pixels of the next issue and of the step
        int ti = t0;
        auto issue = [&](int u) __attribute__((always_inline)) {
            loadf<DPD>(at(cost, pi * (D * 4) + lane_c), qc[u]);
            if constexpr (PHASE == kPairAdd) loadf<DPD>(at(S, pi * (D * 4) + lane_c), qs[u]);
            qp1[u] = loads(at(p1, pi * 4));
            qp2[u] = loads(at(p2, pi * 4));
            pi = rp.move(pi, ++ti);
            __builtin_amdgcn_sched_barrier(0);
        };
        int t = t0;
        auto step = [&](int u) __attribute__((always_inline)) {
            const float m = row_min(lane_min(L));
            const int ks = row_mini(lane_argmin<DPD>(L, m, l));
            const bool start = PHASE != kPairAdd && t == 0;
            const uint32_t w = fwd_step<DPD>(L, qc[u], m, start ? inf : qp1[u], start ? inf : qp2[u]);
            float sv[DPD];
#pragma unroll
            for (int k = 0; k < DPD; ++k) {
                sv[k] = L[k];
                if constexpr (PHASE == kPairAdd) sv[k] = qs[u][k] + L[k];
                if constexpr (PHASE == kPairMiddle) sv[k] = L[k] + other_half(L[k], lane);
            }
            storef<DPD>(at(S, ps * (D * 4) + lane_c), sv);
            store_codes<D>(at(wout, ps * kCodeBytes<D> + lane_w), w);
            storeb(at(kout, ps + plane), ks);           // sixteen lanes, one value
            ps += rp.step;
            ++t;
        };
        if constexpr (PHASE == kPairMiddle) {    // one step at most
            issue(0);
            step(0);
        } else {
            run_steps<NA>(t1 - t0, issue, step);
        }
    };
    walk(std::integral_constant<int, kPairStore>{}, 0, rp.n1);
    walk(std::integral_constant<int, kPairMiddle>{}, rp.n1, rp.n2);
    // the other lanes' stores of the pixels that this phase loads
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    walk(std::integral_constant<int, kPairAdd>{}, rp.n2, rp.n);
}

// Four columns, top->bottom into the workspace volume or (LAST) bottom->top
// with the sum and the soft-argmin.
template <int D, bool LAST, bool WIDE>
__device__ __forceinline__ void fwd_cols(const DsgmArgs& A, int b, int group, int lane) {
    constexpr int DPD = D / 16, NA = kAhead<D, LAST>;
    const float inf = __builtin_inff();
    const int l = lane & 15, W = A.W, H = A.H;
    const Off<WIDE> col = (Off<WIDE>)min(group * 4 + (lane >> 4), W - 1);
    const int64_t npix = (int64_t)A.B * H * W, img = (int64_t)b * H * W, path = LAST ? 2 : 0;
    const Off<WIDE> col_c = col * (D * 4) + (Off<WIDE>)(l * DPD * 4), col_w = col * kCodeBytes<D> + code_byte<D>(l);

    float qc[NA][DPD], qs[NA][DPD], qy[NA][DPD], qp1[NA], qp2[NA];
    int si = 0;
    auto issue = [&](int u) __attribute__((always_inline)) {
        const int s = min(si++, H - 1);
        const int64_t r0 = img + (int64_t)(LAST ? H - 1 - s : s) * W;
        loadf<DPD>(at(A.cost + r0 * D, col_c), qc[u]);
        qp1[u] = loads(at(A.p1 + r0, col * 4));
        qp2[u] = loads(at(A.p2 + r0, col * 4));
        if constexpr (LAST) {
            loadf<DPD>(at(A.S + r0 * D, col_c), qs[u]);
            loadf<DPD>(at(A.vol + r0 * D, col_c), qy[u]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    float L[DPD];
#pragma unroll
    for (int k = 0; k < DPD; ++k) L[k] = 0.f;
    int s = 0;
    auto step = [&](int u) __attribute__((always_inline)) {
        const int64_t r0 = img + (int64_t)(LAST ? H - 1 - s : s) * W;
        const float m = row_min(lane_min(L));
        const int ks = row_mini(lane_argmin<DPD>(L, m, l));
        const uint32_t w = fwd_step<DPD>(L, qc[u], m, s == 0 ? inf : qp1[u], s == 0 ? inf : qp2[u]);
        store_codes<D>(at(A.wins + (path * npix + r0) * kCodeBytes<D>, col_w), w);
        storeb(at(A.kstar + path * npix + r0, col), ks);
        if constexpr (LAST) {
            float sv[DPD], mn, z;
#pragma unroll
            for (int k = 0; k < DPD; ++k) sv[k] = (qs[u][k] + qy[u][k]) + L[k];
            storef<DPD>(at(A.S + r0 * D, col_c), sv);
            const float d = soft_argmin<DPD>(sv, l, A.inv_temperature, &mn, &z);
            store1(at(A.disp + r0, col * 4), d);
            store1(at(A.stats + 2 * r0, col * 8), mn);
            store1(at(A.stats + 2 * r0, col * 8 + 4), z);
        } else {
            storef<DPD>(at(A.vol + r0 * D, col_c), L);
        }
        ++s;
    };
    run_steps<NA>(H, issue, step);
}

// ------------------------------------------------------------ backward ---
template <int D, bool VERT, bool WIDE>
__device__ __forceinline__ void bwd_pair(const DsgmArgs& A, int b, int g, int lane) {
    constexpr int DPD = D / 16, NA = kAhead<D, false>;
    const int l = lane & 15;
    const LinePair<VERT, WIDE> rp(A, b, g, lane, true);
    const int64_t npix = (int64_t)A.B * A.H * A.W;
    const float *S = A.S + rp.q0 * D, *stats = A.stats + 2 * rp.q0;
    const float *disp = A.disp + rp.q0, *gdisp = A.grad_disp + rp.q0;
    float* dc = (VERT ? A.vol : A.grad_cost) + rp.q0 * D;
    float *dp1 = (VERT ? A.vol_p1 : A.grad_p1) + rp.q0, *dp2 = (VERT ? A.vol_p2 : A.grad_p2) + rp.q0;
    constexpr int P = VERT ? 0 : 1;                // the first direction; the second is two planes on
    const uint8_t* win = A.wins + (P * npix + rp.q0) * kCodeBytes<D>;
    const uint8_t* kin = A.kstar + P * npix + rp.q0;
    const Off<WIDE> plane = rp.second ? (Off<WIDE>)(2 * npix) : 0;
    const Off<WIDE> lane_c = (Off<WIDE>)(l * DPD * 4), lane_w = plane * kCodeBytes<D> + (code_byte<D>(l) & ~3u);

    float qs[NA][DPD], qmn[NA], qz[NA], qg[NA], qd[NA], qo[NA][DPD], qo1[NA], qo2[NA];
    uint32_t qw[NA];
    int qk[NA];
    float F[DPD];                              // what the pixel after this one hands to it
#pragma unroll
    for (int k = 0; k < DPD; ++k) F[k] = 0.f;

    auto walk = [&](auto phase, int t0, int t1) __attribute__((always_inline)) {
        constexpr int PHASE = decltype(phase)::value;
        if (t0 >= t1) return;
        Off<WIDE> pi = rp.pix(t0), ps = pi;
        int ti = t0;
        auto issue = [&](int u) __attribute__((always_inline)) {
            loadf<DPD>(at(S, pi * (D * 4) + lane_c), qs[u]);
            qmn[u] = loads(at(stats, pi * 8));
            qz[u] = loads(at(stats, pi * 8 + 4));
            qg[u] = loads(at(gdisp, pi * 4));
            qd[u] = loads(at(disp, pi * 4));
            qw[u] = load_codes(at(win, pi * kCodeBytes<D> + lane_w));
            qk[u] = loadb(at(kin, pi + plane));
            if constexpr (PHASE == kPairAdd) {
                loadf<DPD>(at(dc, pi * (D * 4) + lane_c), qo[u]);
                qo1[u] = loads(at(dp1, pi * 4));
                qo2[u] = loads(at(dp2, pi * 4));
            }
            pi = rp.move(pi, ++ti);
            __builtin_amdgcn_sched_barrier(0);
        };
        int t = t0;
        auto step = [&](int u) __attribute__((always_inline)) {
            float G[DPD], v[DPD], s12, s3;
            grad_s_from<DPD>(qs[u], qmn[u], qz[u], qg[u], qd[u], A.inv_temperature, l, G);
#pragma unroll
            for (int k = 0; k < DPD; ++k) G[k] += F[k];
            // the direction's first pixel (the walk's last) hands on
            // nothing and has no penalty gradient: code 0 everywhere
            const uint32_t w = t == rp.n - 1 ? 0u : shift_codes<D>(qw[u], l);
            float sums[3];
            sums[0] = bwd_flow<DPD>(G, w, F, &s12, &s3);
            sums[1] = s12;
            sums[2] = s3;
            row_sums(sums);
            bwd_jump<DPD>(F, qk[u], sums[0], l);
#pragma unroll
            for (int k = 0; k < DPD; ++k) {
                v[k] = G[k];
                if constexpr (PHASE == kPairAdd) v[k] = qo[u][k] + G[k];
                if constexpr (PHASE == kPairMiddle) v[k] = G[k] + other_half(G[k], lane);
            }
            if constexpr (PHASE == kPairAdd) {
                sums[1] = qo1[u] + sums[1];
                sums[2] = qo2[u] + sums[2];
            }
            if constexpr (PHASE == kPairMiddle) {
                sums[1] += other_half(sums[1], lane);
                sums[2] += other_half(sums[2], lane);
            }
            storef<DPD>(at(dc, ps * (D * 4) + lane_c), v);
            store1(at(dp1, ps * 4), sums[1]);
            store1(at(dp2, ps * 4), sums[2]);
            ps += rp.step;
            ++t;
        };
        if constexpr (PHASE == kPairMiddle) {    // one step at most
            issue(0);
            step(0);
        } else {
            run_steps<NA>(t1 - t0, issue, step);
        }
    };
    walk(std::integral_constant<int, kPairStore>{}, 0, rp.n1);
    walk(std::integral_constant<int, kPairMiddle>{}, rp.n1, rp.n2);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    walk(std::integral_constant<int, kPairAdd>{}, rp.n2, rp.n);
}

// Four columns: top->bottom reversed into the workspace, or (LAST)
// bottom->top reversed, adding both onto the rows' gradients.
template <int D, bool LAST, bool WIDE>
__device__ __forceinline__ void bwd_cols(const DsgmArgs& A, int b, int group, int lane) {
    constexpr int DPD = D / 16, NA = kAhead<D, LAST>;
    const int l = lane & 15, W = A.W, H = A.H;
    const Off<WIDE> col = (Off<WIDE>)min(group * 4 + (lane >> 4), W - 1);
    const int64_t npix = (int64_t)A.B * H * W, img = (int64_t)b * H * W, path = LAST ? 2 : 0;
    const Off<WIDE> col_c = col * (D * 4) + (Off<WIDE>)(l * DPD * 4), col_w = col * kCodeBytes<D> + (code_byte<D>(l) & ~3u);

    float qs[NA][DPD], qmn[NA], qz[NA], qg[NA], qd[NA], qo[NA][DPD], qo1[NA], qo2[NA], qy[NA][DPD], qy1[NA], qy2[NA];
    uint32_t qw[NA];
    int qk[NA];
    int si = 0;
    auto issue = [&](int u) __attribute__((always_inline)) {
        const int s = min(si++, H - 1);
        const int64_t r0 = img + (int64_t)(LAST ? s : H - 1 - s) * W;
        loadf<DPD>(at(A.S + r0 * D, col_c), qs[u]);
        qmn[u] = loads(at(A.stats + 2 * r0, col * 8));
        qz[u] = loads(at(A.stats + 2 * r0, col * 8 + 4));
        qg[u] = loads(at(A.grad_disp + r0, col * 4));
        qd[u] = loads(at(A.disp + r0, col * 4));
        qw[u] = load_codes(at(A.wins + (path * npix + r0) * kCodeBytes<D>, col_w));
        qk[u] = loadb(at(A.kstar + path * npix + r0, col));
        if constexpr (LAST) {
            loadf<DPD>(at(A.grad_cost + r0 * D, col_c), qo[u]);
            loadf<DPD>(at(A.vol + r0 * D, col_c), qy[u]);
            qo1[u] = loads(at(A.grad_p1 + r0, col * 4));
            qo2[u] = loads(at(A.grad_p2 + r0, col * 4));
            qy1[u] = loads(at(A.vol_p1 + r0, col * 4));
            qy2[u] = loads(at(A.vol_p2 + r0, col * 4));
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    float F[DPD];
#pragma unroll
    for (int k = 0; k < DPD; ++k) F[k] = 0.f;
    int s = 0;
    auto step = [&](int u) __attribute__((always_inline)) {
        const int64_t r0 = img + (int64_t)(LAST ? s : H - 1 - s) * W;
        float G[DPD], s12, s3, sums[3];
        grad_s_from<DPD>(qs[u], qmn[u], qz[u], qg[u], qd[u], A.inv_temperature, l, G);
#pragma unroll
        for (int k = 0; k < DPD; ++k) G[k] += F[k];
        sums[0] = bwd_flow<DPD>(G, s == H - 1 ? 0u : shift_codes<D>(qw[u], l), F, &s12, &s3);
        sums[1] = s12;
        sums[2] = s3;
        row_sums(sums);
        bwd_jump<DPD>(F, qk[u], sums[0], l);
        if constexpr (LAST) {
#pragma unroll
            for (int k = 0; k < DPD; ++k) G[k] = (qo[u][k] + qy[u][k]) + G[k];
            storef<DPD>(at(A.grad_cost + r0 * D, col_c), G);
            store1(at(A.grad_p1 + r0, col * 4), (qo1[u] + qy1[u]) + sums[1]);
            store1(at(A.grad_p2 + r0, col * 4), (qo2[u] + qy2[u]) + sums[2]);
        } else {
            storef<DPD>(at(A.vol + r0 * D, col_c), G);
            store1(at(A.vol_p1 + r0, col * 4), sums[1]);
            store1(at(A.vol_p2 + r0, col * 4), sums[2]);
        }
        ++s;
    };
    run_steps<NA>(H, issue, step);
}

// The first launch: the row pairs of every image, then the top->bottom column
// groups; the second: the bottom->top groups.  Column groups are spread so
// that each XCD walks a contiguous run of them: the per-pixel maps (penalties,
// statistics, disparity, gradients) of 32 neighbouring columns share a
// 128-byte line, which is then fetched into one L2 instead of eight.  A
// workgroup is one wave: of few groups, four to a workgroup leave most CUs
// idle, and the walks wait for the memory path of the rest (1242x375, forward
// + backward, four / one: D = 128 2.56 / 1.58 ms, D = 256 6.23 / 3.28 ms;
// 4 images D = 128 5.33 / 4.76 ms).

template <int D, bool BWD, bool WIDE>
__global__ __launch_bounds__(64) void dsgm_first_kernel(DsgmArgs A, int row_blocks) {
    const int lane = threadIdx.x;
    if ((int)blockIdx.x < row_blocks) {
        const int nh = (A.H + 1) / 2, item = blockIdx.x;
        const int b = item / nh;
        if constexpr (BWD) bwd_pair<D, false, WIDE>(A, b, item - b * nh, lane);
        else fwd_pair<D, false, WIDE>(A, b, item - b * nh, lane);
    } else {
        const int nv = (A.W + 3) / 4;
        const int item = dev::xcd_item((int)blockIdx.x - row_blocks, (int)gridDim.x - row_blocks);
        const int b = item / nv;
        if constexpr (BWD) bwd_cols<D, false, WIDE>(A, b, item - b * nv, lane);
        else fwd_cols<D, false, WIDE>(A, b, item - b * nv, lane);
    }
}

template <int D, bool BWD, bool WIDE>
__global__ __launch_bounds__(64) void dsgm_last_kernel(DsgmArgs A) {
    const int nv = (A.W + 3) / 4;
    const int item = dev::xcd_item(blockIdx.x, gridDim.x);
    const int b = item / nv;
    if constexpr (BWD) bwd_cols<D, true, WIDE>(A, b, item - b * nv, threadIdx.x);
    else fwd_cols<D, true, WIDE>(A, b, item - b * nv, threadIdx.x);
}

// The form for little work: all four directions in one launch, rows and columns
// both as pairs walked from both ends, then one pass that joins the two sums,
// S = (L_1 + L_3) + (L_0 + L_2) (and dC, dP1, dP2 likewise).
template <int D, bool BWD>
__global__ __launch_bounds__(64) void dsgm_pairs_kernel(DsgmArgs A, int row_blocks) {
    const int lane = threadIdx.x;
    if ((int)blockIdx.x < row_blocks) {
        const int nh = (A.H + 1) / 2, item = blockIdx.x, b = item / nh;
        if constexpr (BWD) bwd_pair<D, false, false>(A, b, item - b * nh, lane);
        else fwd_pair<D, false, false>(A, b, item - b * nh, lane);
    } else {
        const int nv = (A.W + 1) / 2;
        const int item = dev::xcd_item((int)blockIdx.x - row_blocks, (int)gridDim.x - row_blocks), b = item / nv;
        if constexpr (BWD) bwd_pair<D, true, false>(A, b, item - b * nv, lane);
        else fwd_pair<D, true, false>(A, b, item - b * nv, lane);
    }
}
template <int D, bool BWD>
__global__ __launch_bounds__(256) void dsgm_join_kernel(DsgmArgs A, int64_t npix) {
    constexpr int DPD = D / 16;
    const int l = threadIdx.x & 15;
    const int64_t q = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    if (q >= npix) return;                       // whole 16-lane rows
    float* out = (BWD ? A.grad_cost : A.S) + q * D + l * DPD;
    float x[DPD], y[DPD];
    loadf<DPD>(out, x);
    loadf<DPD>(A.vol + q * D + l * DPD, y);
#pragma unroll
    for (int k = 0; k < DPD; ++k) x[k] += y[k];
    storef<DPD>(out, x);
    if constexpr (BWD) {
        if (l == 0) {
            A.grad_p1[q] += A.vol_p1[q];
            A.grad_p2[q] += A.vol_p2[q];
        }
    } else {
        float mn, z;
        const float d = soft_argmin<DPD>(x, l, A.inv_temperature, &mn, &z);
        if (l == 0) {
            A.disp[q] = d;
            A.stats[2 * q] = mn;
            A.stats[2 * q + 1] = z;
        }
    }
}

template <int D, bool BWD>
hipError_t launch_pairs(const DsgmArgs& A, hipStream_t s) {
    const unsigned rows = (unsigned)A.B * ((A.H + 1) / 2), cols = (unsigned)A.B * ((A.W + 1) / 2);
    const int64_t npix = (int64_t)A.B * A.H * A.W;
    hipLaunchKernelGGL((dsgm_pairs_kernel<D, BWD>), dim3(rows + cols), dim3(64), 0, s, A, (int)rows);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((dsgm_join_kernel<D, BWD>), dim3((unsigned)((npix + 15) / 16)), dim3(256), 0, s, A, npix);
    return hipGetLastError();
}

template <int D, bool BWD, bool WIDE>
hipError_t launch_passes(const DsgmArgs& A, hipStream_t s) {
    const unsigned rows = (unsigned)A.B * ((A.H + 1) / 2);
    const unsigned cols = (unsigned)A.B * ((A.W + 3) / 4);
    hipLaunchKernelGGL((dsgm_first_kernel<D, BWD, WIDE>), dim3(rows + cols), dim3(64), 0, s, A, (int)rows);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((dsgm_last_kernel<D, BWD, WIDE>), dim3(cols), dim3(64), 0, s, A);
    return hipGetLastError();
}

// Where all four directions in one launch are sooner done: the chain is
// max(H, W) steps and a pass over the volumes instead of max(H, W) + H steps, but
// it moves 12 more bytes per cell each way, and past about one wave per SIMD the
// waves share the SIMDs anyway.  Forward + backward, us, separate -> pairs:
//   D = 64: 2 images 321x119 (440 waves) 274 -> 198, 2 640x200 (840) 512 -> 412,
//   4 321x119 (880) 280 -> 222, 1 1242x375 (808, 30M cells) 1010 -> 908, 8 321x119
//   (1760) 320 -> 360
//   D = 128: 1 100x300 (200) 626 -> 269, 3 280x134 (621) 406 -> 302, 4 300x100
//   (800) 387 -> 337, 2 800x100 (900) 797 -> 777, 3 500x200 (1050) 827 -> 938, 1
//   1242x375 (808, 60M cells) 1544 -> 1674
//   D = 256: 1 300x200 (250) 845 -> 509, 2 280x134 (414) 693 -> 509, 3 280x134
//   (621) 773 -> 819
// Below the limit offsets fit 32 bits.
bool pairs_ok(const DsgmArgs& A) {
    const int64_t waves = (int64_t)A.B * ((A.H + 1) / 2 + (A.W + 1) / 2), cells = (int64_t)A.B * A.H * A.W * A.D;
    return waves <= (A.D == 256 ? 500 : 950) && cells <= 30000000;
}

template <bool BWD>
hipError_t launch_by_d(const DsgmArgs& A, hipStream_t s) {
    const int64_t rows = (int64_t)2 * A.W * A.D * 4, codes = ((int64_t)2 * A.B * A.H + 2) * A.W * (A.D / 4);
    const bool wide = std::max(rows, codes) > (int64_t)1 << 31;
    if (pairs_ok(A)) {
        switch (A.D) {
            case 64: return launch_pairs<64, BWD>(A, s);
            case 128: return launch_pairs<128, BWD>(A, s);
            case 256: return launch_pairs<256, BWD>(A, s);
            default: return hipErrorInvalidValue;
        }
    }
    switch (A.D) {
        case 64: return wide ? launch_passes<64, BWD, true>(A, s) : launch_passes<64, BWD, false>(A, s);
        case 128: return wide ? launch_passes<128, BWD, true>(A, s) : launch_passes<128, BWD, false>(A, s);
        case 256: return wide ? launch_passes<256, BWD, true>(A, s) : launch_passes<256, BWD, false>(A, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t dsgm_launch_forward(const DsgmArgs& A, hipStream_t s) {
    return dsgm_sweep_ok(A) ? dsgm_sweep_forward(A, s) : launch_by_d<false>(A, s);
}
hipError_t dsgm_launch_backward(const DsgmArgs& A, hipStream_t s) {
    return dsgm_sweep_ok(A) ? dsgm_sweep_backward(A, s) : launch_by_d<true>(A, s);
}

}  // namespace fsgm
