// Differentiable FP32 SGM, the form for large batches (gfx950): sweeps that
// run a horizontal and a vertical direction of a pixel together.
//
// The separate passes of dsgm_kernels.hip move 93 bytes per cell: every
// direction reads the cost (or S) again and adds onto a volume.  Here one
// wave walks a band of four rows and carries both a horizontal and a vertical
// recurrence, so a pixel's cost is read once for two directions and their sum
// leaves in one store.  Row r of the band runs r steps behind row 0: the
// vertical state of a column passes from row to row through LDS, one step
// after the row above has written it.  A band's first row takes the vertical
// state of the row before it from memory: the edge pass, beforehand, walks
// the columns alone and keeps that state at every fourth row (a quarter of a
// volume per direction).
//
//   forward   edges of top->bottom                  C in, 1/4 out
//             sweep left->right + top->bottom,
//             beside it the edges of bottom->top      C, 1/4 in, S out; C in, 1/4 out
//             sweep right->left + bottom->top         C, S, 1/4 in, S out
//   backward  the same of the reversed directions     S and the codes in place of C, dC of S
//
// About 66 bytes per cell in all.  The second forward sweep and the first
// backward one walk the image turned by 180 degrees: walk pixel p is image
// pixel H W - 1 - p, and nothing else differs.
//
// L, the winner codes and the argmins are those of the separate passes bit
// for bit (the same operations in the same order); the sums are
// S = (L_1 + L_0) + (L_3 + L_2), and dC, dP1, dP2 likewise.
//
// All accesses of a band are buffer accesses from its first pixel with the
// band's size as range; a lane outside the image (the skewed rows' first and
// last steps, a last band of fewer rows) gets an offset past the range, so it
// loads 0 and stores nothing, with no branch around any access: the wait
// counts of the load ring stay exact.
#include "dsgm_device.h"
#include "sgm_device.h"

#pragma clang fp contract(off)

namespace fsgm {
using namespace dsgm;
namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
using Rsrc = __amdgpu_buffer_rsrc_t;

__device__ __forceinline__ Rsrc rsrc_of(const void* p, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
template <int N>
__device__ __forceinline__ void bload(Rsrc r, uint32_t off, float (&v)[N]) {
#pragma unroll
    for (int k = 0; k < N; k += 4) {
        // the whole vector is cast: a bit cast of one element reads element 0
        const f32x4 t = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(off + 4 * k), 0, 0));
        v[k] = t.x; v[k + 1] = t.y; v[k + 2] = t.z; v[k + 3] = t.w;
    }
}
template <int N>
__device__ __forceinline__ void bstore(Rsrc r, uint32_t off, const float (&v)[N]) {
#pragma unroll
    for (int k = 0; k < N; k += 4) {
        const f32x4 t{v[k], v[k + 1], v[k + 2], v[k + 3]};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, t), r, (int)(off + 4 * k), 0, 0);
    }
}
__device__ __forceinline__ float bload1(Rsrc r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}
__device__ __forceinline__ void bstore1(Rsrc r, uint32_t off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, (int)off, 0, 0);
}
// A lane's winner codes are loaded as the dword that holds them and shifted
// at their use: a 1- or 2-byte load leaves its masking for the top of the
// loop, where it waits for the whole ring.
template <int D>
struct CodeLane {
    uint32_t store, load, shift;
    __device__ explicit CodeLane(int l) {
        store = (uint32_t)l * (D / 64);
        load = store & ~3u;
        shift = (store & 3u) * 8;
    }
};
template <int D>
__device__ __forceinline__ void bstore_codes(Rsrc r, uint32_t off, uint32_t w) {
    if constexpr (D == 64) __builtin_amdgcn_raw_buffer_store_b8((uint8_t)w, r, (int)off, 0, 0);
    else if constexpr (D == 128) __builtin_amdgcn_raw_buffer_store_b16((uint16_t)w, r, (int)off, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b32(w, r, (int)off, 0, 0);
}

__device__ __forceinline__ int bands_of(int H) { return (H + 3) / 4; }
// bytes of a pixel's codes of one direction, and of its floats
template <int D> constexpr int kCodeBytes = D / 4;
template <int D> constexpr int kCellBytes = D * 4;
// A band-relative pixel index no band reaches (sweep_ok bounds a band's cells
// to 2^30 bytes): its offset into any of the arrays is past their range.
template <int D> constexpr uint32_t kNoPixel = 0x80000000u / kCellBytes<D>;

// A wave's place in a band: lane (sub, l) stands for disparities
// l D/16 .. of row `sub`, sub steps behind row 0.
template <int D, bool TURNED>
struct Band {
    int W, rows, pixels;
    int64_t q0;            // lowest pixel of the band in the batch
    int x, limit;          // walk column of the next issue; columns of the lane's row (0: no such row)
    int pix;               // its pixel from q0
    __device__ Band(const DsgmArgs& A, int b, int g, int sub) {
        W = A.W;
        rows = min(4, A.H - 4 * g);
        pixels = rows * W;
        const int64_t img = (int64_t)A.H * W;
        q0 = (int64_t)b * img + (TURNED ? img - (int64_t)4 * g * W - pixels : (int64_t)4 * g * W);
        x = -sub;
        limit = sub < rows ? W : 0;
        pix = TURNED ? pixels - 1 - (sub * W - sub) : sub * W - sub;
    }
    // the pixel of the next issue, or kNoPixel; moves on by one column
    __device__ uint32_t next() {
        const uint32_t p = (uint32_t)x < (uint32_t)limit ? (uint32_t)pix : kNoPixel<D>;
        x += 1;
        pix += TURNED ? -1 : 1;
        return p;
    }
};

// The vertical state between the rows of a band: row `sub` writes slot
// sub + 1 and reads slot sub, the state of the row above one step earlier.
// Slot 0 is the band's edge of the next column, which row 0's lanes write;
// the other lanes' writes of it go to slot 4, which is never read.
template <int D>
struct Handover {
    float v[5][D];
    template <int DPD>
    __device__ void put(int slot, int l, const float (&x)[DPD]) {
#pragma unroll
        for (int k = 0; k < DPD; k += 4)
            *reinterpret_cast<f32x4*>(&v[slot][k * 16 + l * 4]) = f32x4{x[k], x[k + 1], x[k + 2], x[k + 3]};
    }
    template <int DPD>
    __device__ void pass(int sub, int l, const float (&own)[DPD], const float (&edge)[DPD], float (&above)[DPD]) {
        put(sub + 1, l, own);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        put(sub == 0 ? 0 : 4, l, edge);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < DPD; k += 4) {
            const f32x4 t = *reinterpret_cast<const f32x4*>(&v[sub][k * 16 + l * 4]);
            above[k] = t.x; above[k + 1] = t.y; above[k + 2] = t.z; above[k + 3] = t.w;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
};

// Edge states of a vertical direction: [direction 0, 2][image][band 1 ..][walk column][D]
__device__ __forceinline__ float* edge_at(const DsgmArgs& A, int second, int b, int band) {
    const int64_t nb1 = bands_of(A.H) - 1;
    return A.vol + ((((int64_t)second * A.B + b) * nb1 + (band - 1)) * A.W) * A.D;
}

// Steps of loads in flight.  A band's walk runs about one wave per SIMD, so
// the ring alone covers the memory latency: four steps of 2-5 KB per wave.
// (Six steps: the same.  At D = 256 four would pass the vector registers.)
template <int D> constexpr int kAheadS = D == 256 ? 2 : 4;

// ------------------------------------------------------------- forward ---
template <int D, bool LAST>
__device__ __forceinline__ void fwd_sweep(const DsgmArgs& A, int b, int g, int lane, Handover<D>& ho) {
    constexpr int DPD = D / 16, NA = kAheadS<D>, PH = LAST ? 3 : 1, PV = LAST ? 2 : 0;
    const float inf = __builtin_inff();
    const int sub = lane >> 4, l = lane & 15;
    const int W = A.W;
    Band<D, LAST> bd(A, b, g, sub);
    const int64_t npix = (int64_t)A.B * A.H * W, px = bd.pixels, q0 = bd.q0;
    const Rsrc rc = rsrc_of(A.cost + q0 * D, px * kCellBytes<D>), rs = rsrc_of(A.S + q0 * D, px * kCellBytes<D>);
    const Rsrc rp1 = rsrc_of(A.p1 + q0, px * 4), rp2 = rsrc_of(A.p2 + q0, px * 4);
    const Rsrc re = rsrc_of(edge_at(A, LAST, b, max(g, 1)), g > 0 ? (int64_t)W * kCellBytes<D> : 0);
    const Rsrc rwh = rsrc_of(A.wins + (PH * npix + q0) * kCodeBytes<D>, px * kCodeBytes<D>);
    const Rsrc rwv = rsrc_of(A.wins + (PV * npix + q0) * kCodeBytes<D>, px * kCodeBytes<D>);
    const Rsrc rkh = rsrc_of(A.kstar + PH * npix + q0, px), rkv = rsrc_of(A.kstar + PV * npix + q0, px);
    const Rsrc rd = rsrc_of(A.disp + q0, px * 4), rst = rsrc_of(A.stats + 2 * q0, px * 8);
    const uint32_t lane_c = (uint32_t)l * DPD * 4;
    const CodeLane<D> cl(l);
    const uint32_t only0 = l == 0 ? 0u : 0x80000000u;       // per-pixel values: stored by lane 0
    // row 0's edge, column by column; other rows stay past the range
    uint32_t eoff = sub == 0 ? lane_c : 0x80000000u;
    const uint32_t estep = sub == 0 ? (uint32_t)kCellBytes<D> : 0u;
    const bool top = g == 0 && sub == 0;                    // the vertical direction starts here

    float qc[NA][DPD], qe[NA][DPD], qs[NA][DPD], qp1[NA], qp2[NA];
    uint32_t qpix[NA];
    auto issue = [&](int u) __attribute__((always_inline)) {
        const uint32_t p = bd.next();
        qpix[u] = p;
        bload<DPD>(rc, p * kCellBytes<D> + lane_c, qc[u]);
        bload<DPD>(re, eoff, qe[u]);
        eoff += estep;
        qp1[u] = bload1(rp1, p * 4);
        qp2[u] = bload1(rp2, p * 4);
        if constexpr (LAST) bload<DPD>(rs, p * kCellBytes<D> + lane_c, qs[u]);
    };
#pragma unroll
    for (int u = 0; u < NA; ++u) {
        issue(u);
        __builtin_amdgcn_sched_barrier(0);
    }

    // L of the horizontal direction and of the row above.  At a direction's
    // first pixel the previous L is 0 and the penalties infinite: L = C.
    // (Columns before the first load a cost of 0, so L stays 0 there.)
    float Lh[DPD], Lv[DPD];
#pragma unroll
    for (int k = 0; k < DPD; ++k) {
        Lh[k] = 0.f;
        Lv[k] = sub == 0 ? qe[0][k] : 0.f;
    }
    int x = -sub;
    int t0 = 0;
    do {   // a loop guard would gather the ring's first loads behind it, out of order
#pragma unroll
        for (int u = 0; u < NA; ++u) {
            float mv = lane_min(Lv), mh = lane_min(Lh);
            row_min_both(mv, mh);
            int kv = lane_argmin<DPD>(Lv, mv, l), kh = lane_argmin<DPD>(Lh, mh, l);
            row_min_both(kv, kh);
            const uint32_t wv = fwd_step<DPD>(Lv, qc[u], mv, top ? inf : qp1[u], top ? inf : qp2[u]);
            float above[DPD];
            ho.pass(sub, l, Lv, qe[(u + 1) % NA], above);
            const uint32_t wh = fwd_step<DPD>(Lh, qc[u], mh, x <= 0 ? inf : qp1[u], x <= 0 ? inf : qp2[u]);
            float sum[DPD];
#pragma unroll
            for (int k = 0; k < DPD; ++k) {
                sum[k] = Lh[k] + Lv[k];
                Lv[k] = above[k];
                if constexpr (LAST) sum[k] = qs[u][k] + sum[k];
            }
            const uint32_t p = qpix[u];
            bstore<DPD>(rs, p * kCellBytes<D> + lane_c, sum);
            bstore_codes<D>(rwh, p * kCodeBytes<D> + cl.store, wh);
            bstore_codes<D>(rwv, p * kCodeBytes<D> + cl.store, wv);
            __builtin_amdgcn_raw_buffer_store_b8((uint8_t)kh, rkh, (int)(p | only0), 0, 0);
            __builtin_amdgcn_raw_buffer_store_b8((uint8_t)kv, rkv, (int)(p | only0), 0, 0);
            if constexpr (LAST) {
                float mn, z;
                const float d = soft_argmin<DPD>(sum, l, A.inv_temperature, &mn, &z);
                bstore1(rd, (p * 4) | only0, d);
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f32x2{mn, z}), rst,
                                                      (int)((p * 8) | only0), 0, 0);
            }
            x += 1;
            issue(u);
            __builtin_amdgcn_sched_barrier(0);   // loads stay a ring apart from their use
        }
        t0 += NA;
    } while (t0 < W + 3);
}

// ------------------------------------------------------------ backward ---
// gS of a pixel from S, its minimum mn, coef = gdisp (-1/T) / z and disp
template <int DPD>
__device__ __forceinline__ void grad_s_coef(const float (&s)[DPD], float mn, float coef, float dq, float c, int l,
                                            float (&g)[DPD]) {
#pragma unroll
    for (int k = 0; k < DPD; ++k) g[k] = coef * soft_weight(s[k], mn, c) * ((float)(l * DPD + k) - dq);
}

template <int D, bool LAST>
__device__ __forceinline__ void bwd_sweep(const DsgmArgs& A, int b, int g, int lane, Handover<D>& ho) {
    constexpr int DPD = D / 16, NA = kAheadS<D>, PH = LAST ? 3 : 1, PV = LAST ? 2 : 0;
    const int sub = lane >> 4, l = lane & 15;
    const int W = A.W;
    Band<D, !LAST> bd(A, b, g, sub);
    const int64_t npix = (int64_t)A.B * A.H * W, px = bd.pixels, q0 = bd.q0;
    const Rsrc rs = rsrc_of(A.S + q0 * D, px * kCellBytes<D>);
    const Rsrc rc = rsrc_of(A.grad_cost + q0 * D, px * kCellBytes<D>);
    const Rsrc rp1 = rsrc_of(A.grad_p1 + q0, px * 4), rp2 = rsrc_of(A.grad_p2 + q0, px * 4);
    const Rsrc re = rsrc_of(edge_at(A, LAST, b, max(g, 1)), g > 0 ? (int64_t)W * kCellBytes<D> : 0);
    const Rsrc rwh = rsrc_of(A.wins + (PH * npix + q0) * kCodeBytes<D>, px * kCodeBytes<D>);
    const Rsrc rwv = rsrc_of(A.wins + (PV * npix + q0) * kCodeBytes<D>, px * kCodeBytes<D>);
    const Rsrc rkh = rsrc_of(A.kstar + PH * npix + q0, px), rkv = rsrc_of(A.kstar + PV * npix + q0, px);
    const Rsrc rd = rsrc_of(A.disp + q0, px * 4), rst = rsrc_of(A.stats + 2 * q0, px * 8);
    const Rsrc rg = rsrc_of(A.vol_p1 + q0, px * 4);   // the pixels' coefficients
    const float sc = soft_scale(A.inv_temperature);
    const uint32_t lane_c = (uint32_t)l * DPD * 4;
    const CodeLane<D> cl(l);
    const uint32_t only0 = l == 0 ? 0u : 0x80000000u;
    uint32_t eoff = sub == 0 ? lane_c : 0x80000000u;
    const uint32_t estep = sub == 0 ? (uint32_t)kCellBytes<D> : 0u;
    // the pixel that each direction starts from (the walk's last column and
    // row) has no previous pixel and no penalty gradient: code 0 everywhere
    const uint32_t keep_v = 4 * g + sub == A.H - 1 ? 0u : ~0u;

    float qs[NA][DPD], qe[NA][DPD], qo[NA][DPD], qo1[NA], qo2[NA], qg[NA], qd[NA], qmn[NA];
    uint32_t qwh[NA], qwv[NA], qkh[NA], qkv[NA], qpix[NA];
    auto issue = [&](int u) __attribute__((always_inline)) {
        const uint32_t p = bd.next();
        qpix[u] = p;
        bload<DPD>(rs, p * kCellBytes<D> + lane_c, qs[u]);
        bload<DPD>(re, eoff, qe[u]);
        eoff += estep;
        qwh[u] = __builtin_amdgcn_raw_buffer_load_b32(rwh, (int)(p * kCodeBytes<D> + cl.load), 0, 0);
        qwv[u] = __builtin_amdgcn_raw_buffer_load_b32(rwv, (int)(p * kCodeBytes<D> + cl.load), 0, 0);
        qkh[u] = __builtin_amdgcn_raw_buffer_load_b8(rkh, (int)p, 0, 0);
        qkv[u] = __builtin_amdgcn_raw_buffer_load_b8(rkv, (int)p, 0, 0);
        qmn[u] = bload1(rst, p * 8);
        qg[u] = bload1(rg, p * 4);
        qd[u] = bload1(rd, p * 4);
        if constexpr (LAST) {
            bload<DPD>(rc, p * kCellBytes<D> + lane_c, qo[u]);
            qo1[u] = bload1(rp1, p * 4);
            qo2[u] = bload1(rp2, p * 4);
        }
    };
#pragma unroll
    for (int u = 0; u < NA; ++u) {
        issue(u);
        __builtin_amdgcn_sched_barrier(0);
    }

    // What the pixels after this one hand to it.  (Columns before the first
    // load a coefficient of 0 and hand on 0.)
    float Fh[DPD], Fv[DPD];
#pragma unroll
    for (int k = 0; k < DPD; ++k) {
        Fh[k] = 0.f;
        Fv[k] = sub == 0 ? qe[0][k] : 0.f;
    }
    int x = -sub;
    int t0 = 0;
    do {
#pragma unroll
        for (int u = 0; u < NA; ++u) {
            const uint32_t p = qpix[u];
            float gs[DPD], Gh[DPD], Gv[DPD], dc[DPD];
            grad_s_coef<DPD>(qs[u], qmn[u], qg[u], qd[u], sc, l, gs);
#pragma unroll
            for (int k = 0; k < DPD; ++k) {
                Gv[k] = gs[k] + Fv[k];
                Gh[k] = gs[k] + Fh[k];
                dc[k] = Gh[k] + Gv[k];
                if constexpr (LAST) dc[k] = qo[u][k] + dc[k];
            }
            bstore<DPD>(rc, p * kCellBytes<D> + lane_c, dc);
            float v12, v3, h12, h3, sums[4], own[DPD];
            sums[0] = bwd_flow<DPD>(Gv, (qwv[u] >> cl.shift) & keep_v, own, &v12, &v3);
            sums[1] = bwd_flow<DPD>(Gh, x == W - 1 ? 0u : qwh[u] >> cl.shift, Fh, &h12, &h3);
            sums[2] = h12 + v12;
            sums[3] = h3 + v3;
            row_sums(sums);
            bwd_jump<DPD>(own, (int)qkv[u], sums[0], l);
            ho.pass(sub, l, own, qe[(u + 1) % NA], Fv);
            bwd_jump<DPD>(Fh, (int)qkh[u], sums[1], l);
            float d1 = sums[2], d2 = sums[3];
            if constexpr (LAST) {
                d1 = qo1[u] + d1;
                d2 = qo2[u] + d2;
            }
            bstore1(rp1, (p * 4) | only0, d1);
            bstore1(rp2, (p * 4) | only0, d2);
            x += 1;
            issue(u);
            __builtin_amdgcn_sched_barrier(0);   // loads stay a ring apart from their use
        }
        t0 += NA;
    } while (t0 < W + 3);
}

// --------------------------------------------------------------- edges ---
// Four columns a wave, one 16-lane row each, walked down (direction 0) or up
// (direction 2; in the backward the reverse of each, 0 upwards).  Rows are
// loaded kAheadE steps ahead from wave-uniform addresses.
constexpr int kAheadE = 4;   // a band: its last step leaves the edge

template <int D, bool BWD>
__device__ __forceinline__ void edge_lines(const DsgmArgs& A, int b, int second, int group, int lane) {
    constexpr int DPD = D / 16, NA = kAheadE;
    const int sub = lane >> 4, l = lane & 15;
    const int W = A.W, H = A.H, nb1 = bands_of(H) - 1;
    const bool turned = BWD ? !second : second;
    const bool active = group * 4 + sub < W;
    const int xw = min(group * 4 + sub, W - 1);             // walk column
    const int col = turned ? W - 1 - xw : xw;
    const int64_t npix = (int64_t)A.B * H * W, img0 = (int64_t)b * H * W;
    const uint32_t lane_c = (uint32_t)col * kCellBytes<D> + l * DPD * 4;
    const CodeLane<D> cl(l);
    const uint32_t eoff = active ? (uint32_t)xw * kCellBytes<D> + l * DPD * 4 : 0x80000000u;
    const int path = second ? 2 : 0;
    const int64_t row_c = (int64_t)W * kCellBytes<D>;

    float q[NA][DPD], q1[NA], q2[NA], q3[NA];
    uint32_t qw[NA], qk[NA];
    auto issue = [&](int u, int s) __attribute__((always_inline)) {
        s = min(s, H - 1);                                   // rows past the end: loaded, not used
        const int64_t r0 = img0 + (int64_t)(turned ? H - 1 - s : s) * W;
        if constexpr (!BWD) {
            bload<DPD>(rsrc_of(A.cost + r0 * D, row_c), lane_c, q[u]);
            q1[u] = bload1(rsrc_of(A.p1 + r0, (int64_t)W * 4), col * 4);
            q2[u] = bload1(rsrc_of(A.p2 + r0, (int64_t)W * 4), col * 4);
        } else {
            bload<DPD>(rsrc_of(A.S + r0 * D, row_c), lane_c, q[u]);
            q1[u] = bload1(rsrc_of(A.stats + 2 * r0, (int64_t)W * 8), col * 8);
            q2[u] = bload1(rsrc_of(A.vol_p1 + r0, (int64_t)W * 4), col * 4);
            q3[u] = bload1(rsrc_of(A.disp + r0, (int64_t)W * 4), col * 4);
            qw[u] = __builtin_amdgcn_raw_buffer_load_b32(
                rsrc_of(A.wins + (path * npix + r0) * kCodeBytes<D>, (int64_t)W * kCodeBytes<D>),
                (int)(col * kCodeBytes<D> + cl.load), 0, 0);
            qk[u] = __builtin_amdgcn_raw_buffer_load_b8(rsrc_of(A.kstar + path * npix + r0, W), col, 0, 0);
        }
    };
#pragma unroll
    for (int u = 0; u < NA; ++u) {
        issue(u, u);
        __builtin_amdgcn_sched_barrier(0);
    }
    // forward: L of the row above (0 and infinite penalties before the first
    // row); backward: what the row after hands over
    float v[DPD];
#pragma unroll
    for (int k = 0; k < DPD; ++k) v[k] = 0.f;
    int band = 0;
    do {
#pragma unroll
        for (int u = 0; u < NA; ++u) {
            if constexpr (!BWD) {
                const bool start = u == 0 && band == 0;
                const float inf = __builtin_inff();
                const float m = row_min(lane_min(v));
                fwd_step<DPD>(v, q[u], m, start ? inf : q1[u], start ? inf : q2[u]);
            } else {
                float gs[DPD], s12, s3;
                grad_s_coef<DPD>(q[u], q1[u], q2[u], q3[u], soft_scale(A.inv_temperature), l, gs);
#pragma unroll
                for (int k = 0; k < DPD; ++k) gs[k] = gs[k] + v[k];
                const float rest = bwd_flow<DPD>(gs, qw[u] >> cl.shift, v, &s12, &s3);
                bwd_jump<DPD>(v, (int)qk[u], row_sumf(rest), l);
            }
            if (u == NA - 1) bstore<DPD>(rsrc_of(edge_at(A, second, b, band + 1), row_c), eoff, v);
            issue(u, band * NA + u + NA);
            __builtin_amdgcn_sched_barrier(0);
        }
    } while (++band < nb1);   // launched where nb1 >= 1
}

// One wave per workgroup: the 752 bands of eight driving frames then spread
// over all CUs (four waves to a workgroup 7.74 ms, one 7.03 ms).  What bounds a
// sweep: 300-420 VALU instructions per step at about 4.5 cycles each (a wave
// alone on its SIMD), 0.9-1.2 ms over 1242 columns, beside its share of HBM.
//
// The first sweep's launch also holds the edges of the second direction: the
// sweep leaves memory bandwidth and wave slots that they fill.
template <int D, bool BWD, bool LAST>
__global__ __launch_bounds__(64) void dsgm_sweep_kernel(DsgmArgs A, int sweeps) {
    __shared__ __align__(16) Handover<D> ho;
    if (LAST || (int)blockIdx.x < sweeps) {
        const int nb = bands_of(A.H), item = blockIdx.x;
        const int b = item / nb, g = item - b * nb;
        if constexpr (BWD) bwd_sweep<D, LAST>(A, b, g, threadIdx.x, ho);
        else fwd_sweep<D, LAST>(A, b, g, threadIdx.x, ho);
    } else {
        const int nv = (A.W + 3) / 4;
        const int item = dev::xcd_item((int)blockIdx.x - sweeps, (int)gridDim.x - sweeps);
        const int b = item / nv;
        edge_lines<D, BWD>(A, b, 1, item - b * nv, threadIdx.x);
    }
}

template <int D, bool BWD>
__global__ __launch_bounds__(64) void dsgm_edge_kernel(DsgmArgs A) {
    const int nv = (A.W + 3) / 4;
    const int item = dev::xcd_item(blockIdx.x, gridDim.x);
    const int b = item / nv;
    edge_lines<D, BWD>(A, b, 0, item - b * nv, threadIdx.x);
}

// gdisp (-1/T) / z of every pixel, which each pass of the backward needs
__global__ __launch_bounds__(256) void dsgm_coef_kernel(DsgmArgs A, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) A.vol_p1[i] = A.grad_disp[i] * (-A.inv_temperature) / A.stats[2 * i + 1];
}

template <int D, bool BWD>
hipError_t launch_sweeps(const DsgmArgs& A, hipStream_t s) {
    const unsigned nb = (unsigned)((A.H + 3) / 4);
    const unsigned sweeps = (unsigned)A.B * nb;
    const unsigned columns = (unsigned)A.B * ((A.W + 3) / 4);
    const unsigned edges = nb > 1 ? columns : 0;
    if constexpr (BWD) {
        const int64_t n = (int64_t)A.B * A.H * A.W;
        hipLaunchKernelGGL(dsgm_coef_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, A, n);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (nb > 1) {
        hipLaunchKernelGGL((dsgm_edge_kernel<D, BWD>), dim3(columns), dim3(64), 0, s, A);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((dsgm_sweep_kernel<D, BWD, false>), dim3(sweeps + edges), dim3(64), 0, s, A,
                       (int)sweeps);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((dsgm_sweep_kernel<D, BWD, true>), dim3(sweeps), dim3(64), 0, s, A, (int)sweeps);
    return hipGetLastError();
}

template <bool BWD>
hipError_t launch_by_d(const DsgmArgs& A, hipStream_t s) {
    switch (A.D) {
        case 64: return launch_sweeps<64, BWD>(A, s);
        case 128: return launch_sweeps<128, BWD>(A, s);
        case 256: return launch_sweeps<256, BWD>(A, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

// Taken from 390 bands on (450 at D = 64), about 0.4 waves per SIMD: the walk of
// a band's W + 3 steps of two directions lasts as long for few images as for
// many, and below that the separate passes are sooner done.  Forward +
// backward, ms, separate -> sweeps, 375 rows of 1242 unless given:
//   D = 128: 4 images (376 bands) 4.76 -> 4.96, 5 (470) 6.40 -> 5.22, 8 (752)
//   9.97 -> 7.03; 8 images 1000x180 (360) 3.60 -> 3.97, 1242x200 (400) 5.75 -> 5.02
//   D = 64: 4 images 2.37 -> 2.80, 5 3.11 -> 2.97, 8 5.07 -> 3.70; 8 images
//   600x196 (392) 1.23 -> 1.35
//   D = 256: 4 images 9.82 -> 9.75; 8 images 600x375 (752) 9.81 -> 7.21, 600x150
//   (304) 4.04 -> 4.45
// With that many bands there also have to be 24M cells (28M at D = 64), or the
// launches and the walks' ends weigh more than the traffic, unless the images are
// tall, whose column walks the sweeps run once fewer (us: D = 64, 32 images 120x64,
// 16M, 217 -> 290, 250x64, 33M, 600 -> 573; D = 128, 32 images 64x64, 17M, 236 -> 293,
// 120x64, 31M, 579 -> 493; D = 256, 100 images 30x20, 15M, 237 -> 270, 64x20, 33M,
// 638 -> 535; 16 images 30x128, D = 64 194 -> 175, 128 302 -> 257; 60 images 8x40,
// D = 64 72 -> 69, but 100 images 8x20, D = 128 64 -> 73), and a last band of
// few rows wastes the rest of its wave (width 1000, of 1, 5, 6, 7, 9, 13 rows: D = 64
// 821 -> 1936, 1624 -> 2176, 1903 -> 2234, 2370 -> 2294, 2098 -> 2254, 2418 -> 2543;
// D = 128 1439 -> 3409, 3262 -> 3872, 3804 -> 3915, 4616 -> 4009, 4220 -> 3974, 4611 ->
// 4665; D = 256 2854 -> 6406, 6730 -> 7446, 7998 -> 7676, 9714 -> 7907, 8801 -> 7775,
// 9476 -> 9546).
// A band's cells stay below 2^30 bytes, so that 32-bit offsets and kNoPixel hold.
bool dsgm_sweep_ok(const DsgmArgs& A) {
    const int64_t bands = (A.H + 3) / 4, cells = (int64_t)A.B * A.H * A.W * A.D;
    const bool tall = A.H >= 40 && 2 * (int64_t)A.H >= 5 * (int64_t)A.W;
    return A.B * bands >= (A.D == 64 ? 450 : 390) && (tall || cells >= (A.D == 64 ? 28000000 : 24000000)) &&
           100 * (int64_t)A.H >= (A.D == 64 ? 85 : 70) * 4 * bands && (int64_t)A.W * A.D <= (int64_t)1 << 26;
}
hipError_t dsgm_sweep_forward(const DsgmArgs& A, hipStream_t s) { return launch_by_d<false>(A, s); }
hipError_t dsgm_sweep_backward(const DsgmArgs& A, hipStream_t s) { return launch_by_d<true>(A, s); }

}  // namespace fsgm
