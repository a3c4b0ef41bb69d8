// Device helpers of the aggregation kernels: one scanline held as packed u16
// pairs over the lanes of a line, its recurrence step, costs from census words,
// and buffer accesses (gfx950, wave64).
#pragma once

#include "sgm_device.h"

namespace fsgm {
namespace dev {

typedef unsigned int buf_u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int buf_u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_at(const uint8_t* p, uint32_t bytes = 0x7fffffffu) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)bytes, 0x00020000);
}
template <int NW>
__device__ __forceinline__ void buf_load(__amdgpu_buffer_rsrc_t r, uint32_t v, int s, uint32_t (&w)[NW]) {
    if constexpr (NW == 1) {
        w[0] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)v, s, 0);
    } else if constexpr (NW == 2) {
        const buf_u32x2 t = __builtin_amdgcn_raw_buffer_load_b64(r, (int)v, s, 0);
        w[0] = t.x; w[1] = t.y;
    } else {
#pragma unroll
        for (int k = 0; k < NW; k += 4) {
            const buf_u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(v + 4 * k), s, 0);
            w[k] = t.x; w[k + 1] = t.y; w[k + 2] = t.z; w[k + 3] = t.w;
        }
    }
}
// A 128-bit store takes its step offset in the vector offset: with a scalar
// offset register the compiler leaves the data registers free to be rewritten
// by the next instruction, and under load such stores have written the later
// values (D = 256 beside two larger pairs); without one it keeps the wait
// state that stores of more than 64 bits need.
template <int NW>
__device__ __forceinline__ void buf_store(__amdgpu_buffer_rsrc_t r, uint32_t v, int s, const uint32_t (&w)[NW]) {
    if constexpr (NW == 1) {
        __builtin_amdgcn_raw_buffer_store_b32(w[0], r, (int)v, s, 0);
    } else if constexpr (NW == 2) {
        __builtin_amdgcn_raw_buffer_store_b64(buf_u32x2{w[0], w[1]}, r, (int)v, s, 0);
    } else {
#pragma unroll
        for (int k = 0; k < NW; k += 4)
            __builtin_amdgcn_raw_buffer_store_b128(buf_u32x4{w[k], w[k + 1], w[k + 2], w[k + 3]}, r,
                                                   (int)(v + 4 * k + s), 0, 0);
    }
}

// value of the previous / next lane of the line; the line's first / last
// lane gets `edge`
template <int LPL>
__device__ __forceinline__ uint32_t from_prev(uint32_t v, uint32_t edge, bool first) {
    if constexpr (LPL == 16) {
        return dpp<kRowShr1>(edge, v);
    } else {
        const uint32_t s = dpp0<kRowShr1>(v);   // every lane moves; the first then takes `edge`
        return first ? edge : s;
    }
}
template <int LPL>
__device__ __forceinline__ uint32_t from_next(uint32_t v, uint32_t edge, bool last) {
    if constexpr (LPL == 16) {
        return dpp<kRowShl1>(edge, v);
    } else {
        const uint32_t s = dpp0<kRowShl1>(v);
        return last ? edge : s;
    }
}

// popcount(a) + acc as two accumulating v_bcnt_u32_b32.  Written out, the
// compiler regroups the sum and packs with a v_lshl_or_b32; this form packs
// the upper count with a v_lshlrev_b32, which issues at twice the rate.
__device__ __forceinline__ uint32_t bcnt_acc(uint32_t x, uint32_t acc) {
    uint32_t r;
    asm("v_bcnt_u32_b32 %0, %1, %2" : "=v"(r) : "v"(x), "v"(acc));
    return r;
}
__device__ __forceinline__ uint32_t popc_acc(uint64_t a, uint32_t acc) {
    return bcnt_acc((uint32_t)a, bcnt_acc((uint32_t)(a >> 32), acc));
}

// One recurrence step of a line, NP packed u16 pairs (2 NP disparities) per lane:
//   L(d) = C(d) + min(L'(d), B-(d), B+(d), m' + P2) - m'
//   B-(d) = d == 0 ? 127 : L'(d-1) + P1,  B+(d) = d == D-1 ? 127 : L'(d+1) + P1
template <int NP>
struct Line {
    uint32_t L[NP];
    uint32_t m;   // the line minimum in both u16 halves
    // 16-lane lines: the neighbours from the lanes beside, whose out-of-row
    // lanes no shift writes and so keep the 127 terms
    uint32_t prev = 127u << 16, next = 127u;
};

// both halves = the smaller half (v_pk_min_u16 with swapped operand halves);
// a u32 minimum of such values is their u16 minimum
__device__ __forceinline__ uint32_t pk_min_halves(uint32_t v) {
    return as_u(__builtin_elementwise_min(as_v(v), as_v(v).yx));
}

template <bool BIG, int LPL, int NP>
__device__ __forceinline__ void line_init(Line<NP>& s, const uint32_t (&c)[NP]) {
#pragma unroll
    for (int k = 0; k < NP; ++k) s.L[k] = c[k];
    s.m = line_min<LPL>(pk_min_halves(pk_min_all<BIG>(s.L)));
}

// The sums of a step never carry or borrow between the u16 halves: costs are
// at most 64, the line minimum is at most the cost at the previous minimum's
// disparity (so below every term, 127 included) and P1 + P2 <= 65000.  So
// they are 32-bit adds and subtracts, which issue in 2 cycles where the packed
// forms take 4.

template <bool BIG, int LPL, int NP>
__device__ __forceinline__ void line_step(Line<NP>& s, const uint32_t (&c)[NP], uint32_t P1v,
                                          uint32_t P2v, bool first, bool last) {
    const uint32_t mv = s.m;
    const uint32_t mp2 = mv + P2v;
    uint32_t R[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) R[k] = s.L[k] + P1v;
    uint32_t prev_last, next_first;
    if constexpr (LPL == 16) {
        prev_last = s.prev = dpp<kRowShr1>(s.prev, R[NP - 1]);
        next_first = s.next = dpp<kRowShl1>(s.next, R[0]);
    } else {
        prev_last = from_prev<LPL>(R[NP - 1], 127u << 16, first);
        next_first = from_next<LPL>(R[0], 127u, last);
    }
    uint32_t E[NP + 1];
    E[0] = __builtin_amdgcn_alignbit(R[0], prev_last, 16);
#pragma unroll
    for (int k = 1; k < NP; ++k) E[k] = __builtin_amdgcn_alignbit(R[k], R[k - 1], 16);
    E[NP] = __builtin_amdgcn_alignbit(next_first, R[NP - 1], 16);
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        const uint32_t v = pk_min(pk_min3<BIG>(s.L[k], E[k], E[k + 1]), mp2);
        s.L[k] = c[k] + v;
    }
    s.m = line_min<LPL>(pk_min_halves(pk_min_all<BIG>(s.L)));
}

// The lane's 2 NP bytes (uint8 truncation).  The volumes these kernels hand
// each other keep a word's bytes in the order d, d + 2, d + 1, d + 3, so the
// reader gets two packed u16 pairs from a word with a 2-cycle mask and one
// packed shift instead of two v_perm.
template <int NP>
__device__ __forceinline__ void pack_lane(const Line<NP>& s, uint32_t sel, uint32_t (&o)[NP / 2]) {
#pragma unroll
    for (int k = 0; k < NP / 2; ++k) o[k] = __builtin_amdgcn_perm(s.L[2 * k + 1], s.L[2 * k], sel);
}
// pairs 2k and 2k + 1 of a word
__device__ __forceinline__ uint32_t word_pair(uint32_t w, int odd) {
    return odd ? as_u(as_v(w) >> (u16x2)8) : (w & 0x00FF00FFu);
}

constexpr uint32_t kSelFwd = 0x06020400u;   // bytes d, d+2, d+1, d+3
// lanes that hold the disparities in reversed order swap a pair's halves, so
// that the reader (which takes their words in reversed order) finds d before d + 1
constexpr uint32_t kSelRev = 0x04000602u;

// packed costs of one lane: pair k = (partner 2k, partner 2k + 1)
template <int NP, class F>
__device__ __forceinline__ void lane_costs(uint64_t own, uint32_t base, F&& partner, uint32_t (&c)[NP]) {
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        uint32_t t;
        asm("v_lshl_add_u32 %0, %1, 16, %2" : "=v"(t) : "v"(popc_acc(own ^ partner(2 * k + 1), 0u)), "v"(base));
        c[k] = popc_acc(own ^ partner(2 * k), t);
    }
}

// value of lane `src` (a compile-time constant after unrolling) of the line,
// on every lane of the line: quad_perm, or row_newbcast (the broadcast of one
// lane of a 16-lane DPP row; two of them, by halves, where a line is 8 lanes)
template <int LPL, int SRC>
__device__ __forceinline__ uint32_t line_bcast_c(uint32_t v) {
    if constexpr (LPL == 4) {
        return dpp0<SRC * 0x55>(v);
    } else if constexpr (LPL == 16) {
        return dpp0<0x150 + SRC>(v);
    } else {
        const int lo = (int)dpp0<0x150 + SRC>(v);
        return (uint32_t)__builtin_amdgcn_update_dpp(lo, (int)v, 0x150 + SRC + 8, 0xF, 0xC, false);
    }
}
template <int LPL>
__device__ __forceinline__ uint32_t line_bcast(uint32_t v, int src) {
    switch (src) {
        case 0: return line_bcast_c<LPL, 0>(v);
        case 1: return line_bcast_c<LPL, 1>(v);
        case 2: return line_bcast_c<LPL, 2>(v);
        case 3: return line_bcast_c<LPL, 3>(v);
        default: break;
    }
    if constexpr (LPL >= 8)
        switch (src) {
            case 4: return line_bcast_c<LPL, 4>(v);
            case 5: return line_bcast_c<LPL, 5>(v);
            case 6: return line_bcast_c<LPL, 6>(v);
            case 7: return line_bcast_c<LPL, 7>(v);
            default: break;
        }
    if constexpr (LPL >= 16)
        switch (src) {
            case 8: return line_bcast_c<LPL, 8>(v);
            case 9: return line_bcast_c<LPL, 9>(v);
            case 10: return line_bcast_c<LPL, 10>(v);
            case 11: return line_bcast_c<LPL, 11>(v);
            case 12: return line_bcast_c<LPL, 12>(v);
            case 13: return line_bcast_c<LPL, 13>(v);
            case 14: return line_bcast_c<LPL, 14>(v);
            case 15: return line_bcast_c<LPL, 15>(v);
            default: break;
        }
    return v;
}
template <int LPL>
__device__ __forceinline__ uint64_t line_bcast64(uint64_t v, int src) {
    const uint32_t lo = line_bcast<LPL>((uint32_t)v, src);
    const uint32_t hi = line_bcast<LPL>((uint32_t)(v >> 32), src);
    return ((uint64_t)hi << 32) | lo;
}

}  // namespace dev
}  // namespace fsgm
