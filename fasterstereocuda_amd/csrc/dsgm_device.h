// Device helpers of the differentiable SGM kernels: 16-lane row reductions,
// the forward step, the soft-argmin and its gradient (gfx950, wave64).
#pragma once

#include <cmath>

#include "dsgm_internal.h"

#pragma clang fp contract(off)

namespace fsgm {
namespace dsgm {

template <int CTRL>
__device__ __forceinline__ float dppf(float old, float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
        __builtin_bit_cast(int, old), __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ __forceinline__ int dppi(int old, int v) {
    return __builtin_amdgcn_update_dpp(old, v, CTRL, 0xF, 0xF, false);
}
constexpr int kShl1 = 0x101, kShr1 = 0x111;

// (written out: fminf of a moved value costs a separate move and a
// canonicalising v_max per stage)
__device__ __forceinline__ float row_min(float a) {
    asm("s_nop 1\n\t"
        "v_min_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_min_f32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_min_f32_dpp %0, %0, %0 row_ror:2 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_min_f32_dpp %0, %0, %0 row_ror:1 row_mask:0xf bank_mask:0xf"
        : "+v"(a));
    return a;
}
__device__ __forceinline__ float row_sumf(float v) {
    v = v + dppf<0x128>(0.f, v);
    v = v + dppf<0x124>(0.f, v);
    v = v + dppf<0x122>(0.f, v);
    v = v + dppf<0x121>(0.f, v);
    return v;
}
__device__ __forceinline__ int row_mini(int v) {
    v = min(v, dppi<0x128>(0, v));
    v = min(v, dppi<0x124>(0, v));
    v = min(v, dppi<0x122>(0, v));
    v = min(v, dppi<0x121>(0, v));
    return v;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) f32x4 g_f4;
typedef __attribute__((address_space(1))) float g_f;

template <int N>
__device__ __forceinline__ void loadf(const float* p, float (&v)[N]) {
#pragma unroll
    for (int k = 0; k < N; k += 4) {
        const f32x4 t = *(const g_f4*)(p + k);
        v[k] = t.x; v[k + 1] = t.y; v[k + 2] = t.z; v[k + 3] = t.w;
    }
}
template <int N>
__device__ __forceinline__ void storef(float* p, const float (&v)[N]) {
#pragma unroll
    for (int k = 0; k < N; k += 4) *(g_f4*)(p + k) = f32x4{v[k], v[k + 1], v[k + 2], v[k + 3]};
}
__device__ __forceinline__ float loads(const float* p) { return *(const g_f*)p; }

// A lane's winner codes of one step: DPD = D / 16 disparities, 2 bits each.
template <int D> struct WinWordOf;
template <> struct WinWordOf<64> { using type = uint8_t; };
template <> struct WinWordOf<128> { using type = uint16_t; };
template <> struct WinWordOf<256> { using type = uint32_t; };
template <int D> using WinWord = typename WinWordOf<D>::type;

// one forward step for a lane's DPD disparities; returns winners packed 2 bits each
template <int DPD>
__device__ __forceinline__ uint32_t fwd_step(float (&L)[DPD], const float (&c)[DPD], float m,
                                             float p1, float p2) {
    const float inf = __builtin_inff();
    const float prev_last = dppf<kShr1>(inf, L[DPD - 1]);
    const float next_first = dppf<kShl1>(inf, L[0]);
    const float c3 = m + p2;
    uint32_t wins = 0;
    float nl[DPD];
#pragma unroll
    for (int k = 0; k < DPD; ++k) {
        const float lm = (k == 0) ? prev_last : L[k - 1];
        const float lp = (k == DPD - 1) ? next_first : L[k + 1];
        float best = L[k];
        uint32_t w = 0;
        const float c1 = lm + p1, c2 = lp + p1;
        if (c1 < best) { best = c1; w = 1; }
        if (c2 < best) { best = c2; w = 2; }
        if (c3 < best) { best = c3; w = 3; }
        nl[k] = (c[k] + best) - m;
        wins |= w << (2 * k);
    }
#pragma unroll
    for (int k = 0; k < DPD; ++k) L[k] = nl[k];
    return wins;
}

template <int DPD>
__device__ __forceinline__ float lane_min(const float (&L)[DPD]) {
    float v = L[0];
#pragma unroll
    for (int k = 1; k < DPD; ++k) v = fminf(v, L[k]);
    return v;
}

// Unnormalised softmax weight exp(-(s - mn) / T) = 2^((mn - s) * c) with
// c = log2(e) / T: one v_exp_f32 after a subtraction and a product.  The
// forward and the backward use this same form.  The argument is <= 0, and a
// weight below 2^-126 (a cost more than 87 T above the minimum) contributes
// nothing to the sums either way.
__device__ __forceinline__ float soft_weight(float s, float mn, float c) {
    return __builtin_amdgcn_exp2f((mn - s) * c);
}
__device__ __forceinline__ float soft_scale(float invT) { return invT * 1.44269504088896340736f; }

// Soft-argmin of one pixel per 16-lane row: s holds S, every lane of the row
// receives the disparity, the minimum mn and the normaliser z.
template <int DPD>
__device__ __forceinline__ float soft_argmin(const float (&s)[DPD], int l, float invT, float* mn_out,
                                             float* z_out) {
    const float mn = row_min(lane_min(s));
    const float c = soft_scale(invT);
    float z = 0.f, acc = 0.f;
#pragma unroll
    for (int k = 0; k < DPD; ++k) {
        const float e = soft_weight(s[k], mn, c);
        z += e;
        acc += (float)(l * DPD + k) * e;
    }
    z = row_sumf(z);
    acc = row_sumf(acc);
    *mn_out = mn;
    *z_out = z;
    return acc / z;
}

// gS(p, d) = gdisp(p) * (-1/T) * prob(p, d) * (d - disp(p)) of one pixel,
// from S and the forward's minimum mn and normaliser z of that pixel.
template <int DPD>
__device__ __forceinline__ void grad_s_from(const float (&s)[DPD], float mn, float z, float gd,
                                            float dq, float invT, int l, float (&g)[DPD]) {
    const float coef = gd * (-invT) / z;
    const float c = soft_scale(invT);
#pragma unroll
    for (int k = 0; k < DPD; ++k)
        g[k] = coef * soft_weight(s[k], mn, c) * ((float)(l * DPD + k) - dq);
}

// Row reductions of several values stage by stage: a DPP read has to wait two
// states after the write of its register, which the other values' moves fill.
__device__ __forceinline__ void row_min_both(float& a, float& b) {
    asm("s_nop 1\n\t"
        "v_min_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_min_f32_dpp %1, %1, %1 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0\n\t"
        "v_min_f32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_min_f32_dpp %1, %1, %1 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0\n\t"
        "v_min_f32_dpp %0, %0, %0 row_ror:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_min_f32_dpp %1, %1, %1 row_ror:2 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0\n\t"
        "v_min_f32_dpp %0, %0, %0 row_ror:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_min_f32_dpp %1, %1, %1 row_ror:1 row_mask:0xf bank_mask:0xf"
        : "+v"(a), "+v"(b));
}
template <int CTRL, int N>
__device__ __forceinline__ void add_stage(float (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] += dppf<CTRL>(0.f, v[i]);
    __builtin_amdgcn_sched_barrier(0);
}
template <int N>
__device__ __forceinline__ void row_sums(float (&v)[N]) {
    add_stage<0x128>(v);
    add_stage<0x124>(v);
    add_stage<0x122>(v);
    add_stage<0x121>(v);
}
// smallest d with L(d) == m in a lane (none: a large value)
template <int DPD>
__device__ __forceinline__ int lane_argmin(const float (&L)[DPD], float m, int l) {
    int idx = 0x7FFFFFFF;
#pragma unroll
    for (int k = DPD - 1; k >= 0; --k)
        if (L[k] == m) idx = l * DPD + k;
    return idx;
}
template <int CTRL>
__device__ __forceinline__ void min_stage(int& a, int& b) {
    a = min(a, dppi<CTRL>(0, a));
    b = min(b, dppi<CTRL>(0, b));
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void row_min_both(int& a, int& b) {
    min_stage<0x128>(a, b);
    min_stage<0x124>(a, b);
    min_stage<0x122>(a, b);
    min_stage<0x121>(a, b);
}

// What a pixel's gradient G of one direction hands to the pixel before it
// (w, ks: the pixel's winner codes and the previous pixel's argmin), and the
// lane's shares of its penalty gradients.
// The codes' two bits become masks, so a share is one three-input bit
// operation; F is left without the argmin's term, whose amount is less the
// sum of F (a code 3 hands nothing on).
template <int DPD>
__device__ __forceinline__ float bwd_flow(const float (&G)[DPD], uint32_t w, float (&F)[DPD], float* s12, float* s3) {
    float A1[DPD], A2[DPD], a12 = 0.f, a3 = 0.f, rest = 0.f;
#pragma unroll
    for (int k = 0; k < DPD; ++k) {
        const uint32_t g = __builtin_bit_cast(uint32_t, G[k]);
        // written out: the compiler turns shifted masks into compares and selects
        uint32_t b0, b1;
        asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(b0) : "v"(w), "i"(2 * k));
        asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(b1) : "v"(w), "i"(2 * k + 1));
        F[k] = __builtin_bit_cast(float, g & ~(b0 | b1));
        A1[k] = __builtin_bit_cast(float, g & b0 & ~b1);   // to d - 1
        A2[k] = __builtin_bit_cast(float, g & b1 & ~b0);   // to d + 1
        a3 += __builtin_bit_cast(float, g & b0 & b1);
        a12 += A1[k] + A2[k];
    }
    const float a1_next = dppf<kShl1>(0.f, A1[0]);
    const float a2_prev = dppf<kShr1>(0.f, A2[DPD - 1]);
#pragma unroll
    for (int k = 0; k < DPD; ++k) {
        F[k] += (k == DPD - 1) ? a1_next : A1[k + 1 < DPD ? k + 1 : k];
        F[k] += (k == 0) ? a2_prev : A2[k > 0 ? k - 1 : 0];
        rest += F[k];
    }
    *s12 = a12;
    *s3 = a3;
    return rest + (a3 - a3);   // a gradient that is no number reaches the argmin too
}
// the argmin's term, to disparity ks
template <int DPD>
__device__ __forceinline__ void bwd_jump(float (&F)[DPD], int ks, float rest, int l) {
    const int kl = ks - l * DPD;
#pragma unroll
    for (int k = 0; k < DPD; ++k) F[k] -= (kl == k) ? rest : 0.f;
}

}  // namespace dsgm
}  // namespace fsgm
