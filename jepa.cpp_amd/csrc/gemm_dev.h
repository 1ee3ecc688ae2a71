// gemm_dev.h - what the GEMM kernels share on the device: the launch arguments and the epilogue of four
// consecutive output features of one row.
#pragma once
#include "kernels.h"

#include <cstdint>

namespace {

struct kargs {
    const _Float16 * A;      // [N][K] weight codes (or f16 / f32 weights)
    const uint16_t * Ad;     // W_Q32, W_Q40: f16 d [N][K/32]; W_Q4K: u32 (d | dmin << 16) [K/256][N]
    const _Float16 * Amin;   // W_Q4K: [N][K/256][16] sub-block mins, each twice
    const uint8_t * Asc;     // W_Q4K: [N][K/256][8] 6-bit sub-block scales
    const _Float16 * B;      // [M][K] activation codes (or f16 / f32 activations)
    const void * Bd;         // A_Q8_0: f16 d [M][K/32]; A_Q8_K: f32 d [M][K/256]
    const _Float16 * Bsum;   // A_Q8_K: f16 bsums [M][K/16]
    const float * bias;
    int64_t M, N, K;
    int tn, tm;              // workgroup tiles along N and M
    int xa, xb;              // tiles per XCD block along N and M (0: plain order)
    int split;               // K halves computed by separate workgroups (1 or 2; q8_0 / q4_0 / q4_K)
    float * part;            // split: raw accumulators of every workgroup [split][tiles][BN*BM]
    int * cnt;               // split: arrivals per tile (0 between launches)
    gemm_epi ep;
};

// GELU(x) = 0.5 x (1 + erf(x / sqrt 2)) = x Phi(x) (ggml_vec_gelu_erf_f32, reference
// docs/ggml-notes.md:291-292), Phi the standard normal CDF, from its tail h(t) = Phi(-t), t = |x|:
//   Phi(x) = 1 - h(t) for x >= 0, h(t) for x < 0,   h(t) = 2^Q(min(t, 5.5)), Q of degree 8 with Q(0) = -1
// One polynomial and one hardware exp2 per value, no branch: 14 VALU ops where erf's two-piece form
// (both pieces evaluated, one selected) took 25. Coefficients from fit_gelu.py (fitted with weight h,
// so the absolute error of Phi is minimised; Q(0) = -1 gives Phi(0) = 1/2 exactly): the float32
// evaluation stays within 1.5 units of 2^-24 of Phi (2.5 with exp2 two units off), about the accuracy
// of the libm erff form. At t = 5.5, h = 1.9e-8 < 2^-25, so 1 - h is 1.0f and GELU(x) = x beyond.
__device__ __forceinline__ float gelu_erf(float x) {
    const float t = fminf(fabsf(x), 5.5f);
    float q = -2.248140163e-06f;
    q = fmaf(q, t, 3.268636283e-05f);
    q = fmaf(q, t, -1.560558158e-04f);
    q = fmaf(q, t, -2.054840443e-04f);
    q = fmaf(q, t, 7.147170603e-03f);
    q = fmaf(q, t, -5.254988000e-02f);
    q = fmaf(q, t, -4.591920078e-01f);
    q = fmaf(q, t, -1.151106834e+00f);
    q = fmaf(q, t, -1.0f);
    const float h = __builtin_amdgcn_exp2f(q);
    return __fmul_rn(x, x >= 0.0f ? __fsub_rn(1.0f, h) : h);
}

__device__ __forceinline__ int perm16(int64_t tok) {
    // position of token `tok` inside its 16-token group of V^T (see attention.hip)
    const int key = (int) (tok & 15);
    const int gg = (key >> 2) & 1, s = (key & 3) + 4 * (key >> 3);
    return (int) (tok & ~(int64_t) 15) + 8 * gg + s;
}

// Epilogue of 4 consecutive features n..n+3 of row m (values t[] = raw accumulators).
template <int EPI>
__device__ __forceinline__ void epi4(const kargs & a, int64_t m, int64_t n, float t[4]) {
    const gemm_epi & ep = a.ep;
    if (a.bias) {
        const float4 b = *(const float4 *) (a.bias + n);
        t[0] = __fadd_rn(t[0], b.x); t[1] = __fadd_rn(t[1], b.y); t[2] = __fadd_rn(t[2], b.z); t[3] = __fadd_rn(t[3], b.w);
    }
    if constexpr (EPI == EPI_F32) {
        if (ep.addvec) {
            const float4 v = *(const float4 *) (ep.addvec + n);
            t[0] = __fadd_rn(t[0], v.x); t[1] = __fadd_rn(t[1], v.y); t[2] = __fadd_rn(t[2], v.z); t[3] = __fadd_rn(t[3], v.w);
        }
        const int64_t item = m / ep.rin, r = m - item * ep.rin;
        const int64_t row = item * ep.rout + ep.pre + r;
        if (ep.addrows) {
            const float4 v = *(const float4 *) (ep.addrows + (ep.pre + r) * ep.ldy + n);
            t[0] = __fadd_rn(t[0], v.x); t[1] = __fadd_rn(t[1], v.y); t[2] = __fadd_rn(t[2], v.z); t[3] = __fadd_rn(t[3], v.w);
        }
        *(float4 *) (ep.y + row * ep.ldy + n) = make_float4(t[0], t[1], t[2], t[3]);
    } else if constexpr (EPI == EPI_RESID) {
        if (ep.ls) {
            const float4 v = *(const float4 *) (ep.ls + n);
            t[0] = __fmul_rn(t[0], v.x); t[1] = __fmul_rn(t[1], v.y); t[2] = __fmul_rn(t[2], v.z); t[3] = __fmul_rn(t[3], v.w);
        }
        float4 * px = (float4 *) (ep.y + m * ep.ldy + n);
        float4 x = *px;
        x.x = __fadd_rn(x.x, t[0]); x.y = __fadd_rn(x.y, t[1]); x.z = __fadd_rn(x.z, t[2]); x.w = __fadd_rn(x.w, t[3]);
        *px = x;
    } else if constexpr (EPI == EPI_GELU_F32) {
        *(float4 *) (ep.y + m * ep.ldy + n) = make_float4(gelu_erf(t[0]), gelu_erf(t[1]), gelu_erf(t[2]), gelu_erf(t[3]));
    } else if constexpr (EPI == EPI_GELU_F16) {
        _Float16 * o = (_Float16 *) ep.oh + m * ep.ldy + n;
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        h4 v = {(_Float16) gelu_erf(t[0]), (_Float16) gelu_erf(t[1]), (_Float16) gelu_erf(t[2]), (_Float16) gelu_erf(t[3])};
        *(h4 *) o = v;
    } else if constexpr (EPI == EPI_QKV) {
        const int D = ep.D, hd = ep.hd, hds = ep.hds ? ep.hds : hd;
        const int64_t ng = n + ep.col0;        // column of the [q | k | v] layout (the bias above is this launch's)
        const int which = (int) (ng / D);
        const int nn = (int) (ng - (int64_t) which * D);
        const int h = nn / hd, d0 = nn - h * hd;
        const int64_t item = m / ep.R, tok = m - item * ep.R;
        const int64_t head = item * ep.n_head + h;
        if (which < 2) {
            float o[4];
            if (ep.rope_c) {
                // out = x*C + swap(x)*S' (reference src/rope3d.cpp:136-164): two products, one add
                const float4 c = *(const float4 *) (ep.rope_c + tok * hd + d0);
                const float4 s = *(const float4 *) (ep.rope_s + tok * hd + d0);
                o[0] = __fadd_rn(__fmul_rn(t[0], c.x), __fmul_rn(t[1], s.x));
                o[1] = __fadd_rn(__fmul_rn(t[1], c.y), __fmul_rn(t[0], s.y));
                o[2] = __fadd_rn(__fmul_rn(t[2], c.z), __fmul_rn(t[3], s.z));
                o[3] = __fadd_rn(__fmul_rn(t[3], c.w), __fmul_rn(t[2], s.w));
            } else {
                o[0] = t[0]; o[1] = t[1]; o[2] = t[2]; o[3] = t[3];
            }
            typedef _Float16 h4 __attribute__((ext_vector_type(4)));
            h4 v = {(_Float16) o[0], (_Float16) o[1], (_Float16) o[2], (_Float16) o[3]};
            _Float16 * dst = (_Float16 *) (which == 0 ? ep.q : ep.k) + (head * ep.R_pad + tok) * hds + d0;
            *(h4 *) dst = v;
        } else {
            _Float16 * vt = (_Float16 *) ep.vt + head * hds * ep.R_pad;
            const int p = perm16(tok);
            for (int e = 0; e < 4; e++) vt[(int64_t) (d0 + e) * ep.R_pad + p] = (_Float16) t[e];
        }
    }
}

}  // namespace
