// gemm_f32.hip - f32 weights x f32 activations (the patch embedding of the image families, f32 files) on
// gfx950's f32 matrix instruction, and the split of f32 QKV rows into the attention operands.
#include "common.h"
#include "gemm_dev.h"
#include "kernels.h"
#include "model.h"

typedef float f16v __attribute__((ext_vector_type(16)));

#define MFMA_F32(a, b, c) __builtin_amdgcn_mfma_f32_32x32x2f32((a), (b), (c), 0, 0, 0)

namespace {

// One workgroup computes a tile of 32 features x 32 tokens; its F32_KS waves each sum one slice of K and
// meet in LDS, in slice order. The slices depend on K alone, so an output's rounding does not depend on
// how many rows share the launch. Small launches are what this is for (one ViT-S/16 image is 196 x 384
// outputs: 84 tiles, 672 waves), and a large one only has more tiles.
//
// v_mfma_f32_32x32x2_f32 runs at the VALU's fma rate (16 lanes' worth per cycle and SIMD: 64 cycles for
// 32 x 32 x 2), so the gain over VALU fmas is in the operands: a lane needs one float of a weight row and
// one of a token row per 16 outputs, where 2 x 4 outputs per lane took six 16-byte LDS reads per 32
// fmas. Operands go from global memory straight to registers, 16 bytes per lane (lane group g holds
// columns 8 j + 4 g .. + 3 of its row for step j; the MFMA pairs columns e and 4 + e), one pair of steps
// ahead; the lines a load leaves half read are finished by the next one out of L1. Each of the four MFMAs
// of a step has its own accumulator: no chain from one to the next, and sums of K / 32 terms.
// Measured against 16 x 32 tiles of VALU fmas (us per launch, tokens x features x K): 196 x 384 x 768 11.4 -> 9.5,
// 256 x 1280 x 588 27.8 -> 13.8, 1024 x 1280 x 588 88.5 -> 36.8 (42 TFLOP/s; the fma rate alone would take 10:
// half-used lines and 32 rows per load bound it), 2048 x 1024 x 1024 218 -> 75.7, one row of 384 x 384 7.2 -> 5.6;
// relative error against 64 bits 1.46e-7 -> 1.12e-7 at K = 768, 1.36e-7 (K = 584) -> 1.05e-7 (588): 32 partial sums
// per output instead of 16. The sums' order is another one than the fmas', so f32 results differ in their last bits
// from that kernel's.
constexpr int F32_KS = 8;

template <int EPI>
__global__ __launch_bounds__(64 * F32_KS) void k_gemm_f32(kargs a) {
    __shared__ __attribute__((aligned(16))) float4 part[F32_KS][4][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, g = lane >> 5;
    const int64_t n0 = (int64_t) blockIdx.x * 32, m0 = (int64_t) blockIdx.y * 32;
    // rows past the end read the last row; their results are dropped
    const int64_t rw = n0 + l32 < a.N ? n0 + l32 : a.N - 1, rx = m0 + l32 < a.M ? m0 + l32 : a.M - 1;
    const float * W = (const float *) a.A + rw * a.K;
    const float * X = (const float *) a.B + rx * a.K;
    const bool al = (a.K & 3) == 0 && (((uintptr_t) a.A | (uintptr_t) a.B) & 15) == 0;   // rows 16-byte aligned
    const int K = (int) a.K;
    // four columns of a row from k; columns past K are zero
    auto ld4 = [&](const float * row, int k) {
        if (al && k + 4 <= K) return *(const float4 *) (row + k);
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (k < K) v.x = row[k];
        if (k + 1 < K) v.y = row[k + 1];
        if (k + 2 < K) v.z = row[k + 2];
        if (k + 3 < K) v.w = row[k + 3];
        return v;
    };
    // this wave's chunks of 16 columns
    const int nch = (K + 15) / 16, c0 = nch * wave / F32_KS, c1 = nch * (wave + 1) / F32_KS;
    f16v acc[4];
#pragma unroll
    for (int e = 0; e < 4; e++) acc[e] = f16v{};
    float4 w[2], x[2];
    auto load = [&](int c, float4 (&wv)[2], float4 (&xv)[2]) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            wv[j] = ld4(W, 16 * c + 8 * j + 4 * g);
            xv[j] = ld4(X, 16 * c + 8 * j + 4 * g);
        }
    };
    if (c0 < c1) load(c0, w, x);
    for (int c = c0; c < c1; c++) {
        float4 wn[2] = {w[0], w[1]}, xn[2] = {x[0], x[1]};
        if (c + 1 < c1) load(c + 1, wn, xn);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            acc[0] = MFMA_F32(w[j].x, x[j].x, acc[0]);
            acc[1] = MFMA_F32(w[j].y, x[j].y, acc[1]);
            acc[2] = MFMA_F32(w[j].z, x[j].z, acc[2]);
            acc[3] = MFMA_F32(w[j].w, x[j].w, acc[3]);
        }
#pragma unroll
        for (int j = 0; j < 2; j++) { w[j] = wn[j]; x[j] = xn[j]; }
    }
    float t[16];
#pragma unroll
    for (int r = 0; r < 16; r++) t[r] = __fadd_rn(__fadd_rn(acc[0][r], acc[1][r]), __fadd_rn(acc[2][r], acc[3][r]));
#pragma unroll
    for (int q = 0; q < 4; q++) part[wave][q][lane] = make_float4(t[4 * q], t[4 * q + 1], t[4 * q + 2], t[4 * q + 3]);
    __syncthreads();
    // wave q < 4 adds the slices of feature group q (features 8 q + 4 g .. + 3 of each token) in order
    if (wave >= 4) return;
    float4 v = part[0][wave][lane];
#pragma unroll
    for (int k = 1; k < F32_KS; k++) {
        const float4 p = part[k][wave][lane];
        v.x = __fadd_rn(v.x, p.x); v.y = __fadd_rn(v.y, p.y); v.z = __fadd_rn(v.z, p.z); v.w = __fadd_rn(v.w, p.w);
    }
    const int64_t m = m0 + l32, n = n0 + 8 * wave + 4 * g;
    float o[4] = {v.x, v.y, v.z, v.w};
    if (m < a.M && n < a.N) epi4<EPI>(a, m, n, o);
}

// f32 fused-qkv rows -> Q, K (RoPE'd) and V^T through the same epilogue the QKV GEMM runs
__global__ void k_qkv_split(kargs a, const float * __restrict__ qkv) {
    const int64_t id = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t groups = a.N / 4;
    if (id >= a.M * groups) return;
    const int64_t m = id / groups, n = (id % groups) * 4;
    const float4 v = *(const float4 *) (qkv + m * a.N + n);
    float t[4] = {v.x, v.y, v.z, v.w};
    epi4<EPI_QKV>(a, m, n, t);
}

}  // namespace

void launch_gemm_f32(const dev_linear & W, const act_view & X, int64_t M, const gemm_epi & ep, hipStream_t s) {
    kargs a{};
    a.A = (const _Float16 *) W.w;
    a.B = (const _Float16 *) X.q;
    a.bias = W.bias;
    a.M = M; a.N = W.n_out; a.K = W.n_in;
    a.ep = ep;
    const dim3 grid((unsigned) ((a.N + 31) / 32), (unsigned) ((M + 31) / 32));
    switch (ep.kind) {
        case EPI_F32:      k_gemm_f32<EPI_F32><<<grid, 64 * F32_KS, 0, s>>>(a); break;
        case EPI_RESID:    k_gemm_f32<EPI_RESID><<<grid, 64 * F32_KS, 0, s>>>(a); break;
        case EPI_GELU_F32: k_gemm_f32<EPI_GELU_F32><<<grid, 64 * F32_KS, 0, s>>>(a); break;
        case EPI_QKV:      k_gemm_f32<EPI_QKV><<<grid, 64 * F32_KS, 0, s>>>(a); break;
        default: jepa_log("jepa: internal error: epilogue %d has no f32 GEMM\n", ep.kind); break;
    }
}

void launch_qkv_split(const float * qkv, int64_t M, int64_t N, const gemm_epi & ep, hipStream_t s) {
    kargs a{};
    a.M = M; a.N = N; a.K = 0;
    a.ep = ep;
    const int64_t total = M * (N / 4);
    if (total > 0) k_qkv_split<<<(unsigned) ((total + 255) / 256), 256, 0, s>>>(a, qkv);
}
