// gemv_q8.hip - q8_0 weights times one row (the one-token linears of the attentive-pool head).
//
// A tile GEMM gives such a linear N / 64 workgroups, each running K / 128 barriered stages over 63 rows of
// padding, and only those few CUs read the weights: 4096 -> 1024 took 25.8 us for 4.5 MB. Here a thread
// takes whole 32-blocks of a weight row (one 32-byte load, eight v_dot4), N / 8 workgroups read the
// weights at once, and only the fma chain over the blocks is serial: block sums and scale products meet in
// LDS, where one lane per feature adds them in K order, with the roundings of the tile kernel (the
// result is the same bits). us per launch: 4096 -> 1024 25.8 -> 5.3, 1024 -> 4096 with GELU and quantization
// 10.7 -> 4.9, 1024 -> 1024 9.4 -> 5.0 (a kernel that does nothing takes about 2.5; 4.5 MB at the copy rate 1).
#include "kernels.h"
#include "model.h"
#include "gemm_dev.h"
#include "quant_dev.h"

namespace {

template <int EPI, int NF>
__global__ __launch_bounds__(256) void k_gemv_q8(kargs a) {
    extern __shared__ __attribute__((aligned(16))) float2 part[];   // [NF][KB + 1]: block sum, scale product
    const int tid = threadIdx.x, KB = (int) (a.K / 32);
    const int64_t n0 = (int64_t) blockIdx.x * NF;
    const uint16_t * bd = (const uint16_t *) a.Bd;
#pragma unroll 4
    for (int i = tid; i < NF * KB; i += 256) {
        const int f = i / KB, b = i - f * KB;
        const uint4 * w = (const uint4 *) ((const int8_t *) a.A + (n0 + f) * a.K + 32 * b);
        const uint4 * x = (const uint4 *) ((const int8_t *) a.B + 32 * b);
        const uint4 w0 = w[0], w1 = w[1], x0 = x[0], x1 = x[1];
        int s = __builtin_amdgcn_sdot4((int) w0.x, (int) x0.x, 0, false);
        s = __builtin_amdgcn_sdot4((int) w0.y, (int) x0.y, s, false);
        s = __builtin_amdgcn_sdot4((int) w0.z, (int) x0.z, s, false);
        s = __builtin_amdgcn_sdot4((int) w0.w, (int) x0.w, s, false);
        s = __builtin_amdgcn_sdot4((int) w1.x, (int) x1.x, s, false);
        s = __builtin_amdgcn_sdot4((int) w1.y, (int) x1.y, s, false);
        s = __builtin_amdgcn_sdot4((int) w1.z, (int) x1.z, s, false);
        s = __builtin_amdgcn_sdot4((int) w1.w, (int) x1.w, s, false);
        const float dw = (float) __builtin_bit_cast(_Float16, a.Ad[(n0 + f) * KB + b]), da = (float) __builtin_bit_cast(_Float16, bd[b]);
        part[f * (KB + 1) + b] = make_float2((float) s, __fmul_rn(dw, da));   // both exact
    }
    __syncthreads();
    if (tid >= NF) return;
    const float2 * p = part + tid * (KB + 1);
    float v = 0.0f;
#pragma unroll 8
    for (int b = 0; b < KB; b++) v = fmaf(p[b].x, p[b].y, v);
    const int64_t n = n0 + tid;
    const gemm_epi & ep = a.ep;
    if (a.bias) v = __fadd_rn(v, a.bias[n]);
    if constexpr (EPI == EPI_F32) {
        if (ep.addvec) v = __fadd_rn(v, ep.addvec[n]);
        if (ep.addrows) v = __fadd_rn(v, ep.addrows[ep.pre * ep.ldy + n]);
        ep.y[ep.pre * ep.ldy + n] = v;
    } else if constexpr (EPI == EPI_RESID) {
        if (ep.ls) v = __fmul_rn(v, ep.ls[n]);
        ep.y[n] = __fadd_rn(ep.y[n], v);
    } else {
        // 32 lanes hold one q8_0 block of the next linear's input
        static_assert(EPI == EPI_GELU_Q8_0 && NF == 32, "one block per workgroup");
        v = gelu_erf(v);
        float am = fabsf(v);
#pragma unroll
        for (int m = 16; m > 0; m >>= 1) am = fmaxf(am, __shfl_xor(am, m, 32));
        const float d = am / 127.0f, id = am != 0.0f ? 127.0f / am : 0.0f;
        ((uint8_t *) ep.oq)[n] = (uint8_t) q8_byte(v, id);
        if (tid == 0) ((uint16_t *) ep.od)[n / 32] = __builtin_bit_cast(uint16_t, (_Float16) d);
    }
}

}  // namespace

bool launch_gemv_q8(const dev_linear & W, const act_view & X, const gemm_epi & ep, hipStream_t s) {
    const int nf = ep.kind == EPI_GELU_Q8_0 ? 32 : 8;
    const size_t lds = (size_t) nf * (W.n_in / 32 + 1) * sizeof(float2);
    if (W.fmt != W_Q32 || W.n_out % nf || W.n_in % 32 || lds > 48 * 1024) return false;
    kargs a{};
    a.A = (const _Float16 *) W.w;
    a.Ad = (const uint16_t *) W.wd;
    a.B = (const _Float16 *) X.q;
    a.Bd = X.d;
    a.bias = W.bias;
    a.M = 1; a.N = W.n_out; a.K = W.n_in;
    a.ep = ep;
    const unsigned grid = (unsigned) (W.n_out / nf);
    switch (ep.kind) {
        case EPI_F32:       k_gemv_q8<EPI_F32, 8><<<grid, 256, lds, s>>>(a); return true;
        case EPI_RESID:     k_gemv_q8<EPI_RESID, 8><<<grid, 256, lds, s>>>(a); return true;
        case EPI_GELU_Q8_0: k_gemv_q8<EPI_GELU_Q8_0, 32><<<grid, 256, lds, s>>>(a); return true;
        default: return false;
    }
}
