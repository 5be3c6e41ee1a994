// Register math of the Tria 3x3 carriers, shared by the Tria kernels and the
// fused decode FFN epilogue.  Row-major 3x3 matrices, fp32.
#pragma once

#include "loom_common.h"

namespace loom {

// tanh(y) for |y| <= sqrt(3) as y N(y^2) / D(y^2), fitted to a relative error
// of 5e-9 there (least squares on the relative error over Chebyshev points);
// with rounding and v_rcp_f32 (1 ulp) it stays within 3.3e-7 relative (every float
// of 2^-31 .. sqrt(3) and the reciprocal's two neighbours).  Fourteen
// operations without a branch, where libm's tanhf with the IEEE square root and
// division around it took most of the element-wise kernels' VALU work; the
// form 1 - 2 / (1 + e^2y) loses the low bits of small y.
__device__ __forceinline__ float tanh_unit(float y) {
    const float z = y * y;
    const float n = fmaf(z, fmaf(z, 0.0019643290f, 0.1206163f), 1.0f);
    const float d = fmaf(z, fmaf(z, fmaf(z, 9.0792593e-5f, 0.019947553f), 0.45394963f), 1.0f);
    return y * n * __builtin_amdgcn_rcpf(d);
}

// The carrier's rows from (a, b, c); the axis is a compile-time parameter: the
// kernels are instantiated per axis.
template <int AXIS>
__device__ __forceinline__ void carrier_rows(float a, float b, float c, float mt[9]) {
    if constexpr (AXIS == 0) {          // about z
        mt[0] = -c;   mt[1] = -1.0f; mt[2] = b;
        mt[3] = 1.0f; mt[4] = -c;    mt[5] = -a;
        mt[6] = a;    mt[7] = b;     mt[8] = 1.0f;
    } else if constexpr (AXIS == 1) {   // about x
        mt[0] = 1.0f; mt[1] = b;     mt[2] = c;
        mt[3] = c;    mt[4] = -a;    mt[5] = -1.0f;
        mt[6] = -b;   mt[7] = 1.0f;  mt[8] = -a;
    } else {                  // about y
        mt[0] = -b;   mt[1] = -c;    mt[2] = 1.0f;
        mt[3] = a;    mt[4] = 1.0f;  mt[5] = c;
        mt[6] = -1.0f; mt[7] = a;    mt[8] = -b;
    }
}

// Local carrier T(r,i,o) = (I + K(a,b,c)) @ R_axis,
// (a,b,c) = alpha * tanh(x / sqrt(mean(x^2) + eps)), x = (ri, ro, io).
// 1/sqrt is v_rsq_f32 (1 ulp), so |y| <= sqrt(3) and tanh is tanh_unit.  A step's rms
// error against 64 bits, in fp32, with this carrier and rms9_inv (with libm's tanh,
// root and division): alpha 0.0375 5.6e-8 (6.1e-8), 0.3 5.8e-8 (6.4e-8), 0.5 6.0e-8
// (6.2e-8), 0.7 6.5e-8 (6.4e-8), 1 6.7e-8 (6.3e-8); a refined reciprocal and root take
// 2% off the last and 3-5% more time.
template <int AXIS>
__device__ __forceinline__ void carrier9(float r, float i, float o, float alpha, float mt[9]) {
    const float x0 = r * i, x1 = r * o, x2 = i * o;
    const float inv = __builtin_amdgcn_rsqf(
        fmaf(fmaf(x0, x0, fmaf(x1, x1, x2 * x2)), 1.0f / 3.0f, 1e-6f));
    carrier_rows<AXIS>(alpha * tanh_unit(x0 * inv), alpha * tanh_unit(x1 * inv),
                       alpha * tanh_unit(x2 * inv), mt);
}

// carrier9 with tanh(y) = 1 - 2/(1 + 2^(2 y log2 e)) on v_exp_f32 and v_rcp_f32
// (1 ulp each), for the streaming chains, which the vector ALU bounds (the
// other form there: 5.63 ms against 4.93 at 24 layers of 8 x 4096 x 3072).  |y| <= sqrt(3),
// so the exponential stays in range and the absolute error of alpha*tanh is a
// few ulp of alpha.
template <int AXIS>
__device__ __forceinline__ void carrier9_fast(float r, float i, float o, float alpha,
                                              float mt[9]) {
    const float x0 = r * i, x1 = r * o, x2 = i * o;
    const float inv = __builtin_amdgcn_rsqf(
        fmaf(fmaf(x0, x0, fmaf(x1, x1, x2 * x2)), 1.0f / 3.0f, 1e-6f));
    const float k = 2.0f * 1.4426950408889634f * inv;   // 2 log2(e) / rms
    const float m2a = -2.0f * alpha;
    const float a = fmaf(m2a, __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x0 * k)), alpha);
    const float b = fmaf(m2a, __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x1 * k)), alpha);
    const float c = fmaf(m2a, __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x2 * k)), alpha);
    carrier_rows<AXIS>(a, b, c, mt);
}

// mean of the squares of 9 entries plus eps
__device__ __forceinline__ float ms9(const float v[9]) {
    float s = v[0] * v[0];
#pragma unroll
    for (int k = 1; k < 9; ++k) s = fmaf(v[k], v[k], s);
    return fmaf(s, 1.0f / 9.0f, 1e-6f);
}
// 1 / sqrt(x) for x > 0: v_rsq_f32 and one Newton step, which leaves the error
// of the correctly rounded root and division at a fifth of their operations.
// x = inf gives 0: the step's 0 * inf is replaced by -1 there, times 0.
__device__ __forceinline__ float rsq_step(float x) {
    const float y = __builtin_amdgcn_rsqf(x);
    const float e = fmaxf(fmaf(-x * y, y, 1.0f), -1.0f);
    return fmaf(0.5f * y, e, y);
}
__device__ __forceinline__ float rms9_inv(const float v[9]) { return rsq_step(ms9(v)); }
// the same with v_rsq_f32 alone (1 ulp), for the streaming chains
__device__ __forceinline__ float rms9_inv_fast(const float v[9]) { return __builtin_amdgcn_rsqf(ms9(v)); }

// out = A @ B for row-major 3x3
__device__ __forceinline__ void mm3(const float A[9], const float B[9], float out[9]) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c)
            out[3 * r + c] = fmaf(A[3 * r + 2], B[6 + c], fmaf(A[3 * r + 1], B[3 + c], A[3 * r] * B[c]));
}

// M <- M (I - beta/2 (G/s - I)), G = M^T M, s = max(mean(diag G), eps)
// (PolARM, tria.py:128-139), in place.
__device__ __forceinline__ void polarm9(float M[9], float beta, float eps) {
    float G[9];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c)
            G[3 * r + c] = fmaf(M[6 + r], M[6 + c], fmaf(M[3 + r], M[3 + c], M[r] * M[c]));
    const float s = fmaxf((G[0] + G[4] + G[8]) * (1.0f / 3.0f), eps);
    float C[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        const float id = (k == 0 || k == 4 || k == 8) ? 1.0f : 0.0f;
        C[k] = id - 0.5f * beta * (G[k] / s - id);
    }
    float R[9];
    mm3(M, C, R);
#pragma unroll
    for (int k = 0; k < 9; ++k) M[k] = R[k];
}

// v <- v / rms(v)
__device__ __forceinline__ void normalize9(float v[9]) {
    const float inv = rms9_inv(v);
#pragma unroll
    for (int k = 0; k < 9; ++k) v[k] *= inv;
}

}  // namespace loom
