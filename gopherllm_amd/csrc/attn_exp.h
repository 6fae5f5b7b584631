// attn_exp.h -- fastExpF32, the exponential of the attention weights.
#pragma once
#include "gllm_common.h"

namespace gllm {

// fastExpF32 (fastmath.go:47-77), operation for operation, without
// branches: the two range checks select the result, so a thread's several
// exps interleave instead of running one exec-masked block after another.
// Inside the range |t| < 128, so the clamp only keeps the int conversion
// defined for inputs the selects discard (a NaN still gives NaN).  The
// empty asm keeps the compiler from turning the first select back into a
// branch around the polynomial.
__device__ __forceinline__ float fast_exp(float x) {
    const float t = x * 1.44269502f;  // float32(1.4426950408889634)
    const float tc = fminf(fmaxf(t, -256.0f), 256.0f);
    const int k = (int)(tc + (tc >= 0.0f ? 0.5f : -0.5f));
    const float r = (float)((double)x - (double)k * 0.6931471805599453);
    const float p = 1.0f + r * (1.0f + r * (0.5f + r * ((float)(1.0 / 6) +
                    r * ((float)(1.0 / 24) + r * ((float)(1.0 / 120) + r * (float)(1.0 / 720))))));
    float v = p * __uint_as_float((uint32_t)(127 + k) << 23);
    asm volatile("" : "+v"(v));  // computed unconditionally: the selects stay selects
    return x > 88.02969f ? __int_as_float(0x7f800000) : x < -87.33654f ? 0.0f : v;
}

// fast_exp of N independent values, step by step across all of them so
// their dependent chains interleave (one wave per SIMD hides no latency
// otherwise); each value sees exactly fast_exp's operations.
template <int N>
__device__ __forceinline__ void fast_exp_n(const float (&x)[N], float (&y)[N]) {
    int k[N];
    float r[N];
#pragma unroll
    for (int i = 0; i < N; i++) {
        const float t = x[i] * 1.44269502f;
        const float tc = fminf(fmaxf(t, -256.0f), 256.0f);
        k[i] = (int)(tc + (tc >= 0.0f ? 0.5f : -0.5f));
    }
#pragma unroll
    for (int i = 0; i < N; i++) r[i] = (float)((double)x[i] - (double)k[i] * 0.6931471805599453);
#pragma unroll
    for (int i = 0; i < N; i++) {
        const float p = 1.0f + r[i] * (1.0f + r[i] * (0.5f + r[i] * ((float)(1.0 / 6) +
                        r[i] * ((float)(1.0 / 24) + r[i] * ((float)(1.0 / 120) + r[i] * (float)(1.0 / 720))))));
        y[i] = p * __uint_as_float((uint32_t)(127 + k[i]) << 23);
    }
#pragma unroll
    for (int i = 0; i < N; i++) asm volatile("" : "+v"(y[i]));
#pragma unroll
    for (int i = 0; i < N; i++)
        y[i] = x[i] > 88.02969f ? __int_as_float(0x7f800000) : x[i] < -87.33654f ? 0.0f : y[i];
}

}  // namespace gllm
