// The activations that products may apply to their sums before they store them, and that the
// element-wise kernels apply: one definition for a type of result, so that all of them round alike.
#pragma once

#include "common.h"

namespace lc {

// ACT_SIGMOID_GATE: times sigmoid of the gate's entry at the output's place; ACT_SIGMOID_GROUP_GATE: times
// sigmoid of ONE gate entry per row and group (a number per token and head)
enum : int { ACT_NONE = 0, ACT_GELU_TANH = 1, ACT_RELU_SQUARED = 2, ACT_SIGMOID_GATE = 3, ACT_SIGMOID_GROUP_GATE = 4,
             ACT_XIELU = 5, ACT_GELU_ERF = 6 };

// The tanh form, z (1 + tanh y) / 2 with y = sqrt(2/pi) (z + 0.044715 z^3), for results of type T.  Those that are rounded to bfloat16 take
// (1 + tanh y) / 2 = 1 / (1 + e^-2y), which loses nothing where tanh is next to -1, with the hardware's exp and reciprocal: the rounding of
// exp's argument makes the relative error grow with |y|, to some 2^-17 at y = -44, where results leave the range of normal numbers; half a
// unit of bfloat16 is 2^-9.
template <typename T>
__device__ __forceinline__ float gelu_tanh(float z) {
    const float inner = 0.7978845608028654f * fmaf(0.044715f * z, z * z, z);
    if constexpr (sizeof(T) == 2) return z * __builtin_amdgcn_rcpf(1.f + __expf(-2.f * inner));
    else return 0.5f * z * (1.f + tanhf(inner));
}

// z Phi(z), Phi the normal distribution, for results of type T.  Those that are rounded to bfloat16 take Phi(-|z|) = erfc(a) / 2, a = |z| / sqrt 2, with
// erfc(a) = e^(-a^2) t P(t), t = 1 / (1 + 0.3 a), P the polynomial of degree 8 whose largest relative error over all a is least
// (1.9e-8; found by reweighted least squares against erfcx): no branches, and nothing cancels where erf is next to -1.  In float32, against 64
// bits: relative to the result 6e-7 at most for |z| < 1 (erff 2e-7), 1.5e-6 down to -5 (erff 5e-2) and 7e-6 beyond; half a unit of bfloat16
// is 2e-3.  6,092 rows by 2,048 in a product's epilogue: 20 us with erff, 5 now (the whole product 99.9 and 80.7).
template <typename T>
__device__ __forceinline__ float gelu_erf(float z) {
    if constexpr (sizeof(T) == 2) {
        const float t = __builtin_amdgcn_rcpf(fmaf(0.3f * 0.70710678f, fabsf(z), 1.f));
        float p = -0.12943172f;
        p = fmaf(p, t, 0.48508397f);
        p = fmaf(p, t, -0.51119810f);
        p = fmaf(p, t, 0.54635904f);
        p = fmaf(p, t, -0.09360332f);
        p = fmaf(p, t, 0.21442275f);
        p = fmaf(p, t, 0.14848642f);
        p = fmaf(p, t, 0.17069128f);
        p = fmaf(p, t, 0.16918966f);
        const float below = 0.5f * p * t * __builtin_amdgcn_exp2f(-0.72134752f * z * z);        // Phi(-|z|)
        return z * (z < 0.f ? below : 1.f - below);
    } else {
        return 0.5f * z * (1.f + erff(z * 0.7071067811865476f));
    }
}

// T: the type of the result
template <typename T>
__device__ __forceinline__ float activate(float z, int kind) {
    if (kind == ACT_GELU_TANH) return gelu_tanh<T>(z);
    if (kind == ACT_GELU_ERF) return gelu_erf<T>(z);
    if (kind == ACT_RELU_SQUARED) {
        const float r = fmaxf(z, 0.f);
        return r * r;
    }
    return z;
}

__device__ __forceinline__ float sigmoid(float z) { return 1.f / (1.f + expf(-z)); }

// xIELU with its two numbers already through softplus: z > 0: a z^2 + z/2;  z <= 0: b (e^z - 1 - z) + z/2
// (a = softplus(p), b = 1/2 + softplus(q)).
__device__ __forceinline__ float xielu(float z, float a, float b) {
    if (z > 0.f) return fmaf(a * z, z, 0.5f * z);
    return fmaf(b, expm1f(z) - z, 0.5f * z);
}

}  // namespace lc
