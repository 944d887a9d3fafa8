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

// z Phi(z), Phi the normal distribution, for results of type T.  Those that are rounded to bfloat16 take z Phi(-|z|), and z less |z| Phi(-|z|) above
// zero, with 2 Phi(-|z|) = 2^-(|z| (|z| / (2 ln 2) + t S(s))), t = 1 / (1 + 0.13 |z|), s = |z| t, S of degree 8 (reweighted least squares
// against erfcx: 1e-8 of Phi for |z| < 0.5, 2e-7 at 8): no branches, nothing cancels where erf is next to -1, and errors of t and s vanish with |z|.
// Largest error in float32 against 64 bits, relative to the result, in units of 10^-7, with erff and so: z in [0, 1) 1.4 and 1.2, beyond 1.4 and
// 0.9; [-0.5, 0) 1.5 and 1.9, [-1, -0.5) 2.6 and 2.3, [-1.5, -1) 6.2 and 3.8, [-2, -1.5) 12 and 4.9, [-2.5, -2) 30 and 6.4, [-4, -3) 4,700 and
// 9.7, beyond -5.6 all of it and 17 to 75; half a unit of bfloat16 is 20,000.  6,092 experts' rows by 2,048, K of 2,048, us: 94 with erff, 84 so, 70
// without an activation.
template <typename T>
__device__ __forceinline__ float gelu_erf(float z) {
    if constexpr (sizeof(T) == 2) {
        const float x = fminf(fabsf(z), 20.f);
        const float t = __builtin_amdgcn_rcpf(fmaf(0.13f, x, 1.f)), s = x * t;
        float q = 2.06598898e-07f;
        q = fmaf(q, s, -4.06970366e-06f);
        q = fmaf(q, s, 3.20552572e-05f);
        q = fmaf(q, s, -8.63060122e-05f);
        q = fmaf(q, s, -0.000308247458f);
        q = fmaf(q, s, 0.00281040324f);
        q = fmaf(q, s, 0.00370200677f);
        q = fmaf(q, s, -0.112473339f);
        q = fmaf(q, s, 1.1511035f);
        const bool far = x > 12.f;              // the hardware's exp2 has no numbers below the normal ones: times 2^64 there
        const float twice = __builtin_amdgcn_exp2f(fmaf(-x, fmaf(0.72134752f, x, q * t), far ? 64.f : 0.f));
        return fmaf((far ? -0x1p-65f : -0.5f) * x, twice, z < 0.f ? 0.f * z : z);            // (0 z: NaN for -inf, as of a product with 0)
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
