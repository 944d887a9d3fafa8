// A short causal convolution over time on one channel of a step's float32 projections, shared by the
// mixers that run their projections through one (attention with convolved q/k/v, the state-space
// mixer): y_t = sum_j taps[c, j] x_(t - K + 1 + j), the last column of the taps being the current
// token's.  Inputs from before the step come from the request's tail: its last K - 1 inputs, oldest
// first, [K - 1, C] per state slot, zeros at a sequence's start.
#pragma once

#include "common.h"

namespace lc {

constexpr int SHORT_CONV_MAX_TAPS = 16;

// Channel c (column c of proj) of token t, the `local`-th token of its request in this step.
// proj [T, cols]; taps [C, K]; tail [K - 1, C] of the request's slot.
__device__ __forceinline__ float short_conv(const float* __restrict__ proj, size_t cols, int t, int local, int c,
                                            const float* __restrict__ taps, int K,
                                            const float* __restrict__ tail, int C) {
    float y = 0.f;
    for (int back = K - 1; back >= 0; --back) {       // oldest input first: the order of the sum is fixed
        const float x = back <= local ? proj[(size_t)(t - back) * cols + c]
                                      : tail[(size_t)((K - 1) - (back - local)) * C + c];
        y = fmaf(taps[(size_t)c * K + (K - 1 - back)], x, y);
    }
    return y;
}

// The same for tokens that follow one another: a thread keeps its channel's taps and last inputs, so that each input is read once and
// not once a tap.  KT: the number of taps, or 0 where it is known at run time alone (then every token reads all of its inputs).  The
// sums are short_conv's, to the bit.
template <int KT>
struct ShortConvRun {
    float w[KT > 0 ? KT : 1], in[KT > 0 ? KT : 1];      // the taps; the inputs up to the token, the oldest first

    __device__ __forceinline__ void start(const float* __restrict__ taps, int c) {
#pragma unroll
        for (int j = 0; j < KT; ++j) w[j] = taps[(size_t)c * KT + j];
    }

    // fresh: the token before was not this request's, or not this thread's
    __device__ __forceinline__ float at(const float* __restrict__ proj, size_t cols, int t, int local, int c, const float* __restrict__ taps,
                                        int K, const float* __restrict__ tail, int C, bool fresh) {
        if constexpr (KT == 0) {
            return short_conv(proj, cols, t, local, c, taps, K, tail, C);
        } else {
#pragma unroll
            for (int j = 0; j < KT - 1; ++j) {
                if (fresh) {
                    const int back = KT - 1 - j;
                    in[j] = back <= local ? proj[(size_t)(t - back) * cols + c] : tail[(size_t)((KT - 1) - (back - local)) * C + c];
                } else {
                    in[j] = in[j + 1];
                }
            }
            in[KT - 1] = proj[(size_t)t * cols + c];
            float y = 0.f;
#pragma unroll
            for (int j = 0; j < KT; ++j) y = fmaf(w[j], in[j], y);
            return y;
        }
    }
};

}  // namespace lc
