// The state-space mixer (Mamba-2's recurrence) around the framework's recurrence kernel.  Per head h of
// group g = h / (heads / groups), with the state S [N, dv] (float32, zeros at a sequence's start):
//   step = softplus(dt_h + dt_bias_h);   S <- exp(-exp(A_log_h) step) S + step B_g x_h^T;   y_h = S^T C_g + D_h x_h
// x, B and C pass a short causal convolution per channel (with a bias) and SiLU first.  That is the
// recurrence S <- diag(decay) S + write v^T, o = S^T read without a removal term, with decay = exp(-exp(A_log)
// step) in every key channel, write = step B, read = C, v = x: this file makes those three vectors a token
// from a step's float32 projections, and the read-out behind the scan:
//   y <- (o + D x) silu(z), divided by its root mean square in `parts` equal parts of the row, times a weight.
// Everything here is float32 arithmetic; only the read-out's result is rounded to the activation type.
#include "common.h"
#include "short_conv.h"

namespace lc {

__device__ __forceinline__ float ss_silu(float z) { return z / (1.f + expf(-z)); }
__device__ __forceinline__ float ss_softplus(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

// A thread per convolved entry and run of `tokens` tokens.  proj [T, cols]: x (heads dv) | B (groups N) | C (groups N) | z (heads dv) | dt
// (heads); the first C = heads dv + 2 groups N columns pass the convolution.  The first x_blocks workgroups of a run take the channels of
// x; the threads of the others a (group, n) pair each, make B and C at n and write them for every head of the group with the head's
// own step and decay, which the workgroup makes once a (token, head) in LDS (KEPT; else, where so many heads do not fit, every thread makes
// those that it needs).  coef [3, T, heads N]; x_out [T, heads dv].
// 2,048 tokens, 16 heads of 128, 4 groups of 128 entries: 83 us with a thread per (token, entry), a 64-bit division, four inputs
// and every head's two exponentials each; 34 us.
template <int KT, bool KEPT>
__global__ __launch_bounds__(256) void state_space_prepare_kernel(
    const float* __restrict__ proj, int cols, int T, int heads, int groups, int N, int dv, const float* __restrict__ taps,
    const float* __restrict__ bias, int K, const float* __restrict__ tails, const float* __restrict__ dt_bias, const float* __restrict__ a_log,
    const int* __restrict__ tok_req, const int* __restrict__ q_offsets, const int* __restrict__ slot_ids, float* __restrict__ coef,
    float* __restrict__ x_out, int tokens, int x_blocks) {
    extern __shared__ float rates[];                // [tokens][heads] steps, then as many decays
    const int inner = heads * dv, C = inner + 2 * groups * N, per_group = heads / groups;
    const int block = blockIdx.y + blockIdx.z * gridDim.y;
    const int t0 = blockIdx.x * tokens, t1 = min(t0 + tokens, T);
    const size_t plane = (size_t)T * heads * N;
    auto tail_of = [&](int r) { return K > 1 ? tails + (size_t)slot_ids[r] * (K - 1) * C : nullptr; };
    if (block < x_blocks) {
        const int i = block * 256 + threadIdx.x;
        if (i >= inner) return;
        ShortConvRun<KT> run;
        run.start(taps, i);
        const float shift = bias[i];
        for (int t = t0, before = -1; t < t1; ++t) {
            const int r = tok_req[t];
            x_out[(size_t)t * inner + i] = ss_silu(run.at(proj, cols, t, t - q_offsets[r], i, taps, K, tail_of(r), C, r != before) + shift);
            before = r;
        }
        return;
    }
    auto step_of = [&](int t, int head) { return ss_softplus(proj[(size_t)t * cols + C + inner + head] + dt_bias[head]); };
    auto decay_of = [&](int head, float step) { return expf(-expf(a_log[head]) * step); };
    if constexpr (KEPT) {
        for (int e = threadIdx.x; e < (t1 - t0) * heads; e += 256) {
            const int head = e % heads;
            const float step = step_of(t0 + e / heads, head);
            rates[e] = step;
            rates[tokens * heads + e] = decay_of(head, step);
        }
        __syncthreads();
    }
    const int i = (block - x_blocks) * 256 + threadIdx.x;
    if (i >= groups * N) return;
    const int g = i / N, n = i % N, cb = inner + i, cc = inner + groups * N + i;
    ShortConvRun<KT> run_b, run_c;
    run_b.start(taps, cb);
    run_c.start(taps, cc);
    const float shift_b = bias[cb], shift_c = bias[cc];
    for (int t = t0, before = -1; t < t1; ++t) {
        const int r = tok_req[t], local = t - q_offsets[r];
        const float* tail = tail_of(r);
        const float b = ss_silu(run_b.at(proj, cols, t, local, cb, taps, K, tail, C, r != before) + shift_b);
        const float c = ss_silu(run_c.at(proj, cols, t, local, cc, taps, K, tail, C, r != before) + shift_c);
        before = r;
        for (int k = 0; k < per_group; ++k) {
            const int head = g * per_group + k, e = (t - t0) * heads + head;
            const size_t at = ((size_t)t * heads + head) * N + n;
            const float step = KEPT ? rates[e] : step_of(t, head);
            coef[at] = KEPT ? rates[tokens * heads + e] : decay_of(head, step);
            coef[plane + at] = step * b;
            coef[2 * plane + at] = c;
        }
    }
}

// One workgroup per token and part of the row.  o, x float32 [T, n]; z float32: columns z_column .. + n of gates
// [T, gate_cols]; skip float32 [heads] (D); weight float32 [n]; the row is normed in `parts` equal parts.
template <typename T>
__global__ void state_space_readout_kernel(const float* __restrict__ o, const float* __restrict__ x,
                                           const float* __restrict__ gates, int gate_cols, int z_column,
                                           const float* __restrict__ skip, int dv, const float* __restrict__ weight,
                                           int parts, float eps, int n, T* __restrict__ out) {
    extern __shared__ float y[];
    __shared__ float scratch[16];
    const size_t t = blockIdx.x;
    const int width = n / parts, first = blockIdx.y * width;
    float ss = 0.f;
    for (int i = threadIdx.x; i < width; i += blockDim.x) {
        const int at = first + i;
        const float v = fmaf(skip[at / dv], x[t * n + at], o[t * n + at]) * ss_silu(gates[t * gate_cols + z_column + at]);
        y[i] = v;                       // a thread meets its own entries only
        ss = fmaf(v, v, ss);
    }
    const float inv = 1.f / sqrtf(block_sum(ss, scratch) / (float)width + eps);
    for (int i = threadIdx.x; i < width; i += blockDim.x) out[t * n + first + i] = from_f32<T>(y[i] * inv * weight[first + i]);
}

// out = a_scale a + b_scale b, float32 arithmetic
template <typename TA, typename TB>
__global__ void scaled_sum_kernel(const TA* __restrict__ a, float a_scale, const TB* __restrict__ b, float b_scale,
                                  float* __restrict__ out, size_t total) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x)
        out[i] = fmaf(b_scale, to_f32(b[i]), a_scale * to_f32(a[i]));
}

}  // namespace lc

using namespace lc;

LC_API int lc_state_space_prepare(const float* proj, int cols, int T, int heads, int groups, int N, int dv,
                                  const float* taps, const float* bias, int K, const float* tails, const float* dt_bias,
                                  const float* a_log, const int* tok_req, const int* q_offsets, const int* slot_ids,
                                  float* coef, float* x_out, hipStream_t stream) {
    LC_CHECK(T >= 0 && heads > 0 && groups > 0 && N > 0 && dv > 0 && heads % groups == 0, "state space prepare: bad sizes");
    LC_CHECK(cols == 2 * heads * dv + 2 * groups * N + heads, "state space prepare: %d columns do not fit the sizes", cols);
    LC_CHECK(K >= 1 && K <= SHORT_CONV_MAX_TAPS, "state space prepare: %d taps (1 to %d)", K, SHORT_CONV_MAX_TAPS);
    if (T == 0) return 0;
    LC_CHECK(proj && taps && bias && dt_bias && a_log && tok_req && q_offsets && slot_ids && coef && x_out && (K == 1 || tails),
             "state space prepare: null pointer");
    const int x_blocks = (heads * dv + 255) / 256, blocks = x_blocks + (groups * N + 255) / 256;
    // Runs of tokens where they leave five workgroups a CU (eight tokens: eight workgroups, and taps whose inputs are kept).  Runs that empty
    // the card only make its threads' chains longer: 4 heads of 32, a group of 16, 1,024 tokens, two workgroups a run: 256 of eight tokens 9.1 us,
    // 6 taps 16.0, 2,048 of one 5.6 and 6.2; 16 heads of 128, 4 groups of 128, 512 tokens in runs of one, two and four 21, 11.5 and 9.7.
    int tokens = 1;
    auto leaves = [&](int run) { return (long long)((T + run - 1) / run) * blocks / device_cus(); };
    while (tokens < 4 && leaves(2 * tokens) >= 5) tokens *= 2;
    if (K >= 2 && K <= 4 && leaves(8) >= 8) tokens = 8;
    while (tokens > 1 && tokens * heads > 4096) tokens /= 2;
    const size_t lds = (size_t)2 * tokens * heads * sizeof(float);
    const bool kept = lds <= 64 * 1024;
    const dim3 grid((T + tokens - 1) / tokens, blocks < 65535 ? blocks : 65535, (blocks + 65534) / 65535);
#define LC_SS_PREPARE(KT, KEPT)                                                                                                       \
    state_space_prepare_kernel<KT, KEPT><<<grid, 256, KEPT ? lds : 0, stream>>>(proj, cols, T, heads, groups, N, dv, taps, bias, K,   \
                                                                                tails, dt_bias, a_log, tok_req, q_offsets, slot_ids,  \
                                                                                coef, x_out, tokens, x_blocks)
    if (!kept) LC_SS_PREPARE(0, false);
    else if (K == 2) LC_SS_PREPARE(2, true);
    else if (K == 3) LC_SS_PREPARE(3, true);
    else if (K == 4) LC_SS_PREPARE(4, true);
    else LC_SS_PREPARE(0, true);
#undef LC_SS_PREPARE
    LC_LAUNCH_CHECK("state_space_prepare");
    return 0;
}

LC_API int lc_state_space_readout(const float* o, const float* x, const float* gates, int gate_cols, int z_column,
                                  const float* skip, int heads, int dv, const float* weight, int parts, float eps, int T,
                                  void* out, int dt, hipStream_t stream) {
    const int n = heads * dv;
    LC_CHECK(T >= 0 && heads > 0 && dv > 0 && parts > 0 && n % parts == 0 && z_column >= 0 && z_column + n <= gate_cols,
             "state space readout: bad sizes");
    if (T == 0) return 0;
    LC_CHECK(o && x && gates && skip && weight && out, "state space readout: null pointer");
    const int width = n / parts;
    const size_t lds = (size_t)width * sizeof(float);
    LC_CHECK(lds <= 48 * 1024, "state space readout: parts of %d entries are too long", width);
    LC_CHECK(parts <= 65535, "state space readout: too many parts (%d)", parts);
    const int threads = width >= 1024 ? 256 : (width >= 256 ? 128 : 64);
    const dim3 grid(T, parts);
    if (dt == DT_F32)
        state_space_readout_kernel<float><<<grid, threads, lds, stream>>>(o, x, gates, gate_cols, z_column, skip, dv, weight,
                                                                          parts, eps, n, (float*)out);
    else if (dt == DT_BF16)
        state_space_readout_kernel<bf16><<<grid, threads, lds, stream>>>(o, x, gates, gate_cols, z_column, skip, dv, weight,
                                                                         parts, eps, n, (bf16*)out);
    else
        LC_CHECK(false, "state space readout: unknown dtype %d", dt);
    LC_LAUNCH_CHECK("state_space_readout");
    return 0;
}

// a [rows, n] of dtype dt_a, b likewise -> out float32
LC_API int lc_scaled_sum(const void* a, int dt_a, float a_scale, const void* b, int dt_b, float b_scale, float* out,
                         long long total, hipStream_t stream) {
    LC_CHECK(total >= 0, "scaled sum: bad size");
    if (total == 0) return 0;
    LC_CHECK(a && b && out, "scaled sum: null pointer");
    const int blocks = (int)((total + 255) / 256 < 8192 ? (total + 255) / 256 : 8192);
#define LC_SS(TA, TB) scaled_sum_kernel<TA, TB><<<blocks, 256, 0, stream>>>((const TA*)a, a_scale, (const TB*)b, b_scale, out, (size_t)total)
    if (dt_a == DT_F32 && dt_b == DT_F32) LC_SS(float, float);
    else if (dt_a == DT_F32 && dt_b == DT_BF16) LC_SS(float, bf16);
    else if (dt_a == DT_BF16 && dt_b == DT_F32) LC_SS(bf16, float);
    else if (dt_a == DT_BF16 && dt_b == DT_BF16) LC_SS(bf16, bf16);
    else LC_CHECK(false, "scaled sum: unknown dtypes %d, %d", dt_a, dt_b);
#undef LC_SS
    LC_LAUNCH_CHECK("scaled_sum");
    return 0;
}
