// float32 attention over the paged cache on the float32 matrix instruction: heads of 16, 32, ... 128 entries, pages of whole groups
// of four tokens, whole 16-byte pieces.  Formulas, cache layouts and what windows mean are those of attention_generic.hip, which
// serves every other size and bfloat16.
//
// A wave works on 16 columns, each a (query row, query head) of one request and kv head, and on 16 keys at a time:
//   S^T = K Q^T, v_mfma_f32_16x16x4_f32: lane (n = lane % 16, g = lane / 16) gives K and Q entries 16 u + 4 g + e to instruction
//   (u, e), whole 16-byte pieces of both, and gets the scores of the keys 4 g .. 4 g + 3 of column n;
//   O^T += V^T P^T: instruction r takes the keys 4 g + r, so those four weights are its operands as they stand and a lane's four
//   keys of a dim are one 16-byte load.
// Each product costs what the instruction costs (16 columns by 16 keys by 128 entries, both products: 2,048 clocks of a SIMD); float32
// multiply-adds with a lane a key spend four instructions on one.  Against that kernel (us, heads of 128, the keys of one layer hot in the
// caches): 566 rows of three prompts of up to 333 tokens, 16 heads over 8, 119 -> 27; 2,048 rows, 32 over 8, 1,373 -> 489 (70 TFLOP/s
// of 157 over the keys that are seen; the rest is the weights between the products and the units that a row sees in part); 576 rows
// after 8,192 tokens 2,806 -> 1,097; lone tokens, which wait for memory: 8 at 8,192 126 -> 112 (4.8 TB/s), 64 at 1,024 123 -> 105,
// 1 at 8,192 39 -> 29.  Its errors against 64 bits are 5 to 30 % smaller, because sums are made in shorter chains.
//
// The order of the additions is a function of the column's query alone.  Keys go in units of 16 at multiples of 16 and in spans of 512
// at multiples of 512; wave w of the four of a workgroup takes the units u % 4 == w.  A wave's maximum, sum and P.V of a span are
// made on their own, are taken into the wave's total span after span, and the four totals are joined in order.  With few
// columns the spans are workgroups of their own that leave the waves' sums in a workspace, and a second kernel takes them in with the
// same operations.  A key that a column does not see has the weight 0 and changes no bit of it, so that a query has the same bits
// alone, beside others and in any part of a prompt.
#include "common.h"

#include "gemm_tile.h"

LC_API int lc_attention_generic_rows(int rows);        // attention_generic.hip

namespace lc {

constexpr int AF_UNIT = 16, AF_SPAN = 512, AF_WAVES = 4;
constexpr int AF_COLUMNS = 16;

struct F32Attention {
    const float* q; int q_stride;
    const float* k_cache; const float* v_cache; float* out;
    const int* tok_req; const int* positions; const int* block_table;
    int max_blocks, T, nh, nkv, page_size;
    float scale; int window;
    float* part; int spans;         // the waves' sums of every span (spans 0: a workgroup works through all of them)
    int rows;                       // rows of the batch a workgroup takes (1, or as many as have heads * rows <= 16)
    int groups;                     // workgroups that take rows
    const int4* lone;               // row, request, position of the requests with a single token, a workgroup each; null: they are rows as all
};

// m, l and the sums of one wave and span, one column's: [m, l, 0, 0, d sums]
__device__ __forceinline__ size_t part_at(const F32Attention& a, int D, int t, int h, int span, int wave) {
    return ((((size_t)t * a.nh + h) * a.spans + span) * AF_WAVES + wave) * (D + 4);
}

// The running (M, L, O) takes in (m, l, o); m = -inf and l = 0: there were no keys.  (Scores that are all NaN leave m at -inf too, for a
// maximum passes NaN by, but their weights make l NaN.)  Explicit operations, so that all who use it round alike.
template <int N>
__device__ __forceinline__ void take_sums(float& M, float& L, floatx4 (&O)[N], float m, float l, const floatx4 (&o)[N]) {
    if (m == -INFINITY && l == 0.f) return;
    const float top = fmaxf(M, m), a = expf(M - top), b = expf(m - top);
    L = fmaf(L, a, __fmul_rn(l, b));
#pragma unroll
    for (int x = 0; x < N; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e) O[x][e] = fmaf(O[x][e], a, __fmul_rn(o[x][e], b));
    M = top;
}

// The rows t0 .. t0 + live - 1, of one request, and `heads` query heads from h0 on: column n is row n / per, head n % per.  position: the
// only row's, where it is known, else -1.
template <int DB>
__device__ __forceinline__ void attend_columns(const F32Attention& a, int t0, int live, int request, int position, int kvh, int h0, int heads,
                                               int per, float* lds) {
    constexpr int D = 16 * DB;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, g = lane >> 4;
    const int row = n / per, head = n % per;
    const bool active = row < live && head < heads;
    const int t = t0 + (active ? row : 0), p = active ? (position >= 0 ? position : a.positions[t]) : -1;
    const int lo = active && a.window > 0 ? max(0, p - a.window + 1) : 0;
    int p_max = p, p_min = active ? p : INT_MAX, lo_min = active ? lo : INT_MAX, lo_max = lo;
#pragma unroll
    for (int s = 1; s < 16; s *= 2) {
        p_max = max(p_max, __shfl_xor(p_max, s));
        p_min = min(p_min, __shfl_xor(p_min, s));
        lo_min = min(lo_min, __shfl_xor(lo_min, s));
        lo_max = max(lo_max, __shfl_xor(lo_max, s));
    }
    p_max = __builtin_amdgcn_readfirstlane(p_max);
    p_min = __builtin_amdgcn_readfirstlane(p_min);
    lo_min = __builtin_amdgcn_readfirstlane(lo_min);
    lo_max = __builtin_amdgcn_readfirstlane(lo_max);
    int from = lo_min, to = p_max;
    if (a.spans > 0) {
        const int s = lo_min / AF_SPAN + blockIdx.z;
        from = max(from, s * AF_SPAN);
        to = min(to, s * AF_SPAN + AF_SPAN - 1);
        if (from > to) return;
    }
    const int* table = a.block_table + (size_t)request * a.max_blocks;

    // the columns' scaled q, the same for all waves, lies in LDS: [block of 16 entries][lane]
    float4* q4 = reinterpret_cast<float4*>(lds);
    __syncthreads();                    // the rows before these may still be read
    for (int i = wave; i < DB; i += AF_WAVES) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (active) v = *reinterpret_cast<const float4*>(a.q + (size_t)t * a.q_stride + (size_t)(h0 + head) * D + 16 * i + 4 * g);
        q4[i * 64 + lane] = make_float4(v.x * a.scale, v.y * a.scale, v.z * a.scale, v.w * a.scale);
    }
    __syncthreads();

    // unit u: this lane's row of K (key 16 u + n) and group of four keys of V (from 16 u + 4 g on), keys outside from .. to replaced by
    // ones that are inside
    const int u_first = from / AF_UNIT, u_last = to / AF_UNIT;
    struct Pages { int k, v; };
    auto k_key = [&](int u) { return min(max(u * AF_UNIT + n, from), to); };
    auto v_key = [&](int u) { return min(max(u * AF_UNIT + 4 * g, from & ~3), to & ~3); };
    auto pages = [&](int u) { return Pages{table[k_key(u) / a.page_size], table[v_key(u) / a.page_size]}; };
    auto load_k = [&](float4 (&k4)[DB], int u, Pages at) {
        const float* k = a.k_cache + (((size_t)at.k * a.nkv + kvh) * a.page_size + k_key(u) % a.page_size) * D + 4 * g;
#pragma unroll
        for (int i = 0; i < DB; ++i) k4[i] = *reinterpret_cast<const float4*>(k + 16 * i);
    };
    auto load_v = [&](float4 (&v4)[DB], int u, Pages at) {
        const float* v = a.v_cache + (((size_t)at.v * a.nkv + kvh) * D + n) * a.page_size + v_key(u) % a.page_size;
#pragma unroll
        for (int i = 0; i < DB; ++i) v4[i] = *reinterpret_cast<const float4*>(v + (size_t)16 * i * a.page_size);
    };

    float M = -INFINITY, L = 0.f, m = -INFINITY, l = 0.f;
    floatx4 O[DB], o[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i) O[i] = o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    int u = u_first + ((wave - u_first) & (AF_WAVES - 1)), span = u / (AF_SPAN / AF_UNIT);
    if (u <= u_last) {
        // the pages of a unit are asked for two turns ahead, its keys one, its values in its own turn before the scores are made
        Pages at = pages(u), next = pages(min(u + AF_WAVES, u_last));
        float4 k4[DB], v4[DB], ahead[DB];
        load_k(k4, u, at);
        for (; u <= u_last; u += AF_WAVES) {
            if (u / (AF_SPAN / AF_UNIT) != span) {
                take_sums<DB>(M, L, O, m, l, o);
                m = -INFINITY;
                l = 0.f;
#pragma unroll
                for (int i = 0; i < DB; ++i) o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
                span = u / (AF_SPAN / AF_UNIT);
            }
            asm volatile("" ::: "memory");      // q is read from LDS every turn: kept in registers it would make the sums spill
            load_v(v4, u, at);
            const Pages later = pages(min(u + 2 * AF_WAVES, u_last));
            load_k(ahead, min(u + AF_WAVES, u_last), next);
            // eight sums of a score's products, added in pairs: shorter chains, and no product waits for the one before it
            constexpr int SUMS = DB > 1 ? 8 : 4;
            floatx4 part[SUMS];
#pragma unroll
            for (int c = 0; c < SUMS; ++c) part[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < DB; ++i) {
                const float4 q = q4[i * 64 + lane];
                floatx4* to_sum = part + (4 * i) % SUMS;
                to_sum[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[i].x, q.x, to_sum[0], 0, 0, 0);
                to_sum[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[i].y, q.y, to_sum[1], 0, 0, 0);
                to_sum[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[i].z, q.z, to_sum[2], 0, 0, 0);
                to_sum[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[i].w, q.w, to_sum[3], 0, 0, 0);
            }
#pragma unroll
            for (int c = 0; c + 4 < SUMS; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r) part[c][r] = __fadd_rn(part[c][r], part[c + 4][r]);
            float s[4];
            const int key = u * AF_UNIT + 4 * g;
            const bool whole = u * AF_UNIT >= lo_max && u * AF_UNIT + AF_UNIT - 1 <= p_min;      // every column sees every key
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[r] = __fadd_rn(__fadd_rn(part[0][r], part[1][r]), __fadd_rn(part[2][r], part[3][r]));
                if (!whole && (key + r < lo || key + r > p)) s[r] = -INFINITY;
            }
            float top = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
            top = fmaxf(top, __shfl_xor(top, 16));
            top = fmaxf(m, fmaxf(top, __shfl_xor(top, 32)));
            const float at0 = top == -INFINITY ? 0.f : top;        // a column that has seen no key yet
            const float alpha = expf(m - at0);
            m = top;
            float w[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) w[r] = expf(s[r] - at0);
            float sum = __fadd_rn(__fadd_rn(w[0], w[1]), __fadd_rn(w[2], w[3]));
            sum = __fadd_rn(sum, __shfl_xor(sum, 16));
            sum = __fadd_rn(sum, __shfl_xor(sum, 32));
            l = fmaf(l, alpha, sum);
            // a unit's products are added up from zero and then taken into the span's sum, four blocks of dims at a time
            auto products = [&](floatx4 (&sums)[DB], const float4 (&values)[DB]) {
                constexpr int AT_ONCE = DB < 4 ? DB : 4;
#pragma unroll
                for (int i0 = 0; i0 < DB; i0 += AT_ONCE) {
                    floatx4 add[AT_ONCE];
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int i = 0; i < AT_ONCE; ++i)
                            if (i0 + i < DB) {
                                const float4& v = values[i0 + i];
                                add[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(r == 0 ? v.x : r == 1 ? v.y : r == 2 ? v.z : v.w, w[r],
                                                                              r == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : add[i], 0, 0, 0);
                            }
#pragma unroll
                    for (int i = 0; i < AT_ONCE; ++i)
                        if (i0 + i < DB)
#pragma unroll
                            for (int e = 0; e < 4; ++e) sums[i0 + i][e] = fmaf(sums[i0 + i][e], alpha, add[i][e]);
                }
            };
            bool apart = false;
            if (!whole) {
                // values outside from .. to are other requests' or none; one that is not finite may only reach columns that see its key
                bool finite = true;
#pragma unroll
                for (int i = 0; i < DB; ++i) {
                    float* v = reinterpret_cast<float*>(&v4[i]);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        v[r] = key + r >= from && key + r <= to ? v[r] : 0.f;
                        finite = finite && fabsf(v[r]) < INFINITY;
                    }
                }
                apart = __any(!finite);
            }
            if (!apart) {
                products(o, v4);
            } else {
#pragma unroll 1
                for (int c = 0; c < AF_COLUMNS; ++c) {
                    const int its_lo = __shfl(lo, c), its_p = __shfl(p, c);
                    floatx4 sums[DB];
                    float4 seen[DB];
#pragma unroll
                    for (int i = 0; i < DB; ++i) {
                        sums[i] = o[i];
                        seen[i] = v4[i];
                        float* v = reinterpret_cast<float*>(&seen[i]);
#pragma unroll
                        for (int r = 0; r < 4; ++r) v[r] = key + r >= its_lo && key + r <= its_p ? v[r] : 0.f;
                    }
                    products(sums, seen);
#pragma unroll
                    for (int i = 0; i < DB; ++i)
                        if (n == c) o[i] = sums[i];
                }
            }
            at = next;
            next = later;
#pragma unroll
            for (int i = 0; i < DB; ++i) k4[i] = ahead[i];
        }
    }

    if (a.spans > 0) {
        // the row's own spans, counted from its first
        const int mine = lo_min / AF_SPAN + blockIdx.z;
        if (active && mine >= lo / AF_SPAN && mine <= p / AF_SPAN) {
            float* to_part = a.part + part_at(a, D, t, h0 + head, mine - lo / AF_SPAN, wave);
            if (g == 0) { to_part[0] = m; to_part[1] = l; }
#pragma unroll
            for (int i = 0; i < DB; ++i) *reinterpret_cast<floatx4*>(to_part + 4 + 16 * i + 4 * g) = o[i];
        }
        return;
    }
    take_sums<DB>(M, L, O, m, l, o);
    // the waves' totals, joined in order: [wave][m, l of 16 columns], then [wave][block of dims][lane]
    float* ml = lds + DB * 256;
    floatx4* sums = reinterpret_cast<floatx4*>(ml + AF_WAVES * 2 * AF_COLUMNS);
    if (g == 0) { ml[wave * 32 + n] = M; ml[wave * 32 + 16 + n] = L; }
#pragma unroll
    for (int i = 0; i < DB; ++i) sums[(wave * DB + i) * 64 + lane] = O[i];
    __syncthreads();
    for (int i = wave; i < DB; i += AF_WAVES) {
        float M4 = -INFINITY, L4 = 0.f;
        floatx4 O4[1] = {floatx4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int w = 0; w < AF_WAVES; ++w) {
            const floatx4 one[1] = {sums[(w * DB + i) * 64 + lane]};
            take_sums<1>(M4, L4, O4, ml[w * 32 + n], ml[w * 32 + 16 + n], one);
        }
        if (active)
            *reinterpret_cast<float4*>(a.out + ((size_t)t * a.nh + h0 + head) * D + 16 * i + 4 * g) =
                make_float4(O4[0][0] / L4, O4[0][1] / L4, O4[0][2] / L4, O4[0][3] / L4);
    }
}

// grid (kv heads by batches of 16 query heads; groups of rows, then lone rows; spans), so that a group's heads start side by side.  A group's
// rows are worked together when they belong to one request, else request by request.
template <int DB>
__global__ __launch_bounds__(64 * AF_WAVES, 2) void attention_f32_kernel(F32Attention a) {
    __shared__ __attribute__((aligned(16))) float lds[DB * 256 + AF_WAVES * (2 * AF_COLUMNS + DB * 256)];
    const int group = a.nh / a.nkv, per = min(group, AF_COLUMNS), batches = (group + per - 1) / per;
    const int at = blockIdx.y, kvh = batches == 1 ? blockIdx.x : blockIdx.x / batches, h0 = kvh * group + (blockIdx.x - kvh * batches) * per;
    const int heads = min(per, (kvh + 1) * group - h0);
    if (at >= a.groups) {
        const int4 row = a.lone[at - a.groups];
        attend_columns<DB>(a, row.x, 1, row.y, row.z, kvh, h0, heads, per, lds);
        return;
    }
    // the last groups, which mostly see the most keys, first
    const int first = (a.groups - 1 - at) * a.rows, end = min(first + a.rows, a.T);
    for (int t = first; t < end;) {
        const int request = a.tok_req[t];
        int n = 1;
        while (t + n < end && a.tok_req[t + n] == request) ++n;
        const bool lone = a.lone && n == 1 && !(t > 0 && a.tok_req[t - 1] == request) && !(t + 1 < a.T && a.tok_req[t + 1] == request);
        if (!lone) attend_columns<DB>(a, t, n, request, -1, kvh, h0, heads, per, lds);
        t += n;
    }
}

// One workgroup per (token, head): a wave for each wave's sums, a lane for four dims; the spans from the first on, then the waves.
template <int DB>
__global__ __launch_bounds__(64 * AF_WAVES) void attention_f32_join_kernel(F32Attention a) {
    constexpr int D = 16 * DB, AHEAD = 4;           // spans asked for before the first is taken in
    __shared__ float ml[AF_WAVES][2];
    __shared__ floatx4 sums[AF_WAVES][D / 4];
    const int t = blockIdx.x, h = blockIdx.y, wave = threadIdx.x >> 6, i = min((int)threadIdx.x & 63, D / 4 - 1);
    const int p = a.positions[t], lo = a.window > 0 ? max(0, p - a.window + 1) : 0, spans = p / AF_SPAN - lo / AF_SPAN + 1;
    float M = -INFINITY, L = 0.f;
    floatx4 O[1] = {floatx4{0.f, 0.f, 0.f, 0.f}};
    for (int s0 = 0; s0 < spans; s0 += AHEAD) {
        float m[AHEAD], l[AHEAD];
        floatx4 one[AHEAD][1];
#pragma unroll
        for (int s = 0; s < AHEAD; ++s) {
            const float* from = a.part + part_at(a, D, t, h, min(s0 + s, spans - 1), wave);
            m[s] = from[0];
            l[s] = from[1];
            one[s][0] = *reinterpret_cast<const floatx4*>(from + 4 + 4 * i);
        }
#pragma unroll
        for (int s = 0; s < AHEAD; ++s)
            if (s0 + s < spans) take_sums<1>(M, L, O, m[s], l[s], one[s]);
    }
    if (((int)threadIdx.x & 63) == i) sums[wave][i] = O[0];
    if ((threadIdx.x & 63) == 0) { ml[wave][0] = M; ml[wave][1] = L; }
    __syncthreads();
    if (wave || (int)threadIdx.x != i) return;
    float M4 = -INFINITY, L4 = 0.f;
    floatx4 O4[1] = {floatx4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int w = 0; w < AF_WAVES; ++w) {
        const floatx4 one[1] = {sums[w][i]};
        take_sums<1>(M4, L4, O4, ml[w][0], ml[w][1], one);
    }
    *reinterpret_cast<float4*>(a.out + ((size_t)t * a.nh + h) * D + 4 * i) =
        make_float4(O4[0][0] / L4, O4[0][1] / L4, O4[0][2] / L4, O4[0][3] / L4);
}

// How a batch's rows are cut: rows a workgroup takes, workgroups that take rows, lone rows with a workgroup of their own.  A workgroup's rows
// of several requests are worked one request after the other, so it takes no more than a portion has on average (64 portions of two rows, 8
// heads over 8 of 128: 16 rows a workgroup 42.7 us, two 8.4; 40 of three after 600, 4 heads over 4 of 16: 57.5 and 15.5).
struct F32Cut { int rows, groups, lone; };

static F32Cut f32_cut(int T, int nh, int nkv, int requests, int lone) {
    const int forced = lc_attention_generic_rows(-1);       // tests: one row, or as many as there is room for; no lone rows then
    if (forced) lone = 0;
    const int per = nh / nkv < AF_COLUMNS ? nh / nkv : AF_COLUMNS, most = AF_COLUMNS / per;
    const int portions = requests - lone > 1 ? requests - lone : 1, mean = (T - lone) / portions;
    const int rows = forced == 1 ? 1 : forced || mean >= most ? most : mean > 1 ? mean : 1;
    return {rows, lone == T ? 0 : (T + rows - 1) / rows, lone};
}

// Spans a launch is cut into (0: it is not): when the workgroups would not fill the card and the block table is wide enough for more
// than one.  Lone tokens wait for memory and want four workgroups a CU, rows of prompts two.
static int f32_spans(int T, int nh, int nkv, int d, int max_blocks, int page_size, F32Cut cut) {
    const int group = nh / nkv, batches = (group + AF_COLUMNS - 1) / AF_COLUMNS;
    const long long workgroups = (long long)(cut.groups + cut.lone) * nkv * batches, keys = (long long)max_blocks * page_size;
    if (workgroups >= (cut.rows > 1 && cut.groups > 0 ? 512 : 1024) || keys <= AF_SPAN) return 0;
    const long long spans = (keys + AF_SPAN - 1) / AF_SPAN;
    if (spans > 65535 || (long long)T * nh * spans * AF_WAVES * (d + 4) > (64ll << 20)) return 0;      // 256 MiB
    return (int)spans;
}

template <int DB>
static void launch_f32(const F32Attention& a, int lone, hipStream_t stream) {
    const int group = a.nh / a.nkv, batches = (group + AF_COLUMNS - 1) / AF_COLUMNS;
    attention_f32_kernel<DB><<<dim3(a.nkv * batches, a.groups + lone, a.spans > 0 ? a.spans : 1), 64 * AF_WAVES, 0, stream>>>(a);
    if (a.spans > 0) attention_f32_join_kernel<DB><<<dim3(a.T, a.nh), 64 * AF_WAVES, 0, stream>>>(a);
}

}  // namespace lc

using namespace lc;

// Whether lc_attention_f32 takes these sizes and operands: 1 or 0.
LC_API int lc_attention_f32_takes(const void* q, int q_stride, const void* k_cache, const void* v_cache, int nh, int nkv, int d,
                                  int page_size) {
    return nh > 0 && nkv > 0 && nh % nkv == 0 && d > 0 && d <= 128 && d % 16 == 0 && page_size > 0 && page_size % 4 == 0 && q_stride % 4 == 0 &&
           ((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) % 16 == 0;
}

// float32 words of workspace that lc_attention_f32 needs (0: none) for T rows of `requests` requests, `lone` of which have a row and a list
// entry each; -1: these sizes or operands are the general kernel's (grids are cut for up to 65,535 groups of rows and heads).
LC_API long long lc_attention_f32_workspace(const void* q, int q_stride, const void* k_cache, const void* v_cache, int T, int nh, int nkv, int d,
                                            int max_blocks, int page_size, int requests, int lone) {
    if (!lc_attention_f32_takes(q, q_stride, k_cache, v_cache, nh, nkv, d, page_size) || T <= 0 || max_blocks <= 0 || lone < 0 || lone > T) return -1;
    const F32Cut cut = f32_cut(T, nh, nkv, requests, lone);
    if (nh > 65535 || (long long)cut.groups + cut.lone > 65535) return -1;
    return (long long)T * nh * f32_spans(T, nh, nkv, d, max_blocks, page_size, cut) * AF_WAVES * (d + 4);
}

// requests: rows of the block table, which tells portions of many rows from portions of few.  lone_rows [lone, 4] (row, request, position,
// any): all requests that have a single row, or none at all (lone 0).
LC_API int lc_attention_f32(const void* q, int q_stride, const void* k_cache, const void* v_cache, void* out, const int* tok_req,
                            const int* positions, const int* block_table, int max_blocks, int T, int nh, int nkv, int d, int page_size,
                            float scale, int window, int requests, const int* lone_rows, int lone, float* workspace, hipStream_t stream) {
    LC_CHECK(T >= 0 && nh > 0 && nkv > 0 && d > 0 && page_size > 0 && max_blocks > 0 && lone >= 0 && lone <= T,
             "attention: bad sizes T=%d nh=%d nkv=%d d=%d page=%d blocks=%d lone=%d", T, nh, nkv, d, page_size, max_blocks, lone);
    if (T == 0) return 0;
    LC_CHECK(nh % nkv == 0, "attention: %d query heads are not a multiple of %d kv heads", nh, nkv);
    LC_CHECK(q && k_cache && v_cache && out && tok_req && positions && block_table && (lone == 0 || lone_rows), "attention: null pointer");
    LC_CHECK(lc_attention_f32_takes(q, q_stride, k_cache, v_cache, nh, nkv, d, page_size) && ((uintptr_t)out | (uintptr_t)lone_rows) % 16 == 0,
             "attention: heads of %d and pages of %d tokens, or unaligned operands, are the general kernel's", d, page_size);
    const F32Cut cut = f32_cut(T, nh, nkv, requests, lone);
    LC_CHECK(nh <= 65535 && (long long)cut.groups + cut.lone <= 65535, "attention: too many heads (%d) or rows (%d)", nh, T);
    const int spans = f32_spans(T, nh, nkv, d, max_blocks, page_size, cut);
    LC_CHECK(spans == 0 || (workspace && (uintptr_t)workspace % 16 == 0), "attention: T=%d with %d blocks needs a workspace", T, max_blocks);
    const F32Attention a{(const float*)q, q_stride, (const float*)k_cache, (const float*)v_cache, (float*)out, tok_req, positions, block_table,
                         max_blocks, T, nh, nkv, page_size, scale, window, workspace, spans, cut.rows, cut.groups,
                         cut.lone > 0 ? (const int4*)lone_rows : nullptr};
    switch (d / 16) {
        case 1: launch_f32<1>(a, cut.lone, stream); break;
        case 2: launch_f32<2>(a, cut.lone, stream); break;
        case 3: launch_f32<3>(a, cut.lone, stream); break;
        case 4: launch_f32<4>(a, cut.lone, stream); break;
        case 5: launch_f32<5>(a, cut.lone, stream); break;
        case 6: launch_f32<6>(a, cut.lone, stream); break;
        case 7: launch_f32<7>(a, cut.lone, stream); break;
        default: launch_f32<8>(a, cut.lone, stream);
    }
    LC_LAUNCH_CHECK("attention_f32");
    return 0;
}
