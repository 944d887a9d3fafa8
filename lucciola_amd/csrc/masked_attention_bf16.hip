// The masked attention of masked_attention.hip on the matrix cores, for bfloat16 caches whose sizes fit:
// key heads of a multiple of 8 entries up to 128, value heads of a multiple of 16 up to 128, pages of a
// multiple of 16 tokens.  Same formulas, same cache (keys token-major, values transposed inside a page);
// scores, softmax, sink, bias and the heads' combination are float32, the two products take bfloat16
// operands: the weights go into P.V as two bfloat16 numbers each (the rounded weight and the rounding's
// remainder, two products), so that they count with 16 bits of mantissa and not with 8.
//
// Work comes as the step's tiles (first token row, tokens, request, first position: up to 16 tokens of one
// request); a workgroup of eight waves serves a tile and one kv head.
//   A tile of several tokens: a wave's 16 columns are the tile's tokens for one query head of the kv head's
//   group; where the group has fewer than eight heads, the waves of a head share out the blocks of keys.
//   A lone token: the 16 columns are query heads of the group, and all eight waves share out the blocks.
// Waves that shared a column's keys leave their maxima, sums and rows in LDS, and the first of them takes the
// others in, in their order.  A wave asks for the next block's keys before it works on this one's.
// In a step of lone tokens only, with fewer workgroups than the card has room for, a token's blocks are also
// shared out over several workgroups (the grid's last place); each leaves its joined sums in a workspace, and a
// second kernel takes them in, in their order, and finishes the columns.
// Keys are walked in blocks of 16 (one part of a page).  S^T = K Q^T (16x16x32: a lane's operand is 16 bytes
// in a row of a key, straight from memory) leaves a lane with four keys of one query column, which is the
// operand P^T of O^T += V^T P^T (16x16x16; V^T's operand is four neighbouring keys of one value entry, 8
// bytes in a row of the transposed page), so the weights never leave the registers.
// The workgroups go tile by tile, a tile's kv heads beside each other, and the list has the longest tiles first: with all tiles of
// one kv head before the next head's, the last head's longest tile began when half of the card had run dry (2,048 tokens, four kv
// heads, a workgroup a CU: 202 -> 136 us for two maps of 64, 207 -> 143 for one of 128 with the bias; 1,523 tokens 102 -> 78; with two
// blocks of keys a step and the scores' forms known to the build 118, 114 and 67; with two stages in LDS, below, 99, 78 and 50).
#include "common.h"

namespace lc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int MB_WAVES = 8;
constexpr int MB_THREADS = MB_WAVES * kWave;

struct MaskedArgs {
    const bf16* q;
    const bf16* k_cache;
    const bf16* v_cache;
    const int* tiles;
    int num_tiles;
    const int* block_table;
    int max_blocks, page_size, heads, kv_heads, d, dv;
    float scale2;       // scores are in units of log 2, here and wherever they meet: the weights are powers of two
    int chunk, window, keep;
    float cap, cap2;    // scores become cap tanh(score / cap) where it is positive; cap2: in the scores' units
    const float* r1;
    const float* r2;
    const float* sink;
    float lambda;
    int unit_out;
    float eps, out_scale;
    const float* gate;
    int gate_stride, gate_column;
    bf16* out;
    float* shares;      // where a lone token's keys are shared out over workgroups: their sums, joined by a second kernel
    int zsplits;
    int lone_only;      // the tiles of several tokens are another kernel's
    int wave_blocks;    // blocks of a stage for every wave that shares a head's keys, in the kernel that stages them
    int at_once;        // the order of the workgroups (below)
};

// floats a wave leaves per lane and map where key ranges are joined: maximum, sum, the lane's part of O^T
template <int DVB> constexpr int share_floats() { return DVB * 4 + 2; }

__device__ __forceinline__ short bits_of(__bf16 v) { return __builtin_bit_cast(short, v); }

constexpr float LOG2E = 1.4426950408889634f;

// s, in units of log 2, held below cap: cap tanh(s / cap) = cap (1 - 2 / (1 + e^(2 s / cap))); the ends saturate to +-cap.  The reciprocal is
// the hardware's with one step of Newton's method, which leaves the last place (a division is ten instructions).
__device__ __forceinline__ float held(float s, float two_by_cap, float cap2) {
    const float x = s * two_by_cap, d = 1.f + __builtin_amdgcn_exp2f(x > 60.f ? 60.f : x);      // (NaN stays)
    float r = __builtin_amdgcn_rcpf(d);
    r = fmaf(fmaf(-d, r, 1.f), r, r);
    return fmaf(-2.f * cap2, r, cap2);
}

// What becomes of the scores, known to the build where it counts (FORM_ANY asks the arguments at every block).
enum : int { FORM_PLAIN = 0, FORM_BIAS = 1, FORM_CAP = 2, FORM_ANY = 4 };

// over the four lanes that hold one query column (lane, lane ^ 16, lane ^ 32, lane ^ 48)
__device__ __forceinline__ float column_max4(float v) {
    v = fmaxf(v, __shfl_xor(v, 16, kWave));
    return fmaxf(v, __shfl_xor(v, 32, kWave));
}
__device__ __forceinline__ float column_sum4(float v) {
    v += __shfl_xor(v, 16, kWave);
    return v + __shfl_xor(v, 32, kWave);
}

template <int DVB, int MAPS>
struct ColumnState {
    float m[MAPS], l[MAPS];     // the column's reference point (the same in its four lanes); the lane's own part of the sum
    floatx4 o[MAPS][DVB];       // O^T: value entries 16 t + 4 (lane / 16) + i of the lane's query column
};

// The upper halves of two float32 numbers side by side.
__device__ __forceinline__ unsigned upper_halves(float first, float second) {
    return __builtin_amdgcn_perm(__float_as_uint(second), __float_as_uint(first), 0x07060302u);
}

// NB blocks of 16 keys for the lane's column: scores from the keys' and the queries' operands, mask, bias, the
// reference point and the sum, and the weighted values taken into O^T.  Two blocks at once take their values with products over 32
// keys (a lane's operand is its four keys of the one and its four of the other), which cost what products over 16 do: 2,048 tokens, 16
// heads over 4, two maps of 64 224 -> 202 us, one of 128 with the bias 210 -> 207 (one stage in LDS).
//
// A score costs its scaling, the maximum, the difference to the reference, exp2, the sum and five instructions for the weight's two numbers;
// the bias five more and a logarithm, the cap six, exp2 and a reciprocal.  With bias and cap asked for at run time, natural exponents and
// divisions, us then and now: 2,048 tokens, 16 heads over 4, two maps of 64 130 and 118, one of 128 with the bias 138 and 114; 1,523 tokens,
// keys of 128, two layers without and one with the cap 246 and 218 together.
template <int FORM, int NB, int DSTEPS, int DVB, int MAPS>
__device__ __forceinline__ void block_step(ColumnState<DVB, MAPS>& st, const MaskedArgs& a,
                                           const bf16x8 (&bq)[MAPS][DSTEPS], const bf16x8 (&ka)[NB][MAPS][DSTEPS],
                                           const short4v (&va)[NB][DVB], const int (&key0)[NB], int pos, int lo, float bias1, float bias2,
                                           const bool (&all_seen)[NB], int lane) {
    const int quad = lane >> 4;
    const bool biased = FORM == FORM_ANY ? a.r1 != nullptr : FORM == FORM_BIAS, capped = FORM == FORM_ANY ? a.cap > 0.f : FORM == FORM_CAP;
    float far[NB][4];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const float first = (float)(pos - (key0[b] + quad * 4));
#pragma unroll
        for (int v = 0; v < 4; ++v) far[b][v] = biased ? bias1 * __builtin_amdgcn_logf(fmaf(bias2, fmaxf(first - (float)v, 0.f), 1.f)) : 0.f;
    }
    const float two_by_cap = capped ? 2.f / a.cap : 0.f;
    auto score = [&](float product, float far_by) {
        const float t = biased ? fmaf(product, a.scale2, -far_by) : product * a.scale2;
        return capped ? held(t, two_by_cap, a.cap2) : t;
    };
#pragma unroll
    for (int m = 0; m < MAPS; ++m) {
        floatx4 s[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) s[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < DSTEPS; ++i)
#pragma unroll
            for (int b = 0; b < NB; ++b) s[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[b][m][i], bq[m][i], s[b], 0, 0, 0);
        float mx = -INFINITY;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (all_seen[b]) {             // every column of the wave sees the whole block: nothing to mask
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    s[b][v] = score(s[b][v], far[b][v]);
                    mx = fmaxf(mx, s[b][v]);
                }
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int j = key0[b] + quad * 4 + v;
                    s[b][v] = ((j >= lo || j < a.keep) && j <= pos) ? score(s[b][v], far[b][v]) : -INFINITY;
                    mx = fmaxf(mx, s[b][v]);
                }
            }
        }
        // The column's reference point st.m moves only when a score outgrows it by 2^12 (or it has none yet): until
        // then no lane asks its column's other three, the weights are 2^(s - reference) <= 2^12, and a lane keeps
        // its own part of the column's sum, which is added up when the column is finished.
        if (__any(mx > st.m[m] + 12.f)) {
            const float top = column_max4(mx);
            const float m_new = top > st.m[m] + 12.f ? top : st.m[m];
            const float alpha = m_new == st.m[m] ? 1.f : __builtin_amdgcn_exp2f(st.m[m] - m_new);       // 0 from no reference at all
            st.l[m] *= alpha;
#pragma unroll
            for (int t = 0; t < DVB; ++t) st.o[m][t] *= alpha;
            st.m[m] = m_new;
        }
        const float base = st.m[m] == -INFINITY ? 0.f : st.m[m];      // a column that has seen no key yet
        // A weight p >= 0 as two bfloat16 numbers: its upper 16 bits, and the upper 16 bits of what they leave
        // (p minus them is exact in float32): together p to 2^-15 of itself.
        float psum = 0.f;
        unsigned hi[2 * NB], lw[2 * NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float p[4], left[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                p[v] = __builtin_amdgcn_exp2f(s[b][v] - base);
                psum += p[v];
                left[v] = p[v] - __uint_as_float(__float_as_uint(p[v]) & 0xffff0000u);
            }
            hi[2 * b] = upper_halves(p[0], p[1]);
            hi[2 * b + 1] = upper_halves(p[2], p[3]);
            lw[2 * b] = upper_halves(left[0], left[1]);
            lw[2 * b + 1] = upper_halves(left[2], left[3]);
        }
        st.l[m] += psum;
        // the weights' upper halves into every block of value entries first, then the remainders: no product waits
        // for the one before it
        if constexpr (NB == 2) {
            typedef unsigned uint4v __attribute__((ext_vector_type(4)));
            auto both = [&](int t) {
                return __builtin_bit_cast(bf16x8, __builtin_shufflevector(va[0][t], va[1][t], 0, 1, 2, 3, 4, 5, 6, 7));
            };
            const bf16x8 hi8 = __builtin_bit_cast(bf16x8, uint4v{hi[0], hi[1], hi[2], hi[3]});
            const bf16x8 lw8 = __builtin_bit_cast(bf16x8, uint4v{lw[0], lw[1], lw[2], lw[3]});
#pragma unroll
            for (int t = 0; t < DVB; ++t) st.o[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(both(t), hi8, st.o[m][t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < DVB; ++t) st.o[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(both(t), lw8, st.o[m][t], 0, 0, 0);
        } else {
            typedef unsigned uint2v __attribute__((ext_vector_type(2)));
            const short4v hi4 = __builtin_bit_cast(short4v, uint2v{hi[0], hi[1]}), lw4 = __builtin_bit_cast(short4v, uint2v{lw[0], lw[1]});
#pragma unroll
            for (int t = 0; t < DVB; ++t) st.o[m][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(va[0][t], hi4, st.o[m][t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < DVB; ++t) st.o[m][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(va[0][t], lw4, st.o[m][t], 0, 0, 0);
        }
    }
}

// The blocks of 16 keys a tile walks: those that hold kept keys and lie before the first visible block, then the blocks
// first .. last.
struct BlockList {
    int kept, first, count;
    __device__ __forceinline__ int block(int i) const { return i < kept ? i : first + (i - kept); }
};
__device__ __forceinline__ BlockList block_list(int keep, int first, int last) {
    const int kept = min((keep + 15) / 16, first);
    return {kept, first, kept + last - first + 1};
}

template <int DSTEPS, int MAPS>
__device__ __forceinline__ void load_queries(bf16x8 (&bq)[MAPS][DSTEPS], const MaskedArgs& a, int tok, int head, int pos,
                                             int lane) {
    const int quad = lane >> 4;
#pragma unroll
    for (int m = 0; m < MAPS; ++m)
#pragma unroll
        for (int s = 0; s < DSTEPS; ++s) {
            const int e = s * 32 + quad * 8;
#pragma unroll
            for (int x = 0; x < 8; ++x) bq[m][s][x] = (__bf16)0.f;
            if (pos >= 0 && e < a.d)
                bq[m][s] = *reinterpret_cast<const bf16x8*>(a.q + ((size_t)tok * a.heads + head) * MAPS * a.d + m * a.d + e);
        }
}

template <int DVB, int MAPS>
__device__ __forceinline__ void clear_state(ColumnState<DVB, MAPS>& st) {
#pragma unroll
    for (int m = 0; m < MAPS; ++m) {
        st.m[m] = -INFINITY;
        st.l[m] = 0.f;
#pragma unroll
        for (int t = 0; t < DVB; ++t) st.o[m][t] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
}

// The lane's column: token row `tok`, head `head`, position `pos` (-1: no such column), first visible key `lo`.
// The blocks of 16 keys to walk are a list, the kept ones in front (BlockList); the lane's wave takes the list's places
// at, at + stride, ... (the same for all lanes): a lane holds the page of one of its next 64 places, so that a block's loads do not wait
// for its page (us, before and so: 64 lone tokens at 2,047 keys, 32 heads over 8, 128, 128 128 and 118, 16 over 16, 64, 32 102 and 94; at 128 to 2,047
// keys, 16 over 4, with the bias 41 and 37; at 2,047, 16 over 4, 256 equal workgroups,
// 48 and 50 with everything in the caches, 71.6 and 70.5 from memory).  Keys seen_from .. seen_to are seen by every column of
// the tile (a block inside them needs no mask).
template <int DSTEPS, int DVB, int MAPS>
__device__ __forceinline__ void attend_blocks(ColumnState<DVB, MAPS>& st, const MaskedArgs& a, int g, int tok, int head,
                                              int pos, int lo, const int* __restrict__ table, const BlockList& blocks,
                                              int at, int stride, int seen_from, int seen_to, int lane) {
    const int quad = lane >> 4, col = lane & 15;
    const size_t k_row = (size_t)a.kv_heads * MAPS * a.d;
    bf16x8 bq[MAPS][DSTEPS];
    load_queries<DSTEPS, MAPS>(bq, a, tok, head, pos, lane);
    const float bias1 = (a.r1 && pos >= 0) ? a.r1[head] : 0.f, bias2 = (a.r1 && pos >= 0) ? a.r2[head] : 0.f;
    clear_state<DVB, MAPS>(st);
    auto pages_from = [&](int i) {
        const int block = blocks.block(min(i + lane * stride, blocks.count - 1));
        return table[a.page_size == 16 ? block : block * 16 / a.page_size];
    };
    struct Block { int page, within; };
    auto found = [&](int pages, int n, int i) {                 // the n-th of the wave's places, i
        return Block{__builtin_amdgcn_readlane(pages, n % kWave), a.page_size == 16 ? 0 : blocks.block(i) * 16 % a.page_size};
    };
    auto load_keys = [&](bf16x8 (&dst)[MAPS][DSTEPS], const Block& b) {
        const size_t row0 = (size_t)b.page * a.page_size + b.within;
#pragma unroll
        for (int m = 0; m < MAPS; ++m)
#pragma unroll
            for (int s = 0; s < DSTEPS; ++s) {
                const int e = s * 32 + quad * 8;
#pragma unroll
                for (int x = 0; x < 8; ++x) dst[m][s][x] = (__bf16)0.f;
                if (e < a.d)
                    dst[m][s] = *reinterpret_cast<const bf16x8*>(a.k_cache + (row0 + col) * k_row + ((size_t)g * MAPS + m) * a.d + e);
            }
    };
    auto load_values = [&](short4v (&dst)[DVB], const Block& b) {
#pragma unroll
        for (int t = 0; t < DVB; ++t) {
            dst[t] = short4v{0, 0, 0, 0};
            if (t * 16 < a.dv)
                dst[t] = *reinterpret_cast<const short4v*>(
                    a.v_cache + ((size_t)b.page * a.kv_heads * a.dv + (size_t)g * a.dv + t * 16 + col) * a.page_size + b.within + quad * 4);
        }
    };
    // the next block's values travel ahead as well where the registers hold them
    constexpr bool VALUES_AHEAD = DSTEPS * MAPS * 4 + DVB * MAPS * 4 + DVB * 4 <= 120;
    bf16x8 ka[1][MAPS][DSTEPS], kn[MAPS][DSTEPS];
    short4v va[1][DVB], vn[DVB];
    if (at >= blocks.count) return;
    int pages = pages_from(at);
    Block now = found(pages, 0, at);
    load_keys(ka[0], now);
    if constexpr (VALUES_AHEAD) load_values(va[0], now);
    for (int i = at, n = 1; i < blocks.count; i += stride, ++n) {
        const int key0 = blocks.block(i) * 16;
        if constexpr (!VALUES_AHEAD) load_values(va[0], now);
        if (i + stride < blocks.count) {            // on their way while this block is worked on
            if (n % kWave == 0) pages = pages_from(i + stride);
            now = found(pages, n, i + stride);
            load_keys(kn, now);
            if constexpr (VALUES_AHEAD) load_values(vn, now);
        }
        block_step<FORM_ANY, 1, DSTEPS, DVB, MAPS>(st, a, bq, ka, va, {key0}, pos, lo, bias1, bias2,
                                         {(key0 >= seen_from || key0 + 15 < a.keep) && key0 + 15 <= seen_to}, lane);
#pragma unroll
        for (int m = 0; m < MAPS; ++m)
#pragma unroll
            for (int i = 0; i < DSTEPS; ++i) ka[0][m][i] = kn[m][i];
        if constexpr (VALUES_AHEAD)
#pragma unroll
            for (int t = 0; t < DVB; ++t) va[0][t] = vn[t];
    }
}

// The lane's column is done: sink, the maps' combination, the unit norm, the gate; four entries a block written.
template <int DVB, int MAPS>
__device__ __forceinline__ void finish_column(const ColumnState<DVB, MAPS>& st, const MaskedArgs& a, int tok, int head,
                                              int pos, int lane) {
    const int quad = lane >> 4;
    floatx4 o[DVB];
#pragma unroll
    for (int m = 0; m < MAPS; ++m) {
        float top = st.m[m], sunk = 0.f;
        if (a.sink && pos >= 0) {
            const float sink2 = a.sink[head] * LOG2E;
            top = fmaxf(st.m[m], sink2);
            sunk = exp2f(sink2 - top);
        }
        const float shrink = pos >= 0 ? exp2f(st.m[m] - top) : 0.f;
        const float denom = fmaf(column_sum4(st.l[m]), shrink, sunk);        // the four lanes' parts of the column's sum
        const float w = denom > 0.f ? shrink / denom : 0.f;
#pragma unroll
        for (int t = 0; t < DVB; ++t) {
            if (m == 0) o[t] = st.o[0][t] * w;
            else o[t] -= st.o[m][t] * (w * a.lambda);
        }
    }
    if (a.unit_out) {
        float ss = 0.f;
#pragma unroll
        for (int t = 0; t < DVB; ++t)
            if (t * 16 < a.dv)
#pragma unroll
                for (int i = 0; i < 4; ++i) ss = fmaf(o[t][i], o[t][i], ss);
        const float inv = a.out_scale / sqrtf(column_sum4(ss) / (float)a.dv + a.eps);
#pragma unroll
        for (int t = 0; t < DVB; ++t) o[t] *= inv;
    }
    if (pos < 0) return;
#pragma unroll
    for (int t = 0; t < DVB; ++t) {
        if (t * 16 >= a.dv) continue;
        const int e = t * 16 + quad * 4;
        short4v packed;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float v = o[t][i];
            if (a.gate) v = v / (1.f + expf(-a.gate[(size_t)tok * a.gate_stride + a.gate_column + (size_t)head * a.dv + e + i]));
            packed[i] = bits_of((__bf16)v);
        }
        *reinterpret_cast<short4v*>(a.out + ((size_t)tok * a.heads + head) * a.dv + e) = packed;
    }
}

// The order in which workgroups start.  Grid (kv heads; tiles; a layer for every 65,535 tiles): a tile's kv heads are neighbours and the longest
// tiles of all heads come first, so that of the two workgroups of a CU one is long and one short.  Lone tokens, up to one workgroup a CU,
// have nothing of that, and a tile's kv heads, whose keys are neighbours in memory, are read by one XCD (workgroup number % 8):
// grid (tiles; kv heads; zsplits).  us, by heads and by tiles, 16 heads over 4, keys of 64 and values of 128: 64 tokens at 2,048, 256
// workgroups, 51 and 37, 8 at 2,048 20.3 and 15.6 (8 at 191 to 2,047, two maps, 25.5 and 30.6: shares of a long token on one XCD); keys and
// values of 128, 64 tokens at 511 to 8,000: heads over 8, 512 workgroups, 180 and 292, over 16 288 and 507.
constexpr int MB_GRID = 65535;

template <int DSTEPS, int DVB, int MAPS>
__global__ __launch_bounds__(MB_THREADS) void masked_attention_bf16_kernel(MaskedArgs a) {
    __shared__ float meet[MB_WAVES - 1][kWave][DVB * 4 + 2];
    const int tile_at = a.at_once ? blockIdx.x : blockIdx.y + blockIdx.z * MB_GRID;
    const int g = a.at_once ? blockIdx.y : blockIdx.x, z = a.at_once ? blockIdx.z : 0;
    if (tile_at >= a.num_tiles) return;
    const int* tile = a.tiles + 4 * tile_at;
    const int t0 = tile[0], n = tile[1], r = tile[2], p0 = tile[3];
    const int group = a.heads / a.kv_heads;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x & (kWave - 1), col = lane & 15;
    const int* table = a.block_table + (size_t)r * a.max_blocks;
    auto first_key = [&](int p) {
        int lo = 0;
        if (a.chunk > 0) lo = p - p % a.chunk;
        if (a.window > 0) lo = max(lo, p - a.window + 1);
        return lo;
    };
    const bool lone = n == 1;
    const int zsplits = lone ? a.zsplits : 1;
    if (!lone && (z > 0 || a.lone_only)) return;
    // head places of a pass (a power of two up to the waves), and the waves that share a place's keys
    int places = 1;
    if (!lone)
        while (places < group && places < MB_WAVES) places *= 2;
    const int splits = MB_WAVES / places;
    const int place = wave % places, split = wave / places;
    // the kept blocks, then those from the first token's first key to the last token
    const BlockList blocks = block_list(a.keep, first_key(p0) / 16, (p0 + n - 1) / 16);
    // what every token of the tile sees: from the last token's first key to the first token (a column without a token
    // or head computes on zeros there and is never written)
    const int seen_from = first_key(p0 + n - 1), seen_to = p0;
    const int heads_a_pass = lone ? 16 : places;
    ColumnState<DVB, MAPS> st;
    for (int h0 = 0; h0 < group; h0 += heads_a_pass) {
        // the lane's column: a token of the tile for the wave's head, or a head of the group for the lone token
        const int hh = lone ? h0 + col : h0 + place;
        const bool on = hh < group && (lone || col < n);
        const int head = g * group + (hh < group ? hh : 0);
        const int tok = lone ? t0 : t0 + (col < n ? col : 0);
        const int pos = on ? (lone ? p0 : p0 + col) : -1;
        const int lo = on ? first_key(pos) : 0;
        const bool wave_on = lone || h0 + place < group;
        if (wave_on)
            attend_blocks<DSTEPS, DVB, MAPS>(st, a, g, tok, head, pos, lo, table, blocks, z * splits + split,
                                             splits * zsplits, seen_from, seen_to, lane);
        if (splits > 1) {
#pragma unroll
            for (int m = 0; m < MAPS; ++m) {
                __syncthreads();            // the rows of the map before this one have been taken in
                if (split > 0 && wave_on) {
                    float* mine = meet[wave - places][lane];
                    mine[0] = st.m[m];
                    mine[1] = st.l[m];
#pragma unroll
                    for (int t = 0; t < DVB; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i) mine[2 + t * 4 + i] = st.o[m][t][i];
                }
                __syncthreads();
                if (split == 0 && wave_on)
                    for (int w = 1; w < splits; ++w) {          // in the waves' order
                        const float* its = meet[place + w * places - places][lane];
                        const float m_new = fmaxf(st.m[m], its[0]);
                        const float base = m_new == -INFINITY ? 0.f : m_new;
                        const float mine_by = exp2f(st.m[m] - base), its_by = exp2f(its[0] - base);
                        st.l[m] = fmaf(st.l[m], mine_by, its[1] * its_by);
#pragma unroll
                        for (int t = 0; t < DVB; ++t)
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                st.o[m][t][i] = fmaf(st.o[m][t][i], mine_by, its[2 + t * 4 + i] * its_by);
                        st.m[m] = m_new;
                    }
            }
        }
        if (split == 0 && wave_on) {
            if (zsplits > 1) {
                const int passes = (group + 15) / 16;
                // [share][lane][map][numbers]: a lane's numbers in a row, which it reads back in wide loads
                float* mine = a.shares + ((((size_t)tile_at * a.kv_heads + g) * passes + h0 / 16) * zsplits + z)
                                             * kWave * MAPS * share_floats<DVB>() + (size_t)lane * MAPS * share_floats<DVB>();
#pragma unroll
                for (int m = 0; m < MAPS; ++m) {
                    mine[m * share_floats<DVB>()] = st.m[m];
                    mine[m * share_floats<DVB>() + 1] = st.l[m];
#pragma unroll
                    for (int t = 0; t < DVB; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i) mine[m * share_floats<DVB>() + 2 + t * 4 + i] = st.o[m][t][i];
                }
            } else {
                finish_column<DVB, MAPS>(st, a, tok, head, pos, lane);
            }
        }
    }
}

// Tiles of several tokens with their keys and values staged through LDS: all waves of the workgroup walk the same
// stage, which is fetched once for all of them, the next one or two stages travelling through registers while this one is
// worked on; LDS holds two stages, so that one barrier a stage is enough.  A stage is `wave_blocks` blocks of 16 keys for every wave that shares a head's keys (one wave a head, or two
// where the group has four heads or fewer): two blocks a wave where a thread's share of a stage is two 16-byte pieces
// of keys and two of values at most, so that a stage's work outlasts the next one's trip from memory; else one.  Keys
// lie in LDS as rows with 16 bytes of padding, values transposed (a value entry's keys of the stage in a row, 16 bytes
// of padding): every operand is one read without bank conflicts.  Lone tokens are left to the kernel above.
//
// One workgroup is what a CU has room for, so nothing hides what its eight waves wait for together: with one stage in LDS, its pages
// looked up as scalars in the chain of the stage's loads, and addresses and places worked out by every thread for every stage, a stage
// took 3.5 us, a sixth of it products.  us, 16 heads over 4, then and now: 2,048 tokens, 128, 128 105 and 75, with the bias 119 and 78, with
// the cap 124 and 84, with both 139 and 95, two maps of 64 120 and 99, with the bias 133 and 105, 64, 64 78 and 53; 16 over 16, 64, 64 147 and 110;
// 576 tokens after 2,048, 128, 128 117 and 78.  (Scores of a standard deviation of one.  In a whole step between products, whose scores spread
// more and whose power the matrix cores have used up, two maps 110 and one with the bias 97.)
// What is left is the operands' way from LDS (16 KB a wave and stage for 16 columns), the scores and the barrier one after the other.
constexpr int MB_STAGE_BLOCKS = 2;

// PAIRS: a wave takes its two blocks of a stage at once.  That needs room for both blocks' operands in registers (MB_ROOM), and those
// take waves off a SIMD: two are left of four with keys and values of 64.  It pays where the products over values are most of the work
// (MB_VALUES: keys and values of 128, 128 1.09 times as fast, 64, 128 1.04, 64, 64 in two maps 1.04), and elsewhere where four heads or more
// share the waves' stage (64, 64 and 64, 32 1.03 over 4 of 16 heads, 32, 32 over 1 of 8 1.07).  With fewer the waves are what is missing, for
// one head leaves half of them idle: 16 heads over 16, 576 to 2,048 tokens after up to 3,000: 64, 64 and 64, 32 0.66 times as fast, 128, 32 0.70;
// over 8, 64, 64 0.75; and 128, 64 in two maps 0.94 with any number.
template <int DSTEPS, int DVB, int MAPS>
constexpr bool MB_ROOM = 2 * MAPS * DSTEPS * 4 + 2 * DVB * 2 + MAPS * DVB * 4 + MAPS * DSTEPS * 4 <= 160;
template <int DSTEPS, int DVB, int MAPS>
constexpr bool MB_VALUES = DVB == 8 || (DVB == 4 && MAPS * DSTEPS == 4);

// The places in LDS are those of the largest stage that a kernel is built for, in bytes.
constexpr int MB_MOST_BLOCKS = 2 * MB_STAGE_BLOCKS, MB_VALUE_PITCH = MB_MOST_BLOCKS * 32 + 16;
constexpr int mb_key_pitch(int dsteps, int maps) { return dsteps * 64 * maps + 16; }
constexpr int mb_stage_bytes(int dsteps, int dvb, int maps) {
    return MB_MOST_BLOCKS * 16 * mb_key_pitch(dsteps, maps) + dvb * 16 * MB_VALUE_PITCH;
}

template <int FORM, int DSTEPS, int DVB, int MAPS, bool PAIRS>
__global__ __launch_bounds__(MB_THREADS) void masked_attention_bf16_staged_kernel(MaskedArgs a) {
    extern __shared__ __align__(16) unsigned char staged[];       // a stage; afterwards where split key ranges meet
    float (*meet)[kWave][DVB * 4 + 2] = reinterpret_cast<float (*)[kWave][DVB * 4 + 2]>(staged);
    const int tile_at = blockIdx.y + blockIdx.z * MB_GRID;
    if (tile_at >= a.num_tiles) return;
    const int* tile = a.tiles + 4 * tile_at;
    const int t0 = tile[0], n = tile[1], r = tile[2], p0 = tile[3];
    if (n == 1) return;
    const int g = blockIdx.x, group = a.heads / a.kv_heads;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x & (kWave - 1), col = lane & 15, quad = lane >> 4;
    const int* table = a.block_table + (size_t)r * a.max_blocks;
    auto first_key = [&](int p) {
        int lo = 0;
        if (a.chunk > 0) lo = p - p % a.chunk;
        if (a.window > 0) lo = max(lo, p - a.window + 1);
        return lo;
    };
    int places = 1;
    while (places < group && places < MB_WAVES) places *= 2;
    const int splits = min(MB_WAVES / places, MB_STAGE_BLOCKS);      // waves that share a head's keys
    const int place = wave % places, split = wave / places;
    const BlockList blocks = block_list(a.keep, first_key(p0) / 16, (p0 + n - 1) / 16);
    const int stage_blocks = splits * a.wave_blocks;
    const int stages = (blocks.count + stage_blocks - 1) / stage_blocks;
    const int seen_from = first_key(p0 + n - 1);        // every token of the tile sees the keys from here to p0
    const bool full_sizes = a.d == DSTEPS * 32 && a.dv == DVB * 16;
    const int d_all = MAPS * a.d;                               // a key row's entries of this kv head
    constexpr int K_PITCH = mb_key_pitch(DSTEPS, MAPS), K_BYTES = MB_MOST_BLOCKS * 16 * K_PITCH, STAGE_BYTES = mb_stage_bytes(DSTEPS, DVB, MAPS);
    const size_t k_row = (size_t)a.kv_heads * d_all;
    constexpr int PIECES = 2;                                   // a thread's pieces of each kind at most
    constexpr int SETS = (MAPS == 2 && DVB == 8) || (MAPS == 1 && !PAIRS) ? 1 : 2;    // stages on their way in registers: two if there is room
    // Where operands and sums leave next to no registers, what a pass over a group's heads needs at its start and at its end is worked out there and
    // not kept through the stages: two maps of 64, values of 128 had 20 to 72 bytes of scratch a lane (2,048 tokens, 16 heads over 4, with the bias 110 us, 103
    // so; without 96.7 and 97.4).  Elsewhere it is kept: one map of 128, 128 68.7 us, and 70 worked out anew.
    constexpr bool FULL = PAIRS && MAPS == 2 && DVB == 8;
    typedef int int4v __attribute__((ext_vector_type(4)));
    struct Pieces { int4v k[PIECES], v[PIECES]; };
    // A thread's places in a stage are counted in units that the build knows (KP pieces a key row, DVB * 32 pieces a
    // block of values: no division by a size that only the launch knows); places beyond the real sizes stay empty.  A
    // block has a whole number of waves' pieces, so a wave's pieces lie in one block each: its page is looked up, and
    // its place in memory worked out, once for the wave (in scalar registers); the thread's offset from there, and
    // where its piece goes in LDS, are the same for every stage.
    constexpr int KP = DSTEPS * 4 * MAPS, VP = DVB * 32;
    static_assert(16 * KP % kWave == 0 && VP % kWave == 0, "a wave's pieces lie in one block");
    static_assert(MB_THREADS % (16 * KP) == 0 && MB_THREADS % VP == 0, "a thread's pieces are the same ones of other blocks");
    constexpr int K_STEP = MB_THREADS / (16 * KP), V_STEP = MB_THREADS / VP;         // blocks from a thread's piece to its next
    const int k_block = wave * kWave / (16 * KP), v_block = wave * kWave / VP;
    const int key = threadIdx.x / KP, piece = threadIdx.x % KP, row = threadIdx.x % VP >> 1, half = threadIdx.x & 1;
    const bool k_real = piece * 8 < d_all, v_real = row < a.dv;
    const int k_from = (int)((key & 15) * k_row) + piece * 8, v_from = row * a.page_size + half * 8;
    const int k_to = key * K_PITCH + piece * 16, v_to = K_BYTES + row * MB_VALUE_PITCH + v_block * 32 + half * 16;
    // The pages' numbers: a lane holds the one of the walk's block 64 c + lane, 64 blocks at a time, the next 64 asked for while these
    // are walked.  (Read as scalars when they are needed they would be waited for at the next operand from LDS: both count there.)
    auto pages_of = [&](int first, int of_lane) {
        const int block = blocks.block(min(first + of_lane, blocks.count - 1));
        return table[a.page_size == 16 ? block : block * 16 / a.page_size];
    };
    int pages_now = 0, pages_next = 0;
    struct Places { int k_page[PIECES], k_within[PIECES], v_page[PIECES], v_within[PIECES]; };       // of the wave
    auto look_up = [&](int stage, Places& of) {                 // stages in their order; stage_blocks divides 64
        const int first = stage * stage_blocks;
        if (first > 0 && first % kWave == 0 && first < blocks.count) {
            pages_now = pages_next;
            pages_next = pages_of(first + kWave, lane);
        }
        auto one = [&](int blk, int& page, int& within) {
            const int at = first + blk;
            page = blk < stage_blocks && at < blocks.count ? __builtin_amdgcn_readlane(pages_now, at % kWave) : -1;
            within = a.page_size == 16 ? 0 : blocks.block(at) * 16 % a.page_size;
        };
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            one(k_block + u * K_STEP, of.k_page[u], of.k_within[u]);
            one(v_block + u * V_STEP, of.v_page[u], of.v_within[u]);
        }
    };
    auto fetch = [&](const Places& of, Pieces& to) {
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            if (of.k_page[u] >= 0) {
                const bf16* from = a.k_cache + ((size_t)of.k_page[u] * a.page_size + of.k_within[u]) * k_row + (size_t)g * d_all;
                if (k_real) to.k[u] = *reinterpret_cast<const int4v*>(from + k_from);
            }
            if (of.v_page[u] >= 0) {
                const bf16* from = a.v_cache + ((size_t)of.v_page[u] * a.kv_heads + g) * a.dv * a.page_size + of.v_within[u];
                if (v_real) to.v[u] = *reinterpret_cast<const int4v*>(from + v_from);
            }
        }
    };
    auto store = [&](unsigned char* stage_at, const Pieces& from) {
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            if (k_block + u * K_STEP < stage_blocks && k_real) *reinterpret_cast<int4v*>(stage_at + k_to + u * K_STEP * 16 * K_PITCH) = from.k[u];
            if (v_block + u * V_STEP < stage_blocks && v_real) *reinterpret_cast<int4v*>(stage_at + v_to + u * V_STEP * 32) = from.v[u];
        }
    };
    ColumnState<DVB, MAPS> st;
    for (int h0 = 0; h0 < group; h0 += places) {
        int lane_now = lane;
        if constexpr (FULL) asm volatile("" : "+v"(lane_now));
        const int col_now = lane_now & 15;
        const int hh = h0 + place;
        const bool wave_on = hh < group && split < splits;
        const bool on = wave_on && col_now < n;
        const int head = g * group + (hh < group ? hh : 0);
        const int tok = t0 + (col_now < n ? col_now : 0);
        const int pos = on ? p0 + col_now : -1;
        const int lo = (FULL ? pos >= 0 : on) ? first_key(pos) : 0;
        bf16x8 bq[MAPS][DSTEPS];
        load_queries<DSTEPS, MAPS>(bq, a, tok, head, pos, lane_now);
        const float bias1 = (a.r1 && pos >= 0) ? a.r1[head] : 0.f, bias2 = (a.r1 && pos >= 0) ? a.r2[head] : 0.f;
        clear_state<DVB, MAPS>(st);
        Places ahead;
        Pieces first, second;
        pages_now = pages_of(0, lane_now);
        pages_next = pages_of(kWave, lane_now);
        look_up(0, ahead);
        fetch(ahead, first);
        look_up(1, ahead);
        if (SETS == 2) {
            fetch(ahead, second);
            look_up(2, ahead);
        }
        __syncthreads();                    // the pass before this one has read its last stage
        store(staged, first);
        if (SETS == 1) {
            fetch(ahead, first);
            look_up(2, ahead);
        }
        __syncthreads();
        // `free` takes the stage after the next; `next` holds the next one, which goes to the other half of LDS
        auto work = [&](int stage, Pieces& free, const Pieces& next) {
            const unsigned char* here = staged + (stage & 1) * STAGE_BYTES;
            if (SETS == 1 && stage + 1 < stages) store(staged + (~stage & 1) * STAGE_BYTES, next);
            fetch(ahead, free);
            look_up(stage + 3, ahead);
            auto operands = [&](int blk, bf16x8 (&ka)[MAPS][DSTEPS], short4v (&va)[DVB]) {
                const unsigned char* krow = here + (blk * 16 + col) * K_PITCH + quad * 16;
                const unsigned char* vrow = here + K_BYTES + col * MB_VALUE_PITCH + blk * 32 + quad * 8;
                if (full_sizes) {           // the sizes the kernel is built for: no operand has empty places
#pragma unroll
                    for (int m = 0; m < MAPS; ++m)
#pragma unroll
                        for (int i = 0; i < DSTEPS; ++i)
                            ka[m][i] = *reinterpret_cast<const bf16x8*>(krow + (m * DSTEPS * 32 + i * 32) * 2);
#pragma unroll
                    for (int t = 0; t < DVB; ++t) va[t] = *reinterpret_cast<const short4v*>(vrow + t * 16 * MB_VALUE_PITCH);
                } else {
#pragma unroll
                    for (int m = 0; m < MAPS; ++m)
#pragma unroll
                        for (int i = 0; i < DSTEPS; ++i) {
                            const int e = i * 32 + quad * 8;
#pragma unroll
                            for (int x = 0; x < 8; ++x) ka[m][i][x] = (__bf16)0.f;
                            if (e < a.d) ka[m][i] = *reinterpret_cast<const bf16x8*>(krow + (m * a.d + i * 32) * 2);
                        }
#pragma unroll
                    for (int t = 0; t < DVB; ++t) {
                        va[t] = short4v{0, 0, 0, 0};
                        if (t * 16 < a.dv) va[t] = *reinterpret_cast<const short4v*>(vrow + t * 16 * MB_VALUE_PITCH);
                    }
                }
            };
            auto seen = [&](int b) { return (b * 16 >= seen_from || b * 16 + 15 < a.keep) && b * 16 + 15 <= p0; };
            const int at0 = stage * stage_blocks + split, at1 = at0 + splits;       // this wave's one or two blocks of the stage
            bool done = false;
            if constexpr (PAIRS) {
                done = wave_on && a.wave_blocks == 2 && at1 < blocks.count;
                if (done) {
                    const int b0 = blocks.block(at0), b1 = blocks.block(at1);
                    bf16x8 ka[2][MAPS][DSTEPS];
                    short4v va[2][DVB];
                    operands(split, ka[0], va[0]);
                    operands(splits + split, ka[1], va[1]);
                    block_step<FORM, 2, DSTEPS, DVB, MAPS>(st, a, bq, ka, va, {b0 * 16, b1 * 16}, pos, lo, bias1, bias2, {seen(b0), seen(b1)}, lane);
                }
            }
            if (!done && wave_on) {
                for (int at = at0, blk = split; at < min(stage * stage_blocks + stage_blocks, blocks.count); at += splits, blk += splits) {
                    const int b0 = blocks.block(at);
                    bf16x8 ka[1][MAPS][DSTEPS];
                    short4v va[1][DVB];
                    operands(blk, ka[0], va[0]);
                    block_step<FORM, 1, DSTEPS, DVB, MAPS>(st, a, bq, ka, va, {b0 * 16}, pos, lo, bias1, bias2, {seen(b0)}, lane);
                }
            }
            if (SETS == 2 && stage + 1 < stages) store(staged + (~stage & 1) * STAGE_BYTES, next);
            __syncthreads();                    // every wave has read this stage and written its part of the next
        };
        if constexpr (SETS == 2) {
            for (int stage = 0; stage < stages; stage += 2) {
                work(stage, first, second);
                if (stage + 1 < stages) work(stage + 1, second, first);
            }
        } else {
            for (int stage = 0; stage < stages; ++stage) work(stage, first, first);
        }
        int lane_then = lane;
        if constexpr (FULL) asm volatile("" : "+v"(lane_then));
        const int col_then = lane_then & 15;
        if (splits > 1) {
#pragma unroll
            for (int m = 0; m < MAPS; ++m) {
                __syncthreads();
                if (split == 1 && wave_on) {
                    float* mine = meet[place][lane_then];
                    mine[0] = st.m[m];
                    mine[1] = st.l[m];
#pragma unroll
                    for (int t = 0; t < DVB; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i) mine[2 + t * 4 + i] = st.o[m][t][i];
                }
                __syncthreads();
                if (split == 0 && wave_on) {
                    const float* its = meet[place][lane_then];
                    const float m_new = fmaxf(st.m[m], its[0]);
                    const float base = m_new == -INFINITY ? 0.f : m_new;
                    const float mine_by = exp2f(st.m[m] - base), its_by = exp2f(its[0] - base);
                    st.l[m] = fmaf(st.l[m], mine_by, its[1] * its_by);
#pragma unroll
                    for (int t = 0; t < DVB; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i) st.o[m][t][i] = fmaf(st.o[m][t][i], mine_by, its[2 + t * 4 + i] * its_by);
                    st.m[m] = m_new;
                }
            }
        }
        if (split == 0 && wave_on) {
            if constexpr (FULL)
                finish_column<DVB, MAPS>(st, a, t0 + (col_then < n ? col_then : 0), head, col_then < n ? p0 + col_then : -1, lane_then);
            else
                finish_column<DVB, MAPS>(st, a, tok, head, pos, lane_then);
        }
    }
}

// One wave per lone token and kv head: the workgroups' shares taken in, in their order; then the columns' end.
template <int DVB, int MAPS>
__global__ __launch_bounds__(kWave) void masked_attention_bf16_join_kernel(MaskedArgs a) {
    const int tile_at = blockIdx.x;
    const int* tile = a.tiles + 4 * tile_at;
    const int t0 = tile[0], n = tile[1], p0 = tile[3];
    if (n != 1) return;
    const int g = blockIdx.y, group = a.heads / a.kv_heads, lane = threadIdx.x, col = lane & 15;
    const int passes = (group + 15) / 16;
    for (int h0 = 0; h0 < group; h0 += 16) {
        const bool on = h0 + col < group;
        const int head = g * group + (on ? h0 + col : 0);
        ColumnState<DVB, MAPS> st;
#pragma unroll
        for (int m = 0; m < MAPS; ++m) {
            st.m[m] = -INFINITY;
            st.l[m] = 0.f;
#pragma unroll
            for (int t = 0; t < DVB; ++t) st.o[m][t] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
        for (int z = 0; z < a.zsplits; ++z) {
            const float* its = a.shares + ((((size_t)tile_at * a.kv_heads + g) * passes + h0 / 16) * a.zsplits + z)
                                              * kWave * MAPS * share_floats<DVB>() + (size_t)lane * MAPS * share_floats<DVB>();
#pragma unroll
            for (int m = 0; m < MAPS; ++m) {
                const float* row = its + m * share_floats<DVB>();
                const float m_new = fmaxf(st.m[m], row[0]);
                const float base = m_new == -INFINITY ? 0.f : m_new;
                const float mine_by = exp2f(st.m[m] - base), its_by = exp2f(row[0] - base);
                st.l[m] = fmaf(st.l[m], mine_by, row[1] * its_by);
#pragma unroll
                for (int t = 0; t < DVB; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) st.o[m][t][i] = fmaf(st.o[m][t][i], mine_by, row[2 + t * 4 + i] * its_by);
                st.m[m] = m_new;
            }
        }
        finish_column<DVB, MAPS>(st, a, t0, head, on ? p0 : -1, lane);
    }
}

}  // namespace lc

using namespace lc;

static thread_local int g_staged = 1;

// Tests and tuning: whether tiles of several tokens may take the kernel that stages keys and values in LDS (for the
// calling thread).  Returns the setting before.
LC_API int lc_masked_attention_bf16_staged(int on) {
    const int before = g_staged;
    if (on >= 0) g_staged = on ? 1 : 0;
    return before;
}

// Whether the matrix-core kernel takes these sizes (else the general kernel serves them).
LC_API int lc_masked_attention_bf16_supported(int d, int dv, int page_size, int maps) {
    return d > 0 && d % 8 == 0 && d <= 128 && dv > 0 && dv % 16 == 0 && dv <= 128 && page_size > 0 && page_size % 16 == 0
           && (maps == 1 || maps == 2);
}

// float32 words of workspace for a step of `num_tiles` lone tokens whose keys are shared out over `zsplits` workgroups
LC_API long long lc_masked_attention_bf16_workspace(int num_tiles, int heads, int kv_heads, int maps, int dv, int zsplits) {
    if (num_tiles <= 0 || kv_heads <= 0 || heads % kv_heads || zsplits <= 1) return 0;
    const int dvb = dv <= 32 ? 2 : (dv <= 64 ? 4 : 8), passes = (heads / kv_heads + 15) / 16;
    return (long long)num_tiles * kv_heads * passes * zsplits * kWave * maps * (dvb * 4 + 2);
}

// tiles int32 [num_tiles, 4]: first token row, tokens (1..16), request, first position.  zsplits > 1 (a step of lone
// tokens only): every token's key blocks are shared out over that many workgroups, through `shares`
// (lc_masked_attention_bf16_workspace words)
LC_API int lc_masked_attention_bf16(const void* q, const void* k_cache, const void* v_cache, const int* tiles,
                                    int num_tiles, const int* block_table, int max_blocks, int page_size, int heads,
                                    int kv_heads, int maps, int d, int dv, float scale, int chunk, int window,
                                    int keep, float cap, const float* r1, const float* r2, const float* sink, float lambda, int unit_out,
                                    float eps, float out_scale, const float* gate, int gate_stride, int gate_column,
                                    void* out, float* shares, int zsplits, int any_portion, int any_lone,
                                    hipStream_t stream) {
    LC_CHECK(zsplits >= 1 && zsplits <= 64 && (zsplits == 1 || shares), "masked attention: bad shares");
    LC_CHECK(num_tiles >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && max_blocks > 0,
             "masked attention: bad sizes");
    LC_CHECK(lc_masked_attention_bf16_supported(d, dv, page_size, maps),
             "masked attention on the matrix cores: sizes d=%d dv=%d page=%d maps=%d are not taken", d, dv, page_size, maps);
    if (num_tiles == 0) return 0;
    LC_CHECK(q && k_cache && v_cache && tiles && block_table && out, "masked attention: null pointer");
    LC_CHECK((r1 == nullptr) == (r2 == nullptr), "masked attention: the bias needs both of its vectors");
    LC_CHECK(kv_heads <= 65535, "masked attention: too many kv heads");
    LC_CHECK(chunk >= 0 && window >= 0 && keep >= 0 && cap >= 0.f, "masked attention: bad mask or cap");
    MaskedArgs a{(const bf16*)q, (const bf16*)k_cache, (const bf16*)v_cache, tiles, num_tiles, block_table, max_blocks, page_size,
                 heads, kv_heads, d, dv, scale * LOG2E, chunk, window, keep, cap, cap * LOG2E, r1, r2, sink, lambda, unit_out, eps, out_scale, gate,
                 gate_stride, gate_column, (bf16*)out, shares, zsplits, 0, 1, 0};
    // tiles of several tokens go through the kernel that stages keys and values in LDS where a stage fits a thread's
    // two pieces of each kind
    const int group = heads / kv_heads;
    int places = 1;
    while (places < group && places < MB_WAVES) places *= 2;
    const int sharing = MB_WAVES / places < MB_STAGE_BLOCKS ? MB_WAVES / places : MB_STAGE_BLOCKS;
    const int dsteps_built = (d + 31) / 32 <= 2 ? 2 : 4, dvb_built = dv <= 32 ? 2 : (dv <= 64 ? 4 : 8);
    auto fits = [&](int blocks) {       // a thread's two places of each kind at most, in the units the kernels are built for
        return blocks * 16 * (dsteps_built * 4 * maps) <= 2 * MB_THREADS && blocks * dvb_built * 32 <= 2 * MB_THREADS;
    };
    const bool staged = any_portion && g_staged && fits(sharing);
    a.wave_blocks = fits(2 * sharing) ? 2 : 1;
    size_t staged_lds = 2 * (size_t)mb_stage_bytes(dsteps_built, dvb_built, maps);
    const size_t meet_lds = (size_t)(MB_WAVES / 2) * kWave * (8 * 4 + 2) * sizeof(float);    // the same memory, later
    if (staged_lds < meet_lds) staged_lds = meet_lds;
    a.lone_only = staged ? 1 : 0;
    const bool main_kernel = !staged || any_lone;
    a.at_once = zsplits > 1 || (long long)num_tiles * kv_heads <= device_cus() ? 1 : 0;
    const dim3 portions_grid(kv_heads, num_tiles < MB_GRID ? num_tiles : MB_GRID, (num_tiles + MB_GRID - 1) / MB_GRID);
    const dim3 grid = a.at_once ? dim3(num_tiles, kv_heads, zsplits) : portions_grid;
    const dim3 join_grid(num_tiles, kv_heads);         // on the XCDs that left the shares
    const int dsteps = (d + 31) / 32, dvb = dv / 16;
    const int form = r1 && cap > 0.f ? FORM_ANY : r1 ? FORM_BIAS : cap > 0.f ? FORM_CAP : FORM_PLAIN;
#define LC_MB_STAGED(FORM, DS, VB, MP, PAIRS)                                                                           \
    do {                                                                                                                \
        if (staged_lds > 64 * 1024)                                                                                     \
            LC_CHECK(hipFuncSetAttribute((const void*)masked_attention_bf16_staged_kernel<FORM, DS, VB, MP, PAIRS>,     \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)staged_lds) == hipSuccess,    \
                     "masked attention: %zu bytes of LDS refused", staged_lds);                                         \
        masked_attention_bf16_staged_kernel<FORM, DS, VB, MP, PAIRS><<<portions_grid, MB_THREADS, staged_lds, stream>>>(a); \
    } while (0)
#define LC_MB_FORM(DS, VB, MP, PAIRS)                                               \
    do {                                                                            \
        if (form == FORM_PLAIN) LC_MB_STAGED(FORM_PLAIN, DS, VB, MP, PAIRS);        \
        else if (form == FORM_BIAS) LC_MB_STAGED(FORM_BIAS, DS, VB, MP, PAIRS);     \
        else if (form == FORM_CAP) LC_MB_STAGED(FORM_CAP, DS, VB, MP, PAIRS);       \
        else LC_MB_STAGED(FORM_ANY, DS, VB, MP, PAIRS);                             \
    } while (0)
#define LC_MB_AS(DS, VB, MP)                                                                                            \
    do {                                                                                                                \
        constexpr bool room = MB_ROOM<DS, VB, MP>, always = room && MB_VALUES<DS, VB, MP>, often = room && MP * DS < 8; \
        if constexpr (often && !always) {                                                                               \
            if (staged && group >= 4) LC_MB_FORM(DS, VB, MP, true);                                                     \
            else if (staged) LC_MB_FORM(DS, VB, MP, false);                                                             \
        } else {                                                                                                        \
            if (staged) LC_MB_FORM(DS, VB, MP, always);                                                                 \
        }                                                                                                               \
        if (main_kernel) masked_attention_bf16_kernel<DS, VB, MP><<<grid, MB_THREADS, 0, stream>>>(a);                  \
        if (zsplits > 1) masked_attention_bf16_join_kernel<VB, MP><<<join_grid, kWave, 0, stream>>>(a);                 \
    } while (0)
#define LC_MB(DS, VB)                          \
    do {                                       \
        if (maps == 1) LC_MB_AS(DS, VB, 1);    \
        else LC_MB_AS(DS, VB, 2);              \
    } while (0)
#define LC_MB_DV(DS)                     \
    do {                                 \
        if (dvb <= 2) LC_MB(DS, 2);      \
        else if (dvb <= 4) LC_MB(DS, 4); \
        else LC_MB(DS, 8);               \
    } while (0)
    if (dsteps <= 2) LC_MB_DV(2);
    else LC_MB_DV(4);
#undef LC_MB_DV
#undef LC_MB
#undef LC_MB_AS
#undef LC_MB_FORM
#undef LC_MB_STAGED
    LC_LAUNCH_CHECK("masked_attention_bf16");
    return 0;
}

template <int DSTEPS, int DVB, int MAPS>
static int staged_scratch() {
    constexpr bool room = MB_ROOM<DSTEPS, DVB, MAPS>, always = room && MB_VALUES<DSTEPS, DVB, MAPS>, often = room && MAPS * DSTEPS < 8;
    const void* kernels[] = {
        (const void*)masked_attention_bf16_staged_kernel<FORM_PLAIN, DSTEPS, DVB, MAPS, always>,
        (const void*)masked_attention_bf16_staged_kernel<FORM_BIAS, DSTEPS, DVB, MAPS, always>,
        (const void*)masked_attention_bf16_staged_kernel<FORM_CAP, DSTEPS, DVB, MAPS, always>,
        (const void*)masked_attention_bf16_staged_kernel<FORM_ANY, DSTEPS, DVB, MAPS, always>,
        (const void*)masked_attention_bf16_staged_kernel<FORM_PLAIN, DSTEPS, DVB, MAPS, often || always>,
        (const void*)masked_attention_bf16_staged_kernel<FORM_BIAS, DSTEPS, DVB, MAPS, often || always>,
        (const void*)masked_attention_bf16_staged_kernel<FORM_CAP, DSTEPS, DVB, MAPS, often || always>,
        (const void*)masked_attention_bf16_staged_kernel<FORM_ANY, DSTEPS, DVB, MAPS, often || always>,
    };
    int most = 0;
    for (const void* kernel : kernels) {
        hipFuncAttributes attr;
        if (hipFuncGetAttributes(&attr, kernel) != hipSuccess) {
            (void)hipGetLastError();
            return -1;
        }
        if ((int)attr.localSizeBytes > most) most = (int)attr.localSizeBytes;
    }
    return most;
}

// Bytes of scratch memory a lane of the staged kernels for d (one map's entries), dv and maps that the library was built with; -1: the runtime could not
// be asked.
LC_API int lc_masked_attention_bf16_scratch(int maps, int d, int dv) {
    const int dsteps = (d + 31) / 32, dvb = dv / 16;
#define LC_MB_SCRATCH(DS, VB) (maps == 1 ? staged_scratch<DS, VB, 1>() : staged_scratch<DS, VB, 2>())
    if (dsteps <= 2) return dvb <= 2 ? LC_MB_SCRATCH(2, 2) : dvb <= 4 ? LC_MB_SCRATCH(2, 4) : LC_MB_SCRATCH(2, 8);
    return dvb <= 2 ? LC_MB_SCRATCH(4, 2) : dvb <= 4 ? LC_MB_SCRATCH(4, 4) : LC_MB_SCRATCH(4, 8);
#undef LC_MB_SCRATCH
}
