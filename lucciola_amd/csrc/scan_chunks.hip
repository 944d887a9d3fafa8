// The recurrence of delta_rule.hip,
//     S <- diag(decay) S - removal (probe^T S) + write v^T,    o = S^T read,
// for portions of prompts, a chunk of SC = 32 tokens at a time on the float32 matrix instruction.  Token by token a step
// is a chain of dependent vector instructions, 0.21 us a token without and 0.29 us with the removal term, on a wave that
// is alone on its SIMD (16 heads of 128 x 128: 437 and 580 us for 2,048 tokens whatever the number of heads; here 88 and 168).
//
// Inside a chunk, from the state S that the chunk before left, with a_i the product of the decays of tokens 0..i (key
// channel by key channel), r_ij that of the tokens j+1..i, and y_i = probe_i^T S_(i-1) what token i takes out:
//     y_i = (probe_i a_(i-1))^T S + sum_(j<i) [M_ij v_j - L_ij y_j]    L_ij = probe_i . (r_(i-1)j removal_j), M_ij with write_j
//     o_i = (read_i a_i)^T S + sum_(j<=i) [W_ij v_j - R_ij y_j]        W_ij = read_i . (r_ij write_j),        R_ij with removal_j
// With T = (1 + L)^-1 (unit lower triangular: forward substitution in blocks of 16), Y = T probe~ S + T M V, and put in:
//     O  = (read~ - R T probe~) S + (W - R T M) V
//     S' = diag(a_last) S + (write~^T - removal~^T T M) V - removal~^T (T probe~ S)
// All that does not hold S or V is made first, chunks and heads side by side (scan_chunk_prepare_kernel); then a workgroup
// per 16 value channels and head walks a request's chunks in order (scan_chunk_walk_kernel), with S in the accumulators.
// Everything is float32: operands, products and sums; products of decays are made in 64 bits and rounded once.  Products between
// blocks of 16 tokens are split at the border, where nothing is divided by.  Inside a block there are two ways.  Where no channel's
// decays multiply to less than 2^-60 or more than 2^60 on the way through a block, the writing vectors are divided by what is left of the
// block's decays and the reading ones multiplied, and a block's pairs are one product: the quotients stay far from float32's ends, so they
// add two roundings a factor and no more (constant decays of 2^-3.74, 2^-59.8 a block: 1.9 to 2.2 units of 2^-24 of the result where token by
// token has 1.3 to 1.5).  Elsewhere (a decay of 0, too) a chunk's pairs are made one by one, each decay multiplied in, none divided by
// (2^-3.76: 1.6 to 2.1 units).
// A token's sums are taken in another order than token by token and depend on where its chunk begins, so callers that
// promise the same bits for every cut of a prompt (float32 models) and steps of few tokens keep the other kernel.
// A chunk's products meet every token of the chunk, and zero times infinity is no number.  So a request with a vector of which
// an entry is NaN, infinite or above SC_MOST goes token by token in the second kernel (walk_tokens), and a value that is not
// finite meets no row of W - R T M above its own: such a token reaches what comes behind it and nothing before.
#include "common.h"

#include <type_traits>

namespace lc {

constexpr int SC = 32;                  // tokens of a chunk: two blocks of 16
constexpr float SC_MOST = 0x1p40f;      // above that a chunk's products could overflow where a token's do not
constexpr int SCP = SC + 4;             // floats of a row of a [SC x SC] matrix in LDS: b128 reads of 16 rows meet no bank twice

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// What the first kernel leaves of a chunk and head, in floats: read^ [SC][DK], Z [DK][SC], the chunk's decay [2][DK] (the
// number in 32 bits and what that leaves out: a model's constant decay would be off by the same last bit in every chunk),
// W^ [SC][SC], and with a removal term T probe~ [SC][DK] and -removal~^T [DK][SC].  The matrices lie as the operands that the
// second kernel loads, 1 KB a [16 x 16] tile: lane (row, quad) has entries 4 quad .. + 3 of a row (in rows
// the walk, whose loads then touch sixteen half lines each, took 109 us where it took 95 and, removing, 199 us where 145, in its form with
// four waves; 63 and 98 now).
template <int DK, bool REMOVE>
struct ChunkRecord {
    static constexpr int READ = 0, Z = SC * DK, DECAY = 2 * SC * DK, MIX = DECAY + 2 * DK, PROBE = MIX + SC * SC,
                         REMOVAL = PROBE + SC * DK, SIZE = REMOVE ? REMOVAL + SC * DK : PROBE;
};

// Where the records of request r's chunks begin, for the requests of at least `least` tokens: no two of them share one, whatever
// the lengths.  Behind such a request q / SC has grown by its whole chunks and the other term by one or more, for the rest of it.
// The many lone tokens that a step may hold beside a portion take no record: their places are those that a request behind them has.
__host__ __device__ __forceinline__ int record_place(int q, int r, int least) { return q / SC + min(r, q / least); }
__device__ __forceinline__ int first_record(const int* __restrict__ q_offsets, int r, int least) {
    return record_place(q_offsets[r], r, least);
}

// The [16 x 16] tile A B over 16 KT k, k = 16 t + 4 (lane / 16) + i: a(t) holds four neighbouring k of the lane's row of A, b(t)
// of its column of B, so that rows are read 16 bytes at a time.  A lane gets rows 4 (lane / 16) .. + 3 of column lane % 16,
// which is in the same order what it holds of a B operand of 16 k.  Every t has a sum of its own, added pairwise: the
// matrix instruction adds one product after the other, and the long sums were what set a chunk's error (16 heads of
// 128, float64 beside it: 2.3e-7 of the result with one sum, 1.5e-7 so; token by token 1.4e-7).
template <int KT, class A, class B>
__device__ __forceinline__ f32x4 tile_product(A a, B b) {
    f32x4 c[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) {
        const f32x4 x = a(t), y = b(t);
        c[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) c[t] = mfma4(x[i], y[i], c[t]);
    }
#pragma unroll
    for (int n = KT / 2; n >= 1; n /= 2)
#pragma unroll
        for (int t = 0; t < n; ++t) c[t] += c[t + n];
    return c[0];
}

// A record of a head is an item; a workgroup takes every gridDim.x-th.  coef [5 or 3][T, heads DK] as delta_rule.hip has it.  alone
// [records][heads][8]: not all zero where the chunk holds what has to go token by token, and its record is not to be used.
// An item asks for the next one's vectors before it makes its pairs, so that loads, products and stores of a CU pass beside each other (with
// a workgroup an item they follow each other; 2,048 tokens, 16 heads of 128 28 -> 21 us, 32 heads 53 -> 40, which is 4.4 TB/s; two workgroups a
// CU, four for heads of 64 without removal, are what its LDS and registers hold and measured best of one to four.  With the walk, before this and the
// walk's loads placed by hand and now: heads of 64, values of 128, 2,048 tokens 73 -> 69 us and, removing, 111 -> 102; 16 portions of 64 tokens 38 -> 35
// and 69 -> 66, 60 of them 107 -> 102 and 204 -> 208, 100 portions of 70 and 4 heads, whose every item looks for its request, 41 -> 36 and 76 -> 68; heads of
// 128, 2,048 tokens 105 -> 88 and 183 -> 168, 60 portions of 64 179 -> 157 and 358 -> 356).  With heads of 128 and
// a removal term a workgroup fills its CU's LDS, has no registers for another item's vectors (29 of them spilled: 66 us against 63) and
// its steps follow each other: 63 us for 2,048 tokens and 16 heads, 16 us an item, whose 155 KB
// in and out take half of that at the rate of a copy.
template <int DK, bool REMOVE> constexpr bool prepare_turns = !(REMOVE && DK == 128);

template <int DK, bool REMOVE, int THREADS>
__global__ __launch_bounds__(THREADS) void scan_chunk_prepare_kernel(const float* __restrict__ coef,
                                                                     const int* __restrict__ q_offsets, int R, int T,
                                                                     int heads, int least, int items, float* __restrict__ records,
                                                                     unsigned char* __restrict__ alone) {
    typedef ChunkRecord<DK, REMOVE> Rec;
    constexpr bool TURNS = prepare_turns<DK, REMOVE>;
    constexpr int DKP = DK + 4, WAVES = THREADS / kWave, NP = REMOVE ? 5 : 3;
    constexpr int DECAY = 0, PROBE = 1, REMOVAL = 2, WRITE = REMOVE ? 3 : 1, READ = REMOVE ? 4 : 2;
    constexpr int MATS = REMOVE ? 4 : 1;                    // W = read x write, R = read x removal, M = probe x write, L = probe x removal
    __shared__ __attribute__((aligned(16))) float plane[NP][SC][DKP];
    __shared__ __attribute__((aligned(16))) float mat[MATS][SC][SCP];
    __shared__ __attribute__((aligned(16))) float inverse[REMOVE ? SC : 1][SCP], scratch[REMOVE ? 16 : 1][20];
    __shared__ __attribute__((aligned(16))) float total[2][DK];     // a block's decay
    __shared__ double whole[2][DK];
    __shared__ int far_waves[WAVES];
    // only LDS has to be in order between the waves: loads and stores of memory stay in flight
    auto meet = []() {
        asm volatile("" ::: "memory");
        wait_lgkmcnt<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // where an item's chunk begins and its tokens; 0: the record is nobody's
    struct Chunk { int record, head, t0, count; };
    auto chunk_of = [&](int item) {
        Chunk c{item / heads, item % heads, 0, 0};
        int low = 0, high = R - 1;                          // the request whose records hold this one
        while (low < high) {
            const int mid = (low + high + 1) / 2;
            if (first_record(q_offsets, mid, least) <= c.record) low = mid;
            else high = mid - 1;
        }
        const int last = q_offsets[low + 1];
        c.t0 = q_offsets[low] + (c.record - first_record(q_offsets, low, least)) * SC;
        if (c.t0 < last && last - q_offsets[low] >= least) c.count = min(SC, last - c.t0);
        return c;
    };
    // the chunk's vectors; a place behind the request's end keeps the state and adds nothing
    constexpr int PIECES = NP * SC * (DK / 4) / THREADS, TOKENS = THREADS / (DK / 4);        // 16 bytes each; tokens a pass of all threads
    static_assert(SC % TOKENS == 0 && PIECES * TOKENS == NP * SC, "whole passes, each within a plane");
    f32x4 held[PIECES];
    auto ask = [&](const Chunk& c) {
        const int tid = threadIdx.x;
        const float* from = coef + ((size_t)c.t0 * heads + c.head) * DK;
        asm volatile("" : "+s"(from));
        const int t = tid / (DK / 4);
#pragma unroll
        for (int n = 0; n < PIECES; ++n) {
            const int p = n * TOKENS / SC, first = n * TOKENS % SC;
            const float pad = p == DECAY ? 1.f : 0.f;
            held[n] = f32x4{pad, pad, pad, pad};
            const float* row = from + ((size_t)p * T + first) * heads * DK;
            if (first + t < c.count) held[n] = *reinterpret_cast<const f32x4*>(row + (unsigned)(t * heads * DK + tid % (DK / 4) * 4));
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    Chunk chunk = chunk_of(blockIdx.x);
    ask(chunk);
    for (int item = blockIdx.x; item < items; item += gridDim.x) {
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));                           // places in LDS are worked out when they are wanted: kept for all turns they spill
        const int wave = tid / kWave, lane = tid % kWave, row = lane & 15, quad = lane >> 4;
        const int record = chunk.record, head = chunk.head, count = chunk.count;
        auto ask_next = [&]() {
            if (TURNS && item + (int)gridDim.x < items) {
                chunk = chunk_of(item + gridDim.x);
                ask(chunk);
            }
        };
        if (count == 0) {
            ask_next();
            continue;
        }
        float* out = records + ((size_t)record * heads + head) * Rec::SIZE;
        meet();                                                 // nobody reads the chunk before any more
        unsigned most = 0;                                      // the largest entry's bits: NaN and infinity lie above all numbers
#pragma unroll
        for (int n = 0; n < PIECES; ++n) {
#pragma unroll
            for (int e = 0; e < 4; ++e) most = max(most, __float_as_uint(held[n][e]) & 0x7FFFFFFFu);
            *reinterpret_cast<f32x4*>(&plane[n * TOKENS / SC][n * TOKENS % SC + tid / (DK / 4)][tid % (DK / 4) * 4]) = held[n];
        }
        const bool odd = __builtin_amdgcn_ballot_w64(most > __float_as_uint(SC_MOST)) != 0;
        if (lane < 8 / WAVES) alone[((size_t)record * heads + head) * 8 + wave * (8 / WAVES) + lane] = odd;
        meet();

        // every vector at its block's border.  A thread is a key channel of a block, and of the reading (read, probe) or the
        // writing side (write, removal); the products of the decays are made in 64 bits and rounded once.
        constexpr int SIDES = THREADS / (2 * DK);
        static_assert(SIDES >= 1, "a thread a channel of a block");
        const int block = tid / DK % 2, channel = tid % DK, side = tid / (2 * DK);
        float decay[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) decay[i] = plane[DECAY][16 * block + i][channel];
        double through = 1.0, least_through = 1.0, most_through = 1.0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            through *= (double)decay[i];
            least_through = fmin(least_through, through);
            most_through = fmax(most_through, through);
        }
        if (side == 0) {
            whole[block][channel] = through;
            total[block][channel] = (float)through;
        }
        // Where no channel's decays multiply to less than 2^-60 or more than 2^60 anywhere in the 16 tokens, the pairs of a block are
        // products of the vectors times and over the decays from the block's first token on, on the matrix instruction: a division
        // by what is far from the smallest number loses nothing.  Else the pairs are made one by one, by vector instructions,
        // several times as long.
        const bool far_here = __builtin_amdgcn_ballot_w64(!(least_through >= 0x1p-60 && most_through <= 0x1p60 && through == through)) != 0;
        if (lane == 0) far_waves[wave] = far_here;
        meet();
        bool far = false;
#pragma unroll
        for (int n = 0; n < WAVES; ++n) far |= far_waves[n] != 0;
        far = __builtin_amdgcn_readfirstlane(far);
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        auto put = [&](float (*to)[SCP], int r0, int c0, f32x4 v) {
#pragma unroll
            for (int i = 0; i < 4; ++i) to[r0 + 4 * quad + i][c0 + row] = v[i];
        };
        auto keep_tile = [&](int matrix, int tile, f32x4 v) { *reinterpret_cast<f32x4*>(out + matrix + tile * 256 + lane * 4) = v; };
        // four neighbouring entries of the lane's row of a matrix or plane, and of its column
        auto along = [&](const float* m, int pitch, int r0, int c0) { return *reinterpret_cast<const f32x4*>(m + (r0 + row) * pitch + c0 + 4 * quad); };
        auto down = [&](const float* m, int pitch, int r0, int c0) {
            f32x4 v;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = m[(r0 + 4 * quad + i) * pitch + c0 + row];
            return v;
        };
        if (far) {
            // lane (j, quad) carries write_j and removal_j through the decays of the tokens behind j, for every fourth group of
            // four key channels, and meets read_i or probe_i (which does not see token i's decay) on the way
            constexpr int ROLES = REMOVE ? 4 : 2;               // (block, read or probe)
            constexpr int G = DK / 16;
            static_assert(WAVES >= ROLES, "a wave a role");
            if (wave < ROLES) {
                const int base = 16 * (wave & 1);
                const bool by_probe = wave >= 2;
                f32x4 w[G], x[REMOVE ? G : 1];
#pragma unroll
                for (int m = 0; m < G; ++m) {
                    w[m] = *reinterpret_cast<const f32x4*>(&plane[WRITE][base + row][16 * m + 4 * quad]);
                    if constexpr (REMOVE) x[m] = *reinterpret_cast<const f32x4*>(&plane[REMOVAL][base + row][16 * m + 4 * quad]);
                }
                for (int i = 0; i < 16; ++i) {
                    const int from = by_probe ? i - 1 : i;      // the last decay that the reader sees
                    float with_w = 0.f, with_x = 0.f;
                    const float* by = &plane[REMOVE && by_probe ? PROBE : READ][base + i][4 * quad];
                    const float* keep = &plane[DECAY][base + max(from, 0)][4 * quad];
#pragma unroll
                    for (int m = 0; m < G; ++m) {
                        const f32x4 d = *reinterpret_cast<const f32x4*>(keep + 16 * m), q = *reinterpret_cast<const f32x4*>(by + 16 * m);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float f = from > row ? d[e] : 1.f;
                            w[m][e] *= f;
                            with_w = fmaf(q[e], w[m][e], with_w);
                            if constexpr (REMOVE) {
                                x[m][e] *= f;
                                with_x = fmaf(q[e], x[m][e], with_x);
                            }
                        }
                    }
                    with_w += __shfl_xor(with_w, 16, kWave);
                    with_w += __shfl_xor(with_w, 32, kWave);
                    const bool seen = by_probe ? row < i : row <= i;
                    if (quad == 0) mat[REMOVE && by_probe ? 2 : 0][base + i][base + row] = seen ? with_w : 0.f;
                    if constexpr (REMOVE) {
                        with_x += __shfl_xor(with_x, 16, kWave);
                        with_x += __shfl_xor(with_x, 32, kWave);
                        if (quad == 0) mat[by_probe ? 3 : 1][base + i][base + row] = seen ? with_x : 0.f;
                    }
                }
            }
            meet();
        }
        // far: read and probe from the block's first token on, write and removal to its last; else those over the decays
        auto scale_reading = [&]() {
            double a = 1.0;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if constexpr (REMOVE) plane[PROBE][16 * block + i][channel] *= (float)a;
                a *= (double)decay[i];
                plane[READ][16 * block + i][channel] *= (float)a;
            }
        };
        auto scale_writing = [&]() {
            double a = far ? 1.0 : 1.0 / through;
#pragma unroll
            for (int i = 15; i >= 0; --i) {
                plane[WRITE][16 * block + i][channel] *= (float)a;
                if constexpr (REMOVE) plane[REMOVAL][16 * block + i][channel] *= (float)a;
                a *= (double)decay[i];
            }
        };
        if (side == 0) scale_reading();
        if (side == SIDES - 1) scale_writing();
        meet();

        // pairs between the two blocks (nothing of the second reaches the first), and, unless they are there, inside them
        auto rows_of = [&](int p, int first) { return [&, p, first](int t) { return along(&plane[p][0][0], DKP, first, 16 * t); }; };
        for (int role = wave; role < MATS * 3; role += WAVES) {
            const int m = role % MATS, tile = role / MATS;      // tile 0: between; 1, 2: inside
            const bool probes = REMOVE && m >= 2;
            const int by = probes ? PROBE : READ, with = REMOVE && (m & 1) ? REMOVAL : WRITE;
            if (tile == 0) {
                auto lasting = [&](int t) {
                    f32x4 v = rows_of(with, 0)(t);
                    if (!far) v *= *reinterpret_cast<const f32x4*>(&total[0][16 * t + 4 * quad]);
                    return v;
                };
                put(mat[m], 16, 0, tile_product<DK / 16>(rows_of(by, 16), lasting));
                put(mat[m], 0, 16, zero);
            } else if (!far) {
                const int base = 16 * (tile - 1);
                f32x4 v = tile_product<DK / 16>(rows_of(by, base), rows_of(with, base));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int reader = 4 * quad + i;
                    v[i] = (probes ? row < reader : row <= reader) ? v[i] : 0.f;
                }
                put(mat[m], base, base, v);
            }
        }
        meet();

        ask_next();
        // from the chunk's first token on, and to its last
        for (int idx = tid; idx < 16 * DK; idx += THREADS) {
            const int i = idx / DK, k = idx % DK;
            const float to_border = far ? 1.f : total[0][k], rest = far ? 1.f : total[1][k];
            plane[READ][16 + i][k] *= total[0][k];
            plane[WRITE][i][k] *= to_border * total[1][k];
            plane[WRITE][16 + i][k] *= rest;
            if constexpr (REMOVE) {
                plane[PROBE][16 + i][k] *= total[0][k];
                plane[REMOVAL][i][k] *= to_border * total[1][k];
                plane[REMOVAL][16 + i][k] *= rest;
            }
        }
        for (int k = tid; k < DK; k += THREADS) {
            const double d = whole[0][k] * whole[1][k];
            const float near = (float)d;
            out[Rec::DECAY + k] = near;
            out[Rec::DECAY + DK + k] = (float)(d - (double)near);
        }

        meet();
        constexpr int KEYS = DK / 16, TILES = 2 * KEYS;
        if constexpr (REMOVE) {
            const float *W = mat[0][0], *Rm = mat[1][0], *M = mat[2][0], *L = mat[3][0];
            float* inv = inverse[0];
            // T's diagonal blocks: lane (column, block) by forward substitution
            if (wave == 0 && lane < 32) {
                const int base = lane & 16, c = lane & 15;
                float x[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    float s = i == c ? 1.f : 0.f;
#pragma unroll
                    for (int j = 0; j < i; ++j) s = fmaf(-L[(base + i) * SCP + base + j], x[j], s);
                    x[i] = s;
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    inverse[base + i][base + c] = x[i];
                    if (base) inverse[i][16 + c] = 0.f;
                }
            }
            meet();
            // T10 = -T11 L10 T00
            if (wave == 0) {
                const f32x4 lt = tile_product<1>([&](int) { return along(L, SCP, 16, 0); }, [&](int) { return down(inv, SCP, 0, 0); });
#pragma unroll
                for (int i = 0; i < 4; ++i) scratch[4 * quad + i][row] = -lt[i];
            }
            meet();
            if (wave == 0)
                put(inverse, 16, 0, tile_product<1>([&](int) { return along(inv, SCP, 16, 16); },
                                                    [&](int) { return down(scratch[0], 20, 0, 0); }));
            meet();
            // T M over M's place (kept in registers until everybody has read M); T probe~, transposed, over the decays
            f32x4 tm = zero;
            if (wave < 4)
                tm = tile_product<2>([&](int t) { return along(inv, SCP, 16 * (wave >> 1), 16 * t); },
                                     [&](int t) { return down(M, SCP, 16 * t, 16 * (wave & 1)); });
            for (int tile = wave; tile < TILES; tile += WAVES) {
                const int t0 = 16 * (tile / KEYS), k0 = 16 * (tile % KEYS);
                const f32x4 v = tile_product<2>([&](int t) { return down(plane[PROBE][0], DKP, 16 * t, k0); },
                                                [&](int t) { return along(inv, SCP, t0, 16 * t); });
                *reinterpret_cast<f32x4*>(&plane[DECAY][t0 + row][k0 + 4 * quad]) = v;
                keep_tile(Rec::PROBE, tile, v);
            }
            meet();
            if (wave < 4) put(mat[2], 16 * (wave >> 1), 16 * (wave & 1), tm);
            meet();
            // read^ = read~ - R (T probe~);  Z = write~^T - removal~^T (T M);  W^ = W - R (T M): each transposed, as a lane's entries lie
            for (int tile = wave; tile < TILES; tile += WAVES) {
                const int t0 = 16 * (tile / KEYS), k0 = 16 * (tile % KEYS);
                const f32x4 v = tile_product<2>([&](int t) { return down(plane[DECAY][0], DKP, 16 * t, k0); },
                                                [&](int t) { return along(Rm, SCP, t0, 16 * t); });
                keep_tile(Rec::READ, tile, along(plane[READ][0], DKP, t0, k0) - v);
            }
            for (int tile = wave; tile < TILES; tile += WAVES) {
                const int k0 = 16 * (tile / 2), t0 = 16 * (tile % 2);
                const f32x4 z = tile_product<2>([&](int t) { return down(M, SCP, 16 * t, t0); },
                                                [&](int t) { return down(plane[REMOVAL][0], DKP, 16 * t, k0); });
                keep_tile(Rec::Z, tile, down(plane[WRITE][0], DKP, t0, k0) - z);
                keep_tile(Rec::REMOVAL, tile, -down(plane[REMOVAL][0], DKP, t0, k0));
            }
            if (wave < 4) {
                const int r0 = 16 * (wave >> 1), c0 = 16 * (wave & 1);
                const f32x4 v = tile_product<2>([&](int t) { return down(M, SCP, 16 * t, c0); },
                                                [&](int t) { return along(Rm, SCP, r0, 16 * t); });
                keep_tile(Rec::MIX, wave, along(W, SCP, r0, c0) - v);
            }
        } else {
            for (int tile = wave; tile < TILES; tile += WAVES) {
                keep_tile(Rec::READ, tile, along(plane[READ][0], DKP, 16 * (tile / KEYS), 16 * (tile % KEYS)));
                keep_tile(Rec::Z, tile, down(plane[WRITE][0], DKP, 16 * (tile % 2), 16 * (tile / 2)));
            }
            for (int tile = wave; tile < 4; tile += WAVES) keep_tile(Rec::MIX, tile, along(mat[0][0], SCP, 16 * (tile >> 1), 16 * (tile & 1)));
        }
    }
}

// The recurrence as it stands, for 16 value channels: 32 lanes a channel, DK / 32 key rows a lane.
template <int DK, bool REMOVE>
__device__ __forceinline__ void walk_tokens(const float* __restrict__ coef, const float* __restrict__ v, float* __restrict__ state,
                                            float* __restrict__ out, int first, int last, int slot, int T, int heads, int head,
                                            int dv, int block) {
    constexpr int N = DK / 32, DECAY = 0, PROBE = 1, REMOVAL = 2, WRITE = REMOVE ? 3 : 1, READ = REMOVE ? 4 : 2;
    const int j = block * 16 + threadIdx.x / 32, k0 = threadIdx.x % 32 * N;
    if (j >= dv) return;
    auto over_rows = [](float x) {
        for (int n = 16; n >= 1; n /= 2) x += __shfl_xor(x, n, 32);
        return x;
    };
    float* home = state + (((size_t)slot * heads + head) * dv + j) * DK + k0;
    float S[N];
    for (int i = 0; i < N; ++i) S[i] = home[i];
    for (int t = first; t < last; ++t) {
        const size_t at = ((size_t)t * heads + head) * dv + j;
        const float value = v[at];
        auto entry = [&](int p, int i) { return coef[(((size_t)p * T + t) * heads + head) * DK + k0 + i]; };
        float held = 0.f, o = 0.f;
        if constexpr (REMOVE) {
            for (int i = 0; i < N; ++i) held = fmaf(entry(PROBE, i), S[i], held);
            held = over_rows(held);
        }
        for (int i = 0; i < N; ++i) {
            S[i] *= entry(DECAY, i);
            if constexpr (REMOVE) S[i] = fmaf(-entry(REMOVAL, i), held, S[i]);
            S[i] = fmaf(entry(WRITE, i), value, S[i]);
            o = fmaf(entry(READ, i), S[i], o);
        }
        o = over_rows(o);
        if (k0 == 0) out[at] = o;
    }
    for (int i = 0; i < N; ++i) home[i] = S[i];
}

// One workgroup per (16 value channels, head, request).  Four waves keep S, a quarter of the key rows each, as accumulators
// (KT tiles of 16), which are B operands of the next products as they are, and take it from chunk to chunk; four others make
// the chunks' read-outs from copies of S that the first leave in LDS, a chunk behind.  So a SIMD has two waves, and one's loads,
// LDS trips and address arithmetic pass beside the other's products (with the read-outs made by the waves that keep S, one wave a
// SIMD: 87 us for the 64 chunks of 2,048 tokens, 16 heads of 128 x 128, and 137 us with a removal term; so 76 and 115, and with the
// loads placed by hand, fewer of them and whole lines stored 63 and 98).  What the waves make of their key rows meets in LDS, two
// buffers in turn, one barrier a chunk.  A chunk's record is asked for two chunks ahead, its values, of which each wave brings an
// eighth for all, four.  A chunk takes 1.0 us and, removing, 1.5, of which the matrix cores 0.5 and 0.9; the rest is the chain: a trip
// through LDS to the readers and back, the barrier, and what the loads' 40 or 70 KB keep the CU's way to L2 busy.  Workgroups are
// numbered so that the blocks of one head, which read the same records, run on one XCD (workgroup i on XCD i % 8) where the heads
// are a multiple of 8.
template <int DK, bool REMOVE>
__global__ __launch_bounds__(512) void scan_chunk_walk_kernel(const float* __restrict__ records, const uint2* __restrict__ alone,
                                                              const float* __restrict__ coef, const float* __restrict__ v,
                                                              float* __restrict__ state, float* __restrict__ out,
                                                              const int* __restrict__ q_offsets,
                                                              const int* __restrict__ slot_ids, int T, int heads, int dv, int least) {
    typedef ChunkRecord<DK, REMOVE> Rec;
    constexpr int KT = DK / 64, TT = SC / 16, KEYS = DK / 16;
    __shared__ f32x4 states[2][4][KT][kWave], reads[2][4][TT][kWave], taken[REMOVE ? 2 : 1][4][TT][kWave];
    __shared__ __attribute__((aligned(16))) float shared_value[3][TT * 4][kWave], shared_decay[3][4][2 * 16 * KT];
    const int lane = threadIdx.x % kWave, row = lane & 15, quad = lane >> 4;
    const int all = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), wave = all & 3;
    const bool keeps = all < 4;
    const int head = blockIdx.x % heads, block = blockIdx.x / heads, req = blockIdx.y;
    const int first = q_offsets[req], last = q_offsets[req + 1];
    if (last - first < least) return;
    const int chunks = (last - first + SC - 1) / SC;
    bool by_token = false;
    for (int c = lane; c < chunks; c += kWave) {
        const uint2 waves = alone[(size_t)(first_record(q_offsets, req, least) + c) * heads + head];
        by_token |= (waves.x | waves.y) != 0;
    }
    if (__builtin_amdgcn_ballot_w64(by_token) != 0) {       // in every wave alike
        walk_tokens<DK, REMOVE>(coef, v, state, out, first, last, slot_ids[req], T, heads, head, dv, block);
        return;
    }
    const int j = block * 16 + row;                         // the value channel
    const bool mine = j < dv;                               // a channel behind dv works through the head's first one's values
    const int column = mine ? j : 0;
    const unsigned line = heads * dv;                       // floats from a token's values to the next one's, below 2^23
    const float* values = v + (size_t)first * line + (size_t)head * dv;
    const float* record = records + ((size_t)first_record(q_offsets, req, least) * heads + head) * Rec::SIZE;
    const size_t record_line = (size_t)heads * Rec::SIZE;
    // A chunk's record, and the value that this wave brings for all of them; behind the last chunk the last one's once more.  Entries that
    // lie behind the request's end are zero in the records, so such a token's value (the last token's) only has to be a number.
    auto record_of = [&](int c) {
        const float* rec = record + (size_t)min(c, chunks - 1) * record_line;
        asm volatile("" : "+s"(rec));
        return rec;
    };
    auto tile = [&](const float* rec, int matrix, int n) { return *reinterpret_cast<const f32x4*>(rec + (matrix + n * 256) + (unsigned)lane * 4); };
    static_assert(TT == 2, "eight waves, a value each");
    const int token = 16 * (all >> 2) + 4 * quad + (all & 3), over = last - first - 1 - (chunks - 1) * SC;
    const unsigned place = __umul24(token, line) + column, place_last = __umul24(min(token, over), line) + column;
    auto fetch_value = [&](int c) {
        const float* at = values + (size_t)(min(c, chunks - 1) * SC) * line;
        asm volatile("" : "+s"(at));
        return at[c >= chunks - 1 ? place_last : place];
    };
    // only LDS has to be in order between the waves: loads from memory stay in flight
    auto meet = []() {
        asm volatile("" ::: "memory");
        wait_lgkmcnt<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // Loads stay where they stand among the products.  Left alone, the compiler put three chunks' loads side by side, so that every third
    // chunk waited for memory twice.  And a CU takes one of these loads in 16 clocks: eight waves that ask for all of a chunk's at once wait a
    // thousand clocks and more for that.  With a removal term they go out between the products (walk of 2,048 tokens, 16 heads of 128 x 128, all
    // at once 122 us, spread 98); without it there are too few products to hide them, and a chunk's go out at its start, where the reading
    // waves have nothing else to do (63 us, spread 71, at other places 66 to 82).
    constexpr bool SPREAD = REMOVE;
    auto pin = []() { __builtin_amdgcn_sched_barrier(6); };
    float raw[3];
#pragma unroll
    for (int n = 0; n < 3; ++n) raw[n] = fetch_value(n);
    shared_value[0][all][lane] = raw[0];
    shared_value[1][all][lane] = raw[1];
    raw[0] = fetch_value(3);
    if (keeps) {
        float* home = state + (((size_t)slot_ids[req] * heads + head) * dv + column) * DK + wave * 16 * KT + 4 * quad;
        f32x4 S[KT];
#pragma unroll
        for (int k = 0; k < KT; ++k) S[k] = *reinterpret_cast<const f32x4*>(home + 16 * k);
        struct Loaded {
            f32x4 z[KT][TT], probe[REMOVE ? TT : 1][KT], removal[KT][REMOVE ? TT : 1];
            float decay;
        };
        const unsigned decay_place = lane / (16 * KT) * DK + wave * 16 * KT + lane % (16 * KT);
        // load number n of a chunk's
        constexpr int TILES = TT * KT, LOADS = 1 + (REMOVE ? 3 : 1) * TILES;
        auto fetch_one = [&](Loaded& l, const float* rec, int n) {
            if (n == 0) l.decay = rec[Rec::DECAY + (16 * KT * 2 == kWave || lane < 32 * KT ? decay_place : 0u)];
            else if (n <= TILES) l.z[(n - 1) % KT][(n - 1) / KT] = tile(rec, Rec::Z, (wave * KT + (n - 1) % KT) * TT + (n - 1) / KT);
            else if constexpr (REMOVE) {
                const int m = n - 1 - TILES;
                if (m < TILES) l.probe[m / KT][m % KT] = tile(rec, Rec::PROBE, m / KT * KEYS + wave * KT + m % KT);
                else l.removal[m % KT][m / KT - TT] = tile(rec, Rec::REMOVAL, (wave * KT + m % KT) * TT + m / KT - TT);
            }
        };
        auto fetch = [&](Loaded& l, int c) {
            const float* rec = record_of(c);
#pragma unroll
            for (int n = 0; n < LOADS; ++n) fetch_one(l, rec, n);
        };
        float value[TT][4];
        f32x4 decay[KT], rest[KT];
        // what the wave works with in the chunk, out of LDS
        auto take = [&](int n) {
#pragma unroll
            for (int k = 0; k < KT; ++k) {
                decay[k] = *reinterpret_cast<const f32x4*>(&shared_decay[n][wave][16 * k + 4 * quad]);
                rest[k] = *reinterpret_cast<const f32x4*>(&shared_decay[n][wave][16 * KT + 16 * k + 4 * quad]);
            }
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) value[t][i] = shared_value[n][4 * t + i][lane];
        };
        auto leave_decay = [&](int n, float d) {
            if (16 * KT * 2 == kWave || lane < 32 * KT) shared_decay[n][wave][lane] = d;
        };
        auto work = [&](const Loaded& l, const Loaded& next, Loaded& coming, int c, auto turn3) {
            constexpr int n = decltype(turn3)::value;       // c % 3
            const int turn = c & 1;
            const float* rec = record_of(c + 2);
            constexpr int EVERY = 2;
            static_assert(!SPREAD || EVERY * LOADS < 12 * TILES, "a product for every load");
            auto ask_all = [&]() {
                pin();
#pragma unroll
                for (int l = 0; l < LOADS; ++l) fetch_one(coming, rec, l);
                raw[(n + 1) % 3] = fetch_value(c + 4);
                pin();
            };
            auto between = [&](int product) {
                if constexpr (!SPREAD) return;
                pin();
                if (product % EVERY == 0 && product / EVERY <= LOADS) {
                    if (product == 0) raw[(n + 1) % 3] = fetch_value(c + 4);
                    else fetch_one(coming, rec, product / EVERY - 1);
                    pin();
                }
            };
            if constexpr (!SPREAD) ask_all();
#pragma unroll
            for (int k = 0; k < KT; ++k) states[turn][wave][k][lane] = S[k];
            if constexpr (REMOVE) {
                f32x4 y[TT];
#pragma unroll
                for (int t = 0; t < TT; ++t) y[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < KT; ++k)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int t = 0; t < TT; ++t) {
                            y[t] = mfma4(l.probe[t][k][i], S[k][i], y[t]);
                            between((k * 4 + i) * TT + t);
                        }
#pragma unroll
                for (int t = 0; t < TT; ++t) taken[turn][wave][t][lane] = y[t];
            }
            shared_value[(n + 2) % 3][all][lane] = raw[(n + 2) % 3];
            leave_decay((n + 1) % 3, next.decay);
#pragma unroll
            for (int k = 0; k < KT; ++k)
#pragma unroll
                for (int i = 0; i < 4; ++i) S[k][i] = fmaf(S[k][i], rest[k][i], S[k][i] * decay[k][i]);
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int k = 0; k < KT; ++k) {
                        S[k] = mfma4(l.z[k][t][i], value[t][i], S[k]);
                        between((REMOVE ? 4 * TILES : 0) + (t * 4 + i) * KT + k);
                    }
            take((n + 1) % 3);
            meet();
            if constexpr (REMOVE) {
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    const f32x4 y = (taken[turn][0][t][lane] + taken[turn][1][t][lane]) +
                                    (taken[turn][2][t][lane] + taken[turn][3][t][lane]);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int k = 0; k < KT; ++k) {
                            S[k] = mfma4(l.removal[k][t][i], y[i], S[k]);
                            between(8 * TILES + (t * 4 + i) * KT + k);
                        }
                }
            }
        };
        Loaded sets[3];
        fetch(sets[0], 0);
        fetch(sets[1], 1);
        leave_decay(0, sets[0].decay);
        meet();                                             // the first two chunks' values are there
        take(0);
        auto turn = [&](int c, auto turn3) {
            constexpr int n = decltype(turn3)::value;
            work(sets[n], sets[(n + 1) % 3], sets[(n + 2) % 3], c, turn3);
        };
        for (int c = 0;;) {
            turn(c, std::integral_constant<int, 0>{});
            if (++c == chunks) break;
            turn(c, std::integral_constant<int, 1>{});
            if (++c == chunks) break;
            turn(c, std::integral_constant<int, 2>{});
            if (++c == chunks) break;
        }
        meet();                                             // the last chunk's read-outs
        if (mine) {
#pragma unroll
            for (int k = 0; k < KT; ++k) *reinterpret_cast<f32x4*>(home + 16 * k) = S[k];
        }
    } else {
        struct Loaded {
            f32x4 read[TT][KT], mix;
        };
        constexpr int LOADS = 1 + TT * KT;
        auto fetch_one = [&](Loaded& l, const float* rec, int n) {
            if (n == 0) l.mix = tile(rec, Rec::MIX, wave);
            else l.read[(n - 1) / KT][(n - 1) % KT] = tile(rec, Rec::READ, (n - 1) / KT * KEYS + wave * KT + (n - 1) % KT);
        };
        auto fetch = [&](Loaded& l, int c) {
            const float* rec = record_of(c);
#pragma unroll
            for (int n = 0; n < LOADS; ++n) fetch_one(l, rec, n);
        };
        // chunk c's read-outs, a tile of tokens by each of two waves, four channels of a token a lane, once every wave has left its part
        float* to = out + (size_t)first * line + (size_t)head * dv;
        const int channel = block * 16 + 4 * quad;
        const bool whole = dv % 4 == 0 && ((uintptr_t)out & 15) == 0;
        const unsigned store_place = __umul24(16 * (wave & 1) + row, line) + channel;
        auto write = [&](int c) {
            if (wave >= TT) return;
            const f32x4* part = &reads[c & 1][0][wave][lane];
            constexpr int NEXT = TT * kWave;                // from a wave's part to the next one's
            const f32x4 o = (part[0] + part[NEXT]) + (part[2 * NEXT] + part[3 * NEXT]);
            float* at = to + (size_t)(c * SC) * line;
            if (16 * wave + row >= last - first - c * SC) return;
            if (whole) {
                if (channel < dv) *reinterpret_cast<f32x4*>(at + store_place) = o;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (channel + i < dv) at[store_place + i] = o[i];
            }
        };
        // a wave takes one of the four blocks of W^ (the one above the diagonal is zero)
        auto mix = [&](const f32x4& w, int n) {
            float value[4];
            f32x4 mixed = {0.f, 0.f, 0.f, 0.f};
            unsigned most = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                value[i] = shared_value[n][4 * (wave & 1) + i][lane];
                most = max(most, __float_as_uint(value[i]) & 0x7FFFFFFFu);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) mixed = mfma4(value[i], w[i], mixed);
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(most >= 0x7F800000u) != 0, 0)) {       // token by token, each for its own row and those behind it
                mixed = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 16; ++s) {
                    const float by = __shfl(w[s & 3], (s >> 2) * 16 + row, kWave);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float of = __shfl(value[s & 3], (s >> 2) * 16 + 4 * quad + i, kWave);
                        if (s <= row + 16 * ((wave >> 1) - (wave & 1))) mixed[i] = fmaf(by, of, mixed[i]);
                    }
                }
            }
            return mixed;
        };
        f32x4 mixed;
        auto work = [&](const Loaded& l, const Loaded& next, Loaded& coming, int c, auto turn3) {
            constexpr int n = decltype(turn3)::value;       // c % 3
            const int turn = c & 1;
            const float* rec = record_of(c + 2);
            constexpr int EVERY = 4 * TT * KT / (LOADS + 1);
            static_assert(EVERY >= 1, "a product for every load");
            auto ask_all = [&]() {
                pin();
#pragma unroll
                for (int l = 0; l < LOADS; ++l) fetch_one(coming, rec, l);
                raw[(n + 1) % 3] = fetch_value(c + 4);
                pin();
            };
            auto between = [&](int product) {
                if constexpr (!SPREAD) return;
                pin();
                if (product % EVERY == 0 && product / EVERY <= LOADS) {
                    if (product == 0) raw[(n + 1) % 3] = fetch_value(c + 4);
                    else fetch_one(coming, rec, product / EVERY - 1);
                    pin();
                }
            };
            if constexpr (!SPREAD) ask_all();
            shared_value[(n + 2) % 3][all][lane] = raw[(n + 2) % 3];
            meet();                                         // the state before chunk c is there, and chunk c - 1's parts
            f32x4 S[KT], o[TT];
#pragma unroll
            for (int k = 0; k < KT; ++k) S[k] = states[turn][wave][k][lane];
#pragma unroll
            for (int t = 0; t < TT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KT; ++k)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int t = 0; t < TT; ++t) {
                        o[t] = mfma4(S[k][i], l.read[t][k][i], o[t]);
                        between((k * 4 + i) * TT + t);
                    }
            const f32x4 mixed_next = mix(next.mix, (n + 1) % 3);
            if (c > 0) write(c - 1);
#pragma unroll
            for (int t = 0; t < TT; ++t) {
#pragma unroll
                for (int i = 0; i < 4; ++i) o[t][i] += wave >> 1 == t ? mixed[i] : 0.f;
                reads[turn][wave][t][lane] = o[t];
            }
            mixed = mixed_next;
        };
        Loaded sets[3];
        fetch(sets[0], 0);
        fetch(sets[1], 1);
        meet();
        mixed = mix(sets[0].mix, 0);
        auto turn = [&](int c, auto turn3) {
            constexpr int n = decltype(turn3)::value;
            work(sets[n], sets[(n + 1) % 3], sets[(n + 2) % 3], c, turn3);
        };
        for (int c = 0;;) {
            turn(c, std::integral_constant<int, 0>{});
            if (++c == chunks) break;
            turn(c, std::integral_constant<int, 1>{});
            if (++c == chunks) break;
            turn(c, std::integral_constant<int, 2>{});
            if (++c == chunks) break;
        }
        meet();
        write(chunks - 1);
    }
}

// Records of a step, one at least: a list of short requests is taken too, and nothing is done for it.
static int record_places(int T, int R, int least) { return max(1, record_place(T, R, least)); }

template <int DK, bool REMOVE>
static void scan_chunks(const float* coef, const float* v, float* state, float* out, float* records, const int* q_offsets,
                        const int* slot_ids, int R, int T, int heads, int dv, int least, hipStream_t stream) {
    constexpr int THREADS = REMOVE ? 4 * DK : 2 * DK;
    const int places = record_places(T, R, least);
    float* alone = records + (size_t)places * heads * ChunkRecord<DK, REMOVE>::SIZE;
    const int items = places * heads, at_once = prepare_turns<DK, REMOVE> ? device_cus() * (DK == 64 && !REMOVE ? 4 : 2) : items;
    scan_chunk_prepare_kernel<DK, REMOVE, THREADS><<<min(items, at_once), THREADS, 0, stream>>>(coef, q_offsets, R, T, heads, least, items, records,
                                                                                                reinterpret_cast<unsigned char*>(alone));
    scan_chunk_walk_kernel<DK, REMOVE><<<dim3(heads * ((dv + 15) / 16), R), 512, 0, stream>>>(
        records, reinterpret_cast<const uint2*>(alone), coef, v, state, out, q_offsets, slot_ids, T, heads, dv, least);
}

}  // namespace lc

using namespace lc;

// Floats that lc_scan_chunks wants as `records` for T tokens of R requests, or 0 where it does not take these sizes.
LC_API long long lc_scan_chunks_records(int planes, int R, int T, int heads, int dk, int dv, int least) {
    if (least < 1 || R <= 0 || T <= 0 || heads <= 0 || dv <= 0 || (long long)heads * dv >= (1 << 23) || (planes != 3 && planes != 5) || (dk != 64 && dk != 128)) return 0;
    const long long size = dk == 64 ? (planes == 5 ? ChunkRecord<64, true>::SIZE : ChunkRecord<64, false>::SIZE)
                                    : (planes == 5 ? ChunkRecord<128, true>::SIZE : ChunkRecord<128, false>::SIZE);
    return (size + 2) * heads * record_places(T, R, least);
}

// The recurrence for the requests of at least `least` tokens; the others' states and rows of out are left alone.
// coef, v, state, out as for lc_delta_scan, all 16-byte aligned.
LC_API int lc_scan_chunks(const float* coef, int planes, const float* v, float* state, int slots, float* out, float* records,
                          const int* q_offsets, const int* slot_ids, int R, int T, int heads, int dk, int dv, int least,
                          hipStream_t stream) {
    LC_CHECK(R >= 0 && T >= 0 && heads > 0 && dk > 0 && dv > 0 && slots >= 0 && least >= 1, "scan_chunks: bad sizes");
    if (R == 0 || T == 0) return 0;
    LC_CHECK(lc_scan_chunks_records(planes, R, T, heads, dk, dv, least) > 0, "scan_chunks: sizes it does not take");
    LC_CHECK(coef && v && state && out && records && q_offsets && slot_ids, "scan_chunks: null pointer");
    LC_CHECK(((uintptr_t)coef | (uintptr_t)state | (uintptr_t)records) % 16 == 0, "scan_chunks: not aligned to 16 bytes");
    LC_CHECK(R <= 65535 && heads <= 65535, "scan_chunks: too many requests or heads for the grid");
    LC_CHECK((long long)heads * dv < (1 << 23), "scan_chunks: a token's values are too many");
#define LC_CHUNKS(DK)                                                                                                      \
    do {                                                                                                                   \
        if (planes == 5)                                                                                                   \
            scan_chunks<DK, true>(coef, v, state, out, records, q_offsets, slot_ids, R, T, heads, dv, least, stream);       \
        else                                                                                                               \
            scan_chunks<DK, false>(coef, v, state, out, records, q_offsets, slot_ids, R, T, heads, dv, least, stream);      \
    } while (0)
    if (dk == 128) LC_CHUNKS(128);
    else LC_CHUNKS(64);
#undef LC_CHUNKS
    LC_LAUNCH_CHECK("scan_chunks");
    return 0;
}
