// Latent attention for a prompt's portion, head by head.
//
// In the latent's space (latent_bf16.hip) a query meets 512 + 64 entries of a cached row and sums 512 of them, whatever the
// head's own size: what a step of lone tokens wants, because it reads nothing but the rows.  A portion of many tokens has
// many queries for every row, so it pays to take the rows out of the latent's space once: k_j = W_uk c_j beside the rotated
// part, v_j = W_uv c_j, and to attend with 128 + 64 and 128 entries a head (320 multiply-adds a query and key where there were 1,088).
// Three steps: latent_rows_kernel lays a request's visible rows side by side out of their pages; two dense products make
// [row][head, entry] keys and, with the operands in the other order, [head, entry][row] values, which is the transposed form
// that O^T = V^T P^T wants; latent_wide_kernel attends and applies the output gate.
#include "common.h"

#include "activations.h"
#include "gemm_tile.h"

namespace lc {

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int LW_KEYS = 64;         // keys of a stage; a request's rows are filled up to whole stages
constexpr int LW_TOKENS = 128;      // queries of a workgroup, 32 a wave
constexpr int LW_DIM = 128, LW_ROT = 64, LW_VDIM = 128;

// grid (rows / 4): a wave a row.  Row i of the request's rows (position lo + i, its page's place in table) -> c [i][R], turned [i][rot];
// zeros behind `count`.
// A query that does not see a key gives it weight zero, and zero times what is not finite would be no number: the later token's row
// would spoil up to a tile's 127 tokens before it.  So a latent with such an entry becomes a value of zeros and a key that is NaN
// in its rotated part, whose score is NaN for the queries that see it and never asked for by the others.
__global__ __launch_bounds__(256) void latent_rows_kernel(const bf16* __restrict__ cache, const int* __restrict__ table, int page_size,
                                                          int R, int rot, int lo, int count, int rows, bf16* __restrict__ c,
                                                          bf16* __restrict__ turned) {
    const int i = blockIdx.x * 4 + threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (i >= rows) return;
    const int j = lo + i, pieces = (R + rot) / 8;
    const bool live = i < count;
    bool odd = false;
    const bf16* row = cache + (size_t)(live ? table[j / page_size] * page_size + j % page_size : 0) * (R + rot);
    for (int p = lane; p < pieces; p += kWave) {
        bf16x8 v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16>(0.f);
        if (live) v = *reinterpret_cast<const bf16x8*>(row + p * 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) odd |= p * 8 < R && (__builtin_bit_cast(unsigned short, static_cast<bf16>(v[e])) & 0x7F80) == 0x7F80;
        if (p * 8 < R) *reinterpret_cast<bf16x8*>(c + (size_t)i * R + p * 8) = v;
        else *reinterpret_cast<bf16x8*>(turned + (size_t)i * rot + (p * 8 - R)) = v;
    }
    if (__builtin_amdgcn_ballot_w64(odd) == 0) return;
    for (int p = lane; p < pieces; p += kWave) {
        const bool rotated = p * 8 >= R;
        bf16x8 v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = static_cast<bf16>(rotated ? __builtin_nanf("") : 0.f);
        *reinterpret_cast<bf16x8*>(rotated ? turned + (size_t)i * rot + (p * 8 - R) : c + (size_t)i * R + p * 8) = v;
    }
}

struct WideArgs {
    const bf16* q; long long ldq;               // [T][head][128 + 64], the rotated entries as they were
    const bf16* q_turned; long long q_row, q_head;   // token t, head h: the 64 rotated entries at t q_row + h q_head
    const bf16* keys; const bf16* turned;       // [row][H 128], [row][64]
    const bf16* values; long long ldv;          // [H 128][row]
    int H, first, tokens, position, lo;         // the portion: its first token's row of q and position; the rows' first position
    float scale_log2; int window;
    const float* sink;
    const bf16* gate; long long ldg, gate_head; // token t, head h: at t ldg + h gate_head, 128 entries or (gate_head 1) one
    bf16* out; long long ldo;
};

// Four operands of LDS, asked for: two places and the same OFFSET bytes further on; lds_have waits until at most LEFT of the reads asked for
// are still on their way and ties the operands to that point.  (The compiler would wait for every load to LDS in flight before an LDS read of
// its own.)
template <int OFFSET>
__device__ __forceinline__ void lds_ask(bf16x8 (&r)[4], unsigned one, unsigned two) {
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:%6\n\tds_read_b128 %2, %5\n\tds_read_b128 %3, %5 offset:%6"
                 : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
                 : "v"(one), "v"(two), "n"(OFFSET)
                 : "memory");
}
template <int LEFT> __device__ __forceinline__ void lds_have(bf16x8 (&r)[4]) {
    wait_lgkmcnt<LEFT>();
    asm volatile("" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]));
    __builtin_amdgcn_sched_barrier(0);
}

// grid (heads, tiles of 128 tokens, the last first: it sees the most keys).  Head h runs on XCD h % 8, whose L2 keeps its keys and
// values for all tiles.  A wave owns 32 queries: S^T = K Q^T by v_mfma_f32_32x32x16_bf16, with the rows of K taken in the order
// that leaves a lane eight neighbouring keys of its query for each 16, which is what P^T needs as an operand; softmax
// base 2 against a reference point that moves when a score outgrows it by 2^8; O^T += V^T P^T.  A stage of 64 keys (40 KB) comes
// straight into LDS while the one before is worked through; 16-byte chunks lie at places xor the row, so that no operand's 16
// rows meet a bank twice.  Two workgroups a CU, whose waves fill each other's waits.
//
// HALVES 2: eight waves, of which four take every other stage of the same queries, with a ring of their own; their sums are joined at the
// end.  A stage keeps a wave that is alone on its SIMD busy for about 1.7 us (its loads, products and weights wait for each other) and
// two waves for little more, so where there are no more workgroups than two a CU the halves are the second wave, and they halve the
// longest chain (us, one and two halves: 2,048 tokens of 16 heads 57 and 43, 1,953 behind 2,048 others 101 and 77, 512 behind 4,000 109 and 75; 4,000
// tokens, 512 workgroups, 119 and 95; not everywhere: 64 heads, 700 tokens, 384 workgroups, 24 and 29, 1,024 behind 4,000, 512 workgroups, 192 and
// 194).  With more workgroups a CU has its second wave anyway, and the halves gain little or only wait for each other (528 workgroups 128 and 111,
// 768 213 and 212 and, 48 heads, 84 and 92, 1,024 337 and 348 and, 64 heads, 99 and 113).
//
// Offset: a lane's place within the rows of a load, in bytes: 32 bits where three rows of the keys and seven of the values fit, so that a load's address
// is one register beside a scalar base; 64 bits for rows longer than that.
template <int HALVES, typename Offset>
__global__ __launch_bounds__(256 * HALVES, 2) void latent_wide_kernel(WideArgs a) {
    constexpr int KB = LW_KEYS * LW_DIM * 2, TB = LW_KEYS * LW_ROT * 2, VB = LW_VDIM * LW_KEYS * 2, STAGE = KB + TB + VB;
    constexpr int KS = (LW_DIM + LW_ROT) / 16, VT = LW_VDIM / 32;
    __shared__ __attribute__((aligned(1024))) char all_lds[HALVES * 2 * STAGE];
    const int lane = threadIdx.x & 63, col = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3, part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    char* lds = all_lds + part * 2 * STAGE;
    const int head = blockIdx.x, tile = gridDim.y - 1 - blockIdx.y;
    const int row = tile * LW_TOKENS + wave * 32 + col;     // the lane's token of the portion
    const bool live = row < a.tokens;
    const int token = a.first + min(row, a.tokens - 1);
    const int tile_last = min(tile * LW_TOKENS + LW_TOKENS, a.tokens) - 1;
    // keys are counted from the rows' first position on
    const int at = a.position - a.lo + min(row, a.tokens - 1);      // the last key that the lane's query sees
    const int from = a.window > 0 ? at - a.window + 1 : 0;          // and the first
    const int wave_first = tile * LW_TOKENS + wave * 32;
    const int wave_lo = a.window > 0 ? a.position - a.lo + wave_first - a.window + 1 : 0;
    const int wave_hi = a.position - a.lo + min(wave_first + 31, a.tokens - 1);
    const bool wave_live = wave_first < a.tokens;
    const int tile_lo = a.window > 0 ? max(0, a.position - a.lo + tile * LW_TOKENS - a.window + 1) : 0;
    const int s_begin = tile_lo / LW_KEYS, s_end = (a.position - a.lo + tile_last) / LW_KEYS + 1;

    const float scale = a.scale_log2 == 0.f ? 1.f : fabsf(a.scale_log2);
    bf16x8 qf[KS];
    {
        const bf16* plain = a.q + (size_t)token * a.ldq + (size_t)head * (LW_DIM + LW_ROT) + 8 * half;
        const bf16* turned = a.q_turned + (size_t)token * a.q_row + (size_t)head * a.q_head + 8 * half;
#pragma unroll
        for (int k = 0; k < KS; ++k)
            qf[k] = *reinterpret_cast<const bf16x8*>(k < LW_DIM / 16 ? plain + 16 * k : turned + 16 * k - LW_DIM);
        if (!(a.scale_log2 > 0.f)) {    // below, the scale of the scores is positive: the largest score times it is the largest
#pragma unroll
            for (int k = 0; k < KS; ++k)
#pragma unroll
                for (int e = 0; e < 8; ++e) qf[k][e] = static_cast<bf16>(static_cast<float>(qf[k][e]) * (a.scale_log2 < 0.f ? -1.f : 0.f));
        }
    }
    // load instructions: four rows of 256 bytes of the keys, eight of 128 of their rotated parts and of the values; a lane's bytes from the
    // first row on, of the first instruction (instruction i of the keys: place xor 4 i) and, the values', of the second
    const int r4 = lane >> 4, r8 = lane >> 3;
    const Offset k_off = (Offset)r4 * a.H * (LW_DIM * 2) + (((lane & 15) ^ r4) * 16), v_row_off = (Offset)(r8 * a.ldv * 2);
    const unsigned t_off = r8 * (LW_ROT * 2) + (((lane & 7) ^ (r8 >> 1)) * 16);
    const Offset v_off[2] = {v_row_off + (((lane & 7) ^ (r8 >> 1)) * 16), v_row_off + (((lane & 7) ^ 4 ^ (r8 >> 1)) * 16)};
    // Load n of a wave, of stage s into that turn's place: 0 to 3 the keys', 4 and 5 their rotated parts', 6 to 9 the values'.
    constexpr int LOADS = 10, KEY_LOADS = 6;
    auto load = [&](int n, int s, int turn) {
        char* stage = lds + (turn & 1) * STAGE;
        const char* from;
        if (n < 4) from = reinterpret_cast<const char*>(a.keys + ((size_t)(s * LW_KEYS + 16 * wave + 4 * n) * a.H + head) * LW_DIM) + (k_off ^ (n * 64));
        else if (n < 6) from = reinterpret_cast<const char*>(a.turned + (size_t)(s * LW_KEYS + 16 * wave + 8 * (n - 4)) * LW_ROT) + (t_off ^ ((n - 4) * 64));
        else from = reinterpret_cast<const char*>(a.values + ((size_t)head * LW_VDIM + 32 * wave + 8 * (n - 6)) * a.ldv + (size_t)s * LW_KEYS) + v_off[n & 1];
        const int at = n < 4 ? (4 * wave + n) * 1024 : n < 6 ? KB + (2 * wave + n - 4) * 1024 : KB + TB + (4 * wave + n - 6) * 1024;
        __builtin_amdgcn_global_load_lds((glb_ptr_t)from, (lds_ptr_t)(stage + at), 16, 0, 0);
    };
    // row r of a tile of S^T is key 16 (r / 16) + 8 ((r / 4) % 2) + 4 ((r / 8) % 2) + r % 4 of its 32: the lane's 16 values, rows
    // 8 (v / 4) + 4 half + v % 4, are then the keys 16 (v / 8) + 8 half + v % 8
    const int key = 16 * (col >> 4) + 8 * ((col >> 2) & 1) + 4 * ((col >> 3) & 1) + (col & 3);
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t)lds;
    // place p of a row of K is chunk p ^ (key % 16): chunk 2 x + half of the lane's row is 32 x further on or back, in these bits alone
    static_assert(STAGE % 1024 == 0 && KB % 1024 == 0 && TB % 1024 == 0, "rows do not reach into the places' bits");
    const unsigned k_row = lds0 + key * 256 + (half ^ (key & 15)) * 16, t_row = lds0 + KB + key * 128 + (half ^ ((key >> 1) & 7)) * 16;
    const unsigned v_row = lds0 + KB + TB + col * 128 + (half ^ ((col >> 1) & 7)) * 16;         // the same for the rows 32 further on

    floatx16 o[VT];
#pragma unroll
    for (int i = 0; i < VT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[i][v] = 0.f;
    float m_ref = -INFINITY, l = 0.f;
    floatx16 sc[2];
    // S^T of the stage in this turn's place; the next four operands are on their way while four are multiplied
    auto scores = [&](unsigned stage) {
        // entries 16 x .. 16 x + 31 of both tiles of 32 keys; the tiles' sums take turns, so that no product waits for the one before it
        constexpr int GROUPS = KS / 2;
        bf16x8 ka[2][4];
        const unsigned k_at = k_row + stage, t_at = t_row + stage;
        auto ask = [&](int g) {
            const int x = 2 * g;
            if (x < LW_DIM / 16) lds_ask<32 * 256>(ka[g & 1], k_at ^ (x * 32), k_at ^ ((x + 1) * 32));
            else lds_ask<32 * 128>(ka[g & 1], t_at ^ ((x - LW_DIM / 16) * 32), t_at ^ ((x + 1 - LW_DIM / 16) * 32));
        };
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) sc[t][v] = 0.f;
        ask(0);
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) {
            if (g + 1 < GROUPS) { ask(g + 1); lds_have<4>(ka[g & 1]); }
            else lds_have<0>(ka[g & 1]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                sc[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[g & 1][i], qf[2 * g + (i >> 1)], sc[i & 1], 0, 0, 0);
        }
    };
    // the weights of stage s, whose scores are in sc, and their products with its values
    auto weigh = [&](int s, unsigned stage) {
        const int c0 = s * LW_KEYS;
        // keys 16 b .. 16 b + 31 of two tiles of 32 entries
        bf16x8 va[2][4];
        const unsigned v_at = v_row + stage;
        auto ask = [&](int g) {
            const int b = g % 2 * 2;
            const unsigned from = v_at + g / 2 * 64 * 128;
            lds_ask<32 * 128>(va[g & 1], from ^ (b * 32), from ^ ((b + 1) * 32));
        };
        // scores in units of log 2; what the query does not see is -infinity
        const bool all = c0 + LW_KEYS - 1 <= wave_hi - 31 && c0 >= wave_lo + 31;       // every query of the wave sees every key
        if (!all) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int j = c0 + 32 * t + 16 * (v >> 3) + 8 * half + (v & 7);
                    sc[t][v] = j <= at && j >= from ? sc[t][v] : -INFINITY;
                }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) mx = fmaxf(mx, sc[t][v]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, kWave)) * scale;
        if (__builtin_amdgcn_ballot_w64(mx > m_ref + 8.f) != 0) {      // also at a query's first visible key
            const float m_new = mx > m_ref + 8.f ? mx : m_ref;
            const float keep = m_ref == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_ref - m_new);
            l *= keep;
#pragma unroll
            for (int i = 0; i < VT; ++i)
#pragma unroll
                for (int v = 0; v < 16; ++v) o[i][v] *= keep;
            m_ref = m_new;
        }
        const float ref = m_ref == -INFINITY ? 0.f : m_ref;
        bf16x8 p[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                float x = sc[b >> 1][(b & 1) * 8 + v] * scale;      // rounded before the reference is taken off, not in one multiply-add:
                asm("" : "+v"(x));                                  // the same bits as ever (2 to 4 % of the kernel's time)
                const float w = __builtin_amdgcn_exp2f(x - ref);
                l += w;
                p[b][v] = static_cast<bf16>(w);
            }
        }
        ask(0);
#pragma unroll
        for (int g = 0; g < VT; ++g) {
            if (g + 1 < VT) { ask(g + 1); lds_have<4>(va[g & 1]); }
            else lds_have<0>(va[g & 1]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                floatx16& sum = o[g / 2 * 2 + (i & 1)];
                sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[g & 1][i], p[g % 2 * 2 + (i >> 1)], sum, 0, 0, 0);
            }
        }
    };
    // The second half is a turn behind with its weights and values: while one half's waves multiply for their scores the other's, on the same
    // SIMDs, work out weights.  A CU takes loads at 64 bytes a clock at most, 1,300 clocks for a turn's 80 KB, and a wave that issues its own in
    // a row does nothing else until they are taken (clock stamps: 700 to 2,000 of a turn's 6,000 clocks): so each half issues them at a moment of
    // its own, the first behind its scores, the second its values at the turn's start and its keys behind its weights.  us, as it was before there was any of
    // this, a turn behind, so, and with the priority below: 1,953 tokens of 16 heads behind 2,048 others 95.4, 89.3, 83.1 and 82; 2,048 tokens
    // 56.6, 54.3, 48.5 and 48; 512 behind 4,000 99.1, 91.0, 78.1 and 77; 1,500 of 32 heads behind 600 (a single half) 79.3, 76.1, 71.5 and 71.
    // All of it beside the kernel before, warm, side by side on another card, a score rounded by itself as there: 88.4 and 76.5, 50.2 and 43.1,
    // 97.0 and 75.2, 70.6 and 63.1.
    const bool behind = HALVES == 2 && part == 1;
    const int turns = (s_end - s_begin + HALVES - 1) / HALVES;
    auto seen = [&](int s) { return wave_live && s < s_end && s * LW_KEYS <= wave_hi && s * LW_KEYS + LW_KEYS > wave_lo; };
#pragma unroll
    for (int n = 0; n < LOADS; ++n)
        if (n < KEY_LOADS || !behind) load(n, min(s_begin + part, s_end - 1), 0);
    for (int turn = 0; turn < turns + HALVES - 1; ++turn) {
        const int s = s_begin + part + turn * HALVES;
        wait_vmcnt<0>();                                    // this wave's loads of the stage have landed
        __builtin_amdgcn_s_barrier();                       // everybody's have; nobody reads the other stage any more
        asm volatile("" ::: "memory");
        // behind the last stage it is loaded again, and not read
        auto ahead = [&](int from, int to) {
            const int s_keys = min(s + HALVES, s_end - 1), s_values = behind ? min(s, s_end - 1) : s_keys;
#pragma unroll
            for (int n = 0; n < LOADS; ++n)
                if (n >= from && n < to) load(n, n < KEY_LOADS ? s_keys : s_values, n >= KEY_LOADS && behind ? turn : turn + 1);
        };
        // (conditions of their own: in one block for each half the compiler makes two loops of the turns, and spills)
        if (behind) ahead(KEY_LOADS, LOADS);
        if (behind && turn > 0 && seen(s - HALVES)) weigh(s - HALVES, ((turn - 1) & 1) * STAGE);
        if (behind) ahead(0, KEY_LOADS);
        const bool see = seen(s);
        __builtin_amdgcn_s_setprio(1);                      // products leave most of the issue slots to the other wave
        if (see) scores((turn & 1) * STAGE);
        __builtin_amdgcn_s_setprio(0);
        if (!behind) ahead(0, LOADS);
        if (!behind && see) weigh(s, (turn & 1) * STAGE);
    }
    wait_vmcnt<0>();
    if constexpr (HALVES == 2) {
        static_assert((VT * 16 + 2) * 256 * 4 <= HALVES * 2 * STAGE, "the second half's sums");
        float* its = reinterpret_cast<float*>(all_lds) + (threadIdx.x & 255);       // [m, l, the sums][thread]
        __syncthreads();                                    // nobody reads a stage any more
        if (part == 1) {
            its[0] = m_ref;
            its[256] = l;
#pragma unroll
            for (int i = 0; i < VT; ++i)
#pragma unroll
                for (int v = 0; v < 16; ++v) its[(2 + 16 * i + v) * 256] = o[i][v];
        }
        __syncthreads();
        if (part == 1) return;
        const float m_its = its[0], m_all = fmaxf(m_ref, m_its);
        const float mine = m_ref == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_ref - m_all);
        const float by = m_its == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_its - m_all);
        l = fmaf(l, mine, its[256] * by);
#pragma unroll
        for (int i = 0; i < VT; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) o[i][v] = fmaf(o[i][v], mine, its[(2 + 16 * i + v) * 256] * by);
        m_ref = m_all;
    }
    if (!live) return;
    l += __shfl_xor(l, 32, kWave);
    float inv = 1.f / l;
    if (a.sink) {       // one more term in the denominator, a key with that score and no value
        const float s2 = a.sink[head] * 1.4426950408889634f, m_all = fmaxf(m_ref, s2);
        const float keep = __builtin_amdgcn_exp2f(m_ref - m_all);
        inv = keep / fmaf(l, keep, __builtin_amdgcn_exp2f(s2 - m_all));
    }
    const bf16* gate = a.gate ? a.gate + (size_t)token * a.ldg + (size_t)head * a.gate_head : nullptr;
    if (gate && a.gate_head == 1) inv *= sigmoid(to_f32(gate[0]));
    bf16* out = a.out + (size_t)token * a.ldo + (size_t)head * LW_VDIM;
#pragma unroll
    for (int i = 0; i < VT; ++i)
#pragma unroll
        for (int v = 0; v < 16; v += 4) {
            const int e = 32 * i + 2 * v + 4 * half;        // rows 8 (v / 4) + 4 half ...
            bf16x4 g, y;
            if (gate && a.gate_head != 1) g = *reinterpret_cast<const bf16x4*>(gate + e);
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                float x = o[i][v + n] * inv;
                if (gate && a.gate_head != 1) x *= sigmoid(static_cast<float>(g[n]));
                y[n] = static_cast<bf16>(x);
            }
            *reinterpret_cast<bf16x4*>(out + e) = y;
        }
}

}  // namespace lc

using namespace lc;

static thread_local int g_wide_halves = 0;

// Tests and tuning: 1 or 2 halves for the calling thread's launches, 0 lets the size decide.  Returns the setting before.
LC_API int lc_latent_wide_halves(int halves) {
    const int before = g_wide_halves;
    if (halves >= 0 && halves <= 2) g_wide_halves = halves;
    return before;
}

// The kernels' operands are asked for and waited for in two pieces of inline assembly (lds_ask, lds_have), and in between the compiler takes
// their registers to hold values already: were one spilled to scratch memory there, the spill would store what it held before.  So the compiled
// kernels are asked, once: 1 all in registers, 0 one uses scratch memory, -1 could not ask.  Unless it is 1, portions stay in the latent's space.
static int wide_state() {
    static const int state = [] {
        const void* kernels[] = {(const void*)latent_wide_kernel<1, unsigned>, (const void*)latent_wide_kernel<2, unsigned>,
                                 (const void*)latent_wide_kernel<1, unsigned long long>, (const void*)latent_wide_kernel<2, unsigned long long>};
        for (const void* kernel : kernels) {
            hipFuncAttributes attr;
            if (hipFuncGetAttributes(&attr, kernel) != hipSuccess) {
                (void)hipGetLastError();
                return -1;
            }
            if (attr.localSizeBytes != 0) return 0;
        }
        return 1;
    }();
    return state;
}
LC_API int lc_latent_wide_ok() { return wide_state(); }

// Whether these heads have a kernel.
LC_API int lc_latent_wide_supported(int R, int dim, int rot, int vdim) {
    return dim == LW_DIM && rot == LW_ROT && vdim == LW_VDIM && R > 0 && R % 64 == 0 && wide_state() == 1 ? 1 : 0;
}

LC_API int lc_latent_rows(const void* cache, const int* table, int page_size, int R, int rot, int lo, int count, int rows, void* c,
                          void* turned, hipStream_t stream) {
    LC_CHECK(page_size > 0 && R > 0 && R % 8 == 0 && rot >= 0 && rot % 8 == 0 && lo >= 0 && count >= 0 && rows >= count, "latent_rows: bad sizes");
    if (rows == 0) return 0;
    LC_CHECK(cache && table && c && (turned || rot == 0), "latent_rows: null pointer");
    LC_CHECK(((uintptr_t)cache | (uintptr_t)c | (uintptr_t)turned) % 16 == 0, "latent_rows: not aligned to 16 bytes");
    latent_rows_kernel<<<(rows + 3) / 4, 256, 0, stream>>>((const bf16*)cache, table, page_size, R, rot, lo, count, rows, (bf16*)c,
                                                           (bf16*)turned);
    LC_LAUNCH_CHECK("latent_rows");
    return 0;
}

// A portion of `tokens` tokens from row `first` of q on, at `position`, over the request's rows from position lo on: keys and
// turned filled up to whole stages of 64 rows, values [H 128][ldv] likewise.
LC_API int lc_latent_wide(const void* q, long long ldq, const void* q_turned, long long q_row, long long q_head, const void* keys,
                          const void* turned, const void* values, long long ldv, int H, int first, int tokens, int position,
                          int lo, float scale, int window, const float* sink, const void* gate, long long ldg, long long gate_head,
                          void* out, long long ldo, hipStream_t stream) {
    LC_CHECK(H > 0 && first >= 0 && tokens >= 0 && lo >= 0 && position >= lo && window >= 0, "latent_wide: bad sizes");
    if (tokens == 0) return 0;
    LC_CHECK(q && q_turned && keys && turned && values && out, "latent_wide: null pointer");
    LC_CHECK(window == 0 ? lo == 0 : lo <= (position - window + 1 > 0 ? position - window + 1 : 0), "latent_wide: rows are missing");
    LC_CHECK(((uintptr_t)q | (uintptr_t)q_turned | (uintptr_t)keys | (uintptr_t)turned | (uintptr_t)values) % 16 == 0 &&
                 (ldq | q_row | q_head | ldv) % 8 == 0, "latent_wide: not aligned to 16 bytes");
    LC_CHECK(ldv >= (position + tokens - lo + LW_KEYS - 1) / LW_KEYS * LW_KEYS, "latent_wide: the values' rows are too short");
    LC_CHECK((uintptr_t)out % 8 == 0 && ldo % 4 == 0, "latent_wide: the output is not aligned to 8 bytes");
    LC_CHECK(!gate || gate_head == 1 || (gate_head == LW_VDIM && (uintptr_t)gate % 8 == 0 && ldg % 4 == 0), "latent_wide: bad gates");
    LC_CHECK(wide_state() != 0, "latent_wide: a kernel uses scratch memory");
    const int tiles = (tokens + LW_TOKENS - 1) / LW_TOKENS;
    LC_CHECK(tiles <= 65535, "latent_wide: too many tokens");
    WideArgs a{(const bf16*)q, ldq, (const bf16*)q_turned, q_row, q_head, (const bf16*)keys, (const bf16*)turned, (const bf16*)values, ldv,
               H, first, tokens, position, lo, scale * 1.4426950408889634f, window, sink, (const bf16*)gate, ldg, gate_head,
               (bf16*)out, ldo};
    const int halves = g_wide_halves ? g_wide_halves : (long long)H * tiles <= 2 * device_cus() ? 2 : 1;
    const bool near = ldv < 1ll << 28 && H < 1 << 22;       // 3 rows of 256 H bytes and 7 of 2 ldv are below 2^32
    if (halves == 2) {
        if (near) latent_wide_kernel<2, unsigned><<<dim3(H, tiles), 512, 0, stream>>>(a);
        else latent_wide_kernel<2, unsigned long long><<<dim3(H, tiles), 512, 0, stream>>>(a);
    } else {
        if (near) latent_wide_kernel<1, unsigned><<<dim3(H, tiles), 256, 0, stream>>>(a);
        else latent_wide_kernel<1, unsigned long long><<<dim3(H, tiles), 256, 0, stream>>>(a);
    }
    LC_LAUNCH_CHECK("latent_wide");
    return 0;
}
