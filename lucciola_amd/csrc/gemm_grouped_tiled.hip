// The grouped products of gemm_grouped.hip for bfloat16 operands, in three shapes of their own:
//
//   even     experts with many rows (prompts): tiles of 256 columns whose height follows from the group's rows, one workgroup a CU,
//            through the loop of the dense products (gemm_tile.h): direct loads to LDS, v_mfma_f32_32x32x16_bf16, scheduled by
//            hand.  8,192 rows over 32 matrices of 2,048 x 2,048 (256 rows each, more or less): 128 us in tiles of 128 x 128,
//            90 (0.76 PFLOP/s); 6,092 rows 102 and 71; 4,096 x 2,048: 258 and 202.  A third of that is that no tile is mostly
//            empty, a third that workgroups do not all ask the same memory channels (below), a third that the tile is found with
//            one trip to memory and stored in whole lines without a test of the epilogue an entry.  What bounds them now is the
//            start (the matrices come from memory once, 45 to 50 us of it) and end of a tile, some 11 us a round, which nothing
//            hides, and 1.0 us a block of 64 k at 160 rows, where LDS is read and written at 0.7 of what it can.
//   tiles    shorter K, fewer columns, products per head: 64 rows by 128 columns through the same loop, four workgroups a CU, because
//            a tile is short and its first loads and its stores pass beside another's products.
//   stream   few rows a group (decoding: 16 rows a tile): bound by reading every group's matrix once, so what counts is
//            how much of it is on its way.  256 rows over 32 matrices of 2,048 x 2,048 (268 MB): 68 -> 51 us (5.3 TB/s); 32 rows,
//            21 matrices: 51 -> 31; 512 rows, 32 matrices of 4,096 x 2,048: 156 -> 98.
//
// Which rows are whose, the gather list and the epilogues are as described there.
#include "common.h"

#include <cmath>

#include "activations.h"
#include "gemm_grouped.h"
#include "gemm_tile.h"

namespace lc {

// One element's epilogue, for a result of type TO.
template <typename TO>
__device__ __forceinline__ float grouped_finish(const GroupedArgs& a, const bf16* gate, int m, int n, float v) {
    if (a.epilogue == ACT_SIGMOID_GATE) return v * sigmoid(to_f32(gate[(size_t)m * a.ldg + n]));
    if (a.epilogue == ACT_SIGMOID_GROUP_GATE) return v * sigmoid(to_f32(gate[(size_t)m * a.ldg]));
    return activate<TO>(v, a.epilogue);
}

// grid (column tiles, row tiles, groups or 1): neighbouring workgroups, which go to different XCDs, take different columns
// of w, and the row tiles of a group that share columns of w run on one XCD where the column tiles are a multiple of 8.
template <typename TO, int BM, int BN, int STAGES, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_grouped_tiled_kernel(GroupedArgs a) {
    typedef TileLoop<BM, BN, STAGES, WM, WN> Loop;
    constexpr int TM = Loop::TM, TN = Loop::TN;
    __shared__ __attribute__((aligned(1024))) char lds[Loop::LDS];
    GroupedTile tile;
    if (!find_tile(a, BM, tile)) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = blockIdx.x * BN, N = a.N, K = a.K;
    const bf16* x = reinterpret_cast<const bf16*>(a.x) + (size_t)tile.group * a.x_group;
    const bf16* w = reinterpret_cast<const bf16*>(a.w) + (size_t)tile.group * N * K;
    const bf16* xg[Loop::LPA];
    const bf16* wg[Loop::LPB];
#pragma unroll
    for (int i = 0; i < Loop::LPA; ++i) {
        const int m = min(tile.first + Loop::row_of(i, wave, lane), tile.end - 1);      // a row behind the group's end is its last one
        xg[i] = x + (size_t)(a.gather ? a.gather[m] : m) * a.ldx + Loop::chunk_of(i, wave, lane) * 8;
    }
#pragma unroll
    for (int i = 0; i < Loop::LPB; ++i)
        wg[i] = w + (size_t)min(n0 + Loop::row_of(i, wave, lane), N - 1) * K + Loop::chunk_of(i, wave, lane) * 8;
    static_assert(Loop::MF == 32, "the epilogue's layout");
    floatx16 acc[TM][TN];
    Loop::run(lds, xg, wg, K / TL_K, 0, wave, lane, acc);

    // acc[i][j][v]: row (v / 4) * 8 + (lane / 32) * 4 + v % 4, column lane % 32 of the 32 x 32 tile
    TO* out = reinterpret_cast<TO*>(a.out) + (size_t)tile.group * a.out_group;
    const bf16* gate = a.gate ? reinterpret_cast<const bf16*>(a.gate) + (size_t)tile.group * a.gate_group : nullptr;
    const int m0 = tile.first + (wave / WN) * (BM / WM) + (lane >> 5) * 4, c0 = n0 + (wave % WN) * (BN / WN) + (lane & 31);
    if (a.pairs) {
        // neighbouring lanes swap every other value and store two columns of a row together: even lanes the even v
        const bool odd = lane & 1;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; v += 2) {
                    const int m = m0 + i * 32 + (v >> 2) * 8 + (v & 3), n = c0 + j * 32, pair = n & ~1;
                    float first = acc[i][j][v], second = acc[i][j][v + 1];
                    asm volatile("" : "+v"(first), "+v"(second));   // two values, not one indexed by `odd`
                    const float got = lane_swap<0xB1>(odd ? first : second);    // lane ^ 1
                    const int row = m + (odd ? 1 : 0);
                    if (row < tile.end && pair < N)
                        store_pair<TO>(out + (size_t)row * a.ldo + pair, grouped_finish<TO>(a, gate, row, pair, odd ? got : first),
                                       grouped_finish<TO>(a, gate, row, pair + 1, odd ? second : got));
                }
    } else {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int m = m0 + i * 32 + (v >> 2) * 8 + (v & 3), n = c0 + j * 32;
                    if (m < tile.end && n < N) store_out<TO>(out + (size_t)m * a.ldo + n, grouped_finish<TO>(a, gate, m, n, acc[i][j][v]));
                }
    }
}

// Experts with many rows: tiles of 256 columns whose height follows from the group.  A group's rows, in units of 32, are cut into the
// fewest tiles of at most `most` units and evenly (257 rows are two tiles of 160 rows' room and not three of 128, the last of
// one row), and `most`, 1 to 8, is what lets the product end first by an estimate: a tile costs its units and two more (its
// columns of w, its first loads and its stores), and the CUs, which hold a workgroup each, take the tiles in rounds.  Every
// workgroup works this out by itself from row_start, a lane per candidate and share of the groups, so that the host need not
// know the routing.
struct EvenTile {
    int group, first, end, units, column;      // units 0: there is none
};

// units divided by `most`, rounded up; inverse: 2^32 divided by `most`, rounded up (0 for 1).  Exact below 2^28 units, for the inverse is too large
// by less than 8.
__device__ __forceinline__ int even_tiles(int units, int most, unsigned inverse) {
    return most == 1 ? units : (int)__umulhi((unsigned)(units + most - 1), inverse);
}
__device__ __forceinline__ unsigned even_inverse(int most) { return most == 1 ? 0u : 0xFFFFFFFFu / (unsigned)most + 1u; }

__device__ __forceinline__ EvenTile find_even_tile(const int* row_start, int G, int id, int columns, int room, int cus, int lane) {
    const int sub = lane >> 3, most = (lane & 7) + 1;
    const unsigned inverse = even_inverse(most);
    int tiles = 0, highest = 0, cost = 0;
    for (int g = sub; g < G; g += 8) {
        // (divisions of integers, some eighty instructions a group, were a quarter of a short product of 256 experts)
        const int units = (row_start[g + 1] - row_start[g] + 31) >> 5, n = even_tiles(units, most, inverse);
        const int h = n ? (int)ceilf((float)units * __builtin_amdgcn_rcpf((float)n) - 0.001f) : 0;
        tiles += n;
        cost += n * (h + 2);
        highest = max(highest, h);
    }
#pragma unroll
    for (int d = 8; d < 64; d *= 2) {
        tiles += __shfl_xor(tiles, d);
        cost += __shfl_xor(cost, d);
        highest = max(highest, __shfl_xor(highest, d));
    }
    const int rounds = (tiles * columns + cus - 1) / cus;
    float until = tiles > room ? INFINITY : tiles ? (float)(rounds - 1) * cost / tiles + (highest + 2) : 0.f;     // `most` 8 always has room
    int best = most;
#pragma unroll
    for (int d = 1; d < 8; d *= 2) {
        const float other = __shfl_xor(until, d);
        const int its = __shfl_xor(best, d);
        if (other < until || (other == until && its > best)) { until = other; best = its; }
    }
    best = __builtin_amdgcn_readfirstlane(best);
    tiles = __shfl(tiles, best - 1);
    const unsigned best_inverse = even_inverse(best);

    // An XCD (workgroup id % 8) takes neighbouring tiles, a group's column by column: its L2 then serves one group's rows to all of its
    // columns and a column of w to all of the group's tiles, and memory is asked for each once.
    const int items = tiles * columns, per = (items + 7) / 8;
    const int item = (id & 7) * per + (id >> 3);
    EvenTile t{0, 0, 0, 0, 0};
    if ((id >> 3) >= per || item >= items) return t;
    int before = 0;
    for (int g0 = 0; g0 < G; g0 += 64) {
        const int g = g0 + lane;
        const int from = g < G ? row_start[g] : 0, to = g < G ? row_start[g + 1] : 0;
        const int units = (to - from + 31) >> 5, n = even_tiles(units, best, best_inverse);
        int upto = n;
#pragma unroll
        for (int d = 1; d < 64; d *= 2) {
            const int v = __shfl_up(upto, d);
            upto += lane >= d ? v : 0;
        }
        const unsigned long long past = __ballot(item < (before + upto) * columns);
        if (past) {
            const int at = __builtin_ctzll(past);
            const int count = __builtin_amdgcn_readfirstlane(__shfl(n, at)), first = __builtin_amdgcn_readfirstlane(__shfl(from, at));
            const int end = __builtin_amdgcn_readfirstlane(__shfl(to, at)), all = __builtin_amdgcn_readfirstlane(__shfl(units, at));
            const int place = __builtin_amdgcn_readfirstlane(item - (before + __shfl(upto, at) - count) * columns);
            t.group = g0 + at;
            t.units = (all + count - 1) / count;
            t.column = place / count;
            t.first = first + (place - t.column * count) * t.units * 32;
            t.end = min(end, t.first + t.units * 32);
            return t;
        }
        before += __builtin_amdgcn_readfirstlane(__shfl(upto, 63));
    }
    return t;
}

constexpr int EVEN_GROUPS = 4096;
constexpr int EVEN_N = 256, EVEN_LDS = 3 * (160 + EVEN_N) * TL_K * 2;

// BM rows from tile.first on by the 256 columns of tile.column.  GATED: these are 128 gate and the 128 up columns that belong to them,
// 32 of each in turn, so that a wave has both of a pair, and 128 columns are stored: 8,192 rows by 4,096 columns would be written
// and read again by a kernel of 49 us (2,048 columns stored, K of 2,048, four choices of 32 weighed: 198 + 49 -> 209 us).
template <typename TO, bool GATED, int BM, int STAGES, int WM, int WN>
__device__ __forceinline__ void even_tile(const GroupedArgs& a, const GroupedGate& gate, const EvenTile& tile, char* lds,
                                          const float* row_weight, int wave, int lane) {
    typedef TileLoop<BM, EVEN_N, STAGES, WM, WN> Loop;
    static_assert(Loop::LDS <= EVEN_LDS, "LDS");
    constexpr int TM = Loop::TM, TN = Loop::TN;
    const int n0 = tile.column * EVEN_N, N = a.N, K = a.K, blocks = K / TL_K;
    const bf16* x = reinterpret_cast<const bf16*>(a.x);
    const bf16* w = reinterpret_cast<const bf16*>(a.w) + (size_t)tile.group * N * K;
    const bf16* xg[Loop::LPA];
    const bf16* wg[Loop::LPB];
#pragma unroll
    for (int i = 0; i < Loop::LPA; ++i) {
        const int m = min(tile.first + Loop::row_of(i, wave, lane), tile.end - 1);      // a row behind the tile's end is its last one
        xg[i] = x + (size_t)(a.gather ? a.gather[m] : m) * a.ldx + Loop::chunk_of(i, wave, lane) * 8;
    }
#pragma unroll
    for (int i = 0; i < Loop::LPB; ++i) {
        const int r = Loop::row_of(i, wave, lane);
        const int n = GATED ? min(n0 / 2 + (r >> 6) * 32 + (r & 31), N / 2 - 1) + ((r >> 5) & 1) * (N / 2) : min(n0 + r, N - 1);
        wg[i] = w + (size_t)n * K + Loop::chunk_of(i, wave, lane) * 8;
    }
    static_assert(Loop::MF == 32, "the epilogue's layout");
    floatx16 acc[TM][TN];
    // Rows of w lie 2 K bytes apart, so workgroups that walk k in step ask the same few memory channels at every moment: each group
    // starts at a block of its own and wraps around.  Its tiles and columns start together, because they share rows in L2.
    Loop::run(lds, xg, wg, blocks, (int)((unsigned)tile.group * 13u % (unsigned)blocks), wave, lane, acc);

    // 32 rows at a time pass through the wave's part of the ring, so that a lane gets neighbouring columns, 16 bytes of them
    // (acc[i][j][v]: row (v / 4) * 8 + (lane / 32) * 4 + v % 4, column lane % 32 of the 32 x 32 product)
    constexpr int WIDTH = 32 * TN, STRIDE = WIDTH + 4;
    static_assert(4 * 32 * STRIDE * 4 <= EVEN_LDS, "a strip of every wave");
    float* strip = reinterpret_cast<float*>(lds) + wave * 32 * STRIDE;
    constexpr int E = PIECE<TO>, OUT = GATED ? WIDTH / 2 : WIDTH, LANES = OUT / E, ROWS = 64 / LANES;      // stored columns, lanes a row, rows a pass
    static_assert(64 % LANES == 0 && 32 % ROWS == 0, "whole passes");
    TO* out = reinterpret_cast<TO*>(a.out);
    const int top_row = (wave / WN) * (BM / WM), columns = GATED ? N / 2 : N;
    const int r0 = lane / LANES, c = lane % LANES * E, n = (GATED ? n0 / 2 : n0) + (wave % WN) * OUT + c;
    const int place = GATED ? c / 32 * 64 + c % 32 : c;         // in the strip; GATED: the up entries stand 32 behind
    // finish: a sum (GATED: a gate's and an up column's) to the stored entry
    auto store = [&](int i, int r, auto finish) {
        const int m = tile.first + top_row + i * 32 + r;
        const float* from = strip + r * STRIDE + place;
        float v[E], u[E];
#pragma unroll
        for (int e = 0; e < E; e += 4) {
            *reinterpret_cast<float4*>(v + e) = *reinterpret_cast<const float4*>(from + e);
            if (GATED) *reinterpret_cast<float4*>(u + e) = *reinterpret_cast<const float4*>(from + 32 + e);
        }
        if (m >= tile.end || n >= columns) return;              // columns % 8 == 0
        const float weight = GATED && gate.weights ? row_weight[top_row + i * 32 + r] : 1.f;
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = GATED ? finish(weight * v[e], weight * u[e]) : finish(v[e], 0.f);
        store_piece<TO>(out + (size_t)m * a.ldo + n, v);
    };
    // one test of the epilogue for 32 rows (one an entry cost 10 to 30 us of a product of 8,192 rows); the long forms stay rolled
    auto finish = [&](int i) {
        auto rolled = [&](auto f) {
#pragma unroll 1
            for (int r = 0; r < 32; r += ROWS) store(i, r0 + r, f);
        };
        auto unrolled = [&](auto f) {
#pragma unroll
            for (int r = 0; r < 32; r += ROWS) store(i, r0 + r, f);
        };
        if constexpr (GATED) {
            if (gate.kind == 0) unrolled([](float g, float u) { return gated_f(g, u, kSilu); });
            else unrolled([](float g, float u) { return gelu_tanh<bf16>(g) * u; });
        } else {
            switch (a.epilogue) {
                case ACT_NONE: unrolled([](float z, float) { return z; }); break;
                case ACT_RELU_SQUARED: unrolled([](float z, float) { return activate<TO>(z, ACT_RELU_SQUARED); }); break;
                case ACT_GELU_ERF: rolled([](float z, float) { return gelu_erf<TO>(z); }); break;
                default:
                    if constexpr (sizeof(TO) == 2) unrolled([](float z, float) { return gelu_tanh<TO>(z); });
                    else rolled([](float z, float) { return gelu_tanh<TO>(z); });
            }
        }
    };
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v)
                strip[((v >> 2) * 8 + (lane >> 5) * 4 + (v & 3)) * STRIDE + j * 32 + (lane & 31)] = acc[i][j][v];
        __builtin_amdgcn_wave_barrier();
        finish(i);
        __builtin_amdgcn_wave_barrier();
    }
}

// (The gated form uses 68 bytes of scratch memory: 16 sums of the highest tile, put aside behind its loop, where no operand is on its way.)
template <typename TO, bool GATED>
__global__ __launch_bounds__(256) void gemm_grouped_even_kernel(GroupedArgs a, GroupedGate gate, int columns, int room, int cus) {
    __shared__ __attribute__((aligned(1024))) char lds[EVEN_LDS];
    __shared__ float row_weight[GATED ? 256 : 1];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int* row_start = reinterpret_cast<int*>(lds);       // G < EVEN_GROUPS
    for (int g = threadIdx.x; g <= a.G; g += 256) row_start[g] = a.row_start[g];
    __syncthreads();
    const EvenTile tile = find_even_tile(row_start, a.G, blockIdx.x, columns, room, cus, lane);
    if (GATED && gate.weights && tile.first + (int)threadIdx.x < tile.end) {
        const int m = tile.first + threadIdx.x, token = a.gather[m];        // one of the token's choices is row m
        for (int k = 0; k < gate.top; ++k)
            if (gate.entry_row[(size_t)token * gate.top + k] == m) row_weight[threadIdx.x] = gate.weights[(size_t)token * gate.top + k];
    }
    __syncthreads();
    switch (tile.units) {
        case 0: return;
        case 1: return even_tile<TO, GATED, 32, 3, 1, 4>(a, gate, tile, lds, row_weight, wave, lane);
        case 2: return even_tile<TO, GATED, 64, 3, 1, 4>(a, gate, tile, lds, row_weight, wave, lane);
        case 3: return even_tile<TO, GATED, 96, 3, 1, 4>(a, gate, tile, lds, row_weight, wave, lane);
        case 4: return even_tile<TO, GATED, 128, 3, 2, 2>(a, gate, tile, lds, row_weight, wave, lane);
        case 5: return even_tile<TO, GATED, 160, 3, 1, 4>(a, gate, tile, lds, row_weight, wave, lane);
        case 6: return even_tile<TO, GATED, 192, 2, 2, 2>(a, gate, tile, lds, row_weight, wave, lane);
        default: return even_tile<TO, GATED, 256, 2, 2, 2>(a, gate, tile, lds, row_weight, wave, lane);
    }
}

// Tiles of 16 rows by 64 columns, K in blocks of 128: a row of w comes 256 bytes at a time, and a ring of STREAM_STAGES blocks
// keeps all but one of them on their way, two workgroups a CU: 120 KB a CU, where the CU's share of the memory's rate
// needs some 64.  A row's 16-byte chunk c lies at place c ^ (row % 16): the 16 rows that LDS serves together meet no bank twice.
// A wave multiplies 16 of the columns by itself.  Every column tile starts at a block of its own and wraps around, so that the
// workgroups, whose rows lie a multiple of 2 K bytes apart, do not all ask the same memory channels at once; the order of
// an element's sum depends on its group and column alone.
constexpr int STREAM_K = 128, STREAM_STAGES = 4, STREAM_N = 64;

template <typename TO>
__global__ __launch_bounds__(256) void gemm_grouped_stream_kernel(GroupedArgs a) {
    constexpr int XB = 16 * STREAM_K * 2, WB = STREAM_N * STREAM_K * 2, LOADS = 5;
    __shared__ __attribute__((aligned(1024))) char lds[STREAM_STAGES * (XB + WB)];
    GroupedTile tile;
    if (!find_tile(a, 16, tile)) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, quad = lane >> 4;
    const int n0 = blockIdx.x * STREAM_N, N = a.N, K = a.K, blocks = K / STREAM_K;
    const bf16* x = reinterpret_cast<const bf16*>(a.x) + (size_t)tile.group * a.x_group;
    const bf16* w = reinterpret_cast<const bf16*>(a.w) + (size_t)tile.group * N * K;
    // a load instruction brings four rows: lane l the chunk at place l % 16 of row l / 16
    const bf16* from[LOADS];
    {
        const int row = 4 * wave + quad, m = min(tile.first + row, tile.end - 1);
        from[0] = x + (size_t)(a.gather ? a.gather[m] : m) * a.ldx + (col ^ row) * 8;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 4 * i + quad;
            from[1 + i] = w + (size_t)min(n0 + 16 * wave + r, N - 1) * K + (col ^ r) * 8;
        }
    }
    const int skew = (int)(((unsigned)blockIdx.x * 17u + (unsigned)tile.group * 5u) % (unsigned)blocks);
    auto issue = [&](int b) {
        char* stage = lds + (b % STREAM_STAGES) * (XB + WB);
        int k = b + skew;
        k -= k >= blocks ? blocks : 0;
        __builtin_amdgcn_global_load_lds((glb_ptr_t)(from[0] + k * STREAM_K), (lds_ptr_t)(stage + wave * 1024), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(from[1 + i] + k * STREAM_K),
                                             (lds_ptr_t)(stage + XB + (4 * wave + i) * 1024), 16, 0, 0);
    };
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t)lds;
    const unsigned row_x = lds0 + col * 256, row_w = lds0 + XB + (16 * wave + col) * 256;
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int b = 0; b < min(STREAM_STAGES - 1, blocks); ++b) issue(b);
    for (int b = 0; b < blocks; ++b) {
        // this wave's loads of block b have landed when only those of the younger blocks are left
        const int younger = min(blocks - 1 - b, STREAM_STAGES - 2);
        if (younger == STREAM_STAGES - 2) wait_vmcnt<(STREAM_STAGES - 2) * LOADS>();
        else if (younger == 1) wait_vmcnt<LOADS>();
        else wait_vmcnt<0>();
        static_assert(STREAM_STAGES == 4, "the waits above");
        __builtin_amdgcn_s_barrier();                       // everybody's have; nobody reads the block before any more
        asm volatile("" ::: "memory");
        if (b + STREAM_STAGES - 1 < blocks) issue(b + STREAM_STAGES - 1);       // into the place of the block before
        const unsigned stage = (b % STREAM_STAGES) * (XB + WB);
        bf16x8 xa[4], wb[4];
        unsigned ax[4], aw[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const unsigned place = ((4 * s + quad) ^ col) * 16;
            ax[s] = row_x + stage + place;
            aw[s] = row_w + stage + place;
        }
        // in inline assembly, because the compiler would wait for every load to LDS in flight before an LDS read
        asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\tds_read_b128 %2, %10\n\tds_read_b128 %3, %11\n\t"
                     "ds_read_b128 %4, %12\n\tds_read_b128 %5, %13\n\tds_read_b128 %6, %14\n\tds_read_b128 %7, %15\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(xa[0]), "=&v"(wb[0]), "=&v"(xa[1]), "=&v"(wb[1]), "=&v"(xa[2]), "=&v"(wb[2]), "=&v"(xa[3]), "=&v"(wb[3])
                     : "v"(ax[0]), "v"(aw[0]), "v"(ax[1]), "v"(aw[1]), "v"(ax[2]), "v"(aw[2]), "v"(ax[3]), "v"(aw[3])
                     : "memory");
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[s], wb[s], acc, 0, 0, 0);
    }
    TO* out = reinterpret_cast<TO*>(a.out) + (size_t)tile.group * a.out_group;
    const bf16* gate = a.gate ? reinterpret_cast<const bf16*>(a.gate) + (size_t)tile.group * a.gate_group : nullptr;
    const int n = n0 + 16 * wave + col;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = tile.first + 4 * quad + i;
        if (m < tile.end && n < N) store_out<TO>(out + (size_t)m * a.ldo + n, grouped_finish<TO>(a, gate, m, n, acc[i]));
    }
}

// Whether gemm_grouped_even_kernel takes these operands: lists, no gates, whole pieces of 8 columns that it stores at once.
static bool even_takes(const GroupedArgs& a) {
    const long long columns = (a.N + EVEN_N - 1) / EVEN_N, room = a.M / 128 + a.G;
    return a.row_start && a.K % TL_K == 0 && a.N % 8 == 0 && a.ldo % 8 == 0 && (uintptr_t)a.out % 16 == 0 && a.G < EVEN_GROUPS &&
           a.epilogue != ACT_SIGMOID_GATE && a.epilogue != ACT_SIGMOID_GROUP_GATE && room * columns < 1 << 30;
}

// Tiles of 64 rows that the experts' rows make, as routers deal them out: about evenly, some sqrt(p) more or fewer than the p rows of each.
static double tiles_of_64(const GroupedArgs& a) {
    const double p = (double)a.M / a.G, spread = sqrt(p);
    double tiles = 1.0 - exp(-p);
    if (p > 1024) tiles = p / 64 + 0.5;
    else
        for (int rows = 64; rows < p + 4 * spread + 1; rows += 64) tiles += 0.5 * erfc((rows - p) / (spread * M_SQRT2));
    return tiles * a.G;
}

// Whether the kernel of even tiles is the faster one of this file's.  Lists for tiles of 128 rows have no other.  With fewer rows an expert
// (lists for tiles of 64 rows, whole K in 64 x 128) it needs 1,024 k and 512 columns (us, 64 x 128 and these, weights cold here and below:
// 2,048 rows over 16 matrices of 512 x 256 8.8 and 9.8, 256 x 1,024 11.6 and 14.4), and what decides then is how many workgroups the tiles of
// 64 x 128 make.  One a CU and fewer bring a CU less per product than a single wide tile does (400 rows, 4 matrices of 1,024 x 2,048 25 and 31;
// 1,520 rows, 8 of them 24 and 31; 1,600 rows, 16 26 and 34; K 4,096 47 and 59), unless w is so large that memory's rate counts, at which
// these are better (640 rows, 32 matrices of 1,024 x 2,048 37 and 33, K 1,024 17.6 and 20.2; 800 rows, 8 of 4,096 x 2,048 37 and 32).  More of
// them share CUs, and the wide tiles win (2,240 rows, 16 of 768 x 2,048 38 and 31; 6,080 rows, 32 of 1,024 x 2,048 58 and 39), but for a short
// K with a tile an expert and many experts, where both wait for w (1,280 rows, 64 of 1,024 x 1,024 30.8 and 32.3, 480 rows, 24 of 2,048 x 1,024
// 25.1 and 23.7).  gated: these save a pass besides, and win
// from one workgroup a CU on (320 rows, 16 of 2 x 1,024 x 1,024 20.9 and 19.1, 1,280 rows, 64 of 2 x 512 x 1,024 32.9 and 31.9), but not
// below (1,120 rows, 8 of 2 x 512 x 2,048 26.7 and 29.8).
static bool even_pays(const GroupedArgs& a, int tile_rows, bool gated) {
    if (tile_rows != 64) return tile_rows == 128;
    if (a.K < 1024 || a.N < 512) return false;
    const double experts = tiles_of_64(a), tiles = experts * ((a.N + 127) / 128), cus = device_cus();
    if (gated) return tiles > 0.98 * cus;
    if (tiles > 1.02 * cus) return a.K >= 1536 || experts > 1.05 * a.G || a.G < 48;
    return (double)a.G * a.N > cus * (80 + 50.0 * 1024 / a.K);
}

template <typename TO, bool GATED>
static void launch_even(const GroupedArgs& a, const GroupedGate& gate, hipStream_t stream) {
    const int columns = (a.N + EVEN_N - 1) / EVEN_N, room = a.M / 128 + a.G;
    gemm_grouped_even_kernel<TO, GATED><<<(room * columns + 7) / 8 * 8, 256, 0, stream>>>(a, gate, columns, room, device_cus());
}

template <typename TO>
static int grouped_tiled(const GroupedArgs& a, int max_tiles, int tile_rows, bool forced, hipStream_t stream) {
    auto grid = [&](int bm, int bn) {
        return dim3((a.N + bn - 1) / bn, a.row_start ? max_tiles : (a.M + bm - 1) / bm, a.row_start ? 1 : a.G);
    };
    if (tile_rows == 16) {
        gemm_grouped_stream_kernel<TO><<<grid(16, STREAM_N), 256, 0, stream>>>(a);
    } else if (even_takes(a) && (forced || even_pays(a, tile_rows, false))) {
        launch_even<TO, false>(a, GroupedGate{}, stream);
    } else {
        gemm_grouped_tiled_kernel<TO, 64, 128, 2, 2, 2><<<grid(64, 128), 256, 0, stream>>>(a);
    }
    LC_LAUNCH_CHECK("gemm_grouped_tiled");
    return 0;
}

bool grouped_tiled_takes(const GroupedArgs& a, int tile_rows) {
    return tile_rows == 16 ? a.K % STREAM_K == 0 : tile_rows == 128 ? even_takes(a) : a.K % TL_K == 0;
}

// What these kernels are faster at is a K long enough to fill their rings; a tile of few blocks is mostly its first loads and its
// stores, which the smaller workgroups of gemm_grouped.hip, of which a CU holds more, hide better.  From 512 k on they are as fast or
// faster at every size tried; below it depends on how many workgroups there are (us, gemm_grouped.hip and these):
//   stream   one round of two workgroups a CU gains (16 heads, 512 columns of 128 k, 64 rows 4.2 and 3.8), more lose: the same
//            at 32 heads 5.1 and 5.4, 400 rows over 32 experts of 2,048 x 128 6.0 and 7.5.  Products per head from 256 k on gain too.
//   128 rows (the even tiles) likewise one round gains (8 experts of 256 rows, 2,048 x 256 16.8 and 10.8, of 400 rows, 512 x 128
//            11.8 and 9.0); less than 192 k has to be one round of one even workgroup a CU, as a round is then mostly what it starts
//            and ends with: 96 experts of 200 rows, 128 columns of 128 k, 13.0 and 11.0, 128 of them (328 workgroups) 13.5 and 14.4,
//            256 20.8 and 26.6.  More rounds than that mostly gain too (8 x 1,024 rows, 2,048 x 256 34.2 and 24.9; 64 x 256 rows,
//            4,096 x 256 102.0 and 111.5) and are not taken.  With the activation in it a
//            product saves a kernel, and the line below 192 k is not drawn (128 x 200 rows, 2 x 64 columns of 128 k 19.7 and 15.5;
//            256 x 200 rows 30.3 and 30.2).
//   64 rows  experts: 384 k and a workgroup for every CU (18.0 and 18.3 at the worst, 116 and 84 at the best); 256 k lose 10 % at
//            few workgroups.  Per head: the shorter K, the more full tiles it takes: of 128 k 160 rows, 16 heads, 512 columns 5.8 and
//            6.6, 2,048 rows 22.7 and 21.6; of 192 k 6.5 and 7.0, and 8.0 and 7.3 at 512 rows; of 64 k it mostly loses (10.1 and 12.4).
static bool rounds_pay(const GroupedArgs& a, int max_tiles, int tile_rows) {
    const double columns = (a.N + (tile_rows == 16 ? STREAM_N : 128) - 1) / (tile_rows == 16 ? STREAM_N : 128);
    const double workgroups =
        columns * (a.row_start ? (max_tiles < a.M ? max_tiles : a.M) : (double)((a.M + tile_rows - 1) / tile_rows) * a.G);
    const double round = 2 * device_cus();
    if (a.K >= 512 || (tile_rows != 64 && workgroups <= round)) return a.K >= 128;
    if (tile_rows == 128) return false;
    if (a.row_start) return tile_rows == 64 && a.K >= 384 && workgroups >= device_cus();
    if (tile_rows == 16) return a.K >= 256;
    const double full = (double)a.M * a.N * a.G / (64 * 128), short_by = 512.0 / a.K;
    return a.K >= 128 && full * full / workgroups >= 32 * short_by * short_by * short_by;
}

bool grouped_tiled_pays(const GroupedArgs& a, int max_tiles, int tile_rows) {
    if (tile_rows == 128 && a.K < 192 && (double)(a.M / 128 + a.G) * ((a.N + EVEN_N - 1) / EVEN_N) > device_cus()) return false;
    return rounds_pay(a, max_tiles, tile_rows);
}

int launch_grouped_tiled(const GroupedArgs& a, int max_tiles, int tile_rows, bool out_bf16, bool forced, hipStream_t stream) {
    return out_bf16 ? grouped_tiled<bf16>(a, max_tiles, tile_rows, forced, stream)
                    : grouped_tiled<float>(a, max_tiles, tile_rows, forced, stream);
}

// a.N: gate and up columns together
bool grouped_gates(const GroupedArgs& a, int tile_rows, bool forced) {
    if (tile_rows == 16 || a.N % 16 || !even_takes(a)) return false;
    return forced || (even_pays(a, tile_rows, true) && rounds_pay(a, a.M / tile_rows + a.G, tile_rows));
}

bool grouped_evens(const GroupedArgs& a, int max_tiles, int tile_rows) {
    return tile_rows != 16 && even_takes(a) && even_pays(a, tile_rows, false) && grouped_tiled_pays(a, max_tiles, tile_rows);
}

int launch_grouped_gated(const GroupedArgs& a, const GroupedGate& gate, hipStream_t stream) {
    launch_even<bf16, true>(a, gate, stream);
    LC_LAUNCH_CHECK("gemm_grouped_gated");
    return 0;
}

}  // namespace lc
