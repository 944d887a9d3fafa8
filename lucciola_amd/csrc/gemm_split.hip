// out[M, N] = x[M, K] . w[N, K]^T for float32 x and bfloat16 w as a true 32-bit product on the bfloat16 matrix instruction: a float32
// number is the sum of three bfloat16 numbers, cut off after 8 bits each (24 in all, so nothing is left over), the product of two
// bfloat16 numbers is exact in float32, and v_mfma_f32_32x32x16_bf16 adds in float32.  x is cut times 2^40: the last bit of the smallest
// float32, 2^-149, then stands at 2^-109, inside bfloat16's range (as they stand, entries below 2^-110 lose their last bits: 2e-5 of one at
// 1e-36), and a chunk's sum is taken times 2^-40.  Three such products cost 3/16 of what
// v_mfma_f32_16x16x4_f32 takes for the same sums (gemm_generic.hip, which serves float32 w and a K that is not whole).
//
// The order of the additions is a function of the output element alone: K goes in steps of 16, the smallest third of x first, in
// chunks of 256 that are summed from zero and added one after the other; with few tiles the chunks are shared out over workgroups
// that leave their sums in a workspace, and a second kernel adds them in the same order.  A row has the same bits alone and among
// thousands.
//
// Three kernels (us; the float32 instruction's general kernel first, then these, weights of several products in turn):
//   tiles    x is cut on its way from registers to LDS.  Tiles of 64 x 128 by eight waves, or of 64 x 64 by four where those make at most a
//            workgroup a CU: x is cut once for every 128 columns (4.5 instructions an entry) and two waves a SIMD fill each other's
//            waits.  64 x 64 and 64 x 128: 566 rows, 6,144 x 1,024 36.1 and 30.8, 1,024 x 3,072 31.8 and 27.4; 2,048 rows, 6,144 x 1,024 114 and
//            100; 100 rows, 1,024 x 2,048 10.6 and 11.4.  (The general kernel 77 for the first, 45 for the second.)  Not taken: 64 x 256
//            and 128 x 128 by eight waves (29.9 and 30.8, but 13.9 and 13.6 for 11.4 at 33 rows), x in the operands' layout past LDS, which every
//            wave cuts (85), blocks of 64 k or loads two blocks ahead (64 and 63).
//   planes   products of several rounds: a kernel of its own cuts x (3 to 14 us), and all operands come straight to LDS in tiles of
//            128 x 256.  566 rows, 151,936 x 1,024 863 and 595 (1,541 in the general kernel); 2,048 rows, 24,576 x 4,096 1,635 and 1,093 (377
//            TFLOP/s: 1.13 of 10^15 products a second), 200 rows 220 and 166.
//   few      up to 16 rows: 24,576 x 4,096, 8 rows 78 and 56 (bound by w: 201 MB); 1 row, 6,144 x 1,024 17 and 13.
// Errors against 64 bits 2.9e-7 in the general kernel and 1.7e-7 here, because 16 products are added at a time.
//
// x is cut on its way from registers to LDS (an entry's remainder is one v_dot2_f32_bf16 with its pair of upper halves; a pair with an
// infinite entry spoils both of its entries, which are one row's).  Infinite entries have no such parts (inf - inf), nor have those of 2^88 and more, three parts
// of x times an infinite w are not x times it, and sums of 2^88 leave the range; all of them give infinity or NaN, and a chunk's sum that is
// not finite is made again from x and w as they are.
#include "common.h"

#include "gemm_split.h"
#include "gemm_tile.h"

namespace lc {

constexpr int GS_CHUNK = 256;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
constexpr float GS_UP = 0x1p40f, GS_DOWN = 0x1p-40f;

// Eight neighbouring entries of x, times GS_UP -> their three parts, operands of a product each.
__device__ __forceinline__ void cut_in_three(const float4& lo, const float4& hi, bf16x8 (&parts)[3]) {
    float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] *= GS_UP;
    // (-1, 0) and (0, -1), from registers: as a constant of the instruction -1 is read into the upper half
    unsigned first_bits = 0x0000BF80u, second_bits = 0xBF800000u;
    asm("" : "+s"(first_bits), "+s"(second_bits));
    const bf16x2 first = __builtin_bit_cast(bf16x2, first_bits), second = __builtin_bit_cast(bf16x2, second_bits);
#pragma unroll
    for (int part = 0; part < 3; ++part) {
        bf16x2 pairs[4];
#pragma unroll
        for (int e = 0; e < 8; e += 2) {            // the upper halves of two entries, and what they leave: one instruction an entry
            pairs[e / 2] = __builtin_bit_cast(bf16x2, __builtin_amdgcn_perm(__float_as_uint(v[e + 1]), __float_as_uint(v[e]), 0x07060302u));
            if (part < 2) {
                v[e] = __builtin_amdgcn_fdot2_f32_bf16(pairs[e / 2], first, v[e], false);
                v[e + 1] = __builtin_amdgcn_fdot2_f32_bf16(pairs[e / 2], second, v[e + 1], false);
            }
        }
        parts[part] = __builtin_bit_cast(bf16x8, pairs);
    }
}

// Eight neighbouring entries; WHOLE: aligned to 16 bytes, else one by one.
template <bool WHOLE>
__device__ __forceinline__ void load8(float4& lo, float4& hi, const float* from) {
    if (WHOLE) {
        lo = *reinterpret_cast<const float4*>(from);
        hi = *reinterpret_cast<const float4*>(from + 4);
    } else {
        lo = make_float4(from[0], from[1], from[2], from[3]);
        hi = make_float4(from[4], from[5], from[6], from[7]);
    }
}
template <bool WHOLE>
__device__ __forceinline__ bf16x8 load8(const bf16* from) {
    if (WHOLE) return *reinterpret_cast<const bf16x8*>(from);
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = from[e];
    return v;
}

// A chunk's sum that is not finite, from x and w as they are, one entry after the other; 16 entries are asked for at a time (one by one,
// each waited for its own trip to the caches, and rows behind the last once more: 1 row with a NaN, N 4,096, K 1,024 247 us, now 14, without the
// NaN 8; 566 rows of which one has it 49 and 31, 28 without).
template <bool WHOLE>
__device__ __forceinline__ float plain_sum(const float* x, const bf16* w, int k0, int k1) {
    float sum = 0.f;
#pragma unroll 1
    for (int k = k0; k < k1; k += 16) {             // K is a multiple of 32
        float4 a[4];
        bf16x8 b[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            load8<WHOLE>(a[2 * i], a[2 * i + 1], x + k + 8 * i);
            b[i] = load8<WHOLE>(w + k + 8 * i);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) sum = fmaf(reinterpret_cast<const float*>(a)[e], to_f32(b[e / 8][e % 8]), sum);
    }
    return sum;
}

// Tile BM x BN, WM x WN waves, KB k a block.  SHARED: blockIdx.z owns the chunks [z * per, (z + 1) * per) and leaves each chunk's sums in
// part[chunk][M][N].
template <int BM, int BN, int WM, int WN, int KB, bool WHOLE, bool SHARED>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_split_kernel(const float* __restrict__ x, const bf16* __restrict__ w, float* __restrict__ out,
                                                            int M, int N, int K, float* __restrict__ part, int per) {
    static_assert(GS_CHUNK % KB == 0, "whole blocks a chunk");
    constexpr int THREADS = 64 * WM * WN;
    constexpr int TM = BM / 32 / WM, TN = BN / 32 / WN;
    constexpr int PIECES = KB / 8, ROWS = THREADS / PIECES;          // 16-byte pieces a row and block, rows that the threads bring at once
    constexpr int XL = (BM + ROWS - 1) / ROWS, WL = BN / ROWS;
    constexpr int PLANE = BM * KB, STAGE = 3 * PLANE + BN * KB;  // entries
    __shared__ __attribute__((aligned(1024))) unsigned short lds[2 * STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);
    const int chunks = (K + GS_CHUNK - 1) / GS_CHUNK;
    const int c_begin = SHARED ? blockIdx.z * per : 0, c_end = SHARED ? min(c_begin + per, chunks) : chunks;
    if (c_begin >= c_end) return;

    // Piece c of row r lies at place c ^ swizzle(r), so that the 16 rows that LDS serves together meet no bank twice.  A row behind the
    // last is the last one again: its products go nowhere.
    auto swizzle = [](int r) { return (r / (128 / KB)) & (PIECES - 1); };
    const int row = tid / PIECES, piece = tid % PIECES;
    const float* xg[XL];
    const bf16* wg[WL];
#pragma unroll
    for (int i = 0; i < XL; ++i) xg[i] = x + (size_t)min(m0 + row + ROWS * i, M - 1) * K + piece * 8;
#pragma unroll
    for (int i = 0; i < WL; ++i) wg[i] = w + (size_t)min(n0 + row + ROWS * i, N - 1) * K + piece * 8;
    float4 xr[XL][2];
    bf16x8 wr[WL];
    auto fetch = [&](int k) {
#pragma unroll
        for (int i = 0; i < XL; ++i)
            if (BM % ROWS == 0 || row < BM) load8<WHOLE>(xr[i][0], xr[i][1], xg[i] + k);
#pragma unroll
        for (int i = 0; i < WL; ++i) wr[i] = load8<WHOLE>(wg[i] + k);
    };
    auto put = [&](int stage) {
        unsigned short* to = lds + stage * STAGE;
#pragma unroll
        for (int i = 0; i < WL; ++i) {
            const int r = row + ROWS * i;
            *reinterpret_cast<bf16x8*>(to + 3 * PLANE + r * KB + (piece ^ swizzle(r)) * 8) = wr[i];
        }
#pragma unroll
        for (int i = 0; i < XL; ++i)
            if (BM % ROWS == 0 || row < BM) {
                const int r = row + ROWS * i;
                bf16x8 parts[3];
                cut_in_three(xr[i][0], xr[i][1], parts);
#pragma unroll
                for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8*>(to + p * PLANE + r * KB + (piece ^ swizzle(r)) * 8) = parts[p];
            }
    };
    const int lr = lane & 31, kg = lane >> 5;
    auto operand = [&](const unsigned short* from, int r, int ks) {
        return *reinterpret_cast<const bf16x8*>(from + r * KB + ((2 * ks + kg) ^ swizzle(r)) * 8);
    };

    // K is a multiple of KB: every block is whole
    const int k_begin = c_begin * GS_CHUNK, k_limit = min(K, c_end * GS_CHUNK);
    floatx16 total[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) total[i][j][v] = 0.f;
    fetch(k_begin);
    put(0);
    fetch(min(k_begin + KB, k_limit - KB));
    int stage = 0;
    for (int c = c_begin; c < c_end; ++c) {
        floatx16 acc[TM][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
        const int k_end = min(K, (c + 1) * GS_CHUNK);
        for (int k = c * GS_CHUNK; k < k_end; k += KB) {
            __syncthreads();                    // this block is written by everybody, and the other stage read
            const unsigned short* from = lds + stage * STAGE;
#pragma unroll
            for (int ks = 0; ks < KB / 16; ++ks) {
                bf16x8 a[3][TM], b[TN];
#pragma unroll
                for (int j = 0; j < TN; ++j) b[j] = operand(from + 3 * PLANE, wn + 32 * j + lr, ks);
#pragma unroll
                for (int p = 2; p >= 0; --p)
#pragma unroll
                    for (int i = 0; i < TM; ++i) a[p][i] = operand(from + p * PLANE, wm + 32 * i + lr, ks);
                if (ks == 0) {
                    put(stage ^ 1);             // the next block (behind the last one: some block once more)
                    fetch(min(k + 2 * KB, k_limit - KB));
                }
#pragma unroll
                for (int p = 2; p >= 0; --p)
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int j = 0; j < TN; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[p][i], b[j], acc[i][j], 0, 0, 0);
            }
            stage ^= 1;
        }
        // lane l holds the rows (v / 4) * 8 + (l / 32) * 4 + v % 4 and column l % 32 of each of its products
        auto m_of = [&](int i, int v) { return m0 + wm + 32 * i + (v >> 2) * 8 + kg * 4 + (v & 3); };
        auto n_of = [&](int j) { return n0 + wn + 32 * j + lr; };
        bool bad = false;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    acc[i][j][v] *= GS_DOWN;
                    bad = bad || !(fabsf(acc[i][j][v]) < INFINITY);
                }
        if (__any(bad)) {
            int first = m0 + wm + kg * 4, n = n0 + wn + lr;
            asm volatile("" : "+v"(first), "+v"(n));        // or all rows' addresses are made before the loop and kept in registers
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int m = first + 32 * i + (v >> 2) * 8 + (v & 3);
                        if (!(fabsf(acc[i][j][v]) < INFINITY) && m < M)
                            acc[i][j][v] = plain_sum<WHOLE>(x + (size_t)m * K, w + (size_t)min(n + 32 * j, N - 1) * K, c * GS_CHUNK, k_end);
                    }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    if (SHARED) {
                        if (m_of(i, v) < M && n_of(j) < N) part[((size_t)c * M + m_of(i, v)) * N + n_of(j)] = acc[i][j][v];
                    } else {
                        total[i][j][v] = __fadd_rn(total[i][j][v], acc[i][j][v]);
                    }
                }
    }
    if (SHARED) return;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int m = m0 + wm + 32 * i + (v >> 2) * 8 + kg * 4 + (v & 3), n = n0 + wn + 32 * j + lr;
                if (m < M && n < N) out[(size_t)m * N + n] = total[i][j][v];
            }
}

// Up to 16 rows: a chunk of x lies in LDS in its three parts, and each of the four waves streams its 32 rows of w past it, a chunk's 16
// loads asked for together in the operands' own layout: nothing is staged and nothing waited for in between.  The products and
// their order are those of the tiles; rows 16 to 31 of a product are the first 16 once more.
constexpr int GS_FEW = 16, GS_FEW_N = 128;

template <bool WHOLE, bool SHARED>
__global__ __launch_bounds__(256, 2) void gemm_split_few_kernel(const float* __restrict__ x, const bf16* __restrict__ w, float* __restrict__ out,
                                                                int M, int N, int K, float* __restrict__ part, int per) {
    constexpr int STEPS = GS_CHUNK / 16, PIECES = GS_CHUNK / 8;
    __shared__ __attribute__((aligned(16))) unsigned short lds[3 * GS_FEW * GS_CHUNK];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 31, kg = lane >> 5;
    const int n0 = blockIdx.x * GS_FEW_N + wave * 32, n = n0 + lr;
    const int chunks = (K + GS_CHUNK - 1) / GS_CHUNK;
    const int c_begin = SHARED ? blockIdx.z * per : 0, c_end = SHARED ? min(c_begin + per, chunks) : chunks;
    const bf16* wg = w + (size_t)min(n, N - 1) * K + 8 * kg;
    const int row = tid / 16;
    const float* xg = x + (size_t)min(row, M - 1) * K;
    floatx16 total;
#pragma unroll
    for (int v = 0; v < 16; ++v) total[v] = 0.f;
    for (int c = c_begin; c < c_end; ++c) {
        const int k0 = c * GS_CHUNK, k_end = min(K, k0 + GS_CHUNK), steps = (k_end - k0) / 16;      // K is a multiple of 32
        bf16x8 b[STEPS];
        if (steps == STEPS) {
#pragma unroll
            for (int s = 0; s < STEPS; ++s) b[s] = load8<WHOLE>(wg + k0 + 16 * s);
        } else {
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
                if (s < steps) b[s] = load8<WHOLE>(wg + k0 + 16 * s);
        }
        if (c > c_begin) __syncthreads();       // the chunk before is read by everybody
#pragma unroll
        for (int i = 0; i < PIECES / 16; ++i) {
            // piece p of row r lies at place p ^ r: the 16 rows that LDS serves together meet no bank twice
            const int piece = tid % 16 + 16 * i;
            if (k0 + 8 * piece < k_end) {
                bf16x8 parts[3];
                float4 lo, hi;
                load8<WHOLE>(lo, hi, xg + k0 + 8 * piece);
                cut_in_three(lo, hi, parts);
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    *reinterpret_cast<bf16x8*>(lds + (p * GS_FEW + row) * GS_CHUNK + (piece ^ row) * 8) = parts[p];
            }
        }
        __syncthreads();
        floatx16 acc;
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v] = 0.f;
#pragma unroll
        for (int s = 0; s < STEPS; ++s)
            if (s < steps)
#pragma unroll
                for (int p = 2; p >= 0; --p) {
                    const int r = lr & (GS_FEW - 1);
                    const bf16x8 a = *reinterpret_cast<const bf16x8*>(lds + (p * GS_FEW + r) * GS_CHUNK + ((2 * s + kg) ^ r) * 8);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[s], acc, 0, 0, 0);
                }
        bool bad = false;
#pragma unroll
        for (int v = 0; v < 8; ++v) {           // the rows up to 15
            acc[v] *= GS_DOWN;
            bad = bad || !(fabsf(acc[v]) < INFINITY);
        }
        if (__any(bad)) {
#pragma unroll
            for (int v = 0; v < 8; ++v)
                if (!(fabsf(acc[v]) < INFINITY) && (v >> 2) * 8 + kg * 4 + (v & 3) < M)
                    acc[v] = plain_sum<WHOLE>(x + (size_t)((v >> 2) * 8 + kg * 4 + (v & 3)) * K, w + (size_t)min(n, N - 1) * K, k0, k_end);
        }
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            const int m = (v >> 2) * 8 + kg * 4 + (v & 3);
            if (SHARED) {
                if (m < M && n < N) part[((size_t)c * M + m) * N + n] = acc[v];
            } else {
                total[v] = __fadd_rn(total[v], acc[v]);
            }
        }
    }
    if (SHARED) return;
#pragma unroll
    for (int v = 0; v < 8; ++v) {
        const int m = (v >> 2) * 8 + kg * 4 + (v & 3);
        if (m < M && n < N) out[(size_t)m * N + n] = total[v];
    }
}

// x [M, K] -> its three parts, planes [3][M][K]; a thread takes eight neighbouring entries.
template <bool WHOLE>
__global__ __launch_bounds__(256) void cut_planes_kernel(const float* __restrict__ x, unsigned short* __restrict__ planes, size_t pieces) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < pieces; i += (size_t)gridDim.x * 256) {
        float4 lo, hi;
        load8<WHOLE>(lo, hi, x + 8 * i);
        bf16x8 parts[3];
        cut_in_three(lo, hi, parts);
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8*>(planes + ((size_t)p * pieces + i) * 8) = parts[p];
    }
}

// The product of the planes: tiles of BM x BN, WM x WN waves, blocks of 32 k in a ring of S stages that direct loads fill S - 1 blocks ahead.
// A block's second k-step's operands are in registers before its barrier, so that its stage is free behind it and the next block's
// first operands are asked for before the last products.  Tiles go in strips of GP_STRIP rows of tiles, which an XCD's L2 serves.
constexpr int GP_K = 32, GP_STRIP = 8, GP_M = 128, GP_N = 256;
template <int BM, int BN, int WM, int WN, int S>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_planes_kernel(const unsigned short* __restrict__ planes, const bf16* __restrict__ w,
                                                                      const float* __restrict__ x, float* __restrict__ out, int M, int N, int K,
                                                                      int tiles_m) {
    constexpr int NW = WM * WN, TM = BM / 32 / WM, TN = BN / 32 / WN;
    constexpr int PLANE = BM * GP_K * 2, STAGE = 3 * PLANE + BN * GP_K * 2;       // bytes
    constexpr int LX = 3 * BM / 16 / NW, LW = BN / 16 / NW, LP = LX + LW;         // load instructions a wave and block
    static_assert(3 * BM % (16 * NW) == 0 && BN % (16 * NW) == 0, "whole load instructions per wave");
    static_assert(S * STAGE <= 160 * 1024 && S >= 3, "LDS");
    __shared__ __attribute__((aligned(1024))) char lds[S * STAGE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int total_tiles = gridDim.x, share = total_tiles >> 3, xcd = blockIdx.x & 7, tiles_n = total_tiles / tiles_m;
    int id = xcd * share + min(xcd, total_tiles & 7) + (blockIdx.x >> 3);          // an XCD takes neighbouring tiles
    const int first_row = id / (GP_STRIP * tiles_n) * GP_STRIP, rows = min(GP_STRIP, tiles_m - first_row);
    id -= first_row * tiles_n;
    const int n0 = id / rows * BN, m0 = (first_row + id % rows) * BM;
    const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);
    const int blocks = K / GP_K;

    auto swizzle = [](int r) { return (r >> 2) & 3; };
    // a load instruction brings 16 rows: lane l the piece at place l % 4 of row l / 4
    const unsigned short* from[LP];
#pragma unroll
    for (int i = 0; i < LP; ++i) {
        const int j = (i < LX ? i : i - LX) * NW + wave, r = (i < LX ? j % (BM / 16) : j) * 16 + (lane >> 2);
        const int piece = (lane & 3) ^ swizzle(r);
        from[i] = i < LX ? planes + ((size_t)(j / (BM / 16)) * M + min(m0 + r, M - 1)) * K + piece * 8
                         : reinterpret_cast<const unsigned short*>(w) + (size_t)min(n0 + r, N - 1) * K + piece * 8;
    }
    auto issue = [&](int b, int stage) {
#pragma unroll
        for (int i = 0; i < LP; ++i)
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(from[i] + b * GP_K),
                (lds_ptr_t)(lds + stage * STAGE + (i < LX ? 0 : 3 * PLANE) + ((i < LX ? i : i - LX) * NW + wave) * 1024), 16, 0, 0);
    };
    const int lr = lane & 31, kg = lane >> 5;
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t)lds;
    unsigned pa[TM], pb[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int r = wm + 32 * i + lr;
        pa[i] = lds0 + r * 64 + ((kg ^ swizzle(r)) * 16);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int r = wn + 32 * j + lr;
        pb[j] = lds0 + 3 * PLANE + r * 64 + ((kg ^ swizzle(r)) * 16);
    }
    bf16x8 a[2][3][TM], b[2][TN];
    // in inline assembly, because the compiler would wait for every load to LDS in flight before an LDS read
    auto read = [&](int stage, int ks, int set) {
        const unsigned at = stage * STAGE;
#pragma unroll
        for (int j = 0; j < TN; ++j) asm volatile("ds_read_b128 %0, %1" : "=v"(b[set][j]) : "v"((pb[j] ^ (ks * 32)) + at));
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
            for (int i = 0; i < TM; ++i)
                asm volatile("ds_read_b128 %0, %1" : "=v"(a[set][p][i]) : "v"((pa[i] ^ (ks * 32)) + at + p * PLANE));
    };
    auto landed = [&](int set) {            // the products that follow stay behind the wait
        wait_lgkmcnt<0>();
#pragma unroll
        for (int j = 0; j < TN; ++j) asm volatile("" : "+v"(b[set][j]));
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int i = 0; i < TM; ++i) asm volatile("" : "+v"(a[set][p][i]));
        __builtin_amdgcn_sched_barrier(0);
    };
    floatx16 total[TM][TN], acc[TM][TN];
    auto products = [&](int set) {
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[set][p][i], b[set][j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto clear = [&](floatx16 (&t)[TM][TN]) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) t[i][j][v] = 0.f;
    };
    clear(total);
    clear(acc);
#pragma unroll
    for (int s = 0; s < S - 1; ++s)
        if (s < blocks) issue(s, s);
    // block 0: this wave's part, then everybody's
    if (blocks >= S - 1) wait_vmcnt<(S - 2) * LP>();
    else wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    read(0, 0, 0);
    int stage = 0;
    for (int it = 0; it < blocks; ++it) {
        const int next = stage + 1 == S ? 0 : stage + 1, last = stage == 0 ? S - 1 : stage - 1;
        landed(0);
        // the stage of the block before is free: everybody had its last operands at the barrier behind it
        if (it + S - 1 < blocks) issue(it + S - 1, last);
        read(stage, 1, 1);
        __builtin_amdgcn_sched_barrier(0);
        products(0);
        landed(1);
        if (it + 1 < blocks) {
            // block it + 1 has landed (this wave's part, then everybody's), and nobody reads this stage any more
            if (it + S - 1 < blocks) wait_vmcnt<(S - 2) * LP>();
            else wait_vmcnt<0>();
            __builtin_amdgcn_s_barrier();
            read(next, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        products(1);
        stage = next;
        if ((it + 1) % (GS_CHUNK / GP_K) != 0 && it + 1 < blocks) continue;
        const int c = it / (GS_CHUNK / GP_K), k_end = min(K, (c + 1) * GS_CHUNK);
        bool bad = false;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    acc[i][j][v] *= GS_DOWN;
                    bad = bad || !(fabsf(acc[i][j][v]) < INFINITY);
                }
        if (__any(bad)) {
            int first = m0 + wm + kg * 4, n = n0 + wn + lr;
            asm volatile("" : "+v"(first), "+v"(n));
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int m = first + 32 * i + (v >> 2) * 8 + (v & 3);
                        if (!(fabsf(acc[i][j][v]) < INFINITY) && m < M)
                            acc[i][j][v] = plain_sum<false>(x + (size_t)m * K, w + (size_t)min(n + 32 * j, N - 1) * K, c * GS_CHUNK, k_end);
                    }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) total[i][j][v] = __fadd_rn(total[i][j][v], acc[i][j][v]);
        clear(acc);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int m = m0 + wm + 32 * i + (v >> 2) * 8 + kg * 4 + (v & 3), n = n0 + wn + 32 * j + lr;
                if (m < M && n < N) out[(size_t)m * N + n] = total[i][j][v];
            }
}

bool gemm_split_takes(int K) { return K % 32 == 0; }

// gemm_planes_kernel reads LDS by inline assembly into registers that the compiler takes to hold values before its wait for them: were
// one spilled to scratch memory in between, the spill would store what the register held before.  So the compiled kernel is asked, once:
// if it uses scratch memory (or cannot be asked), products go by tiles.
static int planes_state() {          // 1: in registers, 0: spilled, -1: could not ask
    static const int state = [] {
        hipFuncAttributes attr;
        if (hipFuncGetAttributes(&attr, (const void*)gemm_planes_kernel<GP_M, GP_N, 2, 4, 4>) != hipSuccess) {
            (void)hipGetLastError();
            return -1;
        }
        return attr.localSizeBytes != 0 ? 0 : 1;
    }();
    return state;
}
LC_API int lc_gemm_planes_ok() { return planes_state(); }

// Whether a product goes by planes.  A round of 256 tiles of 128 x 256 takes 1.53 times as long as one of 512 tiles of 64 x 128, which is
// half as many places (K of 4,096: 182 and 119 us where several rounds follow each other); fewer whole rounds than that pay for the
// cut.  us, tiles of 64 x 128 and planes: 300 rows, 24,576 x 4,096 (2 rounds each) 244 and 314, 566 rows (4 and 2) 424 and 357, 100 rows (1 and 1)
// 118 and 156; 566 rows, 151,936 x 1,024 (21 and 12) 787 and 595; 2,048 rows, 6,144 x 1,024 (3 and 2) 100 and 94 + 5.
static bool planes_pay(int M, int N, int K) {
    if (M <= GS_FEW || !gemm_split_takes(K)) return false;
    auto rounds = [](long long m, long long n, int bm, int bn, int places) {
        return ((m + bm - 1) / bm * ((n + bn - 1) / bn) + places - 1) / places;
    };
    return 1.53 * rounds(M, N, GP_M, GP_N, device_cus()) < rounds(M, N, 64, 128, 2 * device_cus()) &&
           (long long)((M + GP_M - 1) / GP_M) * ((N + GP_N - 1) / GP_N) < 1ll << 30 && planes_state() == 1;
}

// Rows whose parts are in the workspace at once: no more than 64 M words (256 MiB) of them, in whole tiles.
static int rows_at_once(int M, int K) {
    const long long most = (128ll << 20) / 3 / K / GP_M * GP_M;
    return M <= most ? M : most < GP_M ? GP_M : (int)most;
}

long long gemm_split_words(int M, int N, int K) { return planes_pay(M, N, K) ? (3ll * rows_at_once(M, K) * K + 1) / 2 : 0; }

template <bool WHOLE, bool SHARED>
static void launch_split(const float* x, const bf16* w, float* out, int M, int N, int K, float* part, int per, int shares, hipStream_t stream) {
    if (M <= GS_FEW)
        gemm_split_few_kernel<WHOLE, SHARED><<<dim3((N + GS_FEW_N - 1) / GS_FEW_N, 1, shares), 256, 0, stream>>>(x, w, out, M, N, K, part, per);
    else if ((long long)((N + 63) / 64) * ((M + 63) / 64) * shares > device_cus())
        gemm_split_kernel<64, 128, 2, 4, 32, WHOLE, SHARED><<<dim3((N + 127) / 128, (M + 63) / 64, shares), 512, 0, stream>>>(x, w, out, M, N, K,
                                                                                                                     part, per);
    else
        gemm_split_kernel<64, 64, 2, 2, 32, WHOLE, SHARED><<<dim3((N + 63) / 64, (M + 63) / 64, shares), 256, 0, stream>>>(x, w, out, M, N, K,
                                                                                                                    part, per);
}

void launch_gemm_split(const float* x, const bf16* w, float* out, int M, int N, int K, float* part, int per, int shares, float* workspace,
                       hipStream_t stream) {
    if (!part && workspace && (uintptr_t)w % 16 == 0 && (uintptr_t)workspace % 16 == 0 && planes_pay(M, N, K)) {
        unsigned short* planes = reinterpret_cast<unsigned short*>(workspace);
        const int at_once = rows_at_once(M, K);
        for (int first = 0; first < M; first += at_once) {          // one after the other in the workspace
            const int rows = M - first < at_once ? M - first : at_once;
            const float* from = x + (size_t)first * K;
            const size_t pieces = (size_t)rows * K / 8;
            const int blocks = (int)((pieces + 255) / 256 < 2048 ? (pieces + 255) / 256 : 2048);
            if ((uintptr_t)x % 16 == 0) cut_planes_kernel<true><<<blocks, 256, 0, stream>>>(from, planes, pieces);
            else cut_planes_kernel<false><<<blocks, 256, 0, stream>>>(from, planes, pieces);
            const int tiles_m = (rows + GP_M - 1) / GP_M, tiles_n = (N + GP_N - 1) / GP_N;
            gemm_planes_kernel<GP_M, GP_N, 2, 4, 4><<<tiles_m * tiles_n, 512, 0, stream>>>(planes, w, from, out + (size_t)first * N, rows, N, K, tiles_m);
        }
        return;
    }
    const bool whole = ((uintptr_t)x | (uintptr_t)w) % 16 == 0;
    if (whole && part) launch_split<true, true>(x, w, out, M, N, K, part, per, shares, stream);
    else if (whole) launch_split<true, false>(x, w, out, M, N, K, part, per, shares, stream);
    else if (part) launch_split<false, true>(x, w, out, M, N, K, part, per, shares, stream);
    else launch_split<false, false>(x, w, out, M, N, K, part, per, shares, stream);
}

}  // namespace lc
