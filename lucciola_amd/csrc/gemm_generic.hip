// out[M, N] = x[M, K] . w[N, K]^T for any sizes and any mix of float32 / bfloat16 operands, as a
// true 32-bit product: the operands are widened to float32 and multiplied on the matrix cores in
// float32 (v_mfma_f32_16x16x4_f32: float32 products, float32 sums, no reduced-precision mode).
// The weight layout is the checkpoint's: [out_features, in_features] row-major, applied as
// y = x . W^T without bias (reference: src/kernels/linear.cu:24-27, one thread per output
// element; here tiles of 128 x 128, 64 x 64 or, for up to 16 rows, 16 x 64, staged through LDS
// 16 k at a time, four waves with a grid of 16 x 16 products each).
//
// The order of the additions is a function of the output element alone: K is cut into chunks of
// 256; within a chunk the element's sum takes four k at a time, in order (one matrix
// instruction each, the same in every tile shape), and the chunks' sums are added one after the
// other from 0.  With few tiles (a decode step: up to 64 rows and a narrow N) the chunks are
// shared out over workgroups, which leave their sums in a workspace, and a second kernel adds
// them in the same order: a row's result has the same bits whether it is computed alone or
// among thousands.
//
// float32 x by bfloat16 w in whole steps of 32 k has kernels of its own, twice as fast (gemm_split.hip); this entry's workspace and the sum
// of shared chunks serve both.
//
// The figures here are of what those kernels replaced, the product with bfloat16 w on the float32 instruction; the loop is the one
// that float32 w, float32 x of a broken K and 16-bit x of a broken K still run.
//
// Bound by the matrix instruction: 143 TFLOP/s from registers alone on this card.  What kept the first form of the loop
// at 88 (2,048 x 4,096 x 1,024, bfloat16 w, 195 us) was what stood between the products: loads behind a test of k each, whose rows
// were set to zero right behind them, so that each waited for its own trip; LDS writes four to a bank; and all of a stage's LDS work
// in one heap, in which the matrix core had nothing to do.  Now 156 us (110).  566 rows: N 6,144, K 1,024 110 -> 79 us, N 1,024, K 3,072
// 61 -> 46, N 151,936 2,272 -> 1,728; 8 rows, N 6,144 13.6 -> 9.0.
#include "common.h"
#include "gemm_split.h"

#include <type_traits>

namespace lc {

constexpr int GB_M = 64, GB_N = 64, GB_K = 16;
constexpr int GB_CHUNK = 256;   // k elements whose products are added up before they join the total
typedef float floatx4 __attribute__((ext_vector_type(4)));

// four neighbouring k of a row, one load; at(j): entry j, widened
template <typename T> struct Piece;
template <> struct __attribute__((aligned(16))) Piece<float> {
    float v[4];
    __device__ __forceinline__ float at(int j) const { return v[j]; }
    __device__ __forceinline__ void set(int j, const float* p) { v[j] = p ? *p : 0.f; }
};
template <> struct __attribute__((aligned(8))) Piece<bf16> {
    unsigned v[2];
    __device__ __forceinline__ float at(int j) const {
        return __uint_as_float(j & 1 ? v[j / 2] & 0xFFFF0000u : v[j / 2] << 16);
    }
    __device__ __forceinline__ void set(int j, const bf16* p) {
        const unsigned bits = p ? (unsigned)__builtin_bit_cast(unsigned short, *p) : 0u;
        v[j / 2] = j & 1 ? (v[j / 2] & 0xFFFFu) | bits << 16 : bits;
    }
};

// Tile BM x BN, WM x WN waves, each with (BM / 16 / WM) x (BN / 16 / WN) products of 16 x 16.
// part == nullptr: out = x . w^T.  Else blockIdx.z owns the chunks [z * per, (z + 1) * per) and
// writes each chunk's sums to part[chunk][M][N].
//
// WHOLE: K is a multiple of two stages and x and w are aligned to 16 bytes, so that every load is a whole
// piece.  Then nothing stands between a stage's loads and their use at the stage's end: no test of
// k, and no test whether there is a next stage (behind the last one it is the last one again).  A row behind the
// last is the last one again: its products go nowhere.
template <typename TX, typename TW, typename TO, int BM, int BN, int WM, int WN, bool WHOLE, bool SHARED>
__global__ __launch_bounds__(256, 2) void gemm_generic_kernel(const TX* __restrict__ x,
                                                           const TW* __restrict__ w,
                                                           TO* __restrict__ out, int M, int N,
                                                           int K, float* __restrict__ part, int per) {
    static_assert(WM * WN == 4, "four waves");
    constexpr int TM = BM / 16 / WM, TN = BN / 16 / WN;
    constexpr int XL = (BM * 4 + 255) / 256, WL = (BN * 4 + 255) / 256;   // 16-byte pieces a thread loads per stage
    // Two stages: one is filled while the other is multiplied.  Row r of k lies at place
    // r ^ 16 ((k % 4) ^ (k / 4)): the four k of a wave's read (16 rows each) and the four k / 4 of a wave's
    // write (16 rows each) then each lie in banks of their own.
    constexpr int P = BN < 64 ? 64 : BN, STAGE = 2 * GB_K * P;     // floats: a stage's x, then its w
    static_assert(BM <= P, "x's rows have the places of w's");
    __shared__ float lds[2 * STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);
    const int chunks = (K + GB_CHUNK - 1) / GB_CHUNK;
    const int c_begin = SHARED ? blockIdx.z * per : 0;
    const int c_end = SHARED ? min(c_begin + per, chunks) : chunks;
    if (c_begin >= c_end) return;
    floatx4 total[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) total[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    // loader mapping: rows x 16 k; a thread loads 4 consecutive k of a row (of up to XL rows of x
    // and WL of w, 64 apart), a step ahead of the products that use them (the loads of step
    // k0 + 16 are in flight while step k0 is multiplied)
    const int lrow = tid / 4, lk = (tid % 4) * 4;
    // whole 16-byte (8-byte) pieces where the row length allows it
    const bool vec = WHOLE || ((K & 3) == 0 && ((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0));
    Piece<TX> xr[XL];               // as they came: widened on the way to LDS, so that nothing waits for them before
    Piece<TW> wr[WL];
    auto fetch_rows = [&](auto* rows_ptr, int first, int limit, int count, auto* dst, int k0) {
        typedef std::remove_reference_t<decltype(*dst)> P;
#pragma unroll
        for (int u = 0; u < count; ++u) {
            const int row = lrow + 64 * u;
            const auto* p = rows_ptr + (size_t)min(first + row, limit - 1) * K + lk;
            if (WHOLE || (vec && k0 + GB_K <= K)) {         // all four of a row's threads alike: one test a stage
                dst[u] = *reinterpret_cast<const P*>(p + k0);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) dst[u].set(j, k0 + lk + j < K ? p + k0 + j : nullptr);
            }
        }
    };
    auto fetch = [&](int k0) {
        fetch_rows(x, m0, M, XL, xr, k0);
        fetch_rows(w, n0, N, WL, wr, k0);
    };
    // Where this lane writes entry j of its pieces, and where it reads: with wm and wn multiples of TM and TN tiles, tile i of
    // quarter q lies at ((wm / 16) ^ i ^ q ^ g), so that four addresses and constant offsets reach all of them.
    const int g = lane >> 4;
    float* to[4];
    const float* from_x[4];
    const float* from_w[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        to[v] = lds + (lk + v) * P + (lrow ^ (16 * (v ^ (tid & 3))));
        from_x[v] = lds + g * P + 16 * ((wm / 16) ^ v ^ g) + (lane & 15);
        from_w[v] = lds + (GB_K + g) * P + 16 * ((wn / 16) ^ v ^ g) + (lane & 15);
    }
    constexpr int PUTS = 4 * (XL + WL), NM = TM * TN, NR = TM + TN;
    auto put_one = [&](int n, int stage) {
        const int u = n / 4, j = n % 4;
        if (u < XL) {
            if (BM % 64 == 0 || lrow + 64 * u < BM) to[j][stage * STAGE + 64 * u] = xr[u < XL ? u : 0].at(j);
        } else {
            to[j][stage * STAGE + GB_K * P + 64 * (u - XL)] = wr[u < XL ? 0 : u - XL].at(j);
        }
    };
    // the operands of the four k of quarter q: lane l brings x[row l % 16][k l / 16] of each of its tiles, and w likewise
    float a[2][TM], b[2][TN];
    auto read_one = [&](int r, int stage, int q, int buf) {
        if (r < TM) a[buf][r < TM ? r : 0] = from_x[(r ^ q) & 3][stage * STAGE + 4 * q * P];
        else b[buf][r < TM ? 0 : r - TM] = from_w[((r - TM) ^ q) & 3][stage * STAGE + 4 * q * P];
    };
    static_assert(TM <= 4 && TN <= 4 && BN % 64 == 0, "the places above");
    // Every step of 16 k, over all of this workgroup's chunks, is a stage.  While stage s is
    // multiplied, a quarter at a time, the next quarter's operands are read; in its first quarter
    // stage s + 1, whose loads left a stage ago, goes to LDS, in its second the loads of stage s + 2 leave;
    // in its last the waves meet: s + 1 is then written by everybody, and s read.  Each of these goes behind a
    // product of its own: the matrix core is busy with it for 32 clocks, in which the wave issues other work,
    // and what the wave issues beyond that is the matrix core's idle time.
    const int k_begin = c_begin * GB_CHUNK, k_limit = min(K, c_end * GB_CHUNK);
    // The last stage.  Stages go in pairs (a chunk but the last has 16); a K that is not whole may end with half a pair.
    const int k_last = k_begin + (k_limit - k_begin + GB_K - 1) / GB_K * GB_K - GB_K;
    fetch(k_begin);
#pragma unroll
    for (int n = 0; n < PUTS; ++n) put_one(n, 0);
    fetch(min(k_begin + GB_K, k_last));
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NR; ++r) read_one(r, 0, 0, 0);
    for (int c = c_begin; c < c_end; ++c) {
        floatx4 acc[TM][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        constexpr int BAR = NM / 4, AFTER = NM - BAR;              // products of the last quarter before the barrier, and behind it
        constexpr int QR = (NR + NM - 1) / NM, QB = (NR + AFTER - 1) / AFTER, QP = (PUTS + NM - 1) / NM;
        auto step = [&](int k0, auto stage_tag) {
            constexpr int stage = decltype(stage_tag)::value;
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int k = 0; k < NM; ++k) {
                    const int i = k / TN, j = k % TN;
                    if (q == 3 && k == BAR) __syncthreads();
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q & 1][i], b[q & 1][j], acc[i][j], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (q < 3) {
#pragma unroll
                        for (int r = k * QR; r < (k + 1) * QR; ++r)
                            if (r < NR) read_one(r, stage, q + 1, (q + 1) & 1);
                    } else if (k >= BAR) {
#pragma unroll
                        for (int r = (k - BAR) * QB; r < (k - BAR + 1) * QB; ++r)
                            if (r < NR) read_one(r, stage ^ 1, 0, 0);        // behind the last stage: that stage once more
                    }
                    if (q == 0) {
#pragma unroll
                        for (int n = k * QP; n < (k + 1) * QP; ++n)
                            if (n < PUTS) put_one(n, stage ^ 1);
                    }
                    if (q == 1 && k == NM / 2) fetch(min(k0 + 2 * GB_K, k_last));
                    __builtin_amdgcn_sched_barrier(0);
                }
        };
        const int k_end = min(K, (c + 1) * GB_CHUNK);
        for (int k0 = c * GB_CHUNK; k0 < k_end; k0 += 2 * GB_K) {
            step(k0, std::integral_constant<int, 0>{});
            if (WHOLE || k0 + GB_K < k_end) step(k0 + GB_K, std::integral_constant<int, 1>{});
        }
        // lane l holds the rows 4 (l / 16) + r and the column l % 16 of each of its tiles
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (SHARED) {
                        const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + r, n = n0 + wn + 16 * j + (lane & 15);
                        if (m < M && n < N) part[((size_t)c * M + m) * N + n] = acc[i][j][r];
                    } else {
                        total[i][j][r] = __fadd_rn(total[i][j][r], acc[i][j][r]);
                    }
                }
    }
    if (SHARED) return;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + r, n = n0 + wn + 16 * j + (lane & 15);
                if (m < M && n < N) out[(size_t)m * N + n] = from_f32<TO>(total[i][j][r]);
            }
}

constexpr int GF_M = 16;        // rows of the tile for a decode step's few rows

// out = the chunks' sums part[c][M][N] added one after the other from 0, as the kernel above
// adds them when it keeps them to itself
template <typename TO, int VEC>
__global__ void gemm_generic_sum_kernel(const float* __restrict__ part, TO* __restrict__ out, size_t MN,
                                        int chunks) {
    for (size_t idx = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * VEC; idx < MN;
         idx += (size_t)gridDim.x * blockDim.x * VEC) {
        float total[VEC] = {};
#pragma unroll 4
        for (int c = 0; c < chunks; ++c) {
            float got[VEC];
            if constexpr (VEC == 4) load4(got, part + (size_t)c * MN + idx);
            else got[0] = part[(size_t)c * MN + idx];
#pragma unroll
            for (int e = 0; e < VEC; ++e) total[e] = __fadd_rn(total[e], got[e]);
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) out[idx + e] = from_f32<TO>(total[e]);
    }
}

// Chunks a workgroup takes when they are shared out (0: they are not): with fewer than 512
// tiles, as many workgroups as it takes to have about 2048, if the workspace stays modest.  512 tiles are two
// a CU, and a CU keeps five: sharing out then costs the chunks' way through memory and gains nothing (566 rows, K 1,024: N 6,144,
// 864 tiles, 89 us shared out and 80 not; N 4,096, 576 tiles, 61 and 61; 400 rows, 448 tiles: 49 shared out).
static int chunks_per_workgroup(int M, int N, int K) {
    const long long tiles = (long long)((N + GB_N - 1) / GB_N) * ((M + GB_M - 1) / GB_M);
    const int chunks = (K + GB_CHUNK - 1) / GB_CHUNK;
    if (tiles >= 512 || chunks < 2) return 0;
    // the workspace holds every chunk's sums for all of M x N: no more than 64 M floats (256 MiB),
    // beyond which the chunks stay with their tile (the same additions in the same order)
    if ((long long)chunks * M * N > (64ll << 20)) return 0;
    long long shares = (2048 + tiles - 1) / tiles;
    if (shares > chunks) shares = chunks;
    if (shares < 2) return 0;
    return (int)((chunks + shares - 1) / shares);
}

template <typename TX, typename TW, typename TO>
static int launch_generic(const void* x, const void* w, void* out, int M, int N, int K, float* workspace,
                          hipStream_t stream) {
    const int per = chunks_per_workgroup(M, N, K);
    const int chunks = (K + GB_CHUNK - 1) / GB_CHUNK;
    const bool few = M <= GF_M;
    // tiles of 128 x 128 where they fill the card (they bring half as many bytes into a CU per product)
    const bool large = per == 0 && M > GB_M && (long long)((N + 127) / 128) * ((M + 127) / 128) >= device_cus();
    float* part = nullptr;
    int shares = 1;
    if (per > 0) {
        LC_CHECK(workspace, "gemm: M=%d N=%d K=%d needs a workspace", M, N, K);
        part = workspace;
        shares = (chunks + per - 1) / per;
    }
    const bool whole = K % (2 * GB_K) == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0;
    auto launch = [&](auto rows, auto cols, auto wave_rows, auto is_whole, auto is_shared) {
        constexpr int BM = decltype(rows)::value, BN = decltype(cols)::value, WM = decltype(wave_rows)::value;
        const dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM, shares);
        gemm_generic_kernel<TX, TW, TO, BM, BN, WM, 4 / WM, decltype(is_whole)::value, decltype(is_shared)::value>
            <<<grid, 256, 0, stream>>>((const TX*)x, (const TW*)w, (TO*)out, M, N, K, part, per);
    };
    auto with_shape = [&](auto is_whole) {
        typedef std::integral_constant<int, 128> Large;
        typedef std::integral_constant<int, GF_M> Few;
        typedef std::integral_constant<int, GB_M> Tile;
        const std::integral_constant<int, 1> one{};
        const std::integral_constant<int, 2> two{};
        if (few && part) launch(Few{}, Tile{}, one, is_whole, std::true_type{});
        else if (few) launch(Few{}, Tile{}, one, is_whole, std::false_type{});
        else if (large) launch(Large{}, Large{}, two, is_whole, std::false_type{});
        else if (part) launch(Tile{}, Tile{}, two, is_whole, std::true_type{});
        else launch(Tile{}, Tile{}, two, is_whole, std::false_type{});
    };
    constexpr bool SPLITS = std::is_same_v<TX, float> && std::is_same_v<TW, bf16> && std::is_same_v<TO, float>;
    if constexpr (SPLITS) {             // a K that is whole has kernels of its own
        if (gemm_split_takes(K)) launch_gemm_split((const float*)x, (const bf16*)w, (float*)out, M, N, K, part, per, shares, per > 0 ? nullptr : workspace, stream);
        else with_shape(std::false_type{});
    } else {
        if (whole) with_shape(std::true_type{});
        else with_shape(std::false_type{});
    }
    LC_LAUNCH_CHECK("gemm_generic");
    if (per > 0 && out) {
        const size_t MN = (size_t)M * N;
        const size_t threads = MN % 4 == 0 ? MN / 4 : MN;
        const int blocks = (int)((threads + 255) / 256 < 4096 ? (threads + 255) / 256 : 4096);
        if (MN % 4 == 0) gemm_generic_sum_kernel<TO, 4><<<blocks, 256, 0, stream>>>(workspace, (TO*)out, MN, chunks);
        else gemm_generic_sum_kernel<TO, 1><<<blocks, 256, 0, stream>>>(workspace, (TO*)out, MN, chunks);
        LC_LAUNCH_CHECK("gemm_generic_sum");
    }
    return 0;
}

}  // namespace lc

using namespace lc;

// float32 words of workspace that lc_gemm_generic needs for these sizes (0: none), of whatever types the operands are
LC_API long long lc_gemm_generic_workspace(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    return chunks_per_workgroup(M, N, K) > 0 ? (long long)((K + GB_CHUNK - 1) / GB_CHUNK) * M * N : gemm_split_words(M, N, K);
}

// ... and of these types: x's parts are laid out for float32 x, bfloat16 w and a float32 result alone
LC_API long long lc_gemm_generic_workspace_of(int M, int x_dt, int N, int w_dt, int K, int out_dt) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const bool splits = x_dt == DT_F32 && w_dt == DT_BF16 && out_dt == DT_F32;
    return splits || chunks_per_workgroup(M, N, K) > 0 ? lc_gemm_generic_workspace(M, N, K) : 0;
}

// The chunks' float32 sums of a product of float32 x and bfloat16 w that is shared out, for a norm kernel that sums them itself: their
// number (0: the product is not shared out, or its sum is better left to the kernel for it), and part [that number][M][N]
// whose sum in this order, from 0, is what lc_gemm_generic gives.  The norm has a workgroup a row, which asks for eight
// chunks at once where a row is up to 2,048 entries and for four beyond: with fewer rows than CUs, wide rows of many
// chunks are better summed by all CUs first.  Product, sum and norm, us, sum kernel and so: 566 rows, N 1,024, K 2,048
// 26.6 and 24.2, K 3,072 33.4 and 30.1; 2,048 x 6,144 103 and 98; 2,560 x 9,728 194 and 185; one row, 1,024 x 3,072 10.9
// and 10.0, 2,048 x 6,144 (49,152 chunk sums) 17.3 and 16.3; not so: one row of 4,096 x 4,096 17.4 and 19.6, 2,560 x 9,728 22.5 and 30.1.
LC_API int lc_gemm_generic_parts(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const int chunks = (K + GB_CHUNK - 1) / GB_CHUNK;
    if (N % 8 != 0 || N < 512 || N > 8192) return 0;               // rows that the norm takes in 16-byte pieces
    if (M < device_cus() && (N > 2048 || (long long)chunks * N > 49152)) return 0;
    return chunks_per_workgroup(M, N, K) > 0 ? chunks : 0;
}

LC_API int lc_gemm_generic_in_parts(const float* x, const void* w, float* part, int M, int N, int K, hipStream_t stream) {
    LC_CHECK(lc_gemm_generic_parts(M, N, K) > 0, "gemm: the product M=%d N=%d K=%d is not shared out", M, N, K);
    LC_CHECK(x && w && part, "gemm: null pointer");
    LC_CHECK((size_t)((M + GB_M - 1) / GB_M) <= 65535, "gemm: M=%d is too large", M);
    return launch_generic<float, bf16, float>(x, w, nullptr, M, N, K, part, stream);
}

LC_API int lc_gemm_generic(const void* x, int x_dt, const void* w, int w_dt, void* out, int out_dt,
                           int M, int N, int K, float* workspace, hipStream_t stream) {
    LC_CHECK(M >= 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
    if (M == 0) return 0;
    LC_CHECK(x && w && out, "gemm: null pointer");
    LC_CHECK((size_t)((M + GB_M - 1) / GB_M) <= 65535, "gemm: M=%d is too large", M);
    const int key = x_dt * 4 + w_dt * 2 + out_dt;
    switch (key) {
        case 0: return launch_generic<float, float, float>(x, w, out, M, N, K, workspace, stream);
        case 2: return launch_generic<float, bf16, float>(x, w, out, M, N, K, workspace, stream);
        case 4: return launch_generic<bf16, float, float>(x, w, out, M, N, K, workspace, stream);
        case 5: return launch_generic<bf16, float, bf16>(x, w, out, M, N, K, workspace, stream);
        case 6: return launch_generic<bf16, bf16, float>(x, w, out, M, N, K, workspace, stream);
        case 7: return launch_generic<bf16, bf16, bf16>(x, w, out, M, N, K, workspace, stream);
        default:
            LC_CHECK(false, "gemm: unsupported dtypes x=%d w=%d out=%d", x_dt, w_dt, out_dt);
    }
    return 0;
}
