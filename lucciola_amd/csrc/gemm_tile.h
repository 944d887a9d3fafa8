// The inner loop of the tiled bfloat16 products, for kernels that find their rows each in its own way: the dense products
// (gemm_bf16.hip) and the experts' over sorted rows (gemm_grouped_tiled.hip).
#pragma once

#include "common.h"

#include <type_traits>

namespace lc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(1))) const void* glb_ptr_t;

template <typename TO> __device__ __forceinline__ void store_out(TO* p, float v);
template <> __device__ __forceinline__ void store_out<float>(float* p, float v) { *p = v; }
template <> __device__ __forceinline__ void store_out<bf16>(bf16* p, float v) { *p = static_cast<bf16>(v); }

// two adjacent elements in one store; p is aligned to the pair
template <typename TO> __device__ __forceinline__ void store_pair(TO* p, float a, float b);
template <> __device__ __forceinline__ void store_pair<float>(float* p, float a, float b) {
    *reinterpret_cast<float2*>(p) = make_float2(a, b);
}
template <> __device__ __forceinline__ void store_pair<bf16>(bf16* p, float a, float b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    bf16x2 v;
    v[0] = static_cast<bf16>(a);
    v[1] = static_cast<bf16>(b);
    *reinterpret_cast<bf16x2*>(p) = v;
}

// 16 bytes of adjacent elements in one store; p is aligned to 16 bytes
template <typename TO> constexpr int PIECE = 16 / sizeof(TO);
template <typename TO> __device__ __forceinline__ void store_piece(TO* p, const float (&v)[PIECE<TO>]) {
    if constexpr (sizeof(TO) == 2) {
        bf16x8 packed;
#pragma unroll
        for (int e = 0; e < 8; ++e) packed[e] = static_cast<bf16>(v[e]);
        *reinterpret_cast<bf16x8*>(p) = packed;
    } else {
        *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    }
}

// the value of another lane of the same row of 16 lanes, by a DPP move: CTRL 0xB1 swaps
// neighbours (lane ^ 1), 0x128 rotates the row by 8 (lane ^ 8).  All lanes must be active.
template <int CTRL> __device__ __forceinline__ float lane_swap(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// What the gated epilogue makes of a gate and an up entry: with g' = min(g, limit) and u' = u held inside
// -limit .. limit, g' sigmoid(slope g') (u' + shift).  No limit, slope 1 and shift 0 is silu(g) u (reference:
// src/kernels/swiglu.cu:8,31-35), to the bit.
struct GateForm {
    float limit, slope, shift;
};
static constexpr GateForm kSilu{INFINITY, 1.f, 0.f};

// exp and the reciprocal are the hardware's single instructions (about one unit in the last
// place each); the results of these products are rounded to bfloat16 afterwards.
__device__ __forceinline__ float gated_f(float g, float u, GateForm form) {
    g = fminf(g, form.limit);
    u = fminf(fmaxf(u, -form.limit), form.limit);
    return g * __builtin_amdgcn_rcpf(1.f + __expf(-form.slope * g)) * (u + form.shift);
}

// Workgroup tile BM x BN x 64, four waves in a 2 x 2 grid, each owning (BM/64) x (BN/64) tiles
// of 32 x 32.
//
// Operand tiles go from global memory straight into LDS (global_load_lds_dwordx4: lane l's 16
// bytes land at the instruction's LDS base + 16 l, no registers in between) into a ring of
// TL_STAGES stages.  Inside a stage a row's eight 16-byte chunks are stored at column
// (chunk ^ ((row >> 1) & 7)): the 16 lanes that the LDS serves per cycle for a 128-bit read
// (16 consecutive rows, one chunk) then cover all 64 banks.
//
// The loop is scheduled by hand, because a SIMD holds a single wave of this kernel and nothing
// else hides a stall.  Per k-step, which is one product deep (16 or 32 k), the wave issues its
// TM * TN products; between them, one at a time, go the LDS reads of the NEXT k-step's operands (ds_read_b128 in inline
// assembly with explicit waits: the compiler cannot tell the stages apart and would make every
// load in flight land before any read) and the global loads.  In a block's last k-step the wave
// waits for its own loads of the next block and meets the others at a bare barrier, the only one
// of a block: behind it all waves' loads of the next block are visible, and all waves hold the
// last operands of this block in registers, so that its stage is free.  From there on the wave
// reads the next block's first operands and issues, a few products apart, the loads of the block
// TL_STAGES ahead into the freed stage, on into the next block.  sched_barrier pins that order.
// (Figures below that name no product's size are of the loop with products of 32 x 32 x 16.)
//
// The loads are spread because a CU takes them at 64 bytes a clock (58 measured for rows of 128
// bytes that L2 holds): the 16 loads of a wave of the 256 x 256 tile, four waves at once, are a
// thousand clocks in which a wave that issues them in a row issues no product.  In a row, behind
// the barrier or in the first k-step (us; the same sums): 2,048 x 24576 x 4096 with SwiGLU 367,
// 2,048 x 4096 x 12288 193, 2,048 x 2048 x 2048 26.3; spread over the first half: 328, 171 and 22.9 (the matrix cores
// busy 69 % of the clocks instead of 56, at a clock that the power limit takes from 1.84 to
// 1.64 GHz; 2.4 without load).
constexpr int TL_K = 64;

// BM x BN rows of x and of w, TL_STAGES stages, WM x WN waves, each owning (BM / WM) x (BN / WN) of the tile as TM x TN products
// of MF x MF and KP deep.  LATE: of two stages whose loads go out later in a block (below).  FINE: products of 16 x 16 x 32 instead of
// 32 x 32 x 16, the same sums to the bit wherever tried.  Both take the matrix cores' time for as many operations, but the small ones read and
// write each sum half as often, and a product of large tiles is held back by the power limit: at 2,048 rows, held for three seconds, us and the
// clock meanwhile, large (stored in pairs) and small (in whole lines, gemm_bf16.hip): 24576 x 4096 with SwiGLU 325.5 at 1.78 GHz and 315 at 2.00, 6144 x
// 4096 82.4 at 1.82 and 80.3 at 2.08, 4096 x 12288 173 at 1.755 and 169.5 at 1.95, 4096 x 4096 60.4 at 1.86 and 59 at 2.07.  (The first twenty
// after a rest take up to a quarter longer, either way.)  23 products of 233 to 3,868 rows that take
// such tiles: 0.97 of the time in the mean, 0.87 to 1.01.
// Not for tiles whose waves own less than 64 x 128 (bound by the way from L2: no change), nor for the experts' (up to 1.07 of the time: bound by memory).
template <int BM, int BN, int TL_STAGES, int WM, int WN, bool LATE = false, bool FINE = false>
struct TileLoop {
    static constexpr int MF = FINE ? 16 : 32;                 // rows and columns of a product
    typedef typename std::conditional<FINE, floatx4, floatx16>::type Sum;
    static constexpr int SV = MF * MF / 64;                   // sums of a product a lane
    static constexpr int S = TL_STAGES;
    static constexpr int NW = WM * WN;
    static constexpr int TM = BM / (MF * WM), TN = BN / (MF * WN);
    static constexpr int KP = FINE ? 32 : 16;                 // k of a product
    static constexpr int KS = TL_K / KP;                      // k-steps per block
    static constexpr int LPA = BM * 8 / (64 * NW), LPB = BN * 8 / (64 * NW), LP = LPA + LPB;   // load instructions per thread and stage
    static_assert(BM % (MF * WM) == 0 && BN % (MF * WN) == 0, "whole products per wave");
    static_assert((BM * 8) % (64 * NW) == 0 && (BN * 8) % (64 * NW) == 0, "whole load instructions per wave");
    static constexpr int NM = TM * TN, NR = TM + TN;          // products and operand reads per k-step
    static constexpr int A_STAGE = BM * TL_K * 2, B_STAGE = BN * TL_K * 2;   // bytes
    static constexpr int LDS = S * (A_STAGE + B_STAGE);       // A stages, then B stages, aligned to 1,024
    static_assert(S >= 2, "a stage is loaded while another is read");
    static_assert(LDS <= 160 * 1024, "LDS");

    __device__ static __forceinline__ int swz(int row) { return (row >> 1) & 7; }
    // load instruction i of a wave brings, of the stage's rows of x or of w, row row_of(i) and of its chunks of 8 entries
    // chunk chunk_of(i): chunk p = (i * NW + wave) * 64 + lane of a stage holds row p / 8, global chunk (p % 8) ^ swz(row)
    __device__ static __forceinline__ int row_of(int i, int wave, int lane) { return ((i * NW + wave) * 64 + lane) >> 3; }
    __device__ static __forceinline__ int chunk_of(int i, int wave, int lane) { return (lane & 7) ^ swz(row_of(i, wave, lane)); }

    // xg, wg: where load instruction i of this lane reads block 0; nk blocks, the first of them block `skew` (wrapping around)
    __device__ static __forceinline__ void run(char* lds, const bf16* const (&xg)[LPA], const bf16* const (&wg)[LPB], int nk,
                                               int skew, int wave, int lane, Sum (&acc)[TM][TN]) {
    const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);
    const int lr = lane & (MF - 1), kg = lane / MF;
    // load instruction idx (x first, then w) of block kb into a stage
    auto issue_one = [&](int idx, int kb, int stage) {
        kb += skew;
        kb -= kb >= nk ? nk : 0;
        if (idx < LPA)
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(xg[idx] + kb * TL_K),
                (lds_ptr_t)(lds + stage * A_STAGE + (idx * NW + wave) * 1024), 16, 0, 0);
        else
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(wg[idx - LPA] + kb * TL_K),
                (lds_ptr_t)(lds + S * A_STAGE + stage * B_STAGE + ((idx - LPA) * NW + wave) * 1024), 16, 0, 0);
    };
    // Where the loads of a block sit among the products: position 0 is the first product behind the barrier that frees their
    // stage.  With more than two stages they are spread over the whole block but its end (from a third to the whole of it: within
    // 2 %).  With two they have to be back at the next barrier and are issued in its first quarter: in a row, over the first half,
    // over the first quarter, over an eighth (geometric means of four shapes of tile, 212 products of 96 to 4,001 rows on cold data):
    // 1, 1.007, 0.973, 0.989; 192 x 256 of up to 333 rows 1, 1.08, 1.04, 1.04.  Few rows wait for w and want its loads early; many are
    // bound by the matrix cores and want them late (us, in a row, half, quarter: 4,001 x 4096 x 4096 121, 110, 115; 1,024 x 4096 x
    // 4096 49, 43, 45; 2,048 x 4096 x 12288 198, 173, 171; 576 x 19456 x 2560 61, 67, 65).  So the dense tiles of 256 rows, which
    // are taken for many, are LATE: over 50 products of 700 to 4,001 rows for which they are among the best, 256 x 256 0.98 of the
    // time of a quarter (0.94 to 0.99), 256 x 192 0.99 (0.985 to 1.02).  FINE (us, the whole of those two shapes and 256 x 128; 24576 x 4096, 6144 x
    // 4096, 1,523 x 24576 x 4096): barrier after a quarter, loads over 6/16, reads over half of the products 318, 82.9, 252; an eighth and 6/16
    // 308, 82.6, 248; 3/16 and 5/16 313, 81.6, 247; a sixteenth and 5/16 307, 80.9, 248; an eighth, 5/16 and reads over three quarters 310,
    // 81.5, 249; over a quarter 314, 83.6, 252; loads over 12/16 352, 99.6 and 103 for the 94 of 2,039 x 10240 x 2048.
    constexpr int BAR = FINE ? NM / 8 : NM / 4;                // the product after which a block's last k-step syncs
    constexpr int WIN = KS * NM;                               // products between two barriers
    constexpr int NA = NM - 1 - BAR;                           // of them in the block that frees the stage
    constexpr int SPAN = S == 2 ? (LATE ? (FINE ? WIN * 5 / 16 : WIN / 2) : WIN / 4) : WIN * 7 / 8;
    static_assert(SPAN >= 1 && SPAN < WIN, "all loads of a block are issued before the next barrier");
    struct At { static constexpr int of(int l) { return l * SPAN / LP; } };      // load l's position
    // Tiles of two stages with few products a block are several to a CU and bound by how much is on its way, and issue a whole
    // block's loads behind a barrier of their own before they wait for the block before it (8,192 rows over 32 matrices of
    // 2,048 x 2,048 in tiles of 128 x 128: 127 us, 141 spread).
    constexpr bool EARLY = S == 2 && NM * MF * MF <= 4096;
    constexpr int PA = EARLY ? LP : [] { int n = 0; for (int l = 0; l < LP; ++l) n += l * SPAN / LP < NA; return n; }();   // loads in that block
    static_assert((S - 1) * LP + PA <= 63, "the load counter holds 63");
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s < nk) {
#pragma unroll
            for (int i = 0; i < LP; ++i)
                if (s < S - 1 || i < PA) issue_one(i, s, s);
        }

#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < SV; ++v) acc[i][j][v] = 0.f;

    // LDS address of this lane's operand rows in stage 0, with the lane's part of the swizzle;
    // k-step ks flips chunk bits: ((KP / 8 * ks + kg) ^ swz) * 16 = ((kg ^ swz) * 16) ^ (ks * KP * 2)
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t)lds;
    unsigned pa[TM], pb[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int row = wm + i * MF + lr;
        pa[i] = lds0 + row * 128 + ((kg ^ swz(row)) * 16);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int row = wn + j * MF + lr;
        pb[j] = lds0 + S * A_STAGE + row * 128 + ((kg ^ swz(row)) * 16);
    }

    bf16x8 a[2][TM], b[2][TN];
    auto read_one = [&](int r, int stage, int ks, int buf) {
        if (r < TM) {
            const unsigned addr = (pa[r] ^ (ks * KP * 2)) + stage * A_STAGE;
            asm volatile("ds_read_b128 %0, %1" : "=v"(a[buf][r]) : "v"(addr));
        } else {
            const unsigned addr = (pb[r - TM] ^ (ks * KP * 2)) + stage * B_STAGE;
            asm volatile("ds_read_b128 %0, %1" : "=v"(b[buf][r - TM]) : "v"(addr));
        }
    };
    // the products that follow a wait must not be moved above it: tie their operands to that point
    auto tie = [&](int buf) {
#pragma unroll
        for (int i = 0; i < TM; ++i) asm volatile("" : "+v"(a[buf][i]));
#pragma unroll
        for (int j = 0; j < TN; ++j) asm volatile("" : "+v"(b[buf][j]));
    };
    // sums of small products stay in registers of their own, or the compiler moves them about all through the loop
    auto hold = [&](Sum& sum) {
        if constexpr (FINE) asm volatile("" : "+a"(sum));
    };
    auto hold_all = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) hold(acc[i][j]);
    };
    hold_all();
    auto product = [&](int k, int buf) {
        const int i = k / TN, j = k % TN;
        if constexpr (FINE) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[buf][i], b[buf][j], acc[i][j], 0, 0, 0);
            hold(acc[i][j]);
        } else {
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[buf][i], b[buf][j], acc[i][j], 0, 0, 0);
        }
    };

    // where the reads sit among the NM products of a k-step
    constexpr int QR = (2 * NR + NM - 1) / NM;                 // reads after each product, from the first on
    constexpr int QT = NM - BAR - 1 > 0 ? (NR + (NM - BAR - 1) - 1) / (NM - BAR - 1) : NR;
    struct Read {       // the product after which read r goes out, and so behind a block's barrier; FINE: spread over half of the products
        static constexpr int of(int r) { return FINE ? r * (NM / 2) / NR : r / QR; }
        static constexpr int behind(int r) { return FINE ? r * ((NM - BAR - 1) / 2) / NR : r / QT; }
    };

    if (nk >= S) wait_vmcnt<(S - 2) * LP + PA>(); else wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int r = 0; r < NR; ++r) read_one(r, 0, 0, 0);

    int stage = 0, pstage = S - 1;   // the stages of blocks `it` and `it - 1`
    // FREE: block it + S exists, its first loads go into this block's stage once it is free; REST: block it + S - 1 exists, its other
    // loads go where block it - 1 was
    auto block = [&](int it, auto free_tag, auto rest_tag) {
        constexpr bool FREE = decltype(free_tag)::value, REST = decltype(rest_tag)::value;
        const int nstage = stage + 1 == S ? 0 : stage + 1;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int cur = ks & 1, nxt = cur ^ 1;
            wait_lgkmcnt<0>();
            tie(cur);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < NM; ++k) {
                product(k, cur);
                __builtin_amdgcn_sched_barrier(0);
                if (ks < KS - 1) {
#pragma unroll
                    for (int r = 0; r < NR; ++r)
                        if (Read::of(r) == k) read_one(r, stage, ks + 1, nxt);
                }
                if (REST && (ks < KS - 1 || k <= BAR)) {
#pragma unroll
                    for (int l = PA; l < LP; ++l)
                        if (At::of(l) - NA == ks * NM + k) issue_one(l, it + S - 1, pstage);
                }
                if (ks == KS - 1) {
                    if (k == BAR && (REST || it + 1 < nk)) {
                        // block it + 1 has landed (this wave's part, then everybody's), and nobody reads this stage any more
                        if (EARLY && FREE) {
                            __builtin_amdgcn_s_barrier();
#pragma unroll
                            for (int l = 0; l < LP; ++l) issue_one(l, it + S, stage);
                            wait_vmcnt<LP>();
                        } else if (REST) wait_vmcnt<(S - 2) * LP>();
                        else wait_vmcnt<0>();
                        __builtin_amdgcn_s_barrier();
                        if (NM - BAR - 1 == 0) {
#pragma unroll
                            for (int r = 0; r < NR; ++r) read_one(r, nstage, 0, nxt);
                        }
                    }
                    if (k > BAR && (REST || it + 1 < nk)) {
#pragma unroll
                        for (int r = 0; r < NR; ++r)
                            if (Read::behind(r) == k - BAR - 1) read_one(r, nstage, 0, nxt);
                    }
                    if (FREE && !EARLY && k > BAR) {
#pragma unroll
                        for (int l = 0; l < PA; ++l)
                            if (At::of(l) == k - BAR - 1) issue_one(l, it + S, stage);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        pstage = stage;
        stage = nstage;
    };
    int it = 0;
    for (; it + S < nk; ++it) block(it, std::true_type{}, std::true_type{});
    if (it + S - 1 < nk) { block(it, std::false_type{}, std::true_type{}); ++it; }
    for (; it < nk; ++it) block(it, std::false_type{}, std::false_type{});
    hold_all();

    }
};

}  // namespace lc
