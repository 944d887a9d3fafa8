// Latent attention of lone tokens (decoding) for rows of 512 + 64 entries: bound by reading a request's rows once.
//
// The kernel for portions (latent_bf16.hip) brings a stage of rows through registers into LDS twice, as they are and transposed,
// between two barriers, and of a lone token's eight waves only the pair that has its heads works: 1.96 TB/s.  Here every wave
// is by itself (64 requests of 2,048 tokens, 16 heads: 72 us -> 37, 4.1 TB/s; 8 requests 16.7 -> 15.4): it takes every fourth stage of 16 rows of its workgroup's share, straight from memory into two places of LDS of its
// own (one stage is on its way while one is worked through: 74 KB a CU), and keeps its own maximum, sum and row sums for 16
// heads; there is no barrier before the end, where the four waves' sums meet in LDS.  What the second product needs of the rows,
// neighbouring rows' entries of one column, comes out of the same places by the transposing LDS read (ds_read_b64_tr_b16: of 16
// lanes, lane s reads four columns 4 (s % 4) .. of row s / 4 and lane l gets column l of the four rows).
// In LDS a stage lies by chunks of 16 bytes, [chunk][row]: both reads then take whole neighbouring stretches.
#include "common.h"

namespace lc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(1))) const void* glb_ptr_t;

constexpr int LL_R = 512, LL_ROW = 576;             // entries of a row, the first 512 of which are summed
constexpr int LL_KEYS = 16, LL_WAVES = 4;
constexpr int LL_STAGE = LL_KEYS * LL_ROW * 2;      // bytes
constexpr int LL_LOADS = LL_STAGE / 1024;
constexpr int LL_KS = LL_ROW / 32, LL_NR = LL_R / 16;
constexpr int LL_AHEAD = 32;                        // stages whose rows' places a wave looks up at a time

// Operands of LDS with the wait for them in the same piece of assembly: the compiler would make an LDS read of its own wait
// for every load to LDS in flight.
template <int FIRST>
__device__ __forceinline__ void read_rows(bf16x8 (&r)[9], unsigned at) {       // steps FIRST .. + 8 of 32 entries
    asm volatile("ds_read_b128 %0, %9 offset:%10\n\tds_read_b128 %1, %9 offset:%11\n\tds_read_b128 %2, %9 offset:%12\n\t"
                 "ds_read_b128 %3, %9 offset:%13\n\tds_read_b128 %4, %9 offset:%14\n\tds_read_b128 %5, %9 offset:%15\n\t"
                 "ds_read_b128 %6, %9 offset:%16\n\tds_read_b128 %7, %9 offset:%17\n\tds_read_b128 %8, %9 offset:%18\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7]), "=&v"(r[8])
                 : "v"(at), "n"(FIRST * 1024), "n"(FIRST * 1024 + 1024), "n"(FIRST * 1024 + 2048), "n"(FIRST * 1024 + 3072),
                   "n"(FIRST * 1024 + 4096), "n"(FIRST * 1024 + 5120), "n"(FIRST * 1024 + 6144), "n"(FIRST * 1024 + 7168),
                   "n"(FIRST * 1024 + 8192)
                 : "memory");
}
template <int FIRST>
__device__ __forceinline__ void read_columns(short4v (&r)[8], unsigned at) {   // tiles FIRST .. + 7 of 16 columns
    asm volatile("ds_read_b64_tr_b16 %0, %8 offset:%9\n\tds_read_b64_tr_b16 %1, %8 offset:%10\n\tds_read_b64_tr_b16 %2, %8 offset:%11\n\t"
                 "ds_read_b64_tr_b16 %3, %8 offset:%12\n\tds_read_b64_tr_b16 %4, %8 offset:%13\n\tds_read_b64_tr_b16 %5, %8 offset:%14\n\t"
                 "ds_read_b64_tr_b16 %6, %8 offset:%15\n\tds_read_b64_tr_b16 %7, %8 offset:%16\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
                 : "v"(at), "n"(FIRST * 512), "n"(FIRST * 512 + 512), "n"(FIRST * 512 + 1024), "n"(FIRST * 512 + 1536),
                   "n"(FIRST * 512 + 2048), "n"(FIRST * 512 + 2560), "n"(FIRST * 512 + 3072), "n"(FIRST * 512 + 3584)
                 : "memory");
}

// grid (tiles, groups of 16 heads, splits).  A tile [token row, 1, request, position].
__global__ __launch_bounds__(64 * LL_WAVES, 1) void latent_lone_kernel(
    const bf16* __restrict__ qa, int H, const bf16* __restrict__ cache, const int* __restrict__ tiles,
    const int* __restrict__ block_table, int max_blocks, int page_size, float scale_log2, int window,
    const float* __restrict__ sink, bf16* __restrict__ out, int splits, float* __restrict__ part_o, float* __restrict__ part_ml) {
    // the waves' places; at the end, over them, the waves' sums [wave][16 heads][512] of a group of heads at a time
    __shared__ __attribute__((aligned(1024))) char lds[LL_WAVES * 2 * LL_STAGE];
    __shared__ int places[LL_WAVES][LL_AHEAD * LL_KEYS];
    __shared__ float tops[LL_WAVES][16], sums[LL_WAVES][16];
    static_assert(LL_WAVES * 16 * LL_R * 4 <= LL_WAVES * 2 * LL_STAGE, "the sums fit the places");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 15, g = lane >> 4;
    const int* tile = tiles + 4 * blockIdx.x;
    const int token = tile[0], req = tile[2], p = tile[3], h0 = blockIdx.y * 16;
    const int lo = window > 0 && p - window + 1 > 0 ? p - window + 1 : 0;
    const int stages = (p - lo) / LL_KEYS + 1, per = (stages + splits - 1) / splits;
    const int begin = blockIdx.z * per, end = min(stages, begin + per);
    const int mine = end > begin + wave ? (end - begin - wave + LL_WAVES - 1) / LL_WAVES : 0;       // this wave's stages: begin + wave, + 4 ...
    const int* table = block_table + (size_t)req * max_blocks;

    bf16x8 q[LL_KS];
    {
        const bf16* row = qa + ((size_t)token * H + min(h0 + col, H - 1)) * LL_ROW + 8 * g;
#pragma unroll
        for (int k = 0; k < LL_KS; ++k) q[k] = *reinterpret_cast<const bf16x8*>(row + 32 * k);
    }
    char* home = lds + wave * 2 * LL_STAGE;
    const unsigned home_at = (unsigned)(uintptr_t)(lds_ptr_t)home, place_at = (unsigned)(uintptr_t)(lds_ptr_t)&places[wave][0];
    // load instruction i brings chunks 4 i .. 4 i + 3 of the 16 rows: lane l chunk 4 i + l / 16 of row l % 16
    auto issue = [&](int n) {
        int place;
        asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(place) : "v"(place_at + ((n % LL_AHEAD) * LL_KEYS + col) * 4) : "memory");
        const bf16* from = cache + (size_t)place * LL_ROW + g * 8;
        char* to = home + (n & 1) * LL_STAGE;
#pragma unroll
        for (int i = 0; i < LL_LOADS; ++i)
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(from + 32 * i), (lds_ptr_t)(to + i * 1024), 16, 0, 0);
    };
    // where the rows of this wave's next stages lie; a row behind the token's own is that one once more, which counts for nothing
    auto look_up = [&](int n) {
        for (int i = lane; i < LL_AHEAD * LL_KEYS; i += 64) {
            const int stage = begin + wave + (n + i / LL_KEYS) * LL_WAVES;
            const int j = min(lo + stage * LL_KEYS + i % LL_KEYS, p);
            places[wave][i] = table[j / page_size] * page_size + j % page_size;
        }
    };
    const unsigned rows_at = (g * 16 + col) * 16;                       // [chunk 4 k + g][row col]
    const unsigned columns_at = (((col & 3) >> 1) * 16 + 4 * g + (col >> 2)) * 16 + (col & 1) * 8;     // columns 4 (col % 4) .. of row 4 g + col / 4
    floatx4 o[LL_NR];
    float m_ref = -INFINITY, l = 0.f;
#pragma unroll
    for (int d = 0; d < LL_NR; ++d) o[d] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int first = 0; first < mine; first += LL_AHEAD) {
        const int last = min(mine, first + LL_AHEAD);
        look_up(first);
        issue(first);
        for (int n = first; n < last; ++n) {
            if (n + 1 < last) {
                issue(n + 1);                                           // over the stage before, whose reads were waited for
                wait_vmcnt<LL_LOADS>();
            } else {
                wait_vmcnt<0>();
            }
            asm volatile("" ::: "memory");
            const unsigned at = home_at + (n & 1) * LL_STAGE;
            floatx4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
            bf16x8 k[9];
            read_rows<0>(k, at + rows_at);
#pragma unroll
            for (int i = 0; i < 9; ++i) s[i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[i], q[i], s[i & 1], 0, 0, 0);
            read_rows<9>(k, at + rows_at);
#pragma unroll
            for (int i = 0; i < 9; ++i) s[i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[i], q[9 + i], s[i & 1], 0, 0, 0);
            // the lane holds keys 4 g + r of its head; in units of log 2, against a reference point that moves when a score
            // outgrows it by 2^8
            const int j0 = lo + (begin + wave + n * LL_WAVES) * LL_KEYS + 4 * g;
            float mx = -INFINITY;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[0][r] = j0 + r <= p ? (s[0][r] + s[1][r]) * scale_log2 : -INFINITY;
                mx = fmaxf(mx, s[0][r]);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
            mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
            if (__builtin_amdgcn_ballot_w64(mx > m_ref + 8.f) != 0) {
                const float m_new = mx > m_ref + 8.f ? mx : m_ref;
                const float keep = m_ref == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_ref - m_new);
                l *= keep;
#pragma unroll
                for (int d = 0; d < LL_NR; ++d) o[d] *= keep;
                m_ref = m_new;
            }
            const float ref = m_ref == -INFINITY ? 0.f : m_ref;
            bf16x4 weight;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float e = __builtin_amdgcn_exp2f(s[0][r] - ref);
                l += e;
                weight[r] = static_cast<bf16>(e);
            }
            const short4v w = __builtin_bit_cast(short4v, weight);
            auto columns = [&](auto first_tile) {
                constexpr int F = decltype(first_tile)::value;
                short4v c[8];
                read_columns<F>(c, at + columns_at);
#pragma unroll
                for (int d = 0; d < 8; ++d) o[F + d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(c[d], w, o[F + d], 0, 0, 0);
            };
            columns(std::integral_constant<int, 0>{});
            columns(std::integral_constant<int, 8>{});
            columns(std::integral_constant<int, 16>{});
            columns(std::integral_constant<int, 24>{});
        }
    }
    // the four waves' sums: o[d] holds entries 16 d + 4 g + r of head col
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
    if (g == 0) {
        tops[wave][col] = m_ref;
        sums[wave][col] = l;
    }
    float* gathered = reinterpret_cast<float*>(lds);
    __syncthreads();                                                    // every wave is done with its places
    // head by head, 16-byte pieces at places xor the head, so that 16 heads' pieces meet no bank twice
#pragma unroll
    for (int d = 0; d < LL_NR; ++d)
        *reinterpret_cast<floatx4*>(gathered + (wave * 16 + col) * LL_R + (((4 * d + g) ^ col) * 4)) = o[d];
    __syncthreads();
    for (int i = threadIdx.x; i < 16 * (LL_R / 4); i += 64 * LL_WAVES) {
        const int head = i / (LL_R / 4), piece = i % (LL_R / 4), h = h0 + head;
        if (h >= H) break;                                              // the heads come in order
        float top = -INFINITY;
#pragma unroll
        for (int v = 0; v < LL_WAVES; ++v) top = fmaxf(top, tops[v][head]);
        floatx4 sum = {0.f, 0.f, 0.f, 0.f};
        float total = 0.f;
#pragma unroll
        for (int v = 0; v < LL_WAVES; ++v) {
            const float m = tops[v][head];
            const float weight = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - top);
            total = fmaf(sums[v][head], weight, total);
            sum += *reinterpret_cast<const floatx4*>(gathered + (v * 16 + head) * LL_R + ((piece ^ head) * 4)) * weight;
        }
        if (splits == 1) {
            float inv = 1.f / total;
            if (sink) {     // one more term in the denominator, a key with that score and no row
                const float s2 = sink[h] * 1.4426950408889634f, all = fmaxf(top, s2), keep = __builtin_amdgcn_exp2f(top - all);
                inv = keep / fmaf(total, keep, __builtin_amdgcn_exp2f(s2 - all));
            }
            bf16x4 y;
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = static_cast<bf16>(sum[r] * inv);
            *reinterpret_cast<bf16x4*>(out + ((size_t)token * H + h) * LL_R + 4 * piece) = y;
        } else {
            const size_t share = ((size_t)blockIdx.x * H + h) * splits + blockIdx.z;
            *reinterpret_cast<floatx4*>(part_o + share * LL_R + 4 * piece) = sum;
            if (piece == 0) {
                part_ml[share * 2] = top;
                part_ml[share * 2 + 1] = total;
            }
        }
    }
}

bool latent_lone_takes(int R, int rot) { return R == LL_R && R + rot == LL_ROW; }

int launch_latent_lone(const void* qa, int H, const void* cache, const int* tiles, int num_tiles, const int* block_table, int max_blocks,
                       int page_size, float scale, int window, const float* sink, void* out, int splits, float* part_o, float* part_ml,
                       hipStream_t stream) {
    const float scale_log2 = scale * 1.4426950408889634f;
    latent_lone_kernel<<<dim3(num_tiles, (H + 15) / 16, splits), 64 * LL_WAVES, 0, stream>>>(
        (const bf16*)qa, H, (const bf16*)cache, tiles, block_table, max_blocks, page_size, scale_log2, window, sink, (bf16*)out, splits,
        part_o, part_ml);
    LC_LAUNCH_CHECK("latent_lone");
    return 0;
}

}  // namespace lc
