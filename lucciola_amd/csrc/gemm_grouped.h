// What the grouped products' kernels share (gemm_grouped.hip, gemm_grouped_tiled.hip).
#pragma once

#include "common.h"

namespace lc {

struct GroupedArgs {
    const void* x; long long ldx, x_group;
    const void* w;
    void* out; long long ldo, out_group;
    int M, N, K, G;
    const int* gather; const int* row_start; const int* tile_start;
    int epilogue;
    const void* gate; long long ldg, gate_group;
    bool pairs;             // two neighbouring columns of out, the first an even one, may be stored together
};

// A workgroup's group and its rows: first .. end - 1, end being the group's.
struct GroupedTile {
    int group, first, end;
};

// The tile of BM rows that the workgroup (blockIdx.y, blockIdx.z) takes; false: there is none.
__device__ __forceinline__ bool find_tile(const GroupedArgs& a, int BM, GroupedTile& t) {
    if (!a.row_start) {
        t = {(int)blockIdx.z, (int)blockIdx.y * BM, a.M};
        return true;
    }
    const int tile = blockIdx.y;
    if (tile >= a.tile_start[a.G]) return false;
    int lo = 0, hi = a.G - 1;                   // the last group whose first tile is not after this one
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a.tile_start[mid] <= tile) lo = mid;
        else hi = mid - 1;
    }
    t = {lo, a.row_start[lo] + (tile - a.tile_start[lo]) * BM, a.row_start[lo + 1]};
    return true;
}

// What a gated expert makes of its first product's sums (gate rows of w, then as many up rows): act(gate) * up, both first times the
// weight of the row's (token, choice) where weights are given.
struct GroupedGate {
    const float* weights; const int* entry_row;     // [tokens * top]: the choice's weight, the choice's sorted row; null: no weights
    int top;
    int kind;                                       // 0: silu, 1: gelu (tanh form)
};

// Whether gemm_grouped_tiled.hip has a kernel for these bfloat16 operands (whole, aligned 16-byte pieces) and lists, and whether it is
// the faster one.
bool grouped_tiled_takes(const GroupedArgs& a, int tile_rows);
bool grouped_tiled_pays(const GroupedArgs& a, int max_tiles, int tile_rows);
// forced: tests ask for the kernel of even tiles wherever it can run
int launch_grouped_tiled(const GroupedArgs& a, int max_tiles, int tile_rows, bool out_bf16, bool forced, hipStream_t stream);

// whether the gated product is for these sizes (forced: wherever it can run); whether an experts' product goes to the kernel of even tiles
bool grouped_gates(const GroupedArgs& a, int tile_rows, bool forced);
bool grouped_evens(const GroupedArgs& a, int max_tiles, int tile_rows);
int launch_grouped_gated(const GroupedArgs& a, const GroupedGate& gate, hipStream_t stream);

}  // namespace lc
