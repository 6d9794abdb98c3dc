// The matmul on int8 matrix cores with exact results: what gemm.hip needs of gemm_split.hip.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"

namespace dllm_hip {

// Tiles that the split sums hand back to the FP64 matmul.
struct SplitRedo {
    const uint8_t* tile_flags = nullptr;  // [windows in parallel][row tiles][column tiles]: 1 = recompute in FP64
    const uint32_t* tiles = nullptr;      // how many are flagged
    int tile = 0;                         // the tile's side
};

// How a float-A call runs on the int8 path: not at all (rows 0), or in blocks of `rows` rows (a multiple of 128, or I),
// its windows in parallel (into seg_partial) or in sequence.
struct SplitPlan {
    int64_t rows = 0;
    bool parallel = false;
};
SplitPlan split_plan(const GemmCall& g);
// Splits the operands, computes every output that the split sums decide, and recomputes the undecided ones by their own
// chains; the tiles of redo->tile_flags are left to the caller. partial: per-window results instead of C.
int launch_split_gemm(const GemmCall& g, float* partial, hipStream_t stream, SplitRedo* redo);

// Forward matmuls of few outputs, each by its own chain from x and Bt.
bool chain_linear_fits(const GemmCall& g);
int launch_chain_linear(const GemmCall& g, hipStream_t stream);

}  // namespace dllm_hip
