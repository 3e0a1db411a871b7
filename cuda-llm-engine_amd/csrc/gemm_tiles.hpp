// The library's own tiled GEMM for 9 to kTilesMaxRows rows (gemm_tiles.hip): llmk_linear and the
// engine's fused projections (not exported).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace llmk {

constexpr int kTilesMaxRows = 256;

// How a product is cut: the tile shape (an index into gemm_tiles.hip's list) and the number of
// pieces of the in dimension, whose fp32 partial sums a second pass adds.
struct TilePlan {
  int tile, splits;
};

// Whether y[T, out] = x[T, in] W^T runs here: 9 .. kTilesMaxRows rows, in a multiple of 128, out
// of 4, x and w 16-byte and y 8-byte aligned, and not so wide that hipBLASLt wins.
bool tiles_apply(const void* x, const void* w, const void* y, int T, int in, int out);

// The plan for a shape with at most `max_floats` floats of partial sums. `reduce_launch`: whether
// the partial sums cost a launch of their own.
TilePlan tiles_plan(int T, int in, int out, size_t max_floats, bool reduce_launch);

// y = x W^T; `partial` holds splits * T * out floats when the plan has more than one split.
int tiles_linear(const TilePlan& p, const uint16_t* x, const uint16_t* w, uint16_t* y,
                 float* partial, int T, int in, int out, hipStream_t stream);

}  // namespace llmk
