// The library's own tiled GEMM for 9 to kTilesMaxRows rows (gemm_tiles.hip): llmk_linear and the
// engine's fused projections (not exported).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace llmk {

constexpr int kTilesMaxRows = 512;

// How a product is cut: the tile shape (an index into gemm_tiles.hip's list) and the number of
// pieces of the in dimension, whose fp32 partial sums a second pass adds.
struct TilePlan {
  int tile, splits;
};

// Whether y[T, out] = x[T, in] W^T runs here: 9 .. kTilesMaxRows rows, in a multiple of 128, out
// of 4, x and w 16-byte and y 8-byte aligned, and where hipBLASLt does not win. `fused`: the
// product's consumer is part of the launch, or adds up its pieces itself.
bool tiles_apply(const void* x, const void* w, const void* y, int T, int in, int out, bool fused);

// The plan for a shape with at most `max_floats` floats of partial sums. `reduce_launch`: whether
// the partial sums cost a launch of their own.
TilePlan tiles_plan(int T, int in, int out, size_t max_floats, bool reduce_launch);

// y = x W^T; `partial` holds splits * T * out floats when the plan has more than one split.
int tiles_linear(const TilePlan& p, const uint16_t* x, const uint16_t* w, uint16_t* y,
                 float* partial, int T, int in, int out, hipStream_t stream);

// partial[splits, T, out] = the pieces of x W^T (one piece with one split), for a consumer that
// adds them (add_rmsnorm_partial).
int tiles_partial(const TilePlan& p, const uint16_t* x, const uint16_t* w, float* partial, int T,
                  int in, int out, hipStream_t stream);

// act[T, inter] = swiglu of the gate and up halves of fp16(x W^T), W [2 inter, in]; inter a
// multiple of 4. The values of llmk_swiglu_rows.
int tiles_swiglu(const uint16_t* x, const uint16_t* w_gate_up, uint16_t* act, int T, int in,
                 int inter, hipStream_t stream);

// Where the rows of a QKV projection go: q heads rotated to q_out [T, n_heads, 64], k heads rotated
// and v heads to row pool_rows[t] of the pools [rows, n_kv_heads, 64], 16-byte aligned. cos_sin [T,
// 32] (pairs of fp16) and pool_rows come from rope_rows.
struct RopeTarget {
  _Float16 *q_out, *k_pool, *v_pool;
  const uint32_t* cos_sin;
  const long long* pool_rows;
  int n_heads, n_kv_heads;
};
int rope_rows(const int32_t* positions, const int32_t* tables, const float* inv_freq,
              int max_pages, int n, void* cos_sin, long long* pool_rows, hipStream_t stream);
// The values of llmk_qkv_rope_scatter over fp16(x W^T), head_dim 64, page size 16.
int tiles_qkv_rope_scatter(const uint16_t* x, const uint16_t* w_qkv, const RopeTarget& to, int T,
                           int in, hipStream_t stream);

// residual += fp16(sum over splits of partial[s]), out = rmsnorm(residual) * w, row by row;
// hidden a multiple of 8 up to kPartialNormMaxHidden (norm.hip).
constexpr int kPartialNormMaxHidden = 8192;
int add_rmsnorm_partial(const float* partial, int splits, uint16_t* residual, const uint16_t* w,
                        uint16_t* out, int rows, int hidden, float eps, hipStream_t stream);

}  // namespace llmk
