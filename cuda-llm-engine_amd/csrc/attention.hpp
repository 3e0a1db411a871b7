// Attention entry points shared between the attention sources and the engine (not exported).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "prompt_plan.hpp"

namespace llmk {

struct PromptAttention {
  const uint16_t *q, *k_pool, *v_pool;  // as llmk_attention_decode_fast
  const int32_t *tables, *positions;    // [rows, max_pages], [rows]
  const int32_t* lens;                  // [rows]: position + 1 in rows of a tile, 0 elsewhere
  const PromptTile* tiles;              // [n_tiles], device memory
  uint16_t* out;
  float* workspace;  // llmk_attention_decode_fast's, for num_splits splits (unused with 1)
  int n_rows, n_tiles, max_pages, n_heads, n_kv_heads;
  PromptSplits splits;
};

// Attention of the rows in `tiles` over all of their cached positions (their own included); rows
// in no tile are left alone.
int prompt_attention(const PromptAttention& a, hipStream_t stream);

// Merges the pieces of a sequence-split launch (attention.hip): rows of lens[] cut into
// ceil(pages / pages_per_split) pieces, those with more than one.
int merge_split_pieces(const float* workspace, const int32_t* lens, uint16_t* out, int n_rows,
                       int max_pages, int n_heads, int num_splits, int pages_per_split,
                       hipStream_t stream);

}  // namespace llmk
