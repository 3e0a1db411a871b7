// How a pass's prompt rows are cut for attention_prompt.hip: host arithmetic only (not exported).
#pragma once
#include <stdint.h>

namespace llmk {

// A prompt tile: `count` (1 .. kTileRows) consecutive rows of a pass, at consecutive positions of
// one sequence, whose block-table rows agree on every page that the last of them reads.
constexpr int kTileRows = 32;
struct PromptTile {
  int32_t row0, count;
};

// Splits of a launch: up to one block per CU, of at least two chunks of 64 positions: a few rows far
// into a sequence would otherwise run on n_kv_heads CUs, chunk after chunk. Split s of a row is
// pages [s, s + 1) * pages_per_split.
constexpr int kTargetBlocks = 256, kMinSplitPages = 8;
struct PromptSplits {
  int num_splits, pages_per_split;
};

// The splits for n_tiles tiles whose longest attention spans `span` pages. The launch shape is also
// a graph's (llmk_engine_forward_graph), so that spans share it: lengths go up in steps of an
// eighth to a quarter, the number of splits follows the tiles alone, and a single split has one
// length past kMinSplitPages. A prompt of 131072 positions in chunks of any one row count meets at
// most 38 shapes, where exact lengths make hundreds. Splits past a row's end leave at once.
inline PromptSplits prompt_splits(int n_tiles, int n_kv_heads, int span, int max_splits) {
  const long long blocks = (long long)n_tiles * n_kv_heads;
  long long want = blocks > 0 ? kTargetBlocks / blocks : 1;
  if (want > max_splits) want = max_splits;
  if (span <= kMinSplitPages) return {1, kMinSplitPages};
  if (want <= 1) return {1, 1 << 26};
  int pages = (int)((span + want - 1) / want), step = kMinSplitPages;
  while (pages > 8 * step) step *= 2;
  pages = (pages + step - 1) / step * step;
  return {(int)want, pages};
}

}  // namespace llmk
