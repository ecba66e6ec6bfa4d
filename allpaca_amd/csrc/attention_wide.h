// The prompt-portion attention kernel for tiles of 128 rows (attention_wide_bf16.hip), called from the launch code
// in attention_bf16.hip.
#pragma once
#include "common.h"

constexpr int ATTN_WIDE_ROWS = 128;  // rows of a tile

// True for the head sizes (128 and 64) and page sizes the kernel takes (pages of a power of two, 16 to 32,768 positions and less
// than 4 GiB).
bool attn_wide_takes(int Hk, int d, int page_tokens);
// The decoded rows of a step that go beside its tiles: their numbers (null: 0 .. n - 1), and the keys of every row in n_parts ranges,
// four a block, that the last block of a (row, kv head) adds (workspace: n * H * ceil(n_parts / 4) * (d + 2) floats; counters: one a
// (row, tile of 16 heads), zero before and after); workspace null: a block a pair.
struct AttnDecodeRows {
  const int* rows;
  int n, n_parts;
  float* workspace;
  int* counters;
};
// Arguments as apc_attention_prefill_bf16; tiles of up to ATTN_WIDE_ROWS rows.  n_splits > 1: the keys of every tile
// are cut into that many ranges, a block each, and a second kernel adds the ranges; `parts` then has room for
// n_splits * part_rows * H * (d + 2) floats, part_rows being at least the largest row index of a tile + 1.
int launch_attn_prefill_wide(const bf16_t* q, int ldq, int q_off, bf16_t* out, int ldo, int H, int Hk,
                             const bf16_t* cache, int page_tokens, const int* block_table, int max_blocks,
                             const int* positions, const int* row_seg, const int* tile_row0, const int* tile_rows,
                             int n_tiles, int window, float scale, int n_splits, int part_rows, float* parts,
                             int d, hipStream_t stream, const AttnDecodeRows* dec = nullptr);
