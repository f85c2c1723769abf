// GEMMs that do not fill the chip with large tiles: what run_gemm (gemm.hip) hands to gemm_small.hip.
#pragma once
#include "common.h"
#include "gather.h"

namespace tdist {

struct SmallGemmParams {
  const unsigned char* A;
  ShardRows shards;           // rows != 0: A's rows lie in shards, at these offsets from A
  // grouped (sorted_ids != NULL): row r of block b (as many as the tile has) is row sorted_ids[b * rows + r] of the output and row sorted id / topk of A (an id from
  // num_valid on: none); its weights are block_expert[b]'s; post_pad[0] rows are in use
  const int32_t *sorted_ids, *block_expert, *post_pad;
  int64_t b_expert_stride_b;
  int num_blocks, num_valid, a_rows, topk;
  uint32_t topk_magic;
  const unsigned char* B;
  unsigned char* C;           // plain output (scatter_bufs == NULL)
  void* const* scatter_bufs;  // GEMM-RS: rows of owner o go to scatter_bufs[o] from row rank * m_per_rank on
  const float* row_scale;     // e4m3 inputs: fp32 scales or NULL
  const float* col_scale;
  int64_t lda_b, ldb_b;  // byte strides; M * lda_b (of rows in one piece) and N * ldb_b below 2^31
  int64_t ldc;           // elements
  int M, N;              // grouped: M is the rows of all blocks
  int k_bytes;  // a multiple of 16
  int m_per_rank, rank;
  int splits;         // workgroups that share a tile along K
  int tiles_per_split;  // K tiles of 128 bytes per workgroup
  int walk_rows;      // an XCD's run of tiles goes down this many row tiles before the next column (set by launch_gemm_small)
  float* partials;    // splits > 1: fp32 accumulators, a tile per workgroup
  int32_t* counters;  // splits > 1: one per tile, zero, left zero
  int l2_local;       // workgroup i has been seen to run on XCD i % 8: the pieces of a tile meet in that XCD's L2
};

enum SmallGemmElem { kSmallBF16, kSmallF16, kSmallFP8 };
struct SmallGemmTile { int bm, bn; };
constexpr int kNumSmallTiles = 2;
constexpr SmallGemmTile kSmallTiles[kNumSmallTiles] = {{64, 128}, {128, 128}};
constexpr int kSmallMaxSplits = 16;
constexpr int kGroupedFewRows = kSmallTiles[0].bm;   // rows of the smallest blocks of the grouped form

// `deep`: six stages instead of three, one workgroup per compute unit
int launch_gemm_small(const SmallGemmParams& p, SmallGemmElem elem, int tile, bool deep, hipStream_t stream, const char* who);

}  // namespace tdist
