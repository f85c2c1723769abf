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
  int m_per_rank, rank, world;
  // GEMM-RS: this rank's rows are added up beside (out != NULL): its buffer, in which the other ranks' rows lie, and their sum [m_per_rank, N],
  // N and ldc whole 16-byte pieces, all on 16 bytes
  const unsigned char* own;
  unsigned char* out;
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
// `out`: other ranks' rows that the workgroup of a tile adds up, at most. Only the own rows' tiles have them to load, among the stores of all
// the others and with 112 KB in flight; the other calls are better off with the reduction's launch (3 to 5 us). Whole calls in a graph, one
// launch and two: 64-row tiles of 8 ranks, 2048 x 1024 x 768 9.0 and 10.3 us, 5120 x 1280 x 1280 30.2 and 31.6; 128-row ones of 4 ranks,
// 1024 x 3328 x 1792 19.2 and 19.7, of 2, 2048 x 2048 x 8192 63.5 and 65.1; of 8, 1024 x 4096 x 1536, 22.1 and 20.1. (With their lines brought
// into the L2 first, or asked for in front of the products, they were no faster, and the other tiles slower.)
constexpr int kSmallSumRows = 448;
constexpr int kGroupedFewRows = kSmallTiles[0].bm;   // rows of the smallest blocks of the grouped form
static_assert(kGroupedFewRows == TDIST_GROUP_TAIL_BLOCK, "experts' last rows come in the smallest blocks");

// `deep`: six stages instead of three, one workgroup per compute unit
int launch_gemm_small(const SmallGemmParams& p, SmallGemmElem elem, int tile, bool deep, hipStream_t stream, const char* who);

}  // namespace tdist
