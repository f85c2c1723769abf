// The gather of the ranks' shards: what lib.hip launches alone and moe.hip beside the joining of row blocks.
#pragma once
#include "common.h"

namespace tdist {

// status[0..1] of the launch before → first_error[0..1] if that is still clear; status cleared for the next launch
__device__ __forceinline__ void retire_status(int32_t* status, int32_t* first_error) {
  const int32_t code = status[0];
  if (code != 0 && first_error != nullptr && first_error[0] == 0) {
    first_error[1] = status[1];
    first_error[0] = code;
  }
  status[1] = 0;
  status[0] = 0;
}

struct GatherParams {
  unsigned char* workspace;
  const unsigned char* src[TDIST_GATHER_MAX_RANKS];   // (by value: no table in memory to keep in step, none to load first)
  long long rank_bytes;
  int32_t *status, *first_error;   // optional: retired as by tdist_status_retire
};

// Workgroup `block` of the `blocks` that bring rank r's rows: four 16-byte loads in flight per lane.
template <int kThreads>
__device__ __forceinline__ void gather_rows(const GatherParams& p, int r, int block, int blocks) {
  const int4v* const src = (const int4v*)p.src[r];
  int4v* const dst = (int4v*)(p.workspace + r * p.rank_bytes);
  const long long n = p.rank_bytes / 16, step = (long long)blocks * (4 * kThreads);
  for (long long i0 = (long long)block * (4 * kThreads) + threadIdx.x; i0 < n; i0 += step) {
    int4v v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i0 + u * kThreads < n) v[u] = __builtin_nontemporal_load(src + i0 + u * kThreads);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i0 + u * kThreads < n) dst[i0 + u * kThreads] = v[u];   // (read again right away, by the GEMM)
  }
}

// The shards of an all-gather read where they lie: offsets from the lowest one, which a kernel adds to one base as 32-bit lane
// offsets. `rows` = 0: there are none (the rows lie in one piece behind the base).
// Against a gather in front (a read and a write of all rows at HBM speed, a launch, and every panel fetched from a second copy), whole
// calls, the same bits: 8 x 2048 x 8192 by 7168 e4m3 637 -> 606 us, 4 x 50 x 4096 by 1536 bf16 18.6 -> 16.2, a Mixtral-8x7B layer
// of 8 x 1024 tokens 503 -> 485. 32 bits of offset keep the K loops as they were: a scalar base and a lane offset per load.
constexpr int kMaxShards = 16;
struct ShardRows {
  int rows;                           // of every shard
  uint32_t off[kMaxShards];           // bytes
  int32_t *status, *first_error;      // optional: retired by the kernel that reads the rows, as a gather's launch does
};
// What the first workgroup of that kernel does beside its tiles.
__device__ __forceinline__ void retire_beside(const ShardRows& s) {
  if (s.rows != 0 && s.status != nullptr && blockIdx.x == 0 && threadIdx.x == 0) retire_status(s.status, s.first_error);
}
// Fills `out` (but its status) and `base`; false where the shards are too many or do not lie within 4 GiB of each other (or `rows` of them could not be
// told apart by the multiplication that divides by it: see shard_magic; a single row has no such factor).
inline bool shards_in_reach(const void* const* shards, int world_size, int rows, int64_t rank_bytes, ShardRows& out, const unsigned char*& base) {
  if (world_size < 1 || world_size > kMaxShards || rows < 2 || (int64_t)world_size * rows * rows >= (1ll << 32)) return false;
  uintptr_t lo = (uintptr_t)shards[0], hi = lo;
  for (int r = 1; r < world_size; ++r) {
    const uintptr_t at = (uintptr_t)shards[r];
    lo = at < lo ? at : lo;
    hi = at > hi ? at : hi;
  }
  if (hi - lo + (uint64_t)rank_bytes >= (1ull << 32) - 4096) return false;
  base = (const unsigned char*)lo;
  out.rows = rows;
  for (int r = 0; r < kMaxShards; ++r) out.off[r] = r < world_size ? (uint32_t)((uintptr_t)shards[r] - lo) : 0;
  return true;
}
// row / rows for 0 <= row < world_size * rows as the high word of row * shard_magic(rows) (exact while world_size * rows * rows < 2^32)
inline uint32_t shard_magic(int rows) { return (uint32_t)(((1ull << 32) + rows - 1) / rows); }

// Checks the arguments of a gather and fills `p`.
inline int gather_params(GatherParams& p, void* workspace, const void* const* shards, int world_size, int64_t rank_bytes,
                         int32_t* status, int32_t* first_error, const char* who) {
  if (!workspace || !shards) return fail(TDIST_ERR_INVALID, "%s: null pointer", who);
  if (world_size < 1 || world_size > TDIST_GATHER_MAX_RANKS)
    return fail(TDIST_ERR_INVALID, "%s: world_size %d (1 .. %d)", who, world_size, TDIST_GATHER_MAX_RANKS);
  if (rank_bytes <= 0 || rank_bytes % 16 != 0 || !aligned16(workspace))
    return fail(TDIST_ERR_UNSUPPORTED, "%s: shards of whole 16-byte pieces, 16-byte aligned", who);
  p = {};
  p.workspace = (unsigned char*)workspace;
  for (int r = 0; r < world_size; ++r) {
    if (!shards[r]) return fail(TDIST_ERR_INVALID, "%s: null pointer", who);
    if (!aligned16(shards[r])) return fail(TDIST_ERR_UNSUPPORTED, "%s: shards of whole 16-byte pieces, 16-byte aligned", who);
    p.src[r] = (const unsigned char*)shards[r];
  }
  p.rank_bytes = rank_bytes;
  p.status = status;
  p.first_error = first_error;
  return TDIST_OK;
}

}  // namespace tdist
