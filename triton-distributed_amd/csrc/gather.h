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
