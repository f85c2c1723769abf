// (c) MoE low-latency dispatch / combine permute on one GPU.
//
// Index construction (splits, cumsum, stable scatter index, gather index) is a stable counting sort
// of the flat [T*topk] expert ids, restating in parallel form what the reference does with
//   torch.bincount / cumsum / argsort(stable).argsort()      test/nvidia/test_all_to_all.py:42-46,95-96,314
//   calc_gather_index                                         test/nvidia/test_all_to_all.py:49-92
// One launch when the ids fit one co-resident grid (moe_index_fused_kernel: per-block histograms, a grid-wide
// rendezvous, then every block derives its own prefixes and ranks its ids), else three launches (per-block
// histograms, scan, per-block ranking). Inside a wave the rank of an entry among equal ids is found with ballots
// (one per id bit), so no sort is involved and the order of equal ids is their flat order (stability).
//
// Row movement restates all_to_all_kernel (kernels/nvidia/low_latency_all_to_all.py:56-103): the rows
// of destination d are contiguous in the sorted order, and land in that destination's receive slot.
#include <stdlib.h>

#include <mutex>

#include "gather.h"

namespace tdist {

constexpr int kMoeThreads = 256;              // 4 waves
constexpr int kMoeItemsPerBlock = 256;        // ids ranked by one block (64 per wave: one pass)
constexpr int kMoeMaxExperts = 4096;          // LDS: 4 waves * G * 4 B
constexpr int kScanThreads = 1024;

__host__ __device__ static inline int id_bits(int g) {
  int b = 1;
  while ((1 << b) < g) ++b;
  return b;
}

// hist[b][g] = #ids equal to g among block b's items.
__global__ __launch_bounds__(kMoeThreads) void moe_hist_kernel(const int32_t* __restrict__ ids, int64_t n, int G,
                                                              int32_t* __restrict__ hist,
                                                              int32_t* __restrict__ scan_counter) {
  extern __shared__ int32_t s_hist[];
  if (blockIdx.x == 0 && threadIdx.x == 0) *scan_counter = 0;  // arrival counter of the scan that follows
  for (int g = threadIdx.x; g < G; g += kMoeThreads) s_hist[g] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * kMoeItemsPerBlock;
#pragma unroll
  for (int u = 0; u < kMoeItemsPerBlock / kMoeThreads; ++u) {
    const int64_t i = base + u * kMoeThreads + threadIdx.x;
    if (i < n) {
      const int e = ids[i];
      if (e >= 0 && e < G) atomicAdd(&s_hist[e], 1);
    }
  }
  __syncthreads();
  int32_t* out = hist + (int64_t)blockIdx.x * G;
  for (int g = threadIdx.x; g < G; g += kMoeThreads) out[g] = s_hist[g];
}

// Turns hist[b][g] into the exclusive prefix over b, writes splits[g] and cumsum[0..G]. One workgroup per 256
// columns (a single workgroup would move the whole table through one compute unit: 19 us for 2048 groups x 32
// blocks), four row ranges per column; the workgroup that finishes last adds up the column totals. `counter` is zero
// on entry (the histogram kernel clears it) and zero again on exit.
// splits is never NULL here: the host substitutes a row of the workspace when the caller has none.
constexpr int kScanCols = 256, kScanParts = kScanThreads / kScanCols;
__global__ __launch_bounds__(kScanThreads) void moe_scan_kernel(int32_t* __restrict__ hist, int num_blocks, int G,
                                                               int32_t* __restrict__ splits,
                                                               int32_t* __restrict__ cumsum,
                                                               int32_t* __restrict__ counter) {
  __shared__ int32_t s_tot[kScanParts][kScanCols];
  __shared__ int32_t s_part[kScanThreads];
  __shared__ int s_last;
  const int c = threadIdx.x % kScanCols, q = threadIdx.x / kScanCols;
  const int g = blockIdx.x * kScanCols + c;
  const int rows_per = (num_blocks + kScanParts - 1) / kScanParts;
  const int b_begin = min(q * rows_per, num_blocks), b_end = min(b_begin + rows_per, num_blocks);
  constexpr int kDepth = 32;  // loads in flight per thread and round
  int32_t h[kDepth];
  int32_t total = 0;
  if (g < G) {
    for (int b0 = b_begin; b0 < b_end; b0 += kDepth) {
#pragma unroll
      for (int u = 0; u < kDepth; ++u) h[u] = b0 + u < b_end ? hist[(int64_t)(b0 + u) * G + g] : 0;
#pragma unroll
      for (int u = 0; u < kDepth; ++u) total += h[u];
    }
  }
  s_tot[q][c] = total;
  __syncthreads();
  int32_t run = 0, column = 0;
#pragma unroll
  for (int p = 0; p < kScanParts; ++p) {
    if (p < q) run += s_tot[p][c];
    column += s_tot[p][c];
  }
  if (g < G) {
    if (q == 0) splits[g] = column;
    const bool kept = b_end - b_begin <= kDepth;  // the only round's values are still in registers
    for (int b0 = b_begin; b0 < b_end; b0 += kDepth) {
      if (!kept) {
#pragma unroll
        for (int u = 0; u < kDepth; ++u) h[u] = b0 + u < b_end ? hist[(int64_t)(b0 + u) * G + g] : 0;
      }
#pragma unroll
      for (int u = 0; u < kDepth; ++u) {
        if (b0 + u < b_end) hist[(int64_t)(b0 + u) * G + g] = run;
        run += h[u];
      }
    }
  }
  // ---- the last workgroup: cumsum over all columns -------------------------------------------
  if (gridDim.x > 1) {
    __syncthreads();
    if (threadIdx.x == 0) {
      __threadfence();  // this workgroup's splits are visible before its arrival is
      const int arrived = atomicAdd(counter, 1);
      s_last = arrived == (int)gridDim.x - 1;
      if (s_last) {
        *counter = 0;
        __threadfence();
      }
    }
    __syncthreads();
    if (!s_last) return;
  }
  const int per = (G + kScanThreads - 1) / kScanThreads;  // consecutive columns per thread
  const int g0 = threadIdx.x * per;
  int32_t local_total = 0;
  for (int j = 0; j < per; ++j)
    if (g0 + j < G) local_total += __hip_atomic_load(splits + g0 + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  s_part[threadIdx.x] = local_total;
  __syncthreads();
  // Hillis-Steele inclusive scan over the per-thread totals.
  for (int off = 1; off < kScanThreads; off <<= 1) {
    int32_t v = (threadIdx.x >= off) ? s_part[threadIdx.x - off] : 0;
    __syncthreads();
    s_part[threadIdx.x] += v;
    __syncthreads();
  }
  int32_t acc = s_part[threadIdx.x] - local_total;  // exclusive prefix of this thread's first column
  if (threadIdx.x == 0) cumsum[0] = 0;
  for (int j = 0; j < per; ++j) {
    const int gg = g0 + j;
    if (gg < G) {
      acc += __hip_atomic_load(splits + gg, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      cumsum[gg + 1] = acc;
    }
  }
}

// Ranks block b's items. base position of expert g for wave w of block b =
//   cumsum[g] + hist[b][g] (items of earlier blocks) + items of earlier waves of this block.
__global__ __launch_bounds__(kMoeThreads) void moe_rank_kernel(const int32_t* __restrict__ ids, int64_t n, int topk,
                                                              int G, int nbits, const int32_t* __restrict__ hist,
                                                              const int32_t* __restrict__ cumsum,
                                                              int32_t* __restrict__ scatter_idx,
                                                              int32_t* __restrict__ gather_idx,
                                                              int32_t* __restrict__ topk_idx) {
  extern __shared__ int32_t s_cnt[];  // [4][G]
  constexpr int kWaves = kMoeThreads / 64;
  constexpr int kPerWave = kMoeItemsPerBlock / kWaves;
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  for (int g = threadIdx.x; g < kWaves * G; g += kMoeThreads) s_cnt[g] = 0;
  __syncthreads();
  const int64_t wbase = (int64_t)blockIdx.x * kMoeItemsPerBlock + wave * kPerWave;
  int32_t* my_cnt = s_cnt + wave * G;
  // Pass 1: per-wave counts.
#pragma unroll
  for (int u = 0; u < kPerWave / 64; ++u) {
    const int64_t i = wbase + u * 64 + lane;
    if (i < n) {
      const int e = ids[i];
      if (e >= 0 && e < G) atomicAdd(&my_cnt[e], 1);
    }
  }
  __syncthreads();
  // Pass 2: counts → base positions (exclusive over waves, plus the block and expert offsets).
  const int32_t* bh = hist + (int64_t)blockIdx.x * G;
  for (int g = threadIdx.x; g < G; g += kMoeThreads) {
    int32_t run = cumsum[g] + bh[g];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const int32_t c = s_cnt[w * G + g];
      s_cnt[w * G + g] = run;
      run += c;
    }
  }
  __syncthreads();
  // Pass 3: walk the wave's items in flat order, 64 at a time.
  volatile int32_t* pos = my_cnt;
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (int u = 0; u < kPerWave / 64; ++u) {
    const int64_t i = wbase + u * 64 + lane;
    int e = -1;
    if (i < n) {
      e = ids[i];
      if (e < 0 || e >= G) e = -1;
    }
    const bool valid = e >= 0;
    uint64_t peers = __ballot(valid);
    for (int b = 0; b < nbits; ++b) {
      const bool bit = (e >> b) & 1;
      const uint64_t m = __ballot(valid && bit);
      peers &= bit ? m : ~m;
    }
    if (valid) {
      const int32_t start = pos[e];
      const int rank_in = __popcll(peers & lt_mask);
      const int32_t p = start + rank_in;
      scatter_idx[i] = p;
      gather_idx[p] = (int32_t)(i / topk);
      if (topk_idx) topk_idx[p] = (int32_t)(i % topk);
    } else if (i < n) {
      scatter_idx[i] = -1;
    }
    // every lane of the wave has read pos[] before the leaders advance it
    __builtin_amdgcn_wave_barrier();
    if (valid && (peers & lt_mask) == 0) pos[e] = pos[e] + __popcll(peers);
    __builtin_amdgcn_wave_barrier();
  }
}

// ---- the same in one launch ---------------------------------------------------------------------
// Block b owns ids [b * kItems, (b+1) * kItems), kPerWave consecutive ones per wave, in flat order.
//   1. every wave counts its ids per expert in its own row of LDS counters; the block's sum goes to hist[b][.];
//   2. rendezvous: every block needs every other block's histogram (cumsum is a prefix over ALL ids), so the blocks
//      wait for each other. That is safe because the host only takes this path when the grid is at most one block per
//      compute unit, i.e. co-resident (ctrl[0] counts arrivals and is put back to zero by the last one, ctrl[1] is a
//      generation number that the last arrival bumps; the wait is bounded all the same: if it ran out, the block leaves
//      without writing, cumsum[0] is set to -1 instead of 0 and ctrl[2] to 1, where it stays). Co-residency is the
//      caller's to guarantee (nothing else on the GPU may hold compute units for good, e.g. a persistent GEMM that
//      waits for flags), so the host takes this form only on request (TDIST_DEBUG_MOE_INDEX_FORM = 2);
//   3. every block adds up the histogram columns (all rows: the split of the expert; rows before its own: its offset
//      within the expert), scans the splits into cumsum, and turns its waves' counters into start positions;
//   4. ranking as in moe_rank_kernel.
// ctrl[0] must be zero on entry and is zero again on exit.
// A block is 8 waves x 256 ids. (One block of 16 waves x 2048 ids for all of a decode step's 32768 ids, with no
// rendezvous at all, was measured 4 x slower: a wave ranks its ids 64 at a time, each pass behind the previous one's
// counter update, and 32 such passes in a row cost more than the trips through memory they save.) A single block
// (up to 2048 ids) skips the rendezvous.
constexpr int kFusedSpinLimit = 1 << 22;
constexpr int kFusedThreads = 512, kFusedPerWave = 256, kFusedItems = kFusedThreads / 64 * kFusedPerWave;

// kRecount (few ids): no rendezvous and no histogram rows in memory at all. Every block counts, beside its own ids,
// everybody else's (the ids in front of its range and those behind it, into two more rows of LDS counters): reading
// all the ids once more per block (131 KB out of the L2 for a decode step's 32768) is cheaper than the three trips
// through memory of the rendezvous, and with nothing to wait for the blocks can be small (512 or 1024 ids: one or two
// ranking passes per wave). Measured for 32768 ids, launch to launch: 8.7 us with 64 blocks of 512 ids (10.5 with 16
// blocks of 2048) against 12.3 with the rendezvous, of which 2.2 us are the first trip to memory, 2.4 the counting
// (64 LDS atomics per thread), 1.9 column sums and scan, 1.0 the ranking; an empty launch is 3.3 us of the total.
// The work grows with blocks x ids, so the host takes this form up to kRecountMaxBlocks blocks of 1024 ids only.
constexpr int kRecountMaxBlocks = 64;

// kWide: 64-bit ids (torch.topk's), of which the low words count: read as they are instead of converted by a launch of their
// own in front (8000 ids: 3.2 us).
template <int kThreads, int kPerWave, bool kRecount, bool kWide = false>
__global__ __launch_bounds__(kThreads) void moe_index_fused_kernel(const int32_t* __restrict__ ids, int64_t n, int topk,
                                                                  int G, int nbits, int32_t* hist, int32_t* ctrl,
                                                                  int32_t* __restrict__ splits,
                                                                  int32_t* __restrict__ cumsum,
                                                                  int32_t* __restrict__ scatter_idx,
                                                                  int32_t* __restrict__ gather_idx,
                                                                  int32_t* __restrict__ topk_idx) {
  constexpr int kWaves = kThreads / 64, kItems = kWaves * kPerWave, kPasses = kPerWave / 64;
  extern __shared__ int32_t s_mem[];  // [kWaves][G] wave counters, [G] column sums, kRecount: [2][G] ids before / behind
  int32_t* const s_cnt = s_mem;
  int32_t* const s_col = s_mem + kWaves * G;
  int32_t* const s_out = s_col + G;
  __shared__ int32_t s_part[kWaves];
  __shared__ int s_flag;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int B = gridDim.x, b = blockIdx.x;
  int gen0 = 0;
  if (!kRecount && B > 1 && threadIdx.x == 0) gen0 = __hip_atomic_load(ctrl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // the wave's ids first: the loads are in flight while the counters are cleared
  const int64_t wbase = (int64_t)b * kItems + (int64_t)wave * kPerWave;
  int e_of[kPasses];
#pragma unroll
  for (int u = 0; u < kPasses; ++u) {
    const int64_t i = wbase + u * 64 + lane;
    e_of[u] = i < n ? ids[i << (kWide ? 1 : 0)] : -1;
  }
  // kRecount: the other blocks' ids, four per load, kVecBatch loads in flight (the ranges are multiples of four ids,
  // so a vector lies on one side of this block's range or inside it). The first batch (all of a decode step's ids)
  // goes out here, together with the block's own ids, so that there is one wait for memory and not two.
  constexpr int kVecBatch = kRecount ? 16 : 1;
  const int64_t own_lo = (int64_t)b * kItems, own_hi = own_lo + kItems;
  const int64_t n_vec = (n + 3) / 4;
  int4v q[kVecBatch];
  auto load_others = [&](int64_t v0) {
#pragma unroll
    for (int u = 0; u < kVecBatch; ++u) {
      const int64_t vi = v0 + (int64_t)u * kThreads;
      const bool mine = vi * 4 >= own_lo && vi * 4 < own_hi;
      q[u] = int4v{-1, -1, -1, -1};
      if (vi < n_vec && !mine) {
        if (vi * 4 + 3 < n) {
          if constexpr (kWide) {
            const int4v lo = ((const int4v*)ids)[2 * vi], hi = ((const int4v*)ids)[2 * vi + 1];
            q[u] = int4v{lo[0], lo[2], hi[0], hi[2]};
          } else {
            q[u] = ((const int4v*)ids)[vi];
          }
        } else {
          for (int j = 0; j < 4; ++j) q[u][j] = vi * 4 + j < n ? ids[(vi * 4 + j) << (kWide ? 1 : 0)] : -1;
        }
      }
    }
  };
  // (no branch per id: one unsigned compare, and an id out of range counts into a word of its own lane behind the
  // counters; with 64 ids per lane every instruction per id is a quarter of a microsecond per launch)
  int32_t* const s_trash = s_mem + (kWaves + 3) * G + lane;
  auto count_others = [&](int64_t v0) {
#pragma unroll
    for (int u = 0; u < kVecBatch; ++u) {
      const int64_t vi = v0 + (int64_t)u * kThreads;
      if (vi - lane >= n_vec) break;   // (nothing left for this wave)
      int32_t* const row = s_out + (vi * 4 < own_lo ? 0 : G);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t x = (uint32_t)q[u][j];
        atomicAdd(x < (uint32_t)G ? row + x : s_trash, 1);
      }
    }
  };
  if constexpr (kRecount) {
    if (B > 1) load_others(threadIdx.x);
  }
  for (int g = threadIdx.x; g < (kWaves + (kRecount ? 3 : 0)) * G; g += kThreads) s_cnt[g] = 0;
  __syncthreads();
  // 1. per-wave counts
  int32_t* const my_cnt = s_cnt + wave * G;
#pragma unroll
  for (int u = 0; u < kPasses; ++u) {
    if (e_of[u] < 0 || e_of[u] >= G) e_of[u] = -1;
    if (e_of[u] >= 0) atomicAdd(&my_cnt[e_of[u]], 1);
  }
  if constexpr (kRecount) {
    if (B > 1) {
      count_others(threadIdx.x);
      for (int64_t v0 = threadIdx.x + (int64_t)kVecBatch * kThreads; v0 < n_vec; v0 += (int64_t)kVecBatch * kThreads) {
        load_others(v0);
        count_others(v0);
      }
    }
  }
  __syncthreads();
  if (!kRecount && B > 1) {
    for (int g = threadIdx.x; g < G; g += kThreads) {
      int32_t t = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) t += s_cnt[w * G + g];
      // (device-coherent store: it goes through to memory, so no cache has to be written back before the arrival)
      __hip_atomic_store(hist + (int64_t)b * G + g, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // 2. rendezvous. No fence on either side (a release or acquire fence at device scope writes back or invalidates
    // the whole L2 of this XCD, microseconds after a kernel that left it full of dirty lines): every wave waits for
    // its own coherent stores, then the arrival is counted; the histograms are read back with coherent loads.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
      int ok = 1;
      if (__hip_atomic_fetch_add(ctrl, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == B - 1) {
        __hip_atomic_store(ctrl, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(ctrl + 1, gen0 + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        ok = 0;
        for (int it = 0; it < kFusedSpinLimit; ++it) {
          if (__hip_atomic_load(ctrl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != gen0) {
            ok = 1;
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
      }
      s_flag = ok;
    }
    __syncthreads();
    if (!s_flag) {
      // Reported in a word nobody else writes (block 0, if it gets through later, puts cumsum[0] back to 0): ctrl[2]
      // stays non-zero from the first expiry on until the caller clears it.
      if (threadIdx.x == 0) {
        __hip_atomic_store(ctrl + 2, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        cumsum[0] = -1;
      }
      return;
    }
  }
  // 3. column sums: s_col[g] = ids of expert g in all blocks; the blocks before this one go into wave 0's start
  for (int g = threadIdx.x; g < G; g += kThreads) {
    int32_t total = 0, before = 0;
    if (kRecount && B > 1) {
      before = s_out[g];
      total = before + s_out[G + g];
#pragma unroll
      for (int w = 0; w < kWaves; ++w) total += s_cnt[w * G + g];
    } else if (B > 1) {
      for (int r = 0; r < B; ++r) {
        const int32_t h = __hip_atomic_load(hist + (int64_t)r * G + g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        total += h;
        before += r < b ? h : 0;
      }
    }
    // wave starts within the expert: blocks before, then the earlier waves of this block
    int32_t run = before;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const int32_t c = s_cnt[w * G + g];
      s_cnt[w * G + g] = run;
      run += c;
    }
    s_col[g] = B > 1 ? total : run;
  }
  __syncthreads();
  // exclusive scan of s_col over the experts: consecutive experts per thread, an inclusive scan of the threads' totals
  // within the wave by shuffles, then the waves' totals through LDS
  const int per = (G + kThreads - 1) / kThreads;
  const int g0 = threadIdx.x * per;
  int32_t local_total = 0;
  for (int j = 0; j < per; ++j)
    if (g0 + j < G) local_total += s_col[g0 + j];
  const int32_t incl = wave_scan_add(local_total);
  if (lane == 63) s_part[wave] = incl;
  __syncthreads();
  int32_t acc = incl - local_total;  // ids of the experts before this thread's first one
#pragma unroll
  for (int w = 0; w < kWaves; ++w) acc += w < wave ? s_part[w] : 0;
  if (b == 0 && threadIdx.x == 0) cumsum[0] = 0;
  for (int j = 0; j < per; ++j) {
    const int g = g0 + j;
    if (g < G) {
      const int32_t c = s_col[g];
      if (b == 0) {
        if (splits) splits[g] = c;
        cumsum[g + 1] = acc + c;
      }
      // the expert's first position goes into every wave's start
#pragma unroll
      for (int w = 0; w < kWaves; ++w) s_cnt[w * G + g] += acc;
      acc += c;
    }
  }
  __syncthreads();
  if (scatter_idx == nullptr) return;  // splits and cumsum only
  // 4. walk the wave's ids in flat order, 64 at a time
  volatile int32_t* pos = my_cnt;
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int u = 0; u < kPasses; ++u) {
    if (wbase + u * 64 >= n) break;  // (the whole wave is past the end)
    const int64_t i = wbase + u * 64 + lane;
    const int e = e_of[u];
    const bool valid = e >= 0;
    uint64_t peers = __ballot(valid);
    for (int bit = 0; bit < nbits; ++bit) {
      const bool one = (e >> bit) & 1;
      const uint64_t m = __ballot(valid && one);
      peers &= one ? m : ~m;
    }
    if (valid) {
      const int32_t p = pos[e] + __popcll(peers & lt_mask);
      scatter_idx[i] = p;
      gather_idx[p] = (int32_t)(i / topk);
      if (topk_idx) topk_idx[p] = (int32_t)(i % topk);
    } else if (i < n) {
      scatter_idx[i] = -1;
    }
    // every lane of the wave has read pos[] before the leaders advance it
    __builtin_amdgcn_wave_barrier();
    if (valid && (peers & lt_mask) == 0) pos[e] = pos[e] + __popcll(peers);
    __builtin_amdgcn_wave_barrier();
  }
}

// ---- row movement ------------------------------------------------------------------------------

// Finds d with bound[d] <= p < bound[d+1] in a non-decreasing bound[0..W] with bound[W] > p.
__device__ __forceinline__ int find_dest(const int32_t* bound, int stride, int W, int32_t p) {
  int lo = 0, hi = W;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (bound[mid * stride] <= p) lo = mid; else hi = mid;
  }
  return lo;
}

constexpr int kRowsPerWave = 2;
constexpr int kRowsPerBlock = 4 * kRowsPerWave;  // 4 waves

// Copies up to kRowsPerWave rows of n16 16-byte chunks; all loads of a 512-chunk window are issued
// before its stores so each lane keeps up to 16 vectors in flight.
__device__ __forceinline__ void copy_rows_vec(const int4v* const* src, int4v* const* dst, const bool* has, int n16,
                                              int lane) {
  for (int base = 0; base < n16; base += 8 * 64) {
    int4v v[kRowsPerWave][8];
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
      if (has[r]) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int c = base + j * 64 + lane;
          if (c < n16) v[r][j] = __builtin_nontemporal_load(src[r] + c);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
      if (has[r]) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int c = base + j * 64 + lane;
          if (c < n16) __builtin_nontemporal_store(v[r][j], dst[r] + c);
        }
      }
    }
  }
}

// kFromSlots = false: dispatch (sorted/gathered rows → slots); true: post-process (slots → compact).
// s_bound[d] = first sorted row of destination d, s_bound[W] = total.
template <bool kVec16, bool kFromSlots>
__global__ __launch_bounds__(256) void moe_rows_kernel(const unsigned char* __restrict__ in_rows, int64_t row_bytes,
                                                       const float* __restrict__ in_scales,
                                                       const int32_t* __restrict__ gather_idx,
                                                       const int32_t* __restrict__ counts, int64_t n_rows, int W,
                                                       int Er, int max_m, unsigned char* __restrict__ out_rows,
                                                       float* __restrict__ out_scales,
                                                       int32_t* __restrict__ splits_out) {
  extern __shared__ int32_t s_bound[];  // [W+1]
  if (kFromSlots) {
    // counts = splits[G]: per-destination totals, then a serial prefix (W is small).
    for (int d = threadIdx.x; d < W; d += 256) {
      int32_t t = 0;
      for (int j = 0; j < Er; ++j) t += counts[d * Er + j];
      s_bound[d + 1] = t;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      s_bound[0] = 0;
      for (int d = 0; d < W; ++d) s_bound[d + 1] += s_bound[d];
    }
  } else {
    // counts = cumsum[G+1]
    for (int d = threadIdx.x; d <= W; d += 256) s_bound[d] = counts[d * Er];
    if (splits_out && blockIdx.x == 0) {
      const int G = W * Er;
      for (int g = threadIdx.x; g < G; g += 256) splits_out[g] = counts[g + 1] - counts[g];
    }
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int32_t total = s_bound[W];
  const unsigned char* src[kRowsPerWave];
  unsigned char* dst[kRowsPerWave];
  bool has[kRowsPerWave];
#pragma unroll
  for (int r = 0; r < kRowsPerWave; ++r) {
    const int64_t p = (int64_t)blockIdx.x * kRowsPerBlock + wave * kRowsPerWave + r;
    has[r] = false;
    src[r] = in_rows;
    dst[r] = out_rows;
    if (p >= n_rows || p >= total) continue;
    const int d = find_dest(s_bound, 1, W, (int32_t)p);
    const int64_t in_slot = p - s_bound[d];
    if (in_slot >= max_m) continue;
    const int64_t slot_row = (int64_t)d * max_m + in_slot;
    int64_t src_row, dst_row;
    if (kFromSlots) {
      src_row = slot_row;
      dst_row = p;
    } else {
      src_row = gather_idx ? (int64_t)gather_idx[p] : p;
      dst_row = slot_row;
    }
    has[r] = true;
    src[r] = in_rows + src_row * row_bytes;
    dst[r] = out_rows + dst_row * row_bytes;
    if (in_scales && out_scales && lane == 0) out_scales[dst_row] = in_scales[src_row];
  }
  if (kVec16) {
    copy_rows_vec((const int4v* const*)src, (int4v* const*)dst, has, (int)(row_bytes >> 4), lane);
  } else {
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r)
      if (has[r])
        for (int64_t c = lane; c < row_bytes; c += 64) dst[r][c] = src[r][c];
  }
}

// Token-major dispatch: the row of token t is read once and written to the slot rows of its topk sorted
// positions p = scatter_idx[t*topk + k]. One wave per (token, window of 512 16-byte chunks).
template <bool kVec16>
__global__ __launch_bounds__(256) void moe_dispatch_tokens_kernel(const unsigned char* __restrict__ tokens,
                                                                  int64_t row_bytes, const float* __restrict__ scales,
                                                                  const int32_t* __restrict__ scatter_idx, int topk,
                                                                  const int32_t* __restrict__ cumsum, int64_t n_tokens,
                                                                  int W, int Er, int max_m,
                                                                  unsigned char* __restrict__ slot_rows,
                                                                  float* __restrict__ slot_scales,
                                                                  int32_t* __restrict__ splits_out, int windows) {
  if (splits_out && blockIdx.x == 0) {
    const int G = W * Er;
    for (int g = threadIdx.x; g < G; g += 256) splits_out[g] = cumsum[g + 1] - cumsum[g];
  }
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int64_t unit = (int64_t)blockIdx.x * 4 + wave;
  const int64_t t = unit / windows;
  const int win = (int)(unit - t * windows);
  if (t >= n_tokens) return;
  const unsigned char* src = tokens + t * row_bytes;
  // the row's loads go out first: they do not depend on where the copies land
  const int n16 = (int)(row_bytes >> 4);
  const int base = win * 512;
  int4v v[8];
  if (kVec16) {
    const int4v* s16 = (const int4v*)src;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int c = base + j * 64 + lane;
      if (c < n16) v[j] = s16[c];
    }
  }
  // lane k < topk resolves the slot row of copy k; the W+1 slot boundaries sit one per lane, so the search is
  // register work behind a single load
  int32_t my_dst = -1;
  {
    const int32_t p = lane < topk ? scatter_idx[t * topk + lane] : -1;
    if (W < 64) {
      const int32_t bound = lane <= W ? cumsum[lane * Er] : 0x7fffffff;
      const int32_t total = __builtin_amdgcn_readlane(bound, W);
      int d = 0;
      int32_t first = __builtin_amdgcn_readlane(bound, 0);
      for (int i = 1; i < W; ++i) {
        const int32_t b = __builtin_amdgcn_readlane(bound, i);
        if (b <= p) {
          d = i;
          first = b;
        }
      }
      if (p >= 0 && p < total && p - first < max_m) my_dst = d * max_m + (p - first);
    } else if (p >= 0 && p < cumsum[W * Er]) {
      const int d = find_dest(cumsum, Er, W, p);
      const int32_t in_slot = p - cumsum[d * Er];
      if (in_slot < max_m) my_dst = d * max_m + in_slot;
    }
    if (win == 0 && my_dst >= 0 && scales) slot_scales[my_dst] = scales[t];
  }
  if (kVec16) {
    for (int k = 0; k < topk; ++k) {
      const int32_t dst_row = __shfl(my_dst, k);
      if (dst_row < 0) continue;
      int4v* d16 = (int4v*)(slot_rows + (int64_t)dst_row * row_bytes);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int c = base + j * 64 + lane;
        if (c < n16) __builtin_nontemporal_store(v[j], d16 + c);
      }
    }
  } else {
    for (int k = 0; k < topk; ++k) {
      const int32_t dst_row = __shfl(my_dst, k);
      if (dst_row < 0) continue;
      unsigned char* dst = slot_rows + (int64_t)dst_row * row_bytes;
      for (int64_t c = (int64_t)win * 8192 + lane; c < row_bytes && c < (int64_t)(win + 1) * 8192; c += 64) dst[c] = src[c];
    }
  }
}

// ---- dispatch straight from the expert ids: index build and row movement in one launch ---------------------------
// For a decode step's worth of ids (up to kFusedDispatchMaxIds) the index build is cheaper redone by everybody than
// waited for: as in the recounting form of moe_index_fused_kernel, every workgroup counts ALL ids itself (its own
// tokens' per wave, the ids in front of its range and behind it into two more rows of LDS counters), so it knows the
// splits, their prefix sums and the rank of each of its own (token, k) entries without any exchange, and can place its
// rows at once. The row loads go out before the counting starts, so the counting runs while they are in flight. As
// by-products the workgroups write what tdist_moe_scatter_index writes: scatter_idx and gather_idx for their own
// entries, workgroup 0 the splits and cumsum.
// A workgroup is kFdWaves waves; wave w stands for (token, 8 KB window) unit w of the workgroup, as in
// moe_dispatch_tokens_kernel. The window-0 wave of a token counts and ranks that token's ids.
// Few tokens: windows of `vecs` < 8 KB, so that a row is shared by several waves and the rows by more workgroups. What 16
// whole rows per workgroup cost a decode step of 128 tokens x 8 copies of 7168 B is eight compute units storing 7.3 MB:
// 14.5 us, against 12.2 us with eight waves to a row (64 workgroups; twice as many: the same, four times: 18 for 13 us at 600
// tokens). Up to the scan the launch takes 4.3 us; behind it, instructions and waits in a row are what counts, not bytes: 8.4 us
// (from 12.1) since a token's scale is asked for at the start, the copies' rows and windows are the wave's (scalar branches
// instead of eight tests a lane and copy) and the search among the workgroup's own entries has its reads in flight together.
// 64-bit ids are read as they are (a conversion of 1024 of them in front: 3 us and a launch).
constexpr int kFdWaves = 16, kFdThreads = kFdWaves * 64;
constexpr int64_t kFusedDispatchMaxIds = 65536;

// kFew: windows of less than 8 KB (the others' code is left without the tests for them: they cost a prefill's 4096 rows
// and combine 9 of 110 us). kWide: 64-bit ids, of which the low words count.
template <bool kVec16, bool kFew, bool kWide>
__global__ __launch_bounds__(kFdThreads) void moe_dispatch_fused_kernel(
    const unsigned char* __restrict__ tokens, int64_t row_bytes, const float* __restrict__ scales,
    const int32_t* __restrict__ ids, int topk, int64_t n_tokens, int G, int nbits, int W, int Er, uint32_t er_magic, int max_m,
    int windows, int few_vecs, unsigned char* __restrict__ slot_rows, float* __restrict__ slot_scales, int32_t* __restrict__ splits_out,
    int32_t* __restrict__ splits, int32_t* __restrict__ cumsum, int32_t* __restrict__ scatter_idx,
    int32_t* __restrict__ gather_idx) {
  const int vecs = kFew ? few_vecs : 8;   // 16-byte loads per lane and window
  // [3][G] counters: ids in front of this workgroup's range, its own, ids behind it; [G + 1] expert starts (cumsum);
  // then this workgroup's own ids in flat order, padded to a multiple of four with -1
  extern __shared__ int32_t s_fd[];
  int32_t* const s_before = s_fd;
  int32_t* const s_own = s_fd + G;
  int32_t* const s_behind = s_fd + 2 * G;
  int32_t* const s_start = s_fd + 3 * G;
  int32_t* const s_ids = s_fd + 4 * G + 4;
  __shared__ int32_t s_part[kFdWaves];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int tokens_per_block = kFdWaves / windows;
  const int64_t unit = (int64_t)blockIdx.x * kFdWaves + wave;
  const int64_t t = unit / windows;
  const int win = (int)(unit - t * windows);
  const bool live = t < n_tokens;
  // 1. this token's ids, and everybody else's four at a time
  const int64_t n = n_tokens * topk;
  const int own_n = tokens_per_block * topk;
  const int64_t own_lo = (int64_t)blockIdx.x * own_n, own_hi = own_lo + own_n;
  const int own_first = (wave / windows) * topk;   // the token's first entry among the workgroup's own, in flat order
  const int own_f = own_first + lane;              // and this lane's
  int e = -1;
  if (live && lane < topk) e = ids[(t * topk + lane) << (kWide ? 1 : 0)];
  float my_scale = 0.f;   // (asked for here: a load in front of the copies would hold them up for a trip to memory)
  if (scales && live && win == 0) my_scale = scales[t];
  constexpr int kBatch = 8;
  const int64_t n_vec = (n + 3) / 4;
  const bool vec_ok = (reinterpret_cast<uintptr_t>(ids) & 15u) == 0;
  int4v q[kBatch];
  auto load_others = [&](int64_t v0) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int64_t vi = v0 + (int64_t)u * kFdThreads;
      q[u] = int4v{-1, -1, -1, -1};
      if (vi < n_vec) {
        if (vec_ok && vi * 4 + 3 < n) {
          if constexpr (kWide) {
            const int4v lo = ((const int4v*)ids)[2 * vi], hi = ((const int4v*)ids)[2 * vi + 1];
            q[u] = int4v{lo[0], lo[2], hi[0], hi[2]};
          } else {
            q[u] = ((const int4v*)ids)[vi];
          }
        } else {
          for (int j = 0; j < 4; ++j) q[u][j] = vi * 4 + j < n ? ids[(vi * 4 + j) << (kWide ? 1 : 0)] : -1;
        }
      }
    }
  };
  // (no branch per id: a vector that lies wholly in front of the workgroup's range or behind it, as all but one or
  // two do, takes one unsigned compare per id, and what is not counted goes into a word of the lane's own)
  int32_t* const s_trash = s_ids + ((own_n + 4 + 3) & ~3) + lane;
  auto count_others = [&](int64_t v0) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int64_t vi = v0 + (int64_t)u * kFdThreads;
      if (kFew && vi - lane >= n_vec) break;   // (nothing left for this wave)
      const int64_t i0 = vi * 4;
      if (i0 + 3 < own_lo || i0 >= own_hi) {
        int32_t* const row = i0 < own_lo ? s_before : s_behind;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t x = (uint32_t)q[u][j];
          atomicAdd(x < (uint32_t)G ? row + x : s_trash, 1);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int64_t i = i0 + j;
          const int x = q[u][j];
          if (x >= 0 && x < G && (i < own_lo || i >= own_hi)) atomicAdd(i < own_lo ? &s_before[x] : &s_behind[x], 1);
        }
      }
    }
  };
  load_others(threadIdx.x);
  // the row's loads go out behind the ids' (loads return in order, and the counting only needs the ids: it runs while
  // the row is on its way)
  const int n16 = (int)(row_bytes >> 4);
  const int base = win * vecs * 64;
  int4v v[8];
  if (kVec16 && live) {
    const int4v* s16 = (const int4v*)(tokens + t * row_bytes);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int c = base + j * 64 + lane;
      if ((!kFew || j < vecs) && c < n16) v[j] = s16[c];
    }
  }
  for (int g = threadIdx.x; g < 3 * G; g += kFdThreads) s_fd[g] = 0;
  if ((uint32_t)e >= (uint32_t)G) e = -1;
  if (win == 0 && lane < topk) s_ids[own_f] = e;
  if (threadIdx.x < 4) s_ids[own_n + threadIdx.x] = -1;
  __syncthreads();
  if (e >= 0 && win == 0) atomicAdd(&s_own[e], 1);
  count_others(threadIdx.x);
  for (int64_t v0 = threadIdx.x + (int64_t)kBatch * kFdThreads; v0 < n_vec; v0 += (int64_t)kBatch * kFdThreads) {
    load_others(v0);
    count_others(v0);
  }
  __syncthreads();
  // 3. the splits (ids in front + own + behind) and their exclusive scan over the experts: consecutive experts per
  // thread, the threads' totals within the wave by shuffles, the waves' through LDS
  const int per = (G + kFdThreads - 1) / kFdThreads;
  const int g0 = threadIdx.x * per;
  int32_t local_total = 0;
  for (int j = 0; j < per; ++j)
    if (g0 + j < G) local_total += s_before[g0 + j] + s_own[g0 + j] + s_behind[g0 + j];
  const int32_t incl = wave_scan_add(local_total);
  if (lane == 63) s_part[wave] = incl;
  __syncthreads();
  int32_t acc = incl - local_total;
#pragma unroll
  for (int w = 0; w < kFdWaves; ++w) acc += w < wave ? s_part[w] : 0;
  if (threadIdx.x == 0 && blockIdx.x == 0) cumsum[0] = 0;
  for (int j = 0; j < per; ++j) {
    const int g = g0 + j;
    if (g < G) {
      const int32_t c = s_before[g] + s_own[g] + s_behind[g];
      if (blockIdx.x == 0) {
        if (splits) splits[g] = c;
        if (splits_out) splits_out[g] = c;
        cumsum[g + 1] = acc + c;
      }
      s_start[g] = acc;
      acc += c;
    }
  }
  __syncthreads();
  if (!live) return;
  // 4. the sorted position of this token's k-th entry (lane k): the expert's start, the ids in front of the workgroup's
  // range, and the workgroup's own entries before this one in flat order; then its slot row
  int32_t my_dst = -1;
  if (e >= 0) {
    // (the loop's bounds are the wave's, so that its reads go out several at a time)
    int32_t earlier = 0;
    const int32_t start = s_start[e], before = s_before[e];
    const int d = er_magic != 0 ? (int)__umulhi((uint32_t)e, er_magic) : e;   // e / Er
    const int32_t slot_start = s_start[d * Er];
#pragma unroll 4
    for (int f = 0; f < own_first + topk; f += 4) {
      const int4v o = *(const int4v*)(s_ids + f);
#pragma unroll
      for (int j = 0; j < 4; ++j) earlier += (f + j < own_f && o[j] == e) ? 1 : 0;
    }
    const int32_t p = start + before + earlier;
    if (win == 0) {
      scatter_idx[t * topk + lane] = p;
      gather_idx[p] = (int32_t)t;
    }
    const int32_t in_slot = p - slot_start;
    if (in_slot < max_m) my_dst = d * max_m + in_slot;
    if (win == 0 && my_dst >= 0 && scales) slot_scales[my_dst] = my_scale;
  } else if (lane < topk && win == 0) {
    scatter_idx[t * topk + lane] = -1;
  }
  // 5. the copies: row and window of a copy are the wave's, not the lane's (scalar branches, one address a lane)
  if (kVec16) {
    for (int k = 0; k < topk; ++k) {
      const int32_t dst_row = __builtin_amdgcn_readlane(my_dst, k);
      if (dst_row < 0) continue;
      int4v* const d16 = (int4v*)(slot_rows + (int64_t)dst_row * row_bytes) + base;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (kFew && j >= vecs) break;
        if (lane < n16 - base - j * 64) __builtin_nontemporal_store(v[j], d16 + j * 64 + lane);
      }
    }
  } else {
    const unsigned char* src = tokens + t * row_bytes;
    for (int k = 0; k < topk; ++k) {
      const int32_t dst_row = __builtin_amdgcn_readlane(my_dst, k);
      if (dst_row < 0) continue;
      unsigned char* dst = slot_rows + (int64_t)dst_row * row_bytes;
      for (int64_t c = (int64_t)base * 16 + lane; c < row_bytes && c < ((int64_t)base + vecs * 64) * 16; c += 64) dst[c] = src[c];
    }
  }
}

// ---- online e4m3 quantisation in groups of 128 columns -----------------------------------------------------
// Follows _quant_kernel of the reference's tutorials/04-deepseek-infer-all2all.py (:309-329) and its fused form in
// the dispatch kernel (:180-200): per group, scale = max|x| (as fp32) * fp32(1/448), q = e4m3(float(x) / scale).
// A group whose values are all zero divides 0 by 0 there and so it does here (NaN bytes, scale 0).
constexpr int kQuantGroup = 128;

// One lane's 16 consecutive bf16 columns (two 16-byte vectors) → 16 e4m3 bytes; the 8 lanes of a group share the scale.
__device__ __forceinline__ int4v quant16_bf16_e4m3(const int4v& x0, const int4v& x1, float* scale_out) {
  float f[16];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f[2 * j] = BF16::lo((uint32_t)x0[j]);
    f[2 * j + 1] = BF16::hi((uint32_t)x0[j]);
    f[8 + 2 * j] = BF16::lo((uint32_t)x1[j]);
    f[8 + 2 * j + 1] = BF16::hi((uint32_t)x1[j]);
  }
  float amax = 0.f;
#pragma unroll
  for (int j = 0; j < 16; ++j) amax = fmaxf(amax, fabsf(f[j]));
  amax = fmaxf(amax, __shfl_xor(amax, 1));
  amax = fmaxf(amax, __shfl_xor(amax, 2));
  amax = fmaxf(amax, __shfl_xor(amax, 4));
  const float scale = amax * (float)(1.0 / 448.0);
  *scale_out = scale;
  int4v q;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    int w = 0;
    w = __builtin_amdgcn_cvt_pk_fp8_f32(f[4 * j] / scale, f[4 * j + 1] / scale, w, false);
    w = __builtin_amdgcn_cvt_pk_fp8_f32(f[4 * j + 2] / scale, f[4 * j + 3] / scale, w, true);
    q[j] = w;
  }
  return q;
}

// Stand-alone quantiser: one wave per (row, window of 1024 columns).
__global__ __launch_bounds__(256) void quant_groups_kernel(const unsigned short* __restrict__ x, int64_t n_rows, int hidden,
                                                          int windows, unsigned char* __restrict__ q,
                                                          float* __restrict__ scales) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t unit = (int64_t)blockIdx.x * 4 + wave;
  const int64_t r = unit / windows;
  const int win = (int)(unit - r * windows);
  if (r >= n_rows) return;
  const int col = win * 1024 + lane * 16;
  const bool active = col < hidden;
  int4v x0 = {0, 0, 0, 0}, x1 = {0, 0, 0, 0};
  if (active) {
    const int4v* src = (const int4v*)(x + r * hidden + col);
    x0 = src[0];
    x1 = src[1];
  }
  float scale;
  const int4v v = quant16_bf16_e4m3(x0, x1, &scale);
  if (active) {
    *(int4v*)(q + r * hidden + col) = v;
    if ((lane & 7) == 0) scales[r * (hidden / kQuantGroup) + col / kQuantGroup] = scale;
  }
}

// Token-major dispatch with the quantisation fused in: bf16 token rows in, e4m3 slot rows + one fp32 scale per
// group of 128 columns out. One wave per (token, window of 1024 columns).
__global__ __launch_bounds__(256) void moe_dispatch_quant_kernel(const unsigned short* __restrict__ tokens, int hidden,
                                                                const int32_t* __restrict__ scatter_idx, int topk,
                                                                const int32_t* __restrict__ cumsum, int64_t n_tokens,
                                                                int W, int Er, int max_m,
                                                                unsigned char* __restrict__ slot_rows,
                                                                float* __restrict__ slot_scales,
                                                                int32_t* __restrict__ splits_out, int windows) {
  if (splits_out && blockIdx.x == 0) {
    const int G = W * Er;
    for (int g = threadIdx.x; g < G; g += 256) splits_out[g] = cumsum[g + 1] - cumsum[g];
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t unit = (int64_t)blockIdx.x * 4 + wave;
  const int64_t t = unit / windows;
  const int win = (int)(unit - t * windows);
  if (t >= n_tokens) return;
  const int col = win * 1024 + lane * 16;
  const bool active = col < hidden;
  int4v x0 = {0, 0, 0, 0}, x1 = {0, 0, 0, 0};
  if (active) {
    const int4v* src = (const int4v*)(tokens + t * hidden + col);
    x0 = src[0];
    x1 = src[1];
  }
  // lane k < topk resolves the slot row of copy k (slot boundaries one per lane, as in the unquantised dispatch)
  int32_t my_dst = -1;
  {
    const int32_t p = lane < topk ? scatter_idx[t * topk + lane] : -1;
    if (W < 64) {
      const int32_t bound = lane <= W ? cumsum[lane * Er] : 0x7fffffff;
      const int32_t total = __builtin_amdgcn_readlane(bound, W);
      int d = 0;
      int32_t first = __builtin_amdgcn_readlane(bound, 0);
      for (int i = 1; i < W; ++i) {
        const int32_t b = __builtin_amdgcn_readlane(bound, i);
        if (b <= p) {
          d = i;
          first = b;
        }
      }
      if (p >= 0 && p < total && p - first < max_m) my_dst = d * max_m + (p - first);
    } else if (p >= 0 && p < cumsum[W * Er]) {
      const int d = find_dest(cumsum, Er, W, p);
      const int32_t in_slot = p - cumsum[d * Er];
      if (in_slot < max_m) my_dst = d * max_m + in_slot;
    }
  }
  float scale;
  const int4v v = quant16_bf16_e4m3(x0, x1, &scale);
  const int ng = hidden / kQuantGroup;
  for (int k = 0; k < topk; ++k) {
    const int32_t dst_row = __builtin_amdgcn_readlane(my_dst, k);
    if (dst_row < 0) continue;
    if (active) {
      __builtin_nontemporal_store(v, (int4v*)(slot_rows + (int64_t)dst_row * hidden + col));
      if ((lane & 7) == 0) slot_scales[(int64_t)dst_row * ng + col / kQuantGroup] = scale;
    }
  }
}

// Weighted combine: one wave per (token, window of 64 16-byte column chunks). Lane k < topk resolves the k-th
// source row and its coefficient w[t,k] * scale[row]; the wave then reads the rows eight at a time (all loads
// of a batch in flight before the first add) and accumulates in k order.
// kFp8: rows are e4m3 bytes (16 elements per chunk), else bf16 (8 elements per chunk).
constexpr int kCombineMaxTopk = 32;
constexpr int kCombineWaves = 4;

template <bool kFp8>
__global__ __launch_bounds__(kCombineWaves * 64) void moe_combine_kernel(
    const unsigned char* __restrict__ slot_rows, const float* __restrict__ slot_scales,
    const int32_t* __restrict__ scatter_idx, const float* __restrict__ topk_w, const int32_t* __restrict__ cumsum,
    int64_t n_tokens, int topk, int hidden, int W, int Er, int max_m, int scale_group, int n_windows,
    unsigned short* __restrict__ out) {
  // e4m3 rows: a lane ends up with 32 bytes of output; they go through LDS so that each store instruction of the
  // wave writes one contiguous KiB (16 bytes per lane) instead of every other 16 bytes of two
  __shared__ __attribute__((aligned(16))) unsigned char s_tr[kCombineWaves][kFp8 ? 2048 : 16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t gw = (int64_t)blockIdx.x * kCombineWaves + wave;
  if (gw >= n_tokens * n_windows) return;
  const int64_t t = gw / n_windows;
  const int win = (int)(gw - t * n_windows);

  // Lane k resolves source row k. The W+1 slot boundaries sit one per lane (a single load, issued together with
  // the index and weight loads), so the search for the destination is register work, not a chain of loads.
  int64_t row = -1;  // source row of the lane's k, -1 = skip
  const int32_t p = lane < topk ? scatter_idx[t * topk + lane] : -1;
  float coef = (lane < topk && topk_w) ? topk_w[t * topk + lane] : 1.0f;
  if (max_m > 0) {
    if (W < 64) {
      const int32_t bound = lane <= W ? cumsum[lane * Er] : 0x7fffffff;
      const int32_t total = __builtin_amdgcn_readlane(bound, W);
      int d = 0;
      int32_t base = __builtin_amdgcn_readlane(bound, 0);
      for (int i = 1; i < W; ++i) {
        const int32_t b = __builtin_amdgcn_readlane(bound, i);
        if (b <= p) {
          d = i;
          base = b;
        }
      }
      if (p >= 0 && p < total && p - base < max_m) row = (int64_t)d * max_m + (p - base);
    } else if (p >= 0 && p < cumsum[W * Er]) {
      const int d = find_dest(cumsum, Er, W, p);
      const int64_t in_slot = p - cumsum[d * Er];
      if (in_slot < max_m) row = (int64_t)d * max_m + in_slot;
    }
  } else if (p >= 0) {
    row = p;
  }
  // scale_group == 0: one scale per row, folded into the coefficient; else one per 128 columns, read per lane below
  if (row >= 0 && slot_scales && scale_group == 0) coef *= slot_scales[row];
  if (row < 0) coef = 0.f;
  constexpr int kElems = kFp8 ? 16 : 8;
  const int64_t row_bytes = (int64_t)hidden * (kFp8 ? 1 : 2);
  const int n16 = hidden / kElems;
  const int c = win * 64 + lane;
  const bool active = c < n16;
  float acc[kElems];
#pragma unroll
  for (int j = 0; j < kElems; ++j) acc[j] = 0.f;
  const int row_lo = (int)(uint32_t)row, row_hi = (int)(row >> 32);
  const bool grouped = kFp8 && slot_scales != nullptr && scale_group > 0;
  const int ng = grouped ? hidden / scale_group : 0;
  const int my_group = grouped ? (c * kElems) / scale_group : 0;
  for (int k0 = 0; k0 < topk; k0 += 8) {
    int4v v[8];
    float cf[8], gs[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = min(k0 + j, topk - 1);
      const int64_t r = (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane(row_hi, k) << 32) |
                                  (uint32_t)__builtin_amdgcn_readlane(row_lo, k));
      const bool use = (k0 + j < topk) && r >= 0;
      v[j] = (use && active) ? __builtin_nontemporal_load((const int4v*)(slot_rows + r * row_bytes) + c)
                             : int4v{0, 0, 0, 0};
      gs[j] = (grouped && use && active) ? slot_scales[r * ng + my_group] : 1.f;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = min(k0 + j, topk - 1);
      cf[j] = (k0 + j < topk) ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, coef), k)) : 0.f;
      cf[j] *= gs[j];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (kFp8) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float f[4];
          e4m3x4_to_f32((uint32_t)v[j][q], f);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[4 * q + r] += cf[j] * f[r];
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          acc[2 * q] += cf[j] * BF16::lo((uint32_t)v[j][q]);
          acc[2 * q + 1] += cf[j] * BF16::hi((uint32_t)v[j][q]);
        }
      }
    }
  }
  int4v w[kElems / 8];
#pragma unroll
  for (int q = 0; q < kElems / 8; ++q)
#pragma unroll
    for (int j = 0; j < 4; ++j) w[q][j] = (int)pack_bf16x2(acc[8 * q + 2 * j], acc[8 * q + 2 * j + 1]);
  unsigned short* const orow = out + t * hidden + (int64_t)win * 64 * kElems;  // first output element of the window
  if (kFp8) {
    TDIST_AS3 unsigned char* tr = (TDIST_AS3 unsigned char*)s_tr[wave];
    *(TDIST_AS3 int4v*)(tr + lane * 32) = w[0];
    *(TDIST_AS3 int4v*)(tr + lane * 32 + 16) = w[kElems / 8 - 1];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int piece = h * 64 + lane;  // 16-byte piece of the window's 2 KiB of output
      const int4v o = *(TDIST_AS3 int4v*)(tr + piece * 16);
      if (win * 64 + piece / 2 < n16) __builtin_nontemporal_store(o, (int4v*)orow + piece);
    }
  } else {
    if (active) __builtin_nontemporal_store(w[0], (int4v*)orow + lane);
  }
}

// Weighted sum of a token's rows as above (bf16 rows, row t * topk + k), and for the tokens that this rank owns the reduction over
// the ranks' partial results right behind it: the wave that has a piece of such a row rounds it, leaves it in the rank's slice of
// the partials, as the ranks with their own tokens' sums do, and adds the slices up in the order of tdist_reduce_slices, rank + 1 first.
// Memory-bound: 8192 tokens x 2 of 4096 by 8 ranks 48 us, 5.6 TB/s; as three launches (sum, copy of the own slice, reduction) 58 us
// and the gaps between them. The own tokens come first: their waves have the most to read.
template <int kFirst>
__device__ __forceinline__ void add_slices(float* acc, const int4v* own_chunk, int64_t slice16, int first, int rank, int W, const int4v& own) {
  for (int i0 = 0; i0 < W; i0 += kFirst) {
    int4v v[kFirst];
#pragma unroll
    for (int j = 0; j < kFirst; ++j) {
      const int i = min(i0 + j, W - 1);
      const int s = first + i < W ? first + i : first + i - W;
      v[j] = own;
      if (s != rank) v[j] = __builtin_nontemporal_load(own_chunk + (int64_t)s * slice16);
    }
#pragma unroll
    for (int j = 0; j < kFirst; ++j) {
      if (i0 + j < W) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          acc[2 * q] += BF16::lo((uint32_t)v[j][q]);
          acc[2 * q + 1] += BF16::hi((uint32_t)v[j][q]);
        }
      }
    }
  }
}

__global__ __launch_bounds__(kCombineWaves * 64) void moe_combine_reduce_kernel(
    const unsigned char* __restrict__ rows, const float* __restrict__ topk_w, int n_tokens, int topk, int hidden, int n_windows, int rank,
    int W, int m_per, unsigned char* __restrict__ partials, unsigned char* __restrict__ sums, unsigned char* __restrict__ out) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t gw = (int64_t)blockIdx.x * kCombineWaves + wave;
  if (gw >= (int64_t)n_tokens * n_windows) return;
  const int turn = (int)(gw / n_windows), win = (int)(gw - (int64_t)turn * n_windows);
  const int t = turn + rank * m_per < n_tokens ? turn + rank * m_per : turn + rank * m_per - n_tokens;
  const float coef = lane < topk ? topk_w[(int64_t)t * topk + lane] : 0.f;
  const int64_t row16 = hidden / 8;
  const int c = win * 64 + lane;
  const bool active = c < row16;
  const int4v* const src = (const int4v*)rows + (int64_t)t * topk * row16 + c;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < topk; k0 += 8) {
    int4v v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = k0 + j < topk && active ? __builtin_nontemporal_load(src + (k0 + j) * row16) : int4v{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float cf = k0 + j < topk ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, coef), min(k0 + j, topk - 1))) : 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        acc[2 * q] += cf * BF16::lo((uint32_t)v[j][q]);
        acc[2 * q + 1] += cf * BF16::hi((uint32_t)v[j][q]);
      }
    }
  }
  if (!active) return;
  int4v w;
#pragma unroll
  for (int j = 0; j < 4; ++j) w[j] = (int)pack_bf16x2(acc[2 * j], acc[2 * j + 1]);
  if (turn >= m_per) {   // another rank's token
    __builtin_nontemporal_store(w, (int4v*)sums + (int64_t)t * row16 + c);
    return;
  }
  const int64_t slice16 = m_per * row16;
  int4v* const mine = (int4v*)partials + turn * row16 + c;   // of slice 0
  mine[rank * slice16] = w;
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = 0.f;
  add_slices<8>(acc, mine, slice16, rank + 1 < W ? rank + 1 : 0, rank, W, w);
#pragma unroll
  for (int j = 0; j < 4; ++j) w[j] = (int)pack_bf16x2(acc[2 * j], acc[2 * j + 1]);
  __builtin_nontemporal_store(w, (int4v*)out + turn * row16 + c);
}

// ---- align / sort for the grouped GEMM ------------------------------------------------------------------
// Follows moe_ag_scatter_align_block_size_kernel (csrc/lib/moe_utils.cu:60-165): per rank segment, entries grouped
// by expert in flat order, every group padded to a multiple of block_size, groups and segments laid end to end.
// Built on the stable index of this file with the composite key segment * E + expert: the position of an entry in
// the padded layout is its position in the unpadded sorted order moved by the padding in front of its group.

// keys[i] = (i / per_iter) * E + ids[i], or -1 for an id outside [0, E)
// Also pre-fills sorted_ids[0 .. fill_n) with n (the value padding positions keep; fill_n = 0: the caller has done it).
__global__ __launch_bounds__(256) void moe_align_keys_kernel(const void* __restrict__ ids, int ids_int64, int64_t n,
                                                            int64_t per_iter, int E, int32_t* __restrict__ keys,
                                                            int32_t* __restrict__ sorted_ids, int64_t fill_n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < fill_n) sorted_ids[i] = (int32_t)n;
  if (i >= n) return;
  const int64_t id = ids_int64 ? ((const int64_t*)ids)[i] : (int64_t)((const int32_t*)ids)[i];
  keys[i] = (id >= 0 && id < E) ? (int32_t)((i / per_iter) * E + id) : -1;
}

// Padding and placement in one launch. Every workgroup works out the padded exclusive prefix over the G = R * E group
// sizes for itself (G <= 4096 values through LDS: cheaper than a launch of its own and the wait for it), then places
// its 256 entries: an entry's position in the padded layout is its position in the unpadded sorted order moved by the
// padding in front of its group. Workgroup 0 also writes the per-block expert / segment ids, the blocks per segment
// and the padded total.
constexpr int kPlaceThreads = 256;
__global__ __launch_bounds__(kPlaceThreads) void moe_align_place_kernel(
    const int32_t* __restrict__ keys, const int32_t* __restrict__ scatter_idx, const int32_t* __restrict__ splits,
    const int32_t* __restrict__ cumsum, int64_t n, int G, int E, int R, int block_size, int32_t* __restrict__ sorted_ids,
    int32_t* __restrict__ expert_ids, int32_t* __restrict__ block_barrier_ids, int32_t* __restrict__ rank_block_num,
    int32_t* __restrict__ total_post_pad) {
  extern __shared__ int32_t s_pad[];  // [G + 1] padded exclusive prefix
  __shared__ int32_t s_part[kPlaceThreads];
  // the entry's own loads first: they do not depend on the prefix
  const int64_t i = (int64_t)blockIdx.x * kPlaceThreads + threadIdx.x;
  const int32_t k = i < n ? keys[i] : -1;
  const int32_t rank_in_group = k >= 0 ? scatter_idx[i] - cumsum[k] : 0;
  const int per = (G + kPlaceThreads - 1) / kPlaceThreads;  // consecutive groups per thread
  const int g0 = threadIdx.x * per;
  int32_t local_total = 0;
  for (int j = 0; j < per; ++j) {
    const int g = g0 + j;
    if (g < G) local_total += (splits[g] + block_size - 1) / block_size * block_size;
  }
  s_part[threadIdx.x] = local_total;
  __syncthreads();
  for (int off = 1; off < kPlaceThreads; off <<= 1) {
    const int32_t v = (threadIdx.x >= off) ? s_part[threadIdx.x - off] : 0;
    __syncthreads();
    s_part[threadIdx.x] += v;
    __syncthreads();
  }
  int32_t run = s_part[threadIdx.x] - local_total;
  if (threadIdx.x == 0) s_pad[0] = 0;
  for (int j = 0; j < per; ++j) {
    const int g = g0 + j;
    if (g < G) {
      const int32_t padded = (splits[g] + block_size - 1) / block_size * block_size;
      if (blockIdx.x == 0) {
        for (int32_t b = run / block_size; b < (run + padded) / block_size; ++b) {
          expert_ids[b] = g % E;
          block_barrier_ids[b] = g / E;
        }
      }
      run += padded;
      s_pad[g + 1] = run;
    }
  }
  __syncthreads();
  if (blockIdx.x == 0) {
    for (int r = threadIdx.x; r < R; r += kPlaceThreads) rank_block_num[r] = (s_pad[(r + 1) * E] - s_pad[r * E]) / block_size;
    if (threadIdx.x == 0) *total_post_pad = s_pad[G];
  }
  if (k >= 0) sorted_ids[s_pad[k] + rank_in_group] = (int32_t)i;
}

// Align / sort in ONE launch for few entries (up to kRecountMaxBlocks blocks of 1024): the recounting index build above
// with the composite keys formed on the way in and the groups' starts taken from the PADDED prefix, so that an entry's
// rank is its place in the padded layout at once. Every block counts all entries (those in front of its range, its
// own, those behind), works out the padded prefix over the G = R * E groups for itself and places its own entries;
// the padding positions, the per-block expert / segment ids and the positions behind the padded total (up to fill_n)
// are shared out among the blocks, groups in turn; block 0 writes the blocks per segment and the padded total.
// Many groups of few entries: the padding is the larger part (1000 tokens x 8, 256 experts x 8 segments, blocks of 128:
// 260 000 positions for 8000 entries), so the launch has a block per kAlignFillPerBlock positions even where the entries
// alone need fewer: blocks beyond the entries count like the others and only fill (66 blocks 7.8 us, 131 6.8, 256 6.7).
// What bounds it: two trips to memory and the work per group, of which there are thousands. The eight waves' counts of a
// group are the bytes of one 64-bit word (a wave has at most 128 entries), so a group is 20 bytes to clear, to add up (four
// groups a step, the bytes of a word by a sum of absolute differences) and to look up, and nothing is written back per
// wave: the sizes above take 6.4 us, 12.4 with a row of counters per wave (of which 7 were clearing, sums and scan). With
// 32768 entries 12.7 (64 experts: 11.6): there it is the counting, 64 LDS atomics per thread.
constexpr int kAlignFillPerBlock = 1024;
constexpr int kAlignMostQuads = (kMoeMaxExperts / 4 + kFusedThreads - 1) / kFusedThreads;   // steps of four groups per thread
static int64_t align_lds_bytes(int64_t G) { return 20 * ((G + 3) / 4 * 4) + 16 + 256; }
template <int kPasses, bool kIds64>
__global__ __launch_bounds__(kFusedThreads) void moe_align_fused_kernel(
    const void* __restrict__ ids_v, int64_t n, int per_iter, int E, int R, int nbits, int block_size,
    int32_t* __restrict__ sorted_ids, int64_t fill_n, int32_t* __restrict__ expert_ids,
    int32_t* __restrict__ block_barrier_ids, int32_t* __restrict__ rank_block_num, int32_t* __restrict__ total_post_pad,
    uint32_t seg_magic, uint32_t block_magic) {
  constexpr int kThreads = kFusedThreads, kWaves = kThreads / 64, kPerWave = 64 * kPasses, kItems = kWaves * kPerWave;
  static_assert(kWaves == 8 && kPerWave < 256, "a byte of a 64-bit word per wave");
  typedef __attribute__((__vector_size__(2 * sizeof(long long)))) long long long2v;
  const int G = E * R, Gp = (G + 3) & ~3;
  extern __shared__ __attribute__((aligned(16))) int32_t s_mem[];
  unsigned long long* const s_own = (unsigned long long*)s_mem;   // [Gp] entries of this block, a byte per wave
  int32_t* const s_before = s_mem + 2 * Gp;                       // [Gp] entries in front of the block
  int32_t* const s_behind = s_before + Gp;                        // [Gp] those behind it, later all of the group's
  int32_t* const s_start = s_behind + Gp;                         // [Gp + 1] padded exclusive prefix
  __shared__ int32_t s_part[kWaves];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int B = gridDim.x, b = blockIdx.x;
  const int32_t* const ids32 = (const int32_t*)ids_v;
  const long long* const ids64 = (const long long*)ids_v;
  const uint32_t per = (uint32_t)per_iter;
  // the wave's own entries first
  const int64_t wbase = (int64_t)b * kItems + (int64_t)wave * kPerWave;
  long long id_own[kPasses];
#pragma unroll
  for (int u = 0; u < kPasses; ++u) {
    const int64_t i = wbase + u * 64 + lane;
    id_own[u] = i < n ? (kIds64 ? ids64[i] : (long long)ids32[i]) : -1;
  }
  // everybody else's, four per lane and load, all of a batch in flight
  constexpr int kVecBatch = 16;
  const int64_t own_lo = (int64_t)b * kItems, own_hi = own_lo + kItems;
  const int64_t n_vec = (n + 3) / 4;
  int4v q32[kIds64 ? 1 : kVecBatch];
  long2v q64[kIds64 ? 2 * kVecBatch : 1];
  auto load_others = [&](int64_t v0) {   // (v0: the wave's first vector of the batch)
#pragma unroll
    for (int u = 0; u < kVecBatch; ++u) {
      if (v0 + (int64_t)u * kThreads >= n_vec) break;
      const int64_t vi = v0 + (int64_t)u * kThreads + lane;
      const bool take = vi < n_vec && !(vi * 4 >= own_lo && vi * 4 < own_hi);
      const bool whole = vi * 4 + 3 < n;
      if constexpr (kIds64) {
        q64[2 * u] = long2v{-1, -1};
        q64[2 * u + 1] = long2v{-1, -1};
        if (take && whole) {
          q64[2 * u] = ((const long2v*)ids64)[2 * vi];
          q64[2 * u + 1] = ((const long2v*)ids64)[2 * vi + 1];
        } else if (take) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (vi * 4 + j < n) q64[2 * u + j / 2][j % 2] = ids64[vi * 4 + j];
        }
      } else {
        q32[u] = int4v{-1, -1, -1, -1};
        if (take && whole) q32[u] = ((const int4v*)ids32)[vi];
        else if (take) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (vi * 4 + j < n) q32[u][j] = ids32[vi * 4 + j];
        }
      }
    }
  };
  // Every lane counts n / kThreads entries, so an entry costs as few instructions as can be: the segment of a vector's
  // first entry by a multiplication (seg_magic = ceil(2^32 / per), exact below 65536 entries), at most one segment
  // boundary inside a vector (per >= 4), one unsigned compare for the id's range, and no branch: an id out of range
  // counts into a word of its own lane behind the counters.
  int32_t* const s_trash = s_start + Gp + 4 + lane;
  auto count_others = [&](int64_t v0) {
#pragma unroll
    for (int u = 0; u < kVecBatch; ++u) {
      if (v0 + (int64_t)u * kThreads >= n_vec) break;   // (nothing left for this wave)
      const int64_t vi = v0 + (int64_t)u * kThreads + lane;
      int32_t* const row = vi * 4 < own_lo ? s_before : s_behind;
      const uint32_t i0 = (uint32_t)(vi * 4);
      const uint32_t seg = __umulhi(i0, seg_magic);
      const uint32_t to_next = (seg + 1) * per - i0;   // entries of this vector that are still in segment `seg`
      int32_t* const row_seg = row + seg * (uint32_t)E;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t lo;
        bool ok;
        if constexpr (kIds64) {
          const long long id = q64[2 * u + j / 2][j % 2];
          lo = (uint32_t)id;
          ok = (uint32_t)(id >> 32) == 0u && lo < (uint32_t)E;
        } else {
          lo = (uint32_t)q32[u][j];
          ok = lo < (uint32_t)E;
        }
        int32_t* const at = row_seg + (j > 0 && (uint32_t)j >= to_next ? E : 0) + lo;
        atomicAdd(ok ? at : s_trash, 1);
      }
    }
  };
  const int64_t first_vec = wave * 64;
  if (B > 1) load_others(first_vec);
  for (int g = threadIdx.x; g < Gp; g += kThreads) ((int4v*)s_mem)[g] = int4v{0, 0, 0, 0};   // 16 bytes a group
  // the key of each own entry and its place among the wave's entries of that key: those of lower lanes, and of an earlier pass
  int e_of[kPasses], within[kPasses];
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int u = 0; u < kPasses; ++u) {
    const uint32_t i = (uint32_t)(wbase + u * 64 + lane);
    e_of[u] = id_own[u] >= 0 && id_own[u] < E ? (int)__umulhi(i, seg_magic) * E + (int)id_own[u] : -1;
    uint64_t peers[kPasses];
#pragma unroll
    for (int v = 0; v <= u; ++v) peers[v] = __ballot(e_of[v] >= 0);
    for (int bit = 0; bit < nbits; ++bit) {
      const bool one = (e_of[u] >> bit) & 1;
#pragma unroll
      for (int v = 0; v <= u; ++v) {
        const uint64_t m = __ballot((e_of[v] >> bit) & 1);
        peers[v] &= one ? m : ~m;
      }
    }
    within[u] = __popcll(peers[u] & lt_mask);
#pragma unroll
    for (int v = 0; v < u; ++v) within[u] += __popcll(peers[v]);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPasses; ++u)
    if (e_of[u] >= 0) atomicAdd(&s_own[e_of[u]], 1ull << (8 * wave));
  if (B > 1) {
    count_others(first_vec);
    for (int64_t v0 = first_vec + (int64_t)kVecBatch * kThreads; v0 < n_vec; v0 += (int64_t)kVecBatch * kThreads) {
      load_others(v0);
      count_others(v0);
    }
  }
  __syncthreads();
  // group sizes and the exclusive scan of the PADDED ones: consecutive groups per thread, then across threads and waves
  // (whole blocks by a multiplication: exact up to 65536 entries and blocks of 32768; 0: by a division)
  auto padded = [&](int32_t c) {
    const uint32_t x = (uint32_t)(c + block_size - 1);
    return (int32_t)(block_magic != 0 ? __umulhi(x, block_magic) : x / (uint32_t)block_size) * block_size;
  };
  auto sum_bytes = [](unsigned long long w, int32_t to) {
    return (int32_t)__builtin_amdgcn_sad_u8((uint32_t)(w >> 32), 0u, __builtin_amdgcn_sad_u8((uint32_t)w, 0u, (uint32_t)to));
  };
  const int quads = Gp / 4, quads_each = (quads + kThreads - 1) / kThreads;
  int4v size[kAlignMostQuads];   // padded
  int32_t local_total = 0;
#pragma unroll
  for (int k = 0; k < kAlignMostQuads; ++k) {
    const int at = threadIdx.x * quads_each + k;
    size[k] = int4v{0, 0, 0, 0};
    if (k < quads_each && at < quads) {
      const int4v before = ((const int4v*)s_before)[at], behind = ((const int4v*)s_behind)[at];
      const int4v own0 = ((const int4v*)s_own)[2 * at], own1 = ((const int4v*)s_own)[2 * at + 1];
      int4v c = before + behind;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        c[j] = sum_bytes((unsigned long long)(uint32_t)own0[2 * j + 1] << 32 | (uint32_t)own0[2 * j], c[j]);
        c[2 + j] = sum_bytes((unsigned long long)(uint32_t)own1[2 * j + 1] << 32 | (uint32_t)own1[2 * j], c[2 + j]);
      }
      ((int4v*)s_behind)[at] = c;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        size[k][j] = padded(c[j]);
        local_total += size[k][j];
      }
    }
  }
  const int32_t incl = wave_scan_add(local_total);
  if (lane == 63) s_part[wave] = incl;
  __syncthreads();
  int32_t acc = incl - local_total, total = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const int32_t part = s_part[w];
    acc += w < wave ? part : 0;
    total += part;
  }
#pragma unroll
  for (int k = 0; k < kAlignMostQuads; ++k) {
    const int at = threadIdx.x * quads_each + k;
    if (k < quads_each && at < quads) {
      int4v from;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        from[j] = acc;
        acc += size[k][j];
      }
      ((int4v*)s_start)[at] = from;
    }
  }
  if (threadIdx.x == 0) s_start[Gp] = total;
  __syncthreads();
  // the wave's entries
#pragma unroll
  for (int u = 0; u < kPasses; ++u) {
    const int e = e_of[u];
    if (e >= 0) {
      const unsigned long long earlier_waves = s_own[e] & ((1ull << (8 * wave)) - 1);
      sorted_ids[s_start[e] + sum_bytes(earlier_waves, s_before[e] + within[u])] = (int32_t)(wbase + u * 64 + lane);
    }
  }
  if (b == 0) {
    for (int r = threadIdx.x; r < R; r += kThreads) rank_block_num[r] = (s_start[(r + 1) * E] - s_start[r * E]) / block_size;
    if (threadIdx.x == 0) *total_post_pad = total;
  }
  // the groups this block looks after (a wave each, in turn): their padding positions and their blocks' ids
  for (int g = b + B * wave; g < G; g += B * kWaves) {
    const int32_t st = s_start[g], c = s_behind[g], pc = padded(c);
    for (int32_t o = c + lane; o < pc; o += 64) sorted_ids[st + o] = (int32_t)n;
    if (pc > 0) {
      const int seg = g / E, expert = g - seg * E;
      for (int32_t k = st / block_size + lane; k < (st + pc) / block_size; k += 64) {
        expert_ids[k] = expert;
        block_barrier_ids[k] = seg;
      }
    }
  }
  // and its share of the positions behind the padded total
  if (fill_n > total) {
    const int64_t share = (fill_n - total + B - 1) / B;
    const int64_t lo = total + share * b, hi = lo + share < fill_n ? lo + share : fill_n;
    for (int64_t i = lo + threadIdx.x; i < hi; i += kThreads) sorted_ids[i] = (int32_t)n;
  }
}

static int moe_index_common(const int32_t* ids, int64_t n_ids, int topk, int G, int32_t* splits, int32_t* cumsum,
                            int32_t* scatter_idx, int32_t* gather_idx, int32_t* topk_idx, void* workspace,
                            int64_t workspace_bytes, hipStream_t stream, bool want_index, const char* who, bool wide = false) {
  if (!ids || !cumsum) return fail(TDIST_ERR_INVALID, "%s: null ids or cumsum", who);
  if (want_index && (!scatter_idx || !gather_idx)) return fail(TDIST_ERR_INVALID, "%s: null index output", who);
  if (n_ids < 0 || G <= 0 || (want_index && topk <= 0)) return fail(TDIST_ERR_INVALID, "%s: bad sizes", who);
  if (G > kMoeMaxExperts) return fail(TDIST_ERR_UNSUPPORTED, "%s: num_experts %d > %d", who, G, kMoeMaxExperts);
  if (n_ids > 0x7fffffffll) return fail(TDIST_ERR_UNSUPPORTED, "%s: more than 2^31-1 ids", who);
  const int64_t need = tdist_moe_workspace_bytes(n_ids, G);
  if (!workspace || workspace_bytes < need)
    return fail(TDIST_ERR_WORKSPACE, "%s: workspace %lld B < %lld B", who, (long long)workspace_bytes, (long long)need);
  const int num_blocks = (int)ceil_div(n_ids > 0 ? n_ids : 1, kMoeItemsPerBlock);
  // workspace: 256 bytes of control words (always at the start, whatever the sizes of the call), the block
  // histograms, one row for the splits
  int32_t* scan_counter = (int32_t*)workspace;
  int32_t* hist = scan_counter + 64;
  int32_t* splits_buf = splits ? splits : hist + (int64_t)num_blocks * G;
  // One launch for few ids (up to 65536): every block counts all of them itself and nothing is exchanged. Beyond
  // that, three launches. A one-launch form whose blocks (2048 ids each, at most one per compute unit) wait for each
  // other's histograms exists too, but its wait only ends if every block is resident at once, which the library
  // cannot know when other streams hold compute units: it is taken on request only (TDIST_DEBUG_MOE_INDEX_FORM = 2,
  // for tests and measurements; 3 = always three launches). Its histogram rows (one per 2048 ids) fit the rows the
  // workspace holds (one per 256 ids).
  const DeviceInfo& di = device_info();
  const int64_t fused_blocks = ceil_div(n_ids > 0 ? n_ids : 1, kFusedItems);
  const int form_dbg = debug_get(TDIST_DEBUG_MOE_INDEX_FORM);
  constexpr int kLdsLimit = 160 * 1024 - 256;          // (the kernel has a few static words of its own)
  constexpr int kRowsPlain = kFusedThreads / 64 + 1;   // wave counters, column sums
  constexpr int kRowsRecount = kRowsPlain + 2;         // and the ids before / behind the block
  constexpr int kSmall = kFusedThreads;                // ids per block of the recounting forms: 512, or 1024
  const int64_t n1 = n_ids > 0 ? n_ids : 1;
  const bool can_recount = form_dbg != 2 && kRowsRecount * G * 4 + 256 <= kLdsLimit && aligned16(ids);
  // 0: blocks of 2048 ids that exchange their histograms; 1 / 2: blocks of 512 / 1024 ids that count everything
  const int form = !can_recount ? 0 : ceil_div(n1, kSmall) <= kRecountMaxBlocks ? 1 : ceil_div(n1, 2 * kSmall) <= kRecountMaxBlocks ? 2 : 0;
  if (wide && (form == 0 || form_dbg == 2 || form_dbg == 3))
    return fail(TDIST_ERR_UNSUPPORTED, "%s: 64-bit ids are for the one-launch form that counts them all (16-byte aligned, at most "
                "%d of them, counters that fit the LDS): convert them and call tdist_moe_scatter_index", who, kRecountMaxBlocks * 2 * kSmall);
  if (di.ok == 1 && fused_blocks <= di.num_cus && form_dbg != 3 && (form != 0 || form_dbg == 2)) {
    auto kern = form == 1 ? (wide ? moe_index_fused_kernel<kFusedThreads, kSmall / 8, true, true>
                                  : moe_index_fused_kernel<kFusedThreads, kSmall / 8, true>)
              : form == 2 ? (wide ? moe_index_fused_kernel<kFusedThreads, kSmall / 4, true, true>
                                  : moe_index_fused_kernel<kFusedThreads, kSmall / 4, true>)
                          : moe_index_fused_kernel<kFusedThreads, kFusedPerWave, false>;
    const int64_t blocks = form == 1 ? ceil_div(n1, kSmall) : form == 2 ? ceil_div(n1, 2 * kSmall) : fused_blocks;
    const int rows = form != 0 ? kRowsRecount : kRowsPlain;
    static bool attr_set[2][3] = {{false, false, false}, {false, false, false}};
    if (!attr_set[wide][form]) {
      const int most = rows * kMoeMaxExperts * 4 < kLdsLimit ? rows * kMoeMaxExperts * 4 : kLdsLimit;
      if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, most) != hipSuccess)
        return fail(TDIST_ERR_LAUNCH, "%s: cannot reserve LDS for the index kernel", who);
      attr_set[wide][form] = true;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kFusedThreads), (size_t)rows * G * 4 + (form != 0 ? 256 : 0), stream,
                       ids, n_ids, want_index ? topk : 1, G, id_bits(G), hist, scan_counter, splits, cumsum,
                       want_index ? scatter_idx : nullptr, gather_idx, topk_idx);
    return launch_status(who);
  }
  if (wide) return fail(TDIST_ERR_DEVICE, "%s: current device is not gfx950", who);
  hipLaunchKernelGGL(moe_hist_kernel, dim3(num_blocks), dim3(kMoeThreads), (size_t)G * 4, stream, ids, n_ids, G, hist,
                     scan_counter);
  hipLaunchKernelGGL(moe_scan_kernel, dim3((G + kScanCols - 1) / kScanCols), dim3(kScanThreads), 0, stream, hist, num_blocks,
                     G, splits_buf, cumsum, scan_counter);
  if (want_index && n_ids > 0) {
    hipLaunchKernelGGL(moe_rank_kernel, dim3(num_blocks), dim3(kMoeThreads), (size_t)G * 4 * (kMoeThreads / 64), stream,
                       ids, n_ids, topk, G, id_bits(G), hist, cumsum, scatter_idx, gather_idx, topk_idx);
  }
  return launch_status(who);
}

// ---- the index build without a caller's workspace ---------------------------------------------------------
// Scratch for tdist_moe_scatter_index_static: every GPU the library runs on holds its own copy of this array until the
// process ends. Host code never uses the array's name as an address: the per-device address comes from
// hipGetSymbolAddress, once per device, and is what the kernels are given.
constexpr int64_t kMoeStaticScratchBytes = 1 << 20;
static __device__ __align__(256) unsigned char scratch[kMoeStaticScratchBytes];

constexpr int kMoeMaxDevices = 64;
static void* g_scratch_ptr[kMoeMaxDevices];   // device address of `scratch` per device, NULL until looked up
static std::mutex g_scratch_mutex;

// Device address of the current device's copy of `scratch` (looked up on first use, with that device current).
static int moe_static_scratch(void** out, const char* who) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMoeMaxDevices)
    return fail(TDIST_ERR_DEVICE, "%s: no current device (or more than %d devices)", who, kMoeMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr)
      return fail(TDIST_ERR_DEVICE, "%s: hipGetSymbolAddress(scratch) failed on device %d: %s", who, dev, hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return TDIST_OK;
}

int moe_static_scratch_init() {
  void* ptr = nullptr;
  return moe_static_scratch(&ptr, "tdist_init");
}

// ---- row blocks without rank segments ------------------------------------------------------------------------
// The align / sort ends its row blocks with their rank segment, which is what a GEMM needs that starts on one rank's rows while
// the others' are on their way. For a GEMM that has all rows at hand this joins them: the valid entries of all blocks of an
// expert end to end, in the order of the blocks, padded to whole blocks of `out_block` rows. It reads the blocks as they are
// when it runs, so whatever has been written to them since they were sorted is what the GEMM multiplies.
// Every workgroup counts the entries of all blocks (a wave per block, 32 loads per lane in flight) and so knows every expert's
// place; blocks and experts are then shared out among the waves of the grid. The first batch, the experts, the padded total
// and the ids of the first block that a wave will place are all on their way before anything is waited for.
// What bounds it: the launch, one trip to memory, four barriers. 64 blocks 4.5 us a launch with 4 waves to a workgroup (6.4 with
// 16), 160 blocks 6.4 and 512 blocks 8.7 with 16 (7.2 and 14.6 with 4): 4 waves up to kJoinFewBlocks, 16 beyond. (In a graph,
// where a launch that does nothing takes 2.1 us; since then 79 blocks 4.0, 191 5.6, 636 7.4, and with tails 4.5, 6.2, 7.7.)
constexpr int kJoinFewBlocks = 96, kJoinMaxBlock = 512, kJoinCountBits = 10;
constexpr int64_t kJoinLdsLimit = 160 * 1024 - 256;
struct JoinParams {
  const int32_t *sorted_ids, *expert_ids, *post_pad;
  int num_blocks, block_size, num_valid, E, out_block, out_rows;
  int32_t *out_ids, *out_experts, *out_segments, *out_padded;
  int out_shift;   // out_block = 1 << out_shift, or negative: no power of two
  // tail_most != 0: an expert's last rows, where they are at most that many, go into blocks of tail_block rows of a list of their own instead
  // of a block of `out_block` that they would fill in part (both powers of two). Done where it takes a round away from a GEMM of `cols`
  // tiles to a block on `cus` compute units and the list has room for all of them; else it is empty. tail_padded (or NULL) is set either way.
  int tail_most, tail_block, cols, cus, tail_rows;
  int32_t *tail_ids, *tail_experts, *tail_segments, *tail_padded;
};
// Workgroup `block` of `blocks`. kChunks: 64 rows each to a block; 0: any number.
template <int kThreads, int kChunks>
__device__ __forceinline__ void join_blocks(const JoinParams& p, int block, int blocks) {
  const int32_t* __restrict__ const sorted_ids = p.sorted_ids;
  const int32_t* __restrict__ const expert_ids = p.expert_ids;
  int32_t* __restrict__ const out_ids = p.out_ids;
  const int num_blocks = p.num_blocks, block_size = p.block_size, num_valid = p.num_valid, E = p.E, out_block = p.out_block,
            out_rows = p.out_rows;
  constexpr int kWaves = kThreads / 64, kCountMask = (1 << kJoinCountBits) - 1, kMine = kChunks > 0 ? kChunks : 1,
                kBatch = 32 / kMine;   // blocks of a wave in flight
  extern __shared__ int32_t s_mem[];
  int32_t* const s_total = s_mem;           // [E] entries per expert
  int32_t* const s_start = s_mem + E;       // [E] its first row
  int32_t* const s_block = s_mem + 2 * E;   // [num_blocks] expert and number of entries of each block
  int32_t* const s_tail = s_block + num_blocks;   // [E] with tails: the first row of the expert's last rows
  __shared__ int32_t s_part[3][kWaves];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int chunks = kChunks > 0 ? kChunks : (block_size + 63) / 64;
  const int gwave = block * kWaves + wave, waves = blocks * kWaves;
  auto valid = [&](int id) { return (uint32_t)id < (uint32_t)num_valid; };
  // (a block beyond the last of `limit` reads that one again, so that no load depends on a branch; nobody looks at its count)
  auto load = [&](int b, int c, int limit) {
    const int r = c * 64 + lane;
    const int id = sorted_ids[(int64_t)min(b, limit - 1) * block_size + (kChunks > 0 ? r : min(r, block_size - 1))];
    return kChunks > 0 || r < block_size ? id : -1;
  };
  const int total_rows = p.post_pad[0];
  int ids[kBatch][kMine], mine[kMine], expert0 = threadIdx.x < num_blocks ? expert_ids[threadIdx.x] : 0;
  auto load_batch = [&](int b0, int c0, int limit) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
#pragma unroll
      for (int c = 0; c < kMine; ++c) ids[u][c] = load(b0 + u * kWaves, c0 + c, limit);
  };
  load_batch(wave, 0, num_blocks);
#pragma unroll
  for (int c = 0; c < kMine; ++c) mine[c] = load(gwave, c, num_blocks);
  for (int e = threadIdx.x; e < E; e += kThreads) s_total[e] = 0;
  const int used = __builtin_amdgcn_readfirstlane(max(min(total_rows / block_size, num_blocks), 0));
  for (int b = threadIdx.x; b < used; b += kThreads) {
    s_block[b] = min(max(expert0, 0), E - 1) << kJoinCountBits;
    expert0 = b + kThreads < used ? expert_ids[b + kThreads] : 0;
  }
  __syncthreads();
  for (int b0 = wave; b0 < used; b0 += kWaves * kBatch) {
    int n = 0;   // lane u's block is b0 + u * kWaves
    for (int c0 = 0; c0 < chunks; c0 += kMine) {
      if (b0 != wave || c0 != 0) load_batch(b0, c0, used);
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        int count = 0;
#pragma unroll
        for (int c = 0; c < kMine; ++c) count += __popcll(__ballot(valid(ids[u][c])));
        n = lane == u ? n + count : n;
      }
    }
    const int b = b0 + lane * kWaves;
    if (lane < kBatch && b < used) {
      const int e = s_block[b] >> kJoinCountBits;
      s_block[b] = e << kJoinCountBits | n;
      atomicAdd(&s_total[e], n);
    }
  }
  __syncthreads();
  // exclusive prefix of the experts' padded sizes: a thread takes `per` neighbours
  const int per = (E + kThreads - 1) / kThreads;
  const int shift = p.out_shift;   // (a division by a number that is not known is twenty instructions in a row: 0.2 to 0.4 us of a join)
  auto blocks_of = [&](int n) { return shift >= 0 ? n >> shift : n / out_block; };
  auto padded = [&](int n) { return blocks_of(n + out_block - 1) * out_block; };
  auto tail_padded = [&](int n) { return (n + p.tail_block - 1) & -p.tail_block; };
  bool tails = p.tail_most > 0;
  auto tail_of = [&](int total) {   // (rows of an expert in the list of tails)
    const int rest = total & (out_block - 1);
    return tails && rest <= p.tail_most ? rest : 0;
  };
  int own = 0, own_whole = 0, own_tail = 0;
  for (int i = 0; i < per; ++i) {
    const int e = threadIdx.x * per + i;
    if (e < E) {
      const int total = s_total[e];
      own += padded(total);
      if (tails) own_whole += padded(total - tail_of(total)), own_tail += tail_padded(tail_of(total));
    }
  }
  const int sum = wave_scan_add(own);
  if (lane == 63) s_part[0][wave] = sum;
  int sum_whole = 0, sum_tail = 0;
  if (tails) {
    sum_whole = wave_scan_add(own_whole);
    sum_tail = wave_scan_add(own_tail);
    if (lane == 63) s_part[1][wave] = sum_whole, s_part[2][wave] = sum_tail;
  }
  __syncthreads();
  // What the waves before this one have, and all of them. (16 waves: by a scan; three rows of 16 sums read one by one were most of
  // what tails cost a join: 191 blocks 7.3 -> 6.6 us, without tails 6.1 -> 5.8. Four waves' sums are read as fast.)
  auto over_waves = [&](const int32_t* part, int& before, int& all) {
    if constexpr (kWaves > 4) {
      const int v = lane < kWaves ? part[lane] : 0, upto = wave_scan_add(v);
      before = __builtin_amdgcn_readlane(upto, wave) - __builtin_amdgcn_readlane(v, wave);
      all = __builtin_amdgcn_readlane(upto, 63);
    } else {
      before = all = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        before += w < wave ? part[w] : 0;
        all += part[w];
      }
    }
  };
  int before_own, all, at_tail = 0, all_tail = 0;
  over_waves(s_part[0], before_own, all);
  int at = before_own + sum - own;
  if (tails) {
    int before_whole, before_tail, all_whole;
    over_waves(s_part[1], before_whole, all_whole);
    over_waves(s_part[2], before_tail, all_tail);
    const int at_whole = before_whole + sum_whole - own_whole;
    at_tail = before_tail + sum_tail - own_tail;
    // (fewer rounds: the tiles that are left fill at most the whole rounds before the last one of all)
    const uint32_t cus = p.cus, tiles = (uint32_t)blocks_of(all) * p.cols, left = (uint32_t)blocks_of(all_whole) * p.cols;
    tails = all_tail <= p.tail_rows && tiles > 0 && left <= (tiles - 1) / cus * cus;
    if (tails) at = at_whole, all = all_whole;
  }
  if (p.tail_padded && block == 0 && threadIdx.x == 0) p.tail_padded[0] = tails ? all_tail : 0;
  for (int i = 0; i < per; ++i) {
    const int e = threadIdx.x * per + i;
    if (e < E) {
      const int total = s_total[e], tail = tail_of(total);
      s_start[e] = at;
      at += padded(total - tail);
      if (tails) {
        s_tail[e] = at_tail;
        at_tail += tail_padded(tail);
      }
    }
  }
  if (block == 0 && threadIdx.x == 0) p.out_padded[0] = min(all, blocks_of(out_rows) * out_block);
  __syncthreads();
  for (int b = gwave; b < used; b += waves) {
    const int e = s_block[b] >> kJoinCountBits;
    int before = 0;   // entries of the expert's earlier blocks
    for (int i = lane; i < b; i += 64) {
      const int v = s_block[i];
      before += v >> kJoinCountBits == e ? v & kCountMask : 0;
    }
    before = wave_sum(before);
    const int start = s_start[e], total = s_total[e], whole = total - tail_of(total), tail_start = tails ? s_tail[e] : 0;
    int row = before;   // of the expert's
    auto place = [&](int id) {
      const unsigned long long is = __ballot(valid(id));
      const int of = row + __popcll(is & ((1ull << lane) - 1));
      if (valid(id)) {
        if (of < whole) {
          if (start + of < out_rows) out_ids[start + of] = id;
        } else if (tails) {
          p.tail_ids[tail_start + of - whole] = id;   // (all of them fit, or there are no tails)
        }
      }
      row += __popcll(is);
    };
    if (kChunks > 0 && b == gwave) {
#pragma unroll
      for (int c = 0; c < kMine; ++c) place(mine[c]);
    } else {
      for (int c = 0; c < chunks; ++c) place(load(b, c, used));
    }
  }
  for (int e = gwave; e < E; e += waves) {
    const int all_rows = s_total[e], tail = tail_of(all_rows), total = all_rows - tail, lo = s_start[e], hi = min(lo + padded(total), out_rows);
    if (tail > 0) {
      const int first = s_tail[e], end = first + tail_padded(tail);
      for (int r = first + tail + lane; r < end; r += 64) p.tail_ids[r] = num_valid;
      for (int b = first / p.tail_block + lane; b < end / p.tail_block; b += 64) {
        p.tail_experts[b] = e;
        p.tail_segments[b] = 0;
      }
    }
    for (int r = lo + total + lane; r < hi; r += 64) out_ids[r] = num_valid;
    for (int b = blocks_of(lo) + lane; b < blocks_of(hi); b += 64) {
      p.out_experts[b] = e;
      p.out_segments[b] = 0;
    }
  }
}

template <int kThreads, int kChunks>
__global__ __launch_bounds__(kThreads) void moe_join_blocks_kernel(const JoinParams p) {
  join_blocks<kThreads, kChunks>(p, blockIdx.x, gridDim.x);
}

// The same beside the gather of the rows that the GEMM behind will read: the first `join_grid` workgroups join, and are done before
// the rows are there (8 x 1024 rows by 4096: 26 us for both, 23 + 8 us as two launches).
template <int kThreads, int kChunks>
__global__ __launch_bounds__(kThreads) void moe_gather_and_join_kernel(const GatherParams g, const JoinParams p, int join_grid, int per_rank) {
  const int block = blockIdx.x;
  if (block < join_grid) {
    if (g.status != nullptr && block == 0 && threadIdx.x == 0) retire_status(g.status, g.first_error);
    join_blocks<kThreads, kChunks>(p, block, join_grid);
  } else {
    const int r = (block - join_grid) / per_rank;
    gather_rows<kThreads>(g, r, block - join_grid - r * per_rank, per_rank);
  }
}

}  // namespace tdist

using namespace tdist;

extern "C" {

int tdist_moe_scatter_index_static(const int32_t* ids, int64_t n_ids, int topk, int num_experts, int32_t* splits,
                                   int32_t* cumsum, int32_t* scatter_idx, int32_t* gather_idx, int32_t* topk_idx,
                                   void* stream) {
  const char* who = "tdist_moe_scatter_index_static";
  const int64_t need = tdist_moe_workspace_bytes(n_ids, num_experts);
  if (need <= 0) return fail(TDIST_ERR_INVALID, "%s: bad sizes", who);
  if (need > kMoeStaticScratchBytes)
    return fail(TDIST_ERR_UNSUPPORTED, "%s: %lld ids over %d experts need %lld bytes of scratch, the built-in buffer holds "
                "%lld (use tdist_moe_scatter_index with a workspace)", who, (long long)n_ids, num_experts, (long long)need,
                (long long)kMoeStaticScratchBytes);
  void* ws = nullptr;
  if (int rc = moe_static_scratch(&ws, who)) return rc;
  // (the control words are the array's first 256 bytes whatever the call's sizes; they are zero between calls: the
  // kernels leave them so, and the array starts out zero. The rest needs no clearing, every word is written before it
  // is read, so a call after a larger one is not disturbed by what that one left behind.)
  return moe_index_common(ids, n_ids, topk, num_experts, splits, cumsum, scatter_idx, gather_idx, topk_idx, ws, need,
                          (hipStream_t)stream, true, who);
}

int64_t tdist_moe_workspace_bytes(int64_t n_ids, int num_experts) {
  if (n_ids < 0 || num_experts <= 0) return 0;
  const int64_t num_blocks = ceil_div(n_ids > 0 ? n_ids : 1, kMoeItemsPerBlock);
  return 256 + (num_blocks + 1) * (int64_t)num_experts * 4;  // control words + block histograms + one splits row
}

int tdist_moe_splits_cumsum(const int32_t* ids, int64_t n_ids, int num_experts, int32_t* splits, int32_t* cumsum,
                            void* workspace, int64_t workspace_bytes, void* stream) {
  return moe_index_common(ids, n_ids, 1, num_experts, splits, cumsum, nullptr, nullptr, nullptr, workspace,
                          workspace_bytes, (hipStream_t)stream, false, "tdist_moe_splits_cumsum");
}

int tdist_moe_scatter_index(const int32_t* ids, int64_t n_ids, int topk, int num_experts, int32_t* splits,
                            int32_t* cumsum, int32_t* scatter_idx, int32_t* gather_idx, int32_t* topk_idx,
                            void* workspace, int64_t workspace_bytes, void* stream) {
  return moe_index_common(ids, n_ids, topk, num_experts, splits, cumsum, scatter_idx, gather_idx, topk_idx, workspace,
                          workspace_bytes, (hipStream_t)stream, true, "tdist_moe_scatter_index");
}

int tdist_moe_scatter_index64(const int64_t* ids, int64_t n_ids, int topk, int num_experts, int32_t* splits,
                            int32_t* cumsum, int32_t* scatter_idx, int32_t* gather_idx, int32_t* topk_idx,
                            void* workspace, int64_t workspace_bytes, void* stream) {
  return moe_index_common((const int32_t*)ids, n_ids, topk, num_experts, splits, cumsum, scatter_idx, gather_idx, topk_idx, workspace,
                          workspace_bytes, (hipStream_t)stream, true, "tdist_moe_scatter_index64", true);
}

int tdist_moe_dispatch(const void* rows, int64_t row_bytes, const float* scales, const int32_t* gather_idx,
                       const int32_t* cumsum, int64_t n_rows, int world_size, int experts_per_rank, int max_m,
                       void* slot_rows, float* slot_scales, int32_t* splits_out, void* stream) {
  if (!rows || !cumsum || !slot_rows) return fail(TDIST_ERR_INVALID, "tdist_moe_dispatch: null pointer");
  if ((scales != nullptr) != (slot_scales != nullptr))
    return fail(TDIST_ERR_INVALID, "tdist_moe_dispatch: scales and slot_scales must both be given or both NULL");
  if (row_bytes <= 0 || n_rows < 0 || world_size <= 0 || experts_per_rank <= 0 || max_m <= 0)
    return fail(TDIST_ERR_INVALID, "tdist_moe_dispatch: bad sizes");
  if (world_size > 8192) return fail(TDIST_ERR_UNSUPPORTED, "tdist_moe_dispatch: world_size > 8192");
  const int64_t blocks = ceil_div(n_rows > 0 ? n_rows : 1, kRowsPerBlock);
  if (blocks > 0x7fffffff) return fail(TDIST_ERR_UNSUPPORTED, "tdist_moe_dispatch: too many rows");
  const bool vec = (row_bytes % 16 == 0) && aligned16(rows) && aligned16(slot_rows);
  auto kern = vec ? moe_rows_kernel<true, false> : moe_rows_kernel<false, false>;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), (size_t)(world_size + 1) * 4, (hipStream_t)stream,
                     (const unsigned char*)rows, row_bytes, scales, gather_idx, cumsum, n_rows, world_size,
                     experts_per_rank, max_m, (unsigned char*)slot_rows, slot_scales, splits_out);
  return launch_status("tdist_moe_dispatch");
}

int tdist_moe_dispatch_tokens(const void* tokens, int64_t row_bytes, const float* token_scales,
                              const int32_t* scatter_idx, int topk, const int32_t* cumsum, int64_t n_tokens,
                              int world_size, int experts_per_rank, int max_m, void* slot_rows, float* slot_scales,
                              int32_t* splits_out, void* stream) {
  if (!tokens || !scatter_idx || !cumsum || !slot_rows)
    return fail(TDIST_ERR_INVALID, "tdist_moe_dispatch_tokens: null pointer");
  if ((token_scales != nullptr) != (slot_scales != nullptr))
    return fail(TDIST_ERR_INVALID, "tdist_moe_dispatch_tokens: token_scales and slot_scales go together");
  if (row_bytes <= 0 || n_tokens < 0 || world_size <= 0 || experts_per_rank <= 0 || max_m <= 0 || topk <= 0)
    return fail(TDIST_ERR_INVALID, "tdist_moe_dispatch_tokens: bad sizes");
  if (topk > 64) return fail(TDIST_ERR_UNSUPPORTED, "tdist_moe_dispatch_tokens: topk > 64");
  if (world_size > 8192 || (int64_t)world_size * max_m > 0x7fffffff)
    return fail(TDIST_ERR_UNSUPPORTED, "tdist_moe_dispatch_tokens: world_size * max_m too large");
  const int windows = (int)ceil_div(row_bytes, 8192);
  const int64_t units = (n_tokens > 0 ? n_tokens : 1) * windows;
  const int64_t blocks = ceil_div(units, 4);
  if (blocks > 0x7fffffff) return fail(TDIST_ERR_UNSUPPORTED, "tdist_moe_dispatch_tokens: too many tokens");
  const bool vec = (row_bytes % 16 == 0) && aligned16(tokens) && aligned16(slot_rows);
  auto kern = vec ? moe_dispatch_tokens_kernel<true> : moe_dispatch_tokens_kernel<false>;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     (const unsigned char*)tokens, row_bytes, token_scales, scatter_idx, topk, cumsum, n_tokens,
                     world_size, experts_per_rank, max_m, (unsigned char*)slot_rows, slot_scales, splits_out, windows);
  return launch_status("tdist_moe_dispatch_tokens");
}

// (+ a word per lane for what is not counted)
static int64_t from_ids_lds(int64_t G, int topk) { return (3 * G + ((G + 1 + 3) & ~3ll) + kFdWaves * topk + 8 + 64) * 4; }
// The sizes that the launch from ids takes.
static bool from_ids_takes(int64_t n_tokens, int topk, int64_t row_bytes, int64_t G) {
  const int64_t windows = ceil_div(row_bytes, 8192);
  return n_tokens * topk <= kFusedDispatchMaxIds && topk <= 64 && G <= kMoeMaxExperts && windows >= 1 && windows <= kFdWaves &&
         kFdWaves % windows == 0 && from_ids_lds(G, topk) <= 160 * 1024 - 256;
}

int tdist_moe_dispatch_from_ids_takes(int64_t n_tokens, int topk, int64_t row_bytes, int num_experts) {
  return from_ids_takes(n_tokens, topk, row_bytes, num_experts);
}

static int dispatch_tokens_from_ids(const void* tokens, int64_t row_bytes, const float* token_scales, const int32_t* ids,
                                    int ids_wide, int topk, int64_t n_tokens, int world_size, int experts_per_rank, int max_m,
                                    void* slot_rows, float* slot_scales, int32_t* splits_out, int32_t* splits, int32_t* cumsum,
                                    int32_t* scatter_idx, int32_t* gather_idx, void* stream, const char* who) {
  if (!tokens || !ids || !slot_rows || !cumsum || !scatter_idx || !gather_idx) return fail(TDIST_ERR_INVALID, "%s: null pointer", who);
  if ((token_scales != nullptr) != (slot_scales != nullptr))
    return fail(TDIST_ERR_INVALID, "%s: token_scales and slot_scales go together", who);
  if (row_bytes <= 0 || n_tokens < 0 || world_size <= 0 || experts_per_rank <= 0 || max_m <= 0 || topk <= 0)
    return fail(TDIST_ERR_INVALID, "%s: bad sizes", who);
  const int64_t G64 = (int64_t)world_size * experts_per_rank;
  if ((int64_t)world_size * max_m > 0x7fffffff) return fail(TDIST_ERR_UNSUPPORTED, "%s: world_size * max_m too large", who);
  if (!from_ids_takes(n_tokens, topk, row_bytes, G64))
    return fail(TDIST_ERR_UNSUPPORTED, "%s: more than %lld ids, 64 of them to a token or %d experts, or rows above %d bytes (or no power-of-two "
                "number of 8 KB windows): use tdist_moe_scatter_index + tdist_moe_dispatch_tokens", who, (long long)kFusedDispatchMaxIds,
                kMoeMaxExperts, kFdWaves * 8192);
  const int G = (int)G64;
  int windows = (int)ceil_div(row_bytes, 8192);
  const int64_t lds = from_ids_lds(G, topk);
  // Few tokens: smaller windows, as long as there are fewer workgroups than a quarter of the compute units (every
  // workgroup counts all ids, so more of them is not free) and a window holds a KB.
  int vecs = 8;
  const DeviceInfo& di = device_info();
  const int64_t cus = di.ok == 1 ? di.num_cus : 256;
  while (windows < kFdWaves && vecs > 1 && ceil_div(n_tokens * windows, kFdWaves) * 4 < cus) {
    windows *= 2;
    vecs = (int)ceil_div(row_bytes, (int64_t)windows * 1024);
  }
  // (expert / experts_per_rank by a multiplication: exact, both are at most kMoeMaxExperts; 0: the expert itself)
  const uint32_t er_magic = experts_per_rank == 1 ? 0u : (uint32_t)(((1ull << 32) + experts_per_rank - 1) / experts_per_rank);
  const int64_t units = (n_tokens > 0 ? n_tokens : 1) * windows;
  const int64_t blocks = ceil_div(units, kFdWaves);
  const bool vec = (row_bytes % 16 == 0) && aligned16(tokens) && aligned16(slot_rows);
  const bool few = vecs < 8;
  auto kern = !vec ? (ids_wide ? moe_dispatch_fused_kernel<false, true, true> : moe_dispatch_fused_kernel<false, true, false>)
            : few  ? (ids_wide ? moe_dispatch_fused_kernel<true, true, true> : moe_dispatch_fused_kernel<true, true, false>)
                   : (ids_wide ? moe_dispatch_fused_kernel<true, false, true> : moe_dispatch_fused_kernel<true, false, false>);
  static bool attr_set[6] = {false, false, false, false, false, false};
  const int which = (!vec ? 0 : few ? 2 : 4) + ids_wide;
  if (!attr_set[which]) {
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 256) != hipSuccess)
      return fail(TDIST_ERR_LAUNCH, "%s: cannot reserve LDS", who);
    attr_set[which] = true;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kFdThreads), (size_t)lds, (hipStream_t)stream,
                     (const unsigned char*)tokens, row_bytes, token_scales, ids, topk, n_tokens, G, id_bits(G), world_size,
                     experts_per_rank, er_magic, max_m, windows, vecs, (unsigned char*)slot_rows, slot_scales, splits_out, splits, cumsum,
                     scatter_idx, gather_idx);
  return launch_status(who);
}

int tdist_moe_dispatch_tokens_from_ids(const void* tokens, int64_t row_bytes, const float* token_scales,
                                       const int32_t* ids, int topk, int64_t n_tokens, int world_size,
                                       int experts_per_rank, int max_m, void* slot_rows, float* slot_scales,
                                       int32_t* splits_out, int32_t* splits, int32_t* cumsum, int32_t* scatter_idx,
                                       int32_t* gather_idx, void* stream) {
  return dispatch_tokens_from_ids(tokens, row_bytes, token_scales, ids, 0, topk, n_tokens, world_size, experts_per_rank, max_m,
                                  slot_rows, slot_scales, splits_out, splits, cumsum, scatter_idx, gather_idx, stream,
                                  "tdist_moe_dispatch_tokens_from_ids");
}

int tdist_moe_dispatch_tokens_from_ids64(const void* tokens, int64_t row_bytes, const float* token_scales,
                                         const int64_t* ids, int topk, int64_t n_tokens, int world_size,
                                         int experts_per_rank, int max_m, void* slot_rows, float* slot_scales,
                                         int32_t* splits_out, int32_t* splits, int32_t* cumsum, int32_t* scatter_idx,
                                         int32_t* gather_idx, void* stream) {
  return dispatch_tokens_from_ids(tokens, row_bytes, token_scales, (const int32_t*)ids, 1, topk, n_tokens, world_size,
                                  experts_per_rank, max_m, slot_rows, slot_scales, splits_out, splits, cumsum, scatter_idx,
                                  gather_idx, stream, "tdist_moe_dispatch_tokens_from_ids64");
}

int tdist_moe_post_process(const void* slot_rows, int64_t row_bytes, const float* slot_scales, const int32_t* splits,
                           int64_t n_rows, int world_size, int experts_per_rank, int max_m, void* out_rows,
                           float* out_scales, void* stream) {
  if (!slot_rows || !splits || (!out_rows && n_rows > 0))
    return fail(TDIST_ERR_INVALID, "tdist_moe_post_process: null pointer");
  if (row_bytes <= 0 || n_rows < 0 || world_size <= 0 || experts_per_rank <= 0 || max_m <= 0)
    return fail(TDIST_ERR_INVALID, "tdist_moe_post_process: bad sizes");
  if (world_size > 8192) return fail(TDIST_ERR_UNSUPPORTED, "tdist_moe_post_process: world_size > 8192");
  if (n_rows == 0) return TDIST_OK;
  const int64_t blocks = ceil_div(n_rows, kRowsPerBlock);
  if (blocks > 0x7fffffff) return fail(TDIST_ERR_UNSUPPORTED, "tdist_moe_post_process: too many rows");
  const bool vec = (row_bytes % 16 == 0) && aligned16(out_rows) && aligned16(slot_rows);
  auto kern = vec ? moe_rows_kernel<true, true> : moe_rows_kernel<false, true>;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), (size_t)(world_size + 1) * 4, (hipStream_t)stream,
                     (const unsigned char*)slot_rows, row_bytes, slot_scales, (const int32_t*)nullptr, splits, n_rows,
                     world_size, experts_per_rank, max_m, (unsigned char*)out_rows, out_scales, (int32_t*)nullptr);
  return launch_status("tdist_moe_post_process");
}

int tdist_moe_combine_reduce(const void* rows, const float* topk_w, int64_t n_tokens, int topk, int hidden, int rank, int world_size, void* partials,
                             void* sums, void* out, void* stream) {
  const char* who = "tdist_moe_combine_reduce";
  if (!rows || !topk_w || !partials || !sums || !out) return fail(TDIST_ERR_INVALID, "%s: null pointer", who);
  if (n_tokens < 0 || topk <= 0 || topk > kCombineMaxTopk || hidden <= 0)
    return fail(TDIST_ERR_INVALID, "%s: bad sizes (topk <= %d)", who, kCombineMaxTopk);
  if (world_size <= 0 || rank < 0 || rank >= world_size || n_tokens % world_size != 0)
    return fail(TDIST_ERR_INVALID, "%s: rank %d / world_size %d, %lld tokens", who, rank, world_size, (long long)n_tokens);
  if (hidden % 8 != 0 || !aligned16(rows) || !aligned16(partials) || !aligned16(sums) || !aligned16(out))
    return fail(TDIST_ERR_UNSUPPORTED, "%s: hidden must be a multiple of 8 and buffers 16-byte aligned", who);
  if (n_tokens == 0) return TDIST_OK;
  const int n_windows = (hidden / 8 + 63) / 64;
  const int64_t blocks = ceil_div(n_tokens * n_windows, kCombineWaves);
  if (n_tokens > 0x3fffffff || blocks > 0x7fffffff) return fail(TDIST_ERR_UNSUPPORTED, "%s: too many tokens", who);
  hipLaunchKernelGGL(moe_combine_reduce_kernel, dim3((unsigned)blocks), dim3(kCombineWaves * 64), 0, (hipStream_t)stream, (const unsigned char*)rows,
                     topk_w, (int)n_tokens, topk, hidden, n_windows, rank, world_size, (int)(n_tokens / world_size), (unsigned char*)partials,
                     (unsigned char*)sums, (unsigned char*)out);
  return launch_status(who);
}

int tdist_moe_combine(const void* slot_rows, int row_dtype, const float* slot_scales, const int32_t* scatter_idx,
                      const float* topk_w, const int32_t* cumsum, int64_t n_tokens, int topk, int hidden,
                      int world_size, int experts_per_rank, int max_m, int scale_group_size, void* out_bf16,
                      void* stream) {
  if (!slot_rows || !scatter_idx || !out_bf16) return fail(TDIST_ERR_INVALID, "tdist_moe_combine: null pointer");
  if (max_m > 0 && (!cumsum || world_size <= 0 || experts_per_rank <= 0))
    return fail(TDIST_ERR_INVALID, "tdist_moe_combine: slot layout needs cumsum, world_size, experts_per_rank");
  if (n_tokens < 0 || topk <= 0 || topk > kCombineMaxTopk || hidden <= 0)
    return fail(TDIST_ERR_INVALID, "tdist_moe_combine: bad sizes (topk <= %d)", kCombineMaxTopk);
  if (row_dtype != TDIST_F8E4M3 && row_dtype != TDIST_BF16)
    return fail(TDIST_ERR_UNSUPPORTED, "tdist_moe_combine: row dtype %d (e4m3 and bf16 only)", row_dtype);
  if (scale_group_size != 0 && (row_dtype != TDIST_F8E4M3 || scale_group_size < 16 || scale_group_size % 16 != 0 ||
                                hidden % scale_group_size != 0))
    return fail(TDIST_ERR_UNSUPPORTED, "tdist_moe_combine: grouped scales need e4m3 rows and a group size that is a "
                "multiple of 16 and divides hidden");
  const int elems = row_dtype == TDIST_F8E4M3 ? 16 : 8;
  if (hidden % elems != 0 || !aligned16(slot_rows) || !aligned16(out_bf16))
    return fail(TDIST_ERR_UNSUPPORTED, "tdist_moe_combine: hidden must be a multiple of %d and buffers 16-byte aligned", elems);
  if (n_tokens == 0) return TDIST_OK;
  if (n_tokens > 0x7fffffff) return fail(TDIST_ERR_UNSUPPORTED, "tdist_moe_combine: too many tokens");
  const int n_windows = (hidden / elems + 63) / 64;
  const int64_t waves = n_tokens * n_windows;
  const int64_t blocks = ceil_div(waves, kCombineWaves);
  if (blocks > 0x7fffffff) return fail(TDIST_ERR_UNSUPPORTED, "tdist_moe_combine: too many tokens");
  auto kern = row_dtype == TDIST_F8E4M3 ? moe_combine_kernel<true> : moe_combine_kernel<false>;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kCombineWaves * 64), 0, (hipStream_t)stream,
                     (const unsigned char*)slot_rows, slot_scales, scatter_idx, topk_w, cumsum, n_tokens, topk, hidden,
                     world_size, experts_per_rank, max_m, scale_group_size, n_windows, (unsigned short*)out_bf16);
  return launch_status("tdist_moe_combine");
}

int tdist_quant_e4m3_groups(const void* x_bf16, int64_t n_rows, int hidden, int group_size, void* q_out,
                            float* scales_out, void* stream) {
  if (!x_bf16 || !q_out || !scales_out) return fail(TDIST_ERR_INVALID, "tdist_quant_e4m3_groups: null pointer");
  if (n_rows < 0 || hidden <= 0) return fail(TDIST_ERR_INVALID, "tdist_quant_e4m3_groups: bad sizes");
  if (group_size != kQuantGroup || hidden % kQuantGroup != 0 || !aligned16(x_bf16) || !aligned16(q_out))
    return fail(TDIST_ERR_UNSUPPORTED, "tdist_quant_e4m3_groups: group size %d, hidden a multiple of it, 16-byte aligned buffers",
                kQuantGroup);
  if (n_rows == 0) return TDIST_OK;
  const int windows = (hidden + 1023) / 1024;
  const int64_t blocks = ceil_div(n_rows * windows, 4);
  if (blocks > 0x7fffffff) return fail(TDIST_ERR_UNSUPPORTED, "tdist_quant_e4m3_groups: too many rows");
  hipLaunchKernelGGL(quant_groups_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     (const unsigned short*)x_bf16, n_rows, hidden, windows, (unsigned char*)q_out, scales_out);
  return launch_status("tdist_quant_e4m3_groups");
}

int tdist_moe_dispatch_tokens_quant(const void* tokens_bf16, int hidden, int group_size, const int32_t* scatter_idx,
                                    int topk, const int32_t* cumsum, int64_t n_tokens, int world_size,
                                    int experts_per_rank, int max_m, void* slot_rows, float* slot_scales,
                                    int32_t* splits_out, void* stream) {
  const char* who = "tdist_moe_dispatch_tokens_quant";
  if (!tokens_bf16 || !scatter_idx || !cumsum || !slot_rows || !slot_scales) return fail(TDIST_ERR_INVALID, "%s: null pointer", who);
  if (n_tokens < 0 || hidden <= 0 || world_size <= 0 || experts_per_rank <= 0 || max_m <= 0 || topk <= 0)
    return fail(TDIST_ERR_INVALID, "%s: bad sizes", who);
  if (topk > 64) return fail(TDIST_ERR_UNSUPPORTED, "%s: topk > 64", who);
  if (group_size != kQuantGroup || hidden % kQuantGroup != 0 || !aligned16(tokens_bf16) || !aligned16(slot_rows))
    return fail(TDIST_ERR_UNSUPPORTED, "%s: group size %d, hidden a multiple of it, 16-byte aligned buffers", who, kQuantGroup);
  if (world_size > 8192 || (int64_t)world_size * max_m > 0x7fffffff)
    return fail(TDIST_ERR_UNSUPPORTED, "%s: world_size * max_m too large", who);
  const int windows = (hidden + 1023) / 1024;
  const int64_t blocks = ceil_div((n_tokens > 0 ? n_tokens : 1) * windows, 4);
  if (blocks > 0x7fffffff) return fail(TDIST_ERR_UNSUPPORTED, "%s: too many tokens", who);
  hipLaunchKernelGGL(moe_dispatch_quant_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     (const unsigned short*)tokens_bf16, hidden, scatter_idx, topk, cumsum, n_tokens, world_size,
                     experts_per_rank, max_m, (unsigned char*)slot_rows, slot_scales, splits_out, windows);
  return launch_status(who);
}

int64_t tdist_moe_align_workspace_bytes(int64_t n_total, int num_experts, int num_iterations) {
  if (n_total < 0 || num_experts <= 0 || num_iterations <= 0) return 0;
  const int64_t G = (int64_t)num_experts * num_iterations;
  if (G > kMoeMaxExperts) return 0;
  // the index build's own scratch; then keys, scatter index, gather index, group sizes and their prefix
  return (3 * n_total + 3 * (G + 1)) * 4 + tdist_moe_workspace_bytes(n_total, (int)G);
}

int tdist_moe_align_block_size(const void* topk_ids, int ids_int64, int64_t n_total, int num_experts,
                               int num_iterations, int64_t n_per_iteration, int block_size, int32_t* sorted_token_ids,
                               int64_t sorted_fill, int32_t* expert_ids, int32_t* block_barrier_ids,
                               int32_t* rank_block_num, int32_t* total_tokens_post_pad, void* workspace,
                               int64_t workspace_bytes, void* stream) {
  const char* who = "tdist_moe_align_block_size";
  if (!topk_ids || !sorted_token_ids || !expert_ids || !block_barrier_ids || !rank_block_num || !total_tokens_post_pad)
    return fail(TDIST_ERR_INVALID, "%s: null pointer", who);
  if (num_experts <= 0 || num_iterations <= 0 || block_size <= 0 || n_per_iteration < 0 ||
      n_total != n_per_iteration * num_iterations)
    return fail(TDIST_ERR_INVALID, "%s: bad sizes (n_total must be num_iterations * n_per_iteration)", who);
  const int64_t G = (int64_t)num_experts * num_iterations;
  if (G > kMoeMaxExperts)
    return fail(TDIST_ERR_UNSUPPORTED, "%s: num_experts * num_iterations = %lld > %d", who, (long long)G, kMoeMaxExperts);
  if (n_total + G * (int64_t)(block_size - 1) > 0x7fffffffll) return fail(TDIST_ERR_UNSUPPORTED, "%s: too many entries", who);
  if (sorted_fill < 0 || sorted_fill > 0x7fffffffll) return fail(TDIST_ERR_INVALID, "%s: sorted_fill %lld", who, (long long)sorted_fill);
  const int64_t need = tdist_moe_align_workspace_bytes(n_total, num_experts, num_iterations);
  if (!workspace || workspace_bytes < need)
    return fail(TDIST_ERR_WORKSPACE, "%s: workspace %lld B < %lld B", who, (long long)workspace_bytes, (long long)need);
  hipStream_t st = (hipStream_t)stream;
  // the index build's own scratch first, so that its control words are the workspace's first 256 bytes whatever the
  // sizes; then keys, scatter index, gather index, group sizes and two prefix rows
  void* index_ws = workspace;
  int32_t* keys = (int32_t*)((unsigned char*)workspace + tdist_moe_workspace_bytes(n_total, (int)G));
  int32_t* scatter = keys + n_total;
  int32_t* gather = scatter + n_total;
  int32_t* splits = gather + n_total;
  int32_t* cumsum = splits + (G + 1);
  const int64_t blocks = ceil_div(n_total > 0 ? n_total : 1, 256);
  // Few entries: one launch in which every block counts all of them (see moe_align_fused_kernel).
  {
    const int64_t n1 = n_total > 0 ? n_total : 1;
    const int form = ceil_div(n1, kFusedThreads) <= kRecountMaxBlocks ? 1 : ceil_div(n1, 2 * kFusedThreads) <= kRecountMaxBlocks ? 2 : 0;
    const int64_t per_iter = n_per_iteration > 0 ? n_per_iteration : 1;
    // (a vector of four entries may cross one segment boundary, not two; the segment of an entry by multiplication)
    const uint32_t seg_magic = per_iter >= 65536 ? 0u : (uint32_t)(((1ull << 32) + per_iter - 1) / per_iter);
    const uint32_t block_magic = block_size > 1 && block_size <= 32768 ? (uint32_t)(((1ull << 32) + block_size - 1) / block_size) : 0u;
    static_assert(20 * kMoeMaxExperts + 16 + 256 <= 160 * 1024 - 256, "any number of groups has room in the LDS");
    if (form != 0 && device_info().ok == 1 && aligned16(topk_ids) && (per_iter >= 4 || num_iterations == 1) &&
        debug_get(TDIST_DEBUG_MOE_INDEX_FORM) != 3) {
      auto kern = form == 1 ? (ids_int64 ? moe_align_fused_kernel<1, true> : moe_align_fused_kernel<1, false>)
                            : (ids_int64 ? moe_align_fused_kernel<2, true> : moe_align_fused_kernel<2, false>);
      static bool attr_set[4] = {false, false, false, false};
      const int which = (form - 1) * 2 + (ids_int64 ? 1 : 0);
      if (!attr_set[which]) {
        if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)align_lds_bytes(kMoeMaxExperts)) != hipSuccess)
          return fail(TDIST_ERR_LAUNCH, "%s: cannot reserve LDS for the align kernel", who);
        attr_set[which] = true;
      }
      const int64_t for_entries = ceil_div(n1, form == 1 ? kFusedThreads : 2 * kFusedThreads), cus = device_info().num_cus;
      const int64_t for_fill = ceil_div(sorted_fill, kAlignFillPerBlock) < cus ? ceil_div(sorted_fill, kAlignFillPerBlock) : cus;
      const int64_t nblk = for_entries > for_fill ? for_entries : for_fill;
      hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(kFusedThreads), (size_t)align_lds_bytes(G), st, topk_ids, n_total,
                         (int)per_iter, num_experts, num_iterations, id_bits((int)G), block_size, sorted_token_ids, sorted_fill,
                         expert_ids, block_barrier_ids, rank_block_num, total_tokens_post_pad, seg_magic, block_magic);
      return launch_status(who);
    }
  }
  // three launches: keys (and the pre-fill of the padding positions), the stable index on the keys, padding + placement
  const int64_t key_items = n_total > sorted_fill ? n_total : sorted_fill;
  if (key_items > 0)
    hipLaunchKernelGGL(moe_align_keys_kernel, dim3((unsigned)ceil_div(key_items, 256)), dim3(256), 0, st, topk_ids, ids_int64,
                       n_total, n_per_iteration > 0 ? n_per_iteration : 1, num_experts, keys, sorted_token_ids, sorted_fill);
  int rc = moe_index_common(keys, n_total, 1, (int)G, splits, cumsum, scatter, gather, nullptr, index_ws,
                            tdist_moe_workspace_bytes(n_total, (int)G), st, true, who);
  if (rc != TDIST_OK) return rc;
  hipLaunchKernelGGL(moe_align_place_kernel, dim3((unsigned)blocks), dim3(kPlaceThreads), (size_t)(G + 1) * 4, st, keys, scatter,
                     splits, cumsum, n_total, (int)G, num_experts, num_iterations, block_size, sorted_token_ids, expert_ids,
                     block_barrier_ids, rank_block_num, total_tokens_post_pad);
  return launch_status(who);
}

#define TDIST_JOIN_ARGS                                                                                                        \
  const int32_t *sorted_token_ids, const int32_t *expert_ids, const int32_t *num_tokens_post_padded, int num_blocks,           \
      int block_size, int num_valid_tokens, int num_experts, int out_block, int32_t *out_sorted_ids, int64_t out_rows,         \
      int32_t *out_expert_ids, int32_t *out_segment_ids, int32_t *out_post_padded
#define TDIST_JOIN_NAMES                                                                                                        \
  sorted_token_ids, expert_ids, num_tokens_post_padded, num_blocks, block_size, num_valid_tokens, num_experts, out_block,      \
      out_sorted_ids, out_rows, out_expert_ids, out_segment_ids, out_post_padded

// Checks the arguments of a join and fills `p`, the LDS it takes, its threads and workgroups.
struct JoinLaunch {
  JoinParams p;
  int64_t lds;
  int threads, grid;
};
static int join_launch(JoinLaunch& j, const char* who, TDIST_JOIN_ARGS) {
  if (!sorted_token_ids || !expert_ids || !num_tokens_post_padded || !out_sorted_ids || !out_expert_ids || !out_segment_ids ||
      !out_post_padded)
    return fail(TDIST_ERR_INVALID, "%s: null pointer", who);
  if (num_blocks <= 0 || block_size <= 0 || num_valid_tokens < 0 || num_experts <= 0 || out_block <= 0 || out_rows < out_block)
    return fail(TDIST_ERR_INVALID, "%s: sizes must be positive", who);
  j.lds = (2ll * num_experts + num_blocks) * 4;
  if (block_size > kJoinMaxBlock || num_experts > kMoeMaxExperts || j.lds > kJoinLdsLimit || out_rows > 0x7fffffffll)
    return fail(TDIST_ERR_UNSUPPORTED, "%s: %d blocks of %d rows, %d experts", who, num_blocks, block_size, num_experts);
  j.p = {sorted_token_ids, expert_ids, num_tokens_post_padded, num_blocks, block_size, num_valid_tokens, num_experts, out_block,
         (int)out_rows, out_sorted_ids, out_expert_ids, out_segment_ids, out_post_padded,
         (out_block & (out_block - 1)) == 0 ? __builtin_ctz(out_block) : -1, 0, 0, 0, 0, 0, nullptr, nullptr, nullptr, nullptr};
  j.threads = num_blocks <= kJoinFewBlocks ? 256 : 1024;
  const int64_t items = ceil_div(num_blocks > num_experts ? num_blocks : num_experts, j.threads / 64);
  j.grid = (int)(items < 32 ? items : 32);
  return TDIST_OK;
}

// The instance for the launch: the block sizes that the grouped GEMMs take, or any other.
#define TDIST_JOIN_PICK(NAME)                                                                                                 \
  const int which = (j.threads == 256 ? 0 : 3) + (block_size == 128 ? 0 : block_size == 256 ? 1 : 2);                         \
  auto kern = which == 0 ? NAME<256, 2> : which == 1 ? NAME<256, 4> : which == 2 ? NAME<256, 0>                               \
            : which == 3 ? NAME<1024, 2> : which == 4 ? NAME<1024, 4> : NAME<1024, 0>;                                        \
  static bool attr_set[6] = {false, false, false, false, false, false};                                                       \
  if (!attr_set[which]) {                                                                                                     \
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kJoinLdsLimit) != hipSuccess)  \
      return fail(TDIST_ERR_LAUNCH, "%s: cannot reserve LDS", who);                                                           \
    attr_set[which] = true;                                                                                                   \
  }

int tdist_moe_join_blocks(TDIST_JOIN_ARGS, void* stream) {
  const char* who = "tdist_moe_join_blocks";
  JoinLaunch j;
  if (int rc = join_launch(j, who, TDIST_JOIN_NAMES)) return rc;
  TDIST_JOIN_PICK(moe_join_blocks_kernel)
  hipLaunchKernelGGL(kern, dim3((unsigned)j.grid), dim3(j.threads), (size_t)j.lds, (hipStream_t)stream, j.p);
  return launch_status(who);
}

int tdist_moe_join_blocks_tails(TDIST_JOIN_ARGS, int tail_most, int tail_block, int columns, int32_t* tail_ids, int64_t tail_rows,
                                int32_t* tail_experts, int32_t* tail_segments, int32_t* tail_padded, void* stream) {
  const char* who = "tdist_moe_join_blocks_tails";
  JoinLaunch j;
  if (int rc = join_launch(j, who, TDIST_JOIN_NAMES)) return rc;
  if (!tail_ids || !tail_experts || !tail_segments || !tail_padded) return fail(TDIST_ERR_INVALID, "%s: null pointer", who);
  if (tail_most <= 0 || tail_most >= out_block || tail_block <= 0 || columns <= 0 || tail_rows < tail_block || tail_rows > 0x7fffffffll)
    return fail(TDIST_ERR_INVALID, "%s: tails of %d rows in blocks of %d, %d columns", who, tail_most, tail_block, columns);
  if ((out_block & (out_block - 1)) != 0 || (tail_block & (tail_block - 1)) != 0)
    return fail(TDIST_ERR_INVALID, "%s: blocks of %d and %d rows (powers of two)", who, out_block, tail_block);
  const DeviceInfo& di = device_info();
  if (di.ok != 1) return fail(TDIST_ERR_DEVICE, "%s: current device is not gfx950", who);
  j.p.tail_padded = tail_padded;
  // (no room for the tails' places, in the LDS or in 32 bits: the blocks are joined all the same, and no row goes into the second list)
  if (j.lds + 4ll * num_experts <= kJoinLdsLimit && out_rows / out_block * ceil_div(columns, 256) <= 0x7fffffff) {
    j.lds += 4ll * num_experts;
    j.p.tail_most = tail_most, j.p.tail_block = tail_block, j.p.cus = di.num_cus, j.p.tail_rows = (int)tail_rows;
    j.p.cols = (int)ceil_div(columns, 256);
    j.p.tail_ids = tail_ids, j.p.tail_experts = tail_experts, j.p.tail_segments = tail_segments;
  }
  TDIST_JOIN_PICK(moe_join_blocks_kernel)
  hipLaunchKernelGGL(kern, dim3((unsigned)j.grid), dim3(j.threads), (size_t)j.lds, (hipStream_t)stream, j.p);
  return launch_status(who);
}

int tdist_moe_gather_and_join(void* workspace, const void* const* shards, int world_size, int64_t rank_bytes, int32_t* status,
                              int32_t* first_error, TDIST_JOIN_ARGS, void* stream) {
  const char* who = "tdist_moe_gather_and_join";
  GatherParams g;
  if (int rc = gather_params(g, workspace, shards, world_size, rank_bytes, status, first_error, who)) return rc;
  JoinLaunch j;
  if (int rc = join_launch(j, who, TDIST_JOIN_NAMES)) return rc;
  TDIST_JOIN_PICK(moe_gather_and_join_kernel)
  // (four 16-byte loads per lane and turn; at most two million lanes)
  const int64_t wanted = ceil_div(rank_bytes, 16 * 4 * j.threads), most = 2048 * 1024 / j.threads / world_size;
  const int per_rank = (int)(wanted < most ? wanted : most);
  hipLaunchKernelGGL(kern, dim3((unsigned)(j.grid + per_rank * world_size)), dim3(j.threads), (size_t)j.lds, (hipStream_t)stream, g, j.p,
                     j.grid, per_rank);
  return launch_status(who);
}
#undef TDIST_JOIN_PICK
#undef TDIST_JOIN_ARGS
#undef TDIST_JOIN_NAMES

}  // extern "C"
