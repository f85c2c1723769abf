// (d) split-KV GQA flash decode and the LSE-weighted combine.
//
// Restates kernel_gqa_fwd_batch_decode_split_kv (kernels/nvidia/flash_decode.py:129-239) and the
// combine kernels (:392-449, :481-532) for CDNA4:
//
//  * one workgroup per (split, kv head [x block of 16 query heads], sequence); its NW waves each stream
//    an interleaved subset of the split's 16-key blocks and keep a private online-softmax state, merged
//    through LDS at the end, so the main loop has no workgroup barrier;
//  * K and V rows go HBM → LDS with asynchronous 16-byte-per-lane LDS-DMA loads into a per-wave ring of
//    NST stages (P = NST-1 stages in flight), so the only synchronisation is the wave's own vmcnt;
//    the page-table entries a stage needs travel the same way, two rounds ahead of the rows;
//  * scores:  S^T[key, head] = K[16 keys, D] . Q^T[D, 16 heads]   v_mfma_f32_16x16x32 (D/32 steps) per group
//    of 16 keys; the result layout (lane = head, 4 keys per lane) is exactly the B operand of
//    O^T[dv, head] += V^T[16 dv, keys] . P^T[keys, 16 heads]  (v_mfma 16x16x32 over two key groups, or
//    16x16x16 over one), so probabilities never leave registers; the V^T fragments come from the
//    row-major V rows in LDS with the transposing read ds_read_b64_tr_b16, one instruction per 4 keys;
//  * probabilities enter the PV product as a hi+lo pair of 16-bit values, which keeps the product at
//    fp32-level accuracy for the cost of a second (idle anyway) MFMA.
//
//  * heads whose key dimension is not a power of two (192 = 128 + 64, 576 = 512 + 64: flash_decode.py:771-772,
//    BLOCK_DPE) are handled as the reference does: the power-of-two part DM (= the value dimension) and the
//    extra DPE key dimensions are two row sets of the stage, each with its own DMA layout and swizzle;
//  * the fused entry point replaces the reference's persistent kernel (split-KV, grid barrier, combine:
//    flash_decode.py:586-760) by "the last workgroup to arrive merges": every workgroup publishes its partial
//    result, bumps a counter of its (sequence, head block), and the one that finds the counter at S-1 merges the S
//    partials. No workgroup ever waits for another, so nothing depends on the grid being co-resident.
//
// HBM traffic per launch: every K and V row of the split once (len * Hkv * (Dk + Dv) * 2 B per sequence).
#include <type_traits>

#include "common.h"

// Cache policy of the K/V stream: non-temporal (every byte is used once; the hint lets it pass through the
// caches without displacing anything and measurably raises the HBM streaming rate).
#ifndef TDIST_KV_AUX
#define TDIST_KV_AUX 2
#endif

namespace tdist {

struct DecodeParams {
  const unsigned char* q;
  const unsigned char* k;
  const unsigned char* v;
  float* out;  // [B,Hq,S,D]
  float* lse;  // [B,Hq,S]
  const int32_t* table;
  const int32_t* lens;
  float sm_scale;
  float soft_cap;
  int B, Hq, Hkv, S;
  int when_lens;        // 0: run; 1: run only if the sequence lengths are even (decode_lens_even), 2: only if not
  int splits_per_team;  // kWaveHeads: consecutive splits of a sequence that one workgroup streams through (>= 1)
  int d_valid;  // kernels compiled for a padded head dimension: the real one (a multiple of 8), else unused
  int page_size;
  // n / page_size for 0 <= n < 2^31 as (n * page_magic) >> page_shift with
  // page_shift = 31 + ceil(log2 page_size), page_magic = ceil(2^page_shift / page_size)  (exact, Granlund-Montgomery)
  int page_shift;
  uint64_t page_magic;
  // byte strides
  int64_t q_sb, q_sh;
  int64_t k_sp, k_st, k_sh;
  int64_t v_sp, v_st, v_sh;
  int64_t t_s;  // table stride in entries
  // fused merge (null counters = plain split-KV launch)
  int32_t* counters;         // one per (sequence, head block), zero on entry, left zero on exit
  unsigned char* final_out;  // [B,Hq,Dv] of final_dtype
  float* final_lse;          // [B,Hq] or null
  int final_dtype;
  int64_t fo_sb, fo_sh;      // element strides of final_out
  int fo_vec;                // its rows take 8-byte (16-bit types) / 16-byte (fp32) stores
  int part_vec;              // the partial results take 16-byte stores
  // streaming form: ranges the batch's blocks are cut into at most, the fewest blocks of a range, and (for the merge) the
  // width of a result's row
  int ranges, min_blocks, dv;
  const struct RankParams* ranks;   // (host) the other ranks' results to merge with behind the stream, or null
};

struct MmaBF16 {
  typedef bf16x8v frag8;
  typedef short4v frag4;
  __device__ static __forceinline__ float4v mma32(frag8 a, frag8 b, float4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ float4v mma16(frag4 a, frag4 b, float4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
  }
  // p → (hi, lo) 16-bit patterns with hi + lo ≈ p to ~16 mantissa bits
  __device__ static __forceinline__ void split(float p0, float p1, uint32_t& hi, uint32_t& lo) {
    hi = pack_bf16x2(p0, p1);
    lo = pack_bf16x2(p0 - BF16::lo(hi), p1 - BF16::hi(hi));
  }
};
struct MmaF16 {
  typedef f16x8v frag8;
  typedef f16x4v frag4;
  __device__ static __forceinline__ float4v mma32(frag8 a, frag8 b, float4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ float4v mma16(frag4 a, frag4 b, float4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ void split(float p0, float p1, uint32_t& hi, uint32_t& lo) {
    hi = pack_f16x2(p0, p1);
    lo = pack_f16x2(p0 - F16::lo(hi), p1 - F16::hi(hi));
  }
};

// kWaveHeads: splits one workgroup may stream through (the results of all but the last wait in registers: D / 4 each).
// `heavy`: the instances that already fill their registers (soft cap, fused merge, padded rows).
constexpr int decode_max_splits_per_team(int d, bool heavy) { return d <= 64 ? 4 : d <= 128 ? (heavy ? 3 : 4) : 2; }
// a head's row of a wave's result on its way through the LDS
constexpr int decode_acc_row(int d) { return d + 4; }
constexpr int kTableSlots = 8;  // ring of page-table rows per wave (>= 2P+2)

// what the DMA lanes of a padded head dimension read for the dimensions that do not exist
static __device__ __align__(16) const unsigned char kZeroChunk[16] = {0};

// KEYS = keys per block (16 or 32): one or two groups of 16 keys, a group being one MFMA tile of scores.
// DM = value dimension = power-of-two part of the key dimension; DPE = the extra key dimensions (0 or 64).
template <int DM, int DPE, int KEYS, int NST>
struct DecodeCfg {
  static constexpr int kGroups = KEYS / 16;
  static constexpr int kRowBytes = DM * 2;
  static constexpr int kLanesPerRow = kRowBytes / 16;       // 16-byte chunks per row
  static constexpr int kRowsPerInstr = 64 / kLanesPerRow;   // rows one wave-wide DMA covers
  static constexpr int kInstrPerTensor = KEYS / kRowsPerInstr;
  static constexpr int kTensorBytes = KEYS * kRowBytes;
  // the extra key dimensions: rows of DPE * 2 bytes behind the K and V rows of the stage
  static constexpr int kPeRowBytes = DPE * 2;
  static constexpr int kPeLanesPerRow = DPE > 0 ? kPeRowBytes / 16 : 1;
  static constexpr int kPeRowsPerInstr = 64 / kPeLanesPerRow;
  static constexpr int kPeInstr = DPE > 0 ? KEYS / kPeRowsPerInstr : 0;
  static constexpr int kPeBytes = KEYS * kPeRowBytes;
  static constexpr int kVBase = kTensorBytes;
  static constexpr int kPeBase = kVBase + kTensorBytes;
  static constexpr int kStageBytes = kPeBase + kPeBytes;
  static constexpr int kLoadsPerGroup = 1 + 2 * kInstrPerTensor + kPeInstr;  // table row + K + V (+ extra K)
  static constexpr int kP = NST - 1;
  // LDS position of 16-byte chunk c of a row: K rows c ^ kswz(key), V rows c ^ vswz(key).
  // K operand reads: 16 lanes = 16 keys, same chunk      → spread over 16 positions: key & 15.
  // V transposed reads: 32 lanes = 8 keys x 2 adjacent chunks → spread the chunk pairs: (key & 7) << 1.
  static constexpr int kSwzMask = (kLanesPerRow < 16 ? kLanesPerRow : 16) - 1;
  static constexpr int kPeSwzMask = kPeLanesPerRow - 1;
  static constexpr int kTableSlotBytes = KEYS * 4;
  static constexpr int kWaveBytes = NST * kStageBytes + kTableSlots * kTableSlotBytes;
  static_assert(KEYS == 16 || KEYS == 32, "one or two key groups");
  static_assert(kP >= 1 && kP <= 3, "1..3 stages in flight");
  // vmcnt is a 6-bit counter. When a new group is issued, up to kP older ones may still be in flight; where
  // kP + 1 groups do not fit the counter (the 576-dimension heads: 35 loads per group), the loop waits for the
  // block it is about to use BEFORE it issues the next one, so only one group is ever outstanding.
  static constexpr bool kWaitFirst = (kP + 1) * kLoadsPerGroup >= 64;
  static_assert(kLoadsPerGroup < 64 && (!kWaitFirst || kP == 1), "vmcnt is 6 bits");
  static_assert(2 * kP + 2 <= kTableSlots, "table ring too small");
  static_assert(DM % 32 == 0 && DM >= 64 && DM <= 512, "head dim");
  static_assert(DPE == 0 || DPE == 64, "extra key dimensions: none or 64");
  static_assert(DPE == 0 || KEYS % kPeRowsPerInstr == 0, "whole DMA instructions for the extra key rows");
  // Rows shorter than the 256-byte bank window already differ in their row offset: only every kRowsPerWindow-th
  // key needs a new XOR term.
  static constexpr int kRowsPerWindow = kRowBytes >= 256 ? 1 : 256 / kRowBytes;
  static constexpr int kPeRowsPerWindow = DPE > 0 ? 256 / kPeRowBytes : 1;
  __device__ static __forceinline__ int kswz(int key) {
    return (key / kRowsPerWindow) & kSwzMask;
  }
  __device__ static __forceinline__ int vswz(int key) {
    return (((key / kRowsPerWindow) & 7) << 1) & kSwzMask;
  }
  __device__ static __forceinline__ int peswz(int key) { return (key / kPeRowsPerWindow) & kPeSwzMask; }
};

template <int N>
__device__ __forceinline__ void wait_groups(int rem) {
  // rem in [0, P]: number of younger load groups allowed to stay in flight
  if (rem >= 3) wait_vmcnt<(3 * N < 64 ? 3 * N : 63)>();
  else if (rem == 2) wait_vmcnt<(2 * N < 64 ? 2 * N : 63)>();
  else if (rem == 1) wait_vmcnt<N>();
  else wait_vmcnt<0>();
}

// One workgroup's split: streams its keys and writes the partial result and LSE of its 16 heads.
// Partial results that another workgroup of the same launch will read (fused merge) are written through to where
// every XCD sees them (agent-scope store: the L2 caches of the 8 XCDs are not coherent with each other); with that,
// publishing them needs no cache write-back, only the wait for the stores themselves.
template <bool kCoherent>
__device__ __forceinline__ void store_partial(float* p, float v) {
  if constexpr (kCoherent) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}
// Four consecutive floats (16-byte aligned) the same way: one 16-byte vector store, written through at agent scope
// (the sc1 bit, which is what the 4-byte atomic store above carries) where the merge reads them in the same launch.
// A store of more than 8 bytes reads its data registers one cycle after it issues: the s_nop keeps the next
// instruction, which the compiler may let write those registers, out of that cycle (for its own stores the compiler
// does this itself; it does not look into the asm).
template <bool kCoherent>
__device__ __forceinline__ void store_partial4(float* p, float4v v) {
  if constexpr (kCoherent) asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 0" ::"v"(p), "v"(v) : "memory");
  else *(float4v*)p = v;
}

__device__ __forceinline__ float load_elem(const unsigned char* base, int64_t idx, int dtype) {
  if (dtype == TDIST_F32) return ((const float*)base)[idx];
  const uint32_t bits = ((const unsigned short*)base)[idx];
  return dtype == TDIST_BF16 ? bf16_bits_to_f32(bits) : f16_bits_to_f32(bits);
}
__device__ __forceinline__ void store_elem(unsigned char* base, int64_t idx, int dtype, float v) {
  if (dtype == TDIST_F32) ((float*)base)[idx] = v;
  else if (dtype == TDIST_BF16) ((unsigned short*)base)[idx] = (unsigned short)f32_to_bf16_bits(v);
  else ((unsigned short*)base)[idx] = (unsigned short)(pack_f16x2(v, 0.f) & 0xffffu);
}
// Four consecutive elements; `vec`: their address takes one store.
__device__ __forceinline__ void store_elem4(unsigned char* base, int64_t idx, int dtype, int vec, float4v v) {
  if (!vec) {
#pragma unroll
    for (int e = 0; e < 4; ++e) store_elem(base, idx + e, dtype, v[e]);
  } else if (dtype == TDIST_F32) {
    *(float4v*)(base + idx * 4) = v;
  } else {
    const int2v w = dtype == TDIST_BF16 ? int2v{(int)pack_bf16x2(v[0], v[1]), (int)pack_bf16x2(v[2], v[3])}
                                        : int2v{(int)pack_f16x2(v[0], v[1]), (int)pack_f16x2(v[2], v[3])};
    *(int2v*)(base + idx * 2) = w;
  }
}

// Workgroup i of n runs on XCD i % 8: its place when the workgroups are counted XCD by XCD.
__device__ __forceinline__ int xcd_major(int i, int n) {
  const int x = i & 7, q = n >> 3, rest = n & 7;
  return x * q + min(x, rest) + (i >> 3);
}

// ---- streaming form: how a partial result lies in the workspace ---------------------------------------------
// A slot holds Hq x dv floats, one block of up to 16 query heads of a kv head after the other, and a block by tiles of 16 columns:
// tile, head, column. That is the order in which the 64 lanes of a wave hold an MFMA tile of the result (lane: head x = lane % 16,
// four columns g = lane / 16), so that a store of the wave is one run of nvalid x 64 bytes; rows of dv floats were 16 runs of 64
// bytes a store. Where dv is no multiple of 16 the last tile is narrower.
// The stores go through to memory as they are made (store_partial4<true>): what a launch leaves dirty in the L2 caches is written
// back before the next one may begin. Rows, written back at the end, against tiles, written through, whole calls: latent heads,
// 16 sequences up to 4096 keys 26.5 -> 24.7 us,
// 1 x 1000 15.2 -> 13.9; 64 / 8 heads of 128, 64 x 256 keys 19.4 -> 18.6, 48 up to 8192 67.2 -> 66.6. The stores written through alone: 25.6
// and 14.5; non-temporal 26.9 (the merge then finds less in the memory-side cache).
__device__ __forceinline__ int64_t partial_tile(int nvalid, int dv, int tile, int x, int g) {
  return tile * 16 * nvalid + x * min(16, dv - tile * 16) + 4 * g;
}
// The head and the column of 16-byte piece `vec` of a slot.
__device__ __forceinline__ void partial_piece(uint32_t vec, uint32_t group, uint32_t dv, int& head, int& col) {
  const uint32_t kv_vecs = group * dv / 4, kvh = vec / kv_vecs, in_kv = vec - kvh * kv_vecs;
  const uint32_t block = in_kv / (4 * dv), in_block = in_kv - block * 4 * dv, nvalid = min(16u, group - block * 16);
  const uint32_t whole = dv / 16, tile = min(in_block / (4 * nvalid), whole), in_tile = in_block - tile * 4 * nvalid;
  const uint32_t vecs = tile < whole ? 4 : dv % 16 / 4, x = tile < whole ? in_tile / 4 : in_tile / max(vecs, 1u);
  head = (int)(kvh * group + block * 16 + x);
  col = (int)(tile * 16 + (in_tile - x * vecs) * 4);
}

// ---- streaming form: which blocks a range holds -----------------------------------------------------------
struct StreamRange {
  int n;            // blocks in the range (0: the batch has fewer ranges)
  int seq, block;   // the sequence its first block belongs to, and that block's number in the sequence
  int first_block;  // that sequence's first block, numbered over the whole batch
  int per;          // blocks per range
};

// Blocks per range, from the batch's blocks: even shares, but no shorter than min_blocks.
__device__ __forceinline__ int stream_blocks_per_range(const DecodeParams& prm, int total) {
  return max((total + prm.ranges - 1) / prm.ranges, prm.min_blocks);
}

// All sequences' blocks laid end to end and cut into ranges of `per` blocks: the same answer in every wave, from one
// load per 64 sequences and a scan over the lanes.
template <int KEYS>
__device__ __forceinline__ StreamRange stream_range(const DecodeParams& prm, int range) {
  const int lane = threadIdx.x & 63;
  auto blocks = [&](int i) { return i < prm.B ? (max(prm.lens[i], 0) + KEYS - 1) / KEYS : 0; };
  int nb = 0, sum = 0, total = 0;
  auto scan = [&](int i0) {   // sum: this lane's sequence and the ones before it within the 64
    nb = blocks(i0 + lane);
    sum = wave_scan_add(nb);
  };
  for (int i0 = 0; i0 < prm.B; i0 += 64) {
    scan(i0);
    total += __builtin_amdgcn_readlane(sum, 63);
  }
  StreamRange r;
  r.per = stream_blocks_per_range(prm, total);
  const long long g0 = (long long)range * r.per;
  r.seq = r.block = r.first_block = 0;
  if (g0 >= total) {
    r.n = 0;
    return r;
  }
  r.n = min(r.per, total - (int)g0);
  int base = 0;
  for (int i0 = 0;; i0 += 64) {
    if (prm.B > 64) scan(i0);
    const unsigned long long past = __ballot(base + sum > (int)g0);
    if (past) {
      const int at = __builtin_ctzll(past);
      r.seq = i0 + at;
      r.first_block = base + __builtin_amdgcn_readlane(sum, at) - __builtin_amdgcn_readlane(nb, at);
      r.block = (int)g0 - r.first_block;
      return r;
    }
    base += __builtin_amdgcn_readlane(sum, 63);
  }
}

// One sequence: its first block, numbered over the whole batch, and the blocks per range. The loads of all lengths are
// independent of each other.
template <int KEYS>
__device__ __forceinline__ void stream_sequence(const DecodeParams& prm, int seq, int& first_block, int& per) {
  const int lane = threadIdx.x & 63;
  int total = 0, before = 0;
  for (int i = lane; i < prm.B; i += 64) {
    const int nb = (max(prm.lens[i], 0) + KEYS - 1) / KEYS;
    total += nb;
    before += i < seq ? nb : 0;
  }
  first_block = wave_sum(before);
  per = stream_blocks_per_range(prm, wave_sum(total));
}

// Are the B sequence lengths even enough for the form that hands a workgroup 8 kv heads of one (sequence, split)?
// Its time goes with the longest sequence, the other form's (eight times as many, smaller workgroups) with the
// sum: even means mean >= 0.8 max (measured: the one form is 7-11 % faster from mean = 0.9 max on, the other 11 % at
// 0.57 and 6 x with one long sequence among short ones). Every wave computes the same answer from the same loads, so
// two launches, one of each form, can each ask and exactly one of them does the work.
__device__ __forceinline__ bool decode_lens_even(const int32_t* lens, int B) {
  const int lane = threadIdx.x & 63;
  long long sum = 0;
  int mx = 0;
  // sixteen loads in flight per lane: one round trip for up to 1024 sequences
  for (int i0 = 0; i0 < B; i0 += 64 * 16) {
    int l[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int i = i0 + u * 64 + lane;
      l[u] = i < B ? lens[i] : 0;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      sum += max(l[u], 0);
      mx = max(mx, l[u]);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned int lo = __shfl_xor((unsigned int)sum, o), hi = __shfl_xor((unsigned int)(sum >> 32), o);
    sum += (long long)(((unsigned long long)hi << 32) | lo);
    mx = max(mx, __shfl_xor(mx, o));
  }
  return sum * 5 >= (long long)mx * B * 4;
}

// kPadded: the head dimension is prm.d_valid <= D (key and value alike, a multiple of 8): the rows in the LDS are D
// wide, the 16-byte pieces beyond the real row are fetched from a page of zeros (so that the MFMA blocks see exact
// zeros there: the reference masks the same dimensions, kernels/nvidia/flash_decode.py:771-772 with BLOCK_DPE), and
// results are stored d_valid wide.
// kWaveHeads: the NW waves of a workgroup take NW neighbouring kv heads (one each, all keys of the split) instead of
// sharing one kv head's keys: together they read whole stretches of the token rows (NW * 2 * D bytes of every row) at
// the same time, and no wave waits for another: each writes its own heads' results. For at most 16 query heads per kv
// head and a number of kv heads that is a multiple of NW.
// kStream: see decode_stream_kernel; a wave's kv head and its blocks come from its place in the grid.
template <typename MMA, int D, int DPE, int KEYS, int NW, int NST, bool kSoftCap, bool kFuse, bool kPadded, bool kWaveHeads,
          bool kStream = false>
__device__ __forceinline__ void decode_split_body(const DecodeParams& prm) {
  constexpr int DT = D / 16;  // tiles of 16 value dimensions
  typedef DecodeCfg<D, DPE, KEYS, NST> C;
  constexpr int G = C::kGroups;
  constexpr int DK = D + DPE;  // key (and query) dimensions; D is the value dimension
  static_assert(!kPadded || DPE == 0, "padded rows have no extra key dimensions");
  const int Dout = kPadded ? prm.d_valid : D;          // width of the stored results
  const int valid_chunks = kPadded ? prm.d_valid >> 3 : D / 8;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  // kv heads vary fastest over the grid: workgroups that run together then read the neighbouring 2*D-byte
  // pieces of the same token rows
  const int group = prm.Hq / prm.Hkv;
  const int head_blocks = (group + 15) >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform for the compiler too
  const int lane = threadIdx.x & 63;
  // kStream: heads vary fastest over the grid's waves, then the range of blocks
  const int unit = blockIdx.x * NW + wave;
  const int range = kStream ? unit / (prm.Hkv * head_blocks) : 0;
  const int head_unit = kStream ? unit - range * prm.Hkv * head_blocks : blockIdx.x;
  const int kvh = kWaveHeads ? blockIdx.x * NW + wave : head_unit / head_blocks;
  const int hb = kWaveHeads ? 0 : head_unit - kvh * head_blocks;
  int b = blockIdx.z;
  const int h0 = kvh * group + hb * 16;
  const int nvalid = min(16, group - hb * 16);
  // threads that share the work of one (kv head, head block): the workgroup, or the wave
  const int team_tid = kWaveHeads || kStream ? lane : (int)threadIdx.x;
  constexpr int kTeam = kWaveHeads || kStream ? 64 : NW * 64;
  const int g = lane >> 4;   // lane group 0..3
  const int x = lane & 15;   // head (score column) / dv within tile (V^T row) / key (K row)

  StreamRange sr{};
  if constexpr (kStream) {
    sr = stream_range<KEYS>(prm, range);
    for (int i0 = 0; range == 0 && i0 < prm.B; i0 += 64) {
      // sequences without keys: out = 0, lse = -inf
      unsigned long long none = __ballot(i0 + lane < prm.B && prm.lens[min(i0 + lane, prm.B - 1)] <= 0);
      for (; none; none &= none - 1) {
        const int seq = i0 + __builtin_ctzll(none);
        for (int j = team_tid; j < nvalid * Dout; j += kTeam) {
          const int h = j / Dout;
          store_elem(prm.final_out, (int64_t)seq * prm.fo_sb + (int64_t)(h0 + h) * prm.fo_sh + (j - h * Dout), prm.final_dtype, 0.f);
        }
        if (prm.final_lse && team_tid < nvalid) prm.final_lse[(int64_t)seq * prm.Hq + h0 + team_tid] = -INFINITY;
      }
    }
    if (sr.n == 0) return;
  }

  // (the lengths through the scalar cache: a vector load would wait for the stream behind which it is queued)
  const auto lens = (const __attribute__((address_space(4))) int32_t*)(uintptr_t)prm.lens;
  const int len = kStream ? 0 : prm.lens[b];
  const int per = (len + prm.S - 1) / prm.S;
  // kWaveHeads: the team streams through splits split .. split + n_splits - 1 of its sequence, one after the other
  const int split = kWaveHeads ? blockIdx.y * prm.splits_per_team : blockIdx.y;
  const int n_splits = kWaveHeads ? min(prm.splits_per_team, prm.S - split) : 1;
  int start = per * split;
  int end = min(start + per, len);

  float* out_base = prm.out + (((int64_t)b * prm.Hq + h0) * prm.S + split) * Dout;
  float* lse_base = prm.lse + ((int64_t)b * prm.Hq + h0) * prm.S + split;
  if (!kStream && end <= start) {
    // empty split (and with it every later one): zeros and LSE = -inf so that any merge gives it weight 0
    for (int sp = 0; sp < n_splits; ++sp) {
      for (int i = team_tid; i < nvalid * Dout; i += kTeam) {
        const int h = i / Dout, d = i - h * Dout;
        store_partial<kFuse>(out_base + ((int64_t)h * prm.S + sp) * Dout + d, 0.f);
      }
      if (team_tid < nvalid) store_partial<kFuse>(lse_base + (int64_t)team_tid * prm.S + sp, -INFINITY);
    }
    return;
  }

  typedef TDIST_AS3 unsigned char* lds_u8;  // explicit LDS pointers: a generic pointer would turn reads into
                                            // flat loads, which count on vmcnt and break the DMA accounting
  lds_u8 const smem3 = (lds_u8)smem;
  lds_u8 const wbase = smem3 + wave * C::kWaveBytes;
  lds_u8 const tbl_base = wbase + NST * C::kStageBytes;

  const int nb_total = (end - start + KEYS - 1) / KEYS;
  // this wave's blocks: every NW-th one of the kv head's; or all of its own kv head's, split after split (an empty
  // split at the sequence's end runs one block with every key masked, which writes its zeros)
  auto blocks_of = [&](int lo, int hi) { return max(1, (hi - lo + KEYS - 1) / KEYS); };
  int n_w = nb_total > wave ? (nb_total - wave + NW - 1) / NW : 0;
  if constexpr (kWaveHeads) {
    n_w = 0;
    for (int sp = 0; sp < n_splits; ++sp) n_w += blocks_of(start + sp * per, min(start + (sp + 1) * per, len));
  }

  // ---- Q fragments (B operand of the score MFMA): head x, dims 32s + 8g .. +8 -------------------
  typename MMA::frag8 qf[DK / 32];
  auto load_q = [&](int seq) {
    const unsigned char* qrow = prm.q + (int64_t)seq * prm.q_sb + (int64_t)(h0 + x) * prm.q_sh;
#pragma unroll
    for (int s = 0; s < DK / 32; ++s) {
      int4v raw = {0, 0, 0, 0};
      if (x < nvalid && (!kPadded || 4 * s + g < valid_chunks)) raw = *(const int4v*)(qrow + (32 * s + 8 * g) * 2);
      qf[s] = __builtin_bit_cast(typename MMA::frag8, raw);
    }
    // Waited for here: a query fetched inside the stream would otherwise be waited for at every use in the loop, and
    // with it (loads count in order) the whole stream behind it.
    if constexpr (kStream) {
#pragma unroll
      for (int s = 0; s < DK / 32; ++s) {
        int4v raw = __builtin_bit_cast(int4v, qf[s]);
        asm volatile("" : "+v"(raw));
        qf[s] = __builtin_bit_cast(typename MMA::frag8, raw);
      }
    }
  };
  if constexpr (!kStream) load_q(b);

  constexpr float kLog2e = 1.4426950408889634f;
  const float scale_log2 = prm.sm_scale * kLog2e;

  float m_run = -INFINITY;  // running max (log2 domain) of head x, identical in the 4 lane groups
  float l_run = 0.f;        // this lane group's share of the running sum
  float4v acc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) acc[d] = float4v{0.f, 0.f, 0.f, 0.f};

  // Loop-invariant LDS offsets (relative to the stage) of this lane's operand reads. The swizzle moves a chunk within
  // a window of kSwzMask + 1 chunks only, so the windows of a longer row share their offsets.
  // K (A operand of the scores): row = key x of group q, logical chunk 4s+g.
  // The extra key dimensions D + 32s' + 8g live in their own rows behind the K and V rows.
  constexpr int kWinChunks = C::kSwzMask + 1, kWinBytes = kWinChunks * 16;
  constexpr int kKWin = kWinChunks / 4 < D / 32 ? kWinChunks / 4 : D / 32, kVWin = kWinChunks / 2 < DT ? kWinChunks / 2 : DT;
  int koff[G][kKWin], peoff[G][DPE > 0 ? DPE / 32 : 1];
#pragma unroll
  for (int q = 0; q < G; ++q) {
    const int key = 16 * q + x;
#pragma unroll
    for (int s = 0; s < kKWin; ++s) koff[q][s] = key * C::kRowBytes + (((4 * s + g) ^ C::kswz(key)) << 4);
#pragma unroll
    for (int s = 0; s < DPE / 32; ++s) peoff[q][s] = C::kPeBase + key * C::kPeRowBytes + (((4 * s + g) ^ C::peswz(key)) << 4);
  }
  auto k_at = [&](int q, int s) { return s < D / 32 ? koff[q][s % kKWin] + s / kKWin * kWinBytes : peoff[q][s - D / 32]; };
  // V^T (A operand of the output MFMA) through the transposing LDS read: within a 16-lane block, lane x ends
  // up with elements x, 16+x, 32+x, 48+x of the 64 the block loads (lane s loads 4 consecutive ones), so lane s
  // supplies V[key 4g + s/4 of group q][dv 16d + 4(s%4) .. +3] and lane x receives V[4g+j][16d+x], j = 0..3.
  int voff[G][kVWin];
#pragma unroll
  for (int q = 0; q < G; ++q)
#pragma unroll
    for (int d = 0; d < kVWin; ++d) {
      const int key = 16 * q + 4 * g + (x >> 2);
      const int chunk = 2 * d + ((x & 3) >> 1);
      voff[q][d] = C::kVBase + key * C::kRowBytes + ((chunk ^ C::vswz(key)) << 4) + (x & 1) * 8;
    }

  // A block: its first key and the key range [lo, hi) of its split. Keys outside the range are read as the nearest
  // key inside (and, for a split that is empty, as the sequence's last key) and masked in the scores.
  struct Block { int key0, lo, hi, seq; };
  auto clamp_key = [&](int n, const Block& blk) {
    n = max(min(n, blk.hi - 1), blk.lo);
    if constexpr (kWaveHeads) n = min(n, len - 1);
    return n;
  };
  // first key of the wave's j-th block where the workgroup shares one split
  auto shared_block = [&](int j) { return Block{start + (wave + j * NW) * KEYS, start, end, b}; };
  // kWaveHeads: a cursor over the team's blocks in order
  struct Cursor { Block blk; int left; };   // left: blocks of this split still to come, this one included
  auto cursor_begin = [&]() { return Cursor{Block{start, start, end, b}, blocks_of(start, end)}; };
  auto cursor_next = [&](Cursor& c) {
    c.blk.key0 += KEYS;
    if (--c.left == 0) {
      c.blk.lo += per;
      c.blk.hi = min(c.blk.lo + per, len);
      c.blk.key0 = c.blk.lo;
      c.left = blocks_of(c.blk.lo, c.blk.hi);
    }
  };

  // page-table row of block j → table ring slot j % kTableSlots (one entry per key)
  auto issue_table = [&](int j, const Block& blk) {
    if (lane < KEYS) {
      const int n = clamp_key(blk.key0 + lane, blk);
      const int e = (int)(((uint64_t)(uint32_t)n * prm.page_magic) >> prm.page_shift);
      const int32_t* src = prm.table + (int64_t)(kStream ? blk.seq : b) * prm.t_s + e;
      __builtin_amdgcn_global_load_lds((const TDIST_AS1 void*)src,
                                       (TDIST_AS3 void*)(tbl_base + (j % kTableSlots) * C::kTableSlotBytes), 4, 0, 0);
    }
  };

  constexpr int kAux = TDIST_KV_AUX;
  // K and V rows of block j → stage j % NST
  // The byte offset of a row within its cache (page, place in the page, head) is worked out once per block, by one lane
  // per row (K rows in lanes 0 .. KEYS-1, V rows in the next KEYS), and handed to the lanes that fetch the row's chunks.
  auto issue_rows = [&](int j, const Block& blk) {
    const volatile TDIST_AS3 int32_t* tbl =
        (const volatile TDIST_AS3 int32_t*)(tbl_base + (j % kTableSlots) * C::kTableSlotBytes);
    lds_u8 const kst = wbase + (j % NST) * C::kStageBytes;
    lds_u8 const vst = kst + C::kVBase;
    uint32_t off_lo, off_hi;
    {
      const int row = lane & (KEYS - 1);
      const bool is_v = (lane & KEYS) != 0;
      const uint32_t n = (uint32_t)clamp_key(blk.key0 + row, blk);
      const uint32_t in_page = n - (uint32_t)(((uint64_t)n * prm.page_magic) >> prm.page_shift) * (uint32_t)prm.page_size;
      const uint64_t off = (uint64_t)(uint32_t)tbl[row] * (uint64_t)(is_v ? prm.v_sp : prm.k_sp) +
                           (in_page * (uint32_t)(is_v ? prm.v_st : prm.k_st) + (uint32_t)kvh * (uint32_t)(is_v ? prm.v_sh : prm.k_sh));
      off_lo = (uint32_t)off;
      off_hi = (uint32_t)(off >> 32);
    }
    // `row`: which lane's offset; the same for the whole wave where a row takes a whole instruction
    auto row_offset = [&](int row, bool uniform) -> uint64_t {
      const uint32_t lo = uniform ? __builtin_amdgcn_readlane(off_lo, row) : (uint32_t)__shfl((int)off_lo, row);
      const uint32_t hi = uniform ? __builtin_amdgcn_readlane(off_hi, row) : (uint32_t)__shfl((int)off_hi, row);
      return ((uint64_t)hi << 32) | lo;
    };
    constexpr bool kWholeRow = C::kRowsPerInstr == 1;
    constexpr int kInstr = C::kInstrPerTensor, kPe = C::kPeInstr;
    const int chunk = lane % C::kLanesPerRow, pchunk = lane % C::kPeLanesPerRow;
    // all exchanges between lanes first, then the loads: the compiler would wait for each exchange at its load
    uint64_t k_off[kInstr], v_off[kInstr], pe_off[kPe > 0 ? kPe : 1];
#pragma unroll
    for (int u = 0; u < kInstr; ++u) {
      const int key = kWholeRow ? u : u * C::kRowsPerInstr + lane / C::kLanesPerRow;
      k_off[u] = row_offset(key, kWholeRow);
      v_off[u] = row_offset(KEYS + key, kWholeRow);
    }
#pragma unroll
    for (int u = 0; u < kPe; ++u) pe_off[u] = row_offset(u * C::kPeRowsPerInstr + lane / C::kPeLanesPerRow, false);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kInstr; ++u) {
      const int key = kWholeRow ? u : u * C::kRowsPerInstr + lane / C::kLanesPerRow;
      const int kchunk = chunk ^ C::kswz(key), vchunk = chunk ^ C::vswz(key);
      const unsigned char* ksrc = prm.k + k_off[u] + (uint32_t)(kchunk << 4);
      if (kPadded && kchunk >= valid_chunks) ksrc = kZeroChunk;
      __builtin_amdgcn_global_load_lds((const TDIST_AS1 void*)ksrc, (TDIST_AS3 void*)(kst + u * 1024), 16, 0, kAux);
      const unsigned char* vsrc = prm.v + v_off[u] + (uint32_t)(vchunk << 4);
      if (kPadded && vchunk >= valid_chunks) vsrc = kZeroChunk;
      __builtin_amdgcn_global_load_lds((const TDIST_AS1 void*)vsrc, (TDIST_AS3 void*)(vst + u * 1024), 16, 0, kAux);
    }
#pragma unroll
    for (int u = 0; u < kPe; ++u) {
      const int key = u * C::kPeRowsPerInstr + lane / C::kPeLanesPerRow;
      const unsigned char* psrc = prm.k + pe_off[u] + (uint32_t)(C::kRowBytes + ((pchunk ^ C::peswz(key)) << 4));
      __builtin_amdgcn_global_load_lds((const TDIST_AS1 void*)psrc, (TDIST_AS3 void*)(kst + C::kPeBase + u * 1024), 16, 0, kAux);
    }
  };

  auto compute = [&](int j, const Block& blk) {
    const int key0 = blk.key0;
    lds_u8 const st = wbase + (j % NST) * C::kStageBytes;
    // Operand reads run kAhead tiles ahead of their products: two groups of registers in turn.
    // scores: A = K rows (key x of group q, dims 32s+8g..), B = Q  →  sc[q][i]: key 16q+4g+i, head x
    constexpr int kAhead = 4;
    static_assert(DT % kAhead == 0 && kAhead * G < 16, "whole groups of tiles; lgkmcnt counts to 15");
    float4v sc[G];
#pragma unroll
    for (int q = 0; q < G; ++q) {
      sc[q] = float4v{0.f, 0.f, 0.f, 0.f};
      int4v kb[2][kAhead];
      auto read_k = [&](int s0, int4v(&to)[kAhead]) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
          if (s0 + u < DK / 32) to[u] = *(const TDIST_AS3 int4v*)(st + k_at(q, s0 + u));
      };
      read_k(0, kb[0]);
#pragma unroll
      for (int s0 = 0; s0 < DK / 32; s0 += kAhead) {
        if (s0 + kAhead < DK / 32) read_k(s0 + kAhead, kb[(s0 / kAhead + 1) & 1]);
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
          if (s0 + u < DK / 32) sc[q] = MMA::mma32(__builtin_bit_cast(typename MMA::frag8, kb[(s0 / kAhead) & 1][u]), qf[s0 + u], sc[q]);
      }
    }
    // (the first V tiles are on their way while the probabilities are worked out)
    // The transposing reads and the waits for them are written out: for the builtin the compiler waits until every load
    // into the LDS is done, the ones in flight for later blocks included.
    int2v vb[2][kAhead][G];
    const uint32_t v_base = (uint32_t)(uintptr_t)st;
    auto read_v = [&](int d0, int2v(&to)[kAhead][G]) {
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
#pragma unroll
        for (int q = 0; q < G; ++q)
          if (d0 + u < DT)
            asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2"
                         : "=v"(to[u][q])
                         : "v"(v_base + (uint32_t)voff[q][(d0 + u) % kVWin]), "n"((d0 + u) / kVWin * kWinBytes)
                         : "memory");
    };
    auto wait_v = [&](int later, int2v(&of)[kAhead][G]) {   // all but the `later` youngest LDS reads are back
      if (later == 0) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      else asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(kAhead * G) : "memory");
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
#pragma unroll
        for (int q = 0; q < G; ++q) asm volatile("" : "+v"(of[u][q]));
    };
    read_v(0, vb[0]);
    float t[G][4];
    float mx = -INFINITY;
#pragma unroll
    for (int q = 0; q < G; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v;
        if (kSoftCap) {
          v = prm.soft_cap * tanhf(sc[q][i] * prm.sm_scale / prm.soft_cap) * kLog2e;
        } else {
          v = sc[q][i] * scale_log2;
        }
        const bool valid = key0 + 16 * q + 4 * g + i < blk.hi;
        t[q][i] = valid ? v : -INFINITY;
        mx = fmaxf(mx, t[q][i]);
      }
    // The sums are kept relative to m_run, which is raised only when a score lies kSlack above it: their values then stay
    // below 2^kSlack, which costs no precision, and the lanes of a head compare notes and the sums are rescaled a few
    // times per stream instead of per block.
    constexpr float kSlack = 8.f;
    if (__any(mx > m_run + kSlack)) {
      mx = max_lane_xor<32>(max_lane_xor<16>(mx));
      const float m_new = fmaxf(m_run, mx);
      const float alpha = (m_run == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < DT; ++d) acc[d] *= alpha;
      m_run = m_new;
    }
    const float m_safe = (m_run == -INFINITY) ? 0.f : m_run;
    // probabilities as the B operand: k slots 4q..4q+3 of lane group g ↔ keys 16q+4g .. +3
    uint32_t hi[G][2], lo[G][2];
#pragma unroll
    for (int q = 0; q < G; ++q) {
      float p[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[i] = __builtin_amdgcn_exp2f(t[q][i] - m_safe);
        l_run += p[i];
      }
      MMA::split(p[0], p[1], hi[q][0], lo[q][0]);
      MMA::split(p[2], p[3], hi[q][1], lo[q][1]);
    }
    // O^T tiles: A = V^T (dv 16d+x; k slots as above), B = P^T
#pragma unroll
    for (int d0 = 0; d0 < DT; d0 += kAhead) {
      if (d0 + kAhead < DT) read_v(d0 + kAhead, vb[(d0 / kAhead + 1) & 1]);
      wait_v(d0 + kAhead < DT ? 1 : 0, vb[(d0 / kAhead) & 1]);
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int d = d0 + u;
        const auto& v = vb[(d0 / kAhead) & 1][u];
        if constexpr (G == 2) {
          const int2v a0 = v[0], a1 = v[G - 1];
          const int4v vt = {a0[0], a0[1], a1[0], a1[1]};
          const int4v ph = {(int)hi[0][0], (int)hi[0][1], (int)hi[G - 1][0], (int)hi[G - 1][1]};
          const int4v pl = {(int)lo[0][0], (int)lo[0][1], (int)lo[G - 1][0], (int)lo[G - 1][1]};
          const typename MMA::frag8 vf = __builtin_bit_cast(typename MMA::frag8, vt);
          acc[d] = MMA::mma32(vf, __builtin_bit_cast(typename MMA::frag8, ph), acc[d]);
          acc[d] = MMA::mma32(vf, __builtin_bit_cast(typename MMA::frag8, pl), acc[d]);
        } else {
          const int2v ph = {(int)hi[0][0], (int)hi[0][1]};
          const int2v pl = {(int)lo[0][0], (int)lo[0][1]};
          const typename MMA::frag4 vf = __builtin_bit_cast(typename MMA::frag4, v[0]);
          acc[d] = MMA::mma16(vf, __builtin_bit_cast(typename MMA::frag4, ph), acc[d]);
          acc[d] = MMA::mma16(vf, __builtin_bit_cast(typename MMA::frag4, pl), acc[d]);
        }
      }
    }
  };

  constexpr float kLn2 = 0.6931471805599453f;
  if constexpr (kStream) {
    static_assert(!C::kWaitFirst, "a kv head per wave: several groups in flight");
    // One pipeline over the range's blocks, across the sequences in it.
    struct Walk { Block blk; int left, rem; };   // left / rem: blocks of this sequence / of the range, this one included
    auto walk_begin = [&]() {
      const int hi = lens[sr.seq];
      return Walk{Block{sr.block * KEYS, 0, hi, sr.seq}, min((hi + KEYS - 1) / KEYS - sr.block, sr.n), sr.n};
    };
    auto walk_next = [&](Walk& w) {   // (stays on the last block)
      if (w.rem == 1) return;
      --w.rem;
      w.blk.key0 += KEYS;
      if (--w.left == 0) {
        do w.blk.hi = lens[++w.blk.seq];
        while (w.blk.hi <= 0);
        w.blk.key0 = 0;
        w.left = min((w.blk.hi + KEYS - 1) / KEYS, w.rem);
      }
    };
    Walk w_tbl = walk_begin(), w_rows = w_tbl, w_cmp = w_tbl;
    int j_tbl = 0;
    for (; j_tbl <= C::kP; ++j_tbl) {
      issue_table(j_tbl, w_tbl.blk);
      walk_next(w_tbl);
    }
    load_q(sr.seq);   // (one trip to memory with the page-table rows)
    wait_vmcnt<0>();
    for (int gi = 0; gi < C::kP; ++gi) {
      if (gi < sr.n) {
        issue_table(j_tbl++, w_tbl.blk);
        walk_next(w_tbl);
        issue_rows(gi, w_rows.blk);
        walk_next(w_rows);
      }
    }
    // The range's first sequence may have begun in an earlier range (its partial result waits in registers for the
    // end of the stream) and its last may go on in the next one; all between are whole and stored when they end.
    bool begun_here = sr.block == 0;
    float4v held[DT];
    float held_lse = 0.f;
#pragma unroll
    for (int d = 0; d < DT; ++d) held[d] = float4v{0.f, 0.f, 0.f, 0.f};
    bool any_held = false;
    auto part_row = [&](int rg, int slot) { return ((int64_t)rg * 2 + slot) * prm.Hq + h0; };
    auto store_part = [&](int slot, const float4v(&val)[DT], float val_lse) {
      if (x < nvalid) {
        float* o = prm.out + part_row(range, slot) * Dout;
#pragma unroll
        for (int d = 0; d < DT; ++d)
          if (!kPadded || 16 * d + 4 * g < Dout) store_partial4<true>(o + partial_tile(nvalid, Dout, d, x, g), val[d]);
        if (g == 0) store_partial<true>(prm.lse + part_row(range, slot) + x, val_lse);
      }
    };
    for (int i = 0; i < sr.n; ++i) {
      if (i + C::kP < sr.n) {
        issue_table(j_tbl++, w_tbl.blk);
        walk_next(w_tbl);
        issue_rows(i + C::kP, w_rows.blk);
        walk_next(w_rows);
      }
      wait_groups<C::kLoadsPerGroup>(min(C::kP, sr.n - 1 - i));
      compute(i, w_cmp.blk);
      if (w_cmp.left == 1) {
        const float L = sum_lane_xor<32>(sum_lane_xor<16>(l_run));
        const float inv = L > 0.f ? 1.f / L : 0.f;
        const float r_lse = L > 0.f ? (m_run + log2f(L)) * kLn2 : -INFINITY;
        const bool ends = w_cmp.blk.key0 + KEYS >= w_cmp.blk.hi;
#pragma unroll
        for (int d = 0; d < DT; ++d) acc[d] *= inv;
        if (begun_here && ends) {
          if (x < nvalid) {
            const int64_t o = (int64_t)w_cmp.blk.seq * prm.fo_sb + (int64_t)(h0 + x) * prm.fo_sh + 4 * g;
#pragma unroll
            for (int d = 0; d < DT; ++d)
              if (!kPadded || 16 * d + 4 * g < Dout) store_elem4(prm.final_out, o + 16 * d, prm.final_dtype, prm.fo_vec, acc[d]);
            if (prm.final_lse && g == 0) prm.final_lse[(int64_t)w_cmp.blk.seq * prm.Hq + h0 + x] = r_lse;
          }
        } else if (i == sr.n - 1) {
          store_part(begun_here ? 1 : 0, acc, r_lse);
        } else {   // (it began in an earlier range and ends here)
          any_held = true;
          held_lse = r_lse;
#pragma unroll
          for (int d = 0; d < DT; ++d) held[d] = acc[d];
        }
        if (i < sr.n - 1) {
          begun_here = true;
          m_run = -INFINITY;
          l_run = 0.f;
#pragma unroll
          for (int d = 0; d < DT; ++d) acc[d] = float4v{0.f, 0.f, 0.f, 0.f};
          walk_next(w_cmp);
          load_q(w_cmp.blk.seq);
          continue;
        }
      }
      walk_next(w_cmp);
    }
    if (any_held) store_part(0, held, held_lse);
    return;
  }
  if constexpr (kWaveHeads) {
    static_assert(!C::kWaitFirst, "a kv head per wave: several groups in flight");
    // One pipeline over all blocks of the team's splits: the loads of the next split's first blocks are in flight
    // while the last blocks of this one are computed. The results go out of the registers (no LDS: the ring belongs
    // to the loads in flight) when the stream has ended.
    Cursor c_tbl = cursor_begin(), c_rows = cursor_begin(), c_cmp = cursor_begin();
    int j_tbl = 0;
    for (; j_tbl <= C::kP; ++j_tbl) {
      issue_table(j_tbl, c_tbl.blk);
      cursor_next(c_tbl);
    }
    wait_vmcnt<0>();
    for (int gi = 0; gi < C::kP; ++gi) {
      if (gi < n_w) {
        issue_table(j_tbl++, c_tbl.blk);
        cursor_next(c_tbl);
        issue_rows(gi, c_rows.blk);
        cursor_next(c_rows);
      }
    }
    // results of the splits before the team's last one, held until the stream ends
    constexpr int kMaxHeld = decode_max_splits_per_team(D, kSoftCap || kFuse || kPadded) - 1;
    float4v held[kMaxHeld][DT];
    float held_lse[kMaxHeld];
#pragma unroll
    for (int u = 0; u < kMaxHeld; ++u) {
      held_lse[u] = 0.f;
#pragma unroll
      for (int d = 0; d < DT; ++d) held[u][d] = float4v{0.f, 0.f, 0.f, 0.f};
    }
    int sp = 0;
    for (int i = 0; i < n_w; ++i) {
      if (i + C::kP < n_w) {
        issue_table(j_tbl++, c_tbl.blk);
        cursor_next(c_tbl);
        issue_rows(i + C::kP, c_rows.blk);
        cursor_next(c_rows);
      }
      wait_groups<C::kLoadsPerGroup>(min(C::kP, n_w - 1 - i));
      compute(i, c_cmp.blk);
      if (c_cmp.left == 1) {
        // the split's last block: this lane holds dimensions 16d + 4g .. + 3 of head x
        const float L = sum_lane_xor<32>(sum_lane_xor<16>(l_run));
        float4v r[DT];
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
          for (int e = 0; e < 4; ++e) r[d][e] = L > 0.f ? acc[d][e] / L : 0.f;
        const float r_lse = L > 0.f ? (m_run + log2f(L)) * kLn2 : -INFINITY;
        auto store_split = [&](int which, const float4v(&val)[DT], float val_lse) {
          if (x < nvalid) {
            float* o = out_base + ((int64_t)x * prm.S + which) * Dout + 4 * g;
#pragma unroll
            for (int d = 0; d < DT; ++d)
              if (!kPadded || 16 * d + 4 * g < Dout) store_partial4<kFuse>(o + 16 * d, val[d]);
            if (g == 0) store_partial<kFuse>(lse_base + (int64_t)x * prm.S + which, val_lse);
          }
        };
        if (i == n_w - 1) {
          // the team's last split: everything goes out now
#pragma unroll
          for (int u = 0; u < kMaxHeld; ++u)
            if (u < sp) store_split(u, held[u], held_lse[u]);
          store_split(sp, r, r_lse);
        } else {
          // Not yet: stores count on the same counter as the loads, so the next wait for a block would also wait for
          // these stores, which take tens of microseconds to be acknowledged while the read stream runs (measured:
          // 40 us per launch at 8 stores per wave). The result waits in registers for the end of the stream.
#pragma unroll
          for (int u = 0; u < kMaxHeld; ++u)
            if (sp == u) {
#pragma unroll
              for (int d = 0; d < DT; ++d) held[u][d] = r[d];
              held_lse[u] = r_lse;
            }
        }
        ++sp;
        m_run = -INFINITY;
        l_run = 0.f;
#pragma unroll
        for (int d = 0; d < DT; ++d) acc[d] = float4v{0.f, 0.f, 0.f, 0.f};
      }
      cursor_next(c_cmp);
    }
    return;
  }

  if (n_w > 0) {
    // page-table rows of the first P+1 blocks, then the first P row groups
    for (int j = 0; j <= C::kP; ++j) issue_table(j, shared_block(j));
    wait_vmcnt<0>();
    for (int gi = -C::kP; gi < 0; ++gi) {
      if (gi + C::kP < n_w) {
        issue_table(gi + 2 * C::kP + 1, shared_block(gi + 2 * C::kP + 1));
        issue_rows(gi + C::kP, shared_block(gi + C::kP));
      }
    }
  }
  for (int i = 0; i < n_w; ++i) {
    if constexpr (C::kWaitFirst) wait_vmcnt<0>();
    if (i + C::kP < n_w) {
      issue_table(i + 2 * C::kP + 1, shared_block(i + 2 * C::kP + 1));
      issue_rows(i + C::kP, shared_block(i + C::kP));
    }
    if constexpr (!C::kWaitFirst) wait_groups<C::kLoadsPerGroup>(min(C::kP, n_w - 1 - i));
    compute(i, shared_block(i));
  }

  // ---- merge the waves' partial states ---------------------------------------------------------
  l_run = sum_lane_xor<32>(sum_lane_xor<16>(l_run));
  wait_vmcnt<0>();
  __syncthreads();  // every wave is done with its ring; reuse it
  TDIST_AS3 float* s_m = (TDIST_AS3 float*)(wbase);  // [16]
  TDIST_AS3 float* s_l = s_m + 16;                   // [16]
  TDIST_AS3 float* s_acc = s_l + 16;                 // [16][kAccRow]: the 4 floats between rows spread them over the banks
  constexpr int kAccRow = decode_acc_row(D);
  if (lane < 16) {
    s_m[lane] = m_run;
    s_l[lane] = l_run;
  }
#pragma unroll
  for (int d = 0; d < DT; ++d) *(TDIST_AS3 float4v*)(s_acc + x * kAccRow + 16 * d + 4 * g) = acc[d];
  __syncthreads();
  // What each wave counts for in each head: lane l works it out for wave l / 16 and head l % 16 (in every
  // wave: nobody waits), and the LDS hands it round.
  static_assert(kWaveHeads || kStream || NW <= 4, "one lane per wave and head");
  float r_lse16;
  TDIST_AS3 float* const s_w = s_acc + 16 * kAccRow;   // this wave's [4][16]
  {
    const int w = lane >> 4, h = lane & 15;
    const TDIST_AS3 float* wm = (const TDIST_AS3 float*)(smem3 + min(w, NW - 1) * C::kWaveBytes);
    const float mw = w < NW ? wm[h] : -INFINITY;
    const float M = max_lane_xor<32>(max_lane_xor<16>(mw));
    const float sc = (mw == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(mw - M);
    float L = w < NW ? wm[16 + h] * sc : 0.f;
    L = sum_lane_xor<32>(sum_lane_xor<16>(L));
    s_w[lane] = sc / L;
    r_lse16 = (M + log2f(L)) * kLn2;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const int vecs = Dout / 4;
  for (int idx = threadIdx.x; idx < nvalid * vecs; idx += NW * 64) {
    const int h = idx / vecs, dv = (idx - h * vecs) * 4;
    float4v O = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float4v a4 = *(const TDIST_AS3 float4v*)((const TDIST_AS3 float*)(smem3 + w * C::kWaveBytes) + 32 + h * kAccRow + dv);
      const float sc = s_w[w * 16 + h];
#pragma unroll
      for (int e = 0; e < 4; ++e) O[e] += a4[e] * sc;
    }
    float* o = out_base + (int64_t)h * prm.S * Dout + dv;
    if (prm.part_vec) {
      store_partial4<kFuse>(o, O);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) store_partial<kFuse>(o + e, O[e]);
    }
  }
  if (threadIdx.x < nvalid) store_partial<kFuse>(lse_base + (int64_t)threadIdx.x * prm.S, r_lse16);
}

// ---- combine --------------------------------------------------------------------------------------
struct CombineParams {
  const unsigned char* part;
  const float* lse;
  const int32_t* lens;
  unsigned char* out;
  float* lse_out;
  int P, mode, B, Hq, Dv;
  int part_dtype, out_dtype;
  int64_t p_sp, p_sb, p_sh;  // element strides
  int64_t l_sp, l_sb, l_sh;
  int64_t o_sb, o_sh;
};

// One wave per (b,h); lanes stride over Dv. Partial j is weighted by exp(lse_j - max).
// Lane j holds the LSE of partial j (one load per lane instead of a loop of loads in every lane; -inf where the
// partial is skipped), the maximum is a wave reduction, and the partial rows of up to 32 / kPerLane partials are in
// flight together: two round trips to memory for a merge of 16 partials. The sums run over the partials in index
// order, whatever the batching.
template <int kPerLane>
__global__ __launch_bounds__(256) void decode_combine_kernel(const CombineParams prm) {
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int64_t bh = (int64_t)blockIdx.x * 4 + wave;
  if (bh >= (int64_t)prm.B * prm.Hq) return;
  const int b = (int)(bh / prm.Hq);
  const int h = (int)(bh - (int64_t)b * prm.Hq);
  auto skipped = [&](int j) -> bool {
    if (prm.mode == 1) {
      const int len = prm.lens[b];
      const int per = (len + prm.P - 1) / prm.P;
      const int st = per * j;
      return min(st + per, len) <= st;
    }
    if (prm.mode == 2) return prm.lens[(int64_t)j * prm.B + b] == 0;
    return false;
  };
  const float* lse = prm.lse + (int64_t)b * prm.l_sb + (int64_t)h * prm.l_sh;
  // LSE of partial j0 + lane
  auto lse_of_lane = [&](int j0) -> float {
    const int j = j0 + lane;
    return (j < prm.P && !skipped(j)) ? lse[(int64_t)j * prm.l_sp] : -INFINITY;
  };
  float M = -INFINITY;
  for (int j0 = 0; j0 < prm.P; j0 += 64) M = fmaxf(M, lse_of_lane(j0));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o));
  float L = 0.f;
  float acc[kPerLane];
#pragma unroll
  for (int q = 0; q < kPerLane; ++q) acc[q] = 0.f;
  if (M != -INFINITY) {
    constexpr int kBatch = 32 / kPerLane;
    for (int c0 = 0; c0 < prm.P; c0 += 64) {
      const float l_lane = lse_of_lane(c0);
      const int n_here = min(64, prm.P - c0);
      for (int j0 = 0; j0 < n_here; j0 += kBatch) {
        float w[kBatch];
        float x[kBatch][kPerLane];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const int jj = j0 + u;   // (within the chunk; lanes beyond it hold -inf)
          const float lj = jj < 64 ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, l_lane), jj & 63)) : -INFINITY;
          w[u] = lj == -INFINITY ? 0.f : __expf(lj - M);
          const int64_t base = (int64_t)min(c0 + jj, prm.P - 1) * prm.p_sp + (int64_t)b * prm.p_sb + (int64_t)h * prm.p_sh;
#pragma unroll
          for (int q = 0; q < kPerLane; ++q) {
            const int d = lane + q * 64;
            x[u][q] = (d < prm.Dv && lj != -INFINITY) ? load_elem(prm.part, base + d, prm.part_dtype) : 0.f;
          }
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          L += w[u];   // a skipped, empty or out-of-range partial has w = 0 and x = 0: it adds nothing
#pragma unroll
          for (int q = 0; q < kPerLane; ++q) acc[q] += w[u] * x[u][q];
        }
      }
    }
  }
  const int64_t obase = (int64_t)b * prm.o_sb + (int64_t)h * prm.o_sh;
#pragma unroll
  for (int u = 0; u < kPerLane; ++u) {
    const int d = lane + u * 64;
    if (d < prm.Dv) store_elem(prm.out, obase + d, prm.out_dtype, L > 0.f ? acc[u] / L : 0.f);
  }
  if (prm.lse_out && lane == 0) prm.lse_out[bh] = L > 0.f ? M + logf(L) : -INFINITY;
}

static int launch_combine(const CombineParams& prm, hipStream_t stream) {
  const int64_t blocks = ceil_div((int64_t)prm.B * prm.Hq, 4);
  if (blocks > 0x7fffffff) return fail(TDIST_ERR_UNSUPPORTED, "tdist_decode_combine: grid too large");
  auto kern = prm.Dv <= 128 ? decode_combine_kernel<2> : prm.Dv <= 256 ? decode_combine_kernel<4> : decode_combine_kernel<8>;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), 0, stream, prm);
  return launch_status("tdist_decode_combine");
}

// The merge with the other ranks' results that may follow a stream: rank `own`'s place in c.part and c.lse is the stream's output.
struct RankParams {
  CombineParams c;
  int own, part_vec, out_vec;   // rows of four elements take one load / store
};

// Fused tail: publishes this team's partial result (the workgroup's, or with kWaveHeads the wave's); the last of the
// S teams of a (sequence, head block) to get here merges their partials (same arithmetic, in the same order, as
// decode_combine_kernel in mode 1) and puts the counter back to zero for the next launch.
template <int DM, int NW, bool kPadded, bool kWaveHeads>
__device__ __forceinline__ void decode_fused_merge(const DecodeParams& prm) {
  const int D = kPadded ? prm.d_valid : DM;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  TDIST_AS3 int* const s_last = (TDIST_AS3 int*)smem;
  const int group = prm.Hq / prm.Hkv;
  const int head_blocks = (group + 15) >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kvh = kWaveHeads ? blockIdx.x * NW + wave : blockIdx.x / head_blocks;
  const int hb = kWaveHeads ? 0 : blockIdx.x - kvh * head_blocks;
  const int b = blockIdx.z;
  const int h0 = kvh * group + hb * 16;
  const int nvalid = min(16, group - hb * 16);
  const int team_tid = kWaveHeads ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
  constexpr int kTeam = kWaveHeads ? 64 : NW * 64;
  // one counter per (sequence, kv head, head block)
  int32_t* const ctr = prm.counters + ((int64_t)b * prm.Hkv + kvh) * head_blocks + hb;

  // This thread's partial results were stored write-through (store_partial): once the stores have completed they
  // are visible to every XCD. (A release fence here would write back the whole L2 once per wave: measured at 2x the
  // kernel time.)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if constexpr (kWaveHeads) {
    // the wave's stores are complete: its first lane counts, and tells the others
    // (its team brought n_mine of the S splits)
    const int n_mine = min(prm.splits_per_team, prm.S - (int)blockIdx.y * prm.splits_per_team);
    int last = 0;
    if (team_tid == 0) {
      const int old = __hip_atomic_fetch_add(ctr, n_mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = old + n_mine == prm.S;
      if (last) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!__builtin_amdgcn_readfirstlane(last)) return;
  } else {
    // the barrier orders all of the workgroup's stores before thread 0's counter update
    __syncthreads();   // (also: every wave is done with the merge scratch that s_last overlays)
    if (threadIdx.x == 0) {
      const int old = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int last = old == prm.S - 1;
      if (last) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *s_last = last;
    }
    __syncthreads();
    if (!*s_last) return;
  }
  // The counter has reached S: every other team's stores completed before its increment. Only the merging team pays
  // for an acquire (it drops this CU's and this XCD's possibly stale lines; the K/V stream is non-temporal and
  // loses nothing by it), after which plain vector loads may read the partial results.
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");

  const float* lse_p = prm.lse + ((int64_t)b * prm.Hq + h0) * prm.S;
  const float* out_p = prm.out + ((int64_t)b * prm.Hq + h0) * prm.S * D;
  const int kVecs = D / 4;
  for (int idx = team_tid; idx < nvalid * kVecs; idx += kTeam) {
    const int h = idx / kVecs, dv = (idx - h * kVecs) * 4;
    const float* l = lse_p + (int64_t)h * prm.S;
    // sixteen splits at a time: their LSEs, then their rows, are in flight together (two round trips for 16 splits);
    // the sums run over the splits in order
    constexpr int kBatch = 16;
    float M = -INFINITY;
    for (int j0 = 0; j0 < prm.S; j0 += kBatch) {
      float lj[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) lj[u] = j0 + u < prm.S ? l[j0 + u] : -INFINITY;
#pragma unroll
      for (int u = 0; u < kBatch; ++u) M = fmaxf(M, lj[u]);
    }
    float L = 0.f;
    float4v acc = {0.f, 0.f, 0.f, 0.f};
    if (M != -INFINITY) {
      // an empty split has LSE = -inf and zeros: weight exp(-inf) = 0 adds nothing, as skipping it would
      for (int j0 = 0; j0 < prm.S; j0 += kBatch) {
        float lj[kBatch];
        float4v x[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const int j = min(j0 + u, prm.S - 1);
          lj[u] = l[j];
          x[u] = *(const float4v*)(out_p + ((int64_t)h * prm.S + j) * D + dv);
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          if (j0 + u < prm.S) {
            const float w = __expf(lj[u] - M);
            L += w;
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] += w * x[u][e];
          }
        }
      }
    }
    const int64_t o = (int64_t)b * prm.fo_sb + (int64_t)(h0 + h) * prm.fo_sh + dv;
#pragma unroll
    for (int e = 0; e < 4; ++e) store_elem(prm.final_out, o + e, prm.final_dtype, L > 0.f ? acc[e] / L : 0.f);
    if (dv == 0 && prm.final_lse) prm.final_lse[(int64_t)b * prm.Hq + h0 + h] = L > 0.f ? M + logf(L) : -INFINITY;
  }
}

template <typename MMA, int D, int DPE, int KEYS, int NW, int NST, bool kSoftCap, bool kFuse, bool kPadded, bool kWaveHeads = false>
__global__ __launch_bounds__(NW * 64) void decode_split_kv_kernel(const DecodeParams prm) {
  if (prm.when_lens != 0 && decode_lens_even(prm.lens, prm.B) != (prm.when_lens == 1)) return;
  decode_split_body<MMA, D, DPE, KEYS, NW, NST, kSoftCap, kFuse, kPadded, kWaveHeads>(prm);
  if constexpr (kFuse) decode_fused_merge<D, NW, kPadded, kWaveHeads>(prm);
}

template <typename MMA, int D, int DPE, int KEYS, int NW, int NST, bool kSoftCap, bool kFuse, bool kPadded, bool kWaveHeads = false>
static int launch_decode_cfg(const DecodeParams& prm, int head_blocks, hipStream_t stream) {
  typedef DecodeCfg<D, DPE, KEYS, NST> C;
  static_assert((32 + 16 * decode_acc_row(D) + 128) * 4 <= C::kWaveBytes, "merge scratch must fit in a wave's ring");
  const size_t lds = (size_t)NW * C::kWaveBytes;
  static_assert((size_t)NW * C::kWaveBytes <= 160 * 1024, "LDS of one CU");
  auto kern = decode_split_kv_kernel<MMA, D, DPE, KEYS, NW, NST, kSoftCap, kFuse, kPadded, kWaveHeads>;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return fail(TDIST_ERR_LAUNCH, "decode: cannot reserve %zu B of LDS: %s", lds, hipGetErrorString(e));
    attr_set = true;
  }
  dim3 grid(kWaveHeads ? prm.Hkv / NW : prm.Hkv * head_blocks,
            kWaveHeads ? (prm.S + prm.splits_per_team - 1) / prm.splits_per_team : prm.S, prm.B);
  hipLaunchKernelGGL(kern, grid, dim3(NW * 64), lds, stream, prm);
  return launch_status(kFuse ? "tdist_decode_fused" : "tdist_decode_split_kv");
}

constexpr int kMergeBatch = 16;   // partial results in flight per lane of the merge

// The second launch of the streaming form: the partial results of every sequence that is spread over several ranges into its
// result. A workgroup takes 64 16-byte pieces of one sequence's [Hq, Dv] plane; partial j of the sequence lies in the second
// slot of the range in which it begins (j = 0) and in the first slot of the others; a wave takes a run of them, kBatch rows and
// LSEs in flight per lane, and the LDS brings the waves' sums together in order: the result repeats bit for bit.
// Where the batch has fewer sequences than ranges a workgroup asks for its sequence, else for the one that crosses the boundary
// behind range `at` and begins in it (nothing to do at the other boundaries).
// A launch of its own, not the work of the last range to arrive: nobody counts arrivals, so the call holds no state that outlives
// it, and the partials of a long sequence are read by as many waves as its result has pieces.
// What bounds it: the launch and two trips to memory (lengths; rows and LSEs). Against the merge by the last wave to arrive, whole
// calls: 1 x 1320 keys, 32 / 8 heads 16.8 -> 16.0 us; latent heads, 16 up to 4096 keys 60.4 -> 57.7; 48 up to 8192 74.9 -> 75.7;
// 32 x 32768 660 -> 664. One wave could merge 63 ranges of a sequence at most; without that limit 1 x 131072 keys take 36 us
// instead of 156 with 6 / 1 heads and 87 instead of 155 with 32 / 8 (32 splits and their combine: 90, 91).
// 16 waves a workgroup where a sequence may have more partials than four waves hold in flight.
// kAlone: every wave takes 64 pieces of its own and all partials of them, eight in flight, and there is nothing to bring together:
// for batches whose sequences have few partials each (kAloneMost), where the other form's four waves share a handful and
// there are four times as many workgroups, each with its trip for the lengths: latent heads, 16 up to 4096 keys 39.2 -> 31.2 us a
// call, 53 x 100 keys 26.7 -> 18.9, 48 up to 8192 keys with 64 / 8 heads 83.7 -> 80.6, 32 x 32768 655 -> 650. A sequence of many
// partials beside short ones is read eight partials a trip: 4 uneven sequences up to 21874 keys, 256 ranges, 41.2 us with four
// waves to a piece, 45.5 alone, hence the bound.
// kRanks (1: 16-bit results, 2: fp32): the merge with the other ranks' results follows in the same launch, for which every sequence
// has its workgroups: this rank's result goes to its place among the ranks' (or comes from there, where the first launch has left it), as
// it is rounded there, and then the sums over the ranks as in decode_combine_kernel, in the same order and with the same bits.
// The other ranks' rows and LSEs are asked for first. With that merge as a launch of its own (6 us) behind this one a sequence-parallel
// layer of 1 x 1259 keys, 16 heads, 8 ranks took 27.6 us, 18.6 with it; 32 x 32768 keys 658 and 650.
// (Without ranks the launch carries nothing about them: a single sequence's call is as long as its host work.)
struct NoRanks {};
template <int KEYS, int NW, bool kAlone, int kRanks>
__global__ __launch_bounds__(NW * 64) void decode_stream_merge_kernel(const DecodeParams prm, const std::conditional_t<kRanks != 0, RankParams, NoRanks> rk) {
  constexpr int kBatch = kAlone ? kMergeBatch / 2 : kMergeBatch, kPieces = kAlone ? NW * 64 : 64;   // 16-byte pieces of a workgroup
  __shared__ float4v s_acc[kAlone ? 1 : NW][64];
  __shared__ float s_max[kAlone ? 1 : NW][64], s_sum[kAlone ? 1 : NW][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int vecs = prm.Hq * (prm.dv / 4), pieces = (vecs + kPieces - 1) / kPieces;
  const int at = blockIdx.x / pieces, piece = blockIdx.x - at * pieces;
  int seq = at, first_block, per;
  if (kRanks != 0 || prm.B < prm.ranges) {
    stream_sequence<KEYS>(prm, seq, first_block, per);
  } else {
    const StreamRange r = stream_range<KEYS>(prm, at + 1);
    if (r.n == 0 || r.block == 0 || r.first_block / r.per != at) return;
    seq = r.seq;
    first_block = r.first_block;
    per = r.per;
  }
  const int nb = (max(prm.lens[seq], 0) + KEYS - 1) / KEYS;
  if (kRanks == 0 && nb == 0) return;   // (zeros, stored by the first launch)
  const int first = first_block / per, parts = nb == 0 ? 1 : (first_block + nb - 1) / per - first + 1;
  if (kRanks == 0 && parts == 1) return;

  const int my_vec = piece * kPieces + (kAlone ? wave * 64 : 0) + lane, at_vec = min(my_vec, vecs - 1);
  int h, d;
  partial_piece(at_vec, prm.Hq / prm.Hkv, prm.dv, h, d);
  const int64_t plane = (int64_t)prm.Hq * prm.dv;
  auto slot_of = [&](int j) { return ((int64_t)first + j) * 2 + (j == 0 ? 1 : 0); };
  const int share = kAlone ? parts : (parts + NW - 1) / NW, j_begin = kAlone ? 0 : wave * share, j_end = min(parts, j_begin + share);
  // the first ranks' results on their way
  typedef std::conditional_t<kRanks == 2, float4v, int2v> piece_t;
  constexpr int kRankBatch = kRanks != 0 ? 8 : 1;
  piece_t rank_x[kRankBatch];
  float rank_lse[kRankBatch];
  [[maybe_unused]] auto load_ranks = [&](int r0) {
    if constexpr (kRanks != 0) {
#pragma unroll
      for (int u = 0; u < kRankBatch; ++u) {
        const int r = min(r0 + u, rk.c.P - 1);
        const unsigned char* at = rk.c.part + (r * rk.c.p_sp + seq * rk.c.p_sb + h * rk.c.p_sh + d) * (int64_t)(sizeof(piece_t) / 4);
        if (rk.part_vec) {
          rank_x[u] = *(const piece_t*)at;
        } else if constexpr (kRanks == 2) {
#pragma unroll
          for (int e = 0; e < 4; ++e) rank_x[u][e] = ((const float*)at)[e];
        } else {
          const unsigned short* a = (const unsigned short*)at;
          rank_x[u] = int2v{(int)(a[0] | (uint32_t)a[1] << 16), (int)(a[2] | (uint32_t)a[3] << 16)};
        }
        // (a rank without keys of the sequence is left out)
        rank_lse[u] = r0 + u < rk.c.P && r != rk.own && rk.c.lens[(int64_t)r * prm.B + seq] != 0 ? rk.c.lse[r * rk.c.l_sp + seq * rk.c.l_sb + h * rk.c.l_sh] : -INFINITY;
      }
    }
  };
  if constexpr (kRanks != 0) {
    if (parts == 1 && !kAlone && wave != 0) return;   // (nothing to bring together)
    if (kAlone || wave == 0) load_ranks(0);
  }
  float m = -INFINITY, l = 0.f;
  float4v acc = {0.f, 0.f, 0.f, 0.f};
  for (int j0 = kRanks != 0 && parts == 1 ? j_end : j_begin; j0 < j_end; j0 += kBatch) {
    float4v r[kBatch];
    float w[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int64_t slot = slot_of(min(j0 + u, j_end - 1));
      r[u] = *((const float4v*)(prm.out + slot * plane) + at_vec);
      w[u] = prm.lse[slot * prm.Hq + h];
    }
    float m_new = m;
#pragma unroll
    for (int u = 0; u < kBatch; ++u) m_new = fmaxf(m_new, w[u]);
    const float scale = m == -INFINITY ? 0.f : __expf(m - m_new);
    m = m_new;
    l *= scale;
    acc *= scale;
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const float p = j0 + u < j_end && w[u] != -INFINITY ? __expf(w[u] - m) : 0.f;
      l += p;
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += p * r[u][e];
    }
  }
  float M = m, L = l;
  if (!kAlone && !(kRanks != 0 && parts == 1)) {
    s_acc[wave][lane] = acc;
    s_max[wave][lane] = m;
    s_sum[wave][lane] = l;
    __syncthreads();
    if (wave != 0) return;
    M = s_max[0][lane];
#pragma unroll
    for (int v = 1; v < NW; ++v) M = fmaxf(M, s_max[v][lane]);
    L = 0.f;
    acc = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < NW; ++v) {
      const float p = s_max[v][lane] == -INFINITY ? 0.f : __expf(s_max[v][lane] - M);
      L += p * s_sum[v][lane];
      const float4v a = s_acc[v][lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += p * a[e];
    }
  }
  if (my_vec >= vecs) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = L > 0.f ? acc[e] / L : 0.f;
  const int64_t final_at = (int64_t)seq * prm.fo_sb + (int64_t)h * prm.fo_sh + d;
  float lse = L > 0.f ? M + logf(L) : -INFINITY;
  if (kRanks == 0 || parts > 1) {
    store_elem4(prm.final_out, final_at, prm.final_dtype, prm.fo_vec, acc);
    if (prm.final_lse && d == 0) prm.final_lse[(int64_t)seq * prm.Hq + h] = lse;
  }
  if constexpr (kRanks != 0) {
    auto value = [&](const piece_t& x, int e) -> float {
      if constexpr (kRanks == 2) return x[e];
      else {
        const uint32_t bits = (uint32_t)x[e >> 1] >> (16 * (e & 1)) & 0xffffu;
        return rk.c.part_dtype == TDIST_BF16 ? bf16_bits_to_f32(bits) : f16_bits_to_f32(bits);
      }
    };
    if (parts == 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = load_elem(prm.final_out, final_at + e, prm.final_dtype);
      lse = prm.final_lse[(int64_t)seq * prm.Hq + h];
    } else if constexpr (kRanks == 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[e] = rk.c.part_dtype == TDIST_BF16 ? bf16_bits_to_f32(f32_to_bf16_bits(acc[e]) & 0xffffu) : f16_bits_to_f32(pack_f16x2(acc[e], 0.f) & 0xffffu);
      }
    }
    const float own_lse = rk.c.lens[(int64_t)rk.own * prm.B + seq] != 0 ? lse : -INFINITY;
    float top = own_lse;
    for (int r0 = 0; r0 < rk.c.P; r0 += kRankBatch) {
      if (r0 > 0) load_ranks(r0);
#pragma unroll
      for (int u = 0; u < kRankBatch; ++u) top = fmaxf(top, rank_lse[u]);
    }
    float sum = 0.f;
    float4v out = {0.f, 0.f, 0.f, 0.f};
    for (int r0 = 0; r0 < rk.c.P; r0 += kRankBatch) {
      if (rk.c.P > kRankBatch) load_ranks(r0);
#pragma unroll
      for (int u = 0; u < kRankBatch; ++u) {
        if (r0 + u >= rk.c.P) break;
        const bool own = r0 + u == rk.own;
        const float at = own ? own_lse : rank_lse[u];
        const float w = at == -INFINITY ? 0.f : __expf(at - top);
        sum += w;
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] += w * (at == -INFINITY ? 0.f : own ? acc[e] : value(rank_x[u], e));
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = sum > 0.f ? out[e] / sum : 0.f;
    store_elem4(rk.c.out, (int64_t)seq * rk.c.o_sb + (int64_t)h * rk.c.o_sh + d, rk.c.out_dtype, rk.out_vec, out);
  }
}

// Ranges per sequence up to which every wave merges its pieces alone (see above): uneven sequences have several times the average.
// 16 sequences up to 4000 keys, 32 / 8 heads, 8 ranges each: 23.4 us a call alone, 22.2 with four waves to a piece; 10 up to 15128 keys 42.3 and
// 40.0; 30, 4.3 ranges each, 70.6 either way. Latent heads have four times the pieces: 12 sequences up to 4096 keys, 5.3 ranges each, 26.7 and 32.8;
// 8 up to 16000 40.1 and 42.9.
constexpr int kAloneMost = 5, kLatentAloneMost = 16;
template <int KEYS, int NW, bool kAlone>
static int launch_merge_cfg(const DecodeParams& prm, hipStream_t stream) {
  const int64_t pieces = ceil_div((int64_t)prm.Hq * (prm.dv / 4), kAlone ? NW * 64 : 64), places = prm.B < prm.ranges ? prm.B : prm.ranges - 1;
  const dim3 grid((unsigned)(places * pieces)), block(NW * 64);
  if (prm.ranks && prm.B < prm.ranges) {
    if (prm.final_dtype == TDIST_F32) hipLaunchKernelGGL((decode_stream_merge_kernel<KEYS, NW, kAlone, 2>), grid, block, 0, stream, prm, *prm.ranks);
    else hipLaunchKernelGGL((decode_stream_merge_kernel<KEYS, NW, kAlone, 1>), grid, block, 0, stream, prm, *prm.ranks);
    return launch_status("tdist_decode_stream");
  }
  hipLaunchKernelGGL((decode_stream_merge_kernel<KEYS, NW, kAlone, 0>), grid, block, 0, stream, prm, NoRanks{});
  if (int rc = launch_status("tdist_decode_stream")) return rc;
  return prm.ranks ? launch_combine(prm.ranks->c, stream) : TDIST_OK;
}
template <int KEYS>
static int launch_stream_merge(const DecodeParams& prm, int alone_most, hipStream_t stream) {
  if (prm.ranges == 1) return prm.ranks ? launch_combine(prm.ranks->c, stream) : TDIST_OK;   // every sequence lies in the one range
  if (prm.ranges <= alone_most * prm.B) return launch_merge_cfg<KEYS, 4, true>(prm, stream);
  return prm.ranges > 4 * kMergeBatch * 4 ? launch_merge_cfg<KEYS, 16, false>(prm, stream) : launch_merge_cfg<KEYS, 4, false>(prm, stream);
}

// Latent attention: blocks of 16 query heads that share a workgroup (a second one is free where the heads fill more than one: the rows
// come in once for both), and the fewest blocks of 32 keys of a range (1 x 1000 keys, 128 heads: 17.0 us with 2, 18.6 with 4, 21.3
// with 8; longer batches have more in any case).
static int latent_head_blocks(int group) { return group <= 16 ? 1 : 2; }
constexpr int kLatentMinBlocks = 2;

// Streaming form: the whole batch in one launch that fills the chip once. All sequences' blocks of KEYS keys are laid
// end to end and cut into equal ranges; a wave takes one kv head (and up to 16 of its query heads) over one range,
// whatever the lengths are. A sequence that lies in one range is finished by its wave; one that is spread over several
// leaves partial results (at most two per range), which the next launch merges (decode_stream_merge_kernel).
// What bounds it: the K/V stream from HBM (B 32, 64 / 8 heads, 32768 keys: 650 us, 6.6 TB/s), and for little work the
// chain lens -> table -> rows -> merge. Against 32 splits per sequence, a combine launch and the form for even lengths behind
// which the other one was queued, whole calls: 48 sequences of 128 to 8192 keys, f16, 64 / 8 heads 205 -> 72-76 us; B 32 x
// 32768 712 -> 661 us (merge with 7 other ranks' partials included). Eight waves of two stages: the same where the stream is long,
// 15 % behind where it is short (B 64 x 256 keys).
template <typename MMA, int D, int DPE, int KEYS, int NW, int NST, bool kSoftCap, bool kPadded>
__global__ __launch_bounds__(NW * 64) void decode_stream_kernel(const DecodeParams prm) {
  const int group = prm.Hq / prm.Hkv;
  if ((int)(blockIdx.x * NW + (threadIdx.x >> 6)) >= prm.ranges * prm.Hkv * ((group + 15) >> 4)) return;
  decode_split_body<MMA, D, DPE, KEYS, NW, NST, kSoftCap, false, kPadded, false, true>(prm);
}

// The same for heads that share one key and whose value is the first 512 of its 576 columns (latent attention). A workgroup
// takes HB blocks of 16 query heads over one range, 32 keys at a time, in two kinds of waves that work side by side, one
// block of keys apart, and meet once per block:
//  * HB waves work out the scores and probabilities of 16 heads each (query in registers, 36 MFMAs and the softmax), so that a
//    head's running maximum and sum concern one wave alone, and leave the probabilities (hi + lo) in the LDS as their lanes
//    hold them, which is the layout that the output product reads;
//  * four waves own 128 value columns of all heads each (a value is read from the LDS once per workgroup) and rescale their sums
//    where a maximum was raised;
//  * two waves bring the rows in: four stages, two blocks in flight.
// The head blocks of a range run on one XCD, whose L2 fetches its rows once.
// What bounds it: at a few blocks per range the launch, the chain lens -> table -> rows -> scores -> output, and the partial
// results (64 KB a workgroup); in a long stream the instructions of a block, about 1 us for 32 keys by 32 heads (0.5 of it beside
// the products: softmax, exchange, meeting), and with up to 32 heads HBM. Whole calls, against 16 heads a workgroup with eight
// waves that each took every fourth block (scores worked out twice, merged through the LDS; 28 % of the LDS cycles lost to bank
// conflicts, none here): 128 / 1 heads, 16 sequences of 64 to 4096 keys 56.6 -> 27.1 us; 16 x 16384 keys 296 -> 144; 64 x 300
// 44 -> 24; 1 x 1000 19.9 -> 17.0; 16 / 1 heads, 16 x 16384 68.5 -> 63 (4.8 TB/s). The output waves bringing the rows in as well:
// 16 x 16384 166 us; 64 heads a workgroup: 132, but twice the partial results (the batch of 16 uneven ones 45 us against 41).
// A score wave shares its SIMD with an output wave and goes first (s_setprio): 16 x 16384 keys 144 -> 130 us, the 16 uneven ones
// 27.5 -> 26.6. What does not bound it: the rows asked for four blocks ahead by a wave of its own (134 us), or two output waves of 256
// columns on the other SIMDs (127, but 38 us for 31.8 where many sequences end: 40 up to 2000 keys).
template <int HB>
struct LatentCfg {
  static constexpr int kKeys = 32, kDK = 576, kDV = 512;
  static constexpr int kLoaders = 2, kThreads = (4 + HB + kLoaders) * 64;
  static constexpr int kSteps = kDK / 32;        // MFMA steps of a score
  static constexpr int kTiles = kDV / 16 / 4;    // tiles of 16 value columns per wave
  static constexpr int kRow = kDV * 2, kPeRow = (kDK - kDV) * 2;
  // rows of a stage: the first 1024 bytes of the keys, which the output product reads a block after the scores, in four places, the
  // other 128 in three
  static constexpr int kStage = kKeys * kRow, kPeStage = kKeys * kPeRow, kStages = 4, kPeStages = 3;
  static constexpr int kPe = kStages * kStage, kProbs = kPe + kPeStages * kPeStage, kProbBlock = HB * 2048;
  static constexpr int kAlpha = kProbs + 2 * kProbBlock, kEnd = kAlpha + 2 * HB * 64, kRaised = kEnd + 2 * HB * 128;
  static constexpr int kTable = kRaised + 32, kTableSlots = 4, kLds = kTable + kTableSlots * kKeys * 4;
  static constexpr int kRows = kKeys / kLoaders, kLoads = kRows + kRows / 8;   // rows of a loading wave per block, and its loads of them
  static_assert(kLds <= 160 * 1024, "LDS of one CU");
  // 16-byte chunk c of a row's first 1024 bytes sits at c ^ swz(key), of the other 128 at c ^ peswz(key). A score's operand read takes
  // one chunk (or, in half of its lanes, the neighbouring one) of 16 keys, a transposing read two neighbouring chunks of 8 keys:
  // both spread over all banks (no conflict by the counter).
  __host__ __device__ static constexpr int swz(int key) { return ((((key & 7) ^ ((key & 8) >> 1)) << 1) | ((key >> 3) & 1)); }
  __device__ static __forceinline__ int peswz(int key) { return (key >> 1) & 7; }
};

template <typename MMA, int HB, bool kSoftCap>
__global__ __launch_bounds__(LatentCfg<HB>::kThreads) void decode_latent_kernel(const DecodeParams prm) {
  typedef LatentCfg<HB> C;
  constexpr int KEYS = C::kKeys, DV = C::kDV;
  typedef TDIST_AS3 unsigned char* lds_u8;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  lds_u8 const lds = (lds_u8)smem;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int x = lane & 15, g = lane >> 4;
  const int group = prm.Hq / prm.Hkv, head_sets = (group + HB * 16 - 1) / (HB * 16);
  const int unit = xcd_major(blockIdx.x, gridDim.x);
  const int range = unit / (prm.Hkv * head_sets), head_unit = unit - range * prm.Hkv * head_sets;
  const int kvh = head_unit / head_sets, first_head = (head_unit - kvh * head_sets) * HB * 16;
  const int h0 = kvh * group + first_head, nvalid = min(HB * 16, group - first_head);

  const StreamRange sr = stream_range<KEYS>(prm, range);
  for (int i0 = 0; range == 0 && i0 < prm.B; i0 += 64) {
    // sequences without keys: out = 0, lse = -inf
    unsigned long long none = __ballot(i0 + lane < prm.B && prm.lens[min(i0 + lane, prm.B - 1)] <= 0);
    for (; none; none &= none - 1) {
      const int seq = i0 + __builtin_ctzll(none);
      for (int j = threadIdx.x; j < nvalid * DV; j += C::kThreads)
        store_elem(prm.final_out, (int64_t)seq * prm.fo_sb + (int64_t)(h0 + j / DV) * prm.fo_sh + j % DV, prm.final_dtype, 0.f);
      if (prm.final_lse && (int)threadIdx.x < nvalid) prm.final_lse[(int64_t)seq * prm.Hq + h0 + threadIdx.x] = -INFINITY;
    }
  }
  if (sr.n == 0) return;

  // blocks of the range in order, across the sequences in it
  const auto lens = (const __attribute__((address_space(4))) int32_t*)(uintptr_t)prm.lens;
  struct Walk { int key0, hi, seq, left, rem; };   // left / rem: blocks of this sequence / of the range, this one included
  auto walk_begin = [&]() {
    const int hi = lens[sr.seq];
    return Walk{sr.block * KEYS, hi, sr.seq, min((hi + KEYS - 1) / KEYS - sr.block, sr.n), sr.n};
  };
  auto walk_next = [&](Walk& w) {   // (stays on the last block)
    if (w.rem == 1) return;
    --w.rem;
    w.key0 += KEYS;
    if (--w.left == 0) {
      do w.hi = lens[++w.seq];
      while (w.hi <= 0);
      w.key0 = 0;
      w.left = min((w.hi + KEYS - 1) / KEYS, w.rem);
    }
  };
  constexpr float kLog2e = 1.4426950408889634f, kLn2 = 0.6931471805599453f;
  TDIST_AS3 float* const s_alpha = (TDIST_AS3 float*)(lds + C::kAlpha);   // [2][HB][16]
  TDIST_AS3 float* const s_end = (TDIST_AS3 float*)(lds + C::kEnd);       // [2][HB][16] pairs: 1 / sum, lse
  TDIST_AS3 int* const s_raised = (TDIST_AS3 int*)(lds + C::kRaised);     // [2][4]
  lds_u8 const s_p = lds + C::kProbs + lane * 16;                         // [2][HB][2 key groups][64]
  // Step s: the scores of block s and the output product of block s - 1. Blocks 0 .. n - 1, steps 0 .. n: every wave meets n + 1 times.
  if (wave >= 4 && wave < 4 + HB) {
    __builtin_amdgcn_s_setprio(2);   // (ahead of the output wave on the same SIMD: a block's time is this wave's chain)
    const int hb = wave - 4;
    const float scale_log2 = prm.sm_scale * kLog2e;
    // query: head x, columns 32s + 8g .. + 7; operand reads relative to the stage: chunk 4s + g of key x
    typename MMA::frag8 qf[C::kSteps];
    const int h = min(hb * 16 + x, nvalid - 1);
    int koff[4], peoff[2];
#pragma unroll
    for (int s = 0; s < 4; ++s) koff[s] = x * C::kRow + (((4 * s + g) ^ C::swz(x)) << 4);
#pragma unroll
    for (int s = 0; s < 2; ++s) peoff[s] = x * C::kPeRow + (((4 * s + g) ^ C::peswz(x)) << 4);
    float m_run = -INFINITY, l_run = 0.f;   // log2 domain; the sum over this lane's keys
    bool begins = true;
    Walk w = walk_begin();
    for (int i = 0; i < sr.n; ++i) {
      if (begins) {
        const unsigned char* row = prm.q + (int64_t)w.seq * prm.q_sb + (int64_t)(h0 + h) * prm.q_sh + 16 * g;
#pragma unroll
        for (int s = 0; s < C::kSteps; ++s) qf[s] = __builtin_bit_cast(typename MMA::frag8, *(const int4v*)(row + 64 * s));
        m_run = -INFINITY;
        l_run = 0.f;
        begins = false;
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      lds_u8 const st = lds + (i & 3) * C::kStage, pe = lds + C::kPe + i % 3 * C::kPeStage;
      // four chains of products: sc[q], sc[2 + q] for key group q
      float4v sc[4] = {float4v{0.f, 0.f, 0.f, 0.f}, float4v{0.f, 0.f, 0.f, 0.f}, float4v{0.f, 0.f, 0.f, 0.f}, float4v{0.f, 0.f, 0.f, 0.f}};
      // operand n (step n / 2, key group n % 2) is read kAhead products before its own: a step's time is this chain's
      constexpr int kAhead = 12;
      int4v kb[kAhead];
      auto read_k = [&](int n) {
        const int u = n >> 1, q = n & 1;
        return *(const TDIST_AS3 int4v*)(u < 16 ? st + koff[u & 3] + (u >> 2) * 256 + q * 16 * C::kRow : pe + peoff[u & 1] + q * 16 * C::kPeRow);
      };
#pragma unroll
      for (int n = 0; n < kAhead; ++n) kb[n] = read_k(n);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < 2 * C::kSteps; ++n) {
        sc[n & 3] = MMA::mma32(__builtin_bit_cast(typename MMA::frag8, kb[n % kAhead]), qf[n >> 1], sc[n & 3]);
        if (n + kAhead < 2 * C::kSteps) kb[n % kAhead] = read_k(n + kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
      sc[0] += sc[2];
      sc[1] += sc[3];
      // sc[q][e]: key 16q + 4g + e, head x
      float t[2][4], mx = -INFINITY;
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          t[q][e] = kSoftCap ? prm.soft_cap * tanhf(sc[q][e] * prm.sm_scale / prm.soft_cap) * kLog2e : sc[q][e] * scale_log2;
      if (w.key0 + KEYS > w.hi) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int e = 0; e < 4; ++e) t[q][e] = w.key0 + 16 * q + 4 * g + e < w.hi ? t[q][e] : -INFINITY;
      }
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) mx = fmaxf(mx, t[q][e]);
      // The sums are kept relative to m_run, which is raised only when a score lies kSlack above it: their values then stay
      // below 2^kSlack, which costs no precision, and are rescaled a few times per stream instead of per block.
      constexpr float kSlack = 8.f;
      const int raised = __any(mx > m_run + kSlack);
      if (raised) {
        mx = max_lane_xor<32>(max_lane_xor<16>(mx));
        const float m_new = fmaxf(m_run, mx);
        const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_new);
        if (g == 0) s_alpha[((i & 1) * HB + hb) * 16 + x] = alpha;
        l_run *= alpha;
        m_run = m_new;
      }
      if (lane == 0) s_raised[(i & 1) * 4 + hb] = raised;
      const float m_safe = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        float p[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          p[e] = __builtin_amdgcn_exp2f(t[q][e] - m_safe);
          l_run += p[e];
        }
        uint32_t hi[2], lo[2];
        MMA::split(p[0], p[1], hi[0], lo[0]);
        MMA::split(p[2], p[3], hi[1], lo[1]);
        *(TDIST_AS3 int4v*)(s_p + (i & 1) * C::kProbBlock + hb * 2048 + q * 1024) = int4v{(int)hi[0], (int)hi[1], (int)lo[0], (int)lo[1]};
      }
      if (w.left == 1) {
        // the sequence's last block in this range
        const float L = sum_lane_xor<32>(sum_lane_xor<16>(l_run));
        if (g == 0) {
          TDIST_AS3 float* e = s_end + (((i & 1) * HB + hb) * 16 + x) * 2;
          // (a sum that is no number stays one, also as an LSE: -inf would take the sequence for one without keys)
          e[0] = L != 0.f ? 1.f / L : 0.f;
          e[1] = L != 0.f ? (m_run + log2f(L)) * kLn2 : -INFINITY;
        }
        begins = true;
      }
      walk_next(w);
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    return;
  }

  if (wave >= 4 + HB) {
    // Half of a block's rows each; four lanes work out the place of one. Keys behind the end are read as the last one (their
    // probabilities are 0).
    const int first = (wave - 4 - HB) * C::kRows;
    lds_u8 const table = lds + C::kTable + first * 4;
    auto page_slot = [&](uint32_t n) { return (uint32_t)(((uint64_t)n * prm.page_magic) >> prm.page_shift); };
    auto issue_table = [&](int j, const Walk& w) {
      if (lane < C::kRows) {
        const uint32_t n = (uint32_t)min(w.key0 + first + lane, w.hi - 1);
        __builtin_amdgcn_global_load_lds((const TDIST_AS1 void*)(prm.table + (int64_t)w.seq * prm.t_s + page_slot(n)),
                                         (TDIST_AS3 void*)(table + j % C::kTableSlots * (KEYS * 4)), 4, 0, 0);
      }
    };
    auto issue_rows = [&](int j, const Walk& w) {
      const int mine = lane / (64 / C::kRows);
      const uint32_t n = (uint32_t)min(w.key0 + first + mine, w.hi - 1), in_page = n - page_slot(n) * (uint32_t)prm.page_size;
      const uint32_t page = (uint32_t)((const volatile TDIST_AS3 int32_t*)(table + j % C::kTableSlots * (KEYS * 4)))[mine];
      const uint64_t row = (uint64_t)(uintptr_t)prm.k + (uint64_t)page * (uint64_t)prm.k_sp + (in_page * (uint32_t)prm.k_st + (uint32_t)kvh * (uint32_t)prm.k_sh);
      const uint32_t row_lo = (uint32_t)row, row_hi = (uint32_t)(row >> 32);
      lds_u8 const st = lds + (j & 3) * C::kStage + first * C::kRow, pe = lds + C::kPe + j % 3 * C::kPeStage + first * C::kPeRow;
      // (a lane number that the compiler takes for a new one: offsets kept from block to block would be added as 64-bit vectors)
      int l = lane;
      asm volatile("" : "+v"(l));
#pragma unroll
      for (int u = 0; u < C::kRows; ++u) {
        const uint64_t at = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)row_hi, u * (64 / C::kRows)) << 32) |
                            (uint32_t)__builtin_amdgcn_readlane((int)row_lo, u * (64 / C::kRows));
        __builtin_amdgcn_global_load_lds((const TDIST_AS1 void*)((const unsigned char*)(uintptr_t)at + (uint32_t)((l ^ C::swz(u & 15)) << 4)),
                                         (TDIST_AS3 void*)(st + u * C::kRow), 16, 0, 0);
      }
#pragma unroll
      for (int u = 0; u < C::kRows / 8; ++u) {
        const int key = u * 8 + (l >> 3);
        const uint32_t lo = (uint32_t)__shfl((int)row_lo, key * (64 / C::kRows)), hi = (uint32_t)__shfl((int)row_hi, key * (64 / C::kRows));
        const uint64_t at = ((uint64_t)hi << 32) | lo;
        __builtin_amdgcn_global_load_lds((const TDIST_AS1 void*)((const unsigned char*)(uintptr_t)at + (uint32_t)(C::kRow + (((l & 7) ^ C::peswz(key)) << 4))),
                                         (TDIST_AS3 void*)(pe + u * 1024), 16, 0, 0);
      }
    };
    static_assert(C::kRows % 16 == 0, "a wave's rows begin a group of 16");
    Walk w_table = walk_begin(), w_rows = w_table;
    for (int j = 0; j < C::kTableSlots; ++j) {
      issue_table(j, w_table);
      walk_next(w_table);
    }
    wait_vmcnt<0>();
    for (int j = 0; j < 2 && j < sr.n; ++j) {
      issue_rows(j, w_rows);
      walk_next(w_rows);
    }
    for (int s = 0; s <= sr.n; ++s) {
      // block s has landed (and with it the table of block s + 2, which was fetched before); block s + 1 may be on its way
      if (s + 1 < sr.n) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(C::kLoads) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (s + 2 < sr.n) {
        issue_table(s + 4, w_table);
        walk_next(w_table);
        issue_rows(s + 2, w_rows);
        walk_next(w_rows);
      }
    }
    return;
  }

  // transposing reads relative to the stage: chunks of tile d in keys 4g + x / 4
  int voff[C::kTiles];
#pragma unroll
  for (int d = 0; d < C::kTiles; ++d) {
    const int key = 4 * g + (x >> 2);
    voff[d] = key * C::kRow + wave * 256 + (((2 * d + ((x & 3) >> 1)) ^ C::swz(key)) << 4) + (x & 1) * 8;
  }
  static_assert(C::kTiles == 8, "a wave's value columns are one window of 16 chunks");
  float4v acc[C::kTiles][HB];   // value columns wave * 128 + 16d + 4g .. + 3 of head b * 16 + x
  auto reset = [&]() {
#pragma unroll
    for (int d = 0; d < C::kTiles; ++d)
#pragma unroll
      for (int b = 0; b < HB; ++b) acc[d][b] = float4v{0.f, 0.f, 0.f, 0.f};
  };
  reset();

  Walk w_out = walk_begin();
  bool begun_here = sr.block == 0;
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  for (int j = 0; j < sr.n; ++j) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int par = j & 1;
    const uint32_t v_base = (uint32_t)(uintptr_t)(lds + (j & 3) * C::kStage);
    // The transposing reads and the waits for them are written out: for the builtin the compiler waits until every load
    // into the LDS is done, the ones in flight for later blocks included.
    constexpr int kAhead = 6;
    int2v vb[kAhead][2];
    auto read_v = [&](int d) {
      const uint32_t at = v_base + (uint32_t)voff[d];
      asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(vb[d % kAhead][0]) : "v"(at) : "memory");
      asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(vb[d % kAhead][1]) : "v"(at), "n"(16 * C::kRow) : "memory");
    };
    const int4v raised = *(const TDIST_AS3 int4v*)(s_raised + par * 4);
    int4v pa[HB], pc[HB];
#pragma unroll
    for (int b = 0; b < HB; ++b) {
      pa[b] = *(const TDIST_AS3 int4v*)(s_p + par * C::kProbBlock + b * 2048);
      pc[b] = *(const TDIST_AS3 int4v*)(s_p + par * C::kProbBlock + b * 2048 + 1024);
    }
    int any = raised[0];
#pragma unroll
    for (int b = 1; b < HB; ++b) any |= raised[b];
    if (__builtin_amdgcn_readfirstlane(any)) {
#pragma unroll
      for (int b = 0; b < HB; ++b) {
        const float alpha = __builtin_amdgcn_readfirstlane(raised[b]) ? s_alpha[(par * HB + b) * 16 + x] : 1.f;
#pragma unroll
        for (int d = 0; d < C::kTiles; ++d) acc[d][b] *= alpha;
      }
    }
    int4v ph[HB], pl[HB];
#pragma unroll
    for (int b = 0; b < HB; ++b) {
      ph[b] = int4v{pa[b][0], pa[b][1], pc[b][0], pc[b][1]};
      pl[b] = int4v{pa[b][2], pa[b][3], pc[b][2], pc[b][3]};
    }
#pragma unroll
    for (int d = 0; d < kAhead; ++d) read_v(d);
    static_for<C::kTiles>([&](auto tile) {
      constexpr int d = decltype(tile)::value, later = C::kTiles - 1 - d;   // tiles read behind this one
      asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(2 * (later < kAhead - 1 ? later : kAhead - 1)) : "memory");
      int2v(&v)[2] = vb[d % kAhead];
      asm volatile("" : "+v"(v[0]), "+v"(v[1]));
      const typename MMA::frag8 vf = __builtin_bit_cast(typename MMA::frag8, int4v{v[0][0], v[0][1], v[1][0], v[1][1]});
#pragma unroll
      for (int b = 0; b < HB; ++b) acc[d][b] = MMA::mma32(vf, __builtin_bit_cast(typename MMA::frag8, ph[b]), acc[d][b]);
#pragma unroll
      for (int b = 0; b < HB; ++b) acc[d][b] = MMA::mma32(vf, __builtin_bit_cast(typename MMA::frag8, pl[b]), acc[d][b]);
      if constexpr (d + kAhead < C::kTiles) read_v(d + kAhead);
    });

    if (w_out.left == 1) {
      // the sequence's last block in this range: its result, or its part of it
      const bool whole = begun_here && w_out.key0 + KEYS >= w_out.hi;
      const int64_t part = ((int64_t)range * 2 + (begun_here ? 1 : 0)) * prm.Hq + h0;
#pragma unroll
      for (int b = 0; b < HB; ++b) {
        const TDIST_AS3 float* e = s_end + ((par * HB + b) * 16 + x) * 2;
        const float inv = e[0], lse = e[1];
        const int h = b * 16 + x, col = wave * 128 + 4 * g;
        if (h < nvalid) {
          if (whole) {
            const int64_t o = (int64_t)w_out.seq * prm.fo_sb + (int64_t)(h0 + h) * prm.fo_sh + col;
#pragma unroll
            for (int d = 0; d < C::kTiles; ++d) store_elem4(prm.final_out, o + 16 * d, prm.final_dtype, prm.fo_vec, acc[d][b] * inv);
            if (prm.final_lse && wave == 0 && g == 0) prm.final_lse[(int64_t)w_out.seq * prm.Hq + h0 + h] = lse;
          } else {
            float* o = prm.out + (part + b * 16) * DV;
#pragma unroll
            for (int d = 0; d < C::kTiles; ++d) store_partial4<true>(o + partial_tile(min(16, nvalid - b * 16), DV, wave * C::kTiles + d, x, g), acc[d][b] * inv);
            if (wave == 0 && g == 0) store_partial<true>(prm.lse + part + h, lse);
          }
        }
      }
      begun_here = true;
      reset();
    }
    walk_next(w_out);
  }
}

template <typename MMA, int HB, bool kSoftCap>
static int launch_latent_cfg(DecodeParams& prm, hipStream_t stream) {
  typedef LatentCfg<HB> C;
  auto kern = decode_latent_kernel<MMA, HB, kSoftCap>;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::kLds);
    if (e != hipSuccess) return fail(TDIST_ERR_LAUNCH, "decode: cannot reserve %d B of LDS: %s", C::kLds, hipGetErrorString(e));
    attr_set = true;
  }
  prm.min_blocks = kLatentMinBlocks;
  const int64_t sets = ceil_div(prm.Hq / prm.Hkv, HB * 16);
  hipLaunchKernelGGL(kern, dim3((unsigned)((int64_t)prm.ranges * prm.Hkv * sets)), dim3(C::kThreads), C::kLds, stream, prm);
  if (int rc = launch_status("tdist_decode_stream")) return rc;
  return launch_stream_merge<C::kKeys>(prm, kLatentAloneMost, stream);
}

template <typename MMA>
static int launch_latent(DecodeParams& prm, hipStream_t stream) {
  const bool few = latent_head_blocks(prm.Hq / prm.Hkv) == 1;
  if (prm.soft_cap > 0.f) return few ? launch_latent_cfg<MMA, 1, true>(prm, stream) : launch_latent_cfg<MMA, 2, true>(prm, stream);
  return few ? launch_latent_cfg<MMA, 1, false>(prm, stream) : launch_latent_cfg<MMA, 2, false>(prm, stream);
}

template <typename MMA, int D, int DPE, int KEYS, int NW, int NST, bool kSoftCap, bool kPadded>
static int launch_stream_cfg(DecodeParams& prm, int head_blocks, hipStream_t stream) {
  typedef DecodeCfg<D, DPE, KEYS, NST> C;
  const size_t lds = (size_t)NW * C::kWaveBytes;
  static_assert((size_t)NW * C::kWaveBytes <= 160 * 1024, "LDS of one CU");
  auto kern = decode_stream_kernel<MMA, D, DPE, KEYS, NW, NST, kSoftCap, kPadded>;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return fail(TDIST_ERR_LAUNCH, "decode: cannot reserve %zu B of LDS: %s", lds, hipGetErrorString(e));
    attr_set = true;
  }
  // The fewest keys of a range: half of them in one wave are a shorter chain, twice the partial results are a little more to merge (launches of 1 x 1320
  // keys, 32 / 8 heads: 64 keys 9.8 + 3.9 us, 32 7.5 + 4.6, 16 6.5 + 6.4; 2 x up to 1679 of 256-wide heads 16.2 + 4.0, 12.2 + 4.2, 10.3 + 6.6; 20 x up to 400
  // 12.8 + 4.5, 9.2 + 5.1, 9.4 + 5.1).
  prm.min_blocks = 32 / KEYS;
  const int64_t waves = (int64_t)prm.ranges * prm.Hkv * head_blocks;
  hipLaunchKernelGGL(kern, dim3((unsigned)((waves + NW - 1) / NW)), dim3(NW * 64), lds, stream, prm);
  if (int rc = launch_status("tdist_decode_stream")) return rc;
  return launch_stream_merge<KEYS>(prm, kAloneMost, stream);
}

template <typename MMA, int D, int DPE, int KEYS, int NW, int NST, bool kPadded>
static int launch_stream(DecodeParams& prm, int head_blocks, hipStream_t stream) {
  return prm.soft_cap > 0.f ? launch_stream_cfg<MMA, D, DPE, KEYS, NW, NST, true, kPadded>(prm, head_blocks, stream)
                            : launch_stream_cfg<MMA, D, DPE, KEYS, NW, NST, false, kPadded>(prm, head_blocks, stream);
}

template <typename MMA, int D, int DPE, int KEYS, int NW, int NST, bool kPadded = false>
static int launch_decode(const DecodeParams& prm, int head_blocks, hipStream_t stream) {
  const bool fuse = prm.counters != nullptr;
  if (prm.soft_cap > 0.f)
    return fuse ? launch_decode_cfg<MMA, D, DPE, KEYS, NW, NST, true, true, kPadded>(prm, head_blocks, stream)
                : launch_decode_cfg<MMA, D, DPE, KEYS, NW, NST, true, false, kPadded>(prm, head_blocks, stream);
  return fuse ? launch_decode_cfg<MMA, D, DPE, KEYS, NW, NST, false, true, kPadded>(prm, head_blocks, stream)
              : launch_decode_cfg<MMA, D, DPE, KEYS, NW, NST, false, false, kPadded>(prm, head_blocks, stream);
}

}  // namespace tdist

using namespace tdist;

namespace tdist {

struct DecodeCall {
  const void *q, *k_cache, *v_cache;
  float *out_split, *lse_split;
  float sm_scale, soft_cap;
  const int32_t *block_table, *kv_lens;
  int batch, q_heads, kv_heads, head_dim, head_dim_v, page_size, num_splits;
  int64_t q_stride_b, q_stride_h, k_stride_page, k_stride_token, k_stride_head, v_stride_page, v_stride_token,
      v_stride_head, table_stride;
  int dtype;
  // fused merge
  int32_t* counters;
  int64_t n_counters;
  void* out;
  int out_dtype;
  int64_t out_stride_b, out_stride_h;
  float* lse_out;
  void* stream;
  const char* who;
  // streaming form
  void* workspace;
  int64_t workspace_bytes;
  const RankParams* ranks = nullptr;
};

enum DecodeForm { kFormSplit, kFormFused, kFormStream };

static int64_t decode_fused_counters(int batch, int q_heads, int kv_heads) {
  if (batch <= 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0) return -1;
  const int group = q_heads / kv_heads;
  return (int64_t)batch * kv_heads * ((group + 15) / 16);
}

// Streaming form: how many ranges the batch is cut into. `units` waves (kv heads x blocks of query heads) share a
// range, and `slots` waves are resident at a time: as many ranges as fill them once, or, where the units alone nearly
// fill or overfill them, the number of ranges whose last round of waves is the fullest.
static int stream_ranges(int64_t units, int64_t slots) {
  if (units * 4 <= slots) return (int)(slots / units);
  int best = 1;
  double best_cost = 0;
  for (int r = 1; r <= 16; ++r) {
    const double cost = (double)((units * r + slots - 1) / slots) / r;
    if (r == 1 || cost < best_cost * 0.97) best_cost = cost, best = r;
  }
  return best;
}
// Ranges for a call, given its head counts and key dimension. Four waves with rings of up to four stages per compute unit (as much
// in flight as eight waves of two, half the fixed work and half the partial results), a kv head and a block of 16 query heads each;
// or, for latent attention, a workgroup per compute unit with a set of head blocks. With two blocks in a set that is twice the
// ranges, and twice the workspace, of one block per workgroup (128 / 1 heads: 64 ranges, 33.6 MB); a caller who comes with the room
// for `fewest`, as many as there were with one block, gets that many (16 sequences up to 4096 keys 41.5 us a call, 32.6 with 64).
static int stream_ranges_for(int q_heads, int kv_heads, int head_dim, bool fewest = false) {
  const int group = q_heads / kv_heads, cus = device_info().num_cus > 0 ? device_info().num_cus : 256;
  if (head_dim > 256) return stream_ranges((int64_t)kv_heads * ceil_div(group, 16 * (fewest ? 1 : latent_head_blocks(group))), 1ll * cus);
  return stream_ranges((int64_t)kv_heads * ceil_div(group, 16), 4ll * cus);
}
// two partial results per range: rows of head_dim_v floats and one LSE per query head
static int64_t partials_bytes(int ranges, int q_heads, int head_dim_v) { return 2ll * ranges * q_heads * (head_dim_v + 1) * 4; }
static int64_t stream_workspace_bytes(int batch, int q_heads, int kv_heads, int head_dim, int head_dim_v) {
  if (batch <= 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0 || head_dim_v <= 0) return -1;
  return partials_bytes(stream_ranges_for(q_heads, kv_heads, head_dim), q_heads, head_dim_v);
}

static int run_decode(const DecodeCall& c, DecodeForm form) {
  const char* who = c.who;
  const bool whole = form != kFormSplit;   // the call's output is the merged result
  const bool fuse = form == kFormFused;
  if (!c.q || !c.k_cache || !c.v_cache || !c.block_table || !c.kv_lens ||
      (form == kFormStream ? !c.workspace : !c.out_split || !c.lse_split))
    return fail(TDIST_ERR_INVALID, "%s: null pointer", who);
  if (c.batch <= 0 || c.q_heads <= 0 || c.kv_heads <= 0 || c.page_size <= 0 || c.num_splits <= 0)
    return fail(TDIST_ERR_INVALID, "%s: sizes must be positive", who);
  if (c.q_heads % c.kv_heads != 0)
    return fail(TDIST_ERR_INVALID, "%s: q_heads %d not a multiple of kv_heads %d", who, c.q_heads, c.kv_heads);
  if (c.dtype != TDIST_BF16 && c.dtype != TDIST_F16)
    return fail(TDIST_ERR_UNSUPPORTED, "%s: dtype %d (bf16 and f16 only)", who, c.dtype);
  const int dk = c.head_dim, dv = c.head_dim_v;
  const bool padded = dk == dv && dk > 0 && dk < 256 && dk % 8 == 0 && dk != 64 && dk != 128;
  const bool dims_ok = (dk == dv && (dk == 64 || dk == 128 || dk == 256)) || (dk == 192 && dv == 128) ||
                       (dk == 576 && dv == 512) || padded;
  if (!dims_ok)
    return fail(TDIST_ERR_UNSUPPORTED, "%s: head dims (%d, %d): equal ones that are a multiple of 8 up to 256, (192,128) "
                "and (576,512) only", who, dk, dv);
  if (!aligned16(c.q) || !aligned16(c.k_cache) || !aligned16(c.v_cache) || (c.q_stride_b % 8) || (c.q_stride_h % 8) ||
      (c.k_stride_page % 8) || (c.k_stride_token % 8) || (c.k_stride_head % 8) || (c.v_stride_page % 8) ||
      (c.v_stride_token % 8) || (c.v_stride_head % 8))
    return fail(TDIST_ERR_UNSUPPORTED, "%s: q/k/v rows must be 16-byte aligned", who);
  if (c.num_splits > 65535 || c.batch > 65535) return fail(TDIST_ERR_UNSUPPORTED, "%s: grid too large", who);
  DecodeParams prm;
  prm.q = (const unsigned char*)c.q;
  prm.k = (const unsigned char*)c.k_cache;
  prm.v = (const unsigned char*)c.v_cache;
  prm.out = c.out_split;
  prm.lse = c.lse_split;
  prm.table = c.block_table;
  prm.lens = c.kv_lens;
  prm.sm_scale = c.sm_scale;
  prm.soft_cap = c.soft_cap;
  prm.B = c.batch;
  prm.Hq = c.q_heads;
  prm.Hkv = c.kv_heads;
  prm.S = c.num_splits;
  prm.dv = dv;
  prm.d_valid = dk;
  prm.part_vec = aligned16(c.out_split);
  prm.splits_per_team = 1;
  prm.when_lens = 0;
  prm.page_size = c.page_size;
  int lg = 0;
  while ((1ll << lg) < c.page_size) ++lg;
  prm.page_shift = 31 + lg;
  prm.page_magic = ((1ull << prm.page_shift) + (uint64_t)c.page_size - 1) / (uint64_t)c.page_size;
  prm.q_sb = c.q_stride_b * 2;
  prm.q_sh = c.q_stride_h * 2;
  prm.k_sp = c.k_stride_page * 2;
  prm.k_st = c.k_stride_token * 2;
  prm.k_sh = c.k_stride_head * 2;
  prm.v_sp = c.v_stride_page * 2;
  prm.v_st = c.v_stride_token * 2;
  prm.v_sh = c.v_stride_head * 2;
  prm.t_s = c.table_stride;
  prm.ranks = c.ranks;
  prm.counters = nullptr;
  prm.final_out = nullptr;
  prm.final_lse = nullptr;
  prm.final_dtype = TDIST_F32;
  prm.fo_sb = prm.fo_sh = 0;
  if (whole) {
    if ((fuse && !c.counters) || !c.out) return fail(TDIST_ERR_INVALID, "%s: null counters or output", who);
    if (!aligned16(form == kFormStream ? c.workspace : c.out_split))
      return fail(TDIST_ERR_UNSUPPORTED, "%s: %s must be 16-byte aligned", who, form == kFormStream ? "workspace" : "out_split");
    if (c.out_dtype != TDIST_F32 && c.out_dtype != TDIST_BF16 && c.out_dtype != TDIST_F16)
      return fail(TDIST_ERR_UNSUPPORTED, "%s: output dtype %d", who, c.out_dtype);
    if (fuse) {
      const int64_t need = decode_fused_counters(c.batch, c.q_heads, c.kv_heads);
      if (c.n_counters < need)
        return fail(TDIST_ERR_WORKSPACE, "%s: %lld counters given, %lld needed", who, (long long)c.n_counters, (long long)need);
      prm.counters = c.counters;
    }
    prm.final_out = (unsigned char*)c.out;
    prm.final_lse = c.lse_out;
    prm.final_dtype = c.out_dtype;
    prm.fo_sb = c.out_stride_b;
    prm.fo_sh = c.out_stride_h;
    const int esz = c.out_dtype == TDIST_F32 ? 4 : 2;
    prm.fo_vec = ((uintptr_t)c.out % (4 * esz)) == 0 && c.out_stride_b % 4 == 0 && c.out_stride_h % 4 == 0;
  }
  const int group = c.q_heads / c.kv_heads;
  const int head_blocks = (group + 15) / 16;
  if ((int64_t)c.kv_heads * head_blocks > 65535) return fail(TDIST_ERR_UNSUPPORTED, "%s: too many heads", who);
  hipStream_t st = (hipStream_t)c.stream;
  const bool bf = c.dtype == TDIST_BF16;
  if (form == kFormStream) {
    const bool latent = c.v_cache == c.k_cache && prm.v_sp == prm.k_sp && prm.v_st == prm.k_st && (prm.v_sh == prm.k_sh || c.kv_heads == 1);
    if (dk > 256 && !latent)
      return fail(TDIST_ERR_UNSUPPORTED, "%s: head dims (%d, %d) with a value that is no part of the key", who, dk, dv);
    prm.ranges = stream_ranges_for(c.q_heads, c.kv_heads, dk);
    if (c.workspace_bytes < partials_bytes(prm.ranges, c.q_heads, dv)) {
      const int fewest = stream_ranges_for(c.q_heads, c.kv_heads, dk, true);
      if (fewest >= prm.ranges || c.workspace_bytes < partials_bytes(fewest, c.q_heads, dv))
        return fail(TDIST_ERR_WORKSPACE, "%s: %lld bytes of workspace given, %lld needed", who, (long long)c.workspace_bytes,
                    (long long)partials_bytes(prm.ranges, c.q_heads, dv));
      prm.ranges = fewest;
    }
    prm.out = (float*)c.workspace;
    prm.lse = prm.out + 2ll * prm.ranges * c.q_heads * dv;
#define TDIST_STREAM(D_, DPE_, KEYS_, NW_, NST_, PAD_)                                                \
  return bf ? launch_stream<MmaBF16, D_, DPE_, KEYS_, NW_, NST_, PAD_>(prm, head_blocks, st)         \
            : launch_stream<MmaF16, D_, DPE_, KEYS_, NW_, NST_, PAD_>(prm, head_blocks, st);
    if (dk > 256) return bf ? launch_latent<MmaBF16>(prm, st) : launch_latent<MmaF16>(prm, st);
    if (dk == 64) TDIST_STREAM(64, 0, 32, 4, 4, false)
    if (dk == 128) TDIST_STREAM(128, 0, 16, 4, 4, false)
    if (dk == 192 && dv == 128) TDIST_STREAM(128, 64, 16, 4, 3, false)
    if (dk == 256) TDIST_STREAM(256, 0, 16, 4, 2, false)
    if (dk < 64) TDIST_STREAM(64, 0, 32, 4, 4, true)
    if (dk < 128) TDIST_STREAM(128, 0, 16, 4, 4, true)
    TDIST_STREAM(256, 0, 16, 4, 2, true)
#undef TDIST_STREAM
  }
  // <dtype, Dv, extra key dims, keys per block, waves, stages>:
  // LDS = waves * (stages * keys * (Dk + Dv) * 2 B + tables) <= 160 KB
#define TDIST_DEC(D_, DPE_, KEYS_, NW_, NST_)                                             \
  return bf ? launch_decode<MmaBF16, D_, DPE_, KEYS_, NW_, NST_>(prm, head_blocks, st)   \
            : launch_decode<MmaF16, D_, DPE_, KEYS_, NW_, NST_>(prm, head_blocks, st);
#define TDIST_DEC_PADDED(D_, KEYS_, NW_, NST_)                                                 \
  return bf ? launch_decode<MmaBF16, D_, 0, KEYS_, NW_, NST_, true>(prm, head_blocks, st)     \
            : launch_decode<MmaF16, D_, 0, KEYS_, NW_, NST_, true>(prm, head_blocks, st);
  // A kv head per wave (8 waves of 2 stages or 4 waves of 4, 130-136 KB: one workgroup per CU) where the heads allow
  // it, the grid fills the CUs in whole rounds or in many (such a workgroup is NW_ times the work of one of the other
  // form, whose small workgroups fill a small grid's CUs better) and the cache is large enough for a tenth of the
  // kernel's time to outweigh a second launch: the form's time goes with the longest sequence, so the other form is
  // launched behind it and the kernels decide by the sequence lengths which of the two runs (decode_lens_even).
  // tdist_debug_set(TDIST_DEBUG_DECODE_WAVE_HEADS, 0) never takes this form; 2 takes it wherever the heads allow it,
  // alone and whatever the lengths; 4 likewise but only its 4-wave workgroups.
  const int wh_dbg = debug_get(TDIST_DEBUG_DECODE_WAVE_HEADS);
  const int wh_mode = wh_dbg >= 0 ? wh_dbg : 1;
  auto wave_heads = [&](int nw) {
    if (wh_mode == 0 || head_blocks != 1 || c.kv_heads % nw != 0 || (wh_mode == 4 && nw != 4)) return false;
    if (!aligned16(c.out_split)) return false;   // its partial results go out as 16-byte vectors
    // Splits per workgroup: the count that needs the least time in units of (one split on every CU): rounds of
    // workgroups x splits in each; of equal ones the larger, which starts fewer workgroups.
    const int64_t heads_seqs = (int64_t)(c.kv_heads / nw) * c.batch;
    const int cus = device_info().num_cus > 0 ? device_info().num_cus : 256;
    int64_t best_cost = 0;
    int best_w = 1;
    const int max_w = std::min(c.num_splits, decode_max_splits_per_team(dv, c.soft_cap > 0.f || fuse || padded));
    for (int w = 1; w <= max_w; ++w) {
      const int64_t teams = heads_seqs * ((c.num_splits + w - 1) / w);
      const int64_t cost = ((teams + cus - 1) / cus) * w;
      if (w == 1 || cost <= best_cost) best_cost = cost, best_w = w;
    }
    const int spt = debug_get(TDIST_DEBUG_DECODE_SPLITS_PER_TEAM);
    if (spt >= 1) best_w = std::min(spt, max_w);
    prm.splits_per_team = best_w;
    if (wh_mode > 1) return true;
    // the most that the block table lets the call read: below 256 MB (40 us) the form's gain is less than a launch
    const double cap_bytes = (double)c.batch * c.kv_heads * (double)c.table_stride * c.page_size * (dk + dv) * 2.0;
    if (cap_bytes < 256e6) return false;
    // against the time that work spread evenly over the CUs would need: at most a third more
    return best_cost * cus * 3 <= heads_seqs * c.num_splits * 4;
  };
#define TDIST_DEC_WH_(MMA_, D_, KEYS_, NW_, NST_, CAP_, FUSE_, PAD_) \
  launch_decode_cfg<MMA_, D_, 0, KEYS_, NW_, NST_, CAP_, FUSE_, PAD_, true>(prm, head_blocks, st)
#define TDIST_DEC_WH(D_, KEYS_, NW_, NST_) TDIST_DEC_WH_P(D_, KEYS_, NW_, NST_, false)
#define TDIST_DEC_WH_P(D_, KEYS_, NW_, NST_, PAD_)                                                                      \
  if (prm.when_lens == 0 && wave_heads(NW_)) {                                                                       \
    /* chosen for the grid: it runs if the sequence lengths are even, and the other form, launched behind it, if   \
       they are not (forced by the environment: unconditionally, alone) */                                          \
    prm.when_lens = (wh_mode > 1 || c.batch == 1) ? 0 : 1;   /* (one sequence: even by definition) */               \
    int rc_;                                                                                                         \
    if (prm.soft_cap > 0.f) {                                                                                        \
      if (fuse) rc_ = bf ? TDIST_DEC_WH_(MmaBF16, D_, KEYS_, NW_, NST_, true, true, PAD_) : TDIST_DEC_WH_(MmaF16, D_, KEYS_, NW_, NST_, true, true, PAD_);     \
      else rc_ = bf ? TDIST_DEC_WH_(MmaBF16, D_, KEYS_, NW_, NST_, true, false, PAD_) : TDIST_DEC_WH_(MmaF16, D_, KEYS_, NW_, NST_, true, false, PAD_);         \
    } else {                                                                                                         \
      if (fuse) rc_ = bf ? TDIST_DEC_WH_(MmaBF16, D_, KEYS_, NW_, NST_, false, true, PAD_) : TDIST_DEC_WH_(MmaF16, D_, KEYS_, NW_, NST_, false, true, PAD_);   \
      else rc_ = bf ? TDIST_DEC_WH_(MmaBF16, D_, KEYS_, NW_, NST_, false, false, PAD_) : TDIST_DEC_WH_(MmaF16, D_, KEYS_, NW_, NST_, false, false, PAD_);       \
    }                                                                                                                \
    if (rc_ != TDIST_OK || prm.when_lens == 0) return rc_;                                                           \
    prm.when_lens = 2;                                                                                               \
  }
  if (padded) {
    // any other head dimension: the shape of the next power of two, rows filled up with zeros on their way in
    if (dk < 64) TDIST_DEC_PADDED(64, 32, 4, 4)
    if (dk < 128) {
      TDIST_DEC_WH_P(128, 16, 8, 2, true)
      TDIST_DEC_PADDED(128, 16, 3, 3)
    }
    TDIST_DEC_PADDED(256, 16, 2, 3)
  }
  switch (dk) {
    case 64:
      TDIST_DEC_WH(64, 32, 8, 2)
      TDIST_DEC_WH(64, 32, 4, 4)
      TDIST_DEC(64, 0, 32, 4, 4)
    // 16-key blocks, 3 waves, 3 stages = 72 KB of LDS: two workgroups share a CU and two thirds of the ring are
    // in flight
    case 128:
      TDIST_DEC_WH(128, 16, 8, 2)   // (four waves of four stages: no faster than the form below)
      TDIST_DEC(128, 0, 16, 3, 3)
    case 192: TDIST_DEC(128, 64, 16, 2, 3)   // 61 KB: two workgroups per CU
    case 256:
      TDIST_DEC_WH(256, 16, 4, 2)
      TDIST_DEC(256, 0, 16, 2, 3)
    default: TDIST_DEC(512, 64, 16, 2, 2)    // 576 = 512 + 64: 136 KB
  }
#undef TDIST_DEC
#undef TDIST_DEC_WH
#undef TDIST_DEC_WH_P
#undef TDIST_DEC_WH_
#undef TDIST_DEC_PADDED
}

}  // namespace tdist

extern "C" {

int tdist_decode_split_kv(const void* q, const void* k_cache, const void* v_cache, float* out_split, float* lse_split,
                          float sm_scale, float soft_cap, const int32_t* block_table, const int32_t* kv_lens, int batch,
                          int q_heads, int kv_heads, int head_dim, int head_dim_v, int page_size, int num_splits,
                          int64_t q_stride_b, int64_t q_stride_h, int64_t k_stride_page, int64_t k_stride_token,
                          int64_t k_stride_head, int64_t v_stride_page, int64_t v_stride_token, int64_t v_stride_head,
                          int64_t table_stride, int dtype, void* stream) {
  DecodeCall c = {q, k_cache, v_cache, out_split, lse_split, sm_scale, soft_cap, block_table, kv_lens, batch, q_heads,
                  kv_heads, head_dim, head_dim_v, page_size, num_splits, q_stride_b, q_stride_h, k_stride_page,
                  k_stride_token, k_stride_head, v_stride_page, v_stride_token, v_stride_head, table_stride, dtype,
                  nullptr, 0, nullptr, TDIST_F32, 0, 0, nullptr, stream, "tdist_decode_split_kv", nullptr, 0};
  return run_decode(c, kFormSplit);
}

int64_t tdist_decode_fused_counters(int batch, int q_heads, int kv_heads) {
  return decode_fused_counters(batch, q_heads, kv_heads);
}

int tdist_decode_fused(const void* q, const void* k_cache, const void* v_cache, float* out_split, float* lse_split,
                       float sm_scale, float soft_cap, const int32_t* block_table, const int32_t* kv_lens, int batch,
                       int q_heads, int kv_heads, int head_dim, int head_dim_v, int page_size, int num_splits,
                       int64_t q_stride_b, int64_t q_stride_h, int64_t k_stride_page, int64_t k_stride_token,
                       int64_t k_stride_head, int64_t v_stride_page, int64_t v_stride_token, int64_t v_stride_head,
                       int64_t table_stride, int dtype, int32_t* counters, int64_t n_counters, void* out, int out_dtype,
                       int64_t out_stride_b, int64_t out_stride_h, float* lse_out, void* stream) {
  DecodeCall c = {q, k_cache, v_cache, out_split, lse_split, sm_scale, soft_cap, block_table, kv_lens, batch, q_heads,
                  kv_heads, head_dim, head_dim_v, page_size, num_splits, q_stride_b, q_stride_h, k_stride_page,
                  k_stride_token, k_stride_head, v_stride_page, v_stride_token, v_stride_head, table_stride, dtype,
                  counters, n_counters, out, out_dtype, out_stride_b, out_stride_h, lse_out, stream,
                  "tdist_decode_fused", nullptr, 0};
  return run_decode(c, kFormFused);
}

int64_t tdist_decode_stream_workspace_bytes(int batch, int q_heads, int kv_heads, int head_dim, int head_dim_v) {
  return stream_workspace_bytes(batch, q_heads, kv_heads, head_dim, head_dim_v);
}

int tdist_decode_stream(const void* q, const void* k_cache, const void* v_cache, float sm_scale, float soft_cap,
                        const int32_t* block_table, const int32_t* kv_lens, int batch, int q_heads, int kv_heads,
                        int head_dim, int head_dim_v, int page_size, int64_t q_stride_b, int64_t q_stride_h,
                        int64_t k_stride_page, int64_t k_stride_token, int64_t k_stride_head, int64_t v_stride_page,
                        int64_t v_stride_token, int64_t v_stride_head, int64_t table_stride, int dtype, int32_t* /*counters*/,
                        int64_t /*n_counters*/, void* workspace, int64_t workspace_bytes, void* out, int out_dtype,
                        int64_t out_stride_b, int64_t out_stride_h, float* lse_out, void* stream) {
  DecodeCall c = {q, k_cache, v_cache, nullptr, nullptr, sm_scale, soft_cap, block_table, kv_lens, batch, q_heads,
                  kv_heads, head_dim, head_dim_v, page_size, 1, q_stride_b, q_stride_h, k_stride_page,
                  k_stride_token, k_stride_head, v_stride_page, v_stride_token, v_stride_head, table_stride, dtype,
                  nullptr, 0, out, out_dtype, out_stride_b, out_stride_h, lse_out, stream,
                  "tdist_decode_stream", workspace, workspace_bytes};
  return run_decode(c, kFormStream);
}

int tdist_decode_combine(const void* part, int part_dtype, const float* lse, int num_partials, int mode,
                         const int32_t* lens, int batch, int q_heads, int head_dim_v, int64_t part_stride_p,
                         int64_t part_stride_b, int64_t part_stride_h, int64_t lse_stride_p, int64_t lse_stride_b,
                         int64_t lse_stride_h, void* out, int out_dtype, int64_t out_stride_b, int64_t out_stride_h,
                         float* lse_out, void* stream) {
  if (!part || !lse || !out) return fail(TDIST_ERR_INVALID, "tdist_decode_combine: null pointer");
  if (num_partials <= 0 || batch <= 0 || q_heads <= 0 || head_dim_v <= 0)
    return fail(TDIST_ERR_INVALID, "tdist_decode_combine: sizes must be positive");
  if (head_dim_v > 512) return fail(TDIST_ERR_UNSUPPORTED, "tdist_decode_combine: head_dim_v %d > 512", head_dim_v);
  if (mode < 0 || mode > 2 || (mode != 0 && !lens))
    return fail(TDIST_ERR_INVALID, "tdist_decode_combine: mode %d needs lens", mode);
  if ((part_dtype != TDIST_F32 && part_dtype != TDIST_BF16 && part_dtype != TDIST_F16) ||
      (out_dtype != TDIST_F32 && out_dtype != TDIST_BF16 && out_dtype != TDIST_F16))
    return fail(TDIST_ERR_UNSUPPORTED, "tdist_decode_combine: dtype");
  CombineParams prm;
  prm.part = (const unsigned char*)part;
  prm.lse = lse;
  prm.lens = lens;
  prm.out = (unsigned char*)out;
  prm.lse_out = lse_out;
  prm.P = num_partials;
  prm.mode = mode;
  prm.B = batch;
  prm.Hq = q_heads;
  prm.Dv = head_dim_v;
  prm.part_dtype = part_dtype;
  prm.out_dtype = out_dtype;
  prm.p_sp = part_stride_p;
  prm.p_sb = part_stride_b;
  prm.p_sh = part_stride_h;
  prm.l_sp = lse_stride_p;
  prm.l_sb = lse_stride_b;
  prm.l_sh = lse_stride_h;
  prm.o_sb = out_stride_b;
  prm.o_sh = out_stride_h;
  return launch_combine(prm, (hipStream_t)stream);
}

int tdist_decode_stream_ranks(const void* q, const void* k_cache, const void* v_cache, float sm_scale, float soft_cap,
                              const int32_t* block_table, const int32_t* rank_lens, int rank, int num_ranks, int batch, int q_heads, int kv_heads,
                              int head_dim, int head_dim_v, int page_size, int64_t q_stride_b, int64_t q_stride_h, int64_t k_stride_page,
                              int64_t k_stride_token, int64_t k_stride_head, int64_t v_stride_page, int64_t v_stride_token,
                              int64_t v_stride_head, int64_t table_stride, int dtype, void* workspace, int64_t workspace_bytes, void* rank_out,
                              int rank_out_dtype, int64_t out_stride_r, int64_t out_stride_b, int64_t out_stride_h, float* rank_lse,
                              int64_t lse_stride_r, void* out, int out_dtype, void* stream) {
  const char* who = "tdist_decode_stream_ranks";
  if (!rank_lens || !rank_out || !rank_lse || !out) return fail(TDIST_ERR_INVALID, "%s: null pointer", who);
  if (num_ranks <= 0 || rank < 0 || rank >= num_ranks || batch <= 0 || q_heads <= 0 || head_dim_v <= 0)
    return fail(TDIST_ERR_INVALID, "%s: rank %d of %d, sizes must be positive", who, rank, num_ranks);
  if ((rank_out_dtype != TDIST_F32 && rank_out_dtype != TDIST_BF16 && rank_out_dtype != TDIST_F16) ||
      (out_dtype != TDIST_F32 && out_dtype != TDIST_BF16 && out_dtype != TDIST_F16) || head_dim_v > 512)
    return fail(TDIST_ERR_UNSUPPORTED, "%s: dtype, or head_dim_v %d > 512", who, head_dim_v);
  const int esz = rank_out_dtype == TDIST_F32 ? 4 : 2, out_esz = out_dtype == TDIST_F32 ? 4 : 2;
  RankParams r;
  r.c.part = (const unsigned char*)rank_out;
  r.c.lse = rank_lse;
  r.c.lens = rank_lens;
  r.c.out = (unsigned char*)out;
  r.c.lse_out = nullptr;
  r.c.P = num_ranks;
  r.c.mode = 2;
  r.c.B = batch;
  r.c.Hq = q_heads;
  r.c.Dv = head_dim_v;
  r.c.part_dtype = rank_out_dtype;
  r.c.out_dtype = out_dtype;
  r.c.p_sp = out_stride_r;
  r.c.p_sb = out_stride_b;
  r.c.p_sh = out_stride_h;
  r.c.l_sp = lse_stride_r;
  r.c.l_sb = q_heads;
  r.c.l_sh = 1;
  r.c.o_sb = (int64_t)q_heads * head_dim_v;
  r.c.o_sh = head_dim_v;
  r.own = rank;
  r.part_vec = (uintptr_t)rank_out % (4 * esz) == 0 && out_stride_r % 4 == 0 && out_stride_b % 4 == 0 && out_stride_h % 4 == 0;
  r.out_vec = (uintptr_t)out % (4 * out_esz) == 0 && head_dim_v % 4 == 0;
  DecodeCall c = {q, k_cache, v_cache, nullptr, nullptr, sm_scale, soft_cap, block_table, rank_lens + (int64_t)rank * batch, batch, q_heads,
                  kv_heads, head_dim, head_dim_v, page_size, 1, q_stride_b, q_stride_h, k_stride_page,
                  k_stride_token, k_stride_head, v_stride_page, v_stride_token, v_stride_head, table_stride, dtype,
                  nullptr, 0, (unsigned char*)rank_out + rank * out_stride_r * esz, rank_out_dtype, out_stride_b, out_stride_h,
                  rank_lse + rank * lse_stride_r, stream, who, workspace, workspace_bytes, &r};
  return run_decode(c, kFormStream);
}

}  // extern "C"
