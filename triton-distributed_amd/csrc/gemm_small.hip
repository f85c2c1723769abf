// C[M,N] = A[M,K] * B[N,K]^T for shapes whose large tiles would leave most of the chip idle (a decode step's rows, short
// prompts, narrow projections): tiles of 64 or 128 rows, two workgroups of four waves per compute unit, the K dimension
// shared by several workgroups where the tiles alone are too few. Any K whose rows are a multiple of 16 bytes.
//
//  * A and B rows go to the LDS in K tiles of 128 bytes by LDS-DMA, three or four stages, one barrier per K tile; chunk c
//    of row r sits at c ^ ((r >> 1) & 7), so that the 16 rows an operand read touches spread over the banks;
//  * v_mfma 16x16x32 (16-bit) / 16x16x128 (e4m3), D^T = B * A^T, so that a lane holds 4 consecutive columns;
//  * with `splits` > 1 every workgroup leaves its fp32 accumulators in the workspace and bumps its tile's counter; the last
//    to arrive adds the pieces up in their K order, so the result does not depend on timing and nobody waits. The pieces
//    of a tile meet in one XCD's L2 where workgroup i is known to run on XCD i % 8 (written through to memory they cost
//    12 us for 256 tiles of 64 x 128).
#include "gemm_small.h"

namespace tdist {

// what the DMA lanes behind a row's end read
static __device__ __align__(16) const unsigned char kZeroChunk16[16] = {0};

struct SmallBF16 {
  static constexpr int kVecs = 1, kSteps = 2;  // 16-byte pieces per operand fragment, MFMA steps per 128 bytes of K
  typedef int4v frag;
  __device__ static __forceinline__ float4v mma(frag a, frag b, float4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v, a), __builtin_bit_cast(bf16x8v, b), c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pack(float a, float b) { return pack_bf16x2(a, b); }
};
struct SmallF16 : SmallBF16 {
  __device__ static __forceinline__ float4v mma(frag a, frag b, float4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8v, a), __builtin_bit_cast(f16x8v, b), c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pack(float a, float b) { return pack_f16x2(a, b); }
};
struct SmallFP8 {
  static constexpr int kVecs = 2, kSteps = 1;
  typedef int8v frag;
  __device__ static __forceinline__ float4v mma(frag a, frag b, float4v c) {
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pack(float a, float b) { return pack_bf16x2(a, b); }
};

constexpr int kSmallKB = 128;  // bytes of K per tile row

template <int BM, int BN, int NST>
struct SmallCfg {
  static constexpr int kAInstr = BM / 32, kBInstr = BN / 32;  // DMA instructions (8 rows each) per wave and K tile
  static constexpr int kLoads = kAInstr + kBInstr;
  static constexpr int kStageBytes = (BM + BN) * kSmallKB;
  static constexpr int kLdsBytes = NST * kStageBytes;
  static constexpr int kTM = BM / 2 / 16, kTN = BN / 2 / 16;  // 16 x 16 blocks of a wave (2 x 2 waves)
  static constexpr int kEpiPitch = BN * 2 + 16;               // bytes between the staged output rows
  static_assert(BM * kEpiPitch <= kLdsBytes, "the output tile is staged in the ring");
  static_assert((NST - 2) * kLoads < 64, "vmcnt is 6 bits");
};

// kShards: A's rows lie in shards (an instance of its own: the test for them alone costs the other calls 0.3 us of 21)
template <typename E, int BM, int BN, int NST, bool kScales, bool kShards>
__global__ __launch_bounds__(256, 2) void gemm_small_kernel(const SmallGemmParams p) {
  typedef SmallCfg<BM, BN, NST> C;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  typedef TDIST_AS3 unsigned char* lds_u8;
  lds_u8 const ring = (lds_u8)smem;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1, x = lane & 15, g = lane >> 4;

  // Workgroup i runs on XCD i % 8 (checked once per device by tdist_init, and here by every tile's last workgroup): an XCD
  // takes a run of whole tiles, row tiles first, so that it fetches its columns' weights once and the pieces of a tile
  // meet in its L2.
  const int tiles_m = (p.M + BM - 1) / BM, tiles = tiles_m * ((p.N + BN - 1) / BN);
  const int xcd = blockIdx.x & 7, of_xcd = blockIdx.x >> 3;
  const int mine = of_xcd / p.splits, piece = of_xcd - mine * p.splits;
  if constexpr (kShards) retire_beside(p.shards);
  if (mine >= (tiles >> 3) + (xcd < (tiles & 7))) return;
  const int tile = xcd * (tiles >> 3) + min(xcd, tiles & 7) + mine;
  const int tm = tile % tiles_m, tn = tile / tiles_m;
  const int m0 = tm * BM, n0 = tn * BN;
  const int k_tiles = (p.k_bytes + kSmallKB - 1) / kSmallKB;
  const int tail = p.k_bytes % kSmallKB;
  int kt0 = piece * p.tiles_per_split, kt1 = min(kt0 + p.tiles_per_split, k_tiles), splits = p.splits;

  // DMA: instruction i of a wave brings rows (i * 4 + wave) * 8 .. + 7, lane = row * 8 + chunk position
  uint32_t aoff[C::kAInstr], boff[C::kBInstr];
  int chunk_a[C::kAInstr], chunk_b[C::kBInstr];
#pragma unroll
  for (int i = 0; i < C::kAInstr; ++i) {
    const int r = (i * 4 + wave) * 8 + (lane >> 3);
    chunk_a[i] = (lane & 7) ^ ((r >> 1) & 7);
    aoff[i] = (uint32_t)min(m0 + r, p.M - 1) * (uint32_t)p.lda_b + chunk_a[i] * 16;
  }
  if constexpr (kShards) {
    // rows in shards: the tile's few shards one after the other (their offsets by scalar loads), each for the rows from its first on
    const int rows = p.shards.rows, last = min(m0 + BM, p.M) - 1;
    for (int s = m0 / rows, first = s * rows; first <= last; ++s, first += rows) {
      const uint32_t off = p.shards.off[s] - (uint32_t)first * (uint32_t)p.lda_b;
#pragma unroll
      for (int i = 0; i < C::kAInstr; ++i) {
        const int row = min(m0 + (i * 4 + wave) * 8 + (lane >> 3), p.M - 1);
        if (row >= first) aoff[i] = off + (uint32_t)row * (uint32_t)p.lda_b + chunk_a[i] * 16;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < C::kBInstr; ++i) {
    const int r = (i * 4 + wave) * 8 + (lane >> 3);
    chunk_b[i] = (lane & 7) ^ ((r >> 1) & 7);
    boff[i] = (uint32_t)min(n0 + r, p.N - 1) * (uint32_t)p.ldb_b + chunk_b[i] * 16;
  }
  auto dma = [](const unsigned char* src, lds_u8 dst) {
    __builtin_amdgcn_global_load_lds((const TDIST_AS1 void*)src, (TDIST_AS3 void*)dst, 16, 0, 0);
  };
  auto issue = [&](int kt) {
    lds_u8 const st = ring + (kt - kt0) % NST * C::kStageBytes + wave * 1024;
    const unsigned char* a = p.A + (int64_t)kt * kSmallKB;
    const unsigned char* b = p.B + (int64_t)kt * kSmallKB;
    const bool cut = tail != 0 && kt == k_tiles - 1;
#pragma unroll
    for (int i = 0; i < C::kAInstr; ++i) {
      const unsigned char* src = a + aoff[i];
      if (cut && chunk_a[i] * 16 >= tail) src = kZeroChunk16;
      dma(src, st + i * 4096);
    }
#pragma unroll
    for (int i = 0; i < C::kBInstr; ++i) {
      const unsigned char* src = b + boff[i];
      if (cut && chunk_b[i] * 16 >= tail) src = kZeroChunk16;
      dma(src, st + BM * kSmallKB + i * 4096);
    }
  };

  float4v acc[C::kTN][C::kTM];
  // operand reads: row x of block i, chunks of step s and lane group g
  const int a_row = wm * (BM / 2) + x, b_row = wn * (BN / 2) + x;
  auto frag_at = [&](lds_u8 rows, int row, int step) -> typename E::frag {
    const int sw = (row >> 1) & 7;   // (blocks are 16 rows apart: the same for all of them)
    if constexpr (E::kVecs == 1) {
      return *(const TDIST_AS3 int4v*)(rows + row * kSmallKB + (((step * 4 + g) ^ sw) << 4));
    } else {
      // (chunks g and g + 4: the four groups of a read on consecutive chunks, and the order of gemm.hip's sums)
      const int4v lo = *(const TDIST_AS3 int4v*)(rows + row * kSmallKB + ((g ^ sw) << 4));
      const int4v hi = *(const TDIST_AS3 int4v*)(rows + row * kSmallKB + (((g + 4) ^ sw) << 4));
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };

  for (;;) {
#pragma unroll
    for (int j = 0; j < C::kTN; ++j)
#pragma unroll
      for (int i = 0; i < C::kTM; ++i) acc[j][i] = float4v{0.f, 0.f, 0.f, 0.f};
    const int n_kt = kt1 - kt0;
#pragma unroll
    for (int i = 0; i < NST - 1; ++i)
      if (i < n_kt) issue(kt0 + i);
    for (int k = 0; k < n_kt; ++k) {
      // this K tile has arrived (the younger ones may be on their way), and everyone is done with the one before
      if (k + NST - 2 < n_kt) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NST - 2) * C::kLoads) : "memory");
      else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (k + NST - 1 < n_kt) issue(kt0 + k + NST - 1);
      lds_u8 const st = ring + k % NST * C::kStageBytes;
#pragma unroll
      for (int s = 0; s < E::kSteps; ++s) {
        typename E::frag a[C::kTM], b[C::kTN];
#pragma unroll
        for (int i = 0; i < C::kTM; ++i) a[i] = frag_at(st, a_row + i * 16, s);
#pragma unroll
        for (int j = 0; j < C::kTN; ++j) b[j] = frag_at(st + BM * kSmallKB, b_row + j * 16, s);
#pragma unroll
        for (int j = 0; j < C::kTN; ++j)
#pragma unroll
          for (int i = 0; i < C::kTM; ++i) acc[j][i] = E::mma(b[j], a[i], acc[j][i]);
      }
    }
    __syncthreads();
    if (splits == 1) break;

    // ---- this piece of K into the workspace; the last piece's workgroup adds them up -------------------------
    constexpr int kAccs = C::kTM * C::kTN;
    float4v* const slots = (float4v*)p.partials + (int64_t)tile * splits * (kAccs * 256) + threadIdx.x;
    float4v* const own = slots + (int64_t)piece * (kAccs * 256);
    if (p.l2_local) {
#pragma unroll
      for (int u = 0; u < kAccs; ++u) own[u * 256] = acc[u / C::kTM][u % C::kTM];
    } else {
#pragma unroll
      for (int u = 0; u < kAccs; ++u)
        asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 0" ::"v"(own + u * 256), "v"(acc[u / C::kTM][u % C::kTM]) : "memory");
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    TDIST_AS3 int* const s_sum = (TDIST_AS3 int*)ring;
    // the counter sums 1, the XCD id and its square over the pieces: sum and sum of squares tell whether all ids were one
    const int id = __builtin_amdgcn_readfirstlane(xcc_id()), arrive = 1 | id << 8 | (id * id) << 16;
    if (threadIdx.x == 0) {
      const int sum = __hip_atomic_fetch_add(p.counters + tile, arrive, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + arrive;
      if ((sum & 255) == splits) __hip_atomic_store(p.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *s_sum = sum;
    }
    __syncthreads();
    const int sum = __builtin_amdgcn_readfirstlane(*s_sum);
    if ((sum & 255) != splits) return;
    __syncthreads();
    if (p.l2_local && sum != splits * arrive) {
      // pieces from another XCD, whose L2 holds what they left: this workgroup works the whole tile out itself
      kt0 = 0, kt1 = k_tiles, splits = 1;
      continue;
    }
    if (p.l2_local) asm volatile("buffer_inv sc0" ::: "memory");
    else __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#pragma unroll
    for (int u = 0; u < kAccs; ++u) acc[u / C::kTM][u % C::kTM] = float4v{0.f, 0.f, 0.f, 0.f};
    // two pieces in flight at a time, added in order
    for (int z = 0; z < splits; z += 2) {
      const float4v* src = slots + (int64_t)z * (kAccs * 256);
      const float4v* src2 = slots + (int64_t)min(z + 1, splits - 1) * (kAccs * 256);
      float4v v[2][kAccs];
#pragma unroll
      for (int u = 0; u < kAccs; ++u) v[0][u] = src[u * 256], v[1][u] = src2[u * 256];
#pragma unroll
      for (int u = 0; u < kAccs; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[u / C::kTM][u % C::kTM][e] += v[0][u][e];
          if (z + 1 < splits) acc[u / C::kTM][u % C::kTM][e] += v[1][u][e];
        }
    }
    break;
  }

  // ---- epilogue: lane holds columns 4g .. 4g+3 of row x of each block; staged through the LDS so that stores are whole
  // 16-byte pieces of a row
  // (the scales in one round trip, in front of the packing: a load per element and row block in between took longer than a
  // short K's products: 2048 x 1024 x 3328 e4m3 37 -> 26 us per call)
  float4v cs[kScales ? C::kTN : 1];
  float rs[kScales ? C::kTM : 1];
  if constexpr (kScales) {
#pragma unroll
    for (int j = 0; j < C::kTN; ++j) {
      const int col = n0 + wn * (BN / 2) + j * 16 + 4 * g;
#pragma unroll
      for (int e = 0; e < 4; ++e) cs[j][e] = p.col_scale ? p.col_scale[min(col + e, p.N - 1)] : 1.f;
    }
#pragma unroll
    for (int i = 0; i < C::kTM; ++i) rs[i] = p.row_scale ? p.row_scale[min(m0 + wm * (BM / 2) + i * 16 + x, p.M - 1)] : 1.f;
  }
#pragma unroll
  for (int i = 0; i < C::kTM; ++i) {
    const int row = wm * (BM / 2) + i * 16 + x;
#pragma unroll
    for (int j = 0; j < C::kTN; ++j) {
      const int col = wn * (BN / 2) + j * 16 + 4 * g;
      float4v v = acc[j][i];
      if constexpr (kScales) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= rs[i] * cs[j][e];
      }
      *(TDIST_AS3 int2v*)(ring + row * C::kEpiPitch + col * 2) = int2v{(int)E::pack(v[0], v[1]), (int)E::pack(v[2], v[3])};
    }
  }
  __syncthreads();
  unsigned char* c_base = p.C;
  int row_shift = 0;
  if (p.scatter_bufs) {
    const int owner = m0 / p.m_per_rank;
    c_base = (unsigned char*)p.scatter_bufs[owner];
    row_shift = (p.rank - owner) * p.m_per_rank;
  }
  const bool vec = (p.ldc % 8) == 0 && ((uintptr_t)c_base & 15) == 0;
  constexpr int kPieces = BN / 8;
  for (int idx = threadIdx.x; idx < BM * kPieces; idx += 256) {
    const int row = idx / kPieces, col = idx % kPieces * 8;
    if (m0 + row >= p.M || n0 + col >= p.N) continue;
    const int4v v = *(const TDIST_AS3 int4v*)(ring + row * C::kEpiPitch + col * 2);
    unsigned short* dst = (unsigned short*)c_base + (int64_t)(m0 + row + row_shift) * p.ldc + n0 + col;
    if (vec && n0 + col + 8 <= p.N) {
      *(int4v*)dst = v;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (n0 + col + e < p.N) dst[e] = (unsigned short)((uint32_t)v[e >> 1] >> (16 * (e & 1)));
    }
  }
}

template <typename E, int BM, int BN, int NST, bool kScales, bool kShards>
static int launch_shards(const SmallGemmParams& p, hipStream_t stream, const char* who) {
  typedef SmallCfg<BM, BN, NST> C;
  auto kern = gemm_small_kernel<E, BM, BN, NST, kScales, kShards>;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::kLdsBytes);
    if (e != hipSuccess) return fail(TDIST_ERR_LAUNCH, "%s: cannot reserve %d B of LDS: %s", who, C::kLdsBytes, hipGetErrorString(e));
    attr_set = true;
  }
  const int64_t grid = 8 * ceil_div(ceil_div(p.M, BM) * ceil_div(p.N, BN), 8) * p.splits;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), C::kLdsBytes, stream, p);
  return launch_status(who);
}

template <typename E, int BM, int BN, int NST, bool kScales>
static int launch_cfg(const SmallGemmParams& p, hipStream_t stream, const char* who) {
  return p.shards.rows != 0 ? launch_shards<E, BM, BN, NST, kScales, true>(p, stream, who) : launch_shards<E, BM, BN, NST, kScales, false>(p, stream, who);
}

template <int BM, int BN, int NST>
static int launch_tile(const SmallGemmParams& p, SmallGemmElem elem, hipStream_t stream, const char* who) {
  switch (elem) {
    case kSmallBF16: return launch_cfg<SmallBF16, BM, BN, NST, false>(p, stream, who);
    case kSmallF16: return launch_cfg<SmallF16, BM, BN, NST, false>(p, stream, who);
    default:
      return p.row_scale || p.col_scale ? launch_cfg<SmallFP8, BM, BN, NST, true>(p, stream, who)
                                        : launch_cfg<SmallFP8, BM, BN, NST, false>(p, stream, who);
  }
}

int launch_gemm_small(const SmallGemmParams& p, SmallGemmElem elem, int tile, bool deep, hipStream_t stream, const char* who) {
  if (tile == 0) return deep ? launch_tile<64, 128, 6>(p, elem, stream, who) : launch_tile<64, 128, 3>(p, elem, stream, who);
  return deep ? launch_tile<128, 128, 4>(p, elem, stream, who) : launch_tile<128, 128, 2>(p, elem, stream, who);
}

}  // namespace tdist
