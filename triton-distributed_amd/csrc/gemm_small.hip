// C[M,N] = A[M,K] * B[N,K]^T for shapes whose large tiles would leave most of the chip idle (a decode step's rows, short
// prompts, narrow projections): tiles of 64 or 128 rows, two workgroups of four waves per compute unit, the K dimension
// shared by several workgroups where the tiles alone are too few. Any K whose rows are a multiple of 16 bytes.
//
//  * A and B rows go to the LDS in K tiles of 128 bytes by LDS-DMA, two to six stages, one barrier per K tile; chunk c
//    of row r sits at c ^ ((r >> 1) & 7), so that the 16 rows an operand read touches spread over the banks;
//  * a wave reads the operands of its next products (the other half of the K tile, or the next tile) before the products at
//    hand, and a load takes a scalar base and a lane offset that never changes: with one wave per SIMD nothing else hides an LDS
//    read's latency or an address instruction;
//  * a K that is no whole number of K tiles has the ragged one first (its lanes in front of the row fetch zeros), so that only
//    loads outside the loop need to know;
//  * what bounds it: the loads' way into the LDS (64 bytes a clock and compute unit; 24 KB a K tile of 64 x 128 in 0.222 us, 108 GB/s, of
//    128 x 128 32 KB in 0.315 us), at short K the launch and the first trip to memory. Before operands were read ahead and loads went
//    out one by one between products a K tile took 0.505 and 0.655 us whether its rows came from memory or from the L2: 200 x 1536 x 4096
//    16.0 -> 12.1 us, 1024 x 4096 x 4096 47.6 -> 29.6, e4m3 64 x 1536 x 8192 33.7 -> 17.5;
//  * v_mfma 16x16x32 (16-bit) / 16x16x128 (e4m3), D^T = B * A^T, so that a lane holds 4 consecutive columns;
//  * grouped (rows named by sorted ids, weights by a block's expert): for experts of few rows, where a call is a read of the
//    weights. 64 experts of 72 rows in all, 2 x 512 x 2176: 51 us a launch on tiles of 128 x 256 cut along K (86 tiles, a third
//    of their loads rows that are not there), 21 on 64 x 128, or 5.4 TB/s; 311 rows over 16 experts, 1280 x 3200: 62 -> 30;
//    1454 rows over 16, 3584 x 896: 37 -> 25 on 128 x 128;
//  * GEMM-RS (rows to their owners' buffers): this rank's tiles add the other ranks' rows to what they store, where that is little for one
//    workgroup (kSmallSumRows): 2 to 3 us less than a launch for it. 512 x 3840 x 2304 e4m3 of 2 ranks 11.6 -> 9.3 us, 1024 x 3584 x 768 bf16 of 4 12.7 -> 10.9;
//  * with `splits` > 1 every workgroup leaves its fp32 accumulators in the workspace and bumps its tile's counter; the last
//    to arrive adds the pieces up in their K order, so the result does not depend on timing and nobody waits. The pieces
//    of a tile meet in one XCD's L2 where workgroup i is known to run on XCD i % 8 (written through to memory they cost
//    12 us for 256 tiles of 64 x 128).
#include "gemm_small.h"

#include <algorithm>
#include <type_traits>

namespace tdist {

// what the DMA lanes behind a row's end read
static __device__ __align__(16) const unsigned char kZeroChunk16[16] = {0};

struct SmallBF16 {
  typedef BF16 store;   // the results' type
  static constexpr int kVecs = 1, kSteps = 2;  // 16-byte pieces per operand fragment, MFMA steps per 128 bytes of K
  typedef int4v frag;
  __device__ static __forceinline__ float4v mma(frag a, frag b, float4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v, a), __builtin_bit_cast(bf16x8v, b), c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pack(float a, float b) { return pack_bf16x2(a, b); }
};
struct SmallF16 : SmallBF16 {
  typedef F16 store;
  __device__ static __forceinline__ float4v mma(frag a, frag b, float4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8v, a), __builtin_bit_cast(f16x8v, b), c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pack(float a, float b) { return pack_f16x2(a, b); }
};
struct SmallFP8 {
  typedef BF16 store;
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

// kRows: where A's rows lie, or the results' (instances of their own: the test for shards alone costs the other calls 0.3 us of 21)
enum SmallRows { kRowsPlain, kRowsShards, kRowsGrouped, kRowsScatter };
template <typename E, int BM, int BN, int NST, bool kScales, int kRows>
__global__ __launch_bounds__(256, 2) void gemm_small_kernel(const SmallGemmParams p) {
  typedef SmallCfg<BM, BN, NST> C;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  typedef TDIST_AS3 unsigned char* lds_u8;
  lds_u8 const ring = (lds_u8)smem;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = wave >> 1, wn = wave & 1, x = lane & 15, g = lane >> 4;

  // Workgroup i runs on XCD i % 8 (checked once per device by tdist_init, and here by every tile's last workgroup): an XCD
  // takes a run of whole tiles, walk_rows row tiles by all columns at a time, so that the tiles it works on share their rows and
  // weights, and the pieces of a tile meet in its L2.
  // (grouped: of the blocks in use, a load in front of everything. Shared out with those that are not, the XCDs' parts differed by
  // half: 6070 rows over 32 experts, 512 columns, 3712 deep 76 us.)
  const int tiles_m = kRows == kRowsGrouped ? min(__builtin_amdgcn_readfirstlane(p.post_pad[0]) / BM, p.num_blocks) : (p.M + BM - 1) / BM;
  const int tiles_n = (p.N + BN - 1) / BN, tiles = tiles_m * tiles_n;
  const int xcd = blockIdx.x & 7, of_xcd = blockIdx.x >> 3;
  const int mine = of_xcd / p.splits, piece = of_xcd - mine * p.splits;
  constexpr bool kShards = kRows == kRowsShards, kGrouped = kRows == kRowsGrouped;
  if constexpr (kShards || kGrouped) retire_beside(p.shards);
  if (mine >= (tiles >> 3) + (xcd < (tiles & 7))) return;
  const int tile = xcd * (tiles >> 3) + min(xcd, tiles & 7) + mine;
  const int group = tile / (p.walk_rows * tiles_n), in_group = tile - group * p.walk_rows * tiles_n;
  const int rows_g = min(p.walk_rows, tiles_m - group * p.walk_rows), tn = in_group / rows_g;
  int tm = group * p.walk_rows + in_group - tn * rows_g, owner = 0;
  constexpr bool kScatter = kRows == kRowsScatter;
  if constexpr (kScatter) {
    // the owners in turn, this rank first: its tiles, which have the other ranks' rows to add, are spread evenly over the XCDs (8 x 1024
    // rows by 1024 columns in the order of rows: all of them on one)
    const int nth = tm / p.world;
    owner = p.rank + tm - nth * p.world;
    if (owner >= p.world) owner -= p.world;
    tm = owner * (p.m_per_rank / BM) + nth;
  }
  const bool adds = kScatter && p.out != nullptr && owner == p.rank;   // the sum of this tile is this workgroup's
  const int m0 = tm * BM, n0 = tn * BN;
  const int k_tiles = (p.k_bytes + kSmallKB - 1) / kSmallKB;
  const int back = k_tiles * kSmallKB - p.k_bytes;   // bytes of the first K tile in front of the rows
  int kt0 = piece * p.tiles_per_split, kt1 = min(kt0 + p.tiles_per_split, k_tiles), splits = p.splits;

  // DMA: instruction i of a wave brings rows (i * 4 + wave) * 8 .. + 7, lane = row * 8 + chunk position
  uint32_t aoff[C::kAInstr], boff[C::kBInstr];
  const unsigned char* b_base = p.B;
  if constexpr (kGrouped) {
    int ids[C::kAInstr];
#pragma unroll
    for (int i = 0; i < C::kAInstr; ++i) ids[i] = p.sorted_ids[m0 + (i * 4 + wave) * 8 + (lane >> 3)];
    const int expert = __builtin_amdgcn_readfirstlane(p.block_expert[tm]);
    b_base += (int64_t)expert * p.b_expert_stride_b;
#pragma unroll
    for (int i = 0; i < C::kAInstr; ++i) {
      const int r = (i * 4 + wave) * 8 + (lane >> 3);
      // (places without a row read the first one: the same lines for all of them, and what comes of it is not stored)
      int row = (uint32_t)ids[i] < (uint32_t)p.num_valid ? (p.topk == 1 ? ids[i] : (int)__umulhi((uint32_t)ids[i], p.topk_magic)) : 0;
      row = min(row, p.a_rows - 1);
      uint32_t at = (uint32_t)row * (uint32_t)p.lda_b;
      if (p.shards.rows != 0)
        for (int s = 0, first = 0; first < p.a_rows; ++s, first += p.shards.rows)
          if (row >= first) at = p.shards.off[s] + (uint32_t)(row - first) * (uint32_t)p.lda_b;
      aoff[i] = at + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
  } else {
#pragma unroll
    for (int i = 0; i < C::kAInstr; ++i) {
      const int r = (i * 4 + wave) * 8 + (lane >> 3);
      aoff[i] = (uint32_t)min(m0 + r, p.M - 1) * (uint32_t)p.lda_b + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
    }
  }
  if constexpr (kShards) {
    // rows in shards: the tile's few shards one after the other (their offsets by scalar loads), each for the rows from its first on
    const int rows = p.shards.rows, last = min(m0 + BM, p.M) - 1;
    for (int s = m0 / rows, first = s * rows; first <= last; ++s, first += rows) {
      const uint32_t off = p.shards.off[s] - (uint32_t)first * (uint32_t)p.lda_b;
#pragma unroll
      for (int i = 0; i < C::kAInstr; ++i) {
        const int r = (i * 4 + wave) * 8 + (lane >> 3), row = min(m0 + r, p.M - 1);
        if (row >= first) aoff[i] = off + (uint32_t)row * (uint32_t)p.lda_b + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < C::kBInstr; ++i) {
    const int r = (i * 4 + wave) * 8 + (lane >> 3);
    boff[i] = (uint32_t)min(n0 + r, p.N - 1) * (uint32_t)p.ldb_b + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
  }
  // one load: scalar base + lane offset, M0 the LDS address (a register the compiler does not allocate, and nothing else here uses)
  auto dma = [](const unsigned char* base, uint32_t off, lds_u8 dst) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"((uint32_t)(uintptr_t)dst) : "memory");
  };
  const uint32_t dma_lds = (uint32_t)(uintptr_t)ring + wave * 1024;
  // load n of K tile kt into the stage at `stage` bytes
  auto issue_one = [&](const unsigned char* a, const unsigned char* b, int stage, auto n_c) {
    constexpr int n = decltype(n_c)::value;
    lds_u8 const st = (lds_u8)(uintptr_t)(dma_lds + stage);
    if constexpr (n < C::kAInstr) dma(a, aoff[n], st + n * 4096);
    else dma(b, boff[n - C::kAInstr], st + BM * kSmallKB + (n - C::kAInstr) * 4096);
  };
  auto issue = [&](int kt, int stage) {
    const int64_t at = (int64_t)kt * kSmallKB - back;
    static_for<C::kLoads>([&](auto n_c) { issue_one(p.A + at, b_base + at, stage, n_c); });
  };
  // the first K tile where it is ragged: lanes in front of the row read zeros, the others what they read in any tile
  auto issue_ragged = [&](int stage) {
    lds_u8 const st = (lds_u8)(uintptr_t)(dma_lds + stage);
    auto one = [&](const unsigned char* rows, uint32_t off, int r, lds_u8 dst) {
      const unsigned char* src = rows - back + off;
      if ((((lane & 7) ^ ((r >> 1) & 7)) << 4) < back) src = kZeroChunk16;
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"((uint32_t)(uintptr_t)dst) : "memory");
    };
#pragma unroll
    for (int i = 0; i < C::kAInstr; ++i) one(p.A, aoff[i], (i * 4 + wave) * 8 + (lane >> 3), st + i * 4096);
#pragma unroll
    for (int i = 0; i < C::kBInstr; ++i) one(b_base, boff[i], (i * 4 + wave) * 8 + (lane >> 3), st + BM * kSmallKB + i * 4096);
  };

  unsigned char* c_base = p.C;

  float4v acc[C::kTN][C::kTM];
  // operand reads: row x of block i, the chunks of a step (of 16-bit types; e4m3: chunks g and g + 4, the four groups of a read on
  // consecutive chunks, and the order of gemm.hip's sums) and lane group g, relative to the stage; blocks are 16 rows apart, which
  // leaves the swizzle alone
  const int a_row = wm * (BM / 2) + x, b_row = wn * (BN / 2) + x;
  int a_at[2], b_at[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    a_at[c] = a_row * kSmallKB + (((4 * c + g) ^ ((a_row >> 1) & 7)) << 4);
    b_at[c] = BM * kSmallKB + b_row * kSmallKB + (((4 * c + g) ^ ((b_row >> 1) & 7)) << 4);
  }
  auto read = [&](int stage, const int (&at)[2], int step, int i) -> typename E::frag {
    if constexpr (E::kVecs == 1) {
      return *(const TDIST_AS3 int4v*)(ring + stage + at[step] + i * 16 * kSmallKB);
    } else {
      const int4v lo = *(const TDIST_AS3 int4v*)(ring + stage + at[0] + i * 16 * kSmallKB);
      const int4v hi = *(const TDIST_AS3 int4v*)(ring + stage + at[1] + i * 16 * kSmallKB);
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };
  auto after = [](int stage) { return stage + C::kStageBytes == C::kLdsBytes ? 0 : stage + C::kStageBytes; };

  for (;;) {
    // (nothing is outstanding here, and the compiler is told so: on the way round it would count loads of the other pieces, and
    // then wait for every load into the LDS at the first use of a register in the loop below)
    __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
    for (int j = 0; j < C::kTN; ++j)
#pragma unroll
      for (int i = 0; i < C::kTM; ++i) acc[j][i] = float4v{0.f, 0.f, 0.f, 0.f};
    const int n_kt = kt1 - kt0;
    if constexpr (kScatter) c_base = (unsigned char*)p.scatter_bufs[owner];   // (asked for here: its trip to memory is over long before the epilogue)
#pragma unroll
    for (int i = 0; i < NST - 1; ++i) {
      if (i >= n_kt) break;
      if (back != 0 && kt0 + i == 0) issue_ragged(0);
      else issue(kt0 + i, i * C::kStageBytes);
    }
    // all but the `younger` youngest K tiles have arrived
    auto wait_tiles = [&](int younger) {
      static_for<NST - 1>([&](auto n_c) {
        constexpr int n = NST - 2 - decltype(n_c)::value;
        if (younger == n || (n == NST - 2 && younger > n)) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n * C::kLoads) : "memory");
      });
    };
    // everyone has read what they read before this, and everyone's loads that this wave has waited for have arrived
    auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    // A tile's products come in two halves, 16-bit types by K and e4m3 by columns. Between a half's products the operands of the
    // next half are read and, one by one, the loads of tile k + NST - 1 go out: a wave issues in order, and in a burst each
    // would hold the products up until the one before it is through (64 x 128 bf16: 0.31 us a K tile in a burst).
    // Behind the last tile whatever a stage holds is read, and not used: with the reads conditional the compiler would wait for
    // them where the operands before them are used.
    constexpr int kHalves = E::kSteps == 2 ? 1 : 2;             // column halves
    constexpr int kCols = C::kTN / kHalves, kProducts = C::kTM * kCols;
    constexpr int kFirstLoads = NST > 2 ? C::kLoads / 2 : C::kLoads;   // (two stages: the tile is waited for in this very trip)
    typename E::frag a[3 - kHalves][C::kTM], b[2][kCols];       // (e4m3: the same rows for both halves)
    int stage = 0, free_stage = (NST - 1) * C::kStageBytes;   // tile k's stage, and the one that tile k + NST - 1 goes to
    auto half = [&](auto h_c, auto load_c, const unsigned char* ka, const unsigned char* kb, int load_stage) {
      constexpr int h = decltype(h_c)::value;
      constexpr int kLoad0 = h == 0 ? 0 : kFirstLoads, kLoadN = decltype(load_c)::value ? (h == 0 ? kFirstLoads : C::kLoads - kFirstLoads) : 0;
      static_for<kProducts>([&](auto m_c) {
        constexpr int m = decltype(m_c)::value, kNow = m * kLoadN / kProducts, kNext = (m + 1) * kLoadN / kProducts;
        if constexpr (kHalves == 1) {
          if constexpr (m < C::kTM) a[1 - h][m] = read(stage, a_at, 1 - h, m);
          else if constexpr (m < C::kTM + kCols) b[1 - h][m - C::kTM] = read(stage, b_at, 1 - h, m - C::kTM);
          constexpr int j = m / C::kTM, i = m % C::kTM;
          acc[j][i] = E::mma(b[h][j], a[h][i], acc[j][i]);
        } else {
          // row by row: the next tile's row takes a row's place as soon as its products are out
          if constexpr (m < kCols) b[1 - h][m] = read(stage, b_at, 0, (1 - h) * kCols + m);
          constexpr int i = m / kCols, j = m % kCols;
          acc[h * kCols + j][i] = E::mma(b[h][j], a[0][i], acc[h * kCols + j][i]);
          if constexpr (h == 1 && j == kCols - 1) a[0][i] = read(stage, a_at, 0, i);
        }
        static_for<kNext - kNow>([&](auto u_c) { issue_one(ka, kb, load_stage, std::integral_constant<int, kLoad0 + kNow + decltype(u_c)::value>{}); });
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    static_assert(kHalves == 2 || C::kTM + kCols <= kProducts, "a read per product");
    constexpr std::integral_constant<int, 0> zero{};
    constexpr std::integral_constant<int, 1> one{};
    auto tile_of = [&](int k, auto load_c) {
      constexpr bool kLoad = decltype(load_c)::value;
      const int64_t at = (int64_t)(kt0 + k + NST - 1) * kSmallKB - back;
      const unsigned char *ka = p.A + at, *kb = b_base + at;
      const int load_stage = free_stage;
      half(zero, load_c, ka, kb, load_stage);
      // tile k + 1 has arrived
      if constexpr (kLoad) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NST > 2 ? (NST - 3) * C::kLoads + kFirstLoads : 0) : "memory");
      else wait_tiles(n_kt - 2 - k);
      meet();
      free_stage = stage;
      stage = after(stage);
      half(one, load_c, ka, kb, load_stage);
    };
    wait_tiles(n_kt - 1);
    meet();
#pragma unroll
    for (int i = 0; i < C::kTM; ++i) a[0][i] = read(0, a_at, 0, i);
#pragma unroll
    for (int j = 0; j < kCols; ++j) b[0][j] = read(0, b_at, 0, j);
    __builtin_amdgcn_sched_barrier(0);
    int k = 0;
    for (; k + NST - 1 < n_kt; ++k) tile_of(k, std::true_type{});
    for (; k < n_kt; ++k) tile_of(k, std::false_type{});
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
    // added in the pieces' order, eight accumulators of three other pieces in flight at a time; this workgroup's own piece is still
    // in its registers
    constexpr int kBatch = 3;
    static_assert(kAccs % 8 == 0, "eight at a time");
    static_for<kAccs / 8>([&](auto part_c) {
      constexpr int u0 = decltype(part_c)::value * 8;
      float4v total[8];
      auto add_own = [&]() {
#pragma unroll
        for (int u = 0; u < 8; ++u) total[u] += acc[(u0 + u) / C::kTM][(u0 + u) % C::kTM];
      };
#pragma unroll
      for (int u = 0; u < 8; ++u) total[u] = float4v{0.f, 0.f, 0.f, 0.f};
      for (int z0 = 0; z0 < splits - 1; z0 += kBatch) {   // z: the other pieces in order, own one left out
        float4v v[kBatch][8];
#pragma unroll
        for (int w = 0; w < kBatch; ++w) {
          const int z = min(z0 + w, splits - 2);
          const float4v* src = slots + (int64_t)(z + (z >= piece)) * (kAccs * 256) + u0 * 256;
#pragma unroll
          for (int u = 0; u < 8; ++u) v[w][u] = src[u * 256];
        }
#pragma unroll
        for (int w = 0; w < kBatch; ++w) {
          if (z0 + w == piece) add_own();
          if (z0 + w < splits - 1) {
#pragma unroll
            for (int u = 0; u < 8; ++u) total[u] += v[w][u];
          }
        }
      }
      // (own the last, and not met above as the place behind the last batch)
      if (piece == splits - 1 && (splits - 1) % kBatch == 0) add_own();
#pragma unroll
      for (int u = 0; u < 8; ++u) acc[(u0 + u) / C::kTM][(u0 + u) % C::kTM] = total[u];
    });
    break;
  }

  // grouped: the output rows of the pieces that this thread will store
  constexpr int kPieces = BN / 8, kStores = BM * kPieces / 256;
  int out_row[kGrouped ? kStores : 1];
  if constexpr (kGrouped) {
#pragma unroll
    for (int u = 0; u < kStores; ++u) out_row[u] = p.sorted_ids[m0 + (u * 256 + threadIdx.x) / kPieces];
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
  auto stage_tile = [&] {
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
  };
  if constexpr (kScatter) {
    if (adds) {
      // The sum over the ranks: the others' rows, four pieces of every slice in flight at a time, in the order rank + 1, rank + 2, ..., and
      // the own ones last, as they are stored: the order and the bits of reduce.hip. No load is conditional (the compiler would wait for
      // some of them in front of others): slices beyond the last are the last one again.
      auto add_up = [&](auto slices_c) {
        constexpr int kSlices = decltype(slices_c)::value, kBatch = 4;
        static_assert(kStores % kBatch == 0, "whole batches");
        int4v v[kSlices][kBatch];
        auto ask = [&](auto u0_c) {
#pragma unroll
          for (int w = 0; w < kSlices; ++w) {
            const int i = min(1 + w, p.world - 1), s = p.rank + i < p.world ? p.rank + i : p.rank + i - p.world;
            const unsigned char* const src = p.own + ((int64_t)((s - p.rank) * p.m_per_rank + m0) * p.ldc + n0) * 2;
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
              const int idx = (decltype(u0_c)::value + u) * 256 + threadIdx.x, row = idx / kPieces, col = min(idx % kPieces * 8, p.N - 8 - n0);
              v[w][u] = *(const TDIST_AS1 int4v*)(src + ((int64_t)row * p.ldc + col) * 2);
            }
          }
        };
        ask(std::integral_constant<int, 0>{});
        stage_tile();
        static_for<kStores / kBatch>([&](auto b_c) {
          constexpr int u0 = decltype(b_c)::value * kBatch;
          float sum[kBatch][8];
#pragma unroll
          for (int u = 0; u < kBatch; ++u)
#pragma unroll
            for (int e = 0; e < 8; ++e) sum[u][e] = 0.f;
          auto add = [&](int u, const int4v& x) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              sum[u][2 * e] += E::store::lo((uint32_t)x[e]);
              sum[u][2 * e + 1] += E::store::hi((uint32_t)x[e]);
            }
          };
#pragma unroll
          for (int w = 0; w < kSlices; ++w) {
            if (1 + w >= p.world) break;
#pragma unroll
            for (int u = 0; u < kBatch; ++u) add(u, v[w][u]);
          }
          if constexpr (u0 + kBatch < kStores) ask(std::integral_constant<int, u0 + kBatch>{});
#pragma unroll
          for (int u = 0; u < kBatch; ++u) {
            const int idx = (u0 + u) * 256 + threadIdx.x, row = idx / kPieces, col = idx % kPieces * 8;
            if (n0 + col >= p.N) continue;
            const int4v own = *(const TDIST_AS3 int4v*)(ring + row * C::kEpiPitch + col * 2);
            *(int4v*)(c_base + ((int64_t)(m0 + row) * p.ldc + n0 + col) * 2) = own;
            add(u, own);
            int4v o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (int)E::store::pack(sum[u][2 * e], sum[u][2 * e + 1]);
            *(int4v*)(p.out + ((int64_t)(m0 - p.rank * p.m_per_rank + row) * p.N + n0 + col) * 2) = o;
          }
        });
      };
      constexpr int kMost = kSmallSumRows / BM;   // other ranks
      if (p.world <= 2) add_up(std::integral_constant<int, 1>{});
      else if (kMost <= 3 || p.world <= 4) add_up(std::integral_constant<int, 3>{});
      else if constexpr (kMost > 3) add_up(std::integral_constant<int, kMost>{});
      return;
    }
  }
  stage_tile();
  if constexpr (kGrouped) {
    const bool vec = (p.ldc % 8) == 0 && ((uintptr_t)p.C & 15) == 0;
#pragma unroll
    for (int u = 0; u < kStores; ++u) {
      const int idx = u * 256 + threadIdx.x, row = idx / kPieces, col = idx % kPieces * 8;
      if ((uint32_t)out_row[u] >= (uint32_t)p.num_valid || n0 + col >= p.N) continue;
      const int4v v = *(const TDIST_AS3 int4v*)(ring + row * C::kEpiPitch + col * 2);
      unsigned short* dst = (unsigned short*)p.C + (int64_t)out_row[u] * p.ldc + n0 + col;
      if (vec && n0 + col + 8 <= p.N) {
        *(int4v*)dst = v;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (n0 + col + e < p.N) dst[e] = (unsigned short)((uint32_t)v[e >> 1] >> (16 * (e & 1)));
      }
    }
    return;
  }
  const int row_shift = kScatter ? (p.rank - owner) * p.m_per_rank : 0;
  const bool vec = (p.ldc % 8) == 0 && ((uintptr_t)c_base & 15) == 0;
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

// Row tiles that an XCD's run of tiles goes down before the next column. Its 32 to 64 workgroups at work then need few panels: eight rows
// by eight columns, 16, where a run down all row tiles of a long call needs a row panel for every one of them and takes each from
// behind its L2 once per column (12288 x 2304 x 768 bf16 84.0 -> 67.8 us, 4608 x 872 x 1104 18.6 -> 15.6, 7680 x 2888 x 1488 e4m3 62.4 -> 52.2; 4
// and 16 are as good, 1 and 2 are behind in calls of few row tiles). The row tiles of a group belong to one expert or share no
// weights: half of what an expert has, eight at most (6856 rows over 8 experts, 2944 x 512: 57.7 -> 52.5; 3060 over 32, 1152 x 1024: 31.8 -> 27.8;
// 16384 over 8, 4096 x 1792: 372 -> 296, with two rows 328). 90 calls of each kind: 4 and 3.5 % faster on average, 1 % behind the best of 1 to 32.
static int64_t walk_rows(const SmallGemmParams& p, int bm) {
  if (!p.sorted_ids) return 8;
  if ((int64_t)p.num_blocks * bm < p.num_valid) return 2;   // (experts' last rows: one block of each, or two)
  // (experts: what the number of blocks leaves room for, every one pads bm - 1 rows at most)
  const int64_t experts = ((int64_t)p.num_blocks * bm - p.num_valid) / (bm - 1) + 1, blocks = (p.num_valid / std::max<int64_t>(experts, 1) + bm / 2) / bm;
  return blocks >= 16 ? 8 : blocks >= 8 ? 4 : blocks >= 4 ? 2 : 1;
}

template <typename E, int BM, int BN, int NST, bool kScales, int kRows>
static int launch_rows(const SmallGemmParams& p, hipStream_t stream, const char* who) {
  typedef SmallCfg<BM, BN, NST> C;
  auto kern = gemm_small_kernel<E, BM, BN, NST, kScales, kRows>;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, C::kLdsBytes);
    if (e != hipSuccess) return fail(TDIST_ERR_LAUNCH, "%s: cannot reserve %d B of LDS: %s", who, C::kLdsBytes, hipGetErrorString(e));
    attr_set = true;
  }
  const int64_t tiles_m = ceil_div(p.M, BM), tiles_n = ceil_div(p.N, BN), grid = 8 * ceil_div(tiles_m * tiles_n, 8) * p.splits;
  SmallGemmParams q = p;
  q.walk_rows = (int)std::min<int64_t>(walk_rows(p, BM), tiles_m);
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), C::kLdsBytes, stream, q);
  return launch_status(who);
}

template <typename E, int BM, int BN, int NST, bool kScales>
static int launch_cfg(const SmallGemmParams& p, hipStream_t stream, const char* who) {
  if constexpr (!kScales)
    if (p.sorted_ids) return launch_rows<E, BM, BN, NST, kScales, kRowsGrouped>(p, stream, who);
  if (p.scatter_bufs) return launch_rows<E, BM, BN, NST, kScales, kRowsScatter>(p, stream, who);
  return p.shards.rows != 0 ? launch_rows<E, BM, BN, NST, kScales, kRowsShards>(p, stream, who) : launch_rows<E, BM, BN, NST, kScales, kRowsPlain>(p, stream, who);
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
