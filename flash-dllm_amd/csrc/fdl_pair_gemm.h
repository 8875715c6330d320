// GEMM over pairs of weight rows (gfx950, bf16 MFMA, fp32 sums), for many input rows:
//   lo[r][p] = x_r . w_lo(p),  hi[r][p] = x_r . w_hi(p)        (reduction length K)
// handed to an epilogue that sees both members of a pair. The Q/K/V projection pairs the two
// columns that RoPE rotates together.
//
// Tile: 256 rows x 96 pairs (192 weight rows), eight wavefronts (4 x 2, each 64 rows x 48
// pairs, two per SIMD) that load, read LDS and multiply alike.
//
// What bounds it: the L2 -> LDS path moves 26-36 B/clk per CU with every CU loading, and a tile
// of m x n needs 128 (m + n) bytes per 64-deep step of m n / 32 MFMA clocks. 256 x 192 needs 36
// B/clk at the full MFMA rate, the 128 x 192 tile of the smaller shape 53: that one spends its
// time on loads. Both operands are requested two steps ahead (three weight stages: weights may
// come from HBM; two x stages: x is in L2), the weights in the first half of a step and the
// rows in the second, as their stages come free: requesting both in the second half took 5%
// longer (4096 rows 348 -> 329 us). At 4096 rows x 12288 columns x 4096 (us): this tile 326, the
// 128 x 192 one 386; with the loads left out 281, the LDS reads left out 283, the MFMAs left
// out 268 (all in a probe copy), so the three overlap and none is alone the limit; the dense
// MFMA work also pulls the clock down to about 1.9 GHz. The epilogue is about 8 us of the 82
// that a full round of tiles takes. Keeping workgroups resident, with the next tile's first
// loads under an epilogue that stores straight from registers, gained nothing (338 us), nor
// did a five-slot ring of half x tiles (a step further ahead: 327 us at 4096 rows; only a
// half-filled device gained, 76 -> 68 us at 512 rows).
#pragma once

#include <type_traits>

#include "fdl_device.h"

namespace fdl {

constexpr int kPgBM = 256, kPgBP = 96, kPgThreads = 512;
constexpr int kPgKT = 64;                     // reduction step (128 B of a row)
constexpr int kPgABytes = kPgBM * 128;        // x tile of one step
constexpr int kPgBBytes = 2 * kPgBP * 128;    // weight tile of one step (low, high rows)
constexpr int kPgAStages = 2, kPgBStages = 3;
constexpr int kPgBOff = kPgAStages * kPgABytes;
constexpr int kPgMetaOff = kPgBOff + kPgBStages * kPgBBytes;
constexpr int kPgLds = kPgMetaOff + kPgBM * 8;  // 138 KB
constexpr int kPgEpStride = 2 * kPgBP + 4;  // floats per staged row of the epilogue
constexpr int kPgEpRows = 128;              // rows staged at a time
static_assert(kPgEpRows * kPgEpStride * 4 <= kPgMetaOff, "epilogue staging");
constexpr int kPgALoads = kPgABytes / 1024 / 8;  // 1 KB loads per wavefront and step
constexpr int kPgBLoads = kPgBBytes / 1024 / 8;

struct PairGemmTiles {
  const uint16_t* x;  // [n_rows][k]
  int64_t n_rows;
  int k;        // a multiple of 128, at least 256
  int n_mtiles, n_ntiles;
};

// 16 bytes per lane from global memory into LDS at lds + 16 * lane (lds wavefront-uniform),
// issued where the compiler does not see it: it would otherwise wait for every load in flight
// before any LDS read of the wavefront. M0 carries the LDS address and is restored.
__device__ __forceinline__ void pg_dma16(const void* base, uint32_t off, uint32_t lds) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %3\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(off), "s"(base), "s"(lds)
      : "memory");
}
__device__ __forceinline__ void pg_dma16(const void* g, uint32_t lds) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, off\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(g), "s"(lds)
      : "memory");
}
template <int N>
__device__ __forceinline__ void pg_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Tile t -> (n-block, m-block): groups of up to kPgGroupM m-blocks, the m-block fastest within
// a group, so that the tiles of one XCD share x rows and weight rows in its L2.
// At 27 m-blocks (6842 rows): groups of at most 4 / 6 / 8 take 540 / 543 / 567 us.
constexpr int kPgGroupM = 6;
__device__ __forceinline__ void pg_tile(const PairGemmTiles& t, int i, int& nt, int& mt) {
  const int groups = (t.n_mtiles + kPgGroupM - 1) / kPgGroupM;
  const int gm = (t.n_mtiles + groups - 1) / groups;  // m-blocks per group, even groups
  const int per_group = gm * t.n_ntiles;
  const int grp = i / per_group, r = i - grp * per_group;
  const int in_grp = min(gm, t.n_mtiles - grp * gm);
  nt = r / in_grp;
  mt = grp * gm + (r - nt * in_grp);
}

// Epilogue `Ep`: wrow(p, hi) is the first element of pair p's low or high weight row; row(r) ->
// Ep::Row (8 bytes) says where output row r goes (also for r past n_rows: nowhere);
// store(row, r, p, lo, hi) takes the sums of pairs p .. p + 7 (p a multiple of 8) of row r from
// LDS.
template <class Ep>
__global__ __launch_bounds__(kPgThreads, 1) void pair_gemm_kernel(PairGemmTiles t, Ep ep) {
  constexpr int kRB = 4, kPB = 3, kWP = kPgBP / 2;
  __shared__ __align__(1024) uint8_t smem[kPgLds];
  typedef __attribute__((address_space(3))) void* lds_p;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = wave >> 1, wn = wave & 1;
  const int l16 = lane & 15, g4 = lane >> 4;
  const int sw = (l16 >> 1) & 7;
  const int nk = t.k / kPgKT;

  // Workgroup i runs on XCD i % 8: each XCD takes a contiguous run of tiles.
  const int n_tiles = t.n_mtiles * t.n_ntiles;
  int nt, mt;
  pg_tile(t, (n_tiles & 7) == 0 ? (blockIdx.x & 7) * (n_tiles >> 3) + (blockIdx.x >> 3) : blockIdx.x,
          nt, mt);
  const int64_t m0 = int64_t(mt) * kPgBM;

  // Load l of wavefront w fills the 8-row block q = 8 l + w of the x (weight) tile; lane -> row
  // 8 q + lane / 8, LDS chunk lane % 8, which holds the row's chunk (lane % 8) ^ ((row >> 1) & 7):
  // two 128-byte rows share one 256-byte bank line, so 16 consecutive rows read at one chunk
  // land on 16 distinct 4-bank groups.
  const uint16_t* abase = t.x + m0 * t.k;  // the next step to load
  const int last = static_cast<int>(min(t.n_rows - m0, int64_t(kPgBM)) - 1);
  uint32_t aoff[kPgALoads];         // this lane's row and chunk, bytes from abase
  const uint16_t* bsrc[kPgBLoads];  // the next step to load
#pragma unroll
  for (int l = 0; l < kPgALoads; ++l) {
    const int row = 8 * (8 * l + wave) + (lane >> 3);
    const int c = (lane & 7) ^ ((row >> 1) & 7);
    aoff[l] = uint32_t(min(row, last)) * uint32_t(2 * t.k) + 16 * c;
  }
#pragma unroll
  for (int l = 0; l < kPgBLoads; ++l) {
    const int row = 8 * (8 * l + wave) + (lane >> 3);
    const int c = (lane & 7) ^ ((row >> 1) & 7);
    const int hi = row / kPgBP;
    bsrc[l] = ep.wrow(kPgBP * nt + (row - hi * kPgBP), hi) + 8 * c;
  }
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<size_t>((lds_p)smem));
  const uint32_t a_lds = __builtin_amdgcn_readfirstlane(lds0 + 1024 * wave);
  const uint32_t b_lds = __builtin_amdgcn_readfirstlane(lds0 + kPgBOff + 1024 * wave);
  auto load_a = [&](int stage, int l) {
    pg_dma16(abase, aoff[l],
             __builtin_amdgcn_readfirstlane(a_lds + uint32_t(stage * kPgABytes + 8192 * l)));
  };
  auto load_b = [&](int stage, int l) {
    pg_dma16(bsrc[l], __builtin_amdgcn_readfirstlane(b_lds + uint32_t(stage * kPgBBytes + 8192 * l)));
    bsrc[l] += kPgKT;
  };
  u32x4 fa[2][kRB], fb[2][2 * kPB];
  f32x4 acc[kRB][2 * kPB];  // [row block][kPB hi + pair block]
  // fragment addresses: half-step 1 reads the chunk with its bit 2 flipped (byte offset 64)
  const uint32_t fa_off = (64 * wm + l16) * 128 + ((g4 ^ sw) << 4);
  const uint32_t fb_off = kPgBOff + (kWP * wn + l16) * 128 + ((g4 ^ sw) << 4);
  auto read_a = [&](int f, uint32_t at, int rb) {
    fa[f][rb] = *reinterpret_cast<const u32x4*>(smem + at + 2048 * rb);
  };
  auto read_b = [&](int f, uint32_t at, int j) {
    fb[f][j] = *reinterpret_cast<const u32x4*>(smem + at + (j / kPB) * (kPgBP * 128) +
                                               (j % kPB) * 2048);
  };
  auto mma = [&](int f, int rb) {
#pragma unroll
    for (int j = 0; j < 2 * kPB; ++j)
      acc[rb][j] = mfma16(as_bf16x8(fa[f][rb]), as_bf16x8(fb[f][j]), acc[rb][j]);
  };
  typename Ep::Row* meta = reinterpret_cast<typename Ep::Row*>(smem + kPgMetaOff);
  static_assert(sizeof(typename Ep::Row) == 8, "row metadata");

  // steps 0 and 1, in the order in which they are waited for
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int l = 0; l < kPgALoads; ++l) load_a(s, l);
    abase += kPgKT;
#pragma unroll
    for (int l = 0; l < kPgBLoads; ++l) load_b(s, l);
  }
#pragma unroll
  for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
    for (int j = 0; j < 2 * kPB; ++j) acc[rb][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (tid < kPgBM) meta[tid] = ep.row(m0 + tid);
  pg_wait<kPgALoads + kPgBLoads>();  // step 0 landed
  asm volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int rb = 0; rb < kRB; ++rb) read_a(0, fa_off, rb);
#pragma unroll
  for (int j = 0; j < 2 * kPB; ++j) read_b(0, fb_off, j);

  int bs = 0;  // weight stage of the step (the x stage is its parity)
  // One step; kLoad: step kt + 2 exists and is requested; kMore: step kt + 1 exists. The
  // fragments of the next half-step are read, and the weights (first half) and rows (second
  // half) of step kt + 2 requested, between the MFMAs of this half-step; their stages were
  // released by the previous step's barrier and by this step's.
  auto step = [&](int as, auto load_tag, auto more_tag) {
    constexpr bool kLoad = decltype(load_tag)::value, kMore = decltype(more_tag)::value;
    const int bs1 = bs == kPgBStages - 1 ? 0 : bs + 1;
    const int bs2 = bs1 == kPgBStages - 1 ? 0 : bs1 + 1;
    const uint32_t a1 = (fa_off + as * kPgABytes) ^ 64, b1 = (fb_off + bs * kPgBBytes) ^ 64;
    const uint32_t a0 = fa_off + (as ^ 1) * kPgABytes, b0 = fb_off + bs1 * kPgBBytes;
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
      if (kLoad && rb < kPgBLoads) load_b(bs2, rb);
      read_a(1, a1, rb);
      if (rb < kPB) {
        read_b(1, b1, 2 * rb);
        read_b(1, b1, 2 * rb + 1);
      }
      mma(0, rb);
      __builtin_amdgcn_sched_barrier(0);
    }
    // step kt + 1 landed (the weights of step kt + 2 may be in flight); this wave's reads of
    // step kt are done
    pg_wait<kLoad ? kPgBLoads : 0>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
      if (kLoad) load_a(as, rb);
      if (kMore) {
        read_a(0, a0, rb);
        if (rb < kPB) {
          read_b(0, b0, 2 * rb);
          read_b(0, b0, 2 * rb + 1);
        }
      }
      mma(1, rb);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (kLoad) abase += kPgKT;
    bs = bs1;
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  for (int kt = 0; kt < nk - 2; ++kt) step(kt & 1, yes, yes);
  step(0, no, yes);
  step(1, no, no);

  // Epilogue: two halves of 128 rows staged as fp32 rows [low | high] in LDS (every LDS read of
  // the loop came before its last barrier); each thread takes 8-pair groups.
  float* epm = reinterpret_cast<float*>(smem);
  constexpr int kGroups = kPgBP / 8, kPer = kPgEpRows * kGroups / kPgThreads;
  static_assert(kPer * kPgThreads == kPgEpRows * kGroups, "epilogue split");
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    if (half) __syncthreads();
    if ((wm >> 1) == half) {
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float* row = epm + (64 * (wm & 1) + 16 * rb + 4 * g4 + i) * kPgEpStride + kWP * wn + l16;
#pragma unroll
          for (int j = 0; j < 2 * kPB; ++j) row[kPgBP * (j / kPB) + 16 * (j % kPB)] = acc[rb][j][i];
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int it = tid + kPgThreads * j;
      const int row = it / kGroups, g = it - kGroups * row;
      const float* src = epm + row * kPgEpStride + 8 * g;
      const int mrow = kPgEpRows * half + row;
      ep.store(meta[mrow], m0 + mrow, kPgBP * nt + 8 * g, src, src + kPgBP);
    }
  }
}

}  // namespace fdl
