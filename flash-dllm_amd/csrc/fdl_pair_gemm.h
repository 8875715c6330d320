// GEMM over pairs of weight rows (gfx950, bf16 MFMA, fp32 sums):
//   lo[r][p] = x_r . w_lo(p),  hi[r][p] = x_r . w_hi(p)        (reduction length K)
// handed to an epilogue that sees both members of a pair. The Q/K/V projection pairs the two
// columns that RoPE rotates together, the MLP a column's gate and up rows.
//
// pair_pc_kernel: up to 128 rows per tile, wavefronts in two roles (producers that only load,
// consumers that only read LDS and multiply), a deep ring of stages; also the weight-streaming
// kernel of few rows.
//
// pair_gemm_kernel: 256 rows x 96 pairs (192 weight rows) per tile, eight wavefronts (4 x 2, each
// 64 rows x 48 pairs, two per SIMD) that load, read LDS and multiply alike.
//
// What bounds the latter: the L2 -> LDS path moves 26-36 B/clk per CU with every CU loading, and a tile
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

#include <atomic>
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

typedef __attribute__((address_space(3))) void* PgLds;
typedef __attribute__((address_space(1))) void* PgGlb;

struct PairGemmTiles {
  const uint16_t* x;  // [n_rows][ld]
  int64_t n_rows;
  int k;        // reduction length of a workgroup (256-row tiles: a multiple of 128, at least 256)
  int n_mtiles, n_ntiles;
  int ld;       // row stride of x; the weight rows' is the epilogue's business
  int start_mul;  // see pg_start
};

// The reduction step that the tile of pairs p0 .. starts its walk with (it wraps around). Where the
// weight rows are a multiple of 4 KB apart and all workgroups read the same 128 bytes of them at a
// time, the reads crowd on few HBM channels; cold weights, all in step / started apart (us): rows
// of 8 KB, gate and up of 64 rows (201 MB) 44.6 / 36.8, of 128 rows 47.9 / 42.1, the 40-row
// projection (101 MB) 23.5 / 20.8; rows of 4 KB, gate and up of one row 13.4 / 11.7, of 128 rows
// 18.0 / 17.3; other distances (2, 5, 6, 7 KB) the same within 1%, so those start in step. The pairs
// are cut into groups of kPgStartPairs, a multiple of every tile's width, and the groups spread
// over kPgStarts even places (8 places: 128 rows of gate and up 45.4 us; 32 or 64 no better than
// 16). The place depends on the pair, the number of pairs and the rows' length alone, so a row's
// sums are added in the same order, and are the same bits, whatever the number of rows and the
// tile. Launches of many row blocks gain nothing from it and lose nothing (6842 rows of the
// projection 544 / 547 us).
constexpr int kPgStartPairs = 96, kPgStarts = 16, kPgStartStride = 2048;  // (elements)
__device__ __forceinline__ int pg_start(const PairGemmTiles& t, int p0, int nk) {
  return ((p0 / kPgStartPairs * t.start_mul) >> 16) * nk / kPgStarts;
}

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

// Epilogue `Ep`: wrow(p, hi) is the first element of pair p's low or high weight row; row(r) ->
// Ep::Row (8 bytes) says where output row r goes (also for r past n_rows: nowhere); Ep::Group
// takes 8 consecutive pairs of one row: load(ep, row, r, p, lo, hi_off, mine) reads the low sums
// at lo and the high sums at lo + hi_off (p a multiple of 8; nothing is stored unless mine),
// store(ep) writes them.

// ---------------------------------------------------------------------------------------
// Producer / consumer tiles

// LDS tile layout: chunk c (16 B) of tile row r is stored at chunk c ^ ((r >> 1) & 7) of
// that row: two 128-byte rows share one 256-byte bank line, so 16 consecutive rows read at
// the same logical chunk land on 16 distinct 4-bank groups.

// Workgroup i runs on XCD i % 8. Renumber so that each XCD gets a contiguous run of tiles
// (tiles are numbered n-block-major): the m-tiles that share one weight slice then run on
// one XCD and share its L2.
__device__ __forceinline__ int xcd_tile(int bid, int n_tiles) {
  return (n_tiles & 7) == 0 ? (bid & 7) * (n_tiles >> 3) + (bid >> 3) : bid;
}

// Tile t -> (n-block, m-block). Tiles come in groups of kGroupM m-blocks: within a group
// the m-block varies fastest, so the tiles running at the same time on one XCD share both
// X row blocks (kGroupM of them) and weight slices (one per kGroupM tiles) in its L2.
// With at most kGroupM m-blocks this is the plain n-block-major order.
constexpr int kGroupM = 8;
__device__ __forceinline__ void tile_coords(int t, int n_mtiles, int n_tiles, int& nt, int& mt) {
  const int n_ntiles = n_tiles / n_mtiles;
  const int per_group = kGroupM * n_ntiles;
  const int grp = t / per_group, r = t - grp * per_group;
  const int gm = min(kGroupM, n_mtiles - grp * kGroupM);  // m-blocks in this group
  nt = r / gm;
  mt = grp * kGroupM + (r - nt * gm);
}

// Waits until at most n (clamped to 0 .. STAGES - 1) steps of kLoads loads each are in flight.
template <int STAGES, int kLoads>
__device__ __forceinline__ void pg_wait_steps(int n) {
  static_assert(STAGES >= 2 && STAGES <= 8, "stages");
  switch (n <= 0 ? 0 : (n >= STAGES - 1 ? STAGES - 1 : n)) {
    case 0: pg_wait<0>(); break;
    case 1: pg_wait<kLoads>(); break;
    case 2: pg_wait<(STAGES > 2 ? 2 : 0) * kLoads>(); break;
    case 3: pg_wait<(STAGES > 3 ? 3 : 0) * kLoads>(); break;
    case 4: pg_wait<(STAGES > 4 ? 4 : 0) * kLoads>(); break;
    case 5: pg_wait<(STAGES > 5 ? 5 : 0) * kLoads>(); break;
    case 6: pg_wait<(STAGES > 6 ? 6 : 0) * kLoads>(); break;
    default: pg_wait<(STAGES > 7 ? 7 : 0) * kLoads>(); break;
  }
}
// Workgroup barrier without the compiler's memory fence; each side waits for exactly the
// memory operations it must (the fence would drain every outstanding global load).
__device__ __forceinline__ void pg_barrier_lds() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
__device__ __forceinline__ void pg_barrier() { asm volatile("s_barrier" ::: "memory"); }

// ---------------------------------------------------------------------------------------
// Shape of one pair_pc_kernel instance. Consumer (wm, wn) of the WM x (4 / WM) consumers owns
// rows BM/WM * wm .. + BM/WM and columns kCols * wn .. + kCols, counted over [BP low | BP high].
template <int BM, int BP, int NPROD, int STAGES, int WM>
struct PcShape {
  static constexpr int kConsumers = 4, kWN = kConsumers / WM;
  static constexpr int kThreads = (kConsumers + NPROD) * 64;
  static constexpr int kCols = 2 * BP / kWN, kCB = kCols / 16, kRB = BM / (16 * WM);
  static constexpr int kABytes = BM * 128;                 // X tile of one step
  static constexpr int kStageBytes = kABytes + 2 * BP * 128;  // + W tile (low, high columns)
  static constexpr int kLoads = kStageBytes / 1024 / NPROD;   // 1 KB loads per producer/step
  // Epilogue staging in the stage memory once the reduction is done: the fp32 sums as rows
  // of [BP low | BP high] columns (row stride padded by 4 floats), then the rows' places.
  static constexpr int kEpStride = 2 * BP + 4;
  static constexpr int kEpMetaOff = BM * kEpStride * 4;
  static_assert(kCB >= 1 && kRB >= 1 && kCB * 16 * kWN == 2 * BP && kRB * 16 * WM == BM && BP % 8 == 0,
                "tile shape");
  static_assert(kLoads * NPROD * 1024 == kStageBytes, "producer split");
  static_assert((STAGES - 1) * kLoads < 64, "vmcnt range");
  static_assert(STAGES * kStageBytes <= 160 * 1024, "LDS");
  static_assert(kEpMetaOff + BM * 8 <= STAGES * kStageBytes, "epilogue staging");
  static_assert(BM <= kThreads, "row destinations");
};

template <class Ep, int BM, int BP, int NPROD, int STAGES, int WM>
__global__ __launch_bounds__((4 + NPROD) * 64, 1) void pair_pc_kernel(PairGemmTiles t, Ep ep) {
  using Sh = PcShape<BM, BP, NPROD, STAGES, WM>;
  constexpr int kCols = Sh::kCols, kCB = Sh::kCB, kRB = Sh::kRB, kLoads = Sh::kLoads;
  constexpr int kStageBytes = Sh::kStageBytes, kEpStride = Sh::kEpStride;
  constexpr int kThreads = Sh::kThreads, kConsumers = Sh::kConsumers;
  __shared__ __align__(1024) uint8_t smem[STAGES * kStageBytes];

  const int tid = threadIdx.x;
  int nt, mt;
  const int n_tiles = t.n_mtiles * t.n_ntiles;
  tile_coords(xcd_tile(blockIdx.x, n_tiles), t.n_mtiles, n_tiles, nt, mt);
  const int64_t m0 = int64_t(mt) * BM;
  const int64_t ksplit = int64_t(blockIdx.y) * t.k;  // this part's place in the reduction
  // The wavefront index is uniform; readfirstlane makes the role test a scalar branch, so a
  // wavefront executes only its own role's barriers (both roles execute 3 + nk of them).
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const bool producer = wave >= kConsumers;
  const int nk = t.k / kPgKT;

  // Places of tile rows 0 .. BM - 1 (threads 0 .. BM - 1), found now and staged in LDS for the
  // epilogue once the stage memory is free.
  typename Ep::Row my_row = {};
  static_assert(sizeof(my_row) == 8, "row places");
  if (tid < BM) my_row = ep.row(m0 + tid);

  if (producer) {
    const int pw = wave - kConsumers;
    // Load i of producer pw fills LDS bytes [1024 q, 1024 q + 1024) of the step's tile
    // (q = NPROD i + pw, an 8-row block): lane -> row 8 q + lane / 8, LDS chunk lane % 8,
    // which holds the row's logical chunk (lane % 8) ^ ((row >> 1) & 7) (the LDS tile
    // layout). Tile rows past n_rows re-read row n_rows - 1 (never stored). The blocks are
    // dealt round-robin, so every producer requests both X and weight rows: with the X rows
    // on some producers and the weights on the others, the 40-row projection took 2% longer.
    const uint16_t* src[kLoads];
    int dst_off[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int q = NPROD * i + pw;
      const int row = 8 * q + (lane >> 3);
      const int c = (lane & 7) ^ ((row >> 1) & 7);
      if (row < BM) {
        src[i] = t.x + min(m0 + row, t.n_rows - 1) * t.ld + ksplit + 8 * c;
      } else {
        const int wr = row - BM, hlf = wr / BP;
        src[i] = ep.wrow(BP * nt + (wr - hlf * BP), hlf) + ksplit + 8 * c;
      }
      dst_off[i] = 1024 * q;
    }
    const int rot = pg_start(t, BP * nt, nk);
    // Requests step kt (< nk) into `stage`. No step past the end is requested: the tail of the
    // loop waits for fewer steps instead (re-reading the last step there, to keep one wait
    // count, cost 1.3% at 512 rows).
    auto issue = [&](int kt, int stage) {
      const int k0 = (kt + rot < nk ? kt + rot : kt + rot - nk) * kPgKT;
      uint8_t* st = smem + stage * kStageBytes;
#pragma unroll
      for (int i = 0; i < kLoads; ++i)
        __builtin_amdgcn_global_load_lds((PgGlb)(src[i] + k0), (PgLds)(st + dst_off[i]), 16,
                                         0, 0);
    };
    const int first = min(STAGES, nk);  // steps requested before the loop
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
      if (s < first) issue(s, s);
    pg_wait_steps<STAGES, kLoads>(first - 1);  // step 0 landed
    pg_barrier();
    int stage = 0;
    int kt = 0;
    for (; kt + STAGES < nk; ++kt) {
      // step kt + 1 landed (steps kt + 2 .. kt + STAGES - 1 may still be in flight)
      pg_wait<(STAGES - 2) * kLoads>();
      pg_barrier();
      issue(kt + STAGES, stage);  // this stage's last reads came before the barrier
      stage = stage == STAGES - 1 ? 0 : stage + 1;
    }
    // the last steps request nothing: step kt + 1 landed, steps kt + 2 .. nk - 1 in flight
    for (; kt < nk; ++kt) {
      pg_wait_steps<STAGES, kLoads>(nk - 2 - kt);
      pg_barrier();
    }
    pg_wait<0>();  // no load may still be writing LDS when the stages are reused
    pg_barrier();   // -> the consumers may overwrite the stages
    pg_barrier();   // <- the accumulators and destinations are staged
  } else {
    const int wm = wave / Sh::kWN, wn = wave % Sh::kWN;
    const int l16 = lane & 15, g4 = lane >> 4;
    const int sw = (l16 >> 1) & 7;
    struct Frag {
      u32x4 a[kRB];
      u32x4 b[kCB];
    };
    // MFMA operands of half-step ss of the step in `stage`: lane (l16, g4) takes logical
    // chunk 4 ss + g4 of its row.
    auto read_frag = [&](Frag& f, int stage, int ss) {
      const u32x4* st = reinterpret_cast<const u32x4*>(smem + stage * kStageBytes);
      const int c = (4 * ss + g4) ^ sw;
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) f.a[rb] = st[((BM / WM) * wm + 16 * rb + l16) * 8 + c];
#pragma unroll
      for (int cb = 0; cb < kCB; ++cb)
        f.b[cb] = st[Sh::kABytes / 16 + (kCols * wn + 16 * cb + l16) * 8 + c];
    };
    f32x4 acc[kRB][kCB];
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
      for (int cb = 0; cb < kCB; ++cb) acc[rb][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto mma = [&](const Frag& f) {
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
        for (int cb = 0; cb < kCB; ++cb)
          acc[rb][cb] = mfma16(as_bf16x8(f.a[rb]), as_bf16x8(f.b[cb]), acc[rb][cb]);
    };
    // the next half-step's LDS reads spread between this half-step's MFMAs
    constexpr int kReads = kRB + kCB, kMfma = kRB * kCB;
    constexpr int kEvery = kMfma / kReads;  // MFMAs after each read
    auto interleave = [&]() {
      if constexpr (kEvery == 0) return;  // fewer MFMAs than reads: the compiler's order
#pragma unroll
      for (int i = 0; i < kReads; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, kEvery, 0);
      }
      if constexpr (kMfma > kEvery * kReads)
        __builtin_amdgcn_sched_group_barrier(0x008, kMfma - kEvery * kReads, 0);
    };

    Frag f0, f1;
    pg_barrier_lds();  // step 0 landed
    read_frag(f0, 0, 0);
    int stage = 0;
    for (int kt = 0; kt < nk; ++kt) {
      const int next = stage == STAGES - 1 ? 0 : stage + 1;
      read_frag(f1, stage, 1);
      mma(f0);
      interleave();
      __builtin_amdgcn_sched_barrier(0);
      pg_barrier_lds();  // step kt + 1 landed; this wave's reads of step kt done
      __builtin_amdgcn_sched_barrier(0);
      read_frag(f0, next, 0);
      mma(f1);
      interleave();
      __builtin_amdgcn_sched_barrier(0);
      stage = next;
    }

    // Stage the accumulators as fp32 rows in LDS: acc[rb][cb][i] is row
    // BM/WM wm + 16 rb + 4 g4 + i, column kCols wn + 16 cb + l16.
    pg_barrier_lds();  // every LDS read done, every producer load landed
    float* staged = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float* row = staged + ((BM / WM) * wm + 16 * rb + 4 * g4 + i) * kEpStride + kCols * wn + l16;
#pragma unroll
        for (int cb = 0; cb < kCB; ++cb) row[16 * cb] = acc[rb][cb][i];
      }
    if (tid < BM) reinterpret_cast<typename Ep::Row*>(smem + Sh::kEpMetaOff)[tid] = my_row;
    pg_barrier_lds();
  }

  // Every thread stores groups of 8 pairs of one row (16-byte stores): all the reads of its
  // groups first, then the stores.
  const float* staged = reinterpret_cast<const float*>(smem);
  const auto* meta = reinterpret_cast<const typename Ep::Row*>(smem + Sh::kEpMetaOff);
  constexpr int kGroups = BP / 8, kItems = BM * kGroups;
  constexpr int kPer = (kItems + kThreads - 1) / kThreads;
  typename Ep::Group grp[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int it = min(tid + kThreads * j, kItems - 1);
    const int row = it / kGroups, g = it - kGroups * row;
    const bool mine = kItems % kThreads == 0 || tid + kThreads * j < kItems;
    grp[j].load(ep, meta[row], m0 + row, BP * nt + 8 * g, staged + row * kEpStride + 8 * g, BP, mine);
  }
#pragma unroll
  for (int j = 0; j < kPer; ++j) grp[j].store(ep);
}

// ---------------------------------------------------------------------------------------
// 256-row tiles

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

template <class Ep>
__global__ __launch_bounds__(kPgThreads, 1) void pair_gemm_kernel(PairGemmTiles t, Ep ep) {
  constexpr int kRB = 4, kPB = 3, kWP = kPgBP / 2;
  __shared__ __align__(1024) uint8_t smem[kPgLds];

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
  const int start = pg_start(t, kPgBP * nt, nk);
  const uint16_t* abase = t.x + m0 * t.k + start * kPgKT;  // the next step to load
  int to_wrap = nk - 1 - start;  // steps to load before the walk goes back to the first
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
    bsrc[l] = ep.wrow(kPgBP * nt + (row - hi * kPgBP), hi) + start * kPgKT + 8 * c;
  }
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<size_t>((PgLds)smem));
  const uint32_t a_lds = __builtin_amdgcn_readfirstlane(lds0 + 1024 * wave);
  const uint32_t b_lds = __builtin_amdgcn_readfirstlane(lds0 + kPgBOff + 1024 * wave);
  auto load_a = [&](int stage, int l) {
    pg_dma16(abase, aoff[l],
             __builtin_amdgcn_readfirstlane(a_lds + uint32_t(stage * kPgABytes + 8192 * l)));
  };
  int advance = 0;  // elements from the step that is being loaded to the next one
  auto next_step = [&]() { advance = to_wrap-- == 0 ? kPgKT - t.k : kPgKT; };
  auto load_b = [&](int stage, int l) {
    pg_dma16(bsrc[l], __builtin_amdgcn_readfirstlane(b_lds + uint32_t(stage * kPgBBytes + 8192 * l)));
    bsrc[l] += advance;
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
    next_step();
#pragma unroll
    for (int l = 0; l < kPgALoads; ++l) load_a(s, l);
    abase += advance;
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
    if (kLoad) next_step();
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
    if (kLoad) abase += advance;
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
      typename Ep::Group grp;
      grp.load(ep, meta[mrow], m0 + mrow, kPgBP * nt + 8 * g, src, kPgBP, true);
      grp.store(ep);
    }
  }
}

// ---------------------------------------------------------------------------------------
// Launch

// Compute units of the current device (cached per device).
inline int pg_device_cus() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cache[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
      n = 256;
    cache[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// `kernel` of BM-row, BP-pair tiles over n_rows rows and n_pairs pairs (a multiple of BP).
// n_split > 1 (producer / consumer kernels): part z of the reduction, k / n_split long, runs as
// grid row z.
template <class Ep>
hipError_t pair_launch(void (*kernel)(PairGemmTiles, Ep), int bm, int bp, int threads,
                       const uint16_t* x, int64_t n_rows, int64_t k, int64_t n_pairs, const Ep& ep,
                       hipStream_t stream, int64_t n_split = 1) {
  const int64_t n_mtiles = (n_rows + bm - 1) / bm, n_ntiles = n_pairs / bp;
  if (n_mtiles * n_ntiles >= (int64_t(1) << 31)) return hipErrorInvalidValue;
  const int64_t groups = (n_pairs + kPgStartPairs - 1) / kPgStartPairs;
  const PairGemmTiles t = {x, n_rows, static_cast<int>(k / n_split), static_cast<int>(n_mtiles),
                           static_cast<int>(n_ntiles), static_cast<int>(k),
                           k % kPgStartStride ? 0 : static_cast<int>((kPgStarts << 16) / groups)};
  hipLaunchKernelGGL(kernel,
                     dim3(static_cast<unsigned>(n_mtiles * n_ntiles), static_cast<unsigned>(n_split)),
                     dim3(threads), 0, stream, t, ep);
  return hipGetLastError();
}

}  // namespace fdl
