// Products of the block around the attention (gfx950, bf16 MFMA): the gate and up projections
// of the MLP with the SiLU gate in one pass, and split products for few rows (attn_out, ff_out).
//
// The first replaces ff_proj(x), up_proj(x), act and the product (flash_cache_triton.py:628-633):
//   g = bf16(x_r . w_gate[c]),  u = bf16(x_r . w_up[c])       (fp32 sums)
//   out[r][c] = bf16(bf16(silu(g)) * u)
// with the roundings where the unfused code rounds. Column c of both products is one pair of
// the pair GEMM (fdl_pair_gemm.h), so the [rows][2 width] product is neither written nor read.
#include <algorithm>

#include "fdl_device.h"
#include "fdl_host.h"
#include "fdl_pair_gemm.h"

namespace fdl {
namespace {

struct SiluEp {
  const uint16_t* wg;
  const uint16_t* wu;
  uint16_t* out;
  int64_t n_rows;
  int k;
  int chunk;  // columns per output chunk
  struct Row {
    int64_t r;  // output row, -1: not stored
  };
  __device__ __forceinline__ const uint16_t* wrow(int p, int hi) const {
    return (hi ? wu : wg) + int64_t(p) * k;
  }
  __device__ __forceinline__ Row row(int64_t r) const { return {r < n_rows ? r : -1}; }
  struct Group {
    f32x4 g[2], u[2];
    uint16_t* dst;  // null: nothing is stored
    __device__ __forceinline__ void load(const SiluEp& ep, const Row& d, int64_t, int p,
                                         const float* lo, int hi_off, bool mine) {
      const int q = p / ep.chunk;
      dst = mine && d.r >= 0
                ? ep.out + (q * ep.n_rows + d.r) * ep.chunk + (p - q * ep.chunk)
                : nullptr;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        g[h] = *reinterpret_cast<const f32x4*>(lo + 4 * h);
        u[h] = *reinterpret_cast<const f32x4*>(lo + hi_off + 4 * h);
      }
    }
    __device__ __forceinline__ void store(const SiluEp&) const {
      if (dst == nullptr) return;
      u32x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float y[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int i = 2 * j + e;
          const float gv = bf2f(f2bf(g[i >> 2][i & 3])), uv = bf2f(f2bf(u[i >> 2][i & 3]));
          y[e] = bf2f(f2bf(gv / (1.0f + expf(-gv)))) * uv;
        }
        o[j] = pack_bf16x2(y[0], y[1]);
      }
      __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(dst));
    }
  };
};

// ---------------------------------------------------------------------------------------
// Split reductions of a plain product for few rows: part[z][r][n] = sum over chunk z of the
// reduction of x[r][k] w[n][k], in fp32, to be added by the pass that consumes the product
// (fdl_rms_norm_partials, fdl_split_reduce_residual).

// Weights [n_out][k]: columns n and n + n_out / 2 are a pair of the pair GEMM.
struct PartEp {
  const uint16_t* w;
  float* part;
  int64_t n_rows;
  int k, n_out;
  struct Row {
    int64_t r;  // -1: not stored
  };
  __device__ __forceinline__ const uint16_t* wrow(int p, int hi) const {
    return w + int64_t(p + hi * (n_out >> 1)) * k;
  }
  __device__ __forceinline__ Row row(int64_t r) const { return {r < n_rows ? r : -1}; }
  struct Group {
    f32x4 v[2][2];
    float* dst;
    __device__ __forceinline__ void load(const PartEp& ep, const Row& d, int64_t, int p,
                                         const float* lo, int hi_off, bool mine) {
      dst = mine && d.r >= 0
                ? ep.part + (int64_t(blockIdx.y) * ep.n_rows + d.r) * ep.n_out + p
                : nullptr;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          v[h][e] = *reinterpret_cast<const f32x4*>(lo + h * hi_off + 4 * e);
    }
    __device__ __forceinline__ void store(const PartEp& ep) const {
      if (dst == nullptr) return;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          *reinterpret_cast<f32x4*>(dst + h * (ep.n_out >> 1) + 4 * e) = v[h][e];
    }
  };
};

// Weights stored transposed, wt [k][n_out]: BM rows x 128 columns of one chunk of the reduction.
// Four producer wavefronts move 64-deep steps into LDS (64 weight rows of 256 B, BM rows of 128
// B), STAGES deep; four consumers take 32 columns each. The product is formed transposed
// (columns x rows): the weights come as MFMA operands through gfx950's transposing LDS read
// (as V does in the attention), whose 16-lane groups take k-slot (g, j) = 4 g + j of a 32-deep
// half-step for j < 4 and 16 + 4 g + j - 4 beyond; the rows are read in the same order.
// Bound by the weight stream: k 12288, n_out 4096 (101 MB, cold) at 64 rows in 8 parts take 25
// us and 3 more to add them; 4 parts (half of the device) 38, 16 parts (two rounds) 34.
template <int BM, int STAGES>
__global__ __launch_bounds__(512, 1) void part_t_kernel(const uint16_t* __restrict__ x,
                                                        const uint16_t* __restrict__ wt,
                                                        int64_t n_rows, int k, int kc, int n_out,
                                                        float* __restrict__ part) {
  constexpr int kWBytes = 64 * 256, kStageBytes = kWBytes + BM * 128;
  constexpr int kLoads = kStageBytes / 1024 / 4, kRB = BM / 16;
  static_assert(kLoads * 4096 == kStageBytes && STAGES * kStageBytes <= 160 * 1024, "stages");
  static_assert((STAGES - 1) * kLoads < 64, "vmcnt range");
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  __shared__ __align__(1024) uint8_t smem[STAGES * kStageBytes];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int64_t m0 = int64_t(blockIdx.z) * BM;
  const int n0 = 128 * blockIdx.x, nk = kc / kPgKT;
  const int64_t kz = int64_t(blockIdx.y) * kc;

  if (wave >= 4) {
    const int pw = wave - 4;
    // 1 KB block q = 4 i + pw of a step: weight rows 4 q .. + 3 (chunk c of weight row r at c ^
    // ((r & 7) << 1)), then rows 8 (q - 16) .. + 7 (chunk c of row r at c ^ ((r >> 1) & 7); rows
    // past n_rows repeat the last)
    const uint16_t* src[kLoads];
    int64_t step[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int q = 4 * i + pw;
      if (q < 16) {
        const int r = 4 * q + (lane >> 4);
        const int c = (lane & 15) ^ ((r & 7) << 1);
        src[i] = wt + (kz + r) * n_out + n0 + 8 * c;
        step[i] = int64_t(kPgKT) * n_out;
      } else {
        const int r = 8 * (q - 16) + (lane >> 3);
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        src[i] = x + min(m0 + r, n_rows - 1) * k + kz + 8 * c;
        step[i] = kPgKT;
      }
    }
    auto issue = [&](int stage) {
      uint8_t* st = smem + stage * kStageBytes + 1024 * pw;
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        __builtin_amdgcn_global_load_lds((PgGlb)src[i], (PgLds)(st + 4096 * i), 16, 0, 0);
        src[i] += step[i];
      }
    };
    const int first = min(STAGES, nk);
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
      if (s < first) issue(s);
    pg_wait_steps<STAGES, kLoads>(first - 1);  // step 0 landed
    pg_barrier();
    int stage = 0;
    int kt = 0;
    for (; kt + STAGES < nk; ++kt) {
      pg_wait<(STAGES - 2) * kLoads>();  // step kt + 1 landed
      pg_barrier();
      issue(stage);  // this stage's last reads came before the barrier
      stage = stage == STAGES - 1 ? 0 : stage + 1;
    }
    for (; kt < nk; ++kt) {
      pg_wait_steps<STAGES, kLoads>(nk - 2 - kt);
      pg_barrier();
    }
    return;
  }
  const int l16 = lane & 15, g = lane >> 4;
  f32x4 acc[2][kRB];  // [16 columns][16 rows]: lane holds columns 4 g .. + 3 of row l16
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) acc[d][rb] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Frag {
    bf16x8 w[2], x[kRB];
  };
  auto read_frag = [&](Frag& f, int stage, int ks) {
    const uint8_t* wl = smem + stage * kStageBytes;
    const uint8_t* xl = wl + kWBytes;
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const int key = 32 * ks + 4 * g + (l16 >> 2);
      const int col = 32 * wave + 16 * d + 4 * (l16 & 3);
      const int off = (((col >> 3) ^ ((key & 7) << 1)) << 4) + (((col >> 2) & 1) << 3);
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)(PgLds)(wl + key * 256 + off));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)(PgLds)(wl + (key + 16) * 256 + off));
      f.w[d] = as_bf16x8(__builtin_bit_cast(u32x2, lo), __builtin_bit_cast(u32x2, hi));
    }
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
      const int r = 16 * rb + l16, sw = (r >> 1) & 7;
      const int c = 4 * ks + (g >> 1);
      const uint8_t* row = xl + r * 128 + 8 * (g & 1);
      f.x[rb] = as_bf16x8(*reinterpret_cast<const u32x2*>(row + ((c ^ sw) << 4)),
                          *reinterpret_cast<const u32x2*>(row + (((c + 2) ^ sw) << 4)));
    }
  };
  auto mma = [&](const Frag& f) {
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) acc[d][rb] = mfma16(f.w[d], f.x[rb], acc[d][rb]);
  };
  Frag f0, f1;
  pg_barrier_lds();  // step 0 landed
  read_frag(f0, 0, 0);
  int stage = 0;
  for (int kt = 0; kt < nk; ++kt) {
    const int next = stage == STAGES - 1 ? 0 : stage + 1;
    read_frag(f1, stage, 1);
    __builtin_amdgcn_sched_barrier(0);
    mma(f0);
    pg_barrier_lds();  // step kt + 1 landed; this wave's reads of step kt done
    __builtin_amdgcn_sched_barrier(0);
    read_frag(f0, next, 0);  // past the last step: a stage read for nothing
    __builtin_amdgcn_sched_barrier(0);
    mma(f1);
    stage = next;
  }
#pragma unroll
  for (int rb = 0; rb < kRB; ++rb) {
    const int64_t r = m0 + 16 * rb + l16;
    if (r >= n_rows) continue;
    float* dst = part + (int64_t(blockIdx.y) * n_rows + r) * n_out + n0 + 32 * wave + 4 * g;
#pragma unroll
    for (int d = 0; d < 2; ++d) *reinterpret_cast<f32x4*>(dst + 16 * d) = acc[d][rb];
  }
}

struct GuCall {
  const uint16_t* x;
  int64_t k, width;
  SiluEp ep;
  hipStream_t stream;
};

template <int BM, int BP, int NPROD, int STAGES, int WM>
hipError_t gu_pc(const GuCall& c, int64_t n) {
  return pair_launch(pair_pc_kernel<SiluEp, BM, BP, NPROD, STAGES, WM>, BM, BP,
                     PcShape<BM, BP, NPROD, STAGES, WM>::kThreads, c.x, n, c.k, c.width, c.ep,
                     c.stream);
}

// Up to 128 rows the weights stream: 24 pairs a workgroup while that is one round of workgroups
// (width 6144 at 64 rows: 13.4 us, 32 pairs 14.5), else 48 (width 12288: 256 workgroups; 32 pairs
// make one and a half rounds, 51.6 us at 64 rows against 46.4, before the starts were spread).
// Then 128-row tiles while they fit one round (256 rows of width 12288: 57 us, 256-row tiles 85),
// then 256-row tiles. Against a library product over both weights and a separate SiLU pass, k
// 4096, width 12288, cold weights (us): 64 rows 49.6 -> 36.9, 128 rows 52.9 -> 42.5, 256 rows 69 ->
// 57, 512 rows 95 -> 89, 1024 rows 185 -> 176; 384 rows 84 against 86, 640 rows 130 against 157,
// 1900 rows 316 against 340: a caller gains while the tiles fill their rounds.
hipError_t gu_launch(const GuCall& c, int64_t n) {
  const int64_t cus = pg_device_cus();
  if (n <= 128) {
    const bool narrow = c.width / 24 <= cus;
    if (n <= 64) return narrow ? gu_pc<64, 24, 2, 8, 4>(c, n) : gu_pc<64, 48, 4, 8, 4>(c, n);
    return narrow ? gu_pc<128, 24, 2, 6, 4>(c, n) : gu_pc<128, 48, 4, 5, 4>(c, n);
  }
  if ((n + 127) / 128 * (c.width / 96) <= cus) return gu_pc<128, 96, 4, 4, 2>(c, n);
  return pair_launch(pair_gemm_kernel<SiluEp>, kPgBM, kPgBP, kPgThreads, c.x, n, c.k, c.width,
                     c.ep, c.stream);
}

}  // namespace
}  // namespace fdl

extern "C" int fdl_gate_up_silu(const void* x, const void* w_gate, const void* w_up,
                                int64_t n_rows, int64_t k, int64_t width, int64_t out_chunks,
                                void* out, void* stream) {
  using namespace fdl;
  FDL_REQUIRE(n_rows >= 0 && n_rows < (int64_t(1) << 31), FDL_ERR_SHAPE,
              "fdl_gate_up_silu: n_rows = %lld out of range", (long long)n_rows);
  FDL_REQUIRE(k >= 256 && k % 128 == 0 && k <= (1 << 16), FDL_ERR_UNSUPPORTED,
              "fdl_gate_up_silu: k = %lld (a multiple of 128 from 256 to 65536 is implemented)",
              (long long)k);
  FDL_REQUIRE(width >= 96 && width % 96 == 0 && width < (int64_t(1) << 24), FDL_ERR_UNSUPPORTED,
              "fdl_gate_up_silu: width = %lld (a multiple of 96 is implemented)",
              (long long)width);
  FDL_REQUIRE(out_chunks >= 1 && width % (8 * out_chunks) == 0, FDL_ERR_UNSUPPORTED,
              "fdl_gate_up_silu: out_chunks = %lld must divide width / 8 = %lld",
              (long long)out_chunks, (long long)(width / 8));
  if (n_rows == 0) return ok();
  FDL_REQUIRE_PTR(x);
  FDL_REQUIRE_PTR(w_gate);
  FDL_REQUIRE_PTR(w_up);
  FDL_REQUIRE_PTR(out);
  FDL_REQUIRE_ALIGNED(x, 16);
  FDL_REQUIRE_ALIGNED(w_gate, 16);
  FDL_REQUIRE_ALIGNED(w_up, 16);
  FDL_REQUIRE_ALIGNED(out, 16);
  GuCall c;
  c.x = static_cast<const uint16_t*>(x);
  c.k = k;
  c.width = width;
  c.ep.wg = static_cast<const uint16_t*>(w_gate);
  c.ep.wu = static_cast<const uint16_t*>(w_up);
  c.ep.out = static_cast<uint16_t*>(out);
  c.ep.k = static_cast<int>(k);
  c.ep.chunk = static_cast<int>(width / out_chunks);
  c.ep.n_rows = n_rows;
  c.stream = static_cast<hipStream_t>(stream);
  FDL_HIP_CHECK(gu_launch(c, n_rows));
  return ok();
}

extern "C" int fdl_linear_partials(const void* x, const void* w, int64_t n_rows, int64_t k,
                                   int64_t n_out, int64_t n_split, int32_t transposed,
                                   float* part, void* stream) {
  using namespace fdl;
  FDL_REQUIRE(n_rows >= 0 && n_rows < (int64_t(1) << 22), FDL_ERR_SHAPE,
              "fdl_linear_partials: n_rows = %lld out of range", (long long)n_rows);
  FDL_REQUIRE(n_split >= 1 && n_split <= 64 && k >= 64 && k <= (1 << 20) && k % (64 * n_split) == 0,
              FDL_ERR_UNSUPPORTED,
              "fdl_linear_partials: k = %lld (n_split = %lld chunks of a multiple of 64)",
              (long long)k, (long long)n_split);
  FDL_REQUIRE(n_out >= 128 && n_out % 128 == 0 && n_out <= (1 << 20), FDL_ERR_UNSUPPORTED,
              "fdl_linear_partials: n_out = %lld (a multiple of 128 is implemented)",
              (long long)n_out);
  if (n_rows == 0) return ok();
  FDL_REQUIRE_PTR(x);
  FDL_REQUIRE_PTR(w);
  FDL_REQUIRE_PTR(part);
  FDL_REQUIRE_ALIGNED(x, 16);
  FDL_REQUIRE_ALIGNED(w, 16);
  FDL_REQUIRE_ALIGNED(part, 16);
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const auto* xp = static_cast<const uint16_t*>(x);
  const auto* wp = static_cast<const uint16_t*>(w);
  const bool small = n_rows <= 64;
  if (transposed) {
    const int64_t bm = small ? 64 : 128;
    const dim3 grid(static_cast<unsigned>(n_out / 128), static_cast<unsigned>(n_split),
                    static_cast<unsigned>((n_rows + bm - 1) / bm));
    hipLaunchKernelGGL((small ? part_t_kernel<64, 6> : part_t_kernel<128, 5>), grid, dim3(512), 0,
                       st, xp, wp, n_rows, static_cast<int>(k), static_cast<int>(k / n_split),
                       static_cast<int>(n_out), part);
    FDL_HIP_CHECK(hipGetLastError());
    return ok();
  }
  const PartEp ep = {wp, part, n_rows, static_cast<int>(k), static_cast<int>(n_out)};
  if (small)
    FDL_HIP_CHECK((pair_launch(pair_pc_kernel<PartEp, 64, 32, 4, 8, 2>, 64, 32,
                               PcShape<64, 32, 4, 8, 2>::kThreads, xp, n_rows, k, n_out / 2, ep, st,
                               n_split)));
  else
    FDL_HIP_CHECK((pair_launch(pair_pc_kernel<PartEp, 128, 32, 4, 6, 2>, 128, 32,
                               PcShape<128, 32, 4, 6, 2>::kThreads, xp, n_rows, k, n_out / 2, ep,
                               st, n_split)));
  return ok();
}
