// Gate and up projections of the MLP with the SiLU gate in one pass (gfx950, bf16 MFMA).
//
// Replaces ff_proj(x), up_proj(x), act and the product (flash_cache_triton.py:628-633):
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

struct GuCall {
  const uint16_t* x;
  int64_t k, width;
  SiluEp ep;
  hipStream_t stream;
};

template <int BM, int BP, int STAGES, int WM>
hipError_t gu_pc(const GuCall& c, int64_t n) {
  return pair_launch(pair_pc_kernel<SiluEp, BM, BP, 4, STAGES, WM>, BM, BP,
                     PcShape<BM, BP, 4, STAGES, WM>::kThreads, c.x, n, c.k, c.width, c.ep,
                     c.stream);
}

// Up to 128 rows the weights stream: 32 pairs a workgroup while that is one round of
// workgroups, else 48 (width 12288: 256 workgroups; 32 pairs make one and a half rounds, 51.6
// us at 64 rows against 46.4). Then 128-row tiles while they fit one round (256 rows of width
// 12288: 61 us, 256-row tiles 85), then 256-row tiles. Against a library product over both
// weights and a separate SiLU pass, k 4096, width 12288, cold weights (us): 64 rows 50.3 ->
// 37.1, 128 rows 53.5 -> 45.3, 256 rows 67 -> 61, 384 rows 87 -> 93, 512 rows 98 -> 95, 640 rows
// 132 -> 158, 1024 rows 185 -> 177, 1900 rows 308 -> 330: a caller gains while the 128-row tiles
// fit one round, and loses or wins little beyond.
hipError_t gu_launch(const GuCall& c, int64_t n) {
  const int64_t cus = pg_device_cus();
  if (n <= 128) {
    const bool narrow = c.width / 32 <= cus;
    if (n <= 64) return narrow ? gu_pc<64, 32, 8, 2>(c, n) : gu_pc<64, 48, 8, 4>(c, n);
    return narrow ? gu_pc<128, 32, 6, 2>(c, n) : gu_pc<128, 48, 5, 4>(c, n);
  }
  if ((n + 127) / 128 * (c.width / 96) <= cus) return gu_pc<128, 96, 4, 2>(c, n);
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
