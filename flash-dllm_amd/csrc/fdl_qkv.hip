// Fused QKV projection + rotate-half RoPE + direct K/V cache write (gfx950, bf16 MFMA).
//
// Follows _flash_qkv_proj_cache_fwd (flash_cache_triton.py:15-100) and
// _flash_verify_qkv_proj_fwd (flash_cache_triton.py:255-338):
//   q~ = x_r W_q^T, k~ = x_r W_k^T, v~ = x_r W_v^T           (fp32 accumulation)
//   Q[r, h*128 + c]      = q~_c cos[s, c]      - q~_{c+64} sin[s, c]
//   Q[r, h*128 + c + 64] = q~_{c+64} cos[s, c+64] + q~_c sin[s, c+64]       (c < 64)
//   K is rotated the same way; V is not rotated.
//   Q goes to packed row r; K/V go to cache row slot[r] (or packed row r for verify).
//
// The output columns are handled as RoPE pairs (c, c + 64) of a head: pair p of the
// 3 * n_heads * 64 pairs is column c = p % 64 of head (p / 64) % n_heads of matrix
// p / (64 * n_heads). A tile is a block of rows times a block of pairs, and a wavefront
// computes both members of its pairs, so lane l holds (c, c + 64) of the same rows in the
// same accumulator slot and RoPE runs in registers before the bf16 stores.
//
// The products run on the two kernels of the pair GEMM (fdl_pair_gemm.h), whose epilogue here
// rotates and writes 8-pair groups with 16-byte stores. Three kinds of tiles, chosen by the
// number of rows (qkv_split):
//  * many rows: 256 rows x 96 pairs (pair_gemm_kernel);
//  * more than 128 rows: 128 rows x 96 pairs, 4 stages of 40 KB, all of LDS (pair_pc_kernel).
//    512 rows at d_model 4096 give one tile per CU;
//  * up to 128 rows (weight streaming, HBM-bound): 64 or 128 rows x 24 or 32 pairs
//    (pair_pc_kernel), 8 stages of 14 or 16 KB or 6 of 22 or 24 KB, so each workgroup keeps 5-7
//    weight steps in flight.
#include <algorithm>

#include "fdl_device.h"
#include "fdl_host.h"
#include "fdl_pair_gemm.h"

namespace fdl {
namespace {

constexpr int kHeadDim = 128;
constexpr int kHalf = 64;
constexpr int kDAlign = 256;  // d_model must be a multiple of this

struct QkvArgs {
  const uint16_t* x;
  const uint16_t* w[3];
  const float* sin;
  const float* cos;
  const int64_t* slot;
  const int64_t* rope_row;
  uint16_t* q_out;
  uint16_t* k_out;
  uint16_t* v_out;
  int64_t n_rows;
  int64_t n_rope_rows;
  int64_t n_kv_rows;
  int d_model;
  int n_heads;
  int kv_packed;
  int rope_half;  // sin/cos rows repeat their first half: read only that half
};

// Destinations of row r: dq = Q row, dkv = K/V row (cache slot, or the packed row), rope =
// sin/cos row. A row past n_rows, or with an out-of-range slot or rope row, gets -1 in all
// three (skipped in all three outputs).
__device__ __forceinline__ void row_dest(const QkvArgs& a, int64_t r, int64_t& dq, int64_t& dkv,
                                         int64_t& rope) {
  dq = dkv = rope = -1;
  if (r < a.n_rows) {
    const int64_t s = a.slot[r];
    const int64_t rr = a.rope_row ? a.rope_row[r] : s;
    const bool rope_ok = rr >= 0 && rr < a.n_rope_rows;
    const bool slot_ok = a.kv_packed || (s >= 0 && s < a.n_kv_rows);
    if (rope_ok && slot_ok) {
      dq = r;
      dkv = a.kv_packed ? r : s;
      rope = rr;
    }
  }
}

// 8 consecutive pairs (c0 .. c0 + 7 of one head; lo = q~_c, hi = q~_{c+64}) of one row:
// load() reads the fp32 sums from LDS and the sin/cos values, store() rotates and writes two
// 16-byte bf16 chunks. c0 is a multiple of 8, so the sin/cos reads and both stores are
// 16-byte aligned. A group whose row has no destination (dst < 0) reads and writes nothing.
struct EpGroup {
  f32x4 lo[2], hi[2];
  f32x4 s1[2], s2[2], c1[2], c2[2];
  int64_t dst;
  int mat, head, c0;

  __device__ __forceinline__ void load(const QkvArgs& a, const float* src, int hi_off, int m,
                                       int rem, int64_t d, int64_t rope) {
    mat = m;
    head = rem >> 6;
    c0 = rem & 63;
    dst = d;
    if (d < 0) return;
    lo[0] = *reinterpret_cast<const f32x4*>(src);
    lo[1] = *reinterpret_cast<const f32x4*>(src + 4);
    hi[0] = *reinterpret_cast<const f32x4*>(src + hi_off);
    hi[1] = *reinterpret_cast<const f32x4*>(src + hi_off + 4);
    if (m < 2) {
      const float* sn = a.sin + rope * kHeadDim + c0;
      const float* cs = a.cos + rope * kHeadDim + c0;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        s1[h] = *reinterpret_cast<const f32x4*>(sn + 4 * h);
        c1[h] = *reinterpret_cast<const f32x4*>(cs + 4 * h);
        if (a.rope_half) {
          s2[h] = s1[h];
          c2[h] = c1[h];
        } else {
          s2[h] = *reinterpret_cast<const f32x4*>(sn + kHalf + 4 * h);
          c2[h] = *reinterpret_cast<const f32x4*>(cs + kHalf + 4 * h);
        }
      }
    }
  }

  __device__ __forceinline__ void store(const QkvArgs& a) {
    if (dst < 0) return;
    float l[8], r[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      l[j] = lo[j >> 2][j & 3];
      r[j] = hi[j >> 2][j & 3];
    }
    if (mat < 2) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int h = j >> 2, e = j & 3;
        const float rlo = l[j] * c1[h][e] - r[j] * s1[h][e];
        const float rhi = r[j] * c2[h][e] + l[j] * s2[h][e];
        l[j] = rlo;
        r[j] = rhi;
      }
    }
    const u32x4 wlo = {pack_bf16x2(l[0], l[1]), pack_bf16x2(l[2], l[3]), pack_bf16x2(l[4], l[5]),
                       pack_bf16x2(l[6], l[7])};
    const u32x4 whi = {pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3]), pack_bf16x2(r[4], r[5]),
                       pack_bf16x2(r[6], r[7])};
    uint16_t* base = mat == 0 ? a.q_out : (mat == 1 ? a.k_out : a.v_out);
    uint16_t* d = base + dst * a.d_model + int64_t(head) * kHeadDim + c0;
    // non-temporal: the whole grid writes its Q/K/V rows at once at the end (1.5% faster at
    // 512 rows, 2% at 6842; the attention that reads them next is unchanged)
    __builtin_nontemporal_store(wlo, reinterpret_cast<u32x4*>(d));
    __builtin_nontemporal_store(whi, reinterpret_cast<u32x4*>(d + kHalf));
  }
};

// Epilogue of the pair GEMM (fdl_pair_gemm.h).
struct RopeEp {
  QkvArgs a;
  struct Row {
    // K/V row, sin/cos row (both below 2^31: a cache or table row takes at least 512 bytes); -1:
    // not stored
    int dkv, rope;
  };
  __device__ __forceinline__ const uint16_t* wrow(int p, int hi) const {
    const int pairs_per_mat = a.n_heads * kHalf;
    const int mat = p / pairs_per_mat, rem = p - mat * pairs_per_mat;
    // differences of the uniform pointers: an index that differs by lane would read the pointer
    // from the kernel arguments in memory, and each wait for it delays the first loads
    const uint64_t w0 = reinterpret_cast<uint64_t>(a.w[0]), w1 = reinterpret_cast<uint64_t>(a.w[1]),
                   w2 = reinterpret_cast<uint64_t>(a.w[2]);
    const uint64_t w = w0 + (mat >= 1 ? w1 - w0 : 0) + (mat >= 2 ? w2 - w1 : 0);
    return reinterpret_cast<const uint16_t*>(w) +
           int64_t((rem >> 6) * kHeadDim + (rem & 63) + kHalf * hi) * a.d_model;
  }
  __device__ __forceinline__ Row row(int64_t r) const {
    int64_t dq, dkv, rope;
    row_dest(a, r, dq, dkv, rope);
    return {static_cast<int>(dkv), static_cast<int>(rope)};
  }
  struct Group {
    EpGroup g;
    __device__ __forceinline__ void load(const RopeEp& ep, const Row& d, int64_t r, int p,
                                         const float* lo, int hi_off, bool mine) {
      const int pairs_per_mat = ep.a.n_heads * kHalf;
      const int mat = p / pairs_per_mat, rem = p - mat * pairs_per_mat;
      g.load(ep.a, lo, hi_off, mat, rem,
             !mine || d.rope < 0 ? -1 : (mat == 0 ? r : int64_t(d.dkv)), d.rope);
    }
    __device__ __forceinline__ void store(const RopeEp& ep) { g.store(ep.a); }
  };
};

}  // namespace
}  // namespace fdl

namespace fdl {
namespace {

constexpr int kPcBM = 128, kPcBP = 96;

// Rows of a call and the shapes that run them: the first `wide` on 256-row tiles, the next
// `mid` on 128-row tiles, the rest (at most 128) streaming the weights.
struct QkvSplit {
  int64_t wide, mid;
};

// Up to 128 rows the projection streams the weights (128 x 32-pair tiles take 45 us at 192 rows
// against 36 us for the 128 x 96-pair ones). Beyond, two shapes feed the MFMAs: a round of 256-row
// tiles (80 us at d_model 4096, one workgroup per CU) covers as much as two rounds of 128-row
// tiles (47 us each), so whole rounds go to the 256-row tiles and a part of a round to what covers
// it soonest: 512 rows to 128-row tiles (54 us; 256-row tiles fill half of the device and take
// 75), 1024 rows to 256-row tiles (100 -> 86 us), 1536 rows a round of each (140 -> 130 us), 576
// rows a round of 128-row tiles and a 64-row stream (69 us; 256-row tiles 76), 640 rows to
// 256-row tiles (95 -> 76 us). The split with the smallest sum is taken; a launch counts as
// kLaunchUs. At other widths the rounds' costs keep their proportions: over 147 row counts at
// d_model 512 to 8192, timed against every other split, the choice was within 1.6% of the fastest
// but for five (2-6%), and costs scaled with d_model beside a fixed launch choose differently at
// four, by 2% at most.
constexpr int kWideRoundUs = 80, kMidRoundUs = 47, kLaunchUs = 4;
constexpr int kStreamUs[2] = {17, 21};  // up to 64 rows, up to 128
constexpr int kStreamRows = 128;

QkvSplit qkv_split(int64_t n_rows, int64_t n_pairs) {
  const int64_t cus = pg_device_cus();
  auto rounds = [&](int64_t rows, int bm, int bp) {
    return ((rows + bm - 1) / bm * (n_pairs / bp) + cus - 1) / cus;
  };
  auto cost = [&](const QkvSplit& s) {
    const int64_t rest = n_rows - s.wide - s.mid;
    int64_t c = 0;
    if (s.wide) c += rounds(s.wide, kPgBM, kPgBP) * kWideRoundUs + kLaunchUs;
    if (s.mid) c += rounds(s.mid, kPcBM, kPcBP) * kMidRoundUs + kLaunchUs;
    if (rest) c += rounds(rest, kStreamRows, 32) * kStreamUs[rest > 64] + kLaunchUs;
    return c;
  };
  if (n_rows <= kStreamRows) return {0, 0};
  QkvSplit best = {n_rows, 0};
  // wide tiles in whole, the rest on 128-row tiles with or without its last, partial tile (a
  // rest of more than two rounds of 256-row tiles is never the better choice)
  const int64_t whole = n_rows / kPgBM, two_rounds = 2 * (cus / (n_pairs / kPgBP) + 1);
  for (int64_t q = std::max<int64_t>(0, whole - two_rounds); q <= whole; ++q) {
    const int64_t wide = q * kPgBM, rest = n_rows - wide;
    const int64_t full = rest / kPcBM * kPcBM;
    for (const int64_t mid : {rest, full, rest <= kStreamRows ? 0 : rest}) {
      const QkvSplit s = {wide, mid};
      if (cost(s) < cost(best)) best = s;
    }
  }
  return best;
}

// Rows [r0, r0 + n) of the call described by `args`.
QkvArgs qkv_rows(QkvArgs args, int64_t r0, int64_t n) {
  const int64_t D = args.d_model;
  args.x += r0 * D;
  args.slot += r0;
  if (args.rope_row) args.rope_row += r0;
  args.q_out += r0 * D;
  if (args.kv_packed) {
    args.k_out += r0 * D;
    args.v_out += r0 * D;
    args.n_kv_rows = n;
  }
  args.n_rows = n;
  return args;
}

hipError_t qkv_launch(void (*kernel)(PairGemmTiles, RopeEp), int bm, int bp, int threads,
                      const QkvArgs& args, hipStream_t stream) {
  return pair_launch(kernel, bm, bp, threads, args.x, args.n_rows, args.d_model,
                     3 * int64_t(args.n_heads) * kHalf, RopeEp{args}, stream);
}

template <int BM, int BP, int NPROD, int STAGES, int WM>
hipError_t qkv_launch_pc(const QkvArgs& args, hipStream_t stream) {
  return qkv_launch(pair_pc_kernel<RopeEp, BM, BP, NPROD, STAGES, WM>, BM, BP,
                    PcShape<BM, BP, NPROD, STAGES, WM>::kThreads, args, stream);
}

}  // namespace
}  // namespace fdl

extern "C" int fdl_qkv_rope_cache(const void* x, const void* wq, const void* wk,
                                  const void* wv, const float* rope_sin, const float* rope_cos,
                                  int64_t n_rope_rows, const int64_t* slot,
                                  const int64_t* rope_row, int64_t n_rows, int64_t d_model,
                                  int64_t n_heads, int64_t head_dim, void* q_out, void* k_out,
                                  void* v_out, int64_t n_kv_rows, int32_t flags,
                                  void* stream) {
  using namespace fdl;
  FDL_REQUIRE(n_rows >= 0, FDL_ERR_SHAPE, "fdl_qkv_rope_cache: n_rows = %lld < 0",
              (long long)n_rows);
  FDL_REQUIRE(head_dim == kHeadDim, FDL_ERR_UNSUPPORTED,
              "fdl_qkv_rope_cache: head_dim = %lld (only 128 is implemented)",
              (long long)head_dim);
  FDL_REQUIRE(n_heads >= 1 && d_model == n_heads * head_dim, FDL_ERR_SHAPE,
              "fdl_qkv_rope_cache: d_model (%lld) != n_heads (%lld) * head_dim",
              (long long)d_model, (long long)n_heads);
  FDL_REQUIRE(d_model <= (1 << 16), FDL_ERR_UNSUPPORTED,
              "fdl_qkv_rope_cache: d_model = %lld too large", (long long)d_model);
  FDL_REQUIRE(d_model % kDAlign == 0, FDL_ERR_UNSUPPORTED,
              "fdl_qkv_rope_cache: d_model = %lld is not a multiple of %d", (long long)d_model,
              kDAlign);
  FDL_REQUIRE((flags & ~(FDL_QKV_KV_PACKED | FDL_QKV_ROPE_HALVES_EQUAL)) == 0, FDL_ERR_SHAPE,
              "fdl_qkv_rope_cache: flags = %d has unknown bits", flags);
  const int kv_packed = (flags & FDL_QKV_KV_PACKED) ? 1 : 0;
  FDL_REQUIRE(!kv_packed || n_kv_rows == n_rows, FDL_ERR_SHAPE,
              "fdl_qkv_rope_cache: packed K/V needs n_kv_rows == n_rows");
  FDL_REQUIRE(n_kv_rows >= 0 && n_rope_rows >= 0, FDL_ERR_SHAPE,
              "fdl_qkv_rope_cache: negative table size");
  if (n_rows == 0) return ok();
  FDL_REQUIRE_PTR(x);
  FDL_REQUIRE_PTR(wq);
  FDL_REQUIRE_PTR(wk);
  FDL_REQUIRE_PTR(wv);
  FDL_REQUIRE_PTR(rope_sin);
  FDL_REQUIRE_PTR(rope_cos);
  FDL_REQUIRE_PTR(slot);
  FDL_REQUIRE_PTR(q_out);
  FDL_REQUIRE_PTR(k_out);
  FDL_REQUIRE_PTR(v_out);
  FDL_REQUIRE_ALIGNED(x, 16);
  FDL_REQUIRE_ALIGNED(wq, 16);
  FDL_REQUIRE_ALIGNED(wk, 16);
  FDL_REQUIRE_ALIGNED(wv, 16);
  FDL_REQUIRE_ALIGNED(rope_sin, 16);
  FDL_REQUIRE_ALIGNED(rope_cos, 16);
  FDL_REQUIRE_ALIGNED(q_out, 16);
  FDL_REQUIRE_ALIGNED(k_out, 16);
  FDL_REQUIRE_ALIGNED(v_out, 16);
  FDL_REQUIRE((n_rows + 63) / 64 * (3 * n_heads * kHalf / 32) < (int64_t(1) << 31),
              FDL_ERR_UNSUPPORTED, "fdl_qkv_rope_cache: %lld rows is too many",
              (long long)n_rows);
  QkvArgs args;
  args.x = static_cast<const uint16_t*>(x);
  args.w[0] = static_cast<const uint16_t*>(wq);
  args.w[1] = static_cast<const uint16_t*>(wk);
  args.w[2] = static_cast<const uint16_t*>(wv);
  args.sin = rope_sin;
  args.cos = rope_cos;
  args.slot = slot;
  args.rope_row = rope_row;
  args.q_out = static_cast<uint16_t*>(q_out);
  args.k_out = static_cast<uint16_t*>(k_out);
  args.v_out = static_cast<uint16_t*>(v_out);
  args.n_rows = n_rows;
  args.n_rope_rows = n_rope_rows;
  args.n_kv_rows = n_kv_rows;
  args.d_model = static_cast<int>(d_model);
  args.n_heads = static_cast<int>(n_heads);
  args.kv_packed = kv_packed;
  args.rope_half = (flags & FDL_QKV_ROPE_HALVES_EQUAL) ? 1 : 0;
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const QkvSplit split = qkv_split(n_rows, 3 * n_heads * kHalf);
  const int64_t rest = n_rows - split.wide - split.mid;
  if (split.wide > 0)
    FDL_HIP_CHECK(qkv_launch(pair_gemm_kernel<RopeEp>, kPgBM, kPgBP, kPgThreads,
                             qkv_rows(args, 0, split.wide), st));
  if (split.mid > 0)
    FDL_HIP_CHECK((qkv_launch_pc<kPcBM, kPcBP, 4, 4, 2>(qkv_rows(args, split.wide, split.mid), st)));
  if (rest > 0) {
    const QkvArgs tail = qkv_rows(args, split.wide + split.mid, rest);
    // 24-pair tiles, with two producers, which load as fast as more, where they are one round of
    // workgroups on more than half of the CUs (d_model 4096: all 256, against the 192 of 32-pair
    // tiles), and of 65 to 128 rows on more than 7/8. Without / with them, cold and warm weights
    // (us): d_model 4096, 40 rows 22.1 -> 20.9, 17.7 -> 18.3, 64 rows 24.8 -> 23.1, 18.1 -> 18.7, 100
    // rows 29.5 -> 28.3, 19.5 -> 21.1; 2560, 64 rows 17.9 -> 17.3, 12.8 -> 12.1. A model's weights are
    // cold: its other layers come between. Elsewhere they lose more than that warm: 2048, 64 rows
    // 13.5 -> 12.8, 9.7 -> 10.2, 100 rows 16.0 -> 15.8, 10.7 -> 12.3; 3072, 65 rows 21.1 -> 19.9, 14.6
    // -> 15.8; 1024, 64 rows 8.7 -> 8.4, 7.0 -> 7.3.
    const int64_t cus = pg_device_cus(), tiles = n_heads * 3 * kHalf / 24;
    const bool narrow = tiles <= cus && (rest <= 64 ? 2 * tiles > cus : 8 * tiles > 7 * cus);
    FDL_HIP_CHECK((rest <= 64 ? (narrow ? qkv_launch_pc<64, 24, 2, 8, 4>(tail, st)
                                        : qkv_launch_pc<64, 32, 4, 8, 2>(tail, st))
                              : (narrow ? qkv_launch_pc<128, 24, 2, 6, 4>(tail, st)
                                        : qkv_launch_pc<128, 32, 4, 6, 2>(tail, st))));
  }
  return ok();
}
