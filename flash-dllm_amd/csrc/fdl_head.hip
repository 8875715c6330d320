// Confidence of the LM-head rows (gfx950): the float64 softmax maximum and its token, or
// the float64 softmax probability of a given token, one workgroup per row.
//
// Replaces, for bf16 logits,
//   p = softmax(logits.to(float64), -1); x0_p, x0 = max(p, -1)        (generate.py:218, :320)
//   p = softmax(logits.to(float64), -1).gather(1, tok)                  (generate.py:337)
// For row r with maximum m (first index i_max):
//   s = sum_j exp(x_j - m) in float64; max probability = exp(0) / s = 1 / s;
//   probability of token t = exp(x_t - m) / s.
// A row with a NaN, a +inf or only -inf logits has a softmax of NaNs: probability NaN and
// index 0, as torch.max returns for it.
// bf16 -> float -> double is exact. Of few values (below kTableVocab) and where |m| is large,
// the terms are the float64 softmax's and only the order of the float64 sum differs from
// torch's reduction; otherwise s = sum_j exp(x_j) / exp(m), whose terms differ by an ulp or
// two. s >= 1 either way, so no probability exceeds 1, and a row whose maximum holds everything
// has exactly 1.
#include <stdint.h>

#include "fdl_device.h"
#include "fdl_host.h"

namespace fdl {
namespace {

constexpr int kConfThreads = 1024;  // one workgroup per row
constexpr int kConfWaves = kConfThreads / kWave;
constexpr int kDirectThreads = 256;

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) {
  return __builtin_bit_cast(float, w & 0xffff0000u);
}

// (value, index) with the larger value, the smaller index among equal values.
__device__ __forceinline__ void arg_max_merge(float& m, int64_t& i, float m2, int64_t i2) {
  if (m2 > m || (m2 == m && i2 < i)) {
    m = m2;
    i = i2;
  }
}

// vocab below kTableVocab: every exponential computed. vocab % 8 == 0 and 16-byte aligned rows
// (checked on the host).
__global__ __launch_bounds__(kDirectThreads) void softmax_conf_direct_kernel(
    const uint16_t* __restrict__ logits, int64_t vocab, const int64_t* __restrict__ token,
    double* __restrict__ prob, int64_t* __restrict__ arg) {
  __shared__ float s_m[kDirectThreads / kWave];
  __shared__ int64_t s_i[kDirectThreads / kWave];
  __shared__ double s_sum[kDirectThreads / kWave];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint16_t* x = logits + int64_t(blockIdx.x) * vocab;
  const int64_t n8 = vocab / 8;

  // pass 1: maximum and its first index (each thread visits increasing indices; a thread
  // that visits none keeps the index past every real one)
  float m = -INFINITY;
  int64_t im = INT64_MAX;
  for (int64_t c = tid; c < n8; c += kDirectThreads) {
    const u32x4 v = ld16(x + 8 * c);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a = bf16_lo(v[j]), b = bf16_hi(v[j]);
      if (a > m) {
        m = a;
        im = 8 * c + 2 * j;
      }
      if (b > m) {
        m = b;
        im = 8 * c + 2 * j + 1;
      }
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float m2 = __shfl_xor(m, off);
    const int64_t i2 = __shfl_xor(im, off);
    arg_max_merge(m, im, m2, i2);
  }
  if (lane == 0) {
    s_m[wave] = m;
    s_i[wave] = im;
  }
  __syncthreads();
  m = s_m[0];
  im = s_i[0];
#pragma unroll
  for (int w = 1; w < kDirectThreads / kWave; ++w) arg_max_merge(m, im, s_m[w], s_i[w]);

  // pass 2: float64 sum of exp(x - m); per-thread partials, then a fixed reduction tree
  const double md = static_cast<double>(m);
  double s = 0.0;
  for (int64_t c = tid; c < n8; c += kDirectThreads) {
    const u32x4 v = ld16(x + 8 * c);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s += exp(static_cast<double>(bf16_lo(v[j])) - md);
      s += exp(static_cast<double>(bf16_hi(v[j])) - md);
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off);
  if (lane == 0) s_sum[wave] = s;
  __syncthreads();
  if (tid == 0) {
    double sum = s_sum[0];
#pragma unroll
    for (int w = 1; w < kDirectThreads / kWave; ++w) sum += s_sum[w];
    double p;
    if (token) {
      const int64_t t = token[blockIdx.x];
      p = t >= 0 && t < vocab ? exp(static_cast<double>(bf2f(x[t])) - md) / sum : 0.0;
    } else {
      p = 1.0 / sum;
    }
    prob[blockIdx.x] = p;
    // A row with a NaN (no comparison above selects it, but it makes the sum NaN), a +inf or
    // only -inf logits has a softmax of NaNs; torch.max of it returns index 0.
    if (arg) arg[blockIdx.x] = __builtin_isfinite(m) && sum == sum ? im : 0;
  }
}

// ---- vocab from kTableVocab on
//
// What bounds the row: 126464 float64 exponentials by one workgroup are far more work than its
// 253 KB of reads (64 us of the 70 us at 256 rows when each is computed). bf16 logits have few
// distinct values, so the exponentials of the common ones are tabulated once per row in LDS
// (4096 per row instead of 126464) and summed by look-up. The table is of exp(x), not exp(x -
// max): float64 holds it for |x| < 64 with the same relative precision, so a row whose maximum
// lies there is read once, its maximum found and its sum formed as the values arrive (with a
// table of exp(x - max) the look-ups began when the whole row had been read: 24.4 us at 256 rows
// of 126464 against 19.6). Other rows take a second pass that computes every exponential: their
// values mostly lie outside the table as well (a second table, of exp(x - max), took 51.7 us
// against 43.0 at 256 x 126464 N(0, 200^2) values, 12.2 against 9.7 at 32 x 16384 N(0, 40^2)).
// Measured (us), each exponential computed / tabulated: 256 rows of 126464 69.9 / 19.6, 32 rows
// 57.7 / 19.3, 512 rows of 32000 30.9 / 20.1; of a second pass: 256 rows of 126464 70.0 / 43.0,
// of 32000 16.5 / 15.3, of 16384 10.0 / 10.4, the one place that loses. What is left are the
// look-ups (random 8-byte LDS reads: the LDS is active a quarter of the cycles, 59% of that in
// bank conflicts, and wavefronts wait half of theirs) and their addresses: one row alone takes 17
// us. Below 16384 values the table costs more than it saves (512 rows of 8192: 10.0 computed, 14
// tabulated; of 16384: 16.9 and 16.4), so shorter rows keep the direct kernel.
constexpr int64_t kTableVocab = 16384;

// exp of the bf16 values with |x| in [2^-10, 2^6) (16 exponents, both signs) from a table of
// float64 values: a bf16 of those exponents is its sign, the low 4 bits of its exponent and its
// 7 fraction bits. Values outside (also 0, NaN, infinities) take exp() itself.
constexpr uint32_t kTabMagLo = 117u << 7;  // bits of 2^-10
constexpr uint32_t kTabMags = 16u << 7;
constexpr int kTabSize = 2 * kTabMags;  // 4096 values, 32 KB
constexpr float kTabLimit = 64.f;

// whether all 8 values of v are in the table (the smallest and the largest magnitude bits, two
// 16-bit halves at a time)
__device__ __forceinline__ bool in_table(u32x4 v) {
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  u16x2 lo, hi;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const u16x2 mag = __builtin_bit_cast(u16x2, v[j] & 0x7fff7fffu);
    lo = j ? __builtin_elementwise_min(lo, mag) : mag;
    hi = j ? __builtin_elementwise_max(hi, mag) : mag;
  }
  return min(lo[0], lo[1]) >= kTabMagLo && max(hi[0], hi[1]) < kTabMagLo + kTabMags;
}

// sum of the table's values over the 8 values of v (any bits read inside the table)
__device__ __forceinline__ double table_sum8(u32x4 v, const double* tab) {
  double s0 = 0.0, s1 = 0.0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t w = v[j];
    s0 += tab[(w & (kTabMags - 1)) | ((w >> 15) & 1u) * kTabMags];
    s1 += tab[((w >> 16) & (kTabMags - 1)) | (w >> 31) * kTabMags];
  }
  return s0 + s1;
}

__device__ __forceinline__ double exp_sum8(u32x4 v, double md) {
  double s = 0.0;
#pragma unroll 1
  for (int j = 0; j < 4; ++j) {
    s += exp(static_cast<double>(bf16_lo(v[j])) - md);
    s += exp(static_cast<double>(bf16_hi(v[j])) - md);
  }
  return s;
}

// tab[i] = exp(x) of the 4096 values
__device__ __forceinline__ void make_table(double* tab) {
#pragma unroll 1
  for (int i = 0; i < kTabSize / kConfThreads; ++i) {
    const uint32_t t = threadIdx.x + kConfThreads * i;
    const uint32_t low = t & (kTabMags - 1);
    // the magnitude of the range whose low 11 bits these are
    const uint32_t mag = kTabMagLo + ((low - kTabMagLo) & (kTabMags - 1));
    tab[t] = exp(static_cast<double>(bf2f(static_cast<uint16_t>(mag | (t / kTabMags) << 15))));
  }
}

// vocab % 8 == 0 and 16-byte aligned rows (checked on the host). Thread t takes the 16-byte
// chunks t, t + 1024, ..
__global__ __launch_bounds__(kConfThreads) void softmax_conf_kernel(
    const uint16_t* __restrict__ logits, int64_t vocab, const int64_t* __restrict__ token,
    double* __restrict__ prob, int64_t* __restrict__ arg) {
  __shared__ double tab[kTabSize];
  __shared__ float s_m[kConfWaves];
  __shared__ int64_t s_i[kConfWaves];
  __shared__ double s_sum[kConfWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint16_t* x = logits + int64_t(blockIdx.x) * vocab;
  const int64_t n8 = vocab / 8;
  const int n_own = static_cast<int>((n8 - tid + kConfThreads - 1) / kConfThreads);  // n8 >= 2048
  auto chunk = [&](int i) { return ld16(x + 8 * (tid + int64_t(kConfThreads) * min(i, n_own - 1))); };

  constexpr int kAhead = 4;
  u32x4 cur[kAhead];
#pragma unroll
  for (int u = 0; u < kAhead; ++u) cur[u] = chunk(u);  // arrive while the table is made
  make_table(tab);
  __syncthreads();

  // One pass: the maximum, the first own chunk that holds it (a NaN is never the maximum; it
  // makes the sum NaN) and the sum of exp(x). kAhead chunks are in flight. Chunks with values
  // outside the table wait in `rest` (the first 64): a wavefront would pay for every lane's one
  // by one, and a row that takes a second pass need not sum them in the first.
  float m = -INFINITY;
  int best = 0;
  double s = 0.0;
  uint64_t rest = 0;
  for (int i0 = 0; i0 < n_own; i0 += kAhead) {
    u32x4 next[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) next[u] = chunk(i0 + kAhead + u);
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      if (i0 + u < n_own) {
        const u32x4 v = cur[u];
        float top = fmaxf(bf16_lo(v[0]), bf16_hi(v[0]));
#pragma unroll
        for (int j = 1; j < 4; ++j) top = fmaxf(top, fmaxf(bf16_lo(v[j]), bf16_hi(v[j])));
        best = top > m ? i0 + u : best;
        m = fmaxf(m, top);
        if (in_table(v))
          s += table_sum8(v, tab);
        else if (i0 + u < 64)
          rest |= uint64_t(1) << (i0 + u);
        else
          s += exp_sum8(v, 0.0);
      }
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) cur[u] = next[u];
  }

  // the row's maximum and its first index (only threads that hold it look)
  const float m_own = m;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  if (lane == 0) s_m[wave] = m;
  __syncthreads();
  m = s_m[0];
#pragma unroll
  for (int w = 1; w < kConfWaves; ++w) m = fmaxf(m, s_m[w]);
  const double md = static_cast<double>(m);
  int64_t im = INT64_MAX;
  if (m_own == m) {
    const u32x4 v = chunk(best);
    const int64_t c = 8 * (tid + int64_t(kConfThreads) * best);
#pragma unroll
    for (int j = 3; j >= 0; --j) {
      if (bf16_hi(v[j]) == m) im = c + 2 * j + 1;
      if (bf16_lo(v[j]) == m) im = c + 2 * j;
    }
  }
  // a maximum outside the table's range: sums of exp(x) may overflow or vanish
  const bool ranged = m >= -kTabLimit && m < kTabLimit;
  if (!ranged) {
    s = 0.0;
    for (int i = 0; i < n_own; ++i) s += exp_sum8(chunk(i), md);
  } else {
    for (; rest; rest &= rest - 1) s += exp_sum8(chunk(__builtin_ctzll(rest)), 0.0);
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    s += __shfl_xor(s, off);
    im = min(im, __shfl_xor(im, off));
  }
  if (lane == 0) {
    s_sum[wave] = s;
    s_i[wave] = im;
  }
  __syncthreads();
  if (tid == 0) {
    double sum = s_sum[0];
    im = s_i[0];
#pragma unroll
    for (int w = 1; w < kConfWaves; ++w) {
      sum += s_sum[w];
      im = min(im, s_i[w]);
    }
    // The sum of exp(x - m). Divided by exp(m), which is one of its terms: times exp(-m), a row
    // whose maximum holds everything would not give exactly 1 (exp(m) exp(-m) is above or below
    // 1 for a third of the maxima), and its probability could exceed 1.
    if (ranged) sum /= exp(md);
    double p;
    if (token) {
      const int64_t t = token[blockIdx.x];
      p = t >= 0 && t < vocab ? exp(static_cast<double>(bf2f(x[t])) - md) / sum : 0.0;
    } else {
      p = 1.0 / sum;
    }
    prob[blockIdx.x] = p;
    // A row with a NaN (no comparison above selects it, but it makes the sum NaN), a +inf or
    // only -inf logits has a softmax of NaNs; torch.max of it returns index 0.
    if (arg) arg[blockIdx.x] = __builtin_isfinite(m) && sum == sum ? im : 0;
  }
}

}  // namespace
}  // namespace fdl

extern "C" int fdl_softmax_confidence(const void* logits, int64_t n_rows, int64_t vocab,
                                      const int64_t* token, double* prob, int64_t* arg,
                                      void* stream) {
  using namespace fdl;
  FDL_REQUIRE(n_rows >= 0 && n_rows < (int64_t(1) << 31), FDL_ERR_SHAPE,
              "fdl_softmax_confidence: n_rows = %lld out of range", (long long)n_rows);
  FDL_REQUIRE(vocab >= 8 && vocab % 8 == 0, FDL_ERR_UNSUPPORTED,
              "fdl_softmax_confidence: vocab = %lld (a multiple of 8 is implemented)",
              (long long)vocab);
  if (n_rows == 0) return ok();
  FDL_REQUIRE_PTR(logits);
  FDL_REQUIRE_PTR(prob);
  FDL_REQUIRE_ALIGNED(logits, 16);
  const bool direct = vocab < kTableVocab;
  auto* kernel = direct ? softmax_conf_direct_kernel : softmax_conf_kernel;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(n_rows)),
                     dim3(direct ? kDirectThreads : kConfThreads), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(logits), vocab,
                     token, prob, arg);
  FDL_HIP_CHECK(hipGetLastError());
  return ok();
}
