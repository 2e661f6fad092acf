// Training-mode batch norm of a row-major [N, K] fp32 matrix: statistics and normalisation (forward), and the
// backward on the COMPRESSED input (the reference's qbatch_norm, ops.py:206-254, calls at::native_batch_norm and, on
// the dequantised input, at::native_batch_norm_backward).
//
// Every kernel is bound by reading [N, K] once.  A column block (at most 1024 columns, blockIdx.y) is walked by
// whole rows: thread t owns unit t % upr (VEC consecutive columns) of rows t / upr, t / upr + rpp, .., so its columns
// never change and its partial sums and column constants stay in registers.  256 columns fill the workgroup with
// four rows, 512 with two, 1024 with one: every width up to 8192 is served, not only the widths of at most 256
// columns that one row of scalar units covers.

#include <cmath>

#include "exact_common.hpp"

namespace exact {

constexpr int kBnMaxK = 8192;

// One column block's geometry, the same in every kernel below.
struct BnBlock {
  int first, units, rpp;  // first column, units per row, rows per pass
};
template <int VEC>
__device__ __forceinline__ BnBlock bn_block(int K) {
  BnBlock b;
  b.first = static_cast<int>(blockIdx.y) * (kBlock * VEC);
  const int cols = K - b.first < kBlock * VEC ? K - b.first : kBlock * VEC;
  b.units = cols / VEC;  // VEC divides K
  b.rpp = kBlock / b.units;
  return b;
}

template <int VEC>
__device__ __forceinline__ void bn_load(const float* p, float (&v)[VEC]) {
  if constexpr (VEC == 4) {
    const f32x4 q = nt_load4(p);
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
  } else {
    v[0] = __builtin_nontemporal_load(p);
  }
}

// Reductions over rows end in a fixed order whatever the launch does: the threads of a workgroup that share a column
// meet in LDS, the workgroup stores two or three numbers per column, partial[workgroup][2 or 3][K], and one small kernel
// takes the workgroups of a column in their order.  (Atomic adds into the result, half a million of them at
// [169343, 256], cost as much and gave other last bits on every run.)

// Count, mean and sum of squared deviations of two disjoint sets of values make those of their union (Chan, Golub and
// LeVeque 1979): no difference of large sums is formed, however the rows are ordered.  The means are kept in 64 bits, so
// that columns far from zero lose nothing either: deviations are differences of means, of which fp32 at 300 would leave
// 3e-5 units.
__device__ __forceinline__ void bn_join(float na, double& mean, float& dev, float nb, double mean_b, float dev_b) {
  const float share = nb / (na + nb);
  const double d = mean_b - mean;
  const float df = static_cast<float>(d);
  const double both_mean = mean + d * static_cast<double>(share);
  const float both_dev = dev + dev_b + df * df * (na * share);
  // selects, no branches: a chain of joins has its divisions ahead of it
  mean = nb == 0.f ? mean : na == 0.f ? mean_b : both_mean;
  dev = nb == 0.f ? dev : na == 0.f ? dev_b : both_dev;
}

// Mean and squared deviations of a workgroup's rows, per column: partial[workgroup][3][K], the mean as the sum of two
// floats.  A thread takes eight rows at a time: their mean and their deviations from it, formed from the differences to
// the first of them, joined to what it has.  Bound by reading x: with the small kernel behind, [50000, 512] takes 33 us
// and [169343, 256] 43 over operands that rotate.
template <int VEC>
__global__ __launch_bounds__(kBlock) void bn_moments_kernel(const float* __restrict__ x, int64_t N, int K, int64_t rows_per_wg,
                                                            float* __restrict__ partial) {
  constexpr int U = 8;  // rows in flight per thread
  __shared__ double part_mean[kBlock * VEC];
  __shared__ float part_dev[kBlock * VEC];
  __shared__ float count[kBlock];
  const BnBlock b = bn_block<VEC>(K);
  const int t = threadIdx.x;
  const int64_t r0 = static_cast<int64_t>(blockIdx.x) * rows_per_wg;
  const int64_t r1 = r0 + rows_per_wg < N ? r0 + rows_per_wg : N;
  if (t < b.rpp * b.units) {
    const int k = b.first + (t % b.units) * VEC;
    double mean[VEC];
    float dev[VEC], n = 0.f;
#pragma unroll
    for (int c = 0; c < VEC; ++c) mean[c] = 0., dev[c] = 0.f;
    int64_t r = r0 + t / b.units;
    for (; r + static_cast<int64_t>(U - 1) * b.rpp < r1; r += static_cast<int64_t>(U) * b.rpp) {
      float v[U][VEC];
#pragma unroll
      for (int i = 0; i < U; ++i) bn_load<VEC>(x + (r + static_cast<int64_t>(i) * b.rpp) * K + k, v[i]);
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        float e[U], m = 0.f, q = 0.f;
#pragma unroll
        for (int i = 1; i < U; ++i) {
          e[i] = v[i][c] - v[0][c];
          m = __fmaf_rn(e[i], 1.f / U, m);  // an exact eighth: the sum cannot overflow
        }
        e[0] = 0.f;
#pragma unroll
        for (int i = 0; i < U; ++i) {
          const float d = e[i] - m;
          q = __fmaf_rn(d, d, q);
        }
        bn_join(n, mean[c], dev[c], static_cast<float>(U), static_cast<double>(v[0][c]) + static_cast<double>(m), q);
      }
      n += static_cast<float>(U);
    }
    for (; r < r1; r += b.rpp) {
      float v[VEC];
      bn_load<VEC>(x + r * K + k, v);
#pragma unroll
      for (int c = 0; c < VEC; ++c) bn_join(n, mean[c], dev[c], 1.f, static_cast<double>(v[c]), 0.f);
      n += 1.f;
    }
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
      part_mean[t * VEC + c] = mean[c];
      part_dev[t * VEC + c] = dev[c];
    }
    if (t % b.units == 0) count[t / b.units] = n;
  }
  __syncthreads();
  const int cols = b.units * VEC;
  int rows = b.rpp;
  while (rows > 1) {  // the upper half of the row slots joins the lower one
    const int keep = (rows + 1) / 2;
    for (int i = t; i < (rows - keep) * cols; i += kBlock) {
      const int slot = i / cols, other = i + keep * cols;
      bn_join(count[slot], part_mean[i], part_dev[i], count[slot + keep], part_mean[other], part_dev[other]);
    }
    __syncthreads();
    if (t < rows - keep) count[t] += count[t + keep];
    __syncthreads();
    rows = keep;
  }
  float* dst = partial + static_cast<int64_t>(blockIdx.x) * 3 * K + b.first;
  for (int i = t; i < cols; i += kBlock) {
    const float hi = static_cast<float>(part_mean[i]);
    dst[i] = hi;
    dst[K + i] = fabsf(hi) <= 0x1.fffffep+127f ? static_cast<float>(part_mean[i] - static_cast<double>(hi)) : 0.f;
    dst[2 * K + i] = part_dev[i];
  }
}

// The kernels that take the workgroups of a column in their order: 8 columns x 32 groups of workgroups, each group
// every 32nd of them, then the groups.  Bound by latency: a group's numbers are loaded at once (eight at a time with a
// branch around each before) and its divisions are formed ahead of the chain that needs them.  Both on one card:
// statistics at [169343, 256] 44.1 -> 42.7 us, [50000, 512] 33.7 -> 32.6, [9000, 256] 19.8 -> 18.3, [8200, 8000] 58.9 ->
// 59.5; the backward at [9000, 256] 23.8 -> 19.0.  (128 groups joined pair by pair end 2 to 4 us sooner: 40.7, 30.6, 16.8
// and 55.7.  But their statistics have other last bits, and behind a quantiser those are other codes.)
constexpr int kBnCols = 8, kBnGroups = kBlock / kBnCols, kBnFinishFlight = 16, kBnSumsFlight = 32;

// -> mean, 1 / sqrt(var + eps), weight * that, and the running statistics with torch's bookkeeping: one launch where
// the framework's element-wise routines took fourteen.
__global__ __launch_bounds__(kBlock) void bn_finish_kernel(const float* __restrict__ partial, int64_t wgs, int64_t rows_per_wg,
                                                           int64_t N, int K, float eps, float factor,
                                                           const float* __restrict__ weight, float* __restrict__ running_mean,
                                                           float* __restrict__ running_var, float* __restrict__ mean,
                                                           float* __restrict__ invstd, float* __restrict__ mult) {
  __shared__ double part_mean[kBlock];
  __shared__ float part_dev[kBlock], count[kBlock];
  const int t = threadIdx.x, c = t % kBnCols, g = t / kBnCols;
  const int k = static_cast<int>(blockIdx.x) * kBnCols + c;
  const float* src = partial + (k < K ? k : K - 1);
  double m = 0.;
  float n = 0.f, dev = 0.f;
  for (int64_t w = g; w < wgs; w += kBnGroups * kBnFinishFlight) {
    float hi[kBnFinishFlight], lo[kBnFinishFlight], pd[kBnFinishFlight];
#pragma unroll
    for (int i = 0; i < kBnFinishFlight; ++i) {
      const float* p = src + (w + i * kBnGroups < wgs ? w + i * kBnGroups : w) * 3 * K;
      hi[i] = p[0];
      lo[i] = p[K];
      pd[i] = p[2 * K];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kBnFinishFlight; ++i) {
      const int64_t at = w + i * kBnGroups;
      const int64_t left = N - at * rows_per_wg;
      const float rows = at >= wgs ? 0.f : static_cast<float>(left < rows_per_wg ? left : rows_per_wg);
      bn_join(n, m, dev, rows, static_cast<double>(hi[i]) + static_cast<double>(lo[i]), pd[i]);
      n += rows;
    }
  }
  count[t] = n;
  part_mean[t] = m;
  part_dev[t] = dev;
  __syncthreads();
  if (g != 0 || k >= K) return;
#pragma unroll
  for (int i = 1; i < kBnGroups; ++i) {
    const int o = i * kBnCols + c;
    bn_join(n, m, dev, count[o], part_mean[o], part_dev[o]);
    n += count[o];
  }
  const float rows = static_cast<float>(N);
  const float var = dev / rows;
  const float inv = 1.f / sqrtf(var + eps);
  const float m32 = static_cast<float>(m);
  mean[k] = m32;
  invstd[k] = inv;
  mult[k] = weight ? weight[k] * inv : inv;
  if (running_mean) {
    const float unbiased = var * (rows / static_cast<float>(N > 1 ? N - 1 : 1));
    running_mean[k] = running_mean[k] * (1.f - factor) + m32 * factor;
    running_var[k] = running_var[k] * (1.f - factor) + unbiased * factor;
  }
}

// The same for plain sums: sums[0 .. K) and sums[K .. 2 K), and the gradient of the weight.
__global__ __launch_bounds__(kBlock) void bn_sums_kernel(const float* __restrict__ partial, int64_t wgs, int K,
                                                         const float* __restrict__ invstd, float* __restrict__ sums,
                                                         float* __restrict__ grad_weight) {
  __shared__ float part[2][kBlock];
  const int t = threadIdx.x, c = t % kBnCols, g = t / kBnCols;
  const int k = static_cast<int>(blockIdx.x) * kBnCols + c;
  const float* src = partial + (k < K ? k : K - 1);
  float s0 = 0.f, s1 = 0.f;
  for (int64_t w = g; w < wgs; w += kBnGroups * kBnSumsFlight) {
    float p0[kBnSumsFlight], p1[kBnSumsFlight];
#pragma unroll
    for (int i = 0; i < kBnSumsFlight; ++i) {
      const int64_t at = w + i * kBnGroups < wgs ? w + i * kBnGroups : w;
      p0[i] = src[at * 2 * K];
      p1[i] = src[at * 2 * K + K];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kBnSumsFlight; ++i) {
      const bool there = w + i * kBnGroups < wgs;
      s0 = there ? s0 + p0[i] : s0;
      s1 = there ? s1 + p1[i] : s1;
    }
  }
  part[0][t] = s0;
  part[1][t] = s1;
  __syncthreads();
  if (g != 0 || k >= K) return;
#pragma unroll
  for (int i = 1; i < kBnGroups; ++i) {
    s0 += part[0][i * kBnCols + c];
    s1 += part[1][i * kBnCols + c];
  }
  sums[k] = s0;
  sums[K + k] = s1;
  if (grad_weight) grad_weight[k] = s1 * invstd[k];
}

// y = (x - mean) * mult + shift
template <int VEC>
__global__ __launch_bounds__(kBlock) void bn_apply_kernel(const float* __restrict__ x, const float* __restrict__ mean,
                                                          const float* __restrict__ mult, const float* __restrict__ bias,
                                                          int64_t N, int K, int64_t rows_per_wg, float* __restrict__ y) {
  constexpr int U = 4;
  const BnBlock b = bn_block<VEC>(K);
  const int t = threadIdx.x;
  if (t >= b.rpp * b.units) return;
  const int k = b.first + (t % b.units) * VEC;
  const int64_t r0 = static_cast<int64_t>(blockIdx.x) * rows_per_wg;
  const int64_t r1 = r0 + rows_per_wg < N ? r0 + rows_per_wg : N;
  float m[VEC], a[VEC], s[VEC];
#pragma unroll
  for (int c = 0; c < VEC; ++c) {
    m[c] = mean[k + c];
    a[c] = mult[k + c];
    s[c] = bias ? bias[k + c] : 0.f;
  }
  for (int64_t r = r0 + t / b.units; r < r1; r += static_cast<int64_t>(U) * b.rpp) {
    float v[U][VEC];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int64_t row = r + static_cast<int64_t>(i) * b.rpp;
      bn_load<VEC>(x + (row < r1 ? row : r) * K + k, v[i]);
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int64_t row = r + static_cast<int64_t>(i) * b.rpp;
      if (row >= r1) break;
#pragma unroll
      for (int c = 0; c < VEC; ++c) v[i][c] = (v[i][c] - m[c]) * a[c] + s[c];
      float* dst = y + row * K + k;
      if constexpr (VEC == 4) nt_store4(dst, v[i][0], v[i][1], v[i][2], v[i][3]);
      else __builtin_nontemporal_store(v[i][0], dst);
    }
  }
}

// ---- backward on the packed input ------------------------------------------------------------------------------
// With g = the incoming gradient (behind a joint ReLU / dropout mask: bit ? dy / (1 - p) : 0) and x the dequantised
// input, two passes
//   reduce   S0[k] = sum_n g,  S1[k] = sum_n g (x - mean)
//   apply    dx = (g - S0 / N - (x - mean) invstd^2 S1 / N) invstd weight
// each read dy, one mask bit and `bits` code bits per element: neither the masked gradient nor the dequantised
// input is ever written to memory.  A thread takes four consecutive rows of its four columns per step: with 1 and 2
// bits their codes are one 32-bit word, and four 16-byte loads of dy are in flight.  At [169343, 256] INT2 with a
// mask the passes and the sums between them take 115 us where mask 58 + dequantise 36 + reduce 68 + apply
// 100 were; at [50000, 512] without one 83 for dequantise 22 + reduce 699 + apply 59.
struct BnBackward {
  const float* dy;
  const uint32_t* mask;  // null: g = dy
  float p1m, inv_p1m;
  const uint8_t* packed;
  const uint16_t* scale;
  const uint16_t* mn;
  const float* mean;
  const float* invstd;
  const float* weight;  // null: 1
  int64_t N;
  int K;
  int64_t rows_per_wg;  // a multiple of 4
  float* partial;       // [workgroups, 2, K]
  float* sums;          // [2, K]
  float* dx;
};

// MASK: 0 none, 1 behind a mask with 1 - p a power of two (the gradient times its reciprocal is the quotient, exactly),
// 2 behind any other.  Nothing here branches by element: with a branch around each quotient and each masked gradient
// the two passes were bound by the vector instructions (with the sums between them, at [169343, 256] INT2: 160 -> 115 us
// with 1 - p = 1 / 2, 160 -> 126 with 0.7, 116 -> 110 without a mask).
template <int BITS, int MASK>
__device__ __forceinline__ void bn_bwd_rows(const BnBackward& a, int64_t row, int k, float (&g)[4][4], float (&x)[4][4]) {
  constexpr int WPT = 8 / BITS;
  constexpr int WORDS = WPT >= 4 ? 1 : 4 / WPT;
  constexpr uint32_t FIELD = (1u << BITS) - 1u;
  f32x4 d[4];
  uint32_t w[WORDS], mk[4];
  uint16_t sc16[4], mn16[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int64_t n = row + r < a.N ? row + r : a.N - 1;  // rows past the end repeat the last one, with g = 0
    d[r] = nt_load4(a.dy + n * a.K + k);
    if constexpr (MASK != 0) {
      const int64_t e = n * a.K + k;  // K % 4 == 0: the four bits lie in one word
      mk[r] = a.mask[e >> 5] >> (e & 31);
    }
    sc16[r] = a.scale[n];
    mn16[r] = a.mn[n];
  }
#pragma unroll
  for (int i = 0; i < WORDS; ++i) {
    const int64_t n = row + i * WPT < a.N ? row + i * WPT : a.N - 1;
    w[i] = *reinterpret_cast<const uint32_t*>(a.packed + (n / WPT) * a.K + k);
  }
  float scale[4], mn[4];
  bool fast = true;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    scale[r] = bf16_to_f32(sc16[r]);
    mn[r] = bf16_to_f32(mn16[r]);
    const float as = fabsf(scale[r]);
    fast = fast && as >= 0x1p-64f && as <= 0x1p64f;  // exact_quotient's range
  }
  auto code = [&](int r, int c) {
    // row is a multiple of 4, so the shift is known but for which half of an INT1 group the rows are
    const int shift = WPT == 8 ? static_cast<int>((row & 7) + r) : (r % WPT) * BITS;
    return static_cast<float>(((w[r / (4 / WORDS)] >> shift) >> (8 * c)) & FIELD);
  };
  if (fast) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float rcp = 1.f / scale[r];
#pragma unroll
      for (int c = 0; c < 4; ++c) x[r][c] = exact_quotient(code(r, c), scale[r], rcp) + mn[r];
    }
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) x[r][c] = code(r, c) / scale[r] + mn[r];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if constexpr (MASK != 0) mk[r] = row + r < a.N ? mk[r] : 0u;
    const bool live = row + r < a.N;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if constexpr (MASK == 0) {
        g[r][c] = live ? d[r][c] : 0.f;
      } else {
        const float dv = ((mk[r] >> c) & 1u) ? d[r][c] : 0.f;
        g[r][c] = MASK == 1 ? dv * a.inv_p1m : dv / a.p1m;
      }
    }
  }
}

template <int BITS, int MASK>
__global__ __launch_bounds__(kBlock) void bn_bwd_reduce_kernel(const BnBackward a) {
  const BnBlock b = bn_block<4>(a.K);
  const int t = threadIdx.x;
  const int64_t r0 = static_cast<int64_t>(blockIdx.x) * a.rows_per_wg;
  const int64_t r1 = r0 + a.rows_per_wg < a.N ? r0 + a.rows_per_wg : a.N;
  float s0[4] = {0.f, 0.f, 0.f, 0.f}, s1[4] = {0.f, 0.f, 0.f, 0.f};
  if (t < b.rpp * b.units) {
    const int k = b.first + (t % b.units) * 4;
    const f32x4 m = *reinterpret_cast<const f32x4_any*>(a.mean + k);
    for (int64_t row = r0 + 4 * (t / b.units); row < r1; row += 4 * b.rpp) {
      float g[4][4], x[4][4];
      bn_bwd_rows<BITS, MASK>(a, row, k, g, x);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          s0[c] += g[r][c];
          s1[c] = __fmaf_rn(g[r][c], x[r][c] - m[c], s1[c]);
        }
    }
  }
  __shared__ float part[2][kBlock * 4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    part[0][t * 4 + c] = s0[c];
    part[1][t * 4 + c] = s1[c];
  }
  __syncthreads();
  const int cols = b.units * 4;
  float* dst = a.partial + static_cast<int64_t>(blockIdx.x) * 2 * a.K + b.first;
  for (int i = t; i < 2 * cols; i += kBlock) {
    const int which = i >= cols, c = which ? i - cols : i;
    float s = 0.f;
    for (int r = 0; r < b.rpp; ++r) s += part[which][r * cols + c];
    dst[which * a.K + c] = s;
  }
}

template <int BITS, int MASK>
__global__ __launch_bounds__(kBlock) void bn_bwd_apply_kernel(const BnBackward a) {
  const BnBlock b = bn_block<4>(a.K);
  const int t = threadIdx.x;
  if (t >= b.rpp * b.units) return;
  const int k = b.first + (t % b.units) * 4;
  const int64_t r0 = static_cast<int64_t>(blockIdx.x) * a.rows_per_wg;
  const int64_t r1 = r0 + a.rows_per_wg < a.N ? r0 + a.rows_per_wg : a.N;
  const float n = static_cast<float>(a.N);
  float mean[4], m_dy[4], f1[4], f2[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const float inv = a.invstd[k + c];
    mean[c] = a.mean[k + c];
    m_dy[c] = a.sums[k + c] / n;
    f1[c] = inv * inv * (a.sums[a.K + k + c] / n);
    f2[c] = a.weight ? a.weight[k + c] * inv : inv;
  }
  for (int64_t row = r0 + 4 * (t / b.units); row < r1; row += 4 * b.rpp) {
    float g[4][4], x[4][4];
    bn_bwd_rows<BITS, MASK>(a, row, k, g, x);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (row + r >= a.N) break;
      float v[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] = (g[r][c] - m_dy[c] - (x[r][c] - mean[c]) * f1[c]) * f2[c];
      nt_store4(a.dx + (row + r) * a.K + k, v[0], v[1], v[2], v[3]);
    }
  }
}

// Rows per workgroup.  A reduction stores two or three numbers per column and workgroup and reads them again, so its
// workgroups are few and long-lived, with at least 16 KiB of the stream each.  Statistics: 512 in fours of columns
// ([50000, 512] 28 against 34 us with 1024), 1024 otherwise ([100003, 301] 37 against 47 with 512, whose wavefronts have
// a quarter of the bytes in flight).  The backward's: 1024 ([169343, 256] with a mask 114 us, 116 with 512, 118 with 2048;
// [50000, 512] 85.6, 85.8 and 89.4).  An element-wise
// pass has no such end: 8192, which evens out the last wave.
constexpr int kBnApplyWgs = 8192, kBnBackwardWgs = 1024;
template <int VEC>
constexpr int bn_moments_wgs() { return VEC == 4 ? 512 : 1024; }
static int64_t bn_rows_per_wg(int64_t N, int K, int vec, int wgs, int multiple) {
  const int block = kBlock * vec, blocks = (K + block - 1) / block;
  const int cols = K < block ? K : block;
  const int rpp = kBlock / (cols / vec);
  int64_t rows = (N * blocks + wgs - 1) / wgs;
  const int64_t least = (4096 + cols - 1) / cols;
  if (rows < least) rows = least;
  const int64_t pass = static_cast<int64_t>(rpp) * multiple;
  return (rows + pass - 1) / pass * pass;
}
static dim3 bn_grid(int64_t N, int K, int vec, int64_t rows) {
  return dim3(static_cast<unsigned>((N + rows - 1) / rows), static_cast<unsigned>((K + kBlock * vec - 1) / (kBlock * vec)));
}
static bool on(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

template <int BITS, int MASK>
static void launch_bn_backward(BnBackward a, float* grad_weight, hipStream_t s) {
  a.rows_per_wg = bn_rows_per_wg(a.N, a.K, 4, kBnBackwardWgs, 4);
  const dim3 grid = bn_grid(a.N, a.K, 4, a.rows_per_wg);
  hipLaunchKernelGGL((bn_bwd_reduce_kernel<BITS, MASK>), grid, dim3(kBlock), 0, s, a);
  hipLaunchKernelGGL(bn_sums_kernel, dim3(static_cast<unsigned>((a.K + kBnCols - 1) / kBnCols)), dim3(kBlock), 0, s, a.partial,
                     static_cast<int64_t>(grid.x), a.K, a.invstd, a.sums, grad_weight);
  if (a.dx) {
    a.rows_per_wg = bn_rows_per_wg(a.N, a.K, 4, kBnApplyWgs, 4);
    hipLaunchKernelGGL((bn_bwd_apply_kernel<BITS, MASK>), bn_grid(a.N, a.K, 4, a.rows_per_wg), dim3(kBlock), 0, s, a);
  }
}

template <int BITS>
static void launch_bn_backward(const BnBackward& a, float* grad_weight, hipStream_t s) {
  int e;
  if (!a.mask) launch_bn_backward<BITS, 0>(a, grad_weight, s);
  else if (std::frexp(a.p1m, &e) == 0.5f) launch_bn_backward<BITS, 1>(a, grad_weight, s);
  else launch_bn_backward<BITS, 2>(a, grad_weight, s);
}

template <int VEC>
static void launch_bn_moments(const float* x, int64_t N, int K, float* partial, int64_t& rows, int64_t& wgs, hipStream_t s) {
  rows = bn_rows_per_wg(N, K, VEC, bn_moments_wgs<VEC>(), 1);
  const dim3 grid = bn_grid(N, K, VEC, rows);
  wgs = grid.x;
  hipLaunchKernelGGL((bn_moments_kernel<VEC>), grid, dim3(kBlock), 0, s, x, N, K, rows, partial);
}

}  // namespace exact

using namespace exact;

extern "C" {

int64_t exact_bn_work_floats(int64_t N, int64_t K) {
  if (N < 1 || K < 1 || K > kBnMaxK || N > (int64_t{1} << 40) / K) return 0;
  const int k = static_cast<int>(K);
  int64_t most = 3 * static_cast<int64_t>(bn_grid(N, k, 1, bn_rows_per_wg(N, k, 1, bn_moments_wgs<1>(), 1)).x);
  if (K % 4 == 0) {
    const int64_t fours = 3 * static_cast<int64_t>(bn_grid(N, k, 4, bn_rows_per_wg(N, k, 4, bn_moments_wgs<4>(), 1)).x);
    const int64_t back = 2 * static_cast<int64_t>(bn_grid(N, k, 4, bn_rows_per_wg(N, k, 4, kBnBackwardWgs, 4)).x);
    most = fours > most ? fours : most;
    most = back > most ? back : most;
  }
  return most * K;
}

int exact_bn_statistics_f32(const float* x, int64_t N, int64_t K, float eps, float factor, const float* weight,
                            float* running_mean, float* running_var, float* work, float* mean, float* invstd, float* mult,
                            void* stream) {
  if (N < 1 || K < 0 || K > kBnMaxK || N > (int64_t{1} << 40) / (K > 0 ? K : 1)) return EXACT_E_SHAPE;
  if (K == 0) return EXACT_OK;
  if (!x || !work || !mean || !invstd || !mult || (running_mean == nullptr) != (running_var == nullptr)) return EXACT_E_NULL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int k = static_cast<int>(K);
  int64_t rows = 0, wgs = 0;
  if (K % 4 == 0 && on(x, 16)) launch_bn_moments<4>(x, N, k, work, rows, wgs, s);
  else launch_bn_moments<1>(x, N, k, work, rows, wgs, s);
  hipLaunchKernelGGL(bn_finish_kernel, dim3(static_cast<unsigned>((k + kBnCols - 1) / kBnCols)), dim3(kBlock), 0, s, work, wgs, rows, N,
                     k, eps, factor, weight, running_mean, running_var, mean, invstd, mult);
  return launch_status();
}

int exact_bn_apply_f32(const float* x, const float* mean, const float* mult, const float* bias, int64_t N, int64_t K,
                       float* y, void* stream) {
  if (N < 0 || K < 0 || K > kBnMaxK || N > (int64_t{1} << 40) / (K > 0 ? K : 1)) return EXACT_E_SHAPE;
  if (N == 0 || K == 0) return EXACT_OK;
  if (!x || !mean || !mult || !y) return EXACT_E_NULL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int k = static_cast<int>(K);
  if (K % 4 == 0 && on(x, 16) && on(y, 16)) {
    const int64_t rows = bn_rows_per_wg(N, k, 4, kBnApplyWgs, 4);
    hipLaunchKernelGGL((bn_apply_kernel<4>), bn_grid(N, k, 4, rows), dim3(kBlock), 0, s, x, mean, mult, bias, N, k, rows, y);
  } else {
    const int64_t rows = bn_rows_per_wg(N, k, 1, kBnApplyWgs, 4);
    hipLaunchKernelGGL((bn_apply_kernel<1>), bn_grid(N, k, 1, rows), dim3(kBlock), 0, s, x, mean, mult, bias, N, k, rows, y);
  }
  return launch_status();
}

int exact_bn_backward_ordered_f32(const float* dy, const uint32_t* mask, float p, const uint8_t* packed, int bits,
                                 const uint16_t* scale_bf16, const uint16_t* min_bf16, const float* mean, const float* invstd,
                                 const float* weight, int64_t N, int64_t K, float* work, float* sums, float* dx,
                                 float* grad_weight, void* stream) {
  if (bits != 1 && bits != 2 && bits != 4 && bits != 8) return EXACT_E_BITS;
  if (!(p >= 0.f && p < 1.f)) return EXACT_E_ARG;
  if (N < 1 || K < 0 || K > kBnMaxK || K % 4 != 0 || N > (int64_t{1} << 40) / (K > 0 ? K : 1)) return EXACT_E_SHAPE;
  if (K == 0) return EXACT_OK;
  if (!dy || !packed || !scale_bf16 || !min_bf16 || !mean || !invstd || !work || !sums) return EXACT_E_NULL;
  if (!on(dy, 16) || !on(dx, 16) || !on(packed, 4) || !on(mask, 4)) return EXACT_E_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  BnBackward a{};
  a.dy = dy;
  a.mask = mask;
  a.p1m = static_cast<float>(1.0 - static_cast<double>(p));  // as the dropout backward divides
  a.inv_p1m = 1.f / a.p1m;
  a.packed = packed;
  a.scale = scale_bf16;
  a.mn = min_bf16;
  a.mean = mean;
  a.invstd = invstd;
  a.weight = weight;
  a.N = N;
  a.K = static_cast<int>(K);
  a.partial = work;
  a.sums = sums;
  a.dx = dx;
  switch (bits) {
    case 1: launch_bn_backward<1>(a, grad_weight, s); break;
    case 2: launch_bn_backward<2>(a, grad_weight, s); break;
    case 4: launch_bn_backward<4>(a, grad_weight, s); break;
    default: launch_bn_backward<8>(a, grad_weight, s); break;
  }
  return launch_status();
}

}  // extern "C"
