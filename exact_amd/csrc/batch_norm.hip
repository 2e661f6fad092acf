// Training-mode batch norm of a row-major [N, K] fp32 matrix: statistics and normalisation (forward), and the
// backward on the COMPRESSED input (the reference's qbatch_norm, ops.py:206-254, calls at::native_batch_norm and, on
// the dequantised input, at::native_batch_norm_backward).
//
// Every kernel is bound by reading [N, K] once.  A column block (at most 1024 columns, blockIdx.y) is walked by
// whole rows: thread t owns unit t % upr (VEC consecutive columns) of rows t / upr, t / upr + rpp, .., so its columns
// never change and its partial sums and column constants stay in registers.  256 columns fill the workgroup with
// four rows, 512 with two, 1024 with one: every width up to 8192 is served, not only the widths of at most 256
// columns that one row of scalar units covers.

#include "exact_common.hpp"

namespace exact {

constexpr int kBnMaxK = 8192;
constexpr int kBnSample = 256;  // rows whose mean is the centre of the moments

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

// The centre of the moments: the mean of up to 256 rows spread evenly over the matrix (also for sorted or clustered
// rows within a fraction of a standard deviation of the column mean, so that the difference of the moments loses no
// digits).  16 columns x 16 row groups per workgroup, 16 loads in flight per thread: the kernel is a few load
// latencies long whatever N is.  It also clears the two sums, which the next kernel meets with atomics.
__global__ __launch_bounds__(kBlock) void bn_center_kernel(const float* __restrict__ x, int64_t N, int K,
                                                           float* __restrict__ center, float* __restrict__ sums) {
  __shared__ float part[kBlock];
  const int c = threadIdx.x & 15, g = threadIdx.x >> 4;
  const int k = static_cast<int>(blockIdx.x) * 16 + c;
  const int64_t step = N / kBnSample > 0 ? N / kBnSample : 1;
  const int count = static_cast<int>(N < kBnSample ? N : kBnSample);
  float s = 0.f;
  if (k < K) {
    float v[kBnSample / 16];
#pragma unroll
    for (int i = 0; i < kBnSample / 16; ++i) {
      const int row = g + 16 * i;
      v[i] = x[(row < count ? row : 0) * step * K + k];
    }
#pragma unroll
    for (int i = 0; i < kBnSample / 16; ++i) s += g + 16 * i < count ? v[i] : 0.f;
  }
  part[threadIdx.x] = s;
  __syncthreads();
  if (g == 0 && k < K) {
    for (int i = 1; i < 16; ++i) s += part[16 * i + c];
    center[k] = s / static_cast<float>(count);
    sums[k] = 0.f;
    sums[K + k] = 0.f;
  }
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

// The partial sums of the threads that share a column meet in LDS, then one atomic add per column and sum.
template <int VEC>
__device__ __forceinline__ void bn_meet(const BnBlock& b, int K, const float (&s0)[VEC], const float (&s1)[VEC], float* sums) {
  __shared__ float part[2][kBlock * VEC];
  const int t = threadIdx.x;
#pragma unroll
  for (int c = 0; c < VEC; ++c) {
    part[0][t * VEC + c] = s0[c];
    part[1][t * VEC + c] = s1[c];
  }
  __syncthreads();
  const int cols = b.units * VEC;
  for (int i = t; i < 2 * cols; i += kBlock) {
    const int which = i >= cols, c = which ? i - cols : i;
    float s = 0.f;
    for (int r = 0; r < b.rpp; ++r) s += part[which][r * cols + c];
    if (s != 0.f) unsafeAtomicAdd(sums + static_cast<int64_t>(which) * K + b.first + c, s);
  }
}

// sums[k] = sum_n (x - center), sums[K + k] = sum_n (x - center)^2.  [50000, 512]: 36 us (2.8 TB/s); the framework's
// statistics took 504 us there, with two workgroups; [169343, 256]: 42 us.
template <int VEC>
__global__ __launch_bounds__(kBlock) void bn_moments_kernel(const float* __restrict__ x, const float* __restrict__ center,
                                                            int64_t N, int K, int64_t rows_per_wg, float* __restrict__ sums) {
  constexpr int U = 8;  // rows in flight per thread
  const BnBlock b = bn_block<VEC>(K);
  const int t = threadIdx.x;
  const int64_t r0 = static_cast<int64_t>(blockIdx.x) * rows_per_wg;
  const int64_t r1 = r0 + rows_per_wg < N ? r0 + rows_per_wg : N;
  float acc[VEC], acc2[VEC], ctr[VEC];
#pragma unroll
  for (int c = 0; c < VEC; ++c) acc[c] = acc2[c] = ctr[c] = 0.f;
  if (t < b.rpp * b.units) {
    const int k = b.first + (t % b.units) * VEC;
#pragma unroll
    for (int c = 0; c < VEC; ++c) ctr[c] = center[k + c];
    auto add = [&](const float (&v)[VEC]) {
#pragma unroll
      for (int c = 0; c < VEC; ++c) {
        const float d = v[c] - ctr[c];
        acc[c] += d;
        acc2[c] = __fmaf_rn(d, d, acc2[c]);
      }
    };
    int64_t r = r0 + t / b.units;
    for (; r + static_cast<int64_t>(U - 1) * b.rpp < r1; r += static_cast<int64_t>(U) * b.rpp) {
      float v[U][VEC];
#pragma unroll
      for (int i = 0; i < U; ++i) bn_load<VEC>(x + (r + static_cast<int64_t>(i) * b.rpp) * K + k, v[i]);
#pragma unroll
      for (int i = 0; i < U; ++i) add(v[i]);
    }
    for (; r < r1; r += b.rpp) {
      float v[VEC];
      bn_load<VEC>(x + r * K + k, v);
      add(v);
    }
  }
  bn_meet<VEC>(b, K, acc, acc2, sums);
}

// Moments -> mean, 1 / sqrt(var + eps), weight * that, and the running statistics with torch's bookkeeping: one
// launch where the framework's element-wise routines took fourteen.
__global__ __launch_bounds__(kBlock) void bn_finish_kernel(const float* __restrict__ center, const float* __restrict__ sums,
                                                           int64_t N, int K, float eps, float factor,
                                                           const float* __restrict__ weight, float* __restrict__ running_mean,
                                                           float* __restrict__ running_var, float* __restrict__ mean,
                                                           float* __restrict__ invstd, float* __restrict__ mult) {
  const int k = static_cast<int>(blockIdx.x) * kBlock + threadIdx.x;
  if (k >= K) return;
  const float n = static_cast<float>(N);
  const float shift = sums[k] / n;
  const float raw = sums[K + k] / n - shift * shift;
  const float var = raw < 0.f ? 0.f : raw;  // a NaN stays one
  const float m = center[k] + shift;
  const float inv = 1.f / sqrtf(var + eps);
  mean[k] = m;
  invstd[k] = inv;
  mult[k] = weight ? weight[k] * inv : inv;
  if (running_mean) {
    const float unbiased = var * (n / static_cast<float>(N > 1 ? N - 1 : 1));
    running_mean[k] = running_mean[k] * (1.f - factor) + m * factor;
    running_var[k] = running_var[k] * (1.f - factor) + unbiased * factor;
  }
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
// mask the two passes take 76 + 90 us where mask 58 + dequantise 36 + reduce 68 + apply 100 were; at [50000, 512]
// without one 44 + 56 for dequantise 22 + reduce 699 + apply 59.
struct BnBackward {
  const float* dy;
  const uint32_t* mask;  // null: g = dy
  float p1m;
  const uint8_t* packed;
  const uint16_t* scale;
  const uint16_t* mn;
  const float* mean;
  const float* invstd;
  const float* weight;  // null: 1
  int64_t N;
  int K;
  int64_t rows_per_wg;  // a multiple of 4
  float* sums;          // [2, K]
  float* dx;
  float* grad_weight;  // null, or S1 * invstd
};

template <int BITS>
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
    mk[r] = 0xFu;
    if (a.mask) {
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
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float scale = bf16_to_f32(sc16[r]), mn = bf16_to_f32(mn16[r]);
    const float as = fabsf(scale);
    const bool fast = as >= 0x1p-64f && as <= 0x1p64f;  // exact_quotient's range
    const float rcp = 1.f / scale;
    // row is a multiple of 4, so the shift is known but for which half of an INT1 group the rows are
    const int shift = WPT == 8 ? static_cast<int>((row & 7) + r) : (r % WPT) * BITS;
    const uint32_t word = w[r / (4 / WORDS)] >> shift;
    const bool live = row + r < a.N;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float q = static_cast<float>((word >> (8 * c)) & FIELD);
      x[r][c] = (fast ? exact_quotient(q, scale, rcp) : q / scale) + mn;
      const float dv = d[r][c];
      const float gv = a.mask ? (((mk[r] >> c) & 1u) ? dv / a.p1m : 0.f) : dv;
      g[r][c] = live ? gv : 0.f;
    }
  }
}

template <int BITS>
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
      bn_bwd_rows<BITS>(a, row, k, g, x);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          s0[c] += g[r][c];
          s1[c] = __fmaf_rn(g[r][c], x[r][c] - m[c], s1[c]);
        }
    }
  }
  bn_meet<4>(b, a.K, s0, s1, a.sums);
}

template <int BITS>
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
    if (a.grad_weight && blockIdx.x == 0 && t < b.units) a.grad_weight[k + c] = a.sums[a.K + k + c] * inv;
  }
  if (!a.dx) return;
  for (int64_t row = r0 + 4 * (t / b.units); row < r1; row += 4 * b.rpp) {
    float g[4][4], x[4][4];
    bn_bwd_rows<BITS>(a, row, k, g, x);
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

__global__ __launch_bounds__(kBlock) void bn_zero_kernel(float* __restrict__ out, int n) {
  const int i = static_cast<int>(blockIdx.x) * kBlock + threadIdx.x;
  if (i < n) out[i] = 0.f;
}

// Rows per workgroup.  A reduction ends with two atomic adds per column into the same words, which are served one
// after the other: about 1024 long-lived workgroups, at least 16 KiB of the stream each.  An element-wise pass has no
// such end: up to eight times as many, which evens out the last wave.
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

template <int BITS>
static void launch_bn_backward(BnBackward a, hipStream_t s) {
  a.rows_per_wg = bn_rows_per_wg(a.N, a.K, 4, 1024, 4);
  hipLaunchKernelGGL((bn_bwd_reduce_kernel<BITS>), bn_grid(a.N, a.K, 4, a.rows_per_wg), dim3(kBlock), 0, s, a);
  a.rows_per_wg = bn_rows_per_wg(a.N, a.K, 4, 8192, 4);
  if (a.dx || a.grad_weight) {
    const dim3 grid = bn_grid(a.N, a.K, 4, a.rows_per_wg);
    hipLaunchKernelGGL((bn_bwd_apply_kernel<BITS>), a.dx ? grid : dim3(1, grid.y), dim3(kBlock), 0, s, a);
  }
}

}  // namespace exact

using namespace exact;

extern "C" {

int exact_bn_stats_f32(const float* x, int64_t N, int64_t K, float eps, float factor, const float* weight,
                       float* running_mean, float* running_var, float* work, float* mean, float* invstd, float* mult,
                       void* stream) {
  if (N < 1 || K < 0 || K > kBnMaxK || N > (int64_t{1} << 40) / (K > 0 ? K : 1)) return EXACT_E_SHAPE;
  if (K == 0) return EXACT_OK;
  if (!x || !work || !mean || !invstd || !mult || (running_mean == nullptr) != (running_var == nullptr)) return EXACT_E_NULL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int k = static_cast<int>(K);
  float* center = work + 2 * K;
  hipLaunchKernelGGL(bn_center_kernel, dim3(static_cast<unsigned>((K + 15) / 16)), dim3(kBlock), 0, s, x, N, k, center, work);
  if (K % 4 == 0 && on(x, 16)) {
    const int64_t rows = bn_rows_per_wg(N, k, 4, 1024, 1);
    hipLaunchKernelGGL((bn_moments_kernel<4>), bn_grid(N, k, 4, rows), dim3(kBlock), 0, s, x, center, N, k, rows, work);
  } else {
    const int64_t rows = bn_rows_per_wg(N, k, 1, 1024, 1);
    hipLaunchKernelGGL((bn_moments_kernel<1>), bn_grid(N, k, 1, rows), dim3(kBlock), 0, s, x, center, N, k, rows, work);
  }
  hipLaunchKernelGGL(bn_finish_kernel, dim3(static_cast<unsigned>((K + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, center, work, N, k,
                     eps, factor, weight, running_mean, running_var, mean, invstd, mult);
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
    const int64_t rows = bn_rows_per_wg(N, k, 4, 8192, 4);
    hipLaunchKernelGGL((bn_apply_kernel<4>), bn_grid(N, k, 4, rows), dim3(kBlock), 0, s, x, mean, mult, bias, N, k, rows, y);
  } else {
    const int64_t rows = bn_rows_per_wg(N, k, 1, 8192, 4);
    hipLaunchKernelGGL((bn_apply_kernel<1>), bn_grid(N, k, 1, rows), dim3(kBlock), 0, s, x, mean, mult, bias, N, k, rows, y);
  }
  return launch_status();
}

int exact_bn_backward_packed_f32(const float* dy, const uint32_t* mask, float p, const uint8_t* packed, int bits,
                                 const uint16_t* scale_bf16, const uint16_t* min_bf16, const float* mean, const float* invstd,
                                 const float* weight, int64_t N, int64_t K, float* sums, float* dx, float* grad_weight,
                                 void* stream) {
  if (bits != 1 && bits != 2 && bits != 4 && bits != 8) return EXACT_E_BITS;
  if (!(p >= 0.f && p < 1.f)) return EXACT_E_ARG;
  if (N < 1 || K < 0 || K > kBnMaxK || K % 4 != 0 || N > (int64_t{1} << 40) / (K > 0 ? K : 1)) return EXACT_E_SHAPE;
  if (K == 0) return EXACT_OK;
  if (!dy || !packed || !scale_bf16 || !min_bf16 || !mean || !invstd || !sums) return EXACT_E_NULL;
  if (!on(dy, 16) || !on(dx, 16) || !on(packed, 4) || !on(mask, 4)) return EXACT_E_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  BnBackward a{};
  a.dy = dy;
  a.mask = mask;
  a.p1m = static_cast<float>(1.0 - static_cast<double>(p));  // as the dropout backward divides
  a.packed = packed;
  a.scale = scale_bf16;
  a.mn = min_bf16;
  a.mean = mean;
  a.invstd = invstd;
  a.weight = weight;
  a.N = N;
  a.K = static_cast<int>(K);
  a.sums = sums;
  a.dx = dx;
  a.grad_weight = grad_weight;
  hipLaunchKernelGGL(bn_zero_kernel, dim3(static_cast<unsigned>((2 * K + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, sums,
                     static_cast<int>(2 * K));
  switch (bits) {
    case 1: launch_bn_backward<1>(a, s); break;
    case 2: launch_bn_backward<2>(a, s); break;
    case 4: launch_bn_backward<4>(a, s); break;
    default: launch_bn_backward<8>(a, s); break;
  }
  return launch_status();
}

}  // extern "C"
