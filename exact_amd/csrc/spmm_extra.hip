// The remaining sparse kernels of the reference's spmm extension:
//   * max / min aggregation with the arg-entry output
//     (spmm_kernel<.., MAX|MIN, ..> spmm_cuda.cu:27-104, Reducer reducer.cuh:43-85);
//   * the gradient with respect to the edge values, a sampled dense-dense
//     product (spmm_value_bw_kernel spmm_cuda.cu:172-209).
// Neither is on the sum / mean path of the GCN / GraphSAGE benchmarks; they are
// plain one-wavefront-per-row (resp. per-entry) kernels, 64 lanes spanning
// 64 * VEC feature columns.

#include "exact_common.hpp"

namespace exact {

template <int VEC>
__device__ __forceinline__ void load_cols(const float* p, float (&v)[VEC]) {
  if constexpr (VEC == 4) { const float4 q = *reinterpret_cast<const float4*>(p); v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w; }
  else if constexpr (VEC == 2) { const float2 q = *reinterpret_cast<const float2*>(p); v[0] = q.x; v[1] = q.y; }
  else { v[0] = *p; }
}

// out[r, k] = max / min over the entries e of row r of val[e] * X[col[e], k];
// arg_out[r, k] = the entry index that attained it (first one in CSR order),
// nnz for rows without entries, whose output is 0 (reducer.cuh:77-84).
template <typename I, int VEC, bool HAS_VAL, bool IS_MAX>
__global__ __launch_bounds__(kBlock) void spmm_minmax_kernel(const I* __restrict__ rowptr,
                                                             const I* __restrict__ col,
                                                             const float* __restrict__ val,
                                                             const float* __restrict__ X, int64_t M, int64_t K,
                                                             int64_t nnz, float* __restrict__ out,
                                                             I* __restrict__ arg_out) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t r = static_cast<int64_t>(blockIdx.x) * (kBlock / kWave) + (threadIdx.x >> 6);
  if (r >= M) return;
  const int64_t kcol = (static_cast<int64_t>(blockIdx.y) * kWave + lane) * VEC;
  if (kcol >= K) return;
  const int64_t rs = static_cast<int64_t>(rowptr[r]), re = static_cast<int64_t>(rowptr[r + 1]);
  float best[VEC];
  int64_t arg[VEC];
#pragma unroll
  for (int c = 0; c < VEC; ++c) {
    best[c] = IS_MAX ? -3.402823466e+38f : 3.402823466e+38f;  // numeric_limits lowest() / max(), reducer.cuh:47-50
    arg[c] = nnz;
  }
  for (int64_t e = rs; e < re; ++e) {
    const int64_t cidx = static_cast<int64_t>(col[e]);
    float xv[VEC];
    load_cols<VEC>(X + cidx * K + kcol, xv);
    const float w = HAS_VAL ? val[e] : 1.f;
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
      const float t = HAS_VAL ? w * xv[c] : xv[c];
      if (IS_MAX ? (t > best[c]) : (t < best[c])) {  // strict: the first extreme entry wins
        best[c] = t;
        arg[c] = e;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < VEC; ++c) {
    out[r * K + kcol + c] = (re > rs) ? best[c] : 0.f;
    arg_out[r * K + kcol + c] = static_cast<I>((re > rs) ? arg[c] : nnz);
  }
}

// Deterministic sum / mean: one wavefront per row (and per slab of 64 * VEC
// columns), the row's entries taken one after the other in CSR order with one
// multiply and one add each -- the summation order of the reference kernel
// (spmm_cuda.cu:85-90) and of the CPU oracle, so results are reproducible bit
// for bit.  No atomics, every output element is stored exactly once.  Hub rows
// serialise, which is why the default path is the chunked kernel in spmm.hip.
template <typename I, int VEC, bool HAS_VAL, bool MEAN>
__global__ __launch_bounds__(kBlock) void spmm_rowwise_kernel(const I* __restrict__ rowptr,
                                                              const I* __restrict__ col,
                                                              const float* __restrict__ val,
                                                              const float* __restrict__ X, int64_t M, int64_t K,
                                                              float* __restrict__ out) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t r = static_cast<int64_t>(blockIdx.x) * (kBlock / kWave) + (threadIdx.x >> 6);
  if (r >= M) return;
  const int64_t kcol = (static_cast<int64_t>(blockIdx.y) * kWave + lane) * VEC;
  if (kcol >= K) return;
  const int64_t rs = static_cast<int64_t>(rowptr[r]), re = static_cast<int64_t>(rowptr[r + 1]);
  float acc[VEC];
#pragma unroll
  for (int c = 0; c < VEC; ++c) acc[c] = 0.f;
  for (int64_t e = rs; e < re; ++e) {
    float xv[VEC];
    load_cols<VEC>(X + static_cast<int64_t>(col[e]) * K + kcol, xv);
    const float w = HAS_VAL ? val[e] : 1.f;
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
      const float term = HAS_VAL ? w * xv[c] : xv[c];
      acc[c] = acc[c] + term;
    }
  }
  if (MEAN) {
    const float cnt = static_cast<float>(re > rs ? re - rs : 1);  // reducer.cuh:75-76
#pragma unroll
    for (int c = 0; c < VEC; ++c) acc[c] = acc[c] / cnt;
  }
#pragma unroll
  for (int c = 0; c < VEC; ++c) out[r * K + kcol + c] = acc[c];
}

// Gradient with respect to the edge values: out[e] = mat[col[e]] . grad[row[e]]  (/ row length for the mean)
// (spmm_value_bw_cuda, spmm_cuda.cu:172-252).
//
// A group of L lanes (the fewest, 8 to 64, whose four columns each cover K) takes eight consecutive entries: their
// eight rows of `mat` are gathered in one go, and the row of `grad`, which consecutive entries of a CSR matrix mostly
// share, is read once for all eight where they do.  The eight dot products are folded over the group's lanes in
// halves -- 7 exchanges for the first three steps of all eight instead of 24 -- and leave as one 32-byte piece.
// Bound by the gathers of `mat`: 1.8 M entries on 60,000 rows, 128
// columns, 131 us (7.0 TB/s of `mat`); one wavefront per entry, which this replaces, took 338.
constexpr int kSddmmEntries = 8;

template <typename I, int L, bool MEAN>
__global__ __launch_bounds__(kBlock) void sddmm_kernel(const I* __restrict__ row, const I* __restrict__ rowptr,
                                                       const I* __restrict__ col, const float* __restrict__ mat,
                                                       const float* __restrict__ grad, int64_t E, int64_t K,
                                                       float* __restrict__ out) {
  constexpr int U = kSddmmEntries;
  const int gl = threadIdx.x & (L - 1);
  const int64_t e0 = (static_cast<int64_t>(blockIdx.x) * (kBlock / L) + threadIdx.x / L) * U;
  const int64_t mine = e0 + (gl & (U - 1));                 // the entry whose indices this lane fetches
  const int64_t safe = mine < E ? mine : E - 1;             // entries past the end repeat the last one, unstored
  const int64_t my_row = static_cast<int64_t>(row[safe]), my_col = static_cast<int64_t>(col[safe]);
  auto from = [&](int64_t v, int lane) -> int64_t {
    const int src = (static_cast<int>(threadIdx.x) & (kWave - L)) | lane;
    const uint32_t lo = __shfl(static_cast<uint32_t>(v), src), hi = sizeof(I) == 8 ? __shfl(static_cast<uint32_t>(v >> 32), src) : 0u;
    return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
  };
  const int64_t first_row = from(my_row, 0);
  const bool one_row = __ballot(my_row != first_row) == 0;  // in every group of the wavefront
  float acc[U];
#pragma unroll
  for (int u = 0; u < U; ++u) acc[u] = 0.f;
  // A lane's piece past the end of the row is read where the row's last four columns are and left out of the sums: a
  // load behind a branch would make the compiler wait for every load in flight.
  auto load4 = [&](const float* p) -> f32x4 {
    if (K >= 4) return *reinterpret_cast<const f32x4_any*>(p);  // wave-uniform
    f32x4 q = {0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < K; ++i) q[i] = p[i];
    return q;
  };
  for (int64_t k0 = 0; k0 < K; k0 += 4 * L) {
    const int64_t k = k0 + 4 * gl;
    const int64_t at = k + 4 <= K ? k : K >= 4 ? K - 4 : 0;
    const int64_t skip = k - at;  // of the four elements read, those that belong to the lane before
    f32x4 m[U], g[U];
#pragma unroll
    for (int u = 0; u < U; ++u) m[u] = load4(mat + from(my_col, u) * K + at);
    if (one_row) {
      g[0] = load4(grad + first_row * K + at);
#pragma unroll
      for (int u = 1; u < U; ++u) g[u] = g[0];
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) g[u] = load4(grad + from(my_row, u) * K + at);
    }
    if (__ballot(skip != 0) == 0) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[u] = __fmaf_rn(m[u][i], g[u][i], acc[u]);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[u] = i >= skip ? __fmaf_rn(m[u][i], g[u][i], acc[u]) : acc[u];
    }
  }
  // lane bits 0, 1, 2 pick the half of the remaining entries a lane goes on with
#pragma unroll
  for (int step = 0; step < 3; ++step) {
    const bool upper = ((gl >> step) & 1) != 0;
#pragma unroll
    for (int i = 0; i < (U >> (step + 1)); ++i) {
      const float keep = upper ? acc[i + (U >> (step + 1))] : acc[i], give = upper ? acc[i] : acc[i + (U >> (step + 1))];
      acc[i] = keep + __shfl_xor(give, 1 << step);
    }
  }
  float sum = acc[0];
#pragma unroll
  for (int m = 8; m < L; m <<= 1) sum += __shfl_xor(sum, m);
  const int u = ((gl & 1) << 2) | (gl & 2) | ((gl >> 2) & 1);  // the entry whose sum this lane holds
  const int64_t r = from(my_row, u);
  if (gl < U && e0 + u < E) {
    if (MEAN) {
      const int64_t deg = static_cast<int64_t>(rowptr[r + 1]) - static_cast<int64_t>(rowptr[r]);
      sum /= static_cast<float>(deg > 0 ? deg : 1);
    }
    out[e0 + u] = sum;
  }
}

static bool aligned_to(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

template <typename I, int VEC>
static void minmax_dispatch(const I* rowptr, const I* col, const float* val, const float* X, int64_t M, int64_t K,
                            int64_t nnz, bool is_max, float* out, I* arg_out, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>((M + 3) / 4), static_cast<unsigned>((K + kWave * VEC - 1) / (kWave * VEC)));
  const dim3 block(kBlock);
  if (val) {
    if (is_max) hipLaunchKernelGGL((spmm_minmax_kernel<I, VEC, true, true>), grid, block, 0, s, rowptr, col, val, X, M, K, nnz, out, arg_out);
    else hipLaunchKernelGGL((spmm_minmax_kernel<I, VEC, true, false>), grid, block, 0, s, rowptr, col, val, X, M, K, nnz, out, arg_out);
  } else {
    if (is_max) hipLaunchKernelGGL((spmm_minmax_kernel<I, VEC, false, true>), grid, block, 0, s, rowptr, col, val, X, M, K, nnz, out, arg_out);
    else hipLaunchKernelGGL((spmm_minmax_kernel<I, VEC, false, false>), grid, block, 0, s, rowptr, col, val, X, M, K, nnz, out, arg_out);
  }
}

template <typename I, int L>
static void sddmm_dispatch(const I* row, const I* rowptr, const I* col, const float* mat, const float* grad, int64_t E,
                           int64_t K, bool mean, float* out, hipStream_t s) {
  constexpr int64_t per_wg = static_cast<int64_t>(kBlock / L) * kSddmmEntries;
  const dim3 grid(static_cast<unsigned>((E + per_wg - 1) / per_wg));
  if (mean) hipLaunchKernelGGL((sddmm_kernel<I, L, true>), grid, dim3(kBlock), 0, s, row, rowptr, col, mat, grad, E, K, out);
  else hipLaunchKernelGGL((sddmm_kernel<I, L, false>), grid, dim3(kBlock), 0, s, row, rowptr, col, mat, grad, E, K, out);
}

template <typename I, int VEC>
static void rowwise_dispatch(const I* rowptr, const I* col, const float* val, const float* X, int64_t M, int64_t K,
                             bool mean, float* out, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>((M + 3) / 4), static_cast<unsigned>((K + kWave * VEC - 1) / (kWave * VEC)));
  const dim3 block(kBlock);
  if (val) {
    if (mean) hipLaunchKernelGGL((spmm_rowwise_kernel<I, VEC, true, true>), grid, block, 0, s, rowptr, col, val, X, M, K, out);
    else hipLaunchKernelGGL((spmm_rowwise_kernel<I, VEC, true, false>), grid, block, 0, s, rowptr, col, val, X, M, K, out);
  } else {
    if (mean) hipLaunchKernelGGL((spmm_rowwise_kernel<I, VEC, false, true>), grid, block, 0, s, rowptr, col, val, X, M, K, out);
    else hipLaunchKernelGGL((spmm_rowwise_kernel<I, VEC, false, false>), grid, block, 0, s, rowptr, col, val, X, M, K, out);
  }
}

// out[i] = values[index[i]] for the transposed edge values: bound by the lines that the random 4-byte reads fetch (12 TB/s
// of 128-byte lines), so all a thread can do is to keep four in flight, with their indices read in whole runs.  1.8 M
// entries, 8-byte indices: 19.6 us, the framework's index_select 24 and its pass over fp16 values another 5.  An index
// outside the values gives NaN.
template <typename I, typename V>
__global__ __launch_bounds__(kBlock) void gather_values_kernel(const V* __restrict__ values, const I* __restrict__ index, int64_t n,
                                                               int64_t n_values, float* __restrict__ out) {
  constexpr int kEach = 4;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * (2 * kEach * kBlock) + threadIdx.x;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    int64_t at[kEach];
    float v[kEach];
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const int64_t e = first + (h * kEach + i) * kBlock;
      at[i] = static_cast<int64_t>(index[e < n ? e : n - 1]);
    }
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const bool inside = at[i] >= 0 && at[i] < n_values;
      const float got = static_cast<float>(values[inside ? at[i] : 0]);
      v[i] = inside ? got : __builtin_nanf("");
    }
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const int64_t e = first + (h * kEach + i) * kBlock;
      if (e < n) out[e] = v[i];
    }
  }
}

template <typename I>
static void launch_gather_values(const void* values, int half, const void* index, int64_t n, int64_t n_values, float* out, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>((n + 8 * kBlock - 1) / (8 * kBlock)));
  const I* at = static_cast<const I*>(index);
  if (half) hipLaunchKernelGGL((gather_values_kernel<I, half_t>), grid, dim3(kBlock), 0, s, static_cast<const half_t*>(values), at, n, n_values, out);
  else hipLaunchKernelGGL((gather_values_kernel<I, float>), grid, dim3(kBlock), 0, s, static_cast<const float*>(values), at, n, n_values, out);
}

}  // namespace exact

using namespace exact;

extern "C" {

int exact_spmm_csr_minmax_f32(const void* rowptr, const void* col, const float* val, int idx_bytes, const float* X,
                              int64_t M, int64_t n_cols, int64_t K, int64_t nnz, int is_max, float* out,
                              void* arg_out, void* stream) {
  if (idx_bytes != 4 && idx_bytes != 8) return EXACT_E_ARG;
  if (M < 0 || K < 0 || nnz < 0 || n_cols < 0 || n_cols > 0x7FFFFFFFll) return EXACT_E_SHAPE;
  if (idx_bytes == 4 && nnz > 0x7FFFFFFFll) return EXACT_E_SHAPE;
  if (M > (int64_t{1} << 32) || K > (int64_t{1} << 24)) return EXACT_E_SHAPE;  // launch-grid limits
  if (M == 0 || K == 0) return EXACT_OK;
  if (!rowptr || !out || !arg_out || (nnz > 0 && (!col || !X))) return EXACT_E_NULL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int vec = (K % 4 == 0 && aligned_to(X, 16)) ? 4 : (K % 2 == 0 && aligned_to(X, 8)) ? 2 : 1;
#define EXACT_MM_GO(I, V) \
  minmax_dispatch<I, V>(static_cast<const I*>(rowptr), static_cast<const I*>(col), val, X, M, K, nnz, is_max != 0, out, static_cast<I*>(arg_out), s)
  if (idx_bytes == 4) {
    if (vec == 4) EXACT_MM_GO(int32_t, 4); else if (vec == 2) EXACT_MM_GO(int32_t, 2); else EXACT_MM_GO(int32_t, 1);
  } else {
    if (vec == 4) EXACT_MM_GO(int64_t, 4); else if (vec == 2) EXACT_MM_GO(int64_t, 2); else EXACT_MM_GO(int64_t, 1);
  }
#undef EXACT_MM_GO
  return launch_status();
}

int exact_gather_values_f32(const void* values, int half, const void* index, int idx_bytes, int64_t n, int64_t n_values, float* out,
                            void* stream) {
  if ((idx_bytes != 4 && idx_bytes != 8) || (half != 0 && half != 1)) return EXACT_E_ARG;
  if (n < 0 || n_values < 0 || (n > 0 && n_values == 0) || n > (int64_t{1} << 40)) return EXACT_E_SHAPE;
  if (n == 0) return EXACT_OK;
  if (!values || !index || !out) return EXACT_E_NULL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (idx_bytes == 4) launch_gather_values<int32_t>(values, half, index, n, n_values, out, s);
  else launch_gather_values<int64_t>(values, half, index, n, n_values, out, s);
  return launch_status();
}

int exact_sddmm_f32(const void* row, const void* rowptr, const void* col, int idx_bytes, const float* mat,
                    const float* grad, int64_t nnz, int64_t K, int reduce, float* out, void* stream) {
  if (idx_bytes != 4 && idx_bytes != 8) return EXACT_E_ARG;
  if (reduce != EXACT_REDUCE_SUM && reduce != EXACT_REDUCE_MEAN) return EXACT_E_ARG;
  if (nnz < 0 || K < 0 || nnz > (int64_t{1} << 32)) return EXACT_E_SHAPE;  // launch-grid limit
  if (nnz == 0) return EXACT_OK;
  if (!row || !rowptr || !col || !mat || !grad || !out) return EXACT_E_NULL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool mean = reduce == EXACT_REDUCE_MEAN;
#define EXACT_SD_GO(L)                                                                                                 \
  do {                                                                                                                 \
    if (idx_bytes == 4) sddmm_dispatch<int32_t, L>(static_cast<const int32_t*>(row), static_cast<const int32_t*>(rowptr), static_cast<const int32_t*>(col), mat, grad, nnz, K, mean, out, s); \
    else sddmm_dispatch<int64_t, L>(static_cast<const int64_t*>(row), static_cast<const int64_t*>(rowptr), static_cast<const int64_t*>(col), mat, grad, nnz, K, mean, out, s); \
  } while (0)
  if (K <= 32) EXACT_SD_GO(8);
  else if (K <= 64) EXACT_SD_GO(16);
  else if (K <= 128) EXACT_SD_GO(32);
  else EXACT_SD_GO(64);
#undef EXACT_SD_GO
  return launch_status();
}

int exact_spmm_csr_rowwise_f32(const void* rowptr, const void* col, const float* val, int idx_bytes, const float* X,
                               int64_t M, int64_t n_cols, int64_t K, int64_t nnz, int reduce, float* out,
                               void* stream) {
  if (idx_bytes != 4 && idx_bytes != 8) return EXACT_E_ARG;
  if (reduce != EXACT_REDUCE_SUM && reduce != EXACT_REDUCE_MEAN) return EXACT_E_ARG;
  if (M < 0 || K < 0 || nnz < 0 || n_cols < 0 || n_cols > 0x7FFFFFFFll) return EXACT_E_SHAPE;
  if (idx_bytes == 4 && nnz > 0x7FFFFFFFll) return EXACT_E_SHAPE;
  if (M > (int64_t{1} << 32) || K > (int64_t{1} << 24)) return EXACT_E_SHAPE;  // launch-grid limits
  if (M == 0 || K == 0) return EXACT_OK;
  if (!rowptr || !out || (nnz > 0 && (!col || !X))) return EXACT_E_NULL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool mean = reduce == EXACT_REDUCE_MEAN;
  const int vec = (K % 4 == 0 && aligned_to(X, 16)) ? 4 : (K % 2 == 0 && aligned_to(X, 8)) ? 2 : 1;
#define EXACT_RW_GO(I, V) \
  rowwise_dispatch<I, V>(static_cast<const I*>(rowptr), static_cast<const I*>(col), val, X, M, K, mean, out, s)
  if (idx_bytes == 4) {
    if (vec == 4) EXACT_RW_GO(int32_t, 4); else if (vec == 2) EXACT_RW_GO(int32_t, 2); else EXACT_RW_GO(int32_t, 1);
  } else {
    if (vec == 4) EXACT_RW_GO(int64_t, 4); else if (vec == 2) EXACT_RW_GO(int64_t, 2); else EXACT_RW_GO(int64_t, 1);
  }
#undef EXACT_RW_GO
  return launch_status();
}

}  // extern "C"
