// CSR SpMM (sum / mean) for power-law graphs on gfx950:
//   out[r, :] = reduce_{e in row r} val[e] * X[col[e], :]
//
// Semantics restated from the reference (spmm_cuda.cu:27-104 with
// Reducer<SUM|MEAN> reducer.cuh:43-85: fp32 accumulation, mean divides by
// max(row length, 1), empty rows give 0).  The reference gives one 32-lane warp
// to each (row, 32-column tile), which serialises hub rows; this kernel splits
// the ENTRY stream into chunks of C entries, one wavefront each, so the work per
// wavefront is about the same whatever the degree distribution:
//
//   * one coalesced load brings 64 column indices (and values) into lanes; a
//     wave-uniform walk over them gathers X rows, the 64 lanes spanning
//     64 * VEC consecutive feature columns (grid.y tiles wider K);
//   * a row of at most S entries belongs to the wavefront in whose chunk it
//     starts, which walks it to its end and writes it with a plain store; the
//     wavefronts of the chunks it runs on into skip it;
//   * a longer row that straddles chunks is accumulated chunk by chunk and combined with fp32 atomic
//     adds into a row that a small pre-pass has zeroed (the same pre-pass zeroes
//     empty rows); for the mean a small post-pass divides the hubs' totals by
//     the row length.
//
// What bounds it: the gathers, nearly all of which miss L2 -- 7.4 TB/s from the
// memory-side cache on tables of 30 MB to 1 GB and 5.7 TB/s from HBM at 2.5 GB with
// uniformly random columns, whatever the tile width (32 to 256 columns measured) and the
// split.  What the split can save is everything else: where every row cut by a 64-entry chunk met
// in memory, the atomics and the zeroed rows were a fifth of the time at 2.4 M rows.

#include "exact_common.hpp"

namespace exact {

constexpr int kGather = 8;  // X rows in flight per lane (4 and 16 measure the same)
constexpr int kXcds = 8;    // accelerator complex dies of an MI355X, each with its own L2
// Mean aggregation, rows longer than S: up to this length every chunk
// divides its partial sum by the row length before the atomic add (at most 32
// rounded terms); longer rows -- the hubs -- add raw partial sums and are
// divided once by spmm_mean_finish_kernel, like the reference's reducer, so
// hundreds of rounded quotients never pile up.  Dividing every split row at
// the end would re-read and re-write most of the output on dense graphs.
constexpr int64_t kMeanFinishLen = 2048;

// VEC consecutive elements of the operand as they come from memory.  fp16 ones are widened (exactly) where they are
// used: a conversion beside the load would wait for each load before the next is issued.
template <typename T, int VEC> struct Raw { T v __attribute__((ext_vector_type(VEC))); };
template <typename T> struct Raw<T, 1> { T v; };
template <typename T, int VEC>
__device__ __forceinline__ float raw_value(const Raw<T, VEC>& r, int c) {
  if constexpr (VEC == 1) return static_cast<float>(r.v);
  else return static_cast<float>(r.v[c]);
}
template <int VEC>
__device__ __forceinline__ void store_vec(float* p, const float (&v)[VEC]) {
  if constexpr (VEC == 4) *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  else if constexpr (VEC == 2) *reinterpret_cast<float2*>(p) = make_float2(v[0], v[1]);
  else *p = v[0];
}

__device__ __forceinline__ int readlane_i(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float readlane_f(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ int64_t readlane_i64(int64_t v, int lane) {
  const int lo = __builtin_amdgcn_readlane(static_cast<int>(v), lane);
  const int hi = __builtin_amdgcn_readlane(static_cast<int>(v >> 32), lane);
  return (static_cast<int64_t>(hi) << 32) | static_cast<uint32_t>(lo);
}

// A row needs zeroing before the main kernel when nothing stores to it with a
// plain store: it is empty, or longer than S and in more than one chunk.
template <typename I>
__global__ __launch_bounds__(kBlock) void spmm_zero_rows_kernel(const I* __restrict__ rowptr, int64_t M, int C, int S,
                                                                int64_t K, int64_t ldo, float* __restrict__ out) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t base = (static_cast<int64_t>(blockIdx.x) * (kBlock / kWave) + (threadIdx.x >> 6)) * kWave;
  const int64_t r = base + lane;
  bool need = false;
  if (r < M) {
    const int64_t rs = rowptr[r], re = rowptr[r + 1];
    need = (re == rs) || (re - rs > S && rs / C != (re - 1) / C);
  }
  uint64_t todo = __ballot(need);
  while (todo) {
    const int l = __builtin_ctzll(todo);
    todo &= todo - 1;
    float* dst = out + (base + l) * ldo;
    for (int64_t c = lane; c < K; c += kWave) dst[c] = 0.f;
  }
}

// Mean aggregation, rows longer than kMeanFinishLen (which is at least S): the chunk kernel has added up their partial sums; divide by the row
// length (reducer.cuh:75-76).
template <typename I>
__global__ __launch_bounds__(kBlock) void spmm_mean_finish_kernel(const I* __restrict__ rowptr, int64_t M,
                                                                  int64_t K, int64_t ldo, float* __restrict__ out) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t base = (static_cast<int64_t>(blockIdx.x) * (kBlock / kWave) + (threadIdx.x >> 6)) * kWave;
  const int64_t r = base + lane;
  bool split = false;
  float len = 1.f;
  if (r < M) {
    const int64_t rs = rowptr[r], re = rowptr[r + 1];
    split = re - rs > kMeanFinishLen;  // in more than one chunk whatever the split
    len = static_cast<float>(re - rs);
  }
  uint64_t todo = __ballot(split);
  while (todo) {
    const int l = __builtin_ctzll(todo);
    todo &= todo - 1;
    const float d = readlane_f(len, l);
    float* dst = out + (base + l) * ldo;
    for (int64_t c = lane; c < K; c += kWave) dst[c] = dst[c] / d;
  }
}

template <typename I, typename T, int VEC, bool HAS_VAL, bool MEAN, bool OWN>  // OWN: S > 0
__global__ __launch_bounds__(kBlock) void spmm_chunk_kernel(const I* __restrict__ rowptr,
                                                            const I* __restrict__ col,
                                                            const float* __restrict__ val,
                                                            const T* __restrict__ X, int64_t M,
                                                            int64_t nnz, int64_t K, int64_t ldx, int64_t ldo,
                                                            int C, int S, float* __restrict__ out) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  // Workgroups are handed to the 8 XCDs round-robin by index; give each XCD a
  // contiguous range of chunks, so that neighbouring CSR rows (which in real
  // graphs share neighbours) gather through the same L2.  gridDim.x is a
  // multiple of kXcds; logical indices past the last chunk fall out below.
  const int64_t per_xcd = gridDim.x / kXcds;
  const int64_t wg = static_cast<int64_t>(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
  const int64_t e0 = (wg * (kBlock / kWave) + wave) * C;
  if (e0 >= nnz) return;
  const int64_t e1 = nnz - e0 < C ? nnz : e0 + C;
  const int64_t kcol = (static_cast<int64_t>(blockIdx.y) * kWave + lane) * VEC;
  const bool kok = kcol < K;

  // Row that owns entry e0: the last r with rowptr[r] <= e0.  A 64-ary search:
  // every round the 64 lanes probe 64 evenly spaced positions of [lo, hi) at
  // once and a ballot picks the sub-interval, so a graph of M rows costs
  // ceil(log64 M) dependent loads (3 for 169k rows) instead of log2 M.
  // Invariant: rowptr[lo] <= e0, and hi == M or rowptr[hi] > e0.
  int64_t lo = 0, hi = M;
  while (hi - lo > 1) {
    const int64_t step = (hi - lo + kWave - 1) / kWave;
    const int64_t pos = lo + step * lane;
    const bool le = pos < hi && static_cast<int64_t>(rowptr[pos]) <= e0;
    const uint64_t hits = __ballot(le);                 // rowptr is sorted: a run of ones from lane 0
    const int last = 63 - __builtin_clzll(hits | 1u);  // bit 0 is set by the invariant
    lo += step * last;
    hi = (lo + step < hi) ? lo + step : hi;
  }
  int64_t r = lo;

  // row ends for rows r .. r+63, one per lane
  auto load_ends = [&](int64_t first) -> int64_t {
    const int64_t idx = first + 1 + lane;
    return static_cast<int64_t>(rowptr[idx < M ? idx : M]);
  };
  int64_t ends = load_ends(r);
  int rl = 0;
  int64_t row_start = static_cast<int64_t>(rowptr[r]);
  int64_t row_end = readlane_i64(ends, 0);

  // This wavefront's entries [eb, ee): past a row that its predecessor owns, and on to the end of a row of its own
  // that runs past e1.  That row is among the 64 whose ends are at hand or is found row by row.
  int64_t eb = e0, ee = e1;
  if (OWN && row_start < e0 && row_end > e0 && row_end - row_start <= S) eb = row_end;
  if (OWN && e1 < nnz) {
    int64_t first = r, start = row_start, e64 = ends;
    uint64_t past = __ballot(e64 > e1);
    while (past == 0 && first + kWave < M) {  // 64 rows further on: many short or empty rows in one chunk
      start = readlane_i64(e64, kWave - 1);
      first += kWave;
      e64 = load_ends(first);
      past = __ballot(e64 > e1);
    }
    if (past != 0) {
      const int l = __builtin_ctzll(past);
      if (l > 0) start = readlane_i64(e64, l - 1);
      const int64_t end = readlane_i64(e64, l);
      if (start < e1 && end - start <= S) ee = end < nnz ? end : nnz;
    }
  }
  if (eb >= ee) return;

  float acc[VEC], tot[VEC];  // of the row so far: since the last multiple of 64 entries, and before it
#pragma unroll
  for (int c = 0; c < VEC; ++c) acc[c] = tot[c] = 0.f;

  auto flush = [&]() {
    if (row_end > row_start && kok) {
      float* dst = out + r * ldo + kcol;
      const int64_t len = row_end - row_start;
#pragma unroll
      for (int c = 0; c < VEC; ++c) acc[c] += tot[c];
      if ((OWN && len <= S) || (row_start >= e0 && row_end <= e1)) {
        float res[VEC];
#pragma unroll
        for (int c = 0; c < VEC; ++c) res[c] = MEAN ? acc[c] / static_cast<float>(len) : acc[c];  // reducer.cuh:75-76
        store_vec<VEC>(dst, res);
      } else {
        // a long row: its partial sums meet in memory
        const float div = (MEAN && len <= kMeanFinishLen) ? static_cast<float>(len) : 1.f;
#pragma unroll
        for (int c = 0; c < VEC; ++c) unsafeAtomicAdd(dst + c, MEAN ? acc[c] / div : acc[c]);
      }
    }
#pragma unroll
    for (int c = 0; c < VEC; ++c) acc[c] = tot[c] = 0.f;
  };
  auto advance = [&]() {
    ++r;
    ++rl;
    if (rl == kWave) {
      ends = load_ends(r);
      rl = 0;
    }
    row_start = row_end;
    row_end = readlane_i64(ends, rl);
  };

  if (OWN && eb > e0 && r + 1 < M) advance();  // nothing of the skipped row is written here

  int my_col = 0;
  float my_val = 1.f;
  auto load_entries = [&](int64_t first, int& c, float& v) {
    const int64_t e = first + lane < ee ? first + lane : ee - 1;
    c = static_cast<int>(col[e]);
    if constexpr (HAS_VAL) v = val[e];
  };
  load_entries(eb, my_col, my_val);
  for (int64_t sub = eb; sub < ee; sub += kWave) {
    int next_col = 0;
    float next_val = 1.f;
    if (sub + kWave < ee) load_entries(sub + kWave, next_col, next_val);
    const int cnt = static_cast<int>(ee - sub < kWave ? ee - sub : kWave);
#pragma unroll
    for (int c = 0; c < VEC; ++c) {
      tot[c] += acc[c];
      acc[c] = 0.f;
    }
    for (int base = 0; base < cnt; base += kGather) {
      Raw<T, VEC> xv[kGather];
#pragma unroll
      for (int u = 0; u < kGather; ++u) {
        xv[u].v = 0;
        if (base + u < cnt) {  // wave-uniform, so every lane takes part in the broadcast
          const int64_t c = readlane_i(my_col, base + u);
          if (kok) xv[u] = *reinterpret_cast<const Raw<T, VEC>*>(X + c * ldx + kcol);
        }
      }
#pragma unroll
      for (int u = 0; u < kGather; ++u) {
        if (base + u < cnt) {
          const int64_t e = sub + base + u;
          while (e >= row_end && r + 1 < M) {  // r + 1 < M: a malformed rowptr cannot spin
            flush();
            advance();
          }
          const float w = HAS_VAL ? readlane_f(my_val, base + u) : 1.f;
#pragma unroll
          for (int c = 0; c < VEC; ++c) acc[c] = __fmaf_rn(w, raw_value<T, VEC>(xv[u], c), acc[c]);
        }
      }
    }
    my_col = next_col;
    my_val = next_val;
  }
  flush();
}

static bool al(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

template <typename I, typename T, int VEC>
static void spmm_dispatch(const I* rowptr, const I* col, const float* val, const T* X, int64_t M,
                          int64_t nnz, int64_t K, int64_t ldx, int64_t ldo, int reduce, int C, int S, float* out, hipStream_t s) {
  const int64_t chunks = (nnz + C - 1) / C;
  const int64_t wgs = (chunks + 3) / 4;
  const dim3 grid(static_cast<unsigned>((wgs + kXcds - 1) / kXcds * kXcds),
                  static_cast<unsigned>((K + kWave * VEC - 1) / (kWave * VEC)));
  const dim3 block(kBlock);
  const bool mean = reduce == EXACT_REDUCE_MEAN;
#define EXACT_SPMM_CHUNK(HV, MN, OW) \
  hipLaunchKernelGGL((spmm_chunk_kernel<I, T, VEC, HV, MN, OW>), grid, block, 0, s, rowptr, col, val, X, M, nnz, K, ldx, ldo, C, S, out)
#define EXACT_SPMM_OWN(HV, MN) do { if (S > 0) EXACT_SPMM_CHUNK(HV, MN, true); else EXACT_SPMM_CHUNK(HV, MN, false); } while (0)
  if (val) {
    if (mean) EXACT_SPMM_OWN(true, true);
    else EXACT_SPMM_OWN(true, false);
  } else {
    if (mean) EXACT_SPMM_OWN(false, true);
    else EXACT_SPMM_OWN(false, false);
  }
#undef EXACT_SPMM_OWN
#undef EXACT_SPMM_CHUNK
}

// Pre-pass, product and, for the mean, post-pass, with chunks of C entries and rows of up to S in one piece.
template <typename T>
static int spmm_launch(const void* rowptr, const void* col, const float* val, int idx_bytes, const T* X, int64_t ldx,
                       int64_t M, int64_t K, int64_t nnz, int reduce, int vec, int C, int S, float* out, int64_t ldo,
                       hipStream_t s) {
  if ((K + kWave * vec - 1) / (kWave * vec) > 65535) return EXACT_E_SHAPE;  // grid.y limit
  const dim3 rgrid(static_cast<unsigned>((M + kBlock - 1) / kBlock));
  const int32_t* rowptr32 = static_cast<const int32_t*>(rowptr);
  const int64_t* rowptr64 = static_cast<const int64_t*>(rowptr);
  if (idx_bytes == 4) hipLaunchKernelGGL((spmm_zero_rows_kernel<int32_t>), rgrid, dim3(kBlock), 0, s, rowptr32, M, C, S, K, ldo, out);
  else hipLaunchKernelGGL((spmm_zero_rows_kernel<int64_t>), rgrid, dim3(kBlock), 0, s, rowptr64, M, C, S, K, ldo, out);
  if (nnz > 0) {
#define EXACT_SPMM_GO(V)                                                                                                \
  do {                                                                                                                  \
    if (idx_bytes == 4) spmm_dispatch<int32_t, T, V>(rowptr32, static_cast<const int32_t*>(col), val, X, M, nnz, K, ldx, ldo, reduce, C, S, out, s); \
    else spmm_dispatch<int64_t, T, V>(rowptr64, static_cast<const int64_t*>(col), val, X, M, nnz, K, ldx, ldo, reduce, C, S, out, s); \
  } while (0)
    if (vec == 4) {
      if constexpr (sizeof(T) == 2) EXACT_SPMM_GO(4);
    } else if (vec == 2) {
      EXACT_SPMM_GO(2);
    } else {
      EXACT_SPMM_GO(1);
    }
#undef EXACT_SPMM_GO
    if (reduce == EXACT_REDUCE_MEAN) {
      if (idx_bytes == 4) hipLaunchKernelGGL((spmm_mean_finish_kernel<int32_t>), rgrid, dim3(kBlock), 0, s, rowptr32, M, K, ldo, out);
      else hipLaunchKernelGGL((spmm_mean_finish_kernel<int64_t>), rgrid, dim3(kBlock), 0, s, rowptr64, M, K, ldo, out);
    }
  }
  return launch_status();
}

// Entries per wavefront (C) and the longest row one wavefront takes whole (S; 0: none that straddles chunks), by the
// number of wavefronts that chunks of 64 entries make.  Owned rows and longer chunks save atomics and searches but are
// the less even split, so there have to be wavefronts enough to even out their last wave; what a row in pieces costs is
// one atomic instruction per element a lane holds.  Measured on power-law graphs (us, by "C/S"):
//   fp32, two elements   0.7 k wavefronts 64/0 14.3, 64/64 16.3, 128/0 22.4; 28 k (30 entries a row) 157, 151, 132;
//                        39 k 64/0 183, 64/64 167, 128/0 169, 128/128 168; 71 k 292, 271, 269, 267;
//                        3.9 M 64/0 20.7 k, 128/0 17.9 k, 128/128 17.5 k, 256/256 17.2 k
//   fp32, one element    10 k 64/0 36.5, 128/0 39.5; 39 k 103, 100; 71 k 170, 159, 128/128 170; 1.9 M 5.3 k, 4.7 k, 256/0 4.6 k
//   fp16, four elements  10 k 64/0 91, 64/64 61, 128/128 57; 39 k 344, 212, 192; 1.9 M 20.3 k, 13.6 k, 9.6 k, 256/256 8.9 k
struct SpmmSplit { int C, S; };
static SpmmSplit spmm_split(int64_t nnz, int64_t tiles, int vec) {
  const int64_t wavefronts = nnz * tiles / 64;
  if (vec == 1) return wavefronts < 32768 ? SpmmSplit{64, 0} : wavefronts < 262144 ? SpmmSplit{128, 0} : SpmmSplit{256, 0};
  if (wavefronts >= 262144) return {256, 256};
  if (vec == 4) return wavefronts < 8192 ? SpmmSplit{64, 64} : SpmmSplit{128, 128};
  return wavefronts < 16384 ? SpmmSplit{64, 0} : wavefronts < 32768 ? SpmmSplit{128, 0} : SpmmSplit{128, 128};
}

template <typename T>
static int spmm_any(const void* rowptr, const void* col, const float* val, int idx_bytes, const T* X, int64_t ldx,
                    int64_t M, int64_t n_cols, int64_t K, int64_t nnz, int reduce, float* out, int64_t ldo, void* stream) {
  if (idx_bytes != 4 && idx_bytes != 8) return EXACT_E_ARG;
  if (reduce != EXACT_REDUCE_SUM && reduce != EXACT_REDUCE_MEAN) return EXACT_E_ARG;
  if (M < 0 || K < 0 || nnz < 0 || n_cols < 0 || n_cols > 0x7FFFFFFFll) return EXACT_E_SHAPE;
  if (idx_bytes == 4 && nnz > 0x7FFFFFFFll) return EXACT_E_SHAPE;
  // launch-grid limits: 2^31 - 1 workgroups of 256 rows (pre-pass) resp. 256 entries (main kernel)
  if (M > (int64_t{1} << 38) || nnz > (int64_t{1} << 38) || K > (int64_t{1} << 24)) return EXACT_E_SHAPE;
  if (ldx < K || ldo < K) return EXACT_E_SHAPE;
  if (M == 0 || K == 0) return EXACT_OK;
  if (!rowptr || !out || (nnz > 0 && (!col || !X))) return EXACT_E_NULL;
  // Column tile of one wavefront = 64 * vec columns.  Measured on power-law
  // graphs of 170k to 2.4M rows: 8-byte gathers (128 fp32 columns) beat 16-byte
  // ones (256 columns) by 6 to 40 % at every width from 100 to 600 -- twice
  // as many wavefronts share the same gathers -- so 16-byte gathers are not
  // used; rows of at most 64 columns take one element per lane (one tile, more lanes
  // busy than with wider ones).  fp16: four elements per lane from 129 columns on.
  constexpr int E = static_cast<int>(sizeof(T));
  const bool pairs = K > 64 && K % 2 == 0 && ldx % 2 == 0 && ldo % 2 == 0 && al(X, 2 * E) && al(out, 8);
  const bool quads = E == 2 && K > 128 && K % 4 == 0 && ldx % 4 == 0 && ldo % 4 == 0 && al(X, 8) && al(out, 16);
  const int vec = quads ? 4 : pairs ? 2 : 1;
  const SpmmSplit split = spmm_split(nnz, (K + kWave * vec - 1) / (kWave * vec), vec);
  return spmm_launch<T>(rowptr, col, val, idx_bytes, X, ldx, M, K, nnz, reduce, vec, split.C, split.S, out, ldo,
                        static_cast<hipStream_t>(stream));
}

}  // namespace exact

using namespace exact;

extern "C" {

int exact_spmm_csr_strided_f32(const void* rowptr, const void* col, const float* val, int idx_bytes,
                               const float* X, int64_t ldx, int64_t M, int64_t n_cols, int64_t K, int64_t nnz,
                               int reduce, float* out, int64_t ldo, void* stream) {
  return spmm_any<float>(rowptr, col, val, idx_bytes, X, ldx, M, n_cols, K, nnz, reduce, out, ldo, stream);
}

int exact_spmm_csr_strided_f16(const void* rowptr, const void* col, const float* val, int idx_bytes,
                               const uint16_t* X, int64_t ldx, int64_t M, int64_t n_cols, int64_t K, int64_t nnz,
                               int reduce, float* out, int64_t ldo, void* stream) {
  return spmm_any<half_t>(rowptr, col, val, idx_bytes, reinterpret_cast<const half_t*>(X), ldx, M, n_cols, K, nnz, reduce, out, ldo, stream);
}

int exact_spmm_csr_f32(const void* rowptr, const void* col, const float* val, int idx_bytes,
                       const float* X, int64_t M, int64_t n_cols, int64_t K, int64_t nnz, int reduce,
                       float* out, void* stream) {
  return exact_spmm_csr_strided_f32(rowptr, col, val, idx_bytes, X, K, M, n_cols, K, nnz, reduce, out, K, stream);
}

}  // extern "C"
