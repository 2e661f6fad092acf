// Random projection on the bf16 matrix cores of gfx950
// (v_mfma_f32_32x32x16_bf16, fp32 accumulate) with fp32 accuracy:
//   forward   out[N, k] = X[N, D]  . R[D, k]      (input2rp, ops.py:107-118)
//   backward  out[N, D] = Xr[N, k] . R[D, k]^T    (rp2input, ops.py:121-125)
//
// An fp32 number is the exact sum of three bf16 numbers: hi = bf16(x),
// mid = bf16(x - hi), lo = x - hi - mid (each difference is exact in fp32 and
// the last one has at most 8 significant bits).  So
//   * SIGNS: the reference's projection matrix is R = s * c with s = +-1 and
//     one scalar c = 1 / sqrt(k) (ops.py:112-114).  X . R = c * (X . s), and
//     X . s = hi . s + mid . s + lo . s: three bf16 products whose terms are
//     exact, summed in fp32, scaled once at the end.  3 / 16 of the matrix-core
//     time of the fp32 instruction, and one rounding per term less.
//   * SPLIT: any R (e.g. Gaussian) is split the same way and the six products
//     hi.hi, hi.mid, mid.hi, hi.lo, lo.hi, mid.mid are formed; the three left
//     out are below 2^-24 of the leading one, the rounding of an fp32 product.
// Either way the matrix cores are off the critical path and the kernels are
// left with streaming the [N, D] operand, so they are built like streaming
// kernels: many short workgroups, every lane's loads issued at once, no
// prologue.  That needs R in the layout the instruction wants, ready to load:
// exact_rp_prepare_bf16 turns R once into a TABLE of operand fragments (an
// ordinary caller-owned buffer, valid as long as R is), and the kernels read
// 16 bytes per lane from it (it stays in L2).
//
// Register layout of the instruction (wave64): lane l holds, of the A operand,
// row l % 32 and the eight k-slots 8 * (l / 32) .. + 7 (four 32-bit registers
// of two bf16 each); of the B operand column l % 32 and the same eight k-slots;
// accumulator register v of lane l is C[8 * (v / 4) + 4 * (l / 32) + v % 4][l % 32],
// as for every 32 x 32 MFMA.  A k-step covers 16 consecutive features: lane
// (row, h) reads features 8 h .. 8 h + 7 of the step, 32 contiguous bytes.
//
// Table layout (16-byte units): [0] header {c, 0, 0, 0} with c = |R[0][0]|;
// then the forward fragments [step over D][tile over k][piece][lane], lane
// (col, h) of (step, tile) holding R[16 step + 8 h + i][32 tile + col], i = 0..7;
// then the backward fragments [step over k][tile over D][piece][lane], lane
// (col, h) holding R[32 tile + col][16 step + 8 h + i].  SIGNS: one piece (the
// signs as +-1 in bf16); SPLIT: three (hi, mid, lo).  Padding entries are 0.

#include <type_traits>

#include "bf16_split.hpp"
#include "rp_common.hpp"

namespace exact {

constexpr int kStepFeatures = 16;  // K of one MFMA
constexpr int kRpXcds = 8;         // accelerator complex dies of an MI355X, each with its own L2
constexpr int kRpCus = 256;        // compute units

// Eight consecutive floats of a row starting at column `col`, zeros from column
// `limit` on; VEC = the widest aligned access (limit % VEC == 0, col % VEC == 0).
// The loads are unconditional (address clamped to the row's first piece): a
// load behind a branch would make the compiler wait for every load in flight.
template <int VEC>
__device__ __forceinline__ void load8(const float* __restrict__ row, int col, int limit, float (&v)[8]) {
#pragma unroll
  for (int p = 0; p < 8; p += VEC) {
    const bool ok = col + p < limit;
    const float* src = row + (ok ? col + p : 0);
    if constexpr (VEC == 4) {
      const f32x4 q = *reinterpret_cast<const f32x4*>(src);
      v[p] = ok ? q.x : 0.f; v[p + 1] = ok ? q.y : 0.f; v[p + 2] = ok ? q.z : 0.f; v[p + 3] = ok ? q.w : 0.f;
    } else if constexpr (VEC == 2) {
      const floatx2 q = *reinterpret_cast<const floatx2*>(src);
      v[p] = ok ? q.x : 0.f; v[p + 1] = ok ? q.y : 0.f;
    } else {
      const float q = *src;
      v[p] = ok ? q : 0.f;
    }
  }
}

// The same eight floats where they lie inside the row: two 16-byte loads at any element boundary.  Rows whose length
// is no multiple of four took 8- or 4-byte loads here, two to four times as many of the same lines.
__device__ __forceinline__ void load8_inside(const float* __restrict__ src, float (&v)[8]) {
  const f32x4_any* q = reinterpret_cast<const f32x4_any*>(src);
  const f32x4 lo = q[0], hi = q[1];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[i] = lo[i];
    v[4 + i] = hi[i];
  }
}

// ---- the table ---------------------------------------------------------------
struct TableShape {
  int steps_d, tiles_k, steps_k, tiles_d, pieces;
  __host__ __device__ int64_t fwd_units() const { return static_cast<int64_t>(steps_d) * tiles_k * pieces * kWave; }
  __host__ __device__ int64_t bwd_units() const { return static_cast<int64_t>(steps_k) * tiles_d * pieces * kWave; }
};
__host__ __device__ inline TableShape table_shape(int D, int k, int pieces) {
  return TableShape{(D + kStepFeatures - 1) / kStepFeatures, (k + kTile - 1) / kTile, (k + kStepFeatures - 1) / kStepFeatures,
                    (D + kTile - 1) / kTile, pieces};
}

// one thread per (direction, step, tile, lane): eight entries of R -> one fragment per piece
// With `matrix`, R holds 0 and 1 and what is prepared is the matrix of -c and c, which is written there as well.
template <int BP>
__global__ __launch_bounds__(kBlock) void rp_prepare_kernel(const float* __restrict__ R, int D, int k,
                                                            u32x4* __restrict__ table, float* __restrict__ matrix, float c) {
  const TableShape ts = table_shape(D, k, BP);
  const int64_t fwd_frags = static_cast<int64_t>(ts.steps_d) * ts.tiles_k * kWave;
  const int64_t bwd_frags = static_cast<int64_t>(ts.steps_k) * ts.tiles_d * kWave;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (idx == 0) {
    u32x4 head = {__float_as_uint(matrix != nullptr ? c : fabsf(R[0])), 0u, 0u, 0u};
    table[0] = head;
  }
  if (matrix != nullptr) {
    // every fragment is eight entries: the forward ones alone are at least an eighth of the entries
    for (int64_t i = idx; i < static_cast<int64_t>(D) * k; i += static_cast<int64_t>(gridDim.x) * kBlock) matrix[i] = R[i] > 0.f ? c : -c;
  }
  if (idx >= fwd_frags + bwd_frags) return;
  const bool fwd = idx < fwd_frags;
  const int64_t f = fwd ? idx : idx - fwd_frags;
  const int l = static_cast<int>(f & (kWave - 1));
  const int tiles = fwd ? ts.tiles_k : ts.tiles_d;
  const int tile = static_cast<int>((f / kWave) % tiles), step = static_cast<int>(f / (static_cast<int64_t>(kWave) * tiles));
  float r[8];
  bool inside[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    // forward: R[16 step + 8 h + i][32 tile + col];  backward: R[32 tile + col][16 step + 8 h + i]
    const int a = step * kStepFeatures + 8 * (l >> 5) + i, b = tile * kTile + (l & 31);
    const int d = fwd ? a : b, c = fwd ? b : a;
    inside[i] = d < D && c < k;
    r[i] = inside[i] ? R[static_cast<int64_t>(d) * k + c] : 0.f;
  }
  u32x4* dst = table + 1 + (fwd ? 0 : ts.fwd_units()) + (static_cast<int64_t>(step) * tiles + tile) * BP * kWave + l;
  if constexpr (BP == 1) {
    u32x4 w;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (matrix != nullptr) r[i] = r[i] > 0.f ? 1.f : -1.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = sign_bf16(r[2 * i], inside[2 * i]) | (sign_bf16(r[2 * i + 1], inside[2 * i + 1]) << 16);
    dst[0] = w;
  } else {
    const Split8 s = split3x8(r);
    dst[0] = s.hi;
    dst[kWave] = s.mid;
    dst[2 * kWave] = s.lo;
  }
}

// ---- forward -----------------------------------------------------------------
__device__ __forceinline__ void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One wavefront per 32 rows, one wavefront per workgroup: no workgroup barrier
// anywhere.  The wavefront walks the D features in chunks of 64 (four k-steps).  The instruction wants a lane to hold
// eight features of one row, but loads in that arrangement touch 64 pieces of 16 bytes in 32 rows and ran at 3 TB/s
// (190 us at 602 -> 76 columns of 232,965 rows).  So 16 lanes read 256 consecutive bytes of a row, the chunk passes
// through a tile in LDS that belongs to the wavefront (its accesses complete in order), and the lanes read their
// features from there; the next chunk's loads fly while this one is multiplied.  Before -> after, with the quantiser, both on
// one card: 602 -> 76 of 232,965 rows 185 -> 156 us, 301 -> 38 of 100,000 54 -> 37, 100 -> 25 of 2.4 M 269 -> 224, 256 -> 64
// of 2.4 M 581 -> 515, 256 -> 32 of 169,343 39.6 -> 37.6, 602 -> 76 of 20,000 34 -> 24.  At 602 -> 76 the loads and the hand-over alone take 120 us (a
// kernel that only reads in 256-byte runs 98), the split and the products the rest.  Four wavefronts that share the
// fragments through LDS: 148 us there, but 28 instead of 22 at 20,000 rows, whose workgroups then miss half the chip;
// two chunks in flight: 166.
// `frags` holds NT column tiles per k-step.  A feature past the row is zero.
constexpr int kChunkSteps = 4, kChunk = kChunkSteps * kStepFeatures;
constexpr int kChunkPitch = kChunk + 4;  // floats: 16-byte aligned rows; 16 lanes on 16 rows meet 64 different banks
constexpr int kChunkFloats = kTile * kChunkPitch;

// How many of the four columns from `col` on a load that has to stay inside a row of D >= 4 columns starts too early.
__device__ __forceinline__ int early_by(int col, int D) { return col > D - 4 ? col - (D - 4) : 0; }
// What such a load brought -> the four columns, zeros past the row.
__device__ __forceinline__ f32x4 shifted_by(f32x4 v, int early) {
  f32x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float x = 0.f;
#pragma unroll
    for (int j = 3; j >= e; --j) x = early == j - e ? v[j] : x;
    r[e] = x;
  }
  return r;
}

template <int NT, int BP>
__device__ __forceinline__ void rp_fwd_rows(const float* __restrict__ X, const u32x4* __restrict__ frags, int64_t N,
                                            int D, int64_t row0, float* chunk, floatx16 (&acc)[NT]) {
  const int lane = threadIdx.x & (kWave - 1);
  const int half = lane >> 5, l32 = lane & 31, q = lane & 15;
  const int total = (D + kStepFeatures - 1) / kStepFeatures;
  const int last = N - row0 < kTile ? static_cast<int>(N - row0) - 1 : kTile - 1;
  const float* xtile = X + row0 * D;

#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[nt][v] = 0.f;

  if (D < 4) {  // less than a piece a row
    float a[8];
    load8<1>(xtile + static_cast<int64_t>(min(l32, last)) * D, 8 * half, D, a);
    const Split8 pieces = split3x8(a);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      u32x4 b[BP];
#pragma unroll
      for (int p = 0; p < BP; ++p) b[p] = frags[(nt * BP + p) * kWave + lane];
      acc[nt] = step_product<BP>(pieces, b, acc[nt]);
    }
    return;
  }
  uint32_t at[8];  // bytes from the tile's first row to feature 4 q of rows lane / 16 + 4 i; D <= 2^20
#pragma unroll
  for (int i = 0; i < 8; ++i) at[i] = 4u * (static_cast<uint32_t>(min((lane >> 4) + 4 * i, last)) * static_cast<uint32_t>(D) + 4u * q);
  f32x4 ahead[8];
  auto load_inside = [&](int s0) {
    const char* base = reinterpret_cast<const char*>(xtile + s0 * kStepFeatures);
#pragma unroll
    for (int i = 0; i < 8; ++i) ahead[i] = *reinterpret_cast<const f32x4_any*>(base + at[i]);
  };
  auto load_tail = [&](int s0) {  // from the tile's start: less than four columns may be left, and then a piece starts before the chunk
    const char* base = reinterpret_cast<const char*>(xtile);
    const uint32_t shift = 4u * (s0 * kStepFeatures - early_by(s0 * kStepFeatures + 4 * q, D));  // at[] + shift is no less than 0 (mod 2^32)
#pragma unroll
    for (int i = 0; i < 8; ++i) ahead[i] = *reinterpret_cast<const f32x4_any*>(base + (at[i] + shift));
  };
  float* const park = chunk + (lane >> 4) * kChunkPitch + 4 * q;
  const float* const mine = chunk + l32 * kChunkPitch + 8 * half;
  // The chunk in `ahead`, from step s0 on.  NEXT: what follows -- 0 nothing, 1 a chunk inside the row, 2 the row's tail.
  auto multiply_chunk = [&](int s0, auto next) {
    constexpr int NEXT = decltype(next)::value;
    auto load_next = [&]() {
      if constexpr (NEXT == 1) load_inside(s0 + kChunkSteps);
      if constexpr (NEXT == 2) load_tail(s0 + kChunkSteps);
    };
    if (NEXT == 0 && (s0 + kChunkSteps) * kStepFeatures > D) {  // the row's tail, as load_tail brought it
      const int early = early_by(s0 * kStepFeatures + 4 * q, D);
#pragma unroll
      for (int i = 0; i < 8; ++i) ahead[i] = shifted_by(ahead[i], early);
    }
    wave_sync_lds();  // the previous chunk has been read
#pragma unroll
    for (int i = 0; i < 8; ++i) *reinterpret_cast<f32x4*>(park + 4 * i * kChunkPitch) = ahead[i];
    // Loads return in order.  The fragments of a sign matrix are few enough to be asked for before the next rows; those
    // of a split one are not, and the rows wait for them instead.
    u32x4 b[BP == 1 ? kChunkSteps : 1][NT * BP];
    auto load_frags = [&](int st, u32x4 (&f)[NT * BP]) {
      const u32x4* src = frags + static_cast<int64_t>(min(st, total - 1)) * NT * BP * kWave + lane;  // a step past the row meets zeros
#pragma unroll
      for (int p = 0; p < NT * BP; ++p) f[p] = src[p * kWave];
    };
    if constexpr (BP == 1) {
#pragma unroll
      for (int sb = 0; sb < kChunkSteps; ++sb) load_frags(s0 + sb, b[sb]);
      __builtin_amdgcn_sched_barrier(0);
      load_next();
      __builtin_amdgcn_sched_barrier(0);
    }
    wave_sync_lds();
#pragma unroll
    for (int sb = 0; sb < kChunkSteps; ++sb) {
      if (NEXT == 0 && s0 + sb >= total) break;  // wave-uniform
      const f32x4 lo = *reinterpret_cast<const f32x4*>(mine + sb * kStepFeatures);
      const f32x4 hi = *reinterpret_cast<const f32x4*>(mine + sb * kStepFeatures + 4);
      const float a[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      if constexpr (BP != 1) load_frags(s0 + sb, b[0]);
      const Split8 pieces = split3x8(a);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = step_product<BP>(pieces, b[BP == 1 ? sb : 0] + nt * BP, acc[nt]);
    }
    if constexpr (BP != 1) load_next();
  };
  if (kChunk <= D) load_inside(0);
  else load_tail(0);
  int s0 = 0;
#pragma unroll 1
  for (; (s0 + 2 * kChunkSteps) * kStepFeatures <= D; s0 += kChunkSteps) multiply_chunk(s0, std::integral_constant<int, 1>{});
  if (s0 + kChunkSteps < total) {
    multiply_chunk(s0, std::integral_constant<int, 2>{});
    s0 += kChunkSteps;
  }
  multiply_chunk(s0, std::integral_constant<int, 0>{});
}

// Wavefronts a SIMD that the registers have to leave room for (LDS holds three with three tiles, four with fewer).
template <int NT>
constexpr int fwd_waves() { return NT == 1 ? 4 : NT < 4 ? 3 : 2; }

template <int NT, int BP>
__global__ __launch_bounds__(kWave, fwd_waves<NT>()) void rp_fwd_bf16_kernel(const float* __restrict__ X,
                                                            const u32x4* __restrict__ table, int64_t N, int D,
                                                            int k, float* __restrict__ out) {
  HIP_DYNAMIC_SHARED(float, chunk)  // [32][kChunkPitch]
  const int lane = threadIdx.x & (kWave - 1);
  const int half = lane >> 5, l32 = lane & 31;
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kTile;
  floatx16 acc[NT];
  rp_fwd_rows<NT, BP>(X, table + 1, N, D, row0, chunk, acc);
  const float c = BP == 1 ? __uint_as_float(table[0][0]) : 1.f;
  // accumulator register v of lane l is C[8 (v / 4) + 4 (l / 32) + v % 4][l % 32]: a store instruction writes two
  // rows of 32 consecutive columns
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int64_t n = row0 + 8 * (v / 4) + 4 * half + (v % 4);
      const int col = nt * kTile + l32;
      if (n < N && col < k) __builtin_nontemporal_store(BP == 1 ? acc[nt][v] * c : acc[nt][v], out + n * k + col);
    }
}

// Projection and quantisation in one launch.  The wavefront turns its finished
// tile through LDS: out of the accumulator layout (a lane = one column) into the
// layout the row-wise pack kernel works in, where a lane owns an "oct" -- eight
// consecutive columns of one row, the elements of one Philox block (block
// (d / 8, n) serves columns 8 (d / 8) .. + 7 of row n) -- so the row statistics
// are eight local comparisons and a butterfly over the row's lanes, and no
// random number is computed twice.  The sums are those of rp_fwd_bf16_kernel
// (same loop) and the arithmetic is that of exact_minmax_pack_f32
// (quantization_cuda_kernel.cu:89, one rounding per operation), so the bytes
// equal those of the two launches.  The 8 / bits rows that share a packed byte
// meet through a second LDS array: every lane parks its row's bits of eight
// bytes, then one lane per (row group, oct) ORs the group's rows and stores the
// eight bytes.  Both arrays are private to the wavefront, whose LDS accesses
// complete in order: the hand-overs need no workgroup barrier.
constexpr int kStagePitch = 16;  // octs per row in the hand-over array: k <= 128
template <int NT>
constexpr int fwd_tile_pitch() { return NT * kTile + 4; }  // floats per tile row: 16-byte aligned rows, rows 4 apart on other banks

template <int NT, int BP, bool NOISE_IN>
__global__ __launch_bounds__(kWave, fwd_waves<NT>()) void rp_fwd_pack_bf16_kernel(const RpPackArgs a, const u32x4* __restrict__ table) {
  // One after the other in the same bytes: the chunks of X, the tile of sums [32][pitch], the codes uint64 [32][kStagePitch].
  // Each is whole in registers before the next is written, and LDS is what bounds the wavefronts in flight.
  HIP_DYNAMIC_SHARED(float, tile)
  constexpr int PITCH = fwd_tile_pitch<NT>();
  // passes of the 64 lanes over the tile's (row, oct) pairs: 32 rows x (1, 2 or 4 | 8 | 16) lanes per row
  constexpr int PASSES = NT == 1 ? 2 : (NT == 2 ? 4 : 8);
  uint64_t* stage = reinterpret_cast<uint64_t*>(tile);
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kTile;
  {
    floatx16 acc[NT];
    rp_fwd_rows<NT, BP>(a.X, table + 1, a.N, a.D, row0, tile, acc);
    wave_sync_lds();  // the last chunk has been read
    const float c = BP == 1 ? __uint_as_float(table[0][0]) : 1.f;
    const int half = lane >> 5, l32 = lane & 31;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        tile[(8 * (v / 4) + 4 * half + (v % 4)) * PITCH + nt * kTile + l32] = BP == 1 ? acc[nt][v] * c : acc[nt][v];
  }
  wave_sync_lds();
  uint64_t parked[PASSES];  // this lane's words of the passes below
#pragma unroll
  for (int pass = 0; pass < PASSES; ++pass) parked[pass] = 0;
  const int k = a.k, bits = a.bits;
  const int wpt = 8 / bits;
  const float B = static_cast<float>((1 << bits) - 1);
  const int octs = (k + 7) >> 3;
  int opr_log = 0;
  while ((1 << opr_log) < octs) ++opr_log;  // lanes per row: the next power of two
  const int opr = 1 << opr_log;

#pragma unroll
  for (int pass = 0; pass < PASSES; ++pass) {
    if (pass * kWave >= kTile * opr) break;
    const int t = pass * kWave + lane;
    const int i = (t >> opr_log) & (kTile - 1), oct = t & (opr - 1);  // lanes past the tile (k <= 8 only) mirror a real row
    const bool live = t < kTile * opr && oct < octs;
    const int64_t n = row0 + i;
    const int j0 = live ? 8 * oct : 0;
    // ---- the eight sums ------------------------------------------------------
    float x[8];
    {
      const float* src = tile + i * PITCH + j0;
      const f32x4 lo4 = *reinterpret_cast<const f32x4*>(src), hi4 = *reinterpret_cast<const f32x4*>(src + 4);
      x[0] = lo4.x; x[1] = lo4.y; x[2] = lo4.z; x[3] = lo4.w; x[4] = hi4.x; x[5] = hi4.y; x[6] = hi4.z; x[7] = hi4.w;
    }
    // ---- row statistics --------------------------------------------------------
    float mn = __builtin_inff(), mx = -__builtin_inff();
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (live && j0 + e < k) {
        mn = fminf(mn, x[e]);
        mx = fmaxf(mx, x[e]);
      }
    }
    group_minmax(mn, mx, opr);
    const float recip = 1.0f / (mx - mn);  // ops.py:39: reciprocal, then * B -- two roundings
    const float sc = recip * B;
    if (live && oct == 0 && n < a.N) {
      if (a.scale_f32) a.scale_f32[n] = sc;
      if (a.min_f32) a.min_f32[n] = mn;
      if (a.scale_bf16) a.scale_bf16[n] = f32_to_bf16_rne(sc);
      if (a.min_bf16) a.min_bf16[n] = f32_to_bf16_rne(mn);
    }
    // ---- noise -----------------------------------------------------------------
    float u[8];
    if constexpr (NOISE_IN) {
#pragma unroll
      for (int e = 0; e < 8; ++e) u[e] = (live && j0 + e < k && n < a.N) ? a.noise[n * k + j0 + e] : 0.f;
    } else {
      const Philox4 r = philox4x32_10(static_cast<uint32_t>(oct), static_cast<uint32_t>(n), a.off_lo, a.off_hi, a.seed_lo,
                                      a.seed_hi);
      philox_uniform8(r, u);
    }
    // ---- quantise; this row's bits of the eight bytes ------------------------------
    const int shift = (i & (wpt - 1)) * bits;
    uint32_t q[8];  // the code in the low byte
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float tq = x[e] - mn;
      tq = tq * sc;
      tq = tq + u[e];
      q[e] = code_in_low_byte(tq);  // scale and min are this row's own: tq < 2^bits + 2
    }
    // uint8_t arithmetic of the reference: bits shifted past bit 7 of a byte vanish; columns past k and rows
    // past N contribute nothing
    const uint32_t keep = (0xFFu >> shift) * 0x01010101u;
    const int cols = (live && n < a.N) ? (k - j0 < 8 ? (k - j0 < 0 ? 0 : k - j0) : 8) : 0;
    const uint64_t valid = cols >= 8 ? ~uint64_t{0} : ((uint64_t{1} << (8 * cols)) - 1);
    uint32_t word[2];
    word[0] = ((low_bytes4(q[0], q[1], q[2], q[3]) & keep) << shift) & static_cast<uint32_t>(valid);
    word[1] = ((low_bytes4(q[4], q[5], q[6], q[7]) & keep) << shift) & static_cast<uint32_t>(valid >> 32);
    parked[pass] = static_cast<uint64_t>(word[0]) | (static_cast<uint64_t>(word[1]) << 32);
  }
  wave_sync_lds();  // the sums have been read
#pragma unroll
  for (int pass = 0; pass < PASSES; ++pass) {
    const int t = pass * kWave + lane;
    if (t < kTile * opr) stage[((t >> opr_log) & (kTile - 1)) * kStagePitch + (t & (opr - 1))] = parked[pass];
  }
  wave_sync_lds();
  // ---- one lane per (row group, oct): OR the group's rows, store eight bytes -----------
  const int groups = kTile / wpt;
  const bool wide = (k & 7) == 0 && (reinterpret_cast<uintptr_t>(a.packed) & 7u) == 0;
  for (int t = lane; t < groups * octs; t += kWave) {
    const int g = t / octs, oct = t - g * octs;
    if (row0 + static_cast<int64_t>(g) * wpt >= a.N) continue;
    uint64_t w = 0;
    for (int r = 0; r < wpt; ++r) w |= stage[(g * wpt + r) * kStagePitch + oct];
    uint8_t* dst = a.packed + (row0 / wpt + g) * k + 8 * oct;
    if (wide) {
      *reinterpret_cast<uint64_t*>(dst) = w;
    } else {
      const int cnt = (k - 8 * oct < 8) ? k - 8 * oct : 8;
      for (int e = 0; e < cnt; ++e) dst[e] = static_cast<uint8_t>(w >> (8 * e));
    }
  }
  if (blockIdx.x == 0 && lane == 0) a.packed[a.pad_index] = 0;
}

// ---- tall operand times a small dense matrix ----------------------------------------
// out[N, K] = X[N, D] . M[D, K] (+ bias[K]) (+ addend[N, K]) for the linear maps of a
// layer (F.linear and the input gradient of linear_backward, backward_func.cc:83-87):
// the forward loop above with M split in three (six bf16 products per fp32
// product, fp32 accuracy), up to four column tiles per wavefront -- wider
// matrices take one launch per slab of 128 columns -- and an epilogue that adds
// a bias row and / or a matrix (which may be `out` itself: every element is read
// and written by the same lane).  The fragments of M come from
// exact_tall_gemm_prepare_bf16, which also takes M transposed (a weight as
// F.linear holds it).  No atomics: the result does not depend on the launch.
constexpr int kGemmXcds = 8;       // accelerator complex dies of an MI355X, each with its own L2
constexpr int kGemmSlabTiles = 4;  // column tiles (of 32) per wavefront at most

// The ranges in which the pieces carry a row of X and a column of M (by its largest magnitude), see below.
constexpr float kSmallRow = 0x1p-72f, kLargeRow = 0x1p+100f;
constexpr float kSmallColumn = 0x1p-28f, kLargeColumn = 0x1p+10f;

// the larger magnitude, NaN if either is one
__device__ __forceinline__ float magnitude_or(float largest, float v) {
  return __builtin_elementwise_maximum(largest, __builtin_elementwise_abs(v));
}
// The binary exponent that brings a largest magnitude into [1, 2); 0 for a column or row of zeros.
__device__ __forceinline__ int unit_exponent(float largest) {
  int e = 1;
  if (largest > 0.f) frexpf(largest, &e);
  return e - 1;
}
__device__ __forceinline__ float finite_magnitude(float v) {
  const float m = fabsf(v);
  return m <= 0x1.fffffep+127f ? m : 0.f;  // infinities and NaN set no scale
}

// Eight entries of M as pieces whose sum is the entry whatever it is: an infinity or a NaN stands in `hi` alone, a
// finite value beyond bf16's largest takes the largest below it.
__device__ __forceinline__ Split8 split3x8_any(const float (&v)[8]) {
  Split8 s;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float rest[2];
    uint32_t hi = pack_bf16x2(v[2 * i], v[2 * i + 1]);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float x = v[2 * i + j];
      const uint32_t magnitude = __float_as_uint(x) & 0x7FFFFFFFu;
      const uint32_t shift = 16 * j;
      if (magnitude < 0x7F800000u && ((hi >> shift) & 0x7F80u) == 0x7F80u)
        hi = (hi & ~(0xFFFFu << shift)) | ((__float_as_uint(x) >> 16) << shift);
      rest[j] = magnitude < 0x7F800000u ? x - (j ? high_bf16(hi) : low_bf16(hi)) : 0.f;
    }
    const uint32_t mid = pack_bf16x2(rest[0], rest[1]);
    s.hi[i] = hi;
    s.mid[i] = mid;
    s.lo[i] = pack_bf16x2(rest[0] - low_bf16(mid), rest[1] - high_bf16(mid));
  }
  return s;
}

// A workgroup makes `steps_per_wg` k-steps of one column tile.  With `exps` a column whose largest magnitude is not
// between kSmallColumn and kLargeColumn is brought into [1, 2) by a power of two (exact), so that its pieces add up to
// it whatever it is.  The workgroups of a tile each find the 32 exponents (0: as it is) for themselves; behind the
// exponents of all columns one word per tile says whether any is not 0 or any column holds an infinity or a NaN.
__global__ __launch_bounds__(kBlock) void gemm_prepare_kernel(const float* __restrict__ M, int64_t ld, int transposed,
                                                              int D, int K, int steps_per_wg, u32x4* __restrict__ table,
                                                              int32_t* __restrict__ exps) {
  __shared__ float part[2][kBlock];
  __shared__ int column_exp[kTile], flags[kTile];
  const TableShape ts = table_shape(D, K, 3);
  const int t = threadIdx.x, tile = blockIdx.x;
  if (blockIdx.x == 0 && blockIdx.y == 0 && t == 0) {
    const u32x4 head = {0u, 0u, 0u, 0u};
    table[0] = head;
  }
  if (exps) {
    // 8 threads a column; neighbouring lanes on neighbouring addresses either way M lies
    const int cl = transposed ? t >> 3 : t & 31, g = transposed ? t & 7 : t >> 5;
    const int c = tile * kTile + cl;
    const float* src = M + (transposed ? static_cast<int64_t>(c < K ? c : K - 1) * ld : static_cast<int64_t>(c < K ? c : K - 1));
    const int64_t stride = transposed ? 1 : ld;
    float m = 0.f, all = 0.f;  // of the finite entries, of all
    constexpr int kFlight = 32;  // loads in flight per thread: 256 rows in one latency
    for (int d = g; d < D; d += 8 * kFlight) {
      float v[kFlight];
#pragma unroll
      for (int i = 0; i < kFlight; ++i) v[i] = src[(d + 8 * i < D ? d + 8 * i : d) * stride];
#pragma unroll
      for (int i = 0; i < kFlight; ++i) {
        m = fmaxf(m, finite_magnitude(v[i]));
        all = magnitude_or(all, v[i]);
      }
    }
    part[0][cl * 8 + g] = m;
    part[1][cl * 8 + g] = all;
    __syncthreads();
    if (t < kTile) {
      m = all = 0.f;
      for (int i = 0; i < 8; ++i) {
        m = fmaxf(m, part[0][t * 8 + i]);
        all = magnitude_or(all, part[1][t * 8 + i]);
      }
      const bool inside = tile * kTile + t < K;
      const int e = !inside || (m >= kSmallColumn && m < kLargeColumn) ? 0 : unit_exponent(m);
      column_exp[t] = e;
      if (blockIdx.y == 0) exps[tile * kTile + t] = e;
      flags[t] = e != 0 || (inside && !(all <= 0x1.fffffep+127f));
    }
    __syncthreads();
    if (blockIdx.y == 0 && t == 0) {
      int32_t f = 0;
      for (int i = 0; i < kTile; ++i) f |= flags[i];
      exps[ts.tiles_k * kTile + tile] = f;
    }
  }
  const int l = t & (kWave - 1), c = tile * kTile + (l & 31);
  const int first = static_cast<int>(blockIdx.y) * steps_per_wg;
  const int end = first + steps_per_wg < ts.steps_d ? first + steps_per_wg : ts.steps_d;
  for (int step = first + (t >> 6); step < end; step += kBlock / kWave) {
    float r[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int d = step * kStepFeatures + 8 * (l >> 5) + i;
      const bool inside = d < D && c < K;
      r[i] = inside ? (transposed ? M[static_cast<int64_t>(c) * ld + d] : M[static_cast<int64_t>(d) * ld + c]) : 0.f;
      if (exps) r[i] = ldexpf(r[i], -column_exp[l & 31]);
    }
    u32x4* dst = table + 1 + (static_cast<int64_t>(step) * ts.tiles_k + tile) * 3 * kWave + l;
    const Split8 s = split3x8_any(r);
    dst[0] = s.hi;
    dst[kWave] = s.mid;
    dst[2 * kWave] = s.lo;
  }
}

static void gemm_prepare(const float* M, int64_t ld, int transposed, int D, int K, u32x4* table, int32_t* exps, hipStream_t s) {
  const TableShape ts = table_shape(D, K, 3);
  // four steps a workgroup, one per wavefront, while that makes at most 512 workgroups: each reads its tile's columns whole
  const int wanted = ts.tiles_k < 512 ? 512 / ts.tiles_k : 1;
  const int groups = (ts.steps_d + 3) / 4 < wanted ? (ts.steps_d + 3) / 4 : wanted;
  const int per_wg = (ts.steps_d + groups - 1) / groups;
  hipLaunchKernelGGL(gemm_prepare_kernel, dim3(static_cast<unsigned>(ts.tiles_k), static_cast<unsigned>((ts.steps_d + per_wg - 1) / per_wg)),
                     dim3(kBlock), 0, s, M, ld, transposed, D, K, per_wg, table, exps);
}

// ---- values that the three pieces do not carry --------------------------------
// The pieces of an element of X reach from 2^-133 to bf16's largest number: an infinite or larger element turns into
// infinity minus infinity, and one near the smallest normal number keeps its leading digits only.  A wavefront
// therefore keeps the largest magnitude of each of its rows (four instructions a k-step).  Where that is within
// kSmallRow .. kLargeRow, what the pieces of a smaller element lack is below 2^-61 of it, and with the columns of M
// between kSmallColumn and kLargeColumn no product of pieces that counts leaves the normal range either way.  A
// wavefront with a row outside (or a NaN in one), and every wavefront at a tile with such a column, forms the tile on
// the fp32 matrix instruction instead, from the row and the columns scaled by powers of two, in which infinities and
// NaN go through as in any fp32 product.
__device__ __forceinline__ bool row_needs_fp32(float largest) {
  return largest != 0.f && !(largest >= kSmallRow && largest < kLargeRow);
}

__device__ __forceinline__ void tall_gemm_fp32_tiles(const float* xrow, const u32x4* frags, const int32_t* exps, int64_t N, int D, int K,
                                                  int tiles, int tile0, uint32_t which, int64_t row0, const float* bias,
                                                  const float* addend, int64_t ldc, float* out, int64_t ldo) {
  const int lane = threadIdx.x & (kWave - 1), half = lane >> 5, l32 = lane & 31;
  const int total = (D + kStepFeatures - 1) / kStepFeatures;
  float largest = 0.f;
#pragma unroll 1
  for (int st = 0; st < total; ++st) {
    float a[8];
    load8<2>(xrow, st * kStepFeatures + 8 * half, D, a);
#pragma unroll
    for (int e = 0; e < 8; ++e) largest = fmaxf(largest, finite_magnitude(a[e]));
  }
  largest = fmaxf(largest, __shfl_xor(largest, 32));
  const int row_exp = unit_exponent(largest);
  const int rows_left = N - row0 < kTile ? static_cast<int>(N - row0) : kTile;
#pragma unroll 1
  for (int tile = tile0; which != 0; ++tile, which >>= 1) {
    if (!(which & 1u) || tile >= tiles) continue;
    floatx16 c;
#pragma unroll
    for (int v = 0; v < 16; ++v) c[v] = 0.f;
#pragma unroll 1
    for (int st = 0; st < total; ++st) {
      float a[8];
      load8<2>(xrow, st * kStepFeatures + 8 * half, D, a);
      const u32x4* src = frags + (static_cast<int64_t>(st) * tiles + tile) * 3 * kWave + lane;
      const u32x4 hi = src[0], mid = src[kWave], lo = src[2 * kWave];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t h = hi[e / 2], m = mid[e / 2], l = lo[e / 2];
        const float b = e % 2 ? (high_bf16(h) + high_bf16(m)) + high_bf16(l) : (low_bf16(h) + low_bf16(m)) + low_bf16(l);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(ldexpf(a[e], -row_exp), b, c, 0, 0, 0);
      }
    }
    const int col = tile * kTile + l32;
    const int col_exp = exps ? exps[col] : 0;
    const float b = (bias != nullptr && col < K) ? bias[col] : 0.f;
    float* dst = out + (row0 + 4 * half) * ldo + col;
    const float* src = addend == nullptr ? nullptr : addend + (row0 + 4 * half) * ldc + col;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int r = 8 * (v / 4) + 4 * half + (v % 4);
      const int e = static_cast<int>(__shfl(static_cast<uint32_t>(row_exp), r)) + col_exp;
      if (r < rows_left && col < K) {
        float val = ldexpf(c[v], e);
        if (bias != nullptr) val = val + b;
        if (src != nullptr) val = val + *src;
        *dst = val;
      }
      dst += v % 4 == 3 ? 5 * ldo : ldo;
      if (src != nullptr) src += v % 4 == 3 ? 5 * ldc : ldc;
    }
  }
}

// A workgroup of four wavefronts (128 rows) copies the fragments of KS k-steps x NT column tiles into LDS once and all
// read them from there; each wavefront owns 32 rows and a slab of NT column tiles.  What bounds it at [169343, 256] x
// [256, 256]: six matrix-core products per fp32 product (67 us at the 1.9 GHz the chip holds under this load), the
// vector instructions that split X, and HBM (58 us) -- overlapped only by other wavefronts, so their number is what
// counts: four tiles with one k-step per chunk at four wavefronts per SIMD, two steps at three 5 % slower, the next
// chunk fetched ahead into a second buffer at two 40 %, two row tiles per wavefront twice the time.  Narrower slabs take
// longer chunks (two steps for three tiles, four for one and two), and are held to four wavefronts as well: without
// that the compiler leaves two for three tiles (150 against 123 us at 256 -> 160) and three for two (64 against 61 at
// 256 -> 40, both with the fragments' launch).
template <int NT, int KS, bool LINES>  // LINES: every row of the result starts on a 128-byte line
__global__ __launch_bounds__(kBlock, 4) void tall_gemm_kernel(const float* __restrict__ X, const u32x4* __restrict__ table,
                                                              const int32_t* __restrict__ exps, int64_t N, int D, int K,
                                                              int tiles, int slabs, const float* __restrict__ bias,
                                                              const float* addend, int64_t ldc, float* out, int64_t ldo) {
  HIP_DYNAMIC_SHARED(u32x4, shared_frags)  // [KS][NT][3][64]
  // One launch covers `slabs` column slabs of NT tiles each.  Workgroups are handed to the 8 XCDs (each with its own
  // L2) round-robin by index, so the workgroups of one row block -- one per slab -- take indices 8 apart: they run on
  // the same XCD at about the same time and all but the first find the rows of X in that L2.  The grid is a whole
  // number of such groups; row blocks past the last row leave here, before any barrier.
  const int64_t in_group = blockIdx.x % (kGemmXcds * slabs);
  const int64_t row_block = blockIdx.x / (kGemmXcds * slabs) * kGemmXcds + in_group % kGemmXcds;
  const int tile0 = static_cast<int>(in_group / kGemmXcds) * NT;
  if (row_block * (kBlock / kWave) * kTile >= N) return;
  constexpr int kUnits = KS * NT * 3 * kWave;  // 16-byte units per chunk
  constexpr int kPerThread = (kUnits + kBlock - 1) / kBlock;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int half = lane >> 5, l32 = lane & 31;
  const int64_t row0 = (row_block * (kBlock / kWave) + wave) * kTile;
  const u32x4* frags = table + 1;
  const float* xrow = X + (row0 + l32 < N ? row0 + l32 : N - 1) * D;
  const int total = (D + kStepFeatures - 1) / kStepFeatures;
  floatx16 acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[nt][v] = 0.f;
  float row_max = 0.f;
  int32_t flags[NT];  // scalar loads, long done when they are wanted
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) flags[nt] = exps != nullptr ? exps[tiles * kTile + (tile0 + nt < tiles ? tile0 + nt : tiles - 1)] : 0;

  // This thread's share of a chunk's fragments.  A step past the row meets zeros of X and a tile past the last column
  // feeds accumulators that are never stored: any valid fragment will do for either.
  const int step_units = tiles * 3 * kWave;  // of the table: at most 4096 / 32 tiles and 4096 / 16 steps, 32-bit offsets
  auto fetch_frags = [&](int s0, u32x4 (&mine)[kPerThread]) {
#pragma unroll
    for (int u = 0; u < kPerThread; ++u) {
      // units [step][tile][piece][lane] of the chunk, 64 of one fragment piece per wavefront: all but the lane is scalar
      int piece = u * (kBlock / kWave) + wave;
      if (piece >= KS * NT * 3) piece = 0;  // not parked
      const int sb = piece / (NT * 3), tp = piece % (NT * 3);
      const int st = s0 + sb < total ? s0 + sb : s0;
      const int tile = tile0 + tp / 3 < tiles ? tile0 + tp / 3 : tiles - 1;
      const u32x4* src = frags + (st * step_units + (tile * 3 + tp % 3) * kWave);
      mine[u] = src[lane];
    }
  };
  auto fetch_rows = [&](int s0, float (&a)[KS][8]) {
    if ((s0 + KS) * kStepFeatures <= D) {  // wave-uniform: the KS steps lie inside the row, nothing to mask
#pragma unroll
      for (int sb = 0; sb < KS; ++sb) load8_inside(xrow + (s0 + sb) * kStepFeatures + 8 * half, a[sb]);
    } else {
#pragma unroll
      for (int sb = 0; sb < KS; ++sb) load8<2>(xrow, (s0 + sb) * kStepFeatures + 8 * half, D, a[sb]);
    }
  };
  auto multiply = [&](const float (&a)[KS][8]) {
#pragma unroll
    for (int sb = 0; sb < KS; ++sb) {
      u32x4 b[NT][3];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int p = 0; p < 3; ++p) b[nt][p] = shared_frags[((sb * NT + nt) * 3 + p) * kWave + lane];
#pragma unroll
      for (int i = 0; i < 8; ++i) row_max = magnitude_or(row_max, a[sb][i]);
      const Split8 pieces = split3x8(a[sb]);
      // the six products of step_product<3>, in its order for every tile, issued tile after tile: consecutive
      // matrix-core instructions write different accumulators and none waits for its predecessor
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = mfma_bf16(pieces.mid, b[nt][1], acc[nt]);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = mfma_bf16(pieces.lo, b[nt][0], acc[nt]);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = mfma_bf16(pieces.hi, b[nt][2], acc[nt]);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = mfma_bf16(pieces.mid, b[nt][0], acc[nt]);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = mfma_bf16(pieces.hi, b[nt][1], acc[nt]);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = mfma_bf16(pieces.hi, b[nt][0], acc[nt]);
    }
  };

  for (int s0 = 0; s0 < total; s0 += KS) {
    float a[KS][8];
    fetch_rows(s0, a);
    u32x4 mine[kPerThread];
    fetch_frags(s0, mine);
    __syncthreads();  // the previous chunk has been read by every wavefront
#pragma unroll
    for (int u = 0; u < kPerThread; ++u) {
      const int c = u * kBlock + static_cast<int>(threadIdx.x);
      if (kUnits % kBlock == 0 || c < kUnits) shared_frags[c] = mine[u];
    }
    __syncthreads();
    multiply(a);
  }
  row_max = magnitude_or(row_max, __shfl_xor(row_max, 32));
  // tiles that the pieces do not carry, a bit each
  uint32_t again = __ballot(row_needs_fp32(row_max)) != 0 ? (1u << NT) - 1u : 0u;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) again |= flags[nt] != 0 ? 1u << nt : 0u;
  // Accumulator register v is row 8 (v / 4) + 4 half + v % 4 of the wavefront's 32.
  float* first = out + (row0 + 4 * half) * ldo + tile0 * kTile + l32;
  // Rows all inside (all but the last wavefront of the matrix): the addresses advance by additions.  A bounds test
  // and a 64-bit product per element were a third of the kernel's vector instructions (a fifth of the time at 256 x 256).
  if (row0 + kTile <= N) {
    const float* add = addend == nullptr ? nullptr : addend + (row0 + 4 * half) * ldc + tile0 * kTile + l32;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int col = (tile0 + nt) * kTile + l32;
      if ((again >> nt) & 1u) continue;
      if (col >= K) continue;
      const float b = bias != nullptr ? bias[col] : 0.f;
      float* dst = first + nt * kTile;
      if (addend == nullptr) {
        // Whole 128-byte lines stream past the caches (154 against 164 us at 256 x 256); pieces of lines have to meet the
        // neighbouring row's or tile's in L2 first ([300000, 16] x [16, 600] 437 against 262, [2449029, 16] x [16, 70]
        // 651 against 254).
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const float val = bias != nullptr ? acc[nt][v] + b : acc[nt][v];
          if constexpr (LINES) __builtin_nontemporal_store(val, dst);
          else *dst = val;
          dst += v % 4 == 3 ? 5 * ldo : ldo;
        }
      } else {
        const float* src = add + nt * kTile;
        float more[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          more[v] = *src;
          src += v % 4 == 3 ? 5 * ldc : ldc;
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          *dst = (bias != nullptr ? acc[nt][v] + b : acc[nt][v]) + more[v];
          dst += v % 4 == 3 ? 5 * ldo : ldo;
        }
      }
    }
  } else {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int col = (tile0 + nt) * kTile + l32;
      if ((again >> nt) & 1u) continue;
      const float b = (bias != nullptr && col < K) ? bias[col] : 0.f;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t n = row0 + 8 * (v / 4) + 4 * half + (v % 4);
        if (n < N && col < K) {
          float val = acc[nt][v];
          if (bias != nullptr) val = val + b;
          if (addend != nullptr) val = val + addend[n * ldc + col];
          out[n * ldo + col] = val;
        }
      }
    }
  }
  if (__builtin_expect(again != 0, 0))
    tall_gemm_fp32_tiles(xrow, frags, exps, N, D, K, tiles, tile0, again, row0, bias, addend, ldc, out, ldo);
}

// ---- backward ----------------------------------------------------------------
// out[N, D] = Xr[N, k] . R^T: the reduction runs over the k kept columns (at most
// 128: 8 k-steps); a wavefront owns 32 rows and a slab of NT * 32 output columns
// of the result, the four wavefronts of a workgroup four consecutive row
// tiles.  They share the slab's fragments, copied from the table into LDS; the
// [N, D] result leaves through a per-wavefront LDS tile of 8 rows as 16-byte
// stores at any element boundary.  The tile is private to its wavefront, whose
// LDS accesses complete in order, so the hand-over inside it needs no workgroup
// barrier.  Bound by writing [N, D]: with D no multiple of 32 neighbouring slabs
// share lines, so the slabs of one row block take workgroup indices 8 apart (one
// XCD, about the same time: 446 -> 175 us at
// [232965, 76] x [602, 76]^T, where the stores were 4 bytes wide and the slabs apart).
template <int NT>
constexpr int bwd_tile_pitch() { return NT * kTile + 8; }  // 4 * pitch = 32 (mod 64): the two half-waves hit different banks

template <int VEC, int NT, int BP, int KS>  // KS: k-steps whose loads are issued (2, 4 or 8 >= the steps of k)
__global__ __launch_bounds__(kBlock) void rp_bwd_bf16_kernel(const float* __restrict__ Xr,
                                                             const u32x4* __restrict__ table, int64_t N, int D,
                                                             int k, int slabs, float* __restrict__ out) {
  HIP_DYNAMIC_SHARED(u32x4, frag)  // the slab's fragments [step][NT][piece][lane], then the four output tiles
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  const int half = lane >> 5;
  const int l32 = lane & 31;
  const int64_t in_group = blockIdx.x % (kRpXcds * slabs);
  const int slab = static_cast<int>(in_group / kRpXcds);
  const int64_t row_block = blockIdx.x / (kRpXcds * slabs) * kRpXcds + in_group % kRpXcds;
  if (row_block * (kBlock / kWave) * kTile >= N) return;  // whole workgroup, before any barrier
  const int dbase = slab * (NT * kTile);
  const int64_t row0 = (row_block * (kBlock / kWave) + wave) * kTile;
  const int64_t my_row = (row0 + l32 < N) ? row0 + l32 : N - 1;
  const float* xrow = Xr + my_row * k;
  const TableShape ts = table_shape(D, k, BP);
  const int steps = ts.steps_k;  // <= KS
  const u32x4* bwd = table + 1 + ts.fwd_units();

  // my loads first, then the fragments of this slab: tiles slab * NT .. + NT - 1 (past the last tile: zeros)
  float a[KS][8];
#pragma unroll
  for (int sb = 0; sb < KS; ++sb) load8<VEC>(xrow, sb * kStepFeatures + 8 * half, k, a[sb]);
  for (int idx = threadIdx.x; idx < steps * NT * BP * kWave; idx += kBlock) {
    const int l = idx & (kWave - 1), p = (idx / kWave) % BP, nt = (idx / (kWave * BP)) % NT, st = idx / (kWave * BP * NT);
    const int tile = slab * NT + nt;
    u32x4 w = {0u, 0u, 0u, 0u};
    if (tile < ts.tiles_d) w = bwd[((static_cast<int64_t>(st) * ts.tiles_d + tile) * BP + p) * kWave + l];
    frag[idx] = w;
  }
  floatx16 acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[nt][v] = 0.f;
  __syncthreads();

#pragma unroll
  for (int sb = 0; sb < KS; ++sb) {
    if (sb < steps) {
      const Split8 pieces = split3x8(a[sb]);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const u32x4* src = frag + (sb * NT + nt) * BP * kWave + lane;
        u32x4 b[BP];
#pragma unroll
        for (int p = 0; p < BP; ++p) b[p] = src[p * kWave];
        acc[nt] = step_product<BP>(pieces, b, acc[nt]);
      }
    }
  }
  if constexpr (BP == 1) {
    const float c = __uint_as_float(table[0][0]);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[nt][v] = acc[nt][v] * c;
  }

  constexpr int PC = bwd_tile_pitch<NT>();
  constexpr int kQuadsPerRow = NT * kTile / 4;
  float* Ct = reinterpret_cast<float*>(frag + steps * NT * BP * kWave) + wave * (8 * PC);  // [8][PC], this wavefront's own
#pragma unroll
  for (int g = 0; g < 4; ++g) {  // rows 8 g .. 8 g + 7 of the wavefront's 32
    wave_sync_lds();             // the tile's previous contents have been read
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) Ct[(4 * half + r) * PC + nt * kTile + l32] = acc[nt][4 * g + r];
    wave_sync_lds();
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int f = j * kWave + lane;
      const int tr = f / kQuadsPerRow, tq = f - tr * kQuadsPerRow;
      const int64_t rr = row0 + 8 * g + tr;
      const int cj = dbase + 4 * tq;
      const f32x4 q = *reinterpret_cast<const f32x4*>(Ct + tr * PC + 4 * tq);
      if (rr >= N || cj >= D) continue;
      float* dst = out + rr * D + cj;
      if (cj + 4 <= D) {
        *reinterpret_cast<f32x4_any*>(dst) = q;
      } else {
        for (int i = 0; i < D - cj; ++i) dst[i] = q[i];
      }
    }
  }
}

// The same product with the reference's signs where rows of the result do not start on whole lines.  Above, a wavefront
// writes pieces of 512 bytes of 32 rows: with rows of 2408 bytes each piece has two partial lines, and writing alone takes
// 155 us at [232965, 602] where one run takes 104; and every slab loads and splits the rows of Xr anew.  Here a workgroup
// takes 32 whole rows at a time -- one run of memory that starts on a line -- and goes on to the next 32: its four
// wavefronts own TW column tiles each, whose fragments (KS steps at most) stay in registers throughout; the rows of Xr
// come in one run, a tile ahead; and eight rows of the result at a time pass through LDS as they lie in memory (two
// buffers, one barrier each).
template <int TW, int KS>
constexpr int bwd_rows_per_cu() {  // workgroups a compute unit, by registers
  constexpr int regs = 16 * TW + 4 * TW * KS + 2 * KS + 36;
  return regs <= 64 ? 8 : regs <= 80 ? 6 : regs <= 96 ? 5 : regs <= 128 ? 4 : regs <= 168 ? 3 : 2;
}
template <int TW, int KS>
__global__ __launch_bounds__(kBlock, (bwd_rows_per_cu<TW, KS>())) void rp_bwd_rows_kernel(const float* __restrict__ Xr,
                                                                                        const u32x4* __restrict__ table, int64_t N,
                                                                                        int D, int k, float* __restrict__ out) {
  HIP_DYNAMIC_SHARED(float, lds)  // [32][kPitch] of Xr, then two images of eight rows
  constexpr int kPitch = KS * kStepFeatures + 4;  // 16-byte units: an odd number of them, 16 rows meet 64 different banks
  const int t = threadIdx.x, lane = t & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int half = lane >> 5, l32 = lane & 31;
  const int64_t tiles_n = (N + kTile - 1) / kTile;
  const TableShape ts = table_shape(D, k, 1);
  float* image = lds + kTile * kPitch;
  // fragments [step][tile][lane]; a tile past the last column is never stored, a step past k meets zeros: any will do
  u32x4 b[KS][TW];
#pragma unroll
  for (int st = 0; st < KS; ++st)
#pragma unroll
    for (int j = 0; j < TW; ++j)
      b[st][j] = table[1 + ts.fwd_units() + (static_cast<int64_t>(min(st, ts.steps_k - 1)) * ts.tiles_d + min(wave * TW + j, ts.tiles_d - 1)) * kWave + lane];
  const float c = __uint_as_float(table[0][0]);
  for (int e = t; e < kTile * kPitch; e += kBlock) lds[e] = 0.f;  // features past k stay zeros

  constexpr int kPerThread = kTile * KS * kStepFeatures / kBlock;  // of the at most 32 KS 16 features of a tile
  const int drow = kBlock / k, dcol = kBlock - drow * k;
  float x[kPerThread];
  auto load_tile = [&](int64_t tile) {  // one run; zeros past the last row
    const float* src = Xr + tile * kTile * k;
    const int count = static_cast<int>(min<int64_t>(N - tile * kTile, kTile)) * k;
#pragma unroll
    for (int i = 0; i < kPerThread; ++i) {
      const int e = i * kBlock + t;
      const float v = src[min(e, count - 1)];
      x[i] = e < count ? v : 0.f;
    }
  };
  auto park_tile = [&]() {
    int row = t / k, col = t - row * k;
#pragma unroll
    for (int i = 0; i < kPerThread; ++i) {
      if (row < kTile) lds[row * kPitch + col] = x[i];
      row += drow;
      col += dcol;
      if (col >= k) {
        col -= k;
        ++row;
      }
    }
  };
  // One tile; FULL: all its 32 rows are there.  A wait for loads waits for the stores issued ahead of them too, and where
  // some stores may or may not have been issued the compiler has to wait for all: a full tile stores the same number
  // from every lane, lanes past the end the last piece again (860 -> 654 us at 64 -> 256 of 2.4 M rows).
  auto one_tile = [&](int64_t tile, int64_t next, auto whole) {
    constexpr bool FULL = decltype(whole)::value;
    park_tile();  // the tile before was last read ahead of the barrier of its first eight rows
    __syncthreads();
    load_tile(next);
    floatx16 acc[TW];
#pragma unroll
    for (int j = 0; j < TW; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[j][v] = 0.f;
#pragma unroll
    for (int st = 0; st < KS; ++st) {
      const float* src = lds + l32 * kPitch + st * kStepFeatures + 8 * half;
      const f32x4 lo = *reinterpret_cast<const f32x4*>(src), hi = *reinterpret_cast<const f32x4*>(src + 4);
      const float a[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      const Split8 pieces = split3x8(a);
#pragma unroll
      for (int j = 0; j < TW; ++j) acc[j] = step_product<1>(pieces, &b[st][j], acc[j]);
    }
    // Addresses of the epilogue, made anew for every tile: kept across tiles they take more registers than there are
    // (480 us at 602 columns, of which 84 registers spilled).
    int lane_at = 4 * half * D + wave * TW * kTile + l32, quad_at = 4 * t;
    EXACT_VALUE_BARRIER(lane_at);
    EXACT_VALUE_BARRIER(quad_at);
    const int left = D - wave * TW * kTile - l32;  // columns from this lane's first on
#pragma unroll
    for (int g = 0; g < 4; ++g) {  // rows 8 g .. 8 g + 7
      float* eight = image + (g & 1) * 8 * D;  // last read before the barrier of the eight rows in between
#pragma unroll
      for (int j = 0; j < TW; ++j) {
        if (j * kTile < left) {
#pragma unroll
          for (int r = 0; r < 4; ++r) eight[lane_at + r * D + j * kTile] = acc[j][4 * g + r] * c;
        }
      }
      __syncthreads();
      float* dst = out + (tile * kTile + 8 * g) * D;
      constexpr int kQuads = (8 * 4 * kTile * TW / 4 + kBlock - 1) / kBlock;  // of a thread at most
      f32x4 v[kQuads];
#pragma unroll
      for (int i = 0; i < kQuads; ++i) v[i] = *reinterpret_cast<const f32x4*>(eight + min(quad_at + 4 * i * kBlock, 8 * D - 4));
      if constexpr (FULL) {
#pragma unroll
        for (int i = 0; i < kQuads; ++i) *reinterpret_cast<f32x4_any*>(dst + min(quad_at + 4 * i * kBlock, 8 * D - 4)) = v[i];
      } else {
        const int count = min(max(static_cast<int>(N - tile * kTile) - 8 * g, 0), 8) * D;  // floats
#pragma unroll
        for (int i = 0; i < kQuads; ++i) {
          const int e = quad_at + 4 * i * kBlock;
          if (e < count) {
            for (int q = 0; q < min(count - e, 4); ++q) dst[e + q] = v[i][q];
          }
        }
      }
    }
  };
  int64_t tile = blockIdx.x;  // the grid is no larger than the tiles
  load_tile(tile);
  __syncthreads();
  const int64_t whole = N / kTile, step = gridDim.x;
  for (; tile < whole; tile += step) one_tile(tile, tile + step < tiles_n ? tile + step : tiles_n - 1, std::true_type{});
  if (tile < tiles_n) one_tile(tile, tile, std::false_type{});
}

// ---- launches ----------------------------------------------------------------
template <int NT>
constexpr size_t fwd_pack_lds_bytes() {
  constexpr size_t chunk = sizeof(float) * kChunkFloats, sums = sizeof(float) * kTile * fwd_tile_pitch<NT>();
  static_assert(sizeof(uint64_t) * kTile * kStagePitch <= chunk, "the codes fit where a chunk was");
  return chunk > sums ? chunk : sums;
}

template <int BP>
static int rp_fwd_bf16_launch(const float* X, const u32x4* table, int64_t N, int D, int k, float* out, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>((N + kTile - 1) / kTile)), block(kWave);
  switch ((k + kTile - 1) / kTile) {
    case 1: hipLaunchKernelGGL((rp_fwd_bf16_kernel<1, BP>), grid, block, sizeof(float) * kChunkFloats, s, X, table, N, D, k, out); break;
    case 2: hipLaunchKernelGGL((rp_fwd_bf16_kernel<2, BP>), grid, block, sizeof(float) * kChunkFloats, s, X, table, N, D, k, out); break;
    case 3: hipLaunchKernelGGL((rp_fwd_bf16_kernel<3, BP>), grid, block, sizeof(float) * kChunkFloats, s, X, table, N, D, k, out); break;
    case 4: hipLaunchKernelGGL((rp_fwd_bf16_kernel<4, BP>), grid, block, sizeof(float) * kChunkFloats, s, X, table, N, D, k, out); break;
    default: return EXACT_E_SHAPE;
  }
  return launch_status();
}

template <int BP, bool NOISE_IN>
static int rp_fwd_pack_bf16_launch(const RpPackArgs& a, const u32x4* table, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>((a.N + kTile - 1) / kTile)), block(kWave);
  switch ((a.k + kTile - 1) / kTile) {
    case 1: hipLaunchKernelGGL((rp_fwd_pack_bf16_kernel<1, BP, NOISE_IN>), grid, block, fwd_pack_lds_bytes<1>(), s, a, table); break;
    case 2: hipLaunchKernelGGL((rp_fwd_pack_bf16_kernel<2, BP, NOISE_IN>), grid, block, fwd_pack_lds_bytes<2>(), s, a, table); break;
    case 3: hipLaunchKernelGGL((rp_fwd_pack_bf16_kernel<3, BP, NOISE_IN>), grid, block, fwd_pack_lds_bytes<3>(), s, a, table); break;
    case 4: hipLaunchKernelGGL((rp_fwd_pack_bf16_kernel<4, BP, NOISE_IN>), grid, block, fwd_pack_lds_bytes<4>(), s, a, table); break;
    default: return EXACT_E_SHAPE;
  }
  return launch_status();
}

template <int TW, int KS>
static void rp_bwd_rows_launch(const float* Xr, const u32x4* table, int64_t N, int D, int k, float* out, hipStream_t s) {
  const int64_t tiles = (N + kTile - 1) / kTile;
  const int64_t most = static_cast<int64_t>(kRpCus) * bwd_rows_per_cu<TW, KS>();
  const size_t lds = sizeof(float) * (kTile * (KS * kStepFeatures + 4) + 2 * 8 * static_cast<size_t>(D));
  hipLaunchKernelGGL((rp_bwd_rows_kernel<TW, KS>), dim3(static_cast<unsigned>(tiles < most ? tiles : most)), dim3(kBlock), lds, s, Xr, table, N,
                     D, k, out);
}
// Whether rp_bwd_rows_kernel took the product.
static bool rp_bwd_rows(const float* Xr, const u32x4* table, int64_t N, int D, int k, float* out, hipStream_t s) {
  const int steps = (k + kStepFeatures - 1) / kStepFeatures, tw = ((D + kTile - 1) / kTile + 3) / 4;
  // Measured over cold operands, this form / the other: 602 columns of 232,965 rows from 76 133 / 196 us, from 61 131 / 200, 640
  // of 200,000 from 80 123 / 159, 480 of 60,000 30 / 37, 301 of 100,000 28 / 34, 130 of 200,000 30 / 37; more than 5 steps (k > 80)
  // or 5 tiles a wavefront (D > 640) have no instance of this form, and the other takes 256 us for 602 columns of 200,000 rows from
  // 121, 166 for 500 from 100, 148 for 400 from 100 and 181 for 700 from 70 (2.3 - 3.4 TB/s); up to 256 columns of whole lines (256 of
  // 2.4 M rows 654 / 604) and up to 128 of any (100 of 2.4 M 245 / 231) the other is as fast or faster, and so it is
  // where the tiles do not reach every compute unit (602 of 3,000 rows 10.2 / 9.1).
  if (tw > 5 || steps > 5 || N < kRpCus * kTile || !(D > 256 || (D > 128 && D % 32 != 0))) return false;
#define EXACT_RP_ROWS(TW)                                                                  \
  case TW:                                                                                 \
    if (steps <= 2) rp_bwd_rows_launch<TW, 2>(Xr, table, N, D, k, out, s);                 \
    else if (steps <= 4) rp_bwd_rows_launch<TW, 4>(Xr, table, N, D, k, out, s);            \
    else rp_bwd_rows_launch<TW, 5>(Xr, table, N, D, k, out, s);                            \
    break
  switch (tw) {
    EXACT_RP_ROWS(2);
    EXACT_RP_ROWS(3);
    EXACT_RP_ROWS(4);
    EXACT_RP_ROWS(5);
  }
#undef EXACT_RP_ROWS
  return true;
}

template <int VEC, int BP, int KS>
static int rp_bwd_bf16_launch(const float* Xr, const u32x4* table, int64_t N, int D, int k, float* out, hipStream_t s) {
  const int steps = (k + kStepFeatures - 1) / kStepFeatures;
  // output slab per workgroup: 128 columns; 64 when the fragments of a 128-column slab and the tiles pass 64 KB
  const size_t frag4 = static_cast<size_t>(steps) * 4 * BP * kWave * 16;
  const size_t lds4 = frag4 + sizeof(float) * (kBlock / kWave) * 8 * bwd_tile_pitch<4>();
  const size_t lds2 = frag4 / 2 + sizeof(float) * (kBlock / kWave) * 8 * bwd_tile_pitch<2>();
  const int nt = lds4 <= 64 * 1024 ? 4 : 2;
  const int slabs = (D + nt * kTile - 1) / (nt * kTile);
  const int64_t groups = ((N + 127) / 128 + kRpXcds - 1) / kRpXcds * kRpXcds * slabs;
  if (groups > 0x7FFFFFFF) return EXACT_E_SHAPE;
  const dim3 grid(static_cast<unsigned>(groups)), block(kBlock);
  if (nt == 4) hipLaunchKernelGGL((rp_bwd_bf16_kernel<VEC, 4, BP, KS>), grid, block, lds4, s, Xr, table, N, D, k, slabs, out);
  else hipLaunchKernelGGL((rp_bwd_bf16_kernel<VEC, 2, BP, KS>), grid, block, lds2, s, Xr, table, N, D, k, slabs, out);
  return launch_status();
}

template <int VEC, int BP>
static int rp_bwd_bf16_steps(const float* Xr, const u32x4* table, int64_t N, int D, int k, float* out, hipStream_t s) {
  if (BP == 1 && rp_bwd_rows(Xr, table, N, D, k, out, s)) return launch_status();
  const int steps = (k + kStepFeatures - 1) / kStepFeatures;
  if (steps <= 2) return rp_bwd_bf16_launch<VEC, BP, 2>(Xr, table, N, D, k, out, s);
  if (steps <= 4) return rp_bwd_bf16_launch<VEC, BP, 4>(Xr, table, N, D, k, out, s);
  return rp_bwd_bf16_launch<VEC, BP, 8>(Xr, table, N, D, k, out, s);
}

static bool rp_shape_ok(int64_t N, int64_t D, int64_t k) {
  return N >= 0 && D > 0 && k > 0 && D <= (1 << 20) && k <= 128;
}
static bool rp_mode_ok(int mode) { return mode == EXACT_RP_BF16_SPLIT || mode == EXACT_RP_BF16_SIGNS; }
static int rp_pieces(int mode) { return mode == EXACT_RP_BF16_SIGNS ? 1 : 3; }

static int tall_gemm_refused(int64_t N, int64_t D, int64_t K, const float* addend, int64_t ldc, int64_t ldo) {
  if (N < 0 || D <= 0 || K <= 0 || D > 4096 || K > 4096 || D % 2 != 0) return EXACT_E_SHAPE;
  if (ldo < K || (addend && ldc < K)) return EXACT_E_SHAPE;
  return EXACT_OK;
}

static int tall_gemm_launch(const float* X, const u32x4* table, const int32_t* exps, int64_t N, int D, int K, const float* bias,
                            const float* addend, int64_t ldc, float* out, int64_t ldo, hipStream_t s) {
  const int tiles = (K + kTile - 1) / kTile;
  // slabs of equal width, at most four tiles: every slab in one launch, less than one tile per slab for padding
  const int slabs = (tiles + kGemmSlabTiles - 1) / kGemmSlabTiles;
  const int64_t rows = static_cast<int64_t>(kBlock / kWave) * kTile;
  const int64_t groups = ((N + rows - 1) / rows + kGemmXcds - 1) / kGemmXcds;  // groups of 8 row blocks
  if (groups * kGemmXcds * slabs > 0x7FFFFFFF) return EXACT_E_SHAPE;
  const dim3 grid(static_cast<unsigned>(groups * kGemmXcds * slabs)), block(kBlock);
  const bool lines = ldo % 32 == 0 && (reinterpret_cast<uintptr_t>(out) & 127) == 0;
#define EXACT_GEMM_FORM(NT, KS, LINES)                                                                                   \
  hipLaunchKernelGGL((tall_gemm_kernel<NT, KS, LINES>), grid, block, sizeof(u32x4) * KS * NT * 3 * kWave, s, X, table,   \
                     exps, N, D, K, tiles, slabs, bias, addend, ldc, out, ldo)
#define EXACT_GEMM_GO(NT, KS)                      \
  do {                                             \
    if (lines) EXACT_GEMM_FORM(NT, KS, true);      \
    else EXACT_GEMM_FORM(NT, KS, false);           \
  } while (0)
  switch ((tiles + slabs - 1) / slabs) {
    case 1: EXACT_GEMM_GO(1, 4); break;
    case 2: EXACT_GEMM_GO(2, 4); break;
    case 3: EXACT_GEMM_GO(3, 2); break;
    default: EXACT_GEMM_GO(4, 1); break;
  }
#undef EXACT_GEMM_GO
#undef EXACT_GEMM_FORM
  return launch_status();
}

}  // namespace exact

using namespace exact;

extern "C" {

int64_t exact_rp_table_nbytes(int64_t D, int64_t k, int mode) {
  if (!rp_shape_ok(0, D, k) || !rp_mode_ok(mode)) return 0;
  const TableShape ts = table_shape(static_cast<int>(D), static_cast<int>(k), rp_pieces(mode));
  return 16 * (1 + ts.fwd_units() + ts.bwd_units());
}

static int rp_prepare(const float* R, int64_t D, int64_t k, int mode, void* table, float* matrix, float c, void* stream) {
  const TableShape ts = table_shape(static_cast<int>(D), static_cast<int>(k), rp_pieces(mode));
  const int64_t frags = (ts.fwd_units() + ts.bwd_units()) / ts.pieces;
  const dim3 grid(static_cast<unsigned>((frags + kBlock - 1) / kBlock)), block(kBlock);
  hipStream_t s = static_cast<hipStream_t>(stream);
  u32x4* t = static_cast<u32x4*>(table);
  const int d = static_cast<int>(D), kk = static_cast<int>(k);
  if (mode == EXACT_RP_BF16_SIGNS) hipLaunchKernelGGL((rp_prepare_kernel<1>), grid, block, 0, s, R, d, kk, t, matrix, c);
  else hipLaunchKernelGGL((rp_prepare_kernel<3>), grid, block, 0, s, R, d, kk, t, matrix, c);
  return launch_status();
}

int exact_rp_prepare_bf16(const float* R, int64_t D, int64_t k, int mode, void* table, void* stream) {
  if (!rp_shape_ok(0, D, k)) return EXACT_E_SHAPE;
  if (!rp_mode_ok(mode)) return EXACT_E_ARG;
  if (!R || !table) return EXACT_E_NULL;
  if (!al16(table)) return EXACT_E_ALIGN;
  return rp_prepare(R, D, k, mode, table, nullptr, 0.f, stream);
}

int exact_rp_draw_signs_f32(const float* bernoulli, int64_t D, int64_t k, float c, float* R, void* table, void* stream) {
  if (!rp_shape_ok(0, D, k)) return EXACT_E_SHAPE;
  if (!(c > 0.f)) return EXACT_E_ARG;
  if (!bernoulli || !R || !table) return EXACT_E_NULL;
  if (!al16(table)) return EXACT_E_ALIGN;
  return rp_prepare(bernoulli, D, k, EXACT_RP_BF16_SIGNS, table, R, c, stream);
}

int exact_rp_fwd_bf16_f32(const float* X, const void* table, int64_t N, int64_t D, int64_t k, int mode, float* out,
                          void* stream) {
  if (!rp_shape_ok(N, D, k)) return EXACT_E_SHAPE;
  if (!rp_mode_ok(mode)) return EXACT_E_ARG;
  if (N == 0) return EXACT_OK;
  if (!X || !table || !out) return EXACT_E_NULL;
  if (!al16(table)) return EXACT_E_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const u32x4* t = static_cast<const u32x4*>(table);
  const int d = static_cast<int>(D), kk = static_cast<int>(k);
  return mode == EXACT_RP_BF16_SIGNS ? rp_fwd_bf16_launch<1>(X, t, N, d, kk, out, s) : rp_fwd_bf16_launch<3>(X, t, N, d, kk, out, s);
}

int exact_rp_minmax_pack_bf16_f32(const float* X, const void* table, int mode, const float* noise, uint64_t seed,
                                  uint64_t offset, int64_t N, int64_t D, int64_t k, int bits, uint8_t* packed,
                                  float* scale_f32, float* min_f32, uint16_t* scale_bf16, uint16_t* min_bf16,
                                  void* stream) {
  if (bits != 1 && bits != 2 && bits != 4 && bits != 8) return EXACT_E_BITS;
  if (!rp_shape_ok(N, D, k) || N > (int64_t{1} << 31) - 64) return EXACT_E_SHAPE;
  if (!rp_mode_ok(mode)) return EXACT_E_ARG;
  if (!packed) return EXACT_E_NULL;
  RpPackArgs a{};
  a.pad_index = exact_packed_nbytes(N, k, bits) - 1;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (N == 0) {
    hipLaunchKernelGGL(rp_zero_byte_kernel, dim3(1), dim3(1), 0, s, packed + a.pad_index);
    return launch_status();
  }
  if (!X || !table) return EXACT_E_NULL;
  if (!al16(table)) return EXACT_E_ALIGN;
  const u32x4* t = static_cast<const u32x4*>(table);
  a.X = X;
  a.R = nullptr;
  a.noise = noise;
  a.seed_lo = static_cast<uint32_t>(seed);
  a.seed_hi = static_cast<uint32_t>(seed >> 32);
  a.off_lo = static_cast<uint32_t>(offset);
  a.off_hi = static_cast<uint32_t>(offset >> 32);
  a.N = N;
  a.D = static_cast<int>(D);
  a.k = static_cast<int>(k);
  a.bits = bits;
  a.packed = packed;
  a.scale_f32 = scale_f32;
  a.min_f32 = min_f32;
  a.scale_bf16 = scale_bf16;
  a.min_bf16 = min_bf16;
  if (mode == EXACT_RP_BF16_SIGNS) return noise ? rp_fwd_pack_bf16_launch<1, true>(a, t, s) : rp_fwd_pack_bf16_launch<1, false>(a, t, s);
  return noise ? rp_fwd_pack_bf16_launch<3, true>(a, t, s) : rp_fwd_pack_bf16_launch<3, false>(a, t, s);
}

int exact_rp_bwd_bf16_f32(const float* Xr, const void* table, int64_t N, int64_t D, int64_t k, int mode, float* out,
                          void* stream) {
  if (!rp_shape_ok(N, D, k)) return EXACT_E_SHAPE;
  if (!rp_mode_ok(mode)) return EXACT_E_ARG;
  if (N == 0) return EXACT_OK;
  if (!Xr || !table || !out) return EXACT_E_NULL;
  if (!al16(table)) return EXACT_E_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const u32x4* t = static_cast<const u32x4*>(table);
  const int d = static_cast<int>(D), kk = static_cast<int>(k);
#define EXACT_RP_GO(V) \
  (mode == EXACT_RP_BF16_SIGNS ? rp_bwd_bf16_steps<V, 1>(Xr, t, N, d, kk, out, s) : rp_bwd_bf16_steps<V, 3>(Xr, t, N, d, kk, out, s))
  if (k % 4 == 0 && al16(Xr)) return EXACT_RP_GO(4);
  if (k % 2 == 0 && al8(Xr)) return EXACT_RP_GO(2);
  return EXACT_RP_GO(1);
#undef EXACT_RP_GO
}

int64_t exact_tall_gemm_table_nbytes(int64_t D, int64_t K) {
  if (D <= 0 || K <= 0 || D > 4096 || K > 4096) return 0;
  const TableShape ts = table_shape(static_cast<int>(D), static_cast<int>(K), 3);
  return 16 * (1 + ts.fwd_units());
}

int exact_tall_gemm_prepare_bf16(const float* M, int64_t ld, int transposed, int64_t D, int64_t K, void* table,
                                 void* stream) {
  if (D <= 0 || K <= 0 || D > 4096 || K > 4096) return EXACT_E_SHAPE;
  if (transposed != 0 && transposed != 1) return EXACT_E_ARG;
  if (ld < (transposed ? D : K)) return EXACT_E_SHAPE;
  if (!M || !table) return EXACT_E_NULL;
  if (!al16(table)) return EXACT_E_ALIGN;
  gemm_prepare(M, ld, transposed, static_cast<int>(D), static_cast<int>(K), static_cast<u32x4*>(table), nullptr,
               static_cast<hipStream_t>(stream));
  return launch_status();
}

int exact_tall_gemm_bf16_f32(const float* X, const void* table, int64_t N, int64_t D, int64_t K, const float* bias,
                             const float* addend, int64_t ldc, float* out, int64_t ldo, void* stream) {
  if (const int rc = tall_gemm_refused(N, D, K, addend, ldc, ldo)) return rc;
  if (N == 0) return EXACT_OK;
  if (!X || !table || !out) return EXACT_E_NULL;
  if (!al16(table) || !al8(X)) return EXACT_E_ALIGN;
  return tall_gemm_launch(X, static_cast<const u32x4*>(table), nullptr, N, static_cast<int>(D), static_cast<int>(K), bias, addend, ldc,
                          out, ldo, static_cast<hipStream_t>(stream));
}

int64_t exact_tall_product_work_nbytes(int64_t D, int64_t K) {
  const int64_t table = exact_tall_gemm_table_nbytes(D, K);
  return table == 0 ? 0 : table + (K + kTile - 1) / kTile * (kTile + 1) * static_cast<int64_t>(sizeof(int32_t));
}

int exact_tall_product_f32(const float* X, const float* M, int64_t ld, int transposed, int64_t N, int64_t D, int64_t K,
                           const float* bias, const float* addend, int64_t ldc, float* out, int64_t ldo, void* work,
                           void* stream) {
  if (const int rc = tall_gemm_refused(N, D, K, addend, ldc, ldo)) return rc;
  if (transposed != 0 && transposed != 1) return EXACT_E_ARG;
  if (ld < (transposed ? D : K)) return EXACT_E_SHAPE;
  if (N == 0) return EXACT_OK;
  if (!X || !M || !work || !out) return EXACT_E_NULL;
  if (!al16(work) || !al8(X)) return EXACT_E_ALIGN;
  const int d = static_cast<int>(D), k = static_cast<int>(K);
  hipStream_t s = static_cast<hipStream_t>(stream);
  u32x4* table = static_cast<u32x4*>(work);
  int32_t* exps = reinterpret_cast<int32_t*>(static_cast<uint8_t*>(work) + exact_tall_gemm_table_nbytes(D, K));
  gemm_prepare(M, ld, transposed, d, k, table, exps, s);
  return tall_gemm_launch(X, table, exps, N, d, k, bias, addend, ldc, out, ldo, s);
}

}  // extern "C"
