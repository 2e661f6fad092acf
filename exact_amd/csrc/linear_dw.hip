// Weight gradient of a linear layer over a tall batch:
//   dW[Kout, D] = dY[N, Kout]^T . X[N, D]          (backward_func.cc:88-89,
//                                                   grad_output.t().mm(input))
// N is the number of nodes (10^5 .. 10^6), Kout and D a few hundred at most:
// a GEMM whose reduction dimension is the long one, which general GEMM
// libraries tile poorly (a third of the fp32 matrix-core peak at best here).
//
// v_mfma_f32_32x32x2_f32 takes both operands in exactly the order memory has
// them: the A operand of lane l is A[l % 32][l / 32] = dY[n + l / 32][k0 + l % 32]
// and the B operand is B[l / 32][l % 32] = X[n + l / 32][d0 + l % 32], i.e. each
// half-wave reads 128 consecutive bytes of one row -- no transposition, no LDS.
// A wavefront owns a (32 MK) x (32 MD) block of dW in its accumulators and
// walks a slab of rows two at a time; the four wavefronts of a workgroup hold
// neighbouring blocks, so the fragments they share come out of L1.  The row
// range is cut into slabs, one workgroup each, whose blocks meet in memory
// through fp32 atomic adds into the pre-zeroed dW (the order of those
// additions is not fixed).
//
// Addresses past the last row / column are clamped, not branched around (a
// load behind a branch would make the compiler wait for every outstanding
// load at the join and so undo the prefetch): rows past the slab are zeroed
// by a select, and columns past Kout / D only feed accumulators that are never
// stored.
//
// MFMA 32x32x2 f32 accumulator layout (wave64): register v of lane l is
// C[8 * (v / 4) + 4 * (l / 32) + v % 4][l % 32].

#include <cmath>

#include "bf16_split.hpp"

namespace exact {

constexpr int kDwPairs = 4;  // row pairs per batch of loads

__global__ __launch_bounds__(kBlock) void dw_zero_kernel(float* __restrict__ out, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (i < n) out[i] = 0.f;
}

constexpr int kDwXcds = 8;   // accelerator complex dies of an MI355X, each with its own L2

// Workgroup index -> (block of dW, row slab).  Every block of dW reads the same rows of dY and X over a slab, and
// workgroups are handed to the 8 XCDs round-robin by index: the `blocks` workgroups of one slab take indices 8
// apart, so they run on one XCD at about the same time and the rows come from HBM once and from that L2 afterwards.
// The grid is a whole number of groups of 8 slabs; false for a slab past the last one.
__device__ __forceinline__ bool dw_block_and_slab(int blocks, int64_t slabs, int& block, int64_t& slab) {
  const int64_t per_group = static_cast<int64_t>(kDwXcds) * blocks;
  const int64_t in_group = blockIdx.x % per_group;
  block = static_cast<int>(in_group / kDwXcds);
  slab = blockIdx.x / per_group * kDwXcds + in_group % kDwXcds;
  return slab < slabs;
}

// WK x (4 / WK) wavefronts per workgroup along Kout x D.  ORDERED: `out` is scratch [slab][Kout][D] and
// dw_finish_kernel adds the slabs in their order; else they meet in `out` through atomics.
template <int MK, int MD, int WK, bool ORDERED>
__global__ __launch_bounds__(kBlock) void linear_dw_kernel(const float* __restrict__ dY, int64_t ldy,
                                                           const float* __restrict__ X, int64_t ldx, int64_t N,
                                                           int Kout, int D, int64_t rows_per_slab, int blocks_d, int blocks, int64_t slabs,
                                                           float* __restrict__ out) {
  constexpr int WD = 4 / WK;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  const int half = lane >> 5;
  const int l32 = lane & 31;
  int block;
  int64_t slab;
  if (!dw_block_and_slab(blocks, slabs, block, slab)) return;  // whole workgroup
  const int bk = block / blocks_d, bd = block % blocks_d;
  const int k0 = (bk * WK + wave / WD) * (32 * MK);
  const int d0 = (bd * WD + wave % WD) * (32 * MD);
  if (k0 >= Kout || d0 >= D) return;  // whole wavefront: no barrier follows
  const int64_t n_begin = slab * rows_per_slab;
  const int64_t n_end = (n_begin + rows_per_slab < N) ? n_begin + rows_per_slab : N;

  int kcol[MK], dcol[MD];
#pragma unroll
  for (int i = 0; i < MK; ++i) kcol[i] = min(k0 + 32 * i + l32, Kout - 1);
#pragma unroll
  for (int j = 0; j < MD; ++j) dcol[j] = min(d0 + 32 * j + l32, D - 1);

  floatx16 acc[MK][MD];
#pragma unroll
  for (int i = 0; i < MK; ++i)
#pragma unroll
    for (int j = 0; j < MD; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  auto load_batch = [&](int64_t n0, float (&a)[kDwPairs][MK], float (&b)[kDwPairs][MD]) {
#pragma unroll
    for (int p = 0; p < kDwPairs; ++p) {
      const int64_t row = n0 + 2 * p + half;
      const int64_t rc = row < N ? row : N - 1;
      const bool ok = row < n_end;
#pragma unroll
      for (int i = 0; i < MK; ++i) {
        const float v = dY[rc * ldy + kcol[i]];
        a[p][i] = ok ? v : 0.f;
      }
#pragma unroll
      for (int j = 0; j < MD; ++j) {
        const float v = X[rc * ldx + dcol[j]];
        b[p][j] = ok ? v : 0.f;
      }
    }
  };
  auto mfma_batch = [&](const float (&a)[kDwPairs][MK], const float (&b)[kDwPairs][MD]) {
#pragma unroll
    for (int p = 0; p < kDwPairs; ++p)
#pragma unroll
      for (int i = 0; i < MK; ++i)
#pragma unroll
        for (int j = 0; j < MD; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[p][i], b[p][j], acc[i][j], 0, 0, 0);
  };

  constexpr int64_t kStep = 2 * kDwPairs;
  float a0[kDwPairs][MK], b0[kDwPairs][MD], a1[kDwPairs][MK], b1[kDwPairs][MD];
  int64_t n0 = n_begin;
  if (n0 < n_end) load_batch(n0, a0, b0);
  while (n0 < n_end) {
    load_batch(n0 + kStep, a1, b1);  // past the slab: clamped addresses, zeroed values
    mfma_batch(a0, b0);
    n0 += kStep;
    if (n0 >= n_end) break;
    load_batch(n0 + kStep, a0, b0);
    mfma_batch(a1, b1);
    n0 += kStep;
  }

#pragma unroll
  for (int i = 0; i < MK; ++i)
#pragma unroll
    for (int j = 0; j < MD; ++j) {
      const int cj = d0 + 32 * j + l32;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int ri = k0 + 32 * i + 8 * (v / 4) + 4 * half + (v % 4);
        if (ri < Kout && cj < D) {
          if constexpr (ORDERED) out[(slab * Kout + ri) * D + cj] = acc[i][j][v];
          else unsafeAtomicAdd(out + static_cast<int64_t>(ri) * D + cj, acc[i][j][v]);
        }
      }
    }
}

// The same product on the bf16 matrix cores at fp32 accuracy (bf16_split.hpp):
// v_mfma_f32_32x32x16_bf16 reduces over 16 rows per instruction, lane (column,
// g) holding rows n + 8 g .. n + 8 g + 7 of its column -- eight 4-byte loads
// per operand fragment, each again 128 consecutive bytes per half-wave.  Both
// operands are split into three bf16 pieces in registers and every 32 x 32
// block takes six instructions per 16 rows, 3 / 8 of the matrix-core time of
// the fp32 instruction.
template <int MK, int MD, int WK>
__global__ __launch_bounds__(kBlock, 2) void linear_dw_bf16_kernel(const float* __restrict__ dY, int64_t ldy,
                                                                const float* __restrict__ X, int64_t ldx, int64_t N,
                                                                int Kout, int D, int64_t rows_per_slab, int blocks_d, int blocks, int64_t slabs,
                                                                float* __restrict__ out) {
  constexpr int WD = 4 / WK;
  constexpr int64_t kRows = 16;  // rows per step
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  const int half = lane >> 5;
  const int l32 = lane & 31;
  int block;
  int64_t slab;
  if (!dw_block_and_slab(blocks, slabs, block, slab)) return;  // whole workgroup
  const int bk = block / blocks_d, bd = block % blocks_d;
  const int k0 = (bk * WK + wave / WD) * (32 * MK);
  const int d0 = (bd * WD + wave % WD) * (32 * MD);
  if (k0 >= Kout || d0 >= D) return;  // whole wavefront: no barrier follows
  const int64_t n_begin = slab * rows_per_slab;
  const int64_t n_end = (n_begin + rows_per_slab < N) ? n_begin + rows_per_slab : N;

  int kcol[MK], dcol[MD];
#pragma unroll
  for (int i = 0; i < MK; ++i) kcol[i] = min(k0 + 32 * i + l32, Kout - 1);
#pragma unroll
  for (int j = 0; j < MD; ++j) dcol[j] = min(d0 + 32 * j + l32, D - 1);

  floatx16 acc[MK][MD];
#pragma unroll
  for (int i = 0; i < MK; ++i)
#pragma unroll
    for (int j = 0; j < MD; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  const float* ycol[MK];
  const float* xcol[MD];
#pragma unroll
  for (int i = 0; i < MK; ++i) ycol[i] = dY + kcol[i];
#pragma unroll
  for (int j = 0; j < MD; ++j) xcol[j] = X + dcol[j];
  auto load_step = [&](int64_t n0, float (&a)[MK][8], float (&b)[MD][8]) {
    if (n0 + kRows <= n_end) {  // wave-uniform: the whole step lies inside the slab, nothing to clamp or mask
      const int64_t first = n0 + 8 * half;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
#pragma unroll
        for (int i = 0; i < MK; ++i) a[i][e] = ycol[i][(first + e) * ldy];
#pragma unroll
        for (int j = 0; j < MD; ++j) b[j][e] = xcol[j][(first + e) * ldx];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int64_t row = n0 + 8 * half + e;
        const int64_t rc = row < N ? row : N - 1;
        const bool ok = row < n_end;
#pragma unroll
        for (int i = 0; i < MK; ++i) {
          const float v = ycol[i][rc * ldy];
          a[i][e] = ok ? v : 0.f;
        }
#pragma unroll
        for (int j = 0; j < MD; ++j) {
          const float v = xcol[j][rc * ldx];
          b[j][e] = ok ? v : 0.f;
        }
      }
    }
  };
  // One set of raw registers: a step's values are split into their bf16 pieces first, then the
  // loads of the next step are issued into the same registers and fly during this step's MFMAs.
  float a[MK][8], b[MD][8];
  int64_t n0 = n_begin;
  if (n0 < n_end) load_step(n0, a, b);
  while (n0 < n_end) {
    Split8 sa[MK], sb[MD];
#pragma unroll
    for (int i = 0; i < MK; ++i) sa[i] = split3x8(a[i]);
#pragma unroll
    for (int j = 0; j < MD; ++j) sb[j] = split3x8(b[j]);
    load_step(n0 + kRows, a, b);  // past the slab: clamped addresses, zeroed values
#pragma unroll
    for (int i = 0; i < MK; ++i)
#pragma unroll
      for (int j = 0; j < MD; ++j) {
        const u32x4 pieces[3] = {sb[j].hi, sb[j].mid, sb[j].lo};
        acc[i][j] = step_product<3>(sa[i], pieces, acc[i][j]);
      }
    n0 += kRows;
  }

#pragma unroll
  for (int i = 0; i < MK; ++i)
#pragma unroll
    for (int j = 0; j < MD; ++j) {
      const int cj = d0 + 32 * j + l32;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int ri = k0 + 32 * i + 8 * (v / 4) + 4 * half + (v % 4);
        if (ri < Kout && cj < D) unsafeAtomicAdd(out + static_cast<int64_t>(ri) * D + cj, acc[i][j][v]);
      }
    }
}

// The same with the fragments shared.  Above, every wavefront splits the fragments of its own rows and columns, and the
// split (44 vector instructions per fragment) competes with the matrix cores.  Here the four wavefronts divide the
// fragments of a step between them, split each once and hand the pieces round through LDS, in two buffers so that one
// barrier per step suffices; the rows of the step after next are on their way while a step is multiplied.  With operand
// sets in turn, so that none is found in the memory-side cache, [169343, 256]^T x [169343, 256] takes 174 us (own form
// 216 - 231) and 188 under the tracer; with one set 161.
template <int MK, int MD, int WK>
__global__ __launch_bounds__(kBlock, 2) void linear_dw_shared_kernel(const float* __restrict__ dY, int64_t ldy,
                                                                const float* __restrict__ X, int64_t ldx, int64_t N,
                                                                int Kout, int D, int64_t rows_per_slab, int blocks_d, int blocks, int64_t slabs,
                                                                float* __restrict__ out) {
  constexpr int WD = 4 / WK;
  constexpr int KT = MK * WK, DT = MD * WD, F = KT + DT;  // fragments of a step: KT of dY, then DT of X
  constexpr int FPW = (F + 3) / 4;                        // of them, per wavefront: wave, wave + 4, ..
  constexpr int64_t kRows = 16;                           // rows per step
  HIP_DYNAMIC_SHARED(u32x4, shared)                       // [2][F][piece][lane]
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int half = lane >> 5;
  const int l32 = lane & 31;
  int block;
  int64_t slab;
  if (!dw_block_and_slab(blocks, slabs, block, slab)) return;  // whole workgroup, before any barrier
  const int bk = block / blocks_d, bd = block % blocks_d;
  const int wk = wave / WD, wd = wave % WD;
  const int k0 = (bk * WK + wk) * (32 * MK);
  const int d0 = (bd * WD + wd) * (32 * MD);
  const bool active = k0 < Kout && d0 < D;  // wave-uniform; an inactive wavefront still brings its fragments
  const int64_t n_begin = slab * rows_per_slab;
  const int64_t n_end = (n_begin + rows_per_slab < N) ? n_begin + rows_per_slab : N;

  // my fragments' columns; past the last column: clamped, they only feed accumulators that are never stored
  const float* src[FPW];
  int64_t ld[FPW];
#pragma unroll
  for (int j = 0; j < FPW; ++j) {
    const int f = wave + 4 * j < F ? wave + 4 * j : F - 1;
    const bool is_y = f < KT;
    const int c = is_y ? (bk * KT + f) * 32 + l32 : (bd * DT + f - KT) * 32 + l32;
    src[j] = is_y ? dY + min(c, Kout - 1) : X + min(c, D - 1);
    ld[j] = is_y ? ldy : ldx;
  }
  floatx16 acc[MK][MD];
#pragma unroll
  for (int i = 0; i < MK; ++i)
#pragma unroll
    for (int j = 0; j < MD; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  float raw[FPW][8];
  auto load_step = [&](int64_t n0) {
    if (n0 + kRows <= n_end) {  // the same in the whole workgroup: the step lies inside the slab, nothing to clamp
#pragma unroll
      for (int j = 0; j < FPW; ++j) {
        const float* p = src[j] + (n0 + 8 * half) * ld[j];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          raw[j][e] = *p;
          p += ld[j];
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < FPW; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int64_t row = n0 + 8 * half + e;
          const float v = src[j][(row < N ? row : N - 1) * ld[j]];
          raw[j][e] = row < n_end ? v : 0.f;
        }
    }
  };
  auto park_step = [&](int buffer) {
#pragma unroll
    for (int j = 0; j < FPW; ++j) {
      const int f = wave + 4 * j;
      if (f >= F) continue;  // wave-uniform
      const Split8 s = split3x8(raw[j]);
      u32x4* dst = shared + (buffer * F + f) * 3 * kWave + lane;
      dst[0] = s.hi;
      dst[kWave] = s.mid;
      dst[2 * kWave] = s.lo;
    }
  };
  auto multiply = [&](int buffer) {
    const u32x4* base = shared + buffer * F * 3 * kWave + lane;
    u32x4 b[MD][3];
#pragma unroll
    for (int j = 0; j < MD; ++j)
#pragma unroll
      for (int p = 0; p < 3; ++p) b[j][p] = base[((KT + wd * MD + j) * 3 + p) * kWave];
#pragma unroll
    for (int i = 0; i < MK; ++i) {
      const u32x4* fa = base + (wk * MK + i) * 3 * kWave;
      const Split8 a = {fa[0], fa[kWave], fa[2 * kWave]};
#pragma unroll
      for (int j = 0; j < MD; ++j) acc[i][j] = step_product<3>(a, b[j], acc[i][j]);
    }
  };

  if (n_begin >= n_end) return;  // an empty slab: whole workgroup
  load_step(n_begin);
  park_step(0);
  load_step(n_begin + kRows);  // past the slab: clamped addresses, zeroed values
  __syncthreads();
  int buffer = 0;
  for (int64_t n0 = n_begin; n0 < n_end; n0 += kRows) {
    if (active) multiply(buffer);
    buffer ^= 1;
    if (n0 + kRows < n_end) {   // the same in the whole workgroup
      park_step(buffer);        // last read before the barrier that ended the previous step
      load_step(n0 + 2 * kRows);
      __syncthreads();
    }
  }
  if (!active) return;

#pragma unroll
  for (int i = 0; i < MK; ++i)
#pragma unroll
    for (int j = 0; j < MD; ++j) {
      const int cj = d0 + 32 * j + l32;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int ri = k0 + 32 * i + 8 * (v / 4) + 4 * half + (v % 4);
        if (ri < Kout && cj < D) unsafeAtomicAdd(out + static_cast<int64_t>(ri) * D + cj, acc[i][j][v]);
      }
    }
}

// fp16 operands (autocast): the same walk on v_mfma_f32_32x32x16_f16, which takes them as they are -- products of two
// fp16 numbers are exact in fp32, infinities, NaN and subnormal numbers among them.  A fragment is one 16-byte unit per
// lane, so a step is 32 rows.  A slab's block goes to `partial` [slab][Kout][D] and dw_finish_kernel adds the slabs
// in their order: two equal calls give equal bits.
template <int MK, int MD, int WK>
__global__ __launch_bounds__(kBlock, 2) void linear_dw_half_kernel(const half_t* __restrict__ dY, int64_t ldy,
                                                                   const half_t* __restrict__ X, int64_t ldx, int64_t N,
                                                                   int Kout, int D, int64_t rows_per_slab, int blocks_d, int blocks, int64_t slabs,
                                                                   float* __restrict__ partial) {
  constexpr int WD = 4 / WK;
  constexpr int KT = MK * WK, DT = MD * WD, F = KT + DT;  // fragments of 16 rows: KT of dY, then DT of X
  constexpr int FPW = (F + 3) / 4;                        // of them, per wavefront: wave, wave + 4, ..
  constexpr int SUB = 2, kRows = 16 * SUB;                // rows per step
  HIP_DYNAMIC_SHARED(u32x4, shared)                       // [2][SUB][F][lane]
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int half = lane >> 5;
  const int l32 = lane & 31;
  int block;
  int64_t slab;
  if (!dw_block_and_slab(blocks, slabs, block, slab)) return;  // whole workgroup, before any barrier
  const int bk = block / blocks_d, bd = block % blocks_d;
  const int wk = wave / WD, wd = wave % WD;
  const int k0 = (bk * WK + wk) * (32 * MK);
  const int d0 = (bd * WD + wd) * (32 * MD);
  const bool active = k0 < Kout && d0 < D;  // wave-uniform; an inactive wavefront still brings its fragments
  const int64_t n_begin = slab * rows_per_slab;
  const int64_t n_end = (n_begin + rows_per_slab < N) ? n_begin + rows_per_slab : N;

  // my fragments' columns; past the last column: clamped, they only feed accumulators that are never stored
  const half_t* src[FPW];
  int64_t ld[FPW];
#pragma unroll
  for (int j = 0; j < FPW; ++j) {
    const int f = wave + 4 * j < F ? wave + 4 * j : F - 1;
    const bool is_y = f < KT;
    const int c = is_y ? (bk * KT + f) * 32 + l32 : (bd * DT + f - KT) * 32 + l32;
    src[j] = is_y ? dY + min(c, Kout - 1) : X + min(c, D - 1);
    ld[j] = is_y ? ldy : ldx;
  }
  floatx16 acc[MK][MD];
#pragma unroll
  for (int i = 0; i < MK; ++i)
#pragma unroll
    for (int j = 0; j < MD; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  half8 raw[SUB][FPW];
  auto load_step = [&](int64_t n0) {
    if (n0 + kRows <= n_end) {  // the same in the whole workgroup: the step lies inside the slab, nothing to clamp
#pragma unroll
      for (int s = 0; s < SUB; ++s)
#pragma unroll
        for (int j = 0; j < FPW; ++j) {
          const half_t* p = src[j] + (n0 + 16 * s + 8 * half) * ld[j];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            raw[s][j][e] = *p;
            p += ld[j];
          }
        }
    } else {
#pragma unroll
      for (int s = 0; s < SUB; ++s)
#pragma unroll
        for (int j = 0; j < FPW; ++j)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int64_t row = n0 + 16 * s + 8 * half + e;
            const half_t v = src[j][(row < N ? row : N - 1) * ld[j]];
            raw[s][j][e] = row < n_end ? v : static_cast<half_t>(0.f);
          }
    }
  };
  auto park_step = [&](int buffer) {
#pragma unroll
    for (int s = 0; s < SUB; ++s)
#pragma unroll
      for (int j = 0; j < FPW; ++j) {
        const int f = wave + 4 * j;
        if (f < F) shared[((buffer * SUB + s) * F + f) * kWave + lane] = __builtin_bit_cast(u32x4, raw[s][j]);  // wave-uniform
      }
  };
  auto multiply = [&](int buffer) {
#pragma unroll
    for (int s = 0; s < SUB; ++s) {
      const u32x4* base = shared + (buffer * SUB + s) * F * kWave + lane;
      half8 b[MD];
#pragma unroll
      for (int j = 0; j < MD; ++j) b[j] = __builtin_bit_cast(half8, base[(KT + wd * MD + j) * kWave]);
#pragma unroll
      for (int i = 0; i < MK; ++i) {
        const half8 a = __builtin_bit_cast(half8, base[(wk * MK + i) * kWave]);
#pragma unroll
        for (int j = 0; j < MD; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b[j], acc[i][j], 0, 0, 0);
      }
    }
  };

  if (n_begin < n_end) {  // the same in the whole workgroup; the last slabs of a short batch may be empty
    load_step(n_begin);
    park_step(0);
    load_step(n_begin + kRows);  // past the slab: clamped addresses, zeroed values
    __syncthreads();
    int buffer = 0;
    for (int64_t n0 = n_begin; n0 < n_end; n0 += kRows) {
      if (active) multiply(buffer);
      buffer ^= 1;
      if (n0 + kRows < n_end) {  // the same in the whole workgroup
        park_step(buffer);       // last read before the barrier that ended the previous step
        load_step(n0 + 2 * kRows);
        __syncthreads();
      }
    }
  }
  if (!active) return;
  float* mine = partial + slab * Kout * D;
#pragma unroll
  for (int i = 0; i < MK; ++i)
#pragma unroll
    for (int j = 0; j < MD; ++j) {
      const int cj = d0 + 32 * j + l32;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int ri = k0 + 32 * i + 8 * (v / 4) + 4 * half + (v % 4);
        if (ri < Kout && cj < D) mine[static_cast<int64_t>(ri) * D + cj] = acc[i][j][v];
      }
    }
}

// out[i] = the sum over the slabs, rounded to T: eight groups of 32 lanes take every eighth slab, then meet in LDS in
// their order.
template <typename T>
__global__ __launch_bounds__(kBlock) void dw_finish_kernel(const float* __restrict__ partial, int64_t total, int64_t slabs,
                                                           T* __restrict__ out) {
  __shared__ float part[kBlock];
  const int t = threadIdx.x, g = t >> 5;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 32 + (t & 31);
  const float* p = partial + (i < total ? i : total - 1);
  float s = 0.f;
  for (int64_t k = g; k < slabs; k += 64) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[(k + 8 * u < slabs ? k + 8 * u : k) * total];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += k + 8 * u < slabs ? v[u] : 0.f;
  }
  part[t] = s;
  __syncthreads();
  if (g == 0 && i < total) {
#pragma unroll
    for (int k = 1; k < 8; ++k) s += part[32 * k + t];
    out[i] = static_cast<T>(s);
  }
}

// How the forms with a fixed order cut their work.
struct DwOrderedPlan {
  int mk, md, wk, blocks_d, blocks;
  int64_t rows, slabs;
};
static DwOrderedPlan plan_dw_blocks(int K, int D) {
  DwOrderedPlan p{};
  p.mk = K <= 32 ? 1 : 2;
  p.md = (K <= 64 ? D <= 128 : D <= 32) ? 1 : 2;
  p.wk = K <= 64 ? 1 : D <= 64 ? 4 : 2;
  const int kb = 32 * p.mk * p.wk, db = 32 * p.md * (4 / p.wk);
  p.blocks_d = (D + db - 1) / db;
  p.blocks = (K + kb - 1) / kb * p.blocks_d;
  return p;
}
// fp16: about 512 workgroups (two per compute unit), at least 512 rows a slab, whole steps.
static DwOrderedPlan plan_dw_half(int64_t N, int K, int D) {
  DwOrderedPlan p = plan_dw_blocks(K, D);
  const int64_t wanted = (512 + p.blocks - 1) / p.blocks;
  p.rows = (N + wanted - 1) / wanted;
  if (p.rows < 512) p.rows = 512;
  p.rows = (p.rows + 31) / 32 * 32;
  p.slabs = (N + p.rows - 1) / p.rows;
  return p;
}
// Rows of a slab for which the two things that grow with its length and with its number are together least: a
// wavefront's walk, `row_us` a row, and the slabs' results, `value_us` each.  Whole steps of 16, between `least` and 512.
static int64_t dw_slab_rows(int64_t N, int K, int D, double row_us, double value_us, int64_t least) {
  int64_t rows = static_cast<int64_t>(std::sqrt(static_cast<double>(N) * K * D * value_us / row_us));
  rows = rows < least ? least : rows > 512 ? 512 : rows;
  return (rows + 15) / 16 * 16;
}
// fp32, short batches: each further row of a slab costs 0.06 (64 x 64 results) to 0.13 us (256 x 256), taken as 0.11, and
// a result 8 bytes of traffic; the launches, the first loads and the finish are another 6 to 12 us.  Both kernels, 16 / 32
// / 64 / 128 / 256 / 512 rows a slab: 4,096 rows 64 x 64 9.8 / 9.2 / 10.3 / 14.3 / 22.5 / 39 us, 256 x 256 38 / 22 / 21 /
// 28 / 45 / 81; 16,000 rows 17.6 / 14.6 / 13.5 / 17.4 / 27 / 46 and 149 / 90 / 59 / 46 / 49 / 82.  Against the framework's
// GEMM: 4,096 rows 64 x 64 10.2 / 32.7, 128 x 128 17.7 / 25.2, 256 x 256 25.7 / 25.4; 16,383 rows 14.1 / 120, 25.2 / 98,
// 46.8 / 105.
static DwOrderedPlan plan_dw_short(int64_t N, int K, int D) {
  DwOrderedPlan p = plan_dw_blocks(K, D);
  p.rows = dw_slab_rows(N, K, D, 0.11, 2e-6, 64);
  p.slabs = (N + p.rows - 1) / p.rows;
  return p;
}

template <int MK, int MD, int WK>
static void launch_dw_half(const DwOrderedPlan& p, const half_t* dY, int64_t ldy, const half_t* X, int64_t ldx, int64_t N, int Kout, int D,
                           float* partial, hipStream_t s) {
  constexpr size_t lds = sizeof(u32x4) * 2 * 2 * (MK * WK + MD * (4 / WK)) * kWave;
  const dim3 grid(static_cast<unsigned>((p.slabs + kDwXcds - 1) / kDwXcds * kDwXcds * p.blocks));
  hipLaunchKernelGGL((linear_dw_half_kernel<MK, MD, WK>), grid, dim3(kBlock), lds, s, dY, ldy, X, ldx, N, Kout, D, p.rows, p.blocks_d,
                     p.blocks, p.slabs, partial);
}

template <int MK, int MD, int WK>
static void launch_dw_short(const DwOrderedPlan& p, const float* dY, int64_t ldy, const float* X, int64_t ldx, int64_t N, int Kout, int D,
                            float* partial, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>((p.slabs + kDwXcds - 1) / kDwXcds * kDwXcds * p.blocks));
  hipLaunchKernelGGL((linear_dw_kernel<MK, MD, WK, true>), grid, dim3(kBlock), 0, s, dY, ldy, X, ldx, N, Kout, D, p.rows, p.blocks_d, p.blocks,
                     p.slabs, partial);
}

template <int MK, int MD, int WK, bool BF16>
static void launch_dw(const float* dY, int64_t ldy, const float* X, int64_t ldx, int64_t N, int Kout, int D, float* out,
                      hipStream_t s) {
  constexpr int WD = 4 / WK;
  const int blocks_k = (Kout + 32 * MK * WK - 1) / (32 * MK * WK);
  const int blocks_d = (D + 32 * MD * WD - 1) / (32 * MD * WD);
  const int blocks = blocks_k * blocks_d;
  // About 1024 workgroups in all, whole batches per slab, and slabs no shorter than their results are worth.  The bf16
  // forms walk a row in 0.068 us and 100,000 results a microsecond meet in memory; 64 slabs at most are made shorter than 512
  // rows for that, since every slab is one more rounding of the growing sum.  (70,001 rows 20 x 100 in 487 slabs: the worst of
  // 2000 results off by 40 - 71 times 2^-24 of their rms, 28 - 40 in 137 slabs of 512.)  512 rows throughout -> this: 16,384
  // rows 128 x 128 37.4 -> 24.5 us, worst 28.7 -> 24.7 such units on average, 64 x 64 23.8 -> 15.3, 256 x 40 36.7 -> 25.8;
  // 24,000 rows 128 x 128 38.1 -> 32.0, 30.3 -> 27.6 units; the same from 32,768 rows on.
  int64_t slabs = (1024 + blocks - 1) / blocks;
  int64_t rows = (N + slabs - 1) / slabs;
  int64_t least = BF16 ? dw_slab_rows(N, Kout, D, 0.068, 1e-5, 128) : 512;
  if (least < 512 && least * 64 < N) least = N < 512 * 64 ? (N + 63) / 64 : 512;
  if (rows < least) rows = least;
  rows = (rows + 15) / 16 * 16;  // whole batches (8 rows) resp. steps (16 rows)
  slabs = (N + rows - 1) / rows;
  const dim3 grid(static_cast<unsigned>((slabs + kDwXcds - 1) / kDwXcds * kDwXcds * blocks));
  constexpr size_t lds = sizeof(u32x4) * 2 * (MK * WK + MD * WD) * 3 * kWave;
  // Which form, measured as shared / own over 16,384 to 1,000,000 rows (us at 100,000 in brackets):
  //   more than 64 x more than 64    0.72 - 0.98 (157 / 196 at 256 x 300), 1.03 at 16,384 x 100 x 100: shared
  //   33 - 64 x more than 128        1.03 - 1.11 at 16,384 rows, 0.86 - 1.04 at 100,000 (72 / 82 at 64 x 300), 0.79 - 0.89
  //                                  at 1,000,000: shared from 65,536 rows on
  //   up to 32 x more than 128       1.14 - 1.38, 0.97 - 1.31 (95 / 77 at 32 x 602), 0.83 - 0.96: shared from 500,000 on
  //   fewer columns of either        1.02 - 1.5 nearly everywhere (31 / 23 at 8 x 32): own
  constexpr bool can_share = MD == 2 && WK <= 2;
  const bool shared = can_share && (WK == 2 || N >= (MK == 2 ? 65536 : 500000));
  if constexpr (!BF16) {
    hipLaunchKernelGGL((linear_dw_kernel<MK, MD, WK, false>), grid, dim3(kBlock), 0, s, dY, ldy, X, ldx, N, Kout, D, rows, blocks_d, blocks, slabs, out);
  } else {
    if constexpr (can_share) {
      if (shared) {
        hipLaunchKernelGGL((linear_dw_shared_kernel<MK, MD, WK>), grid, dim3(kBlock), lds, s, dY, ldy, X, ldx, N, Kout, D, rows, blocks_d, blocks, slabs, out);
        return;
      }
    }
    hipLaunchKernelGGL((linear_dw_bf16_kernel<MK, MD, WK>), grid, dim3(kBlock), 0, s, dY, ldy, X, ldx, N, Kout, D, rows, blocks_d, blocks, slabs, out);
  }
}

template <bool BF16>
static int linear_dw_any(const float* dY, int64_t ldy, const float* X, int64_t ldx, int64_t N, int64_t Kout, int64_t D,
                         float* out, hipStream_t s) {
  if (N < 0 || Kout < 0 || D < 0 || Kout > 65536 || D > 65536 || N > (int64_t{1} << 40)) return EXACT_E_SHAPE;
  if (ldy < Kout || ldx < D) return EXACT_E_SHAPE;
  if (Kout == 0 || D == 0) return EXACT_OK;
  if (!out || (N > 0 && (!dY || !X))) return EXACT_E_NULL;
  const int64_t total = Kout * D;
  hipLaunchKernelGGL(dw_zero_kernel, dim3(static_cast<unsigned>((total + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, out, total);
  if (N > 0) {
    const int K = static_cast<int>(Kout), Dd = static_cast<int>(D);
    // wavefront block: up to 64 x 64 of dW (wider blocks need more accumulator registers than two wavefronts
    // per SIMD leave); the four wavefronts side by side along the longer extent when the other fits one wavefront
    if (K <= 32) {
      if (Dd <= 128) launch_dw<1, 1, 1, BF16>(dY, ldy, X, ldx, N, K, Dd, out, s);
      else launch_dw<1, 2, 1, BF16>(dY, ldy, X, ldx, N, K, Dd, out, s);
    } else if (K <= 64) {
      if (Dd <= 128) launch_dw<2, 1, 1, BF16>(dY, ldy, X, ldx, N, K, Dd, out, s);
      else launch_dw<2, 2, 1, BF16>(dY, ldy, X, ldx, N, K, Dd, out, s);
    } else {
      if (Dd <= 32) launch_dw<2, 1, 4, BF16>(dY, ldy, X, ldx, N, K, Dd, out, s);
      else if (Dd <= 64) launch_dw<2, 2, 4, BF16>(dY, ldy, X, ldx, N, K, Dd, out, s);
      else launch_dw<2, 2, 2, BF16>(dY, ldy, X, ldx, N, K, Dd, out, s);
    }
  }
  return launch_status();
}

}  // namespace exact

using namespace exact;

extern "C" {

int exact_linear_dw_f32(const float* dY, int64_t ldy, const float* X, int64_t ldx, int64_t N, int64_t Kout, int64_t D,
                        float* out, void* stream) {
  return linear_dw_any<false>(dY, ldy, X, ldx, N, Kout, D, out, static_cast<hipStream_t>(stream));
}

int exact_linear_dw_bf16_f32(const float* dY, int64_t ldy, const float* X, int64_t ldx, int64_t N, int64_t Kout, int64_t D,
                             float* out, void* stream) {
  return linear_dw_any<true>(dY, ldy, X, ldx, N, Kout, D, out, static_cast<hipStream_t>(stream));
}

static bool dw_short_shape_ok(int64_t N, int64_t Kout, int64_t D) { return N >= 0 && Kout >= 0 && D >= 0 && Kout <= 65536 && D <= 65536 && N <= (int64_t{1} << 40); }

int64_t exact_linear_dw_short_work_nbytes(int64_t N, int64_t Kout, int64_t D) {
  if (!dw_short_shape_ok(N, Kout, D) || N == 0 || Kout == 0 || D == 0) return 0;
  return plan_dw_short(N, static_cast<int>(Kout), static_cast<int>(D)).slabs * Kout * D * static_cast<int64_t>(sizeof(float));
}

int exact_linear_dw_short_f32(const float* dY, int64_t ldy, const float* X, int64_t ldx, int64_t N, int64_t Kout, int64_t D, float* out,
                              void* work, void* stream) {
  if (!dw_short_shape_ok(N, Kout, D) || ldy < Kout || ldx < D) return EXACT_E_SHAPE;
  if (Kout == 0 || D == 0) return EXACT_OK;
  if (!out || (N > 0 && (!dY || !X || !work))) return EXACT_E_NULL;
  const int K = static_cast<int>(Kout), Dd = static_cast<int>(D);
  const int64_t total = Kout * D;
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* partial = static_cast<float*>(work);
  int64_t slabs = 0;  // an empty batch: zeros
  if (N > 0) {
    const DwOrderedPlan p = plan_dw_short(N, K, Dd);
    slabs = p.slabs;
    if (p.wk == 1) {
      if (p.mk == 1 && p.md == 1) launch_dw_short<1, 1, 1>(p, dY, ldy, X, ldx, N, K, Dd, partial, s);
      else if (p.mk == 1) launch_dw_short<1, 2, 1>(p, dY, ldy, X, ldx, N, K, Dd, partial, s);
      else if (p.md == 1) launch_dw_short<2, 1, 1>(p, dY, ldy, X, ldx, N, K, Dd, partial, s);
      else launch_dw_short<2, 2, 1>(p, dY, ldy, X, ldx, N, K, Dd, partial, s);
    } else if (p.wk == 4) {
      if (p.md == 1) launch_dw_short<2, 1, 4>(p, dY, ldy, X, ldx, N, K, Dd, partial, s);
      else launch_dw_short<2, 2, 4>(p, dY, ldy, X, ldx, N, K, Dd, partial, s);
    } else {
      launch_dw_short<2, 2, 2>(p, dY, ldy, X, ldx, N, K, Dd, partial, s);
    }
  }
  hipLaunchKernelGGL((dw_finish_kernel<float>), dim3(static_cast<unsigned>((total + 31) / 32)), dim3(kBlock), 0, s, partial, total, slabs, out);
  return launch_status();
}

int64_t exact_linear_dw_f16_work_nbytes(int64_t N, int64_t Kout, int64_t D) {
  if (N < 0 || Kout < 0 || D < 0 || Kout > 65536 || D > 65536 || N > (int64_t{1} << 40)) return 0;
  if (N == 0 || Kout == 0 || D == 0) return 0;
  return plan_dw_half(N, static_cast<int>(Kout), static_cast<int>(D)).slabs * Kout * D * static_cast<int64_t>(sizeof(float));
}

int exact_linear_dw_ordered_f16(const uint16_t* dY, int64_t ldy, const uint16_t* X, int64_t ldx, int64_t N, int64_t Kout, int64_t D,
                                uint16_t* out, void* work, void* stream) {
  if (N < 0 || Kout < 0 || D < 0 || Kout > 65536 || D > 65536 || N > (int64_t{1} << 40)) return EXACT_E_SHAPE;
  if (ldy < Kout || ldx < D) return EXACT_E_SHAPE;
  if (Kout == 0 || D == 0) return EXACT_OK;
  if (!out || (N > 0 && (!dY || !X || !work))) return EXACT_E_NULL;
  const int K = static_cast<int>(Kout), Dd = static_cast<int>(D);
  const int64_t total = Kout * D;
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* partial = static_cast<float*>(work);
  const half_t* y = reinterpret_cast<const half_t*>(dY);
  const half_t* x = reinterpret_cast<const half_t*>(X);
  int64_t slabs = 0;  // an empty batch: zeros
  if (N > 0) {
    const DwOrderedPlan p = plan_dw_half(N, K, Dd);
    slabs = p.slabs;
    if (p.wk == 1) {
      if (p.mk == 1 && p.md == 1) launch_dw_half<1, 1, 1>(p, y, ldy, x, ldx, N, K, Dd, partial, s);
      else if (p.mk == 1) launch_dw_half<1, 2, 1>(p, y, ldy, x, ldx, N, K, Dd, partial, s);
      else if (p.md == 1) launch_dw_half<2, 1, 1>(p, y, ldy, x, ldx, N, K, Dd, partial, s);
      else launch_dw_half<2, 2, 1>(p, y, ldy, x, ldx, N, K, Dd, partial, s);
    } else if (p.wk == 4) {
      if (p.md == 1) launch_dw_half<2, 1, 4>(p, y, ldy, x, ldx, N, K, Dd, partial, s);
      else launch_dw_half<2, 2, 4>(p, y, ldy, x, ldx, N, K, Dd, partial, s);
    } else {
      launch_dw_half<2, 2, 2>(p, y, ldy, x, ldx, N, K, Dd, partial, s);
    }
  }
  hipLaunchKernelGGL((dw_finish_kernel<half_t>), dim3(static_cast<unsigned>((total + 31) / 32)), dim3(kBlock), 0, s, partial, total, slabs,
                     reinterpret_cast<half_t*>(out));
  return launch_status();
}

}  // extern "C"
