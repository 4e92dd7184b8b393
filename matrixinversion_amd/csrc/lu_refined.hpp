// lu_refined.hpp -- inversion and one refinement step in one kernel:
//
//   X = A^-1 (the plain kernel's tile routines), then X <- X + X (I - A X)
//
// with A kept on chip, so the refined inverse moves the plain inverse's bytes
// (A read once, X written once, pivots) instead of a copy, an inversion and
// a separate refinement pass over A and X.  The reference has no refinement:
// its inverse is the FP32 LU result (parallel_pivot/luBatchedInplace.cuh:
// 84-125, stored at :194-197).
//
// Per tile (one wave; 16 lanes per matrix and 4 matrices, or quads and 16
// matrices, as in the plain kernel):
//   1. the tile arrives in registers (TileRegs) and is staged into LDS;
//   2. tile_front + tile_solve (tile_gepp) leave X = A^-1 in the tile's LDS
//      region; the form that refines a given X (kPivGiven) stages X instead;
//   3. per matrix (per 2 or 4 matrices up to n = 8 or 4), the whole wave: A_m
//      is read a second time (normally from the caches) straight into the
//      FP64 product's operand registers, D = A_m X_m is formed on the FP64
//      matrix cores (v_mfma_f64_16x16x4f64: products of FP32 values are exact
//      in FP64, the sums round in FP64), E = D - I (= -R) is rounded to FP32
//      and stays in the registers it was accumulated in, which are exactly
//      the operands of C = X_m E on the FP32 matrix cores
//      (v_mfma_f32_16x16x4f32, accumulated from zero so its roundings stay at
//      the correction's scale), and X_m - C (one rounding) replaces X_m in
//      LDS;
//   4. the tile goes to HBM with the plain kernel's coalesced tile store.
// Nothing but the tile itself lives in LDS, so the kernel keeps the plain
// kernel's occupancy.  Padding: A_m's registers hold zeros outside its n x n
// block and X is read as zero outside its block, so D and C vanish there and
// the padding leaves the n x n result unchanged.
#pragma once

#include "lu_kernel.hpp"

namespace lub {

typedef double f64x4 __attribute__((ext_vector_type(4)));

// Sizes whose first second read of A is issued before the elimination (its
// registers fit beside the elimination's); the others issue it after.
template <int N>
constexpr bool kRfEarly = N <= 24 || N == 32;

// Sizes whose next matrix's A is loaded before the current matrix's step
// (registers permitting); the others load it after.
template <int N>
constexpr bool kRfAhead = N <= 28 || N == 32;

// Sizes that fetch the workgroup's next tile into registers while the
// current tile is refined (registers permitting).
template <int N>
constexpr bool kRfNextTile = N == 32;

// Values of k per lane group in the FP64 product of n = 17..32: step t lets
// group q stand for k = T q + t, so n / 4 steps suffice.
template <int N>
constexpr int kRfSteps = (N + 3) / 4;

// A_m in the FP64 product's operand layout: lane (r = lane % 16,
// q = lane / 16) holds A_m[16 I + r][T q + t], I = 0, 1, t = 0..T-1, and zero
// outside the n x n block.
template <int N>
struct RefinedA {
  float v[2][kRfSteps<N>];
};

// Loads A_m (matrix at `a`) with ordinary loads: the tile's first read used
// them too, so this second read is normally served from the caches.  `vec`:
// the batch is 16-byte aligned (n = 32 then reads 16-byte chunks; other n
// read the T consecutive floats of a row at their own alignment).
template <int N>
__device__ __forceinline__ void refined_load_a(const float* __restrict__ a, RefinedA<N>& r, bool vec, int lane) {
  constexpr int T = kRfSteps<N>;
  const int r16 = lane & 15, q = lane >> 4;
#pragma unroll
  for (int I = 0; I < 2; ++I) {
    const int i = 16 * I + r16;
    const float* const row = a + i * N + T * q;
    if (N == 32 && vec) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4 c = *reinterpret_cast<const f32x4*>(row + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) r.v[I][4 * h + e] = c[e];
      }
    } else {
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const bool in = (N == 32 || I == 0 || i < N) && (N % 4 == 0 || T * q + t < N);
        r.v[I][t] = in ? row[t] : 0.0f;
      }
    }
  }
}

// X_m[i][j] (i, j < 32) from the tile's LDS region, zero outside the n x n
// block.  No branch: the read goes to an address inside the block either way
// and a select supplies the zero, so consecutive reads stay in flight together.
template <int N>
__device__ __forceinline__ float x_at(const float* xm, int i, int j) {
  constexpr int LD = Geo<N, 16>::LD;
  if constexpr (N == 32) {
    return xm[i * LD + j];
  } else {
    const bool in = i < N && j < N;
    const float v = xm[(in ? i : 0) * LD + (in ? j : 0)];
    return in ? v : 0.0f;
  }
}

// One refinement step of matrix m: `am` holds A_m (refined_load_a), xm is
// X_m in the tile's LDS region (row stride Geo::LD), where the refined X_m
// replaces it (every read of X_m precedes the first write).
template <int N>
__device__ __forceinline__ void refined_step(const RefinedA<N>& am, float* xm, int lane) {
  constexpr int LD = Geo<N, 16>::LD;
  const int r16 = lane & 15, q = lane >> 4;
  // D = A_m X_m on the FP64 matrix cores, four 16 x 16 blocks (I, J).  In
  // v_mfma_f64_16x16x4f64 operand lane l holds A[l % 16][kk] and X[kk][l % 16]
  // with kk = l / 16; step t lets lane group q stand for k = T q + t, so A_m's
  // registers are used as loaded.  Accumulator element v of lane l is
  // D[16 I + l / 16 + 4 v][16 J + l % 16].
  f64x4 acc[2][2];
#pragma unroll
  for (int I = 0; I < 2; ++I)
#pragma unroll
    for (int J = 0; J < 2; ++J) acc[I][J] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int t = 0; t < kRfSteps<N>; ++t) {
    const int k = kRfSteps<N> * q + t;
    double xv[2];
#pragma unroll
    for (int J = 0; J < 2; ++J) {
      xv[J] = static_cast<double>(x_at<N>(xm, k, 16 * J + r16));
    }
#pragma unroll
    for (int I = 0; I < 2; ++I) {
      const double av = static_cast<double>(am.v[I][t]);
#pragma unroll
      for (int J = 0; J < 2; ++J) acc[I][J] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, xv[J], acc[I][J], 0, 0, 0);
    }
  }
  // E = D - I rounded to FP32 (E = -R; rounding to nearest is symmetric, so
  // X - X E below equals X + X R bit for bit): ee[I][J][v] = E[16 I + q + 4 v][16 J + r16].
  // Only the diagonal blocks hold ones to subtract (in FP64, before rounding);
  // on the padding diagonal E is -1, which meets only zero columns of X.
  float ee[2][2][4];
#pragma unroll
  for (int I = 0; I < 2; ++I)
#pragma unroll
    for (int J = 0; J < 2; ++J)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (I == J) {
          ee[I][J][v] = static_cast<float>(acc[I][J][v] - (q + 4 * v == r16 ? 1.0 : 0.0));
        } else {
          ee[I][J][v] = static_cast<float>(acc[I][J][v]);
        }
      }
  // C = X_m E on the FP32 matrix cores, four 16 x 16 blocks (Io, J).  In
  // v_mfma_f32_16x16x4f32 operand lane l holds X[l % 16][kk] and E[kk][l % 16]
  // with kk = l / 16; step (I, v) lets lane group q stand for
  // k = 16 I + q + 4 v, the row of E that lane already holds.  Accumulator
  // element v of lane l is C[4 (l / 16) + v][l % 16].
  f32x4 c[2][2];
#pragma unroll
  for (int Io = 0; Io < 2; ++Io)
#pragma unroll
    for (int J = 0; J < 2; ++J) c[Io][J] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int I = 0; I < 2; ++I)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (16 * I + 4 * v >= N) continue;  // rows of E past n
      const int k = 16 * I + q + 4 * v;
      float xa[2];
#pragma unroll
      for (int Io = 0; Io < 2; ++Io) xa[Io] = x_at<N>(xm, 16 * Io + r16, k);
#pragma unroll
      for (int Io = 0; Io < 2; ++Io)
#pragma unroll
        for (int J = 0; J < 2; ++J) c[Io][J] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[Io], ee[I][J][v], c[Io][J], 0, 0, 0);
    }
#pragma unroll
  for (int Io = 0; Io < 2; ++Io)
#pragma unroll
    for (int J = 0; J < 2; ++J)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 16 * Io + 4 * q + v, j = 16 * J + r16;
        if (N == 32 || (i < N && j < N)) xm[i * LD + j] -= c[Io][J][v];
      }
}

// ---- n <= 16: one 16 x 16 product holds P = 16 / S matrices, S = 4, 8 or 16 --
//
// The A operand stacks P matrices' rows (lane (r = lane % 16, q = lane / 16)
// holds row r % S of matrix r / S) and the B operand their columns, so D's
// diagonal S x S blocks are the P products and the rest is never used.  Only
// values of k below 4 T exist: T = ceil(n / 4) matrix instructions.
template <int N>
struct RefinedSmall {
  static constexpr int S = N <= 4 ? 4 : (N <= 8 ? 8 : 16);
  static constexpr int P = 16 / S;         // matrices per product
  static constexpr int T = (N + 3) / 4;    // steps; step t lets lane group q stand for k = T q + t
};

// A operand of matrices m .. m + P - 1 of the tile at `a` (the last `valid`
// matrix stands in for those past the batch; their results are not stored).
template <int N>
__device__ __forceinline__ void refined_small_load(const float* __restrict__ a, int m, int valid,
                                                   float (&v)[RefinedSmall<N>::T], bool vec, int lane) {
  using Z = RefinedSmall<N>;
  const int r = (lane & 15) % Z::S, mm = min(m + (lane & 15) / Z::S, valid - 1), k0 = Z::T * (lane >> 4);
  const float* const row = a + mm * (N * N) + r * N + k0;
  if (N == 16 && vec) {
    const f32x4 c = *reinterpret_cast<const f32x4*>(row);
#pragma unroll
    for (int t = 0; t < Z::T; ++t) v[t] = c[t];
  } else {
#pragma unroll
    for (int t = 0; t < Z::T; ++t) v[t] = (r < N && (N % 4 == 0 || k0 + t < N)) ? row[t] : 0.0f;
  }
}

// One refinement step of the product whose first X starts at xm (LDS, matrix
// stride MS, row stride LD).  Every read of X precedes the first write.
template <int N, int L>
__device__ __forceinline__ void refined_small_step(const float (&av)[RefinedSmall<N>::T], float* xm, int lane) {
  using G = Geo<N, L>;
  using Z = RefinedSmall<N>;
  const int r = lane & 15, q = lane >> 4, rs = r % Z::S;
  float* const mine = xm + (r / Z::S) * G::MS;  // matrix of this lane's row and column
  auto at = [&](int i, int j) {  // X[i][j], zero outside the block; see x_at
    const bool in = i < N && j < N;
    const float v = mine[(in ? i : 0) * G::LD + (in ? j : 0)];
    return in ? v : 0.0f;
  };
  f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int t = 0; t < Z::T; ++t)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(av[t]), static_cast<double>(at(Z::T * q + t, rs)),
                                               acc, 0, 0, 0);
  // acc[v] of this lane is D[q + 4 v][r]; of the lane's own block it has the
  // rows q + 4 w, w = 0 .. S / 4 - 1 (those below n within the first T):
  // E = D - I there, rounded to FP32.
  float ee[Z::T];
#pragma unroll
  for (int w = 0; w < Z::T; ++w) {
    double d = acc[w];
#pragma unroll
    for (int p = 1; p < Z::P; ++p) d = (r / Z::S == p) ? acc[p * (Z::S / 4) + w] : d;
    ee[w] = static_cast<float>(d - (q + 4 * w == rs ? 1.0 : 0.0));
  }
  // C = X E: step w lets lane group q stand for k = q + 4 w of the block.
  f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int w = 0; w < Z::T; ++w) c = __builtin_amdgcn_mfma_f32_16x16x4f32(at(rs, q + 4 * w), ee[w], c, 0, 0, 0);
  // c[v] is C[4 q + v][r]: row (4 q + v) % S of matrix (4 q + v) / S
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int i = 4 * q + v;
    if (i / Z::S == r / Z::S && i % Z::S < N && rs < N) mine[(i % Z::S) * G::LD + rs] -= c[v];
  }
}

// The step for a whole tile in LDS, A's tile at `a`: the next product's A is
// loaded before the current one's step.  (Two or four products interleaved
// were slower, 142 and 159 us against 131 for 300k n = 12: fewer waves fit.)
template <int N, int L>
__device__ __forceinline__ void refined_small_tile(const float* __restrict__ a, float* lds, int valid, bool vec,
                                                   int lane) {
  using G = Geo<N, L>;
  using Z = RefinedSmall<N>;
  float av[Z::T];
  refined_small_load<N>(a, 0, valid, av, vec, lane);
#pragma unroll
  for (int m = 0; m < G::MPW; m += Z::P) {
    float an[Z::T];
    if (m + Z::P < G::MPW) refined_small_load<N>(a, m + Z::P, valid, an, vec, lane);
    refined_small_step<N, L>(av, lds + m * G::MS, lane);
#pragma unroll
    for (int t = 0; t < Z::T; ++t) av[t] = an[t];
  }
}

// The "rule" of the kernel that refines the X it is given instead of inverting A.
constexpr int kPivGiven = -1;

// Out-of-place inverse + one refinement step of `batch` n x n matrices: A is
// only read, X receives the refined inverse, piv (nullable) the pivot vectors
// (kPivGiven: X is refined in place).  `vec`: bit 0, A is 16-byte aligned;
// bit 1, X is.  One workgroup (one wave) per tile, striding when the grid is
// capped; a striding workgroup at n = 32 fetches its next tile into registers
// during the current tile's refinement.  A_m is read a second time for its
// refinement (A_{m+1}'s loads are issued before A_m's refinement starts where
// registers allow); keeping the whole tile in registers through the
// factorisation instead exceeds 256 VGPRs and spills.
// Against copy + inversion + a refinement pass with every matrix padded to
// 32 x 32 (300k matrices): n = 12 0.121 ms instead of 0.71; n = 16 0.19, n = 8
// 0.047.  Bound at n = 12 by the matrix cores' 288 cycles per matrix (35 us)
// on top of the plain inversion's 54 us, and the chain of each step.
template <int N, int L, int PIV>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(2))) void lu_refined_kernel(
    const float* __restrict__ A, float* __restrict__ X, int* __restrict__ piv, int64_t batch, int64_t ntiles,
    int vec) {
  using G = Geo<N, L>;
  constexpr int NN = N * N;
  constexpr bool small = N <= 16;
  __shared__ __attribute__((aligned(16))) float lds[G::LDS_FLOATS];
  const int lane = threadIdx.x;
  const int l = lane % L, g = lane / L;
  const int64_t stride = gridDim.x;
  const float* const src = PIV == kPivGiven ? X : A;  // what is staged
  const bool avec = (vec & 1) != 0;
  auto full = [&](int64_t t) { return (vec & (PIV == kPivGiven ? 2 : 1)) != 0 && (t + 1) * G::MPW <= batch; };
  TileRegs<N, L> next;
  int64_t t = blockIdx.x;
  bool have = t < ntiles && full(t);
  if (have) tile_fetch<N, L, PIV == kPivGiven>(src + t * G::MPW * NN, next, lane);
  for (; t < ntiles; t += stride) {
    const int64_t m0 = t * G::MPW;
    const int64_t left = batch - m0;
    const int valid = left < G::MPW ? static_cast<int>(left) : G::MPW;
    const float* const a = A + m0 * NN;
    RefinedA<N> am;
    if constexpr (PIV == kPivGiven && !small) refined_load_a<N>(a, am, avec, lane);
    if (!have) tile_fetch_part<N, L, PIV == kPivGiven>(src + m0 * NN, next, valid * NN, lane);
    tile_stage<N, L>(next, lds, lane);
    if (valid < G::MPW) tile_identity<N, L>(lds, valid, lane);
    wave_sync();
    if constexpr (PIV == kPivGepp) {
      int prm[G::R];
      tile_gepp<N, L>(prm, lds, lane, nullptr);
      if (piv != nullptr && g < valid) {
#pragma unroll
        for (int h = 0; h < G::R; ++h)
          if (l + L * h < N) piv[(m0 + g) * N + l + L * h] = prm[h];
      }
    } else if constexpr (PIV != kPivGiven) {
      int prm[G::R];
      float w[G::R][N];
      tile_front<N, L, PIV>(w, prm, lds, lane);
      // A_0's second read is in flight during the elimination
      if constexpr (!small && kRfEarly<N>) refined_load_a<N>(a, am, avec, lane);
      tile_solve<N, L>(w, prm, lds, lane);
      if (piv != nullptr && g < valid) {
#pragma unroll
        for (int h = 0; h < G::R; ++h)
          if (l + L * h < N) piv[(m0 + g) * N + l + L * h] = prm[h];
      }
    }
    // the next tile's HBM reads overlap this tile's refinement
    const int64_t tn = t + stride;
    have = tn < ntiles && full(tn);
    if constexpr (kRfNextTile<N>) {
      if (have) tile_fetch<N, L, PIV == kPivGiven>(src + tn * G::MPW * NN, next, lane);
    }
    if constexpr (small) {
      refined_small_tile<N, L>(a, lds, valid, avec, lane);
    } else {
      // Opaque after partial pivoting: keeps the refinement's loads and
      // lane-derived addresses from being live through it (they would spill).
      int ln = lane;
      if constexpr (PIV == kPivGepp) asm volatile("" : "+v"(ln));
      if constexpr (PIV == kPivGepp || (PIV != kPivGiven && !kRfEarly<N>)) refined_load_a<N>(a, am, avec, ln);
#pragma unroll
      for (int m = 0; m < G::MPW; ++m) {
        if (m < valid) {
          if constexpr (kRfAhead<N>) {
            RefinedA<N> an;
            if (m + 1 < valid) refined_load_a<N>(a + (m + 1) * NN, an, avec, ln);
            refined_step<N>(am, lds + m * G::MS, ln);
            am = an;
          } else {
            refined_step<N>(am, lds + m * G::MS, ln);
            if (m + 1 < valid) refined_load_a<N>(a + (m + 1) * NN, am, avec, ln);
          }
        }
      }
    }
    wave_sync();
    tile_store<N, L>(X + m0 * NN, lds, valid, (vec & 2) != 0, lane);
    wave_sync();  // the tile's region is rewritten by the next tile
    if constexpr (!kRfNextTile<N>) {
      if (have) tile_fetch<N, L, PIV == kPivGiven>(src + tn * G::MPW * NN, next, lane);
    }
  }
}

}  // namespace lub
