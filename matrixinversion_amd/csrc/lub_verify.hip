// lub_verify.hip -- device-side inversion check (the C ABI's lu_batched_residual).
//
// The reference checks its results on the host: verifyInv (parallel_pivot/
// verify.hpp:50-103) forms every entry of A*X in FP32 and counts a matrix as
// correct when all n*n entries are within 1e-3 of the identity -- an
// O(batch*n^3) single-threaded loop, the slowest step of each reference run.
// Here a matrix belongs to L lanes of a wave (a 16-lane DPP row, or a quad),
// as in the inversion kernel.  Lane l holds columns l, l + L, ... of X and of
// A; entry (i, j) of A X is formed in the lane that holds column j of X, in
// the reference's l order with a rounded multiply and a rounded add, and
// A[i][l] reaches it by the multiply's DPP broadcast -- two VALU instructions
// per term, no LDS.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <utility>

#include "lu_kernel.hpp"
#include "lubatch.h"

namespace {


// A and X of one tile (64 / L matrices) in registers.
template <int N, int L>
struct Check {
  static constexpr int R = (N + L - 1) / L;  // columns per lane
  static constexpr int MPW = 64 / L;         // matrices per wave
  float a[N][R], x[N][R];

  __device__ __forceinline__ void load(const float* __restrict__ A, const float* __restrict__ X, int64_t m, int l) {
    const float* am = A + m * (N * N);
    const float* xm = X + m * (N * N);
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int h = 0; h < R; ++h) {
        const int j = (N % L == 0 || h + 1 < R) ? l + L * h : min(l + L * h, N - 1);  // lanes past n repeat column n-1
        a[i][h] = __builtin_nontemporal_load(am + i * N + j);
        x[i][h] = __builtin_nontemporal_load(xm + i * N + j);
      }
  }

  // Largest |A X - I| bit pattern over the lane's columns (non-negative
  // floats order like their bit patterns; NaN counts as +inf's pattern + 1),
  // and whether all of them are below thr (false for NaN, as in the
  // reference's '<' test).
  __device__ __forceinline__ void residual(float thr, int l, uint32_t& worst, bool& ok) const {
    worst = 0;
    ok = true;
    lub::static_for<0, N>([&](auto I) {
      constexpr int i = decltype(I)::value;
      float r[R];
      lub::static_for<0, N>([&](auto T) {
        // separate multiply and add: HIP contracts a*b + c into an FMA by
        // default (also through __fmul_rn / __fadd_rn), which rounds once
        // instead of twice and flips borderline counts
#pragma clang fp contract(off)
        constexpr int t = decltype(T)::value;
        const float b = lub::dpp_f32<lub::bcast_ctrl<L, t % L>()>(a[i][t / L]);
#pragma unroll
        for (int h = 0; h < R; ++h) {
          const float p = b * x[t][h];
          r[h] = t == 0 ? p : r[h] + p;
        }
      });
#pragma unroll
      for (int h = 0; h < R; ++h) {
        const int j = l + L * h;
        const float e = fabsf(r[h] - (i == j ? 1.0f : 0.0f));
        const bool mine = N % L == 0 || h + 1 < R || j < N;
        ok = ok && (!mine || e < thr);
        const uint32_t bits = (e == e) ? __float_as_uint(e) : 0x7f800001u;
        worst = max(worst, mine ? bits : 0u);
      }
    });
  }
};

// Per 500k matrices of n = 32: 0.90 ms (4.5 TB/s) where a workgroup of 1024
// threads per matrix with A and X in LDS and two atomics per matrix took
// 12.3 ms.  Bound by VALU issue: 2 n^3 multiplies and adds (no FMA, see
// below) are 0.83 ms at 39.3 T lane-operations/s; the bytes take 0.62 ms.
template <int N, int L, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void residual_kernel(const float* __restrict__ A, const float* __restrict__ X,
                                                            int64_t batch, float thr,
                                                            unsigned long long* __restrict__ correct,
                                                            unsigned int* __restrict__ max_bits) {
  using C = Check<N, L>;
  __shared__ unsigned int part_ok[WAVES], part_max[WAVES];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int l = lane % L, g = lane / L;
  const int64_t ntiles = (batch + C::MPW - 1) / C::MPW;
  uint32_t top = 0, good = 0;  // good: matrices of this wave
  for (int64_t t = int64_t(blockIdx.x) * WAVES + wave; t < ntiles; t += int64_t(gridDim.x) * WAVES) {
    const int64_t m = t * C::MPW + g;
    const bool live = m < batch;
    C c;
    c.load(A, X, live ? m : batch - 1, l);  // groups past the batch repeat its last matrix
    uint32_t worst;
    bool ok;
    c.residual(thr, l, worst, ok);
    top = max(top, worst);
    uint64_t bad = __ballot(!ok);
#pragma unroll
    for (int s = 1; s < L; s <<= 1) bad |= bad >> s;  // lane 0 of a group: any of its lanes
    good += __popcll(__ballot(live && l == 0) & ~bad);
  }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) top = max(top, static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), s)));
  if (lane == 0) {
    part_ok[wave] = good;
    part_max[wave] = top;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned int s = 0, b = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      s += part_ok[w];
      b = max(b, part_max[w]);
    }
    if (s != 0) atomicAdd(correct, static_cast<unsigned long long>(s));
    atomicMax(max_bits, b);
  }
}

using Launch = void (*)(const float*, const float*, int64_t, float, unsigned long long*, unsigned int*, unsigned,
                        hipStream_t);

template <int N, int L, int WAVES>
void launch(const float* A, const float* X, int64_t batch, float thr, unsigned long long* correct,
            unsigned int* max_bits, unsigned max_grid, hipStream_t s) {
  const int64_t per = int64_t(WAVES) * Check<N, L>::MPW;
  const unsigned grid = static_cast<unsigned>(std::min<int64_t>((batch + per - 1) / per, max_grid));
  residual_kernel<N, L, WAVES><<<grid, WAVES * 64, 0, s>>>(A, X, batch, thr, correct, max_bits);
}

// Quads up to n = 4 (19 us against 24 for 500k n = 4), where a row of 16 lanes
// would hold 12 idle ones; above, 16-lane rows: their loads cover up to 64
// consecutive bytes of a matrix row instead of 16 (500k n = 8: 77 us against
// 123, n = 12: 195 against 304).
template <int N>
constexpr int lanes() { return N <= 4 ? 4 : 16; }

template <int N>
constexpr int waves() { return N <= 16 ? 16 : 4; }

template <size_t... I>
Launch pick(int n, std::index_sequence<I...>) {
  static constexpr Launch table[] = {&launch<int(I) + 1, lanes<int(I) + 1>(), waves<int(I) + 1>()>...};
  return table[n - 1];
}

}  // namespace

extern "C" int lu_batched_residual(const float* A, const float* X, int n, int64_t batch, float thr,
                                   unsigned long long* d_correct, unsigned int* d_max_bits, void* stream) {
  if (n < 1 || n > LUB_MAX_N) return LUB_EINVAL_N;
  if (batch < 0) return LUB_EINVAL_BATCH;
  if (batch == 0) return LUB_OK;
  if (A == nullptr || X == nullptr || d_correct == nullptr || d_max_bits == nullptr) return LUB_ENULL;
  // A workgroup ends with two atomics, usually on one cache line: about 20 ns
  // for the pair, one workgroup after the other for the whole device.  So the
  // grid is bounded and its waves stride over the tiles: up to n = 16 512
  // workgroups of 16 waves (500k n = 4: 26 us, 101 with 4,096 of 4 waves),
  // above, where the registers allow 12 waves per CU, 4,096 of 4 (n = 32:
  // 0.90 ms; 0.98 with 12-wave workgroups, 0.93 with one tile per wave).
  const unsigned max_grid = n <= 16 ? 512u : 4096u;
  pick(n, std::make_index_sequence<LUB_MAX_N>())(A, X, batch, thr, d_correct, d_max_bits, max_grid,
                                                 static_cast<hipStream_t>(stream));
  return hipGetLastError() == hipSuccess ? LUB_OK : LUB_EHIP;
}
