// Storage of one FGMRES(m) cycle's small data (Hessenberg columns, rotations, scalars)
// in one device array, and the Givens rotation; shared by the solver's translation
// units.
#pragma once

#include "common.h"

namespace impes {

struct FgmresLayout {
  int m;
  __host__ __device__ int H(int i, int j) const { return i + j * (m + 1); }
  __host__ __device__ int g() const { return (m + 1) * m; }
  __host__ __device__ int cs() const { return g() + m + 1; }
  __host__ __device__ int sn() const { return cs() + m; }
  __host__ __device__ int h() const { return sn() + m; }
  __host__ __device__ int h2() const { return h() + m + 1; }
  __host__ __device__ int y() const { return h2() + m + 1; }
  __host__ __device__ int sc() const { return y() + m; }  // 8 scalars
  // lagged orthogonalisation: provisional column (m+1) and the update's 2 scalars;
  // its coefficients a and c reuse h() and h2()
  __host__ __device__ int hp() const { return sc() + 8; }
  __host__ __device__ int lag() const { return hp() + m + 1; }
  __host__ __device__ int size() const { return lag() + 2; }
};

constexpr int kMaxFusedGs = 32;  // largest basis of the fused Gram-Schmidt kernels

// c, s = the Givens rotation that zeroes b under a
__device__ __forceinline__ void givens(double a, double b, double& c, double& s) {
  if (b == 0.0) { c = 1.0; s = 0.0; }
  else if (fabs(b) > fabs(a)) { const double t = a / b; s = 1.0 / sqrt(1.0 + t * t); c = s * t; }
  else { const double t = b / a; c = 1.0 / sqrt(1.0 + t * t); s = c * t; }
}

// Sums of NV values (a power of two, NV P <= 64) over the wave's lanes of equal
// lane % P: each step sends half of a lane's values to its partner, so NV values take
// NV - 1 + log2(64 / (NV P)) shuffles instead of NV log2(64 / P). Returns the sum of
// value fold_index<NV>(lane).
template <int M, int OFF, int P, int NV>
__device__ __forceinline__ void fold_steps(double (&v)[NV], int lane) {
  if constexpr (M >= 1) {
    const bool hi = (lane & OFF) != 0;
#pragma unroll
    for (int q = 0; q < M; ++q) {
      const double send = hi ? v[q] : v[q + M], keep = hi ? v[q + M] : v[q];
      v[q] = keep + __shfl_xor(send, OFF, kWave);
    }
    fold_steps<M / 2, OFF / 2, P>(v, lane);
  } else if constexpr (OFF >= P) {
    v[0] += __shfl_xor(v[0], OFF, kWave);
    fold_steps<0, OFF / 2, P>(v, lane);
  }
}
template <int NV, int P = 1>
__device__ __forceinline__ double wave_fold(double (&v)[NV]) {
  static_assert(NV * P <= kWave, "one value per lane at the end");
  fold_steps<NV / 2, kWave / 2, P>(v, threadIdx.x & (kWave - 1));
  return v[0];
}
template <int NV>
__device__ __forceinline__ int fold_index(int lane) {
  return lane / (kWave / NV);
}

}  // namespace impes
