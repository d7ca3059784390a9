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

// Sums of NV values (a power of two up to 64) over the wave's lanes: each step sends
// half of a lane's values to its partner, so NV values take NV - 1 + log2(64 / NV)
// shuffles instead of 6 NV. Returns the sum of value fold_index<NV>(lane).
template <int NV>
__device__ __forceinline__ double wave_fold(double (&v)[NV]) {
  const int lane = threadIdx.x & (kWave - 1);
  int off = kWave / 2;
#pragma unroll
  for (int m = NV / 2; m >= 1; m /= 2) {
    const bool hi = (lane & off) != 0;
#pragma unroll
    for (int q = 0; q < m; ++q) {
      const double send = hi ? v[q] : v[q + m], keep = hi ? v[q + m] : v[q];
      v[q] = keep + __shfl_xor(send, off, kWave);
    }
    off /= 2;
  }
#pragma unroll
  for (; off >= 1; off /= 2) v[0] += __shfl_xor(v[0], off, kWave);
  return v[0];
}
template <int NV>
__device__ __forceinline__ int fold_index(int lane) {
  return lane / (kWave / NV);
}

}  // namespace impes
