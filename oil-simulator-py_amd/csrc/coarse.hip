// Coarsest-level direct solve of the V-cycle (classical_amg.py:1045-1069):
// the level matrix is made dense, DOF 0 is optionally pinned (row/column 0 zeroed,
// a_00 = 1, b_0 = 0), and the system is solved exactly. The pin exists for singular
// (pure Neumann) matrices; on a nonsingular but nearly singular operator it removes
// the near-nullspace correction, so the pin decision is a device flag computed from
// the level's row sums (launch_pin_decide). The inverse is formed once per hierarchy
// update, on the matrix cores (dense_mfma.hip) or, for operators that are not SPD, by
// the Gauss-Jordan elimination with partial pivoting here, so each V-cycle visit is a
// single dense matrix-vector product.
#include "amg_kernels.h"

namespace impes {

namespace {

// One workgroup, 8 lanes per row: pin = mode==1 || (mode==2 && no row has
// |row sum| > 1e-8 |a_ii|). Also clears the inverse's failure flag.
constexpr int kPinThreads = 1024;
constexpr int kPinLanes = 8;
__global__ __launch_bounds__(kPinThreads) void k_pin_decide(int n, const int* __restrict__ rp,
                                                            const int* __restrict__ ci, const double* __restrict__ v,
                                                            int mode, int* __restrict__ pin, int* __restrict__ bad) {
  const int g = threadIdx.x % kPinLanes;
  int regular = 0;
  for (int base = 0; base < n; base += kPinThreads / kPinLanes) {
    const int r = base + (int)threadIdx.x / kPinLanes;
    double rs = 0.0, d = 0.0;
    if (r < n) {
      for (int e = rp[r] + g; e < rp[r + 1]; e += kPinLanes) {
        rs += v[e];
        if (ci[e] == r) d += v[e];
      }
    }
    rs = group_sum<kPinLanes>(rs);
    d = group_sum<kPinLanes>(d);
    if (r < n && g == 0 && fabs(rs) > 1e-8 * fabs(d)) regular = 1;
  }
  regular = __syncthreads_or(regular);
  if (threadIdx.x == 0) {
    *pin = (mode == 1) ? 1 : (mode == 2 ? !regular : 0);
    *bad = 0;
  }
}

__global__ void k_pin_rhs(const int* __restrict__ pin, double* __restrict__ b) {
  if (*pin) b[0] = 0.0;
}
__global__ void k_pin_rhs32(const int* __restrict__ pin, float* __restrict__ b) {
  if (*pin) b[0] = 0.f;
}

// Single workgroup Gauss-Jordan with partial pivoting on the n x 2n matrix
// [A_pinned | I] (n <= 512), formed in `aug`; the inverse goes to M (row stride
// n_pad), its transpose behind it. Runs only when the unpivoted elimination on the matrix cores met an
// operator that is not SPD (*bad); else one load and out.
__global__ __launch_bounds__(1024) void k_gauss_jordan(int n, int n_pad, const int* __restrict__ rp,
                                                       const int* __restrict__ ci, const double* __restrict__ v,
                                                       const int* __restrict__ pin_flag, const int* __restrict__ bad,
                                                       double* __restrict__ aug, double* __restrict__ M) {
  if (!*bad) return;
  __shared__ double fcol[512];
  __shared__ double red_v[1024 / kWave];
  __shared__ int red_i[1024 / kWave];
  __shared__ int piv_row;
  const long long w = 2LL * n;
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  const int pin = *pin_flag;
  for (long long t = threadIdx.x; t < n * w; t += blockDim.x) aug[t] = 0.0;
  __syncthreads();
  for (int r = threadIdx.x; r < n; r += blockDim.x) {  // a thread owns whole rows: repeated columns add in order
    aug[r * w + n + r] = 1.0;
    if (pin && r == 0) {
      aug[0] = 1.0;
      continue;
    }
    for (int e = rp[r]; e < rp[r + 1]; ++e)
      if (!(pin && ci[e] == 0)) aug[r * w + ci[e]] += v[e];
  }
  __syncthreads();
  for (int k = 0; k < n; ++k) {
    // pivot search over rows k..n-1 of column k
    double best = -1.0;
    int bi = k;
    for (int r = k + threadIdx.x; r < n; r += blockDim.x) {
      const double a = fabs(aug[(long long)r * w + k]);
      if (a > best) { best = a; bi = r; }
    }
    for (int off = kWave / 2; off > 0; off >>= 1) {
      const double ob = __shfl_xor(best, off, kWave);
      const int oi = __shfl_xor(bi, off, kWave);
      if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
    }
    if (lane == 0) { red_v[wid] = best; red_i[wid] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
      double b = -1.0;
      int i = k;
      for (int q = 0; q < (int)(blockDim.x / kWave); ++q)
        if (red_v[q] > b || (red_v[q] == b && red_i[q] < i)) { b = red_v[q]; i = red_i[q]; }
      piv_row = i;
    }
    __syncthreads();
    const int p = piv_row;
    if (p != k) {
      for (long long c = threadIdx.x; c < w; c += blockDim.x) {
        const double t = aug[(long long)k * w + c];
        aug[(long long)k * w + c] = aug[(long long)p * w + c];
        aug[(long long)p * w + c] = t;
      }
    }
    __syncthreads();
    double piv = aug[(long long)k * w + k];
    if (fabs(piv) < 1e-300) piv = 1e-300;  // singular pivot: keep the elimination finite
    const double inv = 1.0 / piv;
    __syncthreads();
    for (long long c = k + threadIdx.x; c < w; c += blockDim.x) aug[(long long)k * w + c] *= inv;
    for (int r = threadIdx.x; r < n; r += blockDim.x) fcol[r] = (r == k) ? 0.0 : aug[(long long)r * w + k];
    __syncthreads();
    const long long span = w - k;
    for (long long t = threadIdx.x; t < (long long)n * span; t += blockDim.x) {
      const int r = (int)(t / span);
      const long long c = k + t % span;
      const double f = fcol[r];
      if (f != 0.0) aug[(long long)r * w + c] -= f * aug[(long long)k * w + c];
    }
    __syncthreads();
  }
  double* MT = M + (long long)n_pad * n_pad;
  for (long long t = threadIdx.x; t < (long long)n * n; t += blockDim.x) {
    const double a = aug[(t / n) * w + n + t % n];
    M[(t / n) * n_pad + t % n] = a;
    MT[(t % n) * n_pad + t / n] = a;
  }
}

}  // namespace

void launch_pin_decide(int n, const int* rp, const int* ci, const double* v, int mode, int* pin, int* bad,
                       hipStream_t s) {
  k_pin_decide<<<1, kPinThreads, 0, s>>>(n, rp, ci, v, mode, pin, bad);
  IMPES_LAUNCH_CHECK();
}

void launch_pin_rhs_f64(const int* pin, double* b, hipStream_t s) {
  k_pin_rhs<<<1, 1, 0, s>>>(pin, b);
  IMPES_LAUNCH_CHECK();
}

void launch_pin_rhs_f32(const int* pin, float* b, hipStream_t s) {
  k_pin_rhs32<<<1, 1, 0, s>>>(pin, b);
  IMPES_LAUNCH_CHECK();
}

void launch_gauss_jordan_inverse(int n, const int* rp, const int* ci, const double* v, const int* pin, const int* bad,
                                 double* aug, double* M, hipStream_t s) {
  IMPES_REQUIRE(n >= 1 && n <= kDensePivotMax, "pivoted dense inverse supports 1 <= n <= 512");
  k_gauss_jordan<<<1, 1024, 0, s>>>(n, dense_pad(n), rp, ci, v, pin, bad, aug, M);
  IMPES_LAUNCH_CHECK();
}

}  // namespace impes
