// FGMRES steps of small systems in one workgroup each. Up to kSmallRows rows a step's
// kernels (operator apply, two passes over the basis, two Hessenberg updates) move a
// few hundred KB and are bound by their launches: 3-12 us each on the device and
// about as much on the host. One workgroup of 1024 threads holds its rows' vectors
// in registers, so a step is the preconditioner and one launch, and so are a solve's
// start, the start and end of a cycle and the error check. The arithmetic per row is
// that of the kernels in fgmres.hip and spmv.hip; sums over rows run in another order.
// Measured per step (besides the preconditioner): 17 us at 1,200 rows against 23-28 us
// in five launches, and 21 against 26 at 3,600; a step of the 1,200-cell environment
// 931 -> 685 us (the host enqueues 53 instead of 110 launches). What bounds it: the
// chain of far loads, two workgroup folds and the serial rotations.
#include "fgmres_dev.h"
#include "fgmres_small.h"

namespace impes {

namespace {

constexpr int kT = 1024;
constexpr int kW = kT / kWave;
using Layout = FgmresLayout;

// sum over the workgroup; every thread gets it
__device__ __forceinline__ double block_total(double v, double* lds) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == 0) lds[threadIdx.x / kWave] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int q = 0; q < kW; ++q) t += lds[q];
  return t;
}
__device__ __forceinline__ double block_most(double v, double* lds) {
  v = wave_max(v);
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == 0) lds[threadIdx.x / kWave] = v;
  __syncthreads();
  double t = lds[0];
#pragma unroll
  for (int q = 1; q < kW; ++q) t = lds[q] > t ? lds[q] : t;
  return t;
}

// row i of A times x, x given by xv(q), in the term order of the row kernels
template <class F>
__device__ __forceinline__ double row_apply(const SmallOperator& A, int i, F xv) {
  double s = 0.0;
  if (A.stencil) {
    const int sy = A.st.nz, sx = A.st.ny * A.st.nz;
    const int k = i % sy, t = i / sy, j = t % A.st.ny, ix = t / A.st.ny;
    if (ix > 0) s += A.st.ox[i - sx] * xv(i - sx);
    if (j > 0) s += A.st.oy[i - sy] * xv(i - sy);
    if (k > 0) s += A.st.oz[i - 1] * xv(i - 1);
    s += A.st.d[i] * xv(i);
    if (k < A.st.nz - 1) s += A.st.oz[i] * xv(i + 1);
    if (j < A.st.ny - 1) s += A.st.oy[i] * xv(i + sy);
    if (ix < A.st.nx - 1) s += A.st.ox[i] * xv(i + sx);
  } else {
    const int e1 = A.csr.rp[i + 1];
#pragma unroll 4
    for (int e = A.csr.rp[i]; e < e1; ++e) s += A.csr.v[e] * xv(A.csr.ci[e]);
  }
  return s;
}

// r = D^-1 (b - A x) over all rows into V; its squared norm (every thread)
__device__ __forceinline__ double residual_all(const SmallOperator& A, const double* b, const double* x, double* V,
                                               double* lds) {
  double rr = 0.0;
  for (int i = threadIdx.x; i < A.n; i += kT) {
    const double r = A.dinv[i] * (b[i] - row_apply(A, i, [&](int q) { return x[q]; }));
    V[i] = r;
    rr += r * r;
  }
  return block_total(rr, lds);
}

// start of a solve: ||D^-1 b||^2 -> host[5], the scaled residual of x (zeroed first
// without a starting guess) -> V and its squared norm -> sm sc[4], host[4]
__global__ __launch_bounds__(kT) void k_small_start(SmallOperator A, Layout L, double* __restrict__ sm,
                                                    const double* b, double* x, int use_x0, double* V, double* host) {
  __shared__ double lds[kW];
  double bb = 0.0;
  for (int i = threadIdx.x; i < A.n; i += kT) {
    const double s = A.dinv[i] * b[i];
    bb += s * s;
    if (!use_x0) x[i] = 0.0;
  }
  bb = block_total(bb, lds);
  __syncthreads();
  const double rr = residual_all(A, b, x, V, lds);
  if (threadIdx.x == 0) {
    sm[L.sc() + 4] = rr;
    host[4] = rr;
    host[5] = bb;
  }
}

// start of a cycle (k_init_cycle and k_normalize_scale): v_0 = V / beta, g = beta e_1,
// the cycle's first preconditioner input S .* v_0. beta <= 0: V as it is.
template <class T>
__global__ __launch_bounds__(kT) void k_small_begin(int n, Layout L, double* __restrict__ sm, double* __restrict__ V,
                                                    const double* __restrict__ S, T* __restrict__ bout) {
  const double beta = sqrt(sm[L.sc() + 4]);
  const double nrm = (beta > 0.0) ? beta : 1.0;
  const double inv = 1.0 / nrm;
  for (int i = threadIdx.x; i < n; i += kT) {
    const double v = V[i] * inv;
    V[i] = v;
    bout[i] = (T)(S[i] * v);
  }
  for (int i = threadIdx.x; i <= L.m; i += kT) sm[L.g() + i] = (i == 0) ? beta : 0.0;
  if (threadIdx.x == 0) sm[L.sc()] = nrm;
}

// Shared pieces of a lagged step: LDS copies of the column data
struct ColData {
  double part[kW][2 * kMaxFusedGs + 2];
  double val[2 * kMaxFusedGs + 2];                                  // a, c, u.u, u.w
  double hp[kMaxFusedGs + 1], cs[kMaxFusedGs], sn[kMaxFusedGs];     // as on entry, then updated
  double inv_nu, e, gj;
};

// val = a (V^T u), c (V^T w), u.u, u.w over v_0..v_{j-1}; R rows per thread held in
// u, w. All of a chunk's basis loads are in flight before its products.
template <int R>
__device__ __forceinline__ void dots_all(int n, int j, const double* __restrict__ V, const double (&u)[R],
                                         const double (&w)[R], ColData& C) {
  constexpr int K = R > 2 ? 4 : 8;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wid = tid / kWave;
  for (int c0 = 0; c0 < j; c0 += K) {
    double v[K][R];
#pragma unroll
    for (int t = 0; t < K; ++t)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int i = tid + r * kT;
        v[t][r] = (c0 + t < j && i < n) ? V[(long long)(c0 + t) * n + i] : 0.0;
      }
    double s[2 * K];
#pragma unroll
    for (int t = 0; t < K; ++t) {
      s[t] = s[K + t] = 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        s[t] += v[t][r] * u[r];
        s[K + t] += v[t][r] * w[r];
      }
    }
    const double f = wave_fold<2 * K>(s);
    const int q = fold_index<2 * K>(lane), t = c0 + (q % K);
    if (lane % (kWave / (2 * K)) == 0 && t < j) C.part[wid][(q < K ? 0 : j) + t] = f;
  }
  double s[2] = {0.0, 0.0};
#pragma unroll
  for (int r = 0; r < R; ++r) {
    s[0] += u[r] * u[r];
    s[1] += u[r] * w[r];
  }
  const double f = wave_fold<2>(s);
  if (lane % (kWave / 2) == 0) C.part[wid][2 * j + fold_index<2>(lane)] = f;
  __syncthreads();
  if (tid < 2 * j + 2) {
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < kW; ++q) v += C.part[q][tid];
    C.val[tid] = v;
  }
  __syncthreads();
}

// k_lag_colA: column j-1 final, its rotation, the provisional column j
__device__ __forceinline__ void col_final(Layout L, int j, double* __restrict__ sm, ColData& C, double gj1) {
  const double* a = C.val;
  const double* c = C.val + j;
  if (threadIdx.x == 0) {
    const double ss = C.val[2 * j], dd = C.val[2 * j + 1];
    double aa = 0.0, ac = 0.0;
    for (int q = 0; q < j; ++q) {
      aa += a[q] * a[q];
      ac += a[q] * c[q];
    }
    const double nu = (j == 0) ? 1.0 : sqrt(fmax(ss - aa, 0.0));
    double gj = gj1;  // j = 0: g[0]
    if (j > 0) {
      double x = C.hp[0] + a[0];
      for (int q = 0; q + 1 < j; ++q) {
        const double y = C.hp[q + 1] + a[q + 1];
        sm[L.H(q, j - 1)] = C.cs[q] * x + C.sn[q] * y;
        x = -C.sn[q] * x + C.cs[q] * y;
      }
      double cr, sr;
      givens(x, nu, cr, sr);
      C.cs[j - 1] = cr;
      C.sn[j - 1] = sr;
      sm[L.cs() + j - 1] = cr;
      sm[L.sn() + j - 1] = sr;
      sm[L.H(j - 1, j - 1)] = cr * x + sr * nu;
      sm[L.H(j, j - 1)] = 0.0;
      gj = -sr * gj1;
      sm[L.g() + j] = gj;
      sm[L.g() + j - 1] = cr * gj1;
    }
    C.gj = gj;
    C.e = (nu > 0.0) ? (dd - ac) / nu : 0.0;
    C.inv_nu = (nu > 0.0) ? 1.0 / nu : 0.0;
  }
  __syncthreads();
}

// column data of step j into LDS (before the first barrier of the step)
__device__ __forceinline__ double col_load(Layout L, int j, const double* __restrict__ sm, ColData& C) {
  const int t = threadIdx.x;
  if (t < j) {
    C.hp[t] = sm[L.hp() + t];
    C.cs[t] = sm[L.cs() + t];
    C.sn[t] = sm[L.sn() + t];
  }
  return sm[L.g() + (j > 0 ? j - 1 : 0)];
}

// One lagged Arnoldi step (see fgmres.hip) after the preconditioner left x = M u:
// z = sout .* x -> Z, w = D^-1 A z; dots; column j-1 final; v_j and the next u, its
// preconditioner input; the residual estimate of step j -> sm sc[2], *est.
template <class T, int R>
__global__ __launch_bounds__(kT) void k_small_step(SmallOperator A, Layout L, int j, double* __restrict__ sm,
                                                   const T* __restrict__ x, const double* __restrict__ sout,
                                                   double* __restrict__ Z, double* V, const double* __restrict__ S,
                                                   T* __restrict__ bout, double* est) {
  __shared__ ColData C;
  __shared__ double lds[kW];
  const int n = A.n, tid = threadIdx.x;
  const double gj1 = col_load(L, j, sm, C);
  double* uj = V + (long long)j * n;
  double u[R], w[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = tid + r * kT;
    u[r] = w[r] = 0.0;
    if (i < n) {
      u[r] = uj[i];
      auto zv = [&](int q) { return sout[q] * (double)x[q]; };
      w[r] = A.dinv[i] * row_apply(A, i, zv);
      Z[i] = zv(i);
    }
  }
  dots_all<R>(n, j, V, u, w, C);
  col_final(L, j, sm, C, gj1);
  const double* a = C.val;
  const double* c = C.val + j;
  constexpr int K = R > 2 ? 4 : 8;
  double su[R] = {}, sw[R] = {};
  for (int c0 = 0; c0 < j; c0 += K) {
    double v[K][R];
#pragma unroll
    for (int t = 0; t < K; ++t)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int i = tid + r * kT;
        v[t][r] = (c0 + t < j && i < n) ? V[(long long)(c0 + t) * n + i] : 0.0;
      }
#pragma unroll
    for (int t = 0; t < K; ++t) {
      if (c0 + t >= j) break;
      const double at = a[c0 + t], ct = c[c0 + t];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        su[r] += v[t][r] * at;
        sw[r] += v[t][r] * ct;
      }
    }
  }
  double* un = uj + n;
  double ww = 0.0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = tid + r * kT;
    if (i < n) {
      const double vj = (u[r] - su[r]) * C.inv_nu;
      const double w1 = (w[r] - sw[r]) - vj * C.e;
      uj[i] = vj;
      un[i] = w1;
      bout[i] = (T)(S[i] * w1);
      ww += w1 * w1;
    }
  }
  ww = block_total(ww, lds);
  if (tid < j) sm[L.hp() + tid] = c[tid];  // the provisional column starts from c
  if (tid != 0) return;
  sm[L.hp() + j] = C.e;
  // k_lag_colB: rotations 0..j-1 on the provisional column, then the new one
  double y = (j > 0) ? c[0] : C.e;
  for (int q = 0; q < j; ++q) y = -C.sn[q] * y + C.cs[q] * ((q + 1 < j) ? c[q + 1] : C.e);
  double cr, sr;
  givens(y, sqrt(fmax(ww, 0.0)), cr, sr);
  const double v = fabs(sr * C.gj);
  sm[L.sc() + 2] = v;
  *est = v;
}

// End of a cycle of k steps: with `close`, column k-1 is finished first (dots of
// u = V[:, k]); y = H^-1 g, x += Z y, V = D^-1 (b - A x), its squared norm -> sm sc[4],
// host[4], and the error check's preconditioner input S .* V.
template <class T, int R>
__global__ __launch_bounds__(kT) void k_small_end(SmallOperator A, Layout L, int k, int close, double* __restrict__ sm,
                                                  const double* __restrict__ Z, double* V, const double* b, double* x,
                                                  const double* __restrict__ S, T* __restrict__ bout, double* host) {
  __shared__ ColData C;
  __shared__ double lds[kW];
  __shared__ double hs[kMaxFusedGs][kMaxFusedGs + 1], y[kMaxFusedGs];
  const int n = A.n, tid = threadIdx.x;
  if (close) {
    const double gj1 = col_load(L, k, sm, C);
    double u[R];
#pragma unroll
    for (int r = 0; r < R; ++r) u[r] = (tid + r * kT < n) ? V[(long long)k * n + tid + r * kT] : 0.0;
    dots_all<R>(n, k, V, u, u, C);
    col_final(L, k, sm, C, gj1);
  }
  // back substitution, one lane per row (k <= 32)
  for (int q = tid; q < k * k; q += kT) hs[q / k][q % k] = sm[L.H(q % k, q / k)];
  __syncthreads();
  if (tid < kWave) {
    double gj = (tid < k) ? sm[L.g() + tid] : 0.0;
    for (int i = k - 1; i >= 0; --i) {
      const double gi = __shfl(gj, i, kWave);
      const double d = hs[i][i];
      const double yi = (d != 0.0) ? gi / d : 0.0;
      if (tid == i) y[i] = yi;
      if (tid < i) gj -= hs[i][tid] * yi;
    }
  }
  __syncthreads();
  for (int i = tid; i < n; i += kT) {
    double s = x[i];
#pragma unroll 8
    for (int c = 0; c < k; ++c) s += Z[(long long)c * n + i] * y[c];
    x[i] = s;
  }
  __syncthreads();
  const double rr = residual_all(A, b, x, V, lds);
  for (int i = tid; i < n; i += kT) bout[i] = (T)(S[i] * V[i]);
  if (tid == 0) {
    sm[L.sc() + 4] = rr;
    host[4] = rr;
  }
}

// Preconditioner input of the error check where no cycle ran before it
template <class T>
__global__ __launch_bounds__(kT) void k_small_input(int n, const double* __restrict__ V, const double* __restrict__ S,
                                                    T* __restrict__ bout) {
  for (int i = threadIdx.x; i < n; i += kT) bout[i] = (T)(S[i] * V[i]);
}

// Error check: z = sout .* (M V); ||z||_inf -> host[6], x += z, ||x||_inf -> host[7],
// V = D^-1 (b - A x) and its squared norm -> sm sc[4], host[4].
template <class T>
__global__ __launch_bounds__(kT) void k_small_check(SmallOperator A, Layout L, double* __restrict__ sm,
                                                    const T* __restrict__ xc, const double* __restrict__ sout,
                                                    double* V, const double* b, double* x, double* host) {
  __shared__ double lds[kW];
  double zm = 0.0, xm = 0.0;
  for (int i = threadIdx.x; i < A.n; i += kT) {
    const double z = sout[i] * (double)xc[i];
    const double xi = x[i] + z;
    zm = fmax(zm, fabs(z));
    xm = fmax(xm, fabs(xi));
    x[i] = xi;
  }
  zm = block_most(zm, lds);
  xm = block_most(xm, lds);
  __syncthreads();
  const double rr = residual_all(A, b, x, V, lds);
  if (threadIdx.x == 0) {
    sm[L.sc() + 4] = rr;
    host[4] = rr;
    host[6] = zm;
    host[7] = xm;
  }
}

}  // namespace

void small_start(const SmallOperator& A, FgmresLayout L, double* sm, const double* b, double* x, bool use_x0, double* V,
                 double* host, hipStream_t s) {
  k_small_start<<<1, kT, 0, s>>>(A, L, sm, b, x, use_x0 ? 1 : 0, V, host);
  IMPES_LAUNCH_CHECK();
}

template <class T>
void small_begin(int n, FgmresLayout L, double* sm, double* V, const double* S, T* bout, hipStream_t s) {
  k_small_begin<T><<<1, kT, 0, s>>>(n, L, sm, V, S, bout);
  IMPES_LAUNCH_CHECK();
}

template <class T>
void small_step(const SmallOperator& A, FgmresLayout L, int j, double* sm, const T* x, const double* sout, double* Z,
                double* V, const double* S, T* bout, double* est, hipStream_t s) {
  if (A.n <= kT) k_small_step<T, 1><<<1, kT, 0, s>>>(A, L, j, sm, x, sout, Z, V, S, bout, est);
  else if (A.n <= 2 * kT) k_small_step<T, 2><<<1, kT, 0, s>>>(A, L, j, sm, x, sout, Z, V, S, bout, est);
  else k_small_step<T, 4><<<1, kT, 0, s>>>(A, L, j, sm, x, sout, Z, V, S, bout, est);
  IMPES_LAUNCH_CHECK();
}
static_assert(kSmallRows <= 4 * kT, "rows per thread");

template <class T>
void small_end(const SmallOperator& A, FgmresLayout L, int k, bool close, double* sm, const double* Z, double* V,
               const double* b, double* x, const double* S, T* bout, double* host, hipStream_t s) {
  const int c = close ? 1 : 0;
  if (A.n <= kT) k_small_end<T, 1><<<1, kT, 0, s>>>(A, L, k, c, sm, Z, V, b, x, S, bout, host);
  else if (A.n <= 2 * kT) k_small_end<T, 2><<<1, kT, 0, s>>>(A, L, k, c, sm, Z, V, b, x, S, bout, host);
  else k_small_end<T, 4><<<1, kT, 0, s>>>(A, L, k, c, sm, Z, V, b, x, S, bout, host);
  IMPES_LAUNCH_CHECK();
}

template <class T>
void small_input(int n, const double* V, const double* S, T* bout, hipStream_t s) {
  k_small_input<T><<<1, kT, 0, s>>>(n, V, S, bout);
  IMPES_LAUNCH_CHECK();
}

template <class T>
void small_check(const SmallOperator& A, FgmresLayout L, double* sm, const T* xc, const double* sout, double* V,
                 const double* b, double* x, double* host, hipStream_t s) {
  k_small_check<T><<<1, kT, 0, s>>>(A, L, sm, xc, sout, V, b, x, host);
  IMPES_LAUNCH_CHECK();
}

#define IMPES_SMALL(T)                                                                                             \
  template void small_begin<T>(int, FgmresLayout, double*, double*, const double*, T*, hipStream_t);              \
  template void small_step<T>(const SmallOperator&, FgmresLayout, int, double*, const T*, const double*, double*, \
                              double*, const double*, T*, double*, hipStream_t);                                  \
  template void small_end<T>(const SmallOperator&, FgmresLayout, int, bool, double*, const double*, double*,      \
                             const double*, double*, const double*, T*, double*, hipStream_t);                    \
  template void small_input<T>(int, const double*, const double*, T*, hipStream_t);                               \
  template void small_check<T>(const SmallOperator&, FgmresLayout, double*, const T*, const double*, double*,     \
                               const double*, double*, double*, hipStream_t);
IMPES_SMALL(float)
IMPES_SMALL(double)
#undef IMPES_SMALL

}  // namespace impes
