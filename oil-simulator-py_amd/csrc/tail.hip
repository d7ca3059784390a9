// The coarse end of the V-cycle as one matrix. From a level of at most kTailMax rows
// down, a V-cycle that starts from zero is a fixed linear operator B until the next
// numeric update: B = V(I). It is formed once per update by running the cycle on the
// columns of the identity, and each V-cycle then applies it as one dense
// matrix-vector product instead of about six dependent launches per level.
//
// What it replaces is bound by launches: a level of 1,894 rows costs 25 us per visit
// for 2.4 MB, and a whole hierarchy of a 1,200-cell reservoir 14 launches of ~3 us.
// The product reads n^2 values once (14 MB in FP32 at 1,894 rows, from the L2s).
//
// Forming: a workgroup takes M columns through all levels with its vectors in LDS,
// so there is no launch per level, and n / M workgroups fill the chip. The operators
// are read in sliced form (64 rows per slice, entry k of a slice's rows side by side),
// a row per lane: each load is one contiguous 64-entry line, and the M values of the
// gathered row are one or two 16-byte LDS reads.
//
// B is formed in FP64 for both cycles and rounded once for the FP32 one. An FP32 cycle
// level by level applies the coarsest inverse in FP64, so a B of FP32 operations would
// hold fewer bits than what it replaces: over 48 operators of 400-1,600 rows its error
// against the FP64 cycle was 1.05 times the level-by-level FP32 cycle's in the mean and
// up to 4.3 times; rounded once it is 0.55 times (the rest is the rounding of b). The
// FP64 operations cost 72 us against 50 at 1,200 rows, once per update.
#include <algorithm>
#include <vector>

#include "amg_kernels.h"
#include "prims.h"

namespace impes {

namespace {

constexpr int kTailThreads = 1024;

struct EllEntry {
  double v;
  int c;
};

// Slice offsets of a level: the exclusive sums of the longest row of each 64 rows
// (at most kTailMax / 64 slices) and, behind them, the total. One workgroup.
__global__ __launch_bounds__(kTailThreads) void k_tail_slices(int n, const int* __restrict__ rp, int* __restrict__ so) {
  __shared__ int width[kWave];
  static_assert(kTailMax <= kWave * kWave, "one lane per slice");
  const int lane = threadIdx.x & (kWave - 1), ns = (n + kWave - 1) / kWave;
  for (int sl = threadIdx.x / kWave; sl < ns; sl += kTailThreads / kWave) {
    const int r = sl * kWave + lane;
    const int len = wave_max(r < n ? rp[r + 1] - rp[r] : 0);
    if (lane == 0) width[sl] = len;
  }
  __syncthreads();
  if (threadIdx.x >= kWave) return;
  const int w = lane < ns ? width[lane] : 0;
  int sum = w;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int u = __shfl_up(sum, d, kWave);
    if (lane >= d) sum += u;
  }
  if (lane < ns) so[lane] = sum - w;
  if (lane == ns - 1) so[ns] = sum;
}

// The sliced operator: padding entries have value 0 and their own row as column.
__global__ __launch_bounds__(256) void k_tail_pack(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                                                   const double* __restrict__ v, const int* __restrict__ so,
                                                   EllEntry* __restrict__ ell) {
  // a wave per quarter of a slice's width: the rows' loads are spread over four waves
  const int sl = blockIdx.x, lane = threadIdx.x & (kWave - 1), part = threadIdx.x / kWave;
  const int r = sl * kWave + lane;
  const int k1 = so[sl + 1] - so[sl];
  const int e0 = r < n ? rp[r] : 0, len = r < n ? rp[r + 1] - e0 : 0;
  for (int k = part; k < k1; k += 256 / kWave) {
    EllEntry e{0.0, r < n ? r : 0};
    if (k < len) {
      e.v = v[e0 + k];
      e.c = ci[e0 + k];
    }
    ell[(long long)(so[sl] + k) * kWave + lane] = e;
  }
}

template <class T, int M>
struct Vec {
  T v[M];
};
template <class T, int M>
__device__ __forceinline__ Vec<T, M> ld_vec(const T* __restrict__ p) {
  Vec<T, M> r;
  __builtin_memcpy(&r, __builtin_assume_aligned(p, 16), sizeof(r));
  return r;
}

// A workgroup's M columns of an LDS vector: planes of 16 bytes per row, so that the
// reads of neighbouring rows fall on neighbouring banks.
template <class T, int M>
struct Cols {
  static constexpr int V = 16 / sizeof(T);
  T* p;
  int n;  // rows
  __device__ __forceinline__ Vec<T, M> get(int i) const {
    Vec<T, M> r;
#pragma unroll
    for (int q = 0; q < M / V; ++q)
      __builtin_memcpy(&r.v[q * V], __builtin_assume_aligned(p + ((long long)q * n + i) * V, 16), 16);
    return r;
  }
  __device__ __forceinline__ void put(int i, const Vec<T, M>& r) const {
#pragma unroll
    for (int q = 0; q < M / V; ++q)
      __builtin_memcpy(__builtin_assume_aligned(p + ((long long)q * n + i) * V, 16), &r.v[q * V], 16);
  }
};

template <class T, int M>
__device__ __forceinline__ void add(Vec<T, M>& acc, T a, const Vec<T, M>& x) {
#pragma unroll
  for (int m = 0; m < M; ++m) acc.v[m] += a * x.v[m];
}

// Rows i and i + kTailThreads of a sliced operator times X (so: its slice offsets in
// LDS), both rows' loads in flight at once; rows past n give 0.
template <class T, int M>
struct RowPair {
  Vec<T, M> a, b;
};
template <class T, int M>
__device__ __forceinline__ RowPair<T, M> rows_times(const TailLevel& L, const int* __restrict__ so, int i,
                                                    const Cols<T, M>& X) {
  RowPair<T, M> r{};
  const EllEntry* ell = static_cast<const EllEntry*>(L.ell) + i % kWave;
  const int s0 = i / kWave, s1 = s0 + kTailThreads / kWave, ns = (L.n + kWave - 1) / kWave;
  const int q0 = s0 < ns ? so[s0] : 0, w0 = s0 < ns ? so[s0 + 1] - q0 : 0;
  const int q1 = s1 < ns ? so[s1] : 0, w1 = s1 < ns ? so[s1 + 1] - q1 : 0;
  const EllEntry* e0 = ell + (long long)q0 * kWave;
  const EllEntry* e1 = ell + (long long)q1 * kWave;
  const int both = w0 < w1 ? w0 : w1;
  int k = 0;
#pragma unroll 4
  for (; k < both; ++k) {
    const EllEntry x = e0[k * kWave], y = e1[k * kWave];
    add<T, M>(r.a, x.v, X.get(x.c));
    add<T, M>(r.b, y.v, X.get(y.c));
  }
  const int k0 = k;
#pragma unroll 8
  for (k = k0; k < w0; ++k) {
    const EllEntry x = e0[k * kWave];
    add<T, M>(r.a, x.v, X.get(x.c));
  }
#pragma unroll 8
  for (k = k0; k < w1; ++k) {
    const EllEntry y = e1[k * kWave];
    add<T, M>(r.b, y.v, X.get(y.c));
  }
  return r;
}

// entries g, g + G, .. of row i of a CSR transfer (P or R) times X
template <class T, int M, int G>
__device__ __forceinline__ Vec<T, M> csr_row_times(const int* __restrict__ rp, const int* __restrict__ ci,
                                                   const double* __restrict__ v, int i, int g, const Cols<T, M>& X) {
  Vec<T, M> acc{};
  const int e1 = rp[i + 1];
#pragma unroll 4
  for (int e = rp[i] + g; e < e1; e += G) add<T, M>(acc, (T)v[e], X.get(ci[e]));
  return acc;
}
constexpr int kRowLanes = 4;

// Columns blockIdx.x * M .. of B = V(I). Vectors in LDS: x and y (ping-pong, y also
// the residual) per level, b below the first level (whose right-hand side is the
// identity's columns). The coarsest level's solve sums in FP64 over the transposed
// inverse, so that a wave reads contiguous lines: two rows per thread and the columns
// split over the remaining threads; its x overwrites its b.
// What bounds it: at 1,200 rows the ~17 dependent phases of 1-6 us (72 us together);
// on dense levels (852 rows with 24 entries each: 136 us) the LDS reads of the gathered
// rows.
constexpr int kTailSlices = kTailLevels * (kTailMax / kWave + 1);
template <class S, int M>
__global__ __launch_bounds__(kTailThreads) void k_tail_form(TailArgs A) {
  using T = double;
  extern __shared__ __align__(16) unsigned char raw[];
  __shared__ int so[kTailSlices];
  T* lds = reinterpret_cast<T*>(raw);
  const int tid = threadIdx.x;
  const int c0 = blockIdx.x * M;
  const T w = (T)A.omega;
  const int nd = A.levels;  // non-coarsest levels
  for (int q = tid; q < A.so_len; q += kTailThreads) so[q] = A.so[q];
  unsigned flip = 0;  // bit l: the iterate of level l is in its y, the other buffer its x
  auto cur = [&](int l) {
    return Cols<T, M>{lds + ((flip >> l & 1u) ? A.lv[l].y : A.lv[l].x), A.lv[l].n};
  };
  auto oth = [&](int l) {
    return Cols<T, M>{lds + ((flip >> l & 1u) ? A.lv[l].x : A.lv[l].y), A.lv[l].n};
  };
  // the right-hand side of level l at row i
  auto rhs = [&](int l, int i) {
    if (l > 0) return Cols<T, M>{lds + A.lv[l].b, A.lv[l].n}.get(i);
    Vec<T, M> r;
#pragma unroll
    for (int m = 0; m < M; ++m) r.v[m] = (i == c0 + m) ? T(1) : T(0);
    return r;
  };
  auto sweep = [&](int l) {
    const TailLevel& L = A.lv[l];
    const Cols<T, M> xi = cur(l), xo = oth(l);
    for (int i = tid; i < L.n; i += 2 * kTailThreads) {
      const RowPair<T, M> s = rows_times<T, M>(L, so + L.so, i, xi);
      auto put = [&](int r, const Vec<T, M>& sum) {
        const Vec<T, M> b = rhs(l, r);
        Vec<T, M> x = xi.get(r);
        const T a = w * (T)L.ir[r];
#pragma unroll
        for (int m = 0; m < M; ++m) x.v[m] += a * (b.v[m] - sum.v[m]);
        xo.put(r, x);
      };
      put(i, s.a);
      if (i + kTailThreads < L.n) put(i + kTailThreads, s.b);
    }
    flip ^= 1u << l;
    __syncthreads();
  };
  for (int l = 0; l < nd; ++l) {
    const TailLevel& L = A.lv[l];
    const Cols<T, M> x0{lds + L.x, L.n};
    for (int i = tid; i < L.n; i += kTailThreads) {  // first sweep from zero
      Vec<T, M> x = rhs(l, i);
      const T a = A.pre > 0 ? w * (T)L.ir[i] : T(0);
#pragma unroll
      for (int m = 0; m < M; ++m) x.v[m] *= a;
      x0.put(i, x);
    }
    __syncthreads();
    for (int it = 1; it < A.pre; ++it) sweep(l);
    const Cols<T, M> xi = cur(l), res = oth(l);
    for (int i = tid; i < L.n; i += 2 * kTailThreads) {  // residual
      RowPair<T, M> s{};
      if (A.pre > 0) s = rows_times<T, M>(L, so + L.so, i, xi);
      auto put = [&](int r, const Vec<T, M>& sum) {
        Vec<T, M> v = rhs(l, r);
#pragma unroll
        for (int m = 0; m < M; ++m) v.v[m] -= sum.v[m];
        res.put(r, v);
      };
      put(i, s.a);
      if (i + kTailThreads < L.n) put(i + kTailThreads, s.b);
    }
    __syncthreads();
    const Cols<T, M> bc{lds + A.lv[l + 1].b, A.lv[l + 1].n};
    for (int i = tid / kRowLanes; i < bc.n; i += kTailThreads / kRowLanes) {
      // the ~20 entries of a restriction row over kRowLanes lanes
      Vec<T, M> r = csr_row_times<T, M, kRowLanes>(L.rrp, L.rci, L.rv, i, tid % kRowLanes, res);
#pragma unroll
      for (int m = 0; m < M; ++m) r.v[m] = group_sum<kRowLanes>(r.v[m]);
      if (tid % kRowLanes == 0) bc.put(i, r);
    }
    __syncthreads();
  }
  {
    // coarsest: x = A^-1 b (b_0 = 0 when pinned)
    const TailLevel& L = A.lv[nd];
    const Cols<T, M> x{lds + L.x, L.n};
    double* part = reinterpret_cast<double*>(lds + A.part);  // partial sums [split][column][row]
    const int pairs = (L.n + 1) / 2;
    const int tr = (pairs + kWave - 1) / kWave * kWave;  // threads over the rows
    const int splits = A.splits;
    const int p = tid % tr, sp = tid / tr;
    if (sp < splits && p < pairs) {
      const int r0 = p, r1 = p + pairs;
      const bool two = r1 < L.n;
      double s0[M] = {}, s1[M] = {};
      const int k0 = max((int)((long long)L.n * sp / splits), *A.pin ? 1 : 0);
      const int k1 = (int)((long long)L.n * (sp + 1) / splits);
      const double* col = A.inv_t + r0;
      const int off = two ? pairs : 0;
#pragma unroll 8
      for (int k = k0; k < k1; ++k) {
        const double a0 = col[(long long)k * A.inv_ld];
        const double a1 = col[(long long)k * A.inv_ld + off];
        const Vec<T, M> v = x.get(k);
#pragma unroll
        for (int m = 0; m < M; ++m) {
          s0[m] += a0 * (double)v.v[m];
          s1[m] += a1 * (double)v.v[m];
        }
      }
#pragma unroll
      for (int m = 0; m < M; ++m) {
        part[(sp * M + m) * L.n + r0] = s0[m];
        if (two) part[(sp * M + m) * L.n + r1] = s1[m];
      }
    }
    __syncthreads();
    for (int r = tid; r < L.n; r += kTailThreads) {
      Vec<T, M> v;
#pragma unroll
      for (int m = 0; m < M; ++m) {
        double t = 0.0;
        for (int q = 0; q < splits; ++q) t += part[(q * M + m) * L.n + r];
        v.v[m] = (T)t;
      }
      x.put(r, v);
    }
    __syncthreads();
  }
  for (int l = nd - 1; l >= 0; --l) {
    const TailLevel& L = A.lv[l];
    const Cols<T, M> xc = cur(l + 1), xf = cur(l);
#pragma unroll 2
    for (int i = tid; i < L.n; i += kTailThreads) {
      const Vec<T, M> e = csr_row_times<T, M, 1>(L.prp, L.pci, L.pv, i, 0, xc);
      Vec<T, M> x = xf.get(i);
#pragma unroll
      for (int m = 0; m < M; ++m) x.v[m] += e.v[m];
      xf.put(i, x);
    }
    __syncthreads();
    for (int it = 0; it < A.post; ++it) sweep(l);
  }
  // the row stride holds the last workgroup's padding columns
  S* B = static_cast<S*>(A.B);
  const Cols<T, M> xb = cur(0);
  for (int i = tid; i < A.lv[0].n; i += kTailThreads) {
    const Vec<T, M> x = xb.get(i);
    Vec<S, M> r;
#pragma unroll
    for (int m = 0; m < M; ++m) r.v[m] = (S)x.v[m];
    constexpr int align = sizeof(r) % 16 == 0 ? 16 : 8;  // c0 is a multiple of M, ld of 8
    __builtin_memcpy(__builtin_assume_aligned(B + (long long)i * A.ld + c0, align), &r, sizeof(r));
  }
}

// x = B b: a wavefront per row with 16-byte loads, sums in FP64. Columns past n hold
// the cycle of a zero right-hand side, zero; b is not read there.
template <class T>
__global__ __launch_bounds__(256) void k_tail_mv(int n, int ld, const T* __restrict__ B, const T* __restrict__ b,
                                                 T* __restrict__ x) {
  constexpr int V = 16 / sizeof(T);
  const int lane = threadIdx.x & (kWave - 1);
  const int r = (int)xcd_block() * (256 / kWave) + threadIdx.x / kWave;
  if (r >= n) return;
  const T* row = B + (long long)r * ld;
  double s[V] = {};
  int c = lane * V;
#pragma unroll 4
  for (; c + V <= n; c += kWave * V) {
    const Vec<T, V> a = ld_vec<T, V>(row + c), v = ld_vec<T, V>(b + c);
#pragma unroll
    for (int m = 0; m < V; ++m) s[m] += (double)a.v[m] * (double)v.v[m];
  }
  if (c < n)
    for (int m = 0; c + m < n; ++m) s[0] += (double)row[c + m] * (double)b[c + m];
  double t = s[0];
#pragma unroll
  for (int m = 1; m < V; ++m) t += s[m];
  t = wave_sum(t);
  if (lane == 0) x[r] = (T)t;
}

template <class S, int M>
void form(const TailArgs& A, size_t lds, hipStream_t s) {
  IMPES_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_tail_form<S, M>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  k_tail_form<S, M><<<div_up(A.lv[0].n, M), kTailThreads, lds, s>>>(A);
  IMPES_LAUNCH_CHECK();
}

}  // namespace

int tail_slices(int n) { return div_up(n, kWave); }

void launch_tail_slices(int n, const int* rp, int* so, hipStream_t s) {
  k_tail_slices<<<1, kTailThreads, 0, s>>>(n, rp, so);
  IMPES_LAUNCH_CHECK();
}

size_t tail_ell_bytes(long long lines) { return (size_t)lines * kWave * sizeof(EllEntry); }

void launch_tail_pack(int n, const int* rp, const int* ci, const double* v, const int* so, void* ell, hipStream_t s) {
  k_tail_pack<<<tail_slices(n), 256, 0, s>>>(n, rp, ci, v, so, static_cast<EllEntry*>(ell));
  IMPES_LAUNCH_CHECK();
}

// LDS offsets for M columns a workgroup; the bytes. Once a level's residual has been
// restricted, the buffer that held it is free until the level's first post-sweep: the
// next level's x and y lie in it where they fit, or the coarsest solve's partial sums.
static size_t layout(TailArgs& A, int M) {
  long long at = 0;
  auto take = [&](int n) {
    const long long o = at;
    at += (long long)n * M;
    return (int)o;
  };
  int room = 0, free_at = 0;  // rows and offset of the level above's free buffer
  for (int l = 0; l <= A.levels; ++l) {
    TailLevel& L = A.lv[l];
    if (l > 0) L.b = take(L.n);
    if (l == A.levels) {
      L.x = L.b;
      L.y = 0;
      break;
    }
    const bool inside = 2 * L.n <= room;
    L.x = inside ? free_at : take(L.n);
    L.y = inside ? free_at + L.n * M : take(L.n);
    room = L.n;
    free_at = A.pre > 1 && (A.pre - 1) % 2 == 1 ? L.x : L.y;  // the residual's (cur after the sweeps is the other)
  }
  // one split per group of threads over the row pairs, as many as fit
  const int n = A.lv[A.levels].n;
  const size_t used = (size_t)at * sizeof(double), one = (size_t)n * M * sizeof(double);
  const int groups = kTailThreads / (div_up((n + 1) / 2, kWave) * kWave);
  const int in_room = std::min(groups, room / n);
  const int behind = used < kTailLds ? (int)std::min<size_t>(groups, (kTailLds - used) / one) : 0;
  A.splits = std::max(in_room, behind);
  A.part = in_room >= behind ? free_at : (int)at;
  if (A.splits == 0) return kTailLds + 1;
  return in_room >= behind ? used : used + A.splits * one;
}

// Columns a workgroup: the fewest that take at most one workgroup per CU, since a second
// round of workgroups costs as much as the first (1,200 rows: 99 us with 4, in two
// rounds, 72 with 6; 1,072 rows 118 and 84), where six columns fit the LDS; else 4.
static int tail_cols(TailArgs& A) {
  for (int M : {2, 4, 6})
    if (div_up(A.lv[0].n, M) <= 256 && layout(A, M) <= kTailLds) return M;
  return 4;
}

// Two or four columns of every vector side by side (x and y, b below the first level,
// the partial sums) fit the LDS: up to about 1,500 rows. Larger ones would fit as well
// with the shared buffers, but take two rounds of long passes and do not pay.
bool tail_fits(const TailArgs& A) {
  const int n0 = A.lv[0].n, nc = A.lv[A.levels].n;
  long long rows = 2LL * n0 + (n0 > 512 && n0 <= 1024 ? 2LL : 3LL) * nc;
  for (int l = 1; l < A.levels; ++l) rows += 3LL * A.lv[l].n;
  return rows * (n0 <= 512 ? 16 : 32) <= (long long)kTailLds;
}

void launch_tail_form(int precision, TailArgs A, hipStream_t s) {
  const int M = tail_cols(A);
  const size_t lds = layout(A, M);
  IMPES_REQUIRE(lds <= kTailLds, "tail: vectors exceed LDS");
  IMPES_REQUIRE(A.ld % 2 == 0 && A.ld >= div_up(A.lv[0].n, M) * M, "tail: row stride");
  if (precision == 32) {
    if (M == 6) form<float, 6>(A, lds, s);
    else if (M == 4) form<float, 4>(A, lds, s);
    else form<float, 2>(A, lds, s);
  } else {
    if (M == 6) form<double, 6>(A, lds, s);
    else if (M == 4) form<double, 4>(A, lds, s);
    else form<double, 2>(A, lds, s);
  }
}

void launch_tail_mv_f32(int n, int ld, const float* B, const float* b, float* x, hipStream_t s) {
  k_tail_mv<float><<<div_up(n, 4), 256, 0, s>>>(n, ld, B, b, x);
  IMPES_LAUNCH_CHECK();
}

void launch_tail_mv_f64(int n, int ld, const double* B, const double* b, double* x, hipStream_t s) {
  k_tail_mv<double><<<div_up(n, 4), 256, 0, s>>>(n, ld, B, b, x);
  IMPES_LAUNCH_CHECK();
}

}  // namespace impes
