// Dense inverse of a large coarsest AMG operator (classical_amg.py:1045-1069 solves
// the coarsest level densely) on the matrix cores: blocked Gauss-Jordan without
// pivoting, whose rank-64 updates run as 64 x 64 x 64 FP64 tiles of
// v_mfma_f64_16x16x4_f64. The operator is symmetric positive definite (a Galerkin
// product of the SPD pressure matrix, with DOF 0 optionally pinned), so every
// diagonal block met during the elimination is a Schur complement of an SPD
// matrix and itself SPD: no pivoting is needed.
//
// The matrix (n x n, row-major) is padded to n_pad = 64 nb with an identity block.
// For each block column k (one step of Gauss-Jordan on 64 columns at once):
//   P = A_kk^-1                          one workgroup, the block in registers (4 x 4 pivot blocks)
//   from A into A':                      one workgroup per 64 x 64 block, MFMA
// where the first P comes from its own launch and each later one from the
// workgroup of the previous step that produces that pivot block (so one launch
// per block column after the first)
//     A'_kk = P;  A'_kj = P A_kj;  A'_ik = -A_ik P;  A'_ij = A_ij - A_ik (P A_kj)
// which is the scalar elimination (a_kj /= a_kk; a_ij -= a_ik a_kj; a_ik = -a_ik /
// a_kk; a_kk = 1 / a_kk) on 64 x 64 blocks. Writing into a second matrix lets
// every block read the old row and column panels, so each block forms its own
// P A_kj instead of waiting on a row-panel launch. After the last block column
// the inverse is in M (the elimination starts in W when nb is odd). Each visit of
// the V-cycle then applies the inverse as one dense matrix-vector product (a
// wavefront per row, FP64 accumulation).
#include <utility>

#include "amg_kernels.h"

namespace impes {

namespace {

constexpr int kB = 64;        // block size of the elimination
// LDS row strides (doubles). A wave reads A operands at (row i, column kk) and B
// operands at (row kk, column i), i < 16, kk < 4: with these strides the 64 lanes
// spread evenly over the banks (a common stride of 65 left both 4-way conflicted).
constexpr int kLdA = kB + 4;
constexpr int kLdB = kB + 16;
constexpr int kGemmThreads = 256;
typedef double v4d __attribute__((ext_vector_type(4)));

// C = A B for 64 x 64 tiles in LDS (row strides kLdA, kLdB). Wave w owns rows
// 16w..16w+15 as four 16 x 16 output tiles t (columns 16t..16t+15).
// v_mfma_f64_16x16x4_f64 lane layout (measured on gfx950): A[i][k] at lane i + 16k,
// B[k][j] at lane j + 16k, D[i][j] at lane j + 16 (i % 4), element i / 4.
// kDepth: how many of the 64 inner indices count (the rest add zeros)
template <int kDepth>
__device__ __forceinline__ void tile_mma_depth(const double* __restrict__ As, const double* __restrict__ Bs,
                                               v4d (&acc)[4]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = lane & 15, kk = lane >> 4;
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
  for (int k0 = 0; k0 < kDepth; k0 += 4) {
    const double a = As[(16 * w + i) * kLdA + k0 + kk];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const double b = Bs[(k0 + kk) * kLdB + 16 * t + i];
      acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[t], 0, 0, 0);
    }
  }
}

// rows: the inner indices that belong to the matrix
__device__ __forceinline__ void tile_mma(const double* __restrict__ As, const double* __restrict__ Bs, int rows,
                                         v4d (&acc)[4]) {
  if (rows <= kB / 4) tile_mma_depth<kB / 4>(As, Bs, acc);
  else if (rows <= kB / 2) tile_mma_depth<kB / 2>(As, Bs, acc);
  else tile_mma_depth<kB>(As, Bs, acc);
}

// (row, column) within the 64 x 64 tile of element e of output tile t
__device__ __forceinline__ void tile_pos(int t, int e, int& r, int& c) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  r = 16 * w + 4 * e + (lane >> 4);
  c = 16 * t + (lane & 15);
}

// A 64 x 64 block (row-major, leading dimension ld, 16-byte aligned rows) to an LDS
// tile with row stride kS: 16-byte loads, all of a thread's in flight at once.
struct TileRegs {
  double2 v[kB * kB / 2 / kGemmThreads];
};
__device__ __forceinline__ void tile_fetch(const double* __restrict__ g, long long ld, TileRegs& t) {
#pragma unroll
  for (int m = 0; m < kB * kB / 2 / kGemmThreads; ++m) {
    const int q = threadIdx.x + m * kGemmThreads;
    t.v[m] = *reinterpret_cast<const double2*>(g + (long long)(q / (kB / 2)) * ld + 2 * (q % (kB / 2)));
  }
}
template <int kS>
__device__ __forceinline__ void tile_put(const TileRegs& t, double* __restrict__ s) {
#pragma unroll
  for (int m = 0; m < kB * kB / 2 / kGemmThreads; ++m) {
    const int q = threadIdx.x + m * kGemmThreads;
    *reinterpret_cast<double2*>(s + (q / (kB / 2)) * kS + 2 * (q % (kB / 2))) = t.v[m];
  }
}

// Dense n_pad x n_pad from CSR: one workgroup per row; the row is zeroed in LDS, then the
// thread of the first entry of each column adds that column's entries in order (repeated
// columns are adjacent where the columns are sorted, as a setup's own levels have them;
// else one thread adds the row up) and the row is written out. Padding rows are identity
// rows; a pinned DOF 0 keeps only a_00 = 1 in its row and column. A one-thread scatter of the row took 14.8 us at 450 rows.
// A level far from 1 (a_00 beyond 2^+-400) is scaled by a power of two, and its inverse
// with it in the last launch: the pivot blocks' 2 x 2 determinants would leave the range
// of doubles where the pivots do not. Entries may still differ by 30 orders and more.
constexpr int kFillThreads = 256;
__device__ __forceinline__ double range_scale(double a00) {
  if (!(fabs(a00) > 0.0 && fabs(a00) <= 1.7976931348623157e308)) return 1.0;
  const int e = ilogb(a00);
  return e >= -400 && e <= 400 ? 1.0 : ldexp(1.0, e > 0 ? -e : (e < -1000 ? 1000 : -e));
}
__global__ __launch_bounds__(kFillThreads) void k_fill_padded(int n, int n_pad, const int* __restrict__ rp,
                                                              const int* __restrict__ ci, const double* __restrict__ v,
                                                              const int* __restrict__ pin_flag, double* __restrict__ M) {
  extern __shared__ double row[];
  const int r = blockIdx.x;
  const int pin = *pin_flag;
  for (int c = threadIdx.x; c < n_pad; c += blockDim.x) row[c] = 0.0;
  __syncthreads();
  if (r >= n || (pin && r == 0)) {
    if (threadIdx.x == 0) row[r] = 1.0;
  } else {
    const int e0 = rp[r], e1 = rp[r + 1];
    const double scale = range_scale(*v);
    bool sorted = true;
    for (int e = e0 + 1 + threadIdx.x; e < e1; e += kFillThreads) sorted = sorted && ci[e - 1] <= ci[e];
    if (__syncthreads_and(sorted)) {
      for (int e = e0 + threadIdx.x; e < e1; e += kFillThreads) {
        const int c = ci[e];
        if ((e > e0 && ci[e - 1] == c) || (pin && c == 0)) continue;
        double sum = v[e];
        for (int q = e + 1; q < e1 && ci[q] == c; ++q) sum += v[q];
        row[c] = sum * scale;
      }
    } else if (threadIdx.x == 0) {
      for (int e = e0; e < e1; ++e)
        if (!(pin && ci[e] == 0)) row[ci[e]] += v[e] * scale;
    }
  }
  __syncthreads();
  for (int c = threadIdx.x; c < n_pad; c += blockDim.x) M[(long long)r * n_pad + c] = row[c];
}

// 1 / d to the last bit or one beside it: the hardware estimate and two Newton steps
// (a full division is a chain three times as long, and the elimination waits on it)
__device__ __forceinline__ double recip(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = fma(fma(-d, r, 1.0), r, r);
  return fma(fma(-d, r, 1.0), r, r);
}

// Inverse of the 2 x 2 matrix (a b; c d). ok: both elimination pivots a and
// d - c b / a = det / a exceed ta and tb.
struct M2 {
  double a, b, c, d;
};
__device__ __forceinline__ M2 inv2(const M2& m, double ta, double tb, bool& ok) {
  const double det = fma(m.a, m.d, -m.b * m.c);
  ok = ok && m.a > ta && det > tb * m.a;
  const double r = recip(det);
  return M2{m.d * r, -m.b * r, -m.c * r, m.a * r};
}
__device__ __forceinline__ M2 mul2(const M2& x, const M2& y) {
  return M2{fma(x.a, y.a, x.b * y.c), fma(x.a, y.b, x.b * y.d), fma(x.c, y.a, x.d * y.c), fma(x.c, y.b, x.d * y.d)};
}

// In-place inverse of the 64 x 64 block that one workgroup of four waves holds in the
// MFMA accumulator layout (tile_pos), by unpivoted Gauss-Jordan on 4 x 4 pivot
// blocks. Step q (pivot rows and columns 4q..4q+3): the pivot rows and columns pass
// through LDS (double-buffered, one barrier per step); every lane inverts the 4 x 4
// pivot block by 2 x 2 blocks (two reciprocals on the chain) and forms its entry of
// R = B^-1 A_Pj, which is at once the MFMA's B operand and, in the pivot rows, the
// result; the rank-4 update A_ij -= A_iP R_j is one v_mfma_f64_16x16x4_f64 per tile.
// Inside the pivot columns R is B^-1 and the old entries count as zero, which leaves
// -A_iP B^-1 there.
// What bounds it: the chain of 16 steps (exchange, two reciprocals, four MFMAs of 64
// cycles). The launch with one block: 31 -> 20 us against vector updates from one
// thread column each with four divisions per step.
// A pivot not above tol times its diagonal entry of dg (or above zero when dg is
// null) clears the return value. rows: the block's rows that belong to the matrix; the
// padding behind them is an identity and needs no step (at 83 rows 21 steps in all
// instead of 32, 60 -> 46 us for the whole inverse; 142 -> 134 us at 275).
constexpr int kGjLds = 2 * 4 * kB + 2 * kB * 4;
template <bool kPartial>
__device__ __forceinline__ bool invert_block_rows(v4d (&acc)[4], double* __restrict__ lds, const double* __restrict__ dg,
                                             double tol, int rows) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = lane & 15, kk = lane >> 4;
  double* rowb = lds;               // [2][4][64]
  double* colb = lds + 2 * 4 * kB;  // [2][64][4]
  bool ok = true;
  for (int q4 = 0; q4 < 4; ++q4) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int p0 = 16 * q4 + 4 * e;
      if (kPartial && p0 >= rows) return ok;  // uniform
      double* rb = rowb + (e & 1) * 4 * kB;
      double* cb = colb + (e & 1) * kB * 4;
      if (w == q4) {
#pragma unroll
        for (int t = 0; t < 4; ++t) rb[kk * kB + 16 * t + i] = acc[t][e];
      }
      const bool jp = (i >> 2) == e;  // in tile q4 this lane holds a pivot column
      if (jp) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          double v = acc[0][m];
          v = (q4 == 1) ? acc[1][m] : v;
          v = (q4 == 2) ? acc[2][m] : v;
          v = (q4 == 3) ? acc[3][m] : v;
          cb[(16 * w + 4 * m + kk) * 4 + (i & 3)] = v;
        }
      }
      __syncthreads();
      const double a_op = -cb[(16 * w + i) * 4 + kk];
      const M2 E{rb[p0], rb[p0 + 1], rb[kB + p0], rb[kB + p0 + 1]};
      const M2 F{rb[p0 + 2], rb[p0 + 3], rb[kB + p0 + 2], rb[kB + p0 + 3]};
      const M2 G{rb[2 * kB + p0], rb[2 * kB + p0 + 1], rb[3 * kB + p0], rb[3 * kB + p0 + 1]};
      const M2 H{rb[2 * kB + p0 + 2], rb[2 * kB + p0 + 3], rb[3 * kB + p0 + 2], rb[3 * kB + p0 + 3]};
      double rv[4][4];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int c = 0; c < 4; ++c) rv[t][c] = rb[c * kB + 16 * t + i];
      double t0 = 0.0, t1 = 0.0, t2 = 0.0, t3 = 0.0;
      if (dg) {
        t0 = tol * dg[p0];
        t1 = tol * dg[p0 + 1];
        t2 = tol * dg[p0 + 2];
        t3 = tol * dg[p0 + 3];
      }
      // B^-1 from the Schur complement of its leading 2 x 2 block
      const M2 Ei = inv2(E, t0, t1, ok);
      const M2 T = mul2(G, Ei), U = mul2(Ei, F);
      const M2 TF = mul2(T, F);
      const M2 Si = inv2(M2{H.a - TF.a, H.b - TF.b, H.c - TF.c, H.d - TF.d}, t2, t3, ok);
      const M2 US = mul2(U, Si), ST = mul2(Si, T);
      const M2 UST = mul2(US, T);
      // row kk of B^-1
      const bool hi = kk >= 2, odd = (kk & 1) != 0;
      double b0 = hi ? (odd ? -ST.c : -ST.a) : (odd ? Ei.c + UST.c : Ei.a + UST.a);
      double b1 = hi ? (odd ? -ST.d : -ST.b) : (odd ? Ei.d + UST.d : Ei.b + UST.b);
      double b2 = hi ? (odd ? Si.c : Si.a) : (odd ? -US.c : -US.a);
      double b3 = hi ? (odd ? Si.d : Si.b) : (odd ? -US.d : -US.b);
      const double bj = (i & 2) ? ((i & 1) ? b3 : b2) : ((i & 1) ? b1 : b0);
      double R[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const double v = fma(b0, rv[t][0], b1 * rv[t][1]) + fma(b2, rv[t][2], b3 * rv[t][3]);
        const bool piv = jp && t == q4;
        R[t] = piv ? bj : v;
#pragma unroll
        for (int m = 0; m < 4; ++m) acc[t][m] = piv ? 0.0 : acc[t][m];
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a_op, R[t], acc[t], 0, 0, 0);
        if (w == q4) acc[t][e] = R[t];
      }
    }
  }
  return ok;
}
// The exit test inside the unrolled steps costs a full block 3 us: two forms.
__device__ __forceinline__ bool invert_block(v4d (&acc)[4], double* __restrict__ lds, const double* __restrict__ dg,
                                             double tol, int rows) {
  return rows >= kB ? invert_block_rows<false>(acc, lds, dg, tol, rows)
                    : invert_block_rows<true>(acc, lds, dg, tol, rows);
}

// Block 0: the inverse of the first 64 x 64 pivot block, into P (leading dimension
// 64; straight into the result, with its transpose PT, when the matrix has no other
// block). Blocks 1..: with
// sym_rows > 0, block b checks row b - 1 for symmetry, |a_ij - a_ji| <= 1e-10
// sqrt(a_ii a_jj) (the rounding asymmetry of a Galerkin product passes, a
// non-symmetric operator does not; well rows can exceed interior rows by 15 orders,
// so the scale is per entry), and for a positive diagonal, and keeps the diagonal. a00:
// the level's first entry, from which a result takes its scale (range_scale).
__global__ __launch_bounds__(kGemmThreads) void k_gj_diag(int n, int n_pad, int sym_rows, const double* __restrict__ M,
                                                          double* __restrict__ P, double* __restrict__ PT,
                                                          double* __restrict__ dg, double tol,
                                                          int* __restrict__ bad, const double* __restrict__ a00) {
  if (blockIdx.x > 0) {
    const int r = blockIdx.x - 1;
    const double dr = M[(long long)r * n_pad + r];
    bool wrong = !(dr > 0.0);
    for (int c = threadIdx.x; c < r; c += blockDim.x) {
      const double d = fabs(M[(long long)r * n_pad + c] - M[(long long)c * n_pad + r]);
      const double dc = M[(long long)c * n_pad + c];
      wrong = wrong || !(d <= 1e-10 * sqrt(fabs(dr) * fabs(dc)));
    }
    if (wrong) *bad = 1;
    return;
  }
  __shared__ double lds[kGjLds];
  __shared__ double d0[kB];
  if (dg)
    for (int r = threadIdx.x; r < n_pad; r += blockDim.x) {
      const double d = M[(long long)r * n_pad + r];
      dg[r] = d;
      if (r < kB) d0[r] = d;
    }
  v4d acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int r, c;
      tile_pos(t, e, r, c);
      acc[t][e] = M[(long long)r * n_pad + c];
    }
  __syncthreads();
  if (!invert_block(acc, lds, dg ? d0 : nullptr, tol, min(n, kB))) *bad = 1;
  const double scale = PT ? range_scale(*a00) : 1.0;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int r, c;
      tile_pos(t, e, r, c);
      const double x = acc[t][e] * scale;
      P[r * kB + c] = x;
      if (PT) PT[c * kB + r] = x;
    }
}

// One elimination step from A into A' (see the header), one workgroup per block
// (blockIdx.x = j, blockIdx.y = i). Every block of column j != k forms P A_kj
// itself with the same MFMA sequence, so the row panel it subtracts equals the one
// its own row-k block stores. The longest path of a launch is the workgroup that
// also inverts the next pivot block (fetches, two products of 1.7 us, the inverse);
// every tile it needs is fetched before the first product. The last block column
// also scales the inverse (a00, range_scale) and writes its transpose (AnT). One launch per block
// column: 47-49 -> 13-24 us at 83-576 rows.
__global__ __launch_bounds__(kGemmThreads) void k_gj_step(int k, int n, int n_pad, const double* __restrict__ A,
                                                          double* __restrict__ An, const double* __restrict__ P,
                                                          double* __restrict__ Pn, double* __restrict__ AnT,
                                                          const double* __restrict__ dg, double tol,
                                                          int* __restrict__ bad, const double* __restrict__ a00) {
  __shared__ double As[kB * kLdA], Bs[kB * kLdB], Cs[kB * kLdA];
  __shared__ double d0[kB];  // the next pivot block's entries of dg
  const int j = blockIdx.x, i = blockIdx.y;
  const double* blk = A + (long long)i * kB * n_pad + (long long)j * kB;
  double* out = An + (long long)i * kB * n_pad + (long long)j * kB;
  double* outT = AnT ? AnT + (long long)j * kB * n_pad + (long long)i * kB : nullptr;
  const double scale = AnT ? range_scale(*a00) : 1.0;
  if (i == k && j == k) {
    for (int q = threadIdx.x; q < kB * kB; q += blockDim.x) {
      const double x = P[q] * scale;
      out[(long long)(q / kB) * n_pad + q % kB] = x;
      if (outT) outT[(long long)(q % kB) * n_pad + q / kB] = x;
    }
    return;
  }
  v4d acc[4];
  TileRegs ta, tb;
  // inner indices past the matrix's last row meet zeros: of A_ik, and of P left of its
  // identity
  const int depth = n - k * kB;
  if (j == k) {  // A'_ik = -A_ik P
    tile_fetch(blk, n_pad, ta);
    tile_fetch(P, kB, tb);
    tile_put<kLdA>(ta, As);
    tile_put<kLdB>(tb, Bs);
    __syncthreads();
    tile_mma(As, Bs, depth, acc);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        int r, c;
        tile_pos(t, e, r, c);
        const double x = -acc[t][e] * scale;
        out[(long long)r * n_pad + c] = x;
        if (outT) outT[(long long)c * n_pad + r] = x;
      }
    return;
  }
  tile_fetch(P, kB, ta);
  tile_fetch(A + (long long)k * kB * n_pad + (long long)j * kB, n_pad, tb);
  if (i == k) {
    tile_put<kLdA>(ta, As);
    tile_put<kLdB>(tb, Bs);
    __syncthreads();
    tile_mma(As, Bs, depth, acc);  // P A_kj
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        int r, c;
        tile_pos(t, e, r, c);
        const double x = acc[t][e] * scale;
        out[(long long)r * n_pad + c] = x;
        if (outT) outT[(long long)c * n_pad + r] = x;
      }
    return;
  }
  if (dg && i == k + 1 && threadIdx.x < kB) d0[threadIdx.x] = dg[(long long)i * kB + threadIdx.x];
  TileRegs tc;
  tile_fetch(A + (long long)i * kB * n_pad + (long long)k * kB, n_pad, tc);
  v4d own[4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int r, c;
      tile_pos(t, e, r, c);
      own[t][e] = blk[(long long)r * n_pad + c];
    }
  tile_put<kLdA>(ta, As);
  tile_put<kLdB>(tb, Bs);
  tile_put<kLdA>(tc, Cs);
  __syncthreads();
  tile_mma(As, Bs, depth, acc);  // P A_kj
  __syncthreads();        // every wave is done reading Bs
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int r, c;
      tile_pos(t, e, r, c);
      Bs[r * kLdB + c] = acc[t][e];
    }
  __syncthreads();
  tile_mma(Cs, Bs, depth, acc);  // A_ik (P A_kj)
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int r, c;
      tile_pos(t, e, r, c);
      own[t][e] -= acc[t][e];
      out[(long long)r * n_pad + c] = own[t][e] * scale;
      if (outT) outT[(long long)c * n_pad + r] = own[t][e] * scale;
    }
  if (i != k + 1 || j != k + 1 || Pn == nullptr) return;
  // this block is the next step's pivot block: its inverse goes to step k + 1 in Pn
  // (As is free: every wave has passed the barrier behind its last read of it)
  if (!invert_block(own, As, dg ? d0 : nullptr, tol, min(n - i * kB, kB))) *bad = 1;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int r, c;
      tile_pos(t, e, r, c);
      Pn[r * kB + c] = own[t][e];
    }
}

// x = A^-1 b (b_0 taken as 0 when DOF 0 is pinned): a wavefront per row, four
// independent partial sums per lane (four loads in flight), folded at the end.
template <class T>
__global__ __launch_bounds__(256) void k_dense_mv(int n, int n_pad, const int* __restrict__ pin_flag,
                                                  const double* __restrict__ M, const T* __restrict__ b,
                                                  T* __restrict__ x) {
  const int pin = *pin_flag;
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = (blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int nwaves = (gridDim.x * blockDim.x) / kWave;
  for (int r = wid; r < n; r += nwaves) {
    const double* row = M + (long long)r * n_pad;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int c = (pin ? 1 : 0) + lane;
    for (; c + 3 * kWave < n; c += 4 * kWave) {
      s0 += row[c] * (double)b[c];
      s1 += row[c + kWave] * (double)b[c + kWave];
      s2 += row[c + 2 * kWave] * (double)b[c + 2 * kWave];
      s3 += row[c + 3 * kWave] * (double)b[c + 3 * kWave];
    }
    for (; c < n; c += kWave) s0 += row[c] * (double)b[c];
    const double s = wave_sum((s0 + s1) + (s2 + s3));
    if (lane == 0) x[r] = (T)s;
  }
}

}  // namespace

int dense_pad(int n) { return div_up(n, kB) * kB; }

void launch_dense_inverse_mfma(int n, const int* rp, const int* ci, const double* v, const int* pin, double* M,
                               double* W, double* P, int* bad, hipStream_t s) {
  IMPES_REQUIRE(n >= 1 && n <= kDenseMfmaMax, "MFMA dense inverse supports 1 <= n <= 4096");
  const int n_pad = dense_pad(n), nb = n_pad / kB;
  double* MT = M + (long long)n_pad * n_pad;
  // small operators are checked for symmetry and their pivots against the diagonal
  // (a pivot of rounding size: not numerically SPD), so that a failed check reaches
  // the pivoted elimination; larger ones for positive pivots only
  const bool strict = n <= kDenseStrictMax;
  const double tol = strict ? 1e-13 : 0.0;
  double* dg = strict ? P + 2 * kB * kB : nullptr;
  // each step swaps the two matrices: start where nb steps end in M
  double* cur = (nb % 2 == 0) ? M : W;
  double* nxt = (nb % 2 == 0) ? W : M;
  k_fill_padded<<<n_pad, kFillThreads, n_pad * sizeof(double), s>>>(n, n_pad, rp, ci, v, pin, cur);
  IMPES_LAUNCH_CHECK();
  // P holds two 64 x 64 pivot inverses: step k reads P_k and its block (k+1, k+1)
  // workgroup writes P_{k+1} into the other half. With one block its inverse is the
  // result (n_pad = 64 = the leading dimension of P).
  k_gj_diag<<<1 + (strict ? n : 0), kGemmThreads, 0, s>>>(n, n_pad, strict ? n : 0, cur, nb == 1 ? M : P,
                                                              nb == 1 ? MT : nullptr, dg, tol, bad, v);
  IMPES_LAUNCH_CHECK();
  if (nb == 1) return;
  for (int k = 0; k < nb; ++k) {
    double* Pk = P + (k & 1) * kB * kB;
    double* Pn = (k + 1 < nb) ? P + ((k + 1) & 1) * kB * kB : nullptr;
    k_gj_step<<<dim3(nb, nb), kGemmThreads, 0, s>>>(k, n, n_pad, cur, nxt, Pk, Pn, k + 1 == nb ? MT : nullptr, dg,
                                                    tol, bad, v);
    IMPES_LAUNCH_CHECK();
    std::swap(cur, nxt);
  }
}

void launch_dense_mv_f64(int n, const int* pin, const double* M, const double* b, double* x, hipStream_t s) {
  k_dense_mv<double><<<div_up(n, 4), 256, 0, s>>>(n, dense_pad(n), pin, M, b, x);
  IMPES_LAUNCH_CHECK();
}

void launch_dense_mv_f32(int n, const int* pin, const double* M, const float* b, float* x, hipStream_t s) {
  k_dense_mv<float><<<div_up(n, 4), 256, 0, s>>>(n, dense_pad(n), pin, M, b, x);
  IMPES_LAUNCH_CHECK();
}

}  // namespace impes
