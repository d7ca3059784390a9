// Sparse operator kernels of the V-cycle and of the outer Krylov method.
//
// CSR: G lanes of a wavefront share one row (G = 1..64 chosen from the mean row
// length), lanes walk the row with stride G so a group's loads are contiguous,
// and the partial sums fold with cross-lane shuffles. Every variant is fused
// with the vector update it feeds (residual, L1-Jacobi sweep, prolongation
// add, row scaling) so each sweep streams the matrix once.
//
// Stencil7: the level-0 IMPES pressure operator is a symmetric 7-point stencil,
// so it is stored index-free as one diagonal and three face-coefficient arrays
// (4 values per cell instead of CSR's ~7 values + 7 indices + row pointers).
#include <cstdint>
#include <cstdlib>
#include <type_traits>

#include "kernels.h"
#include "ktimer.h"

namespace impes {

namespace {
constexpr int kBlock = 256;

// kRestrictJ0: y = A x (a restriction R r) and y2 = w * aux .* y (the first
// L1-Jacobi sweep of the coarse level from a zero guess, aux = its inv_relax)
// kYPlusB: y = b + A x (an add into another buffer; same arithmetic as kYAdd)
// kJacZ0 (stencil): two L1-Jacobi sweeps from a zero guess in one pass: the first
// sweep's x = w * aux .* b is formed at every stencil point instead of being read
// (the expression of k_jacobi0), then y = x + w * aux .* (b - A x) as kJac
// kProlongJac (padded tiles): y = y2 + w * aux .* b + A x, the prolongation and the first
// L1-Jacobi sweep after it with A = P - w diag(aux) (A_l P), x the coarse correction, b
// the residual and y2 the iterate before the correction (y may be y2)
enum Mode {
  kY = 0, kYAdd = 1, kRes = 2, kJac = 3, kRowScaled = 4, kRowScaledRes = 5, kRestrictJ0 = 6, kYPlusB = 7, kJacZ0 = 8,
  kProlongJac = 9
};

template <int G, class T, class TA, int MODE>
__global__ __launch_bounds__(kBlock) void k_csr(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                                                 const T* __restrict__ v, const T* __restrict__ x,
                                                 const T* __restrict__ b, const TA* __restrict__ aux, T w,
                                                 T* __restrict__ y, T* __restrict__ y2) {
  constexpr int RPB = kBlock / G;  // rows per block
  const int g = threadIdx.x % G;
  for (long long base = xcd_block() * RPB; base < n; base += (long long)gridDim.x * RPB) {
    const long long row = base + threadIdx.x / G;
    const bool active = row < n;
    // the row's own operands are loaded before the row walk, so their latency
    // overlaps the (row pointer -> column -> gather) chain instead of following it
    T ob = T(0), ox = T(0), oy = T(0), oa = T(0);
    if (active && g == 0) {
      if (MODE == kYPlusB || MODE == kRes || MODE == kJac || MODE == kRowScaledRes) ob = b[row];
      if (MODE == kJac) ox = x[row];
      if (MODE == kYAdd) oy = y[row];
      if (MODE == kJac || MODE == kRowScaled || MODE == kRowScaledRes || MODE == kRestrictJ0) oa = (T)aux[row];
    }
    T sum = T(0);
    if (active) {
      const int e1 = rp[row + 1];
#pragma unroll 4
      for (int e = rp[row] + g; e < e1; e += G) sum += v[e] * x[ci[e]];
    }
    if (G > 1) sum = group_sum<G>(sum);
    if (active && g == 0) {
      if (MODE == kY) y[row] = sum;
      else if (MODE == kYAdd) y[row] = oy + sum;
      else if (MODE == kYPlusB) y[row] = ob + sum;
      else if (MODE == kRes) y[row] = ob - sum;
      else if (MODE == kJac) y[row] = ox + w * oa * (ob - sum);
      else if (MODE == kRowScaled) y[row] = oa * sum;
      else if (MODE == kRowScaledRes) y[row] = oa * (ob - sum);
      else if (MODE == kRestrictJ0) {
        y[row] = sum;
        y2[row] = w * oa * sum;
      }
    }
  }
}

// Padded FP32 CSR (Csr4F32): G lanes per row, each lane 4 entries per 16-byte load.
template <int G, int MODE, bool OFF16>
__global__ __launch_bounds__(kBlock) void k_csr4(int n, const int* __restrict__ rp4, const int4* __restrict__ ci4,
                                                  const short4* __restrict__ co4, const float4* __restrict__ v4,
                                                  const float* __restrict__ x, const float* __restrict__ b,
                                                  const float* __restrict__ aux, float w, float* __restrict__ y) {
  constexpr int RPB = kBlock / G;
  const int g = threadIdx.x % G;
  for (long long base = xcd_block() * RPB; base < n; base += (long long)gridDim.x * RPB) {
    const long long row = base + threadIdx.x / G;
    const bool active = row < n;
    // the row's own operands are loaded before the row walk (as in k_csr)
    float ob = 0.f, ox = 0.f, oa = 0.f;
    if (active && g == 0) {
      ob = b[row];
      if (MODE == kJac) {
        ox = x[row];
        oa = aux[row];
      }
    }
    float sum = 0.f;
    if (active) {
      const int q1 = rp4[row + 1] >> 2;
#pragma unroll 2
      for (int q = (rp4[row] >> 2) + g; q < q1; q += G) {
        const float4 a = v4[q];
        int4 c;
        if (OFF16) {
          const short4 o = co4[q];
          const int r = (int)row;
          c = make_int4(r + o.x, r + o.y, r + o.z, r + o.w);
        } else {
          c = ci4[q];
        }
        sum += a.x * x[c.x];
        sum += a.y * x[c.y];
        sum += a.z * x[c.z];
        sum += a.w * x[c.w];
      }
    }
    if (G > 1) sum = group_sum<G>(sum);
    if (active && g == 0) {
      if (MODE == kRes) y[row] = ob - sum;
      else y[row] = ox + w * oa * (ob - sum);
    }
  }
}

// Padded FP32 CSR over wave tiles: a wave takes one tile of 64 four-entry chunks, one
// per lane, so no lane idles on a short row. A lane's row and its place in the row
// come with the chunk (tag), and the tile's address from its number alone, so all of
// a tile's operator loads issue at once and the gathers wait on nothing else; the
// lanes of a row add up by a segmented scan of as many steps as the tile's longest
// row needs, and the row's last lane applies the update.
// What bounds it: the chain of dependent loads per wave at full occupancy
// (operator -> gather -> update), then the gathers. The first tiled form (tiles of
// whole rows packed without gaps) read each tile's bounds first, found the lane's row
// by six dependent shuffles over a load of the row starts, and scanned six steps of
// two shuffles: 8.6 -> 7.6 us per sweep over the 1M-cell hierarchy's levels (level 1,
// 58 MB: 15.2 -> 13.7 us), 4.2 -> 3.6 us over the 200k-cell hierarchy's; the sums are
// the same bits.
// FP64 values (two 16-byte loads per chunk) serve the FP64 cycle: against a group of lanes
// per CSR row, sweeps over 116,000 rows 9.6 -> 7.4 us, over 35,000 rows of 29 entries
// 8.4 -> 6.3 us.
template <class T>
__device__ __forceinline__ void ld_chunk(const T* __restrict__ v, long long q, T (&a)[4]) {
#pragma unroll
  for (int h = 0; h < 4 * (int)sizeof(T) / 16; ++h)
    __builtin_memcpy(reinterpret_cast<unsigned char*>(a) + 16 * h,
                     __builtin_assume_aligned(reinterpret_cast<const unsigned char*>(v + 4 * q) + 16 * h, 16), 16);
}

template <class T, int MODE, bool OFF16>
__global__ __launch_bounds__(kBlock) void k_csr4_tile(int nw, const int* __restrict__ wrow,
                                                       const unsigned short* __restrict__ tag,
                                                       const int4* __restrict__ ci4, const short4* __restrict__ co4,
                                                       const T* __restrict__ v4, const T* __restrict__ x,
                                                       const T* __restrict__ b, const T* __restrict__ aux, T w, T* y,
                                                       T* y2) {
  constexpr int WPB = kBlock / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  for (int t = (int)xcd_block() * WPB + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave); t < nw;
       t += gridDim.x * WPB) {
    const long long q = (long long)t * kWave + lane;
    T a[4];
    ld_chunk(v4, q, a);
    const unsigned tg = tag[q];
    int4 c;
    short4 o;
    if (OFF16) o = co4[q];
    else c = ci4[q];
    const int row = wrow[t] + (int)(tg & 63u);
    const int pos = (int)(tg >> 6 & 63u);
    const bool last = (tg >> 12) != 0;
    if (OFF16) c = make_int4(row + o.x, row + o.y, row + o.z, row + o.w);
    T ob = T(0), ox = T(0), oa = T(0);
    if (last) {
      if (MODE == kRes || MODE == kJac || MODE == kProlongJac) ob = b[row];
      if (MODE == kJac) ox = x[row];
      if (MODE == kProlongJac) ox = y2[row];
      if (MODE == kJac || MODE == kRestrictJ0 || MODE == kProlongJac) oa = aux[row];
    }
    T sum = T(0);
    sum += a[0] * x[c.x];
    sum += a[1] * x[c.y];
    sum += a[2] * x[c.z];
    sum += a[3] * x[c.w];
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      if (!__any(pos >= d)) break;  // uniform
      const T u = __shfl_up(sum, d, kWave);
      if (pos >= d) sum += u;
    }
    if (last) {
      if (MODE == kRes) y[row] = ob - sum;
      else if (MODE == kJac) y[row] = ox + w * oa * (ob - sum);
      else if (MODE == kProlongJac) y[row] = (ox + w * oa * ob) + sum;
      else if (MODE == kY) y[row] = sum;
      else if (MODE == kRestrictJ0) {
        y[row] = sum;
        y2[row] = w * oa * sum;
      }
    }
  }
}

// chunks of row r (an empty row has one)
__device__ __forceinline__ int row_chunks(const int* __restrict__ rp, int r) {
  const int len = rp[r + 1] - rp[r];
  return len > 0 ? (len + 3) >> 2 : 1;
}

// Greedy tiles of one segment, a wave each: per tile the wave looks at the next 64
// rows and takes those whose chunks fit. FILL writes the tiles' first rows and the
// rows' first entries, else the segment's tile count.
template <bool FILL>
__global__ __launch_bounds__(kBlock) void k_tile4_rows(int n, const int* __restrict__ rp,
                                                       const long long* __restrict__ base, int* __restrict__ cnt,
                                                       int* __restrict__ wrow, int* __restrict__ rp4) {
  const int seg = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int r0 = seg * kTileSeg, r1 = min(n, r0 + kTileSeg);
  if (r0 >= n) return;
  long long t = FILL ? base[seg] : 0;
  for (int r = r0; r < r1;) {
    const int mine = r + lane;
    const int c = mine < r1 ? row_chunks(rp, mine) : kWave + 1;
    int sum = c;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int u = __shfl_up(sum, d, kWave);
      if (lane >= d) sum += u;
    }
    const int take = __popcll(__ballot(mine < r1 && sum <= kWave));
    if (take == 0) {  // a row longer than a tile
      if (!FILL && lane == 0) cnt[seg] = kTileNone;
      return;
    }
    if (FILL) {
      if (lane == 0) wrow[t] = r;
      if (lane < take) rp4[mine] = (int)((t * kWave + sum - c) * 4);
    }
    r += take;
    ++t;
  }
  if (!FILL && lane == 0) cnt[seg] = (int)t;
  if (FILL && r1 == n && lane == 0) wrow[t] = n;
}

// One tile per wave: every lane finds its chunk's row among the tile's row starts
__global__ __launch_bounds__(kBlock) void k_tile4_fill(int nw, const int* __restrict__ wrow,
                                                       const int* __restrict__ rp, const int* __restrict__ ci,
                                                       const double* __restrict__ v, const int* __restrict__ rp4,
                                                       int4* __restrict__ ci4, short4* __restrict__ co4,
                                                       float4* __restrict__ v4, unsigned short* __restrict__ tag,
                                                       int* __restrict__ maxabs, int square) {
  const int lane = threadIdx.x & (kWave - 1);
  int far = 0;
  for (int t = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; t < nw; t += gridDim.x * (kBlock / kWave)) {
    const int r0 = wrow[t], nr = wrow[t + 1] - r0;
    const int q0 = t * kWave;
    // first chunk, relative to the tile, of row r0 + 1 + lane (64: no such row)
    const int ps = (lane + 1 < nr) ? (rp4[r0 + 1 + lane] >> 2) - q0 : kWave;
    int lo = 0;
#pragma unroll
    for (int st = kWave / 2; st >= 1; st >>= 1) {
      const int pc = __shfl(ps, lo + st - 1, kWave);
      if (pc <= lane) lo += st;
    }
    const int row = r0 + lo;
    const int e0 = rp[row], len = rp[row + 1] - e0;
    const int pos = q0 + lane - (rp4[row] >> 2), chunks = row_chunks(rp, row);
    const bool used = pos < chunks;
    const int pad = square ? row : (len > 0 ? ci[e0] : 0);
    int c[4];
    float a[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int k = 4 * pos + m;
      const bool in = used && k < len;
      c[m] = in ? ci[e0 + k] : pad;
      a[m] = in ? (float)v[e0 + k] : 0.f;
      far = max(far, abs(c[m] - row));
    }
    const long long q = (long long)q0 + lane;
    ci4[q] = make_int4(c[0], c[1], c[2], c[3]);
    v4[q] = make_float4(a[0], a[1], a[2], a[3]);
    if (co4) {
      short o[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) o[m] = (short)max(-32768, min(32767, c[m] - row));
      co4[q] = make_short4(o[0], o[1], o[2], o[3]);
    }
    tag[q] = (unsigned short)(used ? (lo | pos << 6 | (pos + 1 == chunks ? 1 << 12 : 0)) : lo);
  }
  if (!maxabs) return;
  far = wave_max(far);
  if (lane == 0 && far > 0) atomicMax(maxabs, far);
}

// FP64 values of a tiled matrix from its CSR values
__global__ __launch_bounds__(kBlock) void k_tile4_values_f64(int nw, const int* __restrict__ wrow,
                                                             const unsigned short* __restrict__ tag,
                                                             const int* __restrict__ rp4, const int* __restrict__ rp,
                                                             const double* __restrict__ v, double2* __restrict__ v8) {
  const int lane = threadIdx.x & (kWave - 1);
  for (int t = (int)xcd_block() * (kBlock / kWave) + threadIdx.x / kWave; t < nw; t += gridDim.x * (kBlock / kWave)) {
    const long long q = (long long)t * kWave + lane;
    const unsigned tg = tag[q];
    const int row = wrow[t] + (int)(tg & 63u), pos = (int)(tg >> 6 & 63u);
    const bool used = (rp4[row] >> 2) + pos == q;  // not a spare chunk at the tile's end
    const int e0 = rp[row] + 4 * pos, e1 = used ? rp[row + 1] : 0;
    double a[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) a[m] = e0 + m < e1 ? v[e0 + m] : 0.0;
    v8[2 * q] = make_double2(a[0], a[1]);
    v8[2 * q + 1] = make_double2(a[2], a[3]);
  }
}

// Values of a tiled P - w diag(ir) AP on AP's pattern (P's is part of it: A has its
// diagonal): a lane per chunk, its row's few entries of P compared with the chunk's four
// columns. Formed in FP64, rounded once for FP32. miss (or null): adds the entries of P that AP's
// pattern lacks (a row without a diagonal entry).
template <class T>
__global__ __launch_bounds__(kBlock) void k_tile4_prolong_sweep(int nw, const int* __restrict__ wrow,
                                                                const unsigned short* __restrict__ tag,
                                                                const int* __restrict__ rp4,
                                                                const int4* __restrict__ ci4,
                                                                const int* __restrict__ aprp,
                                                                const double* __restrict__ apv,
                                                                const int* __restrict__ prp,
                                                                const int* __restrict__ pci,
                                                                const double* __restrict__ pv,
                                                                const double* __restrict__ ir, double w,
                                                                T* __restrict__ v4, int* __restrict__ miss) {
  const int lane = threadIdx.x & (kWave - 1);
  int lack = 0;
  for (int t = (int)xcd_block() * (kBlock / kWave) + threadIdx.x / kWave; t < nw; t += gridDim.x * (kBlock / kWave)) {
    const long long q = (long long)t * kWave + lane;
    const unsigned tg = tag[q];
    const int4 c4 = ci4[q];
    const int row = wrow[t] + (int)(tg & 63u), pos = (int)(tg >> 6 & 63u);
    const bool used = (rp4[row] >> 2) + pos == q;  // not a spare chunk at the tile's end
    const int e0 = aprp[row] + 4 * pos, e1 = used ? aprp[row + 1] : 0, p0 = prp[row], p1 = prp[row + 1];
    const double s = w * ir[row];
    const int c[4] = {c4.x, c4.y, c4.z, c4.w};
    double a[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) a[m] = e0 + m < e1 ? -s * apv[e0 + m] : 0.0;
    for (int e = p0; e < p1; ++e) {
      const int col = pci[e];
      const double v = pv[e];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const bool hit = e0 + m < e1 && c[m] == col;
        a[m] += hit ? v : 0.0;
        lack -= hit ? 1 : 0;
      }
    }
    if (tg >> 12) lack += p1 - p0;
    if constexpr (sizeof(T) == 4) {
      reinterpret_cast<float4*>(v4)[q] = make_float4((float)a[0], (float)a[1], (float)a[2], (float)a[3]);
    } else {
      reinterpret_cast<double2*>(v4)[2 * q] = make_double2(a[0], a[1]);
      reinterpret_cast<double2*>(v4)[2 * q + 1] = make_double2(a[2], a[3]);
    }
  }
  if (!miss) return;
  lack = wave_sum(lack);
  if (lane == 0 && lack != 0) atomicAdd(miss, lack);
}

template <int MODE, bool OFF16>
void csr4_tile_launch(const Csr4F32& A, const float* x, const float* b, const float* aux, float w, float* y,
                      hipStream_t s, float* y2 = nullptr) {
  const int grid = grid_for(A.nw, kBlock / kWave, 1 << 18);
  klaunch(k_csr4_tile<float, MODE, OFF16>, dim3(grid), dim3(kBlock), 0, s, A.nw, A.wrow, A.tag, A.ci4, A.co4,
          reinterpret_cast<const float*>(A.v4), x, b, aux, w, y, y2);
}

// the same pattern with FP64 values v8
template <int MODE>
void csr4_tile_f64(const Csr4F32& A, const double* v8, const double* x, const double* b, const double* aux, double w,
                   double* y, hipStream_t s, double* y2 = nullptr) {
  if (A.n <= 0) return;
  IMPES_REQUIRE(A.nw > 0 && ((uintptr_t)v8 & 15) == 0, "FP64 tiles: aligned values of a tiled pattern required");
  const int grid = grid_for(A.nw, kBlock / kWave, 1 << 18);
  if (A.co4)
    klaunch(k_csr4_tile<double, MODE, true>, dim3(grid), dim3(kBlock), 0, s, A.nw, A.wrow, A.tag, A.ci4, A.co4, v8, x,
            b, aux, w, y, y2);
  else
    klaunch(k_csr4_tile<double, MODE, false>, dim3(grid), dim3(kBlock), 0, s, A.nw, A.wrow, A.tag, A.ci4, A.co4, v8, x,
            b, aux, w, y, y2);
  IMPES_LAUNCH_CHECK();
}

template <int MODE, bool OFF16>
void csr4_launch(const Csr4F32& A, int G, const float* x, const float* b, const float* aux, float w, float* y,
                 hipStream_t s) {
  const int grid = grid_for(A.n, kBlock / G, 1 << 18);
#define IMPES_CSR4_CASE(GG)                                                                                     \
  case GG:                                                                                                     \
    klaunch(k_csr4<GG, MODE, OFF16>, dim3(grid), dim3(kBlock), 0, s, A.n, A.rp4, A.ci4, A.co4, A.v4, x, b, aux, \
            w, y);                                                                                             \
    break;
  switch (G) {
    IMPES_CSR4_CASE(1)
    IMPES_CSR4_CASE(2)
    IMPES_CSR4_CASE(4)
    IMPES_CSR4_CASE(8)
    IMPES_CSR4_CASE(16)
    IMPES_CSR4_CASE(32)
    default:
      klaunch(k_csr4<64, MODE, OFF16>, dim3(grid), dim3(kBlock), 0, s, A.n, A.rp4, A.ci4, A.co4, A.v4, x, b, aux,
              w, y);
      break;
  }
#undef IMPES_CSR4_CASE
  IMPES_LAUNCH_CHECK();
}

template <int MODE>
void csr4_dispatch(const Csr4F32& A, int G, const float* x, const float* b, const float* aux, float w, float* y,
                   hipStream_t s) {
  if (A.n <= 0) return;
  IMPES_REQUIRE(((uintptr_t)A.ci4 & 15) == 0 && ((uintptr_t)A.v4 & 15) == 0, "padded CSR: arrays not 16-byte aligned");
  if (A.co4) IMPES_REQUIRE(((uintptr_t)A.co4 & 7) == 0, "padded CSR: offsets not 8-byte aligned");
  if (A.nw > 0) {
    if (A.co4) csr4_tile_launch<MODE, true>(A, x, b, aux, w, y, s);
    else csr4_tile_launch<MODE, false>(A, x, b, aux, w, y, s);
  } else if (A.co4) {
    csr4_launch<MODE, true>(A, G, x, b, aux, w, y, s);
  } else {
    csr4_launch<MODE, false>(A, G, x, b, aux, w, y, s);
  }
}

__global__ void k_csr4_count(int n, const int* __restrict__ rp, int* __restrict__ cnt) {
  for (long long r = blockIdx.x * (long long)blockDim.x + threadIdx.x; r < n; r += (long long)gridDim.x * blockDim.x)
    cnt[r] = max(4, (rp[r + 1] - rp[r] + 3) & ~3);
}

__global__ void k_csr4_pattern(int n, const int* __restrict__ rp, const int* __restrict__ ci,
                               const int* __restrict__ rp4, int* __restrict__ ci4) {
  for (long long r = blockIdx.x * (long long)blockDim.x + threadIdx.x; r < n; r += (long long)gridDim.x * blockDim.x) {
    const int e0 = rp[r], len = rp[r + 1] - e0, q0 = rp4[r], len4 = rp4[r + 1] - q0;
    for (int k = 0; k < len4; ++k) ci4[q0 + k] = (k < len) ? ci[e0 + k] : (int)r;
  }
}

__global__ void k_csr4_offsets(int n, const int* __restrict__ rp4, const int* __restrict__ ci4,
                               short* __restrict__ co4, int* __restrict__ maxabs) {
  int m = 0;
  for (long long r = blockIdx.x * (long long)blockDim.x + threadIdx.x; r < n; r += (long long)gridDim.x * blockDim.x) {
    for (int e = rp4[r]; e < rp4[r + 1]; ++e) {
      const int d = ci4[e] - (int)r;
      m = max(m, abs(d));
      co4[e] = (short)max(-32768, min(32767, d));
    }
  }
  m = wave_max(m);
  if ((threadIdx.x & (kWave - 1)) == 0 && m > 0) atomicMax(maxabs, m);
}

// G lanes per row (entries strided by G): consecutive lanes write consecutive entries
template <int G>
__global__ void k_csr4_values(int n, const int* __restrict__ rp, const double* __restrict__ v,
                              const int* __restrict__ rp4, float* __restrict__ v4) {
  const int g = threadIdx.x % G;
  for (long long r = (blockIdx.x * (long long)blockDim.x + threadIdx.x) / G; r < n;
       r += (long long)gridDim.x * blockDim.x / G) {
    const int e0 = rp[r], len = rp[r + 1] - e0, q0 = rp4[r], len4 = rp4[r + 1] - q0;
    for (int k = g; k < len4; k += G) v4[q0 + k] = (k < len) ? (float)v[e0 + k] : 0.f;
  }
}

template <class T, class TA, int MODE>
void csr_dispatch(int n, const int* rp, const int* ci, const T* v, const T* x, const T* b, const TA* aux, T w, T* y,
                  int G, hipStream_t s, T* y2 = nullptr) {
  if (n <= 0) return;
  const int rpb = kBlock / G;
  const int grid = grid_for(n, rpb, 1 << 18);
  switch (G) {
    case 1: klaunch(k_csr<1, T, TA, MODE>, dim3(grid), dim3(kBlock), 0, s, n, rp, ci, v, x, b, aux, w, y, y2); break;
    case 2: klaunch(k_csr<2, T, TA, MODE>, dim3(grid), dim3(kBlock), 0, s, n, rp, ci, v, x, b, aux, w, y, y2); break;
    case 4: klaunch(k_csr<4, T, TA, MODE>, dim3(grid), dim3(kBlock), 0, s, n, rp, ci, v, x, b, aux, w, y, y2); break;
    case 8: klaunch(k_csr<8, T, TA, MODE>, dim3(grid), dim3(kBlock), 0, s, n, rp, ci, v, x, b, aux, w, y, y2); break;
    case 16: klaunch(k_csr<16, T, TA, MODE>, dim3(grid), dim3(kBlock), 0, s, n, rp, ci, v, x, b, aux, w, y, y2); break;
    case 32: klaunch(k_csr<32, T, TA, MODE>, dim3(grid), dim3(kBlock), 0, s, n, rp, ci, v, x, b, aux, w, y, y2); break;
    default: klaunch(k_csr<64, T, TA, MODE>, dim3(grid), dim3(kBlock), 0, s, n, rp, ci, v, x, b, aux, w, y, y2); break;
  }
  IMPES_LAUNCH_CHECK();
}

// ---------------------------------------------------------------- stencil 7
// sum_j A[c,j] x[j] in the column order of the CSR form (c-sx, c-nz, c-1, c, c+1, c+nz,
// c+sx), x[q] given by xv(q). A missing neighbour is read as the cell itself and left
// out of the sum: with the loads under the boundary conditions instead, a wave waited
// for memory once per neighbour (FP32 sweeps of 76,800 rows 3.5 us, now 2.5; the FP64 operator apply 4.8 and 3.8).
template <class T, class F>
__device__ __forceinline__ T st7_row(const Stencil7<T>& S, F xv, long long c, int i, int j, int k) {
  const long long sy = S.nz;
  const long long sx = (long long)S.ny * S.nz;
  const bool w = i > 0, e = i < S.nx - 1, o = j > 0, n = j < S.ny - 1, b = k > 0, t = k < S.nz - 1;
  const long long qw = w ? c - sx : c, qo = o ? c - sy : c, qb = b ? c - 1 : c;
  const T fw = S.ox[qw], fo = S.oy[qo], fb = S.oz[qb], d = S.d[c], ft = S.oz[c], fn = S.oy[c], fe = S.ox[c];
  const T xw = xv(qw), xo = xv(qo), xb = xv(qb), xc = xv(c);
  const T xt = xv(t ? c + 1 : c), xn = xv(n ? c + sy : c), xe = xv(e ? c + sx : c);
  T s = T(0);
  s = w ? s + fw * xw : s;
  s = o ? s + fo * xo : s;
  s = b ? s + fb * xb : s;
  s += d * xc;
  s = t ? s + ft * xt : s;
  s = n ? s + fn * xn : s;
  s = e ? s + fe * xe : s;
  return s;
}

template <class T, class TA, int MODE>
__global__ __launch_bounds__(kBlock) void k_st7(Stencil7<T> S, const T* __restrict__ x, const T* __restrict__ b,
                                                const TA* __restrict__ aux, T w, T* __restrict__ y) {
  const long long n = (long long)S.nx * S.ny * S.nz;
  for (long long c = xcd_block() * blockDim.x + threadIdx.x; c < n; c += (long long)gridDim.x * blockDim.x) {
    int i, j, k;
    cell_ijk(c, S.ny, S.nz, i, j, k);
    if constexpr (MODE == kJacZ0) {
      auto xv = [&](long long q) { return w * (T)aux[q] * b[q]; };
      const T bc = b[c], ac = (T)aux[c];
      const T sum = st7_row(S, xv, c, i, j, k);
      y[c] = xv(c) + w * ac * (bc - sum);
      continue;
    }
    // the row's own operands are loaded with the row's
    constexpr bool uses_b = MODE == kRes || MODE == kJac || MODE == kRowScaledRes;
    constexpr bool uses_aux = MODE == kJac || MODE == kRowScaled || MODE == kRowScaledRes;
    const T bc = uses_b ? b[c] : T(0), ac = uses_aux ? (T)aux[c] : T(0);
    const T sum = st7_row(S, [&](long long q) { return x[q]; }, c, i, j, k);
    if (MODE == kY) y[c] = sum;
    else if (MODE == kRes) y[c] = bc - sum;
    else if (MODE == kJac) y[c] = x[c] + w * ac * (bc - sum);
    else if (MODE == kRowScaled) y[c] = ac * sum;
    else if (MODE == kRowScaledRes) y[c] = ac * (bc - sum);
  }
}

// Wide form of k_st7 for nz a multiple of V = 16 / sizeof(T): a thread takes V
// consecutive cells of one z-column (same i, j) and reads every coefficient and
// x array with 16-byte loads (the +-x and +-y neighbours of V aligned cells are
// V aligned cells), plus oz[c-1], x[c-1] and x[c+V] for the column ends. Each
// cell's sum is formed in st7_row's order, so the results equal k_st7's.
template <class T>
struct Wide;
template <>
struct Wide<float> { using type = float4; };
template <>
struct Wide<double> { using type = double2; };

template <class T, int V>
__device__ __forceinline__ void ld_wide(const T* __restrict__ p, T (&a)[V]) {
  static_assert(V * sizeof(T) == 16, "16-byte vectors");
  const typename Wide<T>::type v = *reinterpret_cast<const typename Wide<T>::type*>(p);
  __builtin_memcpy(a, &v, 16);
}
template <class T, int V>
__device__ __forceinline__ void st_wide(T* __restrict__ p, const T (&a)[V]) {
  typename Wide<T>::type v;
  __builtin_memcpy(&v, a, 16);
  *reinterpret_cast<typename Wide<T>::type*>(p) = v;
}

template <class T, int MODE>
__global__ __launch_bounds__(kBlock) void k_st7_wide(Stencil7<T> S, const T* __restrict__ x, const T* __restrict__ b,
                                                     const T* __restrict__ aux, T w, T* __restrict__ y) {
  constexpr int V = 16 / sizeof(T);
  const long long n = (long long)S.nx * S.ny * S.nz;
  const long long sy = S.nz;
  const long long sx = (long long)S.ny * S.nz;
  for (long long q = xcd_block() * blockDim.x + threadIdx.x; q * V < n; q += (long long)gridDim.x * blockDim.x) {
    const long long c = q * V;
    int i, j, k0;
    cell_ijk(c, S.ny, S.nz, i, j, k0);
    T xc[V], dd[V], fz[V], fy[V], fx[V];
    T fw[V] = {}, xw[V] = {}, fs[V] = {}, xs[V] = {}, xn[V] = {}, xe[V] = {}, bb[V] = {}, aa[V] = {};
    // x at V aligned cells: read, or (kJacZ0) the first sweep w * aux .* b formed in place
    auto xg = [&](long long q, T (&dst)[V]) {
      if constexpr (MODE == kJacZ0) {
        T bq[V], aq[V];
        ld_wide(b + q, bq);
        ld_wide(aux + q, aq);
#pragma unroll
        for (int m = 0; m < V; ++m) dst[m] = w * aq[m] * bq[m];
      } else {
        ld_wide(x + q, dst);
      }
    };
    auto x1 = [&](long long q) {
      if constexpr (MODE == kJacZ0) return w * aux[q] * b[q];
      else return x[q];
    };
    xg(c, xc);
    ld_wide(S.d + c, dd);
    ld_wide(S.oz + c, fz);
    ld_wide(S.oy + c, fy);
    ld_wide(S.ox + c, fx);
    // a missing neighbour is read as the cells themselves and left out of the sum
    const long long qw = i > 0 ? c - sx : c, qs = j > 0 ? c - sy : c, qb = k0 > 0 ? c - 1 : c;
    ld_wide(S.ox + qw, fw);
    xg(qw, xw);
    ld_wide(S.oy + qs, fs);
    xg(qs, xs);
    xg(j < S.ny - 1 ? c + sy : c, xn);
    xg(i < S.nx - 1 ? c + sx : c, xe);
    const T zb = S.oz[qb];
    const T xb = x1(qb);
    const T xa = x1(k0 + V < S.nz ? c + V : c);
    if (MODE == kRes || MODE == kJac || MODE == kRowScaledRes || MODE == kJacZ0) ld_wide(b + c, bb);
    if (MODE == kJac || MODE == kRowScaled || MODE == kRowScaledRes || MODE == kJacZ0) ld_wide(aux + c, aa);
    T out[V];
#pragma unroll
    for (int m = 0; m < V; ++m) {
      const int k = k0 + m;
      T sum = T(0);
      if (i > 0) sum += fw[m] * xw[m];
      if (j > 0) sum += fs[m] * xs[m];
      if (k > 0) sum += (m == 0 ? zb : fz[m > 0 ? m - 1 : 0]) * (m == 0 ? xb : xc[m > 0 ? m - 1 : 0]);
      sum += dd[m] * xc[m];
      if (k < S.nz - 1) sum += fz[m] * (m == V - 1 ? xa : xc[m < V - 1 ? m + 1 : 0]);
      if (j < S.ny - 1) sum += fy[m] * xn[m];
      if (i < S.nx - 1) sum += fx[m] * xe[m];
      if (MODE == kY) out[m] = sum;
      else if (MODE == kRes) out[m] = bb[m] - sum;
      else if (MODE == kJac || MODE == kJacZ0) out[m] = xc[m] + w * aa[m] * (bb[m] - sum);
      else if (MODE == kRowScaled) out[m] = aa[m] * sum;
      else out[m] = aa[m] * (bb[m] - sum);
    }
    st_wide(y + c, out);
  }
}

// y = dinv .* (A z) and z itself, with z = sout .* x formed on the fly from the
// V-cycle's output x (FP32 or FP64): the preconditioner's output scaling fused
// into the Krylov operator apply. Same operation order as k_scale followed by
// k_st7<kRowScaled>, so the result is identical to the two-kernel form.
template <class TX>
__global__ __launch_bounds__(kBlock) void k_st7_rowscaled_z(Stencil7<double> S, const double* __restrict__ dinv,
                                                            const double* __restrict__ sout,
                                                            const TX* __restrict__ x, double* __restrict__ z,
                                                            double* __restrict__ y) {
  const long long n = (long long)S.nx * S.ny * S.nz;
  const long long sy = S.nz;
  const long long sx = (long long)S.ny * S.nz;
  for (long long c = xcd_block() * blockDim.x + threadIdx.x; c < n; c += (long long)gridDim.x * blockDim.x) {
    int i, j, k;
    cell_ijk(c, S.ny, S.nz, i, j, k);
    auto zv = [&](long long q) { return sout[q] * (double)x[q]; };
    const double di = dinv[c];
    const double s = st7_row(S, zv, c, i, j, k);
    z[c] = zv(c);
    y[c] = di * s;
  }
}

// Wide form of k_st7_rowscaled_z for even nz: two cells of one z-column per
// thread, 16-byte loads of every FP64 array (8-byte loads of an FP32 x), the same
// operation order per cell.
template <class TX>
struct Pair;
template <>
struct Pair<float> { using type = float2; };
template <>
struct Pair<double> { using type = double2; };

template <class TX>
__device__ __forceinline__ void ld_pair(const TX* __restrict__ p, TX (&a)[2]) {
  const typename Pair<TX>::type v = *reinterpret_cast<const typename Pair<TX>::type*>(p);
  a[0] = v.x;
  a[1] = v.y;
}

template <class TX>
__global__ __launch_bounds__(kBlock) void k_st7_rowscaled_z_wide(Stencil7<double> S, const double* __restrict__ dinv,
                                                                 const double* __restrict__ sout,
                                                                 const TX* __restrict__ x, double* __restrict__ z,
                                                                 double* __restrict__ y) {
  const long long n = (long long)S.nx * S.ny * S.nz;
  const long long sy = S.nz;
  const long long sx = (long long)S.ny * S.nz;
  for (long long q = xcd_block() * blockDim.x + threadIdx.x; q * 2 < n; q += (long long)gridDim.x * blockDim.x) {
    const long long c = q * 2;
    int i, j, k0;
    cell_ijk(c, S.ny, S.nz, i, j, k0);
    // z = sout .* x at the cell pair and at each neighbour pair
    auto zpair = [&](long long p0, double (&zz)[2]) {
      TX xx[2];
      double ss[2];
      ld_pair(x + p0, xx);
      ld_pair(sout + p0, ss);
      zz[0] = ss[0] * (double)xx[0];
      zz[1] = ss[1] * (double)xx[1];
    };
    double zc[2], dd[2], fz[2], fy[2], fx[2], di[2];
    double zw[2] = {}, fw[2] = {}, zs[2] = {}, fs[2] = {}, zn[2] = {}, ze[2] = {};
    zpair(c, zc);
    ld_pair(S.d + c, dd);
    ld_pair(S.oz + c, fz);
    ld_pair(S.oy + c, fy);
    ld_pair(S.ox + c, fx);
    ld_pair(dinv + c, di);
    // a missing neighbour is read as the cells themselves and left out of the sum
    const long long qw = i > 0 ? c - sx : c, qs = j > 0 ? c - sy : c, qb = k0 > 0 ? c - 1 : c;
    const long long qa = k0 + 2 < S.nz ? c + 2 : c;
    ld_pair(S.ox + qw, fw);
    zpair(qw, zw);
    ld_pair(S.oy + qs, fs);
    zpair(qs, zs);
    zpair(j < S.ny - 1 ? c + sy : c, zn);
    zpair(i < S.nx - 1 ? c + sx : c, ze);
    const double fb = S.oz[qb];
    const double zb = sout[qb] * (double)x[qb];
    const double za = sout[qa] * (double)x[qa];
    double out[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int k = k0 + m;
      double sum = 0.0;
      if (i > 0) sum += fw[m] * zw[m];
      if (j > 0) sum += fs[m] * zs[m];
      if (k > 0) sum += (m == 0 ? fb : fz[0]) * (m == 0 ? zb : zc[0]);
      sum += dd[m] * zc[m];
      if (k < S.nz - 1) sum += fz[m] * (m == 1 ? za : zc[1]);
      if (j < S.ny - 1) sum += fy[m] * zn[m];
      if (i < S.nx - 1) sum += fx[m] * ze[m];
      out[m] = di[m] * sum;
    }
    *reinterpret_cast<double2*>(z + c) = make_double2(zc[0], zc[1]);
    *reinterpret_cast<double2*>(y + c) = make_double2(out[0], out[1]);
  }
}

template <class T>
__global__ void k_jacobi0(const T* __restrict__ b, const T* __restrict__ inv_relax, T w, T* __restrict__ xo, int n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    xo[i] = w * inv_relax[i] * b[i];
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

template <class T, class TA, int MODE>
void st7_launch(const Stencil7<T>& S, const T* x, const T* b, const TA* aux, T w, T* y, hipStream_t s) {
  const long long n = (long long)S.nx * S.ny * S.nz;
  if (n <= 0) return;
  constexpr int V = 16 / sizeof(T);
  constexpr bool uses_b = MODE == kRes || MODE == kJac || MODE == kRowScaledRes || MODE == kJacZ0;
  constexpr bool uses_aux = MODE == kJac || MODE == kRowScaled || MODE == kRowScaledRes || MODE == kJacZ0;
  if constexpr (std::is_same<T, TA>::value) {
    // the wide form needs whole 16-byte vectors along z and 16-byte aligned arrays
    if (S.nz % V == 0 && aligned16(x) && aligned16(y) && aligned16(S.d) && aligned16(S.ox) && aligned16(S.oy) &&
        aligned16(S.oz) && (!uses_b || aligned16(b)) && (!uses_aux || aligned16(aux))) {
      klaunch(k_st7_wide<T, MODE>, dim3(grid_for(n / V, kBlock, 1 << 18)), dim3(kBlock), 0, s, S, x, b, aux, w, y);
      IMPES_LAUNCH_CHECK();
      return;
    }
  }
  klaunch(k_st7<T, TA, MODE>, dim3(grid_for(n, kBlock, 1 << 18)), dim3(kBlock), 0, s, S, x, b, aux, w, y);
  IMPES_LAUNCH_CHECK();
}

}  // namespace

// Algorithmic HBM bytes of one pass (each operand read or written once):
// CSR: row pointers + (column, value) per entry + `vecs` row vectors besides x
// (x read once, e.g. b, inv_relax and the output for Jacobi);
// stencil: four coefficient arrays + x + `vecs` row vectors.
double csr_bytes(long long n, long long nnz, int val_bytes, int vecs) {
  return (double)(n + 1) * 4 + (double)nnz * (4 + val_bytes) + (double)n * val_bytes * (1 + vecs);
}
template <class T>
double st7_bytes(const Stencil7<T>& S, int val_bytes, int vecs) {
  const double n = (double)S.nx * S.ny * S.nz;
  return n * val_bytes * (4 + 1 + vecs);
}

// Lanes per row: the smallest power of two with at most ~4 entries per lane, so a
// lane has several independent (value, column, gather) loads in flight (one entry
// per lane is latency-bound). A sweep too small to fill the GPU (fewer than 2^18
// lanes) is bound by each row's serial chain instead of by throughput: it takes
// twice the lanes (~2 entries per lane). Measured at 1M cells: level-1/2 sweeps
// 21.9/23.6 us at ~4 per lane against 25.5/28.4 us at ~2; level-4+ sweeps and
// coarse restrictions 7-12 us at ~4 against 5-8 us at ~2.
int csr_group_for(int n_rows, int nnz) {
  if (n_rows <= 0) return 1;
  const double mean = (double)nnz / (double)n_rows;
  int g = 1;
  while (g < 64 && g * 4 < mean) g <<= 1;
  if ((long long)n_rows * g < (1LL << 18) && g < 64 && g * 2 < mean) g <<= 1;
  return g;
}

void launch_spmv_f64(const CsrF64& A, const double* x, double* y, int G, hipStream_t s) {
  csr_dispatch<double, double, kY>(A.n_rows, A.rp, A.ci, A.v, x, nullptr, (const double*)nullptr, 0.0, y, G, s);
}
void launch_spmv_f32(const CsrF32& A, const float* x, float* y, int G, hipStream_t s) {
  csr_dispatch<float, float, kY>(A.n_rows, A.rp, A.ci, A.v, x, nullptr, (const float*)nullptr, 0.f, y, G, s);
}
void launch_spmv_add_f64(const CsrF64& A, const double* x, double* y, int G, hipStream_t s) {
  csr_dispatch<double, double, kYAdd>(A.n_rows, A.rp, A.ci, A.v, x, nullptr, (const double*)nullptr, 0.0, y, G, s);
}
void launch_spmv_add_f32(const CsrF32& A, const float* x, float* y, int G, hipStream_t s) {
  csr_dispatch<float, float, kYAdd>(A.n_rows, A.rp, A.ci, A.v, x, nullptr, (const float*)nullptr, 0.f, y, G, s);
}
void launch_spmv_add_to_f64(const CsrF64& A, const double* x, const double* y0, double* y, int G, hipStream_t s) {
  csr_dispatch<double, double, kYPlusB>(A.n_rows, A.rp, A.ci, A.v, x, y0, (const double*)nullptr, 0.0, y, G, s);
}
void launch_spmv_add_to_f32(const CsrF32& A, const float* x, const float* y0, float* y, int G, hipStream_t s) {
  csr_dispatch<float, float, kYPlusB>(A.n_rows, A.rp, A.ci, A.v, x, y0, (const float*)nullptr, 0.f, y, G, s);
}
void launch_residual_f64(const CsrF64& A, const double* x, const double* b, double* r, int G, hipStream_t s) {
  csr_dispatch<double, double, kRes>(A.n_rows, A.rp, A.ci, A.v, x, b, (const double*)nullptr, 0.0, r, G, s);
}
void launch_residual_f32(const CsrF32& A, const float* x, const float* b, float* r, int G, hipStream_t s) {
  KScope ks("csr_residual_f32", csr_bytes(A.n_rows, A.nnz, 4, 2), s);
  csr_dispatch<float, float, kRes>(A.n_rows, A.rp, A.ci, A.v, x, b, (const float*)nullptr, 0.f, r, G, s);
}
void launch_jacobi_f64(const CsrF64& A, const double* xi, const double* b, const double* inv_relax, double w,
                       double* xo, int G, hipStream_t s) {
  KScope ks("csr_jacobi_f64", csr_bytes(A.n_rows, A.nnz, 8, 3), s);
  csr_dispatch<double, double, kJac>(A.n_rows, A.rp, A.ci, A.v, xi, b, inv_relax, w, xo, G, s);
}
void launch_jacobi_f32(const CsrF32& A, const float* xi, const float* b, const float* inv_relax, float w, float* xo,
                       int G, hipStream_t s) {
  KScope ks("csr_jacobi_f32", csr_bytes(A.n_rows, A.nnz, 4, 3), s);
  csr_dispatch<float, float, kJac>(A.n_rows, A.rp, A.ci, A.v, xi, b, inv_relax, w, xo, G, s);
}
int csr4_group_for(int n_rows, long long nnz4) {
  if (n_rows <= 0) return 1;
  // at most one 4-entry chunk per lane on a row of mean length: the smallest power
  // of two not below the mean number of chunks (measured on the 1M-cell IMPES
  // hierarchy: 8 lanes on level 1 with ~4 chunks per row beat 4 lanes by 7%)
  const double chunks = (double)nnz4 / 4.0 / (double)n_rows;
  int g = 1;
  while (g < 64 && g < chunks) g <<= 1;
  return g;
}
void launch_csr4_count(int n, const int* rp, int* cnt, hipStream_t s) {
  if (n <= 0) return;
  k_csr4_count<<<grid_for(n, kBlock, 1 << 16), kBlock, 0, s>>>(n, rp, cnt);
  IMPES_LAUNCH_CHECK();
}
void launch_tile4_count(int n, const int* rp, int* cnt, hipStream_t s) {
  const int segs = div_up(n, kTileSeg);
  k_tile4_rows<false><<<div_up(segs, kBlock / kWave), kBlock, 0, s>>>(n, rp, nullptr, cnt, nullptr, nullptr);
  IMPES_LAUNCH_CHECK();
}
void launch_tile4_rows(int n, const int* rp, const long long* base, int* wrow, int* rp4, hipStream_t s) {
  const int segs = div_up(n, kTileSeg);
  k_tile4_rows<true><<<div_up(segs, kBlock / kWave), kBlock, 0, s>>>(n, rp, base, nullptr, wrow, rp4);
  IMPES_LAUNCH_CHECK();
}
void launch_tile4_fill(int nw, const int* wrow, const int* rp, const int* ci, const double* v, const int* rp4,
                       int* ci4, short* co4, float* v4, unsigned short* tag, int* maxabs, bool square, hipStream_t s) {
  if (nw <= 0) return;
  k_tile4_fill<<<grid_for(nw, kBlock / kWave, 1 << 16), kBlock, 0, s>>>(
      nw, wrow, rp, ci, v, rp4, reinterpret_cast<int4*>(ci4), reinterpret_cast<short4*>(co4),
      reinterpret_cast<float4*>(v4), tag, maxabs, square ? 1 : 0);
  IMPES_LAUNCH_CHECK();
}
void launch_csr4_pattern(int n, const int* rp, const int* ci, const int* rp4, int* ci4, hipStream_t s) {
  if (n <= 0) return;
  k_csr4_pattern<<<grid_for(n, kBlock, 1 << 16), kBlock, 0, s>>>(n, rp, ci, rp4, ci4);
  IMPES_LAUNCH_CHECK();
}
void launch_csr4_values(int n, const int* rp, const double* v, const int* rp4, float* v4, hipStream_t s) {
  if (n <= 0) return;
  k_csr4_values<8><<<grid_for((long long)n * 8, kBlock, 1 << 16), kBlock, 0, s>>>(n, rp, v, rp4, v4);
  IMPES_LAUNCH_CHECK();
}
void launch_csr4_offsets(int n, const int* rp4, const int* ci4, short* co4, int* maxabs, hipStream_t s) {
  if (n <= 0) return;
  k_csr4_offsets<<<grid_for(n, kBlock, 1 << 16), kBlock, 0, s>>>(n, rp4, ci4, co4, maxabs);
  IMPES_LAUNCH_CHECK();
}
void launch_residual4_f32(const Csr4F32& A, int G, const float* x, const float* b, float* r, hipStream_t s) {
  KScope ks("csr_residual_f32", csr_bytes(A.n, A.nnz, 4, 2), s);
  csr4_dispatch<kRes>(A, G, x, b, nullptr, 0.f, r, s);
}
void launch_jacobi4_f32(const Csr4F32& A, int G, const float* xi, const float* b, const float* inv_relax, float w,
                        float* xo, hipStream_t s) {
  KScope ks("csr_jacobi_f32", csr_bytes(A.n, A.nnz, 4, 3), s);
  csr4_dispatch<kJac>(A, G, xi, b, inv_relax, w, xo, s);
}
void launch_spmv4_f32(const Csr4F32& A, const float* x, float* y, hipStream_t s) {
  IMPES_REQUIRE(A.nw > 0 && !A.co4, "padded transfer: wave tiles and column indices required");
  if (A.n <= 0) return;
  csr4_tile_launch<kY, false>(A, x, nullptr, nullptr, 0.f, y, s);
  IMPES_LAUNCH_CHECK();
}
void launch_restrict4_j0_f32(const Csr4F32& R, const float* r, const float* inv_relax_c, float w, float* bc, float* xc,
                             hipStream_t s) {
  IMPES_REQUIRE(R.nw > 0 && !R.co4, "padded transfer: wave tiles and column indices required");
  if (R.n <= 0) return;
  csr4_tile_launch<kRestrictJ0, false>(R, r, nullptr, inv_relax_c, w, bc, s, xc);
  IMPES_LAUNCH_CHECK();
}
void launch_prolong_sweep4_f32(const Csr4F32& S, const float* e, const float* r, const float* inv_relax, float w,
                               float* x0, float* x, hipStream_t s) {
  IMPES_REQUIRE(S.nw > 0 && !S.co4, "padded transfer: wave tiles and column indices required");
  if (S.n <= 0) return;
  KScope ks("csr_prolong_sweep_f32", csr_bytes(S.n, S.nnz, 4, 4), s);
  csr4_tile_launch<kProlongJac, false>(S, e, r, inv_relax, w, x, s, x0);
  IMPES_LAUNCH_CHECK();
}
void launch_tile4_values_f64(const Csr4F32& A, const int* rp, const double* v, double* v8, hipStream_t s) {
  if (A.nw <= 0) return;
  k_tile4_values_f64<<<grid_for(A.nw, kBlock / kWave, 1 << 18), kBlock, 0, s>>>(A.nw, A.wrow, A.tag, A.rp4, rp, v,
                                                                               reinterpret_cast<double2*>(v8));
  IMPES_LAUNCH_CHECK();
}
void launch_residual4_f64(const Csr4F32& A, const double* v8, const double* x, const double* b, double* r,
                          hipStream_t s) {
  KScope ks("csr_residual_f64", csr_bytes(A.n, A.nnz, 8, 2), s);
  csr4_tile_f64<kRes>(A, v8, x, b, nullptr, 0.0, r, s);
}
void launch_jacobi4_f64(const Csr4F32& A, const double* v8, const double* xi, const double* b, const double* inv_relax,
                        double w, double* xo, hipStream_t s) {
  KScope ks("csr_jacobi_f64", csr_bytes(A.n, A.nnz, 8, 3), s);
  csr4_tile_f64<kJac>(A, v8, xi, b, inv_relax, w, xo, s);
}
void launch_spmv4_f64(const Csr4F32& A, const double* v8, const double* x, double* y, hipStream_t s) {
  csr4_tile_f64<kY>(A, v8, x, nullptr, nullptr, 0.0, y, s);
}
void launch_restrict4_j0_f64(const Csr4F32& R, const double* v8, const double* r, const double* inv_relax_c, double w,
                             double* bc, double* xc, hipStream_t s) {
  csr4_tile_f64<kRestrictJ0>(R, v8, r, nullptr, inv_relax_c, w, bc, s, xc);
}
void launch_prolong_sweep4_f64(const Csr4F32& S, const double* v8, const double* e, const double* r,
                               const double* inv_relax, double w, double* x0, double* x, hipStream_t s) {
  csr4_tile_f64<kProlongJac>(S, v8, e, r, inv_relax, w, x, s, x0);
}
void launch_tile4_prolong_sweep(int nw, const int* wrow, const unsigned short* tag, const int* rp4, const int* ci4,
                                const int* aprp, const double* apv, const int* prp, const int* pci, const double* pv, const double* ir,
                                double w, float* v4, double* v8, int* miss, hipStream_t s) {
  if (nw <= 0) return;
  if (v8) {
    k_tile4_prolong_sweep<<<grid_for(nw, kBlock / kWave, 1 << 18), kBlock, 0, s>>>(
        nw, wrow, tag, rp4, reinterpret_cast<const int4*>(ci4), aprp, apv, prp, pci, pv, ir, w, v8, miss);
    IMPES_LAUNCH_CHECK();
    return;
  }
  k_tile4_prolong_sweep<<<grid_for(nw, kBlock / kWave, 1 << 18), kBlock, 0, s>>>(
      nw, wrow, tag, rp4, reinterpret_cast<const int4*>(ci4), aprp, apv, prp, pci, pv, ir, w, v4, miss);
  IMPES_LAUNCH_CHECK();
}
void launch_restrict_j0_f64(const CsrF64& R, const double* r, const double* inv_relax_c, double w, double* bc,
                            double* xc, int G, hipStream_t s) {
  csr_dispatch<double, double, kRestrictJ0>(R.n_rows, R.rp, R.ci, R.v, r, nullptr, inv_relax_c, w, bc, G, s, xc);
}
void launch_restrict_j0_f32(const CsrF32& R, const float* r, const float* inv_relax_c, float w, float* bc, float* xc,
                            int G, hipStream_t s) {
  csr_dispatch<float, float, kRestrictJ0>(R.n_rows, R.rp, R.ci, R.v, r, nullptr, inv_relax_c, w, bc, G, s, xc);
}
void launch_jacobi0_f64(const double* b, const double* inv_relax, double w, double* xo, int n, hipStream_t s) {
  if (n <= 0) return;
  k_jacobi0<double><<<grid_for(n, kBlock, 1 << 18), kBlock, 0, s>>>(b, inv_relax, w, xo, n);
  IMPES_LAUNCH_CHECK();
}
void launch_jacobi0_f32(const float* b, const float* inv_relax, float w, float* xo, int n, hipStream_t s) {
  if (n <= 0) return;
  k_jacobi0<float><<<grid_for(n, kBlock, 1 << 18), kBlock, 0, s>>>(b, inv_relax, w, xo, n);
  IMPES_LAUNCH_CHECK();
}
void launch_csr_rowscaled_spmv_f64(const CsrF64& A, const double* dinv, const double* x, double* y, int G,
                                   hipStream_t s) {
  csr_dispatch<double, double, kRowScaled>(A.n_rows, A.rp, A.ci, A.v, x, nullptr, dinv, 0.0, y, G, s);
}
void launch_csr_rowscaled_residual_f64(const CsrF64& A, const double* dinv, const double* x, const double* b,
                                       double* r, int G, hipStream_t s) {
  csr_dispatch<double, double, kRowScaledRes>(A.n_rows, A.rp, A.ci, A.v, x, b, dinv, 0.0, r, G, s);
}

void launch_st7_spmv_f64(const Stencil7<double>& S, const double* x, double* y, hipStream_t s) {
  st7_launch<double, double, kY>(S, x, nullptr, (const double*)nullptr, 0.0, y, s);
}
void launch_st7_residual_f64(const Stencil7<double>& S, const double* x, const double* b, double* r, hipStream_t s) {
  st7_launch<double, double, kRes>(S, x, b, (const double*)nullptr, 0.0, r, s);
}
void launch_st7_jacobi_z0_f64(const Stencil7<double>& S, const double* b, const double* inv_relax, double w,
                              double* xo, hipStream_t s) {
  KScope ks("st7_jacobi_z0_f64", st7_bytes(S, 8, 2), s);
  st7_launch<double, double, kJacZ0>(S, nullptr, b, inv_relax, w, xo, s);
}
void launch_st7_jacobi_z0_f32(const Stencil7<float>& S, const float* b, const float* inv_relax, float w, float* xo,
                              hipStream_t s) {
  KScope ks("st7_jacobi_z0_f32", st7_bytes(S, 4, 2), s);
  st7_launch<float, float, kJacZ0>(S, nullptr, b, inv_relax, w, xo, s);
}
void launch_st7_residual_f32(const Stencil7<float>& S, const float* x, const float* b, float* r, hipStream_t s) {
  KScope ks("st7_residual_f32", st7_bytes(S, 4, 2), s);
  st7_launch<float, float, kRes>(S, x, b, (const float*)nullptr, 0.f, r, s);
}
void launch_st7_jacobi_f64(const Stencil7<double>& S, const double* xi, const double* b, const double* inv_relax,
                           double w, double* xo, hipStream_t s) {
  KScope ks("st7_jacobi_f64", st7_bytes(S, 8, 3), s);
  st7_launch<double, double, kJac>(S, xi, b, inv_relax, w, xo, s);
}
void launch_st7_jacobi_f32(const Stencil7<float>& S, const float* xi, const float* b, const float* inv_relax, float w,
                           float* xo, hipStream_t s) {
  KScope ks("st7_jacobi_f32", st7_bytes(S, 4, 3), s);
  st7_launch<float, float, kJac>(S, xi, b, inv_relax, w, xo, s);
}
void launch_st7_rowscaled_spmv_f64(const Stencil7<double>& S, const double* dinv, const double* x, double* y,
                                   hipStream_t s) {
  KScope ks("st7_rowscaled_spmv_f64", st7_bytes(S, 8, 2), s);
  st7_launch<double, double, kRowScaled>(S, x, nullptr, dinv, 0.0, y, s);
}
template <class TX>
static void st7_rowscaled_z(const Stencil7<double>& S, const double* dinv, const double* sout, const TX* x, double* z,
                            double* y, hipStream_t s) {
  const long long n = (long long)S.nx * S.ny * S.nz;
  if (n <= 0) return;
  // x and sout, 4 coefficient arrays and dinv read; z and y written
  KScope ks(sizeof(TX) == 4 ? "st7_rowscaled_z_f32in" : "st7_rowscaled_z_f64in",
            (double)n * (sizeof(TX) + 8 * 8), s);
  if (S.nz % 2 == 0 && aligned16(dinv) && aligned16(sout) && aligned16(z) && aligned16(y) && aligned16(S.d) &&
      aligned16(S.ox) && aligned16(S.oy) && aligned16(S.oz) && ((uintptr_t)x % (2 * sizeof(TX))) == 0) {
    klaunch(k_st7_rowscaled_z_wide<TX>, dim3(grid_for(n / 2, kBlock, 1 << 18)), dim3(kBlock), 0, s, S, dinv, sout, x,
            z, y);
  } else {
    klaunch(k_st7_rowscaled_z<TX>, dim3(grid_for(n, kBlock, 1 << 18)), dim3(kBlock), 0, s, S, dinv, sout, x, z, y);
  }
  IMPES_LAUNCH_CHECK();
}
void launch_st7_rowscaled_spmv_z_f64(const Stencil7<double>& S, const double* dinv, const double* sout,
                                     const float* x, double* z, double* y, hipStream_t s) {
  st7_rowscaled_z<float>(S, dinv, sout, x, z, y, s);
}
void launch_st7_rowscaled_spmv_z_f64(const Stencil7<double>& S, const double* dinv, const double* sout,
                                     const double* x, double* z, double* y, hipStream_t s) {
  st7_rowscaled_z<double>(S, dinv, sout, x, z, y, s);
}
void launch_st7_rowscaled_residual_f64(const Stencil7<double>& S, const double* dinv, const double* x,
                                       const double* b, double* r, hipStream_t s) {
  st7_launch<double, double, kRowScaledRes>(S, x, b, dinv, 0.0, r, s);
}

}  // namespace impes
