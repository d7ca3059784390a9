// Scans, segmented sort and small reductions for the AMG setup phase.
#include <mutex>
#include <vector>

#include "prims.h"

namespace impes {

namespace {
constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;
constexpr int kTile = kScanBlock * kScanItems;

template <class T>
__device__ __forceinline__ T wave_incl_scan(T v) {
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    T t = __shfl_up(v, off, kWave);
    if (lane >= off) v += t;
  }
  return v;
}

// exclusive block scan; returns the exclusive prefix of v and writes the block total
template <class T>
__device__ __forceinline__ T block_excl_scan(T v, T* lds, T& total) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = threadIdx.x / kWave;
  constexpr int nw = kScanBlock / kWave;
  T inc = wave_incl_scan(v);
  __syncthreads();
  if (lane == kWave - 1) lds[wid] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    T run = 0;
    for (int w = 0; w < nw; ++w) { T t = lds[w]; lds[w] = run; run += t; }
    lds[nw] = run;
  }
  __syncthreads();
  T res = lds[wid] + inc - v;
  total = lds[nw];
  __syncthreads();
  return res;
}

template <class TO>
__global__ __launch_bounds__(kScanBlock) void k_tile_sums(const int* __restrict__ in, long long n,
                                                          TO* __restrict__ bsum) {
  __shared__ TO lds[kScanBlock / kWave + 1];
  const long long base = (long long)blockIdx.x * kTile + (long long)threadIdx.x * kScanItems;
  TO s = 0;
#pragma unroll
  for (int t = 0; t < kScanItems; ++t) {
    long long i = base + t;
    if (i < n) s += (TO)in[i];
  }
  TO tot;
  (void)block_excl_scan<TO>(s, lds, tot);
  if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// single block: exclusive scan of nb tile sums in place, total -> *total
template <class TO>
__global__ __launch_bounds__(kScanBlock) void k_scan_tiles(TO* __restrict__ bsum, long long nb, TO* __restrict__ total) {
  __shared__ TO lds[kScanBlock / kWave + 1];
  TO carry = 0;
  for (long long c0 = 0; c0 < nb; c0 += kScanBlock) {
    long long i = c0 + threadIdx.x;
    TO v = (i < nb) ? bsum[i] : (TO)0;
    TO tot;
    TO ex = block_excl_scan<TO>(v, lds, tot);
    if (i < nb) bsum[i] = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) *total = carry;
}

template <class TO>
__global__ __launch_bounds__(kScanBlock) void k_tile_scan(const int* __restrict__ in, long long n,
                                                          const TO* __restrict__ bsum, TO* __restrict__ out) {
  __shared__ TO lds[kScanBlock / kWave + 1];
  const long long base = (long long)blockIdx.x * kTile + (long long)threadIdx.x * kScanItems;
  TO vals[kScanItems];
  TO s = 0;
#pragma unroll
  for (int t = 0; t < kScanItems; ++t) {
    long long i = base + t;
    vals[t] = (i < n) ? (TO)in[i] : (TO)0;
    s += vals[t];
  }
  TO tot;
  TO ex = block_excl_scan<TO>(s, lds, tot) + bsum[blockIdx.x];
#pragma unroll
  for (int t = 0; t < kScanItems; ++t) {
    long long i = base + t;
    if (i < n) out[i] = ex;
    ex += vals[t];
  }
}

template <class TO>
void scan_impl(const int* in, TO* out, long long n, hipStream_t s) {
  if (n <= 0) {
    IMPES_HIP_CHECK(hipMemsetAsync(out, 0, sizeof(TO), s));
    return;
  }
  const long long nb = (n + kTile - 1) / kTile;
  DevBuf<TO> bsum;
  bsum.alloc((size_t)nb);
  k_tile_sums<TO><<<(unsigned)nb, kScanBlock, 0, s>>>(in, n, bsum.p);
  IMPES_LAUNCH_CHECK();
  k_scan_tiles<TO><<<1, kScanBlock, 0, s>>>(bsum.p, nb, out + n);
  IMPES_LAUNCH_CHECK();
  k_tile_scan<TO><<<(unsigned)nb, kScanBlock, 0, s>>>(in, n, bsum.p, out);
  IMPES_LAUNCH_CHECK();
  sync_before_release(s);  // bsum must outlive the kernels
}

// ---------------------------------------------------------------- segmented sort
// Segments are binned by length (k_seg_bin), and each bin is sorted by a
// kernel sized for it: a thread per segment of <= 16 keys (registers), else a
// workgroup per segment with the keys staged in LDS and bitonic-sorted over the
// next power of two >= the segment length (padding with all-ones keys), from
// one wavefront for <= 64 keys up to 1024 threads for <= 8192 keys (64 KiB of
// LDS); longer segments are sorted in place. Bins only choose the kernel: each
// segment is sorted on its own, so the result does not depend on the binning.
constexpr int kSortBins = 7;  // <= 16, 64, 256, 1024, 4096, 8192 keys, and longer

__device__ __forceinline__ int sort_bin(long long len) {
  return len <= 16 ? 0 : len <= 64 ? 1 : len <= 256 ? 2 : len <= 1024 ? 3 : len <= 4096 ? 4 : len <= 8192 ? 5 : 6;
}

// Segments of at most 16 keys: a thread per segment, bitonic network over 16
// registers (padding with all-ones keys).
__global__ void k_segsort_regs(unsigned long long* __restrict__ keys, const long long* __restrict__ seg,
                               const int* __restrict__ list, const int* __restrict__ count) {
  const int n = *count;
  for (long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x; q < n;
       q += (long long)gridDim.x * blockDim.x) {
    const long long sg = list[q];
    const long long b = seg[sg];
    const int len = (int)(seg[sg + 1] - b);
    unsigned long long r[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) r[t] = (t < len) ? keys[b + t] : ~0ull;
#pragma unroll
    for (int size = 2; size <= 16; size <<= 1) {
#pragma unroll
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
#pragma unroll
        for (int t = 0; t < 16; ++t) {
          const int partner = t ^ stride;
          if (partner > t) {
            const bool asc = (t & size) == 0;
            const unsigned long long a = r[t], c = r[partner];
            if ((a > c) == asc) { r[t] = c; r[partner] = a; }
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < 16; ++t)
      if (t < len) keys[b + t] = r[t];
  }
}

__global__ void k_fill_zero(int* __restrict__ counts, int n) {
  if (threadIdx.x < n) counts[threadIdx.x] = 0;
}

// Bin lists: each wavefront claims its slots with one atomic per bin present
// in it (a single counter per bin would otherwise take one atomic per segment).
__global__ void k_seg_bin(const long long* __restrict__ seg, long long nseg, int* __restrict__ counts,
                          int* __restrict__ lists) {
  const int lane = threadIdx.x & (kWave - 1);
  const unsigned long long below = lane ? (~0ull >> (kWave - lane)) : 0ull;
  for (long long i0 = blockIdx.x * (long long)blockDim.x + (threadIdx.x & ~(kWave - 1)); i0 < nseg;
       i0 += (long long)gridDim.x * blockDim.x) {
    const long long i = i0 + lane;
    int bin = -1;
    long long len = 0;
    if (i < nseg) {
      len = seg[i + 1] - seg[i];
      if (len > 1) bin = sort_bin(len);
    }
    for (int b = 0; b < kSortBins; ++b) {
      const unsigned long long m = __ballot(bin == b);
      if (!m) continue;
      const int leader = __ffsll((long long)m) - 1;
      int base = 0;
      if (lane == leader) base = atomicAdd(&counts[b], __popcll(m));
      base = __shfl(base, leader, kWave);
      if (bin == b) lists[(long long)b * nseg + base + __popcll(m & below)] = (int)i;
    }
  }
}

template <class K>
__device__ __forceinline__ void bitonic_block(K* sk, long long p2) {
  for (long long size = 2; size <= p2; size <<= 1) {
    for (long long stride = size >> 1; stride > 0; stride >>= 1) {
      for (long long t = threadIdx.x; t < p2; t += blockDim.x) {
        const long long partner = t ^ stride;
        if (partner > t) {
          const bool asc = (t & size) == 0;
          const K a = sk[t], c = sk[partner];
          if ((a > c) == asc) { sk[t] = c; sk[partner] = a; }
        }
      }
      __syncthreads();
    }
  }
}

// In-place sort of any number of keys by the workgroup: the bitonic network with every
// comparator ascending (the first one of a size pairs t with its mirror image), so
// that the missing keys up to the next power of two, the largest of all, would never
// move and need no storage.
__device__ __forceinline__ void bitonic_any(unsigned long long* sk, long long len) {
  for (long long size = 2; size < 2 * len; size <<= 1) {
    for (long long stride = size >> 1; stride > 0; stride >>= 1) {
      const long long flip = stride == size >> 1 ? size - 1 : stride;
      for (long long t = threadIdx.x; t < len; t += blockDim.x) {
        const long long partner = t ^ flip;
        if (partner > t && partner < len) {
          const unsigned long long a = sk[t], c = sk[partner];
          if (a > c) { sk[t] = c; sk[partner] = a; }
        }
      }
      __syncthreads();
    }
  }
}

// list and *count: the segments of one length class
template <int CAP, int NT>
__global__ __launch_bounds__(NT) void k_segsort_bin(unsigned long long* __restrict__ keys,
                                                    const long long* __restrict__ seg, const int* __restrict__ list,
                                                    const int* __restrict__ count) {
  __shared__ unsigned long long sk[CAP];
  const int n = *count;
  for (int q = blockIdx.x; q < n; q += gridDim.x) {
    const long long sg = list[q];
    const long long b = seg[sg];
    const int len = (int)(seg[sg + 1] - b);
    int p2 = 2;
    while (p2 < len) p2 <<= 1;
    for (int t = threadIdx.x; t < p2; t += NT) sk[t] = (t < len) ? keys[b + t] : ~0ull;
    __syncthreads();
    bitonic_block(sk, (long long)p2);
    for (int t = threadIdx.x; t < len; t += NT) keys[b + t] = sk[t];
    __syncthreads();
  }
}

// Few segments: a workgroup per segment without the classes (nine launches otherwise,
// which bind a small level's sort), the same network in LDS. Segments above kSortAnyLds
// keys are left to k_segsort_few_long.
constexpr int kSortAny = 4096, kSortAnyLds = 4096;
__global__ __launch_bounds__(256) void k_segsort_any(unsigned long long* __restrict__ keys,
                                                     const long long* __restrict__ seg) {
  __shared__ unsigned long long sk[kSortAnyLds];
  const long long b = seg[blockIdx.x], len = seg[blockIdx.x + 1] - b;
  if (len <= 1 || len > kSortAnyLds) return;
  int p2 = 2;
  while (p2 < len) p2 <<= 1;
  for (int t = threadIdx.x; t < p2; t += 256) sk[t] = (t < len) ? keys[b + t] : ~0ull;
  __syncthreads();
  bitonic_block(sk, (long long)p2);
  for (int t = threadIdx.x; t < len; t += 256) keys[b + t] = sk[t];
}

// The long ones among few segments: in LDS up to 8192 keys, else in place. With 256
// threads to such a segment (in k_segsort_any) the sorts of a hierarchy of 20,000 rows and
// 2M entries took 166 ms, with 1024 they take 60; looking the lengths over takes about 3 us.
constexpr int kSortLongLds = 8192;
__global__ __launch_bounds__(1024) void k_segsort_few_long(unsigned long long* __restrict__ keys,
                                                           const long long* __restrict__ seg, int nseg) {
  __shared__ unsigned long long sk[kSortLongLds];
  for (int sg = blockIdx.x; sg < nseg; sg += gridDim.x) {
    const long long b = seg[sg], len = seg[sg + 1] - b;
    if (len <= kSortAnyLds) continue;
    if (len > kSortLongLds) {
      bitonic_any(keys + b, len);
      continue;
    }
    for (int t = threadIdx.x; t < kSortLongLds; t += 1024) sk[t] = (t < len) ? keys[b + t] : ~0ull;
    __syncthreads();
    bitonic_block(sk, (long long)kSortLongLds);
    for (int t = threadIdx.x; t < len; t += 1024) keys[b + t] = sk[t];
    __syncthreads();
  }
}

// Segments longer than the LDS classes, a workgroup each, in place
__global__ __launch_bounds__(1024) void k_segsort_global(unsigned long long* __restrict__ keys,
                                                         const long long* __restrict__ seg,
                                                         const int* __restrict__ list, const int* __restrict__ count) {
  const int n = *count;
  for (int q = blockIdx.x; q < n; q += gridDim.x) bitonic_any(keys + seg[list[q]], seg[list[q] + 1] - seg[list[q]]);
}

__global__ void k_sum_i32(const int* __restrict__ x, long long n, long long* __restrict__ part) {
  __shared__ long long lds[256 / kWave];
  long long m = 0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    m += x[i];
  m = block_sum<long long>(m, lds);
  if (threadIdx.x == 0) part[blockIdx.x] = m;
}

__global__ void k_count_i8(const signed char* __restrict__ x, long long n, signed char v, long long* __restrict__ part) {
  __shared__ long long lds[256 / kWave];
  long long m = 0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    m += (x[i] == v) ? 1 : 0;
  m = block_sum<long long>(m, lds);
  if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// Readback: wave w handles item w (a value, or the sum of m)
struct ReadItems {
  const void* p[8];
  int bytes[8], m[8];
};
__global__ __launch_bounds__(8 * kWave) void k_readback(ReadItems it, long long* __restrict__ out) {
  const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
  long long v = 0;
  for (int q = lane; q < it.m[w]; q += kWave)
    v += it.bytes[w] == 4 ? (long long)static_cast<const int*>(it.p[w])[q] : static_cast<const long long*>(it.p[w])[q];
  v = wave_sum(v);
  if (lane == 0) out[w] = v;
}

// Pinned words of a readback: from those that no other thread uses, so there are as many
// as readbacks ever ran at once, however many threads come and go. They stay until the
// process ends (after the HIP runtime may be gone).
struct ReadbackWords {
  long long* p = nullptr;
  static std::mutex& lock() {
    static std::mutex* m = new std::mutex();
    return *m;
  }
  static std::vector<long long*>& unused() {
    static std::vector<long long*>* v = new std::vector<long long*>();
    return *v;
  }
  ReadbackWords() {
    {
      std::lock_guard<std::mutex> g(lock());
      if (!unused().empty()) {
        p = unused().back();
        unused().pop_back();
        return;
      }
    }
    IMPES_HIP_CHECK(hipHostMalloc((void**)&p, 8 * sizeof(long long), hipHostMallocMapped | hipHostMallocPortable));
  }
  void give_back() {  // once the device has written them (a failed readback keeps its words)
    std::lock_guard<std::mutex> g(lock());
    unused().push_back(p);
  }
};

// Order statistic of max(|x|, floor) by its bit pattern (positive doubles order like
// their bits), digit by digit from the top: a histogram of the digit over the values
// that share the digits found so far, then the bin that holds the k-th value.
__device__ __forceinline__ unsigned long long abs_bits(double x, double floor) {
  return (unsigned long long)__double_as_longlong(fmax(fabs(x), floor));
}
struct SelectState {
  unsigned long long prefix;  // digits found, in place
  long long k;                // rank among the values that share them
};

// one workgroup, digits of 8 bits, the values re-read from the L2
constexpr int kSelectSmall = 32768;
__global__ __launch_bounds__(1024) void k_select_small(const double* __restrict__ x, int n, long long k, double floor,
                                                       SelectState* __restrict__ st) {
  __shared__ int hist[256];
  __shared__ unsigned long long prefix_s;
  __shared__ long long k_s;
  unsigned long long prefix = 0, mask = 0;
  for (int shift = 56; shift >= 0; shift -= 8) {
    if (threadIdx.x < 256) hist[threadIdx.x] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
      const unsigned long long b = abs_bits(x[i], floor);
      if ((b & mask) == prefix) atomicAdd(&hist[b >> shift & 255], 1);
    }
    __syncthreads();
    if (threadIdx.x < kWave) {  // lane l: bins 4 l .. 4 l + 3
      const int l = threadIdx.x;
      int h[4], c = 0;
      for (int q = 0; q < 4; ++q) c += h[q] = hist[4 * l + q];
      const int incl = wave_incl_scan(c);
      long long r = k - (incl - c);
      if (r >= 0 && r < c) {
        int q = 0;
        while (r >= h[q]) r -= h[q++];
        prefix_s = prefix | (unsigned long long)(4 * l + q) << shift;
        k_s = r;
      }
    }
    __syncthreads();
    prefix = prefix_s;
    k = k_s;
    mask |= 255ull << shift;
  }
  if (threadIdx.x == 0) {
    st->prefix = prefix;
    st->k = k;
  }
}

// the whole device, digits of 11 bits (the last of 9)
constexpr int kSelectBins = 2048;
__global__ __launch_bounds__(256) void k_select_hist(const double* __restrict__ x, long long n, double floor, int shift,
                                                     unsigned long long mask, const SelectState* __restrict__ st,
                                                     int* __restrict__ hist) {
  __shared__ int h[kSelectBins];
  for (int b = threadIdx.x; b < kSelectBins; b += blockDim.x) h[b] = 0;
  __syncthreads();
  const unsigned long long prefix = st->prefix;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const unsigned long long b = abs_bits(x[i], floor);
    if ((b & mask) == prefix) atomicAdd(&h[b >> shift & (kSelectBins - 1)], 1);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < kSelectBins; b += blockDim.x)
    if (h[b]) atomicAdd(&hist[b], h[b]);
}
// start (k >= 0): the state; else the bin of the k-th value; hist cleared either way
__global__ __launch_bounds__(kScanBlock) void k_select_pick(int shift, long long k, SelectState* __restrict__ st,
                                                            int* __restrict__ hist) {
  __shared__ long long lds[kScanBlock / kWave + 1];
  constexpr int per = kSelectBins / kScanBlock;
  int h[per];
  long long c = 0;
#pragma unroll
  for (int q = 0; q < per; ++q) {
    h[q] = k >= 0 ? 0 : hist[threadIdx.x * per + q];
    c += h[q];
    hist[threadIdx.x * per + q] = 0;
  }
  if (k >= 0) {
    if (threadIdx.x == 0) *st = SelectState{0, k};
    return;
  }
  const SelectState s = *st;
  long long tot;
  long long r = s.k - block_excl_scan<long long>(c, lds, tot);
  if (r >= 0 && r < c) {
#pragma unroll
    for (int q = 0; q < per; ++q) {
      if (r >= 0 && r < h[q]) *st = SelectState{s.prefix | (unsigned long long)(threadIdx.x * per + q) << shift, r};
      r -= h[q];
    }
  }
}

}  // namespace

void scan_i32_to_i64(const int* in, long long* out, long long n, hipStream_t s) { scan_impl<long long>(in, out, n, s); }
void scan_i32_to_i32(const int* in, int* out, long long n, hipStream_t s) { scan_impl<int>(in, out, n, s); }

void segmented_sort_u64(unsigned long long* keys, const long long* seg, long long nseg, long long total,
                        hipStream_t s) {
  if (nseg <= 0) return;
  IMPES_REQUIRE(nseg < (1LL << 31), "segmented sort: too many segments");
  if (nseg <= kSortAny) {
    k_segsort_any<<<(int)nseg, 256, 0, s>>>(keys, seg);
    IMPES_LAUNCH_CHECK();
    if (total <= kSortAnyLds) return;
    k_segsort_few_long<<<(int)(nseg < 512 ? nseg : 512), 1024, 0, s>>>(keys, seg, (int)nseg);
    IMPES_LAUNCH_CHECK();
    return;
  }
  DevBuf<int> counts, lists;
  counts.alloc(kSortBins);
  lists.alloc((size_t)kSortBins * nseg);
  k_fill_zero<<<1, 64, 0, s>>>(counts.p, kSortBins);
  IMPES_LAUNCH_CHECK();
  k_seg_bin<<<grid_for(nseg, 256, 2048), 256, 0, s>>>(seg, nseg, counts.p, lists.p);
  IMPES_LAUNCH_CHECK();
  // the grids are sized without the classes' counts: workgroups walk their class
  auto grid = [&](int most) { return (int)(nseg < most ? nseg : most); };
  const int* L = lists.p;
  const int* c = counts.p;
  k_segsort_regs<<<grid_for(nseg, 256, 8192), 256, 0, s>>>(keys, seg, L, c);
  k_segsort_bin<64, 64><<<grid(8192), 64, 0, s>>>(keys, seg, L + nseg, c + 1);
  k_segsort_bin<256, 128><<<grid(8192), 128, 0, s>>>(keys, seg, L + 2 * nseg, c + 2);
  k_segsort_bin<1024, 256><<<grid(4096), 256, 0, s>>>(keys, seg, L + 3 * nseg, c + 3);
  k_segsort_bin<4096, 512><<<grid(1024), 512, 0, s>>>(keys, seg, L + 4 * nseg, c + 4);
  k_segsort_bin<8192, 1024><<<grid(512), 1024, 0, s>>>(keys, seg, L + 5 * nseg, c + 5);
  k_segsort_global<<<grid(256), 1024, 0, s>>>(keys, seg, L + 6 * nseg, c + 6);
  IMPES_LAUNCH_CHECK();
  sync_before_release(s);  // the bin lists must outlive the kernels
}

int launch_sum_i32(const int* x, long long n, long long* part, hipStream_t s) {
  if (n <= 0) return 0;
  const int m = grid_for(n, 1024, kSumParts);
  k_sum_i32<<<m, 256, 0, s>>>(x, n, part);
  IMPES_LAUNCH_CHECK();
  return m;
}

int launch_count_i8(const signed char* x, long long n, signed char v, long long* part, hipStream_t s) {
  if (n <= 0) return 0;
  const int m = grid_for(n, 1024, kSumParts);
  k_count_i8<<<m, 256, 0, s>>>(x, n, v, part);
  IMPES_LAUNCH_CHECK();
  return m;
}

int Readback::add(const void* p, int bytes, int m) {
  IMPES_REQUIRE(n_ < 8, "readback: too many values");
  p_[n_] = p;
  bytes_[n_] = bytes;
  m_[n_] = m;
  return n_++;
}

void Readback::fetch(hipStream_t s) {
  if (n_ == 0) return;
  ReadbackWords words;
  long long* w = words.p;
  long long* dev = nullptr;
  IMPES_HIP_CHECK(hipHostGetDevicePointer((void**)&dev, w, 0));
  ReadItems it{};
  for (int q = 0; q < n_; ++q) {
    it.p[q] = p_[q];
    it.bytes[q] = bytes_[q];
    it.m[q] = m_[q];
  }
  k_readback<<<1, n_ * kWave, 0, s>>>(it, dev);
  IMPES_LAUNCH_CHECK();
  IMPES_HIP_CHECK(hipStreamSynchronize(s));
  for (int q = 0; q < n_; ++q) v_[q] = static_cast<volatile long long*>(w)[q];
  words.give_back();
}

long long sum_i32(const int* x, long long n, hipStream_t s) {
  if (n <= 0) return 0;
  DevBuf<long long> part;
  part.alloc(kSumParts);
  Readback r;
  r.sum(part.p, launch_sum_i32(x, n, part.p, s));
  r.fetch(s);
  return r[0];
}

double select_abs_f64(const double* x, long long n, long long k, double floor, hipStream_t s) {
  IMPES_REQUIRE(n >= 1 && k >= 0 && k < n && floor > 0.0, "select: bad rank");
  DevBuf<SelectState> st;
  DevBuf<int> hist;
  st.alloc(1);
  if (n <= kSelectSmall) {
    k_select_small<<<1, 1024, 0, s>>>(x, (int)n, k, floor, st.p);
    IMPES_LAUNCH_CHECK();
  } else {
    hist.alloc(kSelectBins);
    k_select_pick<<<1, kScanBlock, 0, s>>>(0, k, st.p, hist.p);
    IMPES_LAUNCH_CHECK();
    unsigned long long mask = 0;
    for (int shift = 53; shift > -11; shift -= 11) {
      const int sh = shift < 0 ? 0 : shift;  // the last digit overlaps the one before, whose bits then all agree
      k_select_hist<<<grid_for(n, 2048, 512), 256, 0, s>>>(x, n, floor, sh, mask, st.p, hist.p);
      IMPES_LAUNCH_CHECK();
      k_select_pick<<<1, kScanBlock, 0, s>>>(sh, -1, st.p, hist.p);
      IMPES_LAUNCH_CHECK();
      mask |= (unsigned long long)(kSelectBins - 1) << sh;
    }
  }
  Readback r;
  r.i64(reinterpret_cast<const long long*>(&st.p->prefix));
  r.fetch(s);
  const long long bits = r[0];
  double v;
  std::memcpy(&v, &bits, sizeof(v));
  return v;
}

}  // namespace impes
