// Device primitives used by the AMG setup: exclusive scans, a segmented sort of
// 64-bit keys, and integer reductions. All deterministic (no order-dependent
// atomics in anything whose result is observable).
#pragma once

#include "common.h"

namespace impes {

// out[0..n] = exclusive scan of in[0..n-1], out[n] = total. Returns nothing;
// the total can be read from out[n]. Work buffers are allocated internally.
void scan_i32_to_i64(const int* in, long long* out, long long n, hipStream_t s);
void scan_i32_to_i32(const int* in, int* out, long long n, hipStream_t s);

// Sort every segment [seg[i], seg[i+1]) of the `total` keys ascending. Does not wait for
// the stream: the number of segments per length class stays on the device.
void segmented_sort_u64(unsigned long long* keys, const long long* seg, long long nseg, long long total,
                        hipStream_t s);

// Partial sums of an int32 array, and of the count of int8 entries equal to v, into
// part (kSumParts values); returns how many were written (Readback::sum adds them up).
constexpr int kSumParts = 256;
int launch_sum_i32(const int* x, long long n, long long* part, hipStream_t s);
int launch_count_i8(const signed char* x, long long n, signed char v, long long* part, hipStream_t s);

// Device values for the host, up to 8 at once: one kernel writes them to pinned host
// memory and the stream is waited for. A blocking copy of a scalar takes 25 us (a
// blit, its staging and two waits), the kernel and one wait about 12.
class Readback {
 public:
  int i32(const int* p) { return add(p, 4, 1); }
  int i64(const long long* p) { return add(p, 8, 1); }
  int sum(const long long* part, int m) { return add(part, 8, m); }
  void fetch(hipStream_t s);  // later reads see the values as of this point of the stream
  long long operator[](int k) const { return v_[k]; }

 private:
  int add(const void* p, int bytes, int m);
  const void* p_[8] = {};
  int bytes_[8] = {}, m_[8] = {};
  int n_ = 0;
  long long v_[8] = {};
};

// sum of an int32 array (synchronises, returns host value)
long long sum_i32(const int* x, long long n, hipStream_t s);
// one int or long long device->host (synchronises)
inline int read_scalar(const int* dev, hipStream_t s) {
  Readback r;
  r.i32(dev);
  r.fetch(s);
  return (int)r[0];
}
inline long long read_scalar(const long long* dev, hipStream_t s) {
  Readback r;
  r.i64(dev);
  r.fetch(s);
  return r[0];
}

// The k-th smallest (from 0) of max(|x_i|, floor), floor > 0, exactly (synchronises).
double select_abs_f64(const double* x, long long n, long long k, double floor, hipStream_t s);

}  // namespace impes
