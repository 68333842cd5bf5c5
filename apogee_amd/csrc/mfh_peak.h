// Where a filter launch writes its peaks: separate index and value arrays, or
// 16-byte {int64 index; complex64 value} records.  Either may be page-locked
// host memory: a caller's result buffer is then written by the filter itself,
// with no readback launch behind it (6 us for 16384 peaks, and the gap).
#pragma once
#include "mfh_dft.h"

namespace mfh {

struct PeakOut {
  int64_t *idx = nullptr;
  cf *val = nullptr;
  int4 *rec = nullptr;  // if set, used instead of idx and val
  __device__ __forceinline__ void put(long long o, long long k, cf z) const {
    if (rec) {
      // one 16-byte store: over the host link, half the packets of two
      rec[o] = int4{(int)(unsigned)(unsigned long long)k, (int)(k >> 32), __float_as_int(z.x), __float_as_int(z.y)};
    } else {
      idx[o] = k;
      val[o] = z;
    }
  }
  // a record as put() stores it
  __device__ __forceinline__ void put_record(long long o, int4 r) const {
    if (rec) {
      rec[o] = r;
    } else {
      idx[o] = (long long)(((unsigned long long)(unsigned)r.y << 32) | (unsigned)r.x);
      val[o] = cf{__int_as_float(r.z), __int_as_float(r.w)};
    }
  }
  __device__ __forceinline__ void none(long long o) const { put(o, -1, cf{0.f, 0.f}); }
  PeakOut at(size_t o) const {
    PeakOut r;
    if (rec) {
      r.rec = rec + o;
    } else {
      r.idx = idx + o;
      r.val = val + o;
    }
    return r;
  }
};

}  // namespace mfh
