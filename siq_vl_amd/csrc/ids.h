// Sorting runs of token ids, shared by the embedding-table gradient and the
// cross-entropy's label terms.
#pragma once
#include "common.h"

namespace siq {

// Ids are sorted in chunks of kIdChunk positions, one 1024-thread workgroup
// each: 64-bit keys (id << 32 | position in the chunk), kNoKey (sorts last) for
// positions without an id.
constexpr int kIdChunk = 2048;  // two keys per thread
constexpr uint64_t kNoKey = ~0ull;
static_assert(kIdChunk == 2 * 1024, "one compare-exchange pair per thread and stage");

// Bitonic network over the np2 (a power of two, at most kIdChunk) keys in
// LDS: in each stage thread t owns the pair (i, i + j), i = t with a zero bit
// inserted at j.  The keys are in LDS (behind a barrier) on entry, sorted
// behind a barrier on exit.
__device__ __forceinline__ void sort_keys(uint64_t* sk, int np2) {
  const int t = threadIdx.x;
  for (int k = 2; k <= np2; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      const int i = 2 * t - (t & (j - 1));
      if (i + j < np2) {
        const uint64_t a = sk[i], b = sk[i + j];
        if ((a > b) == ((i & k) == 0)) {
          sk[i] = b;
          sk[i + j] = a;
        }
      }
      __syncthreads();
    }
  }
}

// The run [first, end) of id v among the kIdChunk sorted keys (both bounds
// searched together: their loads overlap).
__device__ __forceinline__ int2 id_run(const uint64_t* keys, uint32_t v) {
  const uint64_t a = (uint64_t)v << 32, b = ((uint64_t)v + 1) << 32;
  int lo = 0, hi = 0;  // keys below a, below b, found so far
#pragma unroll
  for (int step = kIdChunk / 2; step > 0; step >>= 1) {
    const uint64_t x = keys[lo + step - 1], y = keys[hi + step - 1];
    lo += x < a ? step : 0;
    hi += y < b ? step : 0;
  }
  lo += keys[lo] < a ? 1 : 0;  // (at most kIdChunk - 1 here)
  hi += keys[hi] < b ? 1 : 0;
  return make_int2(lo, hi);
}

}  // namespace siq
