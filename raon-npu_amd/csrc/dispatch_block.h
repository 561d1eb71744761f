// The dispatch's histogram of one chunk as a device function: moe_dispatch.hip runs it as a
// kernel of its own, the grouped prefill inside its preparation launch (moe_prefill.hip).
#pragma once

#include "rmoe_internal.h"

namespace rmoe {

// counts[c][e]: assignments of chunk c routed to expert e.  256 threads; hist: 256 ints of LDS.
__device__ __forceinline__ void dispatch_count_block(const int32_t* __restrict__ ids, int n, int E,
                                                     int32_t* __restrict__ counts, int* err, int c, int* hist) {
  hist[threadIdx.x] = 0;
  __syncthreads();
  const int begin = c * kDispatchChunk;
  int ev[kDispatchChunk / 256];
#pragma unroll
  for (int j = 0; j < kDispatchChunk / 256; ++j) {
    const int i = begin + 256 * j + threadIdx.x;
    ev[j] = i < n ? ids[i] : 0x7fffffff;
  }
#pragma unroll
  for (int j = 0; j < kDispatchChunk / 256; ++j) {
    if (ev[j] == 0x7fffffff) continue;
    if (ev[j] >= 0 && ev[j] < E) atomicAdd(&hist[ev[j]], 1);
    else atomicOr(err, 4);
  }
  __syncthreads();
  if ((int)threadIdx.x < E) counts[(size_t)c * E + threadIdx.x] = hist[threadIdx.x];
}

}  // namespace rmoe
