// The dispatch's per-chunk work as device functions: the histogram of a chunk and its stable
// scatter.  moe_dispatch.hip runs them as kernels of their own; the prefill runs them inside
// launches that are there anyway (moe_prefill.hip).
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

// Chunk c's stable scatter; the workgroup of chunk 0 also writes offsets[e] (E + 1 entries)
// and, when asked for, the tile table.  256 threads.  kShared: ids and counts were written by
// other workgroups of the same launch (device-scope loads).
struct ScatterArgs {
  const int32_t* ids;
  int n, E;
  const int32_t* counts;
  int nchunks;
  int32_t *offsets, *order, *inv;
  uint32_t* tiles;
  int* ntiles;
  int cap, shared_rows, bm;
};
template <bool kShared>
__device__ __forceinline__ void dispatch_scatter_block(const ScatterArgs& a, int c) {
  __shared__ int slot[4][256];  // per wave: counts, then next output slot per expert
  __shared__ int wsum[4];
  const int n = a.n, E = a.E, nchunks = a.nchunks;
  int32_t *offsets = a.offsets, *order = a.order, *inv = a.inv;
  auto ld = [](const int32_t* p) {
    return kShared ? (int)ld_dev_u32(reinterpret_cast<const uint32_t*>(p)) : *p;
  };
  const int tid = threadIdx.x, wave = wave_id(), lane = tid & 63;
  for (int i = tid; i < 4 * 256; i += 256) (&slot[0][0])[i] = 0;
  // This wave's assignments (loaded first, so that their latency overlaps the count reads).
  const int begin = c * kDispatchChunk + 256 * wave;
  int ev[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = begin + 64 * j + lane;
    ev[j] = i < n ? ld(a.ids + i) : -1;
  }
  // Thread e: expert e's assignments in the chunks before this one and in all chunks;
  // the expert's offset is the exclusive scan of the totals (wave scans, then the four
  // wave sums).  The counts are read 32 chunks at a time, all loads in flight together.
  int before = 0, total = 0;
  if (tid < E) {
    for (int q0 = 0; q0 < nchunks; q0 += 32) {
      int v[32];
#pragma unroll
      for (int i = 0; i < 32; ++i) v[i] = q0 + i < nchunks ? ld(a.counts + (size_t)(q0 + i) * E + tid) : 0;
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        before += q0 + i < c ? v[i] : 0;
        total += v[i];
      }
    }
  }
  int incl = total;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(incl, d, 64);
    if (lane >= d) incl += y;
  }
  if (lane == 63) wsum[wave] = incl;
  unsigned long long same[4];
  __syncthreads();
  // Lanes of one round with the same expert agree on every bit of the id.
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int e = ev[j];
    const bool ok = e >= 0 && e < E;
    unsigned long long m = __ballot(ok);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const unsigned long long bb = __ballot((e >> b) & 1);
      m &= ((e >> b) & 1) ? bb : ~bb;
    }
    same[j] = ok ? m : 0ull;
    // The last lane of each expert group adds the group's size (one writer per expert).
    if (ok && (m >> lane) == 1ull) slot[wave][e] += __popcll(m);
  }
  __syncthreads();
  // Expert e's first slot for wave w: offset + earlier chunks + counts of waves 0..w-1.
  // (Thread E's exclusive prefix is the number of routed rows.)
  int woff = 0;
  for (int w = 0; w < wave; ++w) woff += wsum[w];
  const int offset = woff + incl - total;
  if (tid < E) {
    if (c == 0) {
      offsets[tid] = offset;
      if (tid == E - 1) offsets[E] = offset + total;
    }
    int run = offset + before;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int v = slot[w][tid];
      slot[w][tid] = run;
      run += v;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int e = ev[j];
    if (same[j]) {
      const int pos = slot[wave][e] + __popcll(same[j] & ((1ull << lane) - 1ull));
      const int i = begin + 64 * j + lane;
      order[pos] = i;
      if (inv) inv[i] = pos;
    }
    if (same[j] && (same[j] >> lane) == 1ull) slot[wave][e] += __popcll(same[j]);
  }
  // The grouped GEMM's tile table (when asked for): routed group e holds sorted rows
  // [offset, offset + total); the shared group (shared_rows > 0) starts at row n (after
  // every assignment, whether or not its id was valid), where the GEMM places it.
  if (c == 0 && a.tiles) {
    __shared__ int tsum[kTileClasses][4];
    const int ng = E + (a.shared_rows > 0 ? 1 : 0);
    const int gb = tid < E ? offset : n;
    tile_table_block<4>(tid, ng, gb, gb + (tid < E ? total : a.shared_rows), a.tiles, a.ntiles, a.cap, a.bm, tsum);
  }
}

}  // namespace rmoe
