// q4nx format kernels: pack_gemv <-> device tile layout, and the device quantizer.
//
// pack_gemv layout: quant/q4nx.py:335-393 (32x256 blocks of 5,120 B, block order
// ((slice*k_blocks + kb)*4 + r), scales/mins [group][row], codes in
// (half, group, col, row16) order with two rows per byte).  The device tile layout
// is described in rmoe_internal.h.
#include "rmoe_internal.h"

namespace rmoe {
namespace {

// Position of (row r, group g) inside a pack_gemv buffer.
struct PackPos {
  size_t base;  // block byte offset
  int r32, half, r16, gg;
};

__device__ __forceinline__ PackPos pack_pos(int r, int g, int K) {
  const int kblocks = K / 256;
  const int slice = r / 128, rw = (r % 128) / 32, r32 = r % 32;
  const int kb = g / 8, gg = g % 8;
  PackPos p;
  p.base = ((size_t)(slice * kblocks + kb) * 4 + rw) * 5120;
  p.r32 = r32;
  p.half = r32 / 16;
  p.r16 = r32 % 16;
  p.gg = gg;
  return p;
}

// Column c (0..31) of a group -> (dword, nibble) inside the lane's 16 bytes.
__device__ __forceinline__ int tile_nibble_index(int c) {
  const int d = c >> 3, w = c & 7;
  const int q = (w & 1) ? (w >> 1) + 4 : (w >> 1);
  return d * 8 + q;  // nibble index 0..31 over the 4 dwords
}

// Thread = (tile, j, lane): gathers row (64*rt + lane), group (4*kt + j).
__global__ void relayout_in_kernel(const uint8_t* __restrict__ packed, uint8_t* __restrict__ tiles, int M, int K) {
  const int G = K / 32, nkt = K / 128;
  const size_t n = (size_t)M * G;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n) return;
  const int lane = idx & 63;
  const size_t rest = idx >> 6;
  const int j = rest & 3;
  const size_t tile = rest >> 2;
  const int rt = (int)(tile / nkt), kt = (int)(tile % nkt);
  const int r = rt * 64 + lane, g = kt * 4 + j;
  const PackPos p = pack_pos(r, g, K);
  const uint16_t* sm = reinterpret_cast<const uint16_t*>(packed + p.base);
  const uint32_t scale = sm[p.gg * 32 + p.r32];
  const uint32_t mn = sm[256 + p.gg * 32 + p.r32];
  uint32_t w[4] = {0u, 0u, 0u, 0u};
  const uint8_t* cbase = packed + p.base + 1024 + (size_t)((p.half * 8 + p.gg) * 32) * 8 + (p.r16 >> 1);
  const int shift = (p.r16 & 1) ? 4 : 0;
#pragma unroll 8
  for (int c = 0; c < 32; ++c) {
    const uint32_t code = (cbase[c * 8] >> shift) & 15u;
    const int ni = tile_nibble_index(c);
    w[ni >> 3] |= code << (4 * (ni & 7));
  }
  uint8_t* t = tiles + tile * kTileBytes;
  *reinterpret_cast<uint4*>(t + j * 1024 + lane * 16) = make_uint4(w[0], w[1], w[2], w[3]);
  *reinterpret_cast<uint32_t*>(t + kCodeBytes + lane * 16 + j * 4) = scale | (mn << 16);
}

// One workgroup per 64 rows x 256 columns: two K tiles, 10 KB in a row in the tile layout,
// become two pack_gemv blocks, 10 KB in a row there, through LDS, so that both sides move
// 16 bytes per lane.  (One thread per row pair and group, storing 32 single bytes 8 apart,
// took 16.4 us for 1536 x 2048; this takes 5.3 us.)  A group's 1 KB of codes is followed by
// 16 bytes of padding in LDS: the lanes of a wave read one row of four groups at a time.
constexpr int kRelayoutGroup = 1024 + 16;  // bytes per group of 64 rows in LDS
__global__ __launch_bounds__(256) void relayout_out_kernel(const uint8_t* __restrict__ tiles,
                                                           uint8_t* __restrict__ packed, int K, unsigned first) {
  __shared__ __attribute__((aligned(16))) uint8_t codes[8 * kRelayoutGroup];
  __shared__ __attribute__((aligned(16))) uint32_t sm[2][64 * 4];
  const int kblocks = K / 256, tid = threadIdx.x;
  // Workgroups in the order of the output: the two 64-row bands of a 128-row slice alternate.
  const unsigned unit = first + blockIdx.x;
  const int band = (int)(unit / (2 * kblocks)) * 2 + (int)(unit & 1), kb = (int)((unit >> 1) % kblocks);
  const uint4* src = reinterpret_cast<const uint4*>(tiles + ((size_t)band * kblocks + kb) * 2 * kTileBytes);
  constexpr int kUnits = kTileBytes / 16;  // 320: four groups of 64 rows, then the scale|min words
  uint4 v[3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (tid + 256 * i < 2 * kUnits) v[i] = src[tid + 256 * i];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int u = tid + 256 * i;
    if (u >= 2 * kUnits) continue;
    const int t = u / kUnits, o = u % kUnits;
    if (o < 256) *reinterpret_cast<uint4*>(codes + (4 * t + (o >> 6)) * kRelayoutGroup + (o & 63) * 16) = v[i];
    else *reinterpret_cast<uint4*>(&sm[t][(o - 256) * 4]) = v[i];
  }
  __syncthreads();
  uint4* dst = reinterpret_cast<uint4*>(packed + (size_t)blockIdx.x * kRelayoutBytes);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int u = tid + 256 * i;
    if (u >= 2 * kUnits) continue;
    const int blk = u / kUnits, o = u % kUnits;
    uint32_t w[4];
    if (o < 64) {  // 8 rows' scales (units 0..31) or mins of one group
      const int gg = (o & 31) >> 2, r0 = 32 * blk + 8 * (o & 3), hi = o >> 5;
      const uint32_t* p = &sm[gg >> 2][r0 * 4 + (gg & 3)];
      const uint32_t sel = hi ? 0x07060302u : 0x05040100u;
#pragma unroll
      for (int q = 0; q < 4; ++q) w[q] = __builtin_amdgcn_perm(p[8 * q + 4], p[8 * q], sel);
    } else {  // columns 2 cp and 2 cp + 1 of one group, 16 rows: 8 bytes each, two rows per byte
      const int q = o - 64, cp = q & 15, gg = (q >> 4) & 7, r0 = 32 * blk + 16 * (q >> 7);
      const uint8_t* p = codes + gg * kRelayoutGroup + r0 * 16 + 4 * (cp >> 2);
      const int sh = 4 * (cp & 3);  // nibbles cp % 4 (even column) and cp % 4 + 4 (odd column)
      uint32_t b[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t lo = *reinterpret_cast<const uint32_t*>(p + 32 * j) >> sh;
        const uint32_t hi = *reinterpret_cast<const uint32_t*>(p + 32 * j + 16) >> sh;
        b[j] = (lo & 0x000f000fu) | ((hi & 0x000f000fu) << 4);  // bytes 0 and 2
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = 4 * (j & 1);  // even column: bytes 0 of b; odd column: bytes 2
        const uint32_t sel = j < 2 ? 0x0c0c0400u : 0x0c0c0602u;
        const uint32_t p0 = __builtin_amdgcn_perm(b[k + 1], b[k], sel), p1 = __builtin_amdgcn_perm(b[k + 3], b[k + 2], sel);
        w[j] = p0 | (p1 << 16);
      }
    }
    dst[u] = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// ------------------------------------------------------------ Q4_K -> tiles --
// llama.cpp block_q4_K (quant/gguf_q4k.py:189-233): 144 bytes per 256 weights of a row --
// d (fp16), dmin (fp16), eight 6-bit scales and mins in 12 bytes, 128 code bytes (sub-
// block 2p = low nibbles of bytes 32p..32p+31, 2p+1 = their high nibbles).  q4nx keeps
// every code; group j's parameters are RTNE bf16 of d*sc[j] and -dmin*mn[j] (exact fp32
// products).  Thread = (tile row band, K tile, group j, lane): row row0 + 64*band + lane,
// group 4*kt + j of a tile matrix Kt wide; groups at or past K are the zero padding
// (codes 0, scale 0, min 0).
__global__ void q4k_to_tiles_kernel(const uint8_t* __restrict__ q4k, int M, int K, uint8_t* __restrict__ tiles,
                                    int Kt, int row0) {
  const int nkt = Kt / 128;
  const size_t n = (size_t)M * (Kt / 32);
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n) return;
  const int lane = (int)(idx & 63);
  const size_t rest = idx >> 6;
  const int j = (int)(rest & 3);
  const size_t rest2 = rest >> 2;
  const int kt = (int)(rest2 % nkt), band = (int)(rest2 / nkt);
  const int r = 64 * band + lane, g = 4 * kt + j;
  uint32_t w[4] = {0u, 0u, 0u, 0u};
  uint32_t sm = 0u;
  if (32 * g < K) {
    const uint8_t* b = q4k + ((size_t)r * (K / 256) + g / 8) * 144;
    const int jj = g % 8;
    const uint16_t dh = (uint16_t)(b[0] | (b[1] << 8)), mh = (uint16_t)(b[2] | (b[3] << 8));
    const float d = (float)__builtin_bit_cast(_Float16, dh), dmin = (float)__builtin_bit_cast(_Float16, mh);
    uint32_t sc, mn;
    if (jj < 4) {
      sc = b[4 + jj] & 0x3Fu;
      mn = b[8 + jj] & 0x3Fu;
    } else {
      sc = (b[12 + jj - 4] & 0x0Fu) | ((uint32_t)(b[4 + jj - 4] >> 6) << 4);
      mn = (uint32_t)(b[12 + jj - 4] >> 4) | ((uint32_t)(b[8 + jj - 4] >> 6) << 4);
    }
    sm = f32_to_bf16(__fmul_rn(d, (float)sc)) | (f32_to_bf16(__fmul_rn(-dmin, (float)mn)) << 16);
    const uint8_t* cb = b + 16 + 32 * (jj / 2);
    const int shift = (jj & 1) ? 4 : 0;
#pragma unroll 8
    for (int c = 0; c < 32; ++c) {
      const uint32_t code = ((uint32_t)cb[c] >> shift) & 15u;
      const int ni = tile_nibble_index(c);
      w[ni >> 3] |= code << (4 * (ni & 7));
    }
  }
  const int R = row0 + r;
  uint8_t* t = tiles + ((size_t)(R / 64) * nkt + kt) * kTileBytes;
  *reinterpret_cast<uint4*>(t + j * 1024 + (R % 64) * 16) = make_uint4(w[0], w[1], w[2], w[3]);
  *reinterpret_cast<uint32_t*>(t + kCodeBytes + (R % 64) * 16 + j * 4) = sm;
}

// ------------------------------------------------------------------ quantizer --
// Bit-exact restatement of quant/q4nx.py:127-200 per (row, group), in float64 where
// the reference uses float64.
__device__ __forceinline__ float bits_f(uint32_t u) { return __uint_as_float(u); }

__device__ __forceinline__ float bf16_floor_f32(float x) {
  const uint32_t u = __float_as_uint(x);
  const uint32_t bump = ((u >> 31) && (u & 0xffffu)) ? 1u : 0u;
  return bits_f(((u >> 16) + bump) << 16);
}

__device__ __forceinline__ float bf16_ceil_f64(double x) {
  float f = __double2float_rn(x);
  if ((double)f < x) f = nextafterf(f, __builtin_inff());
  const uint32_t u = __float_as_uint(f);
  const uint32_t bump = (!(u >> 31) && (u & 0xffffu)) ? 1u : 0u;
  return bits_f(((u >> 16) + bump) << 16);
}

__device__ __forceinline__ float bf16_next_up(float x) {
  uint32_t h = __float_as_uint(x) >> 16;
  if (h == 0x8000u) h = 0u;
  uint32_t nx;
  if (h == 0u) nx = 1u;
  else if (h & 0x8000u) nx = (h == 0x8001u) ? 0u : h - 1u;
  else nx = h + 1u;
  return bits_f(nx << 16);
}

// Quantize one (row, group) of 32 fp32 values and store it at (tile, j, lane).
__device__ void quantize_group(const float (&v)[32], uint8_t* tile, int j, int lane, int* err) {
  bool finite = true;
#pragma unroll
  for (int c = 0; c < 32; ++c) finite = finite && isfinite(v[c]);
  if (!finite) atomicOr(err, 1);
  float lo = v[0], hi = v[0];
#pragma unroll
  for (int c = 1; c < 32; ++c) {
    lo = fminf(lo, v[c]);
    hi = fmaxf(hi, v[c]);
  }
  const float minq = bf16_floor_f32(lo);
  const double min64 = (double)minq, hi64 = (double)hi;
  const double span = hi64 - min64;
  float sc = bf16_ceil_f64(span / 15.0);
  for (int it = 0; it < 64; ++it) {
    if (!isfinite(sc)) break;
    if (min64 + 15.0 * (double)sc >= hi64) break;
    sc = bf16_next_up(sc);
  }
  const bool flat = span == 0.0;
  if (flat) sc = 0.f;
  if (!isfinite(minq) || !isfinite(sc)) atomicOr(err, 2);
  const double div = flat ? 1.0 : (double)sc;
  uint32_t words[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int c = 0; c < 32; ++c) {
    double q = rint(((double)v[c] - min64) / div);
    q = q < 0.0 ? 0.0 : (q > 15.0 ? 15.0 : q);
    const uint32_t code = flat ? 0u : (uint32_t)q;
    const int ni = tile_nibble_index(c);
    words[ni >> 3] |= code << (4 * (ni & 7));
  }
  *reinterpret_cast<uint4*>(tile + j * 1024 + lane * 16) = make_uint4(words[0], words[1], words[2], words[3]);
  const uint32_t sb = __float_as_uint(sc) >> 16, mb = __float_as_uint(minq) >> 16;
  *reinterpret_cast<uint32_t*>(tile + kCodeBytes + lane * 16 + j * 4) = sb | (mb << 16);
}

// Thread = (tile, j, lane) -> (row, group), coalesced on the tile side.
struct GroupIndex {
  size_t tile;
  int j, lane, r, g;
};
__device__ __forceinline__ GroupIndex group_index(size_t idx, int nkt) {
  GroupIndex gi;
  gi.lane = idx & 63;
  const size_t rest = idx >> 6;
  gi.j = rest & 3;
  gi.tile = rest >> 2;
  const int rt = (int)(gi.tile / nkt), kt = (int)(gi.tile % nkt);
  gi.r = rt * 64 + gi.lane;
  gi.g = kt * 4 + gi.j;
  return gi;
}

// One workgroup per tile of 64 rows x 128 columns, whose fp32 values come through LDS: a
// wave loads its 16 rows by whole 256-byte lines, then takes group `wave` of row `lane`.
// (A thread loading its own 128 bytes touched 64 lines per load: 15.4 us for 1536 x 2048;
// this takes 9.7 us.  The rest is the serial fp64 divisions of 1.5 waves per SIMD.)
constexpr int kQuantRow = 128 + 4;  // floats per row in LDS: 16-byte reads of 64 rows spread over the banks
__global__ __launch_bounds__(256) void quantize_kernel(const float* __restrict__ w, int K, int ld, int k_valid,
                                                       uint8_t* __restrict__ tiles, int* __restrict__ err) {
  __shared__ __attribute__((aligned(16))) float rows[64 * kQuantRow];
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int nkt = K / kTileCols, rt = blockIdx.x / nkt, kt = blockIdx.x % nkt;
  const float* src = w + (size_t)(rt * 64 + 16 * wave) * ld + kt * kTileCols;
  float x[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const int c = lane + 64 * (i & 1);
    x[i] = kt * kTileCols + c < k_valid ? src[(size_t)(i >> 1) * ld + c] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 32; ++i) rows[(16 * wave + (i >> 1)) * kQuantRow + lane + 64 * (i & 1)] = x[i];
  __syncthreads();
  float v[32];
#pragma unroll
  for (int c = 0; c < 32; c += 4) {
    const float4 f = *reinterpret_cast<const float4*>(&rows[lane * kQuantRow + 32 * wave + c]);
    v[c] = f.x;
    v[c + 1] = f.y;
    v[c + 2] = f.z;
    v[c + 3] = f.w;
  }
  quantize_group(v, tiles + (size_t)blockIdx.x * kTileBytes, wave, lane, err);
}

// Counter-based N(0, std) weights: splitmix64 of (seed, row*k_valid + col) -> Box-Muller.
__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

__device__ __forceinline__ float synth_normal(uint64_t seed, uint64_t i) {
  const uint64_t h = splitmix64(seed * 0x100000001B3ull ^ splitmix64(i));
  const float u1 = ((uint32_t)(h >> 40) + 1u) * (1.0f / 16777217.0f);  // (0, 1)
  const float u2 = (uint32_t)(h & 0xFFFFFFu) * (1.0f / 16777216.0f);   // [0, 1)
  return sqrtf(-2.0f * logf(u1)) * cospif(2.0f * u2);
}

__global__ void synth_quantize_kernel(uint64_t seed, float std, int M, int K, int k_valid,
                                      uint8_t* __restrict__ tiles, int* __restrict__ err) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)M * (K / 32)) return;
  const GroupIndex gi = group_index(idx, K / 128);
  float v[32];
#pragma unroll
  for (int c = 0; c < 32; ++c) {
    const int col = gi.g * 32 + c;
    v[c] = col < k_valid ? std * synth_normal(seed, (uint64_t)gi.r * k_valid + col) : 0.f;
  }
  quantize_group(v, tiles + gi.tile * kTileBytes, gi.j, gi.lane, err);
}

}  // namespace

hipError_t launch_relayout_in(const uint8_t* packed, uint8_t* tiles, int M, int K, hipStream_t st) {
  const size_t n = (size_t)M * (K / 32);
  const unsigned blocks = (unsigned)((n + 255) / 256);
  hipLaunchKernelGGL(relayout_in_kernel, dim3(blocks), dim3(256), 0, st, packed, tiles, M, K);
  return hipGetLastError();
}

hipError_t launch_q4k_to_tiles(const uint8_t* q4k, int M, int K, uint8_t* tiles, int Kt, int row0, hipStream_t st) {
  if (M % 64 || row0 % 64 || K % 256 || Kt % 128 || K > Kt) return hipErrorInvalidValue;
  const size_t n = (size_t)M * (Kt / 32);
  const unsigned blocks = (unsigned)((n + 255) / 256);
  hipLaunchKernelGGL(q4k_to_tiles_kernel, dim3(blocks), dim3(256), 0, st, q4k, M, K, tiles, Kt, row0);
  return hipGetLastError();
}

hipError_t launch_relayout_out(const uint8_t* tiles, uint8_t* packed, int M, int K, size_t first, size_t n,
                               hipStream_t st) {
  const size_t total = (size_t)(M / 64) * (K / 256);
  if (M % 128 || K % 256 || first >= total) return hipErrorInvalidValue;
  const size_t count = n ? min(n, total - first) : total - first;
  hipLaunchKernelGGL(relayout_out_kernel, dim3((unsigned)count), dim3(256), 0, st, tiles, packed, K, (unsigned)first);
  return hipGetLastError();
}

hipError_t launch_quantize(const float* w, int M, int K, int ld, int k_valid, uint8_t* tiles, int* err,
                           hipStream_t st) {
  if (M % 64 || K % kTileCols) return hipErrorInvalidValue;
  const unsigned blocks = (unsigned)((M / 64) * (K / kTileCols));
  hipLaunchKernelGGL(quantize_kernel, dim3(blocks), dim3(256), 0, st, w, K, ld, k_valid, tiles, err);
  return hipGetLastError();
}

hipError_t launch_synth_quantize(uint64_t seed, float std, int M, int K, int k_valid, uint8_t* tiles, int* err,
                                 hipStream_t st) {
  const size_t n = (size_t)M * (K / 32);
  const unsigned blocks = (unsigned)((n + 255) / 256);
  hipLaunchKernelGGL(synth_quantize_kernel, dim3(blocks), dim3(256), 0, st, seed, std, M, K, k_valid, tiles, err);
  return hipGetLastError();
}

}  // namespace rmoe
