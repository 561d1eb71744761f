// Dense y[T, M] = RTNE(x[T, K] @ W^T), q4nx or bfp16 weights, on bf16 MFMA (wave_gemm.h):
// NumpyBackend.linear (host/backend.py:402-417) with fp32 accumulation and one rounding.
//
// What bounds it: few tokens read the weights once and are bound by that stream (HBM), or
// for small matrices by the latency of one load round and of the final sum; from some 100
// tokens on the VALU work around the MFMAs (unpacking, and for q4nx one FMA per group and
// output) is the bound, which grows with the number of token tiles.  Measured against the
// GEMV kernels that served every token count (four tokens per weight pass): q4nx [1536,
// 2048], 445 tokens 65.8 -> 11.4 us; bfp16 [2176, 2560], 256 tokens 77.6 -> 13.1 us; bfp16
// [260096, 2560], one token 114.5 -> 113.8 us (6.6 TB/s).
//
// One workgroup takes 16 MF tokens x 16 NF weight rows, its W waves a W-th of K each; the
// waves' sums meet in LDS and are added in wave order.  W depends on K only and a row's
// sums do not depend on MF and NF, so a token's result is the same in a batch of any size:
// linear_batch equals stacked linear calls.  (One token of a small q4nx matrix on device
// pointers runs linear_lane_kernel instead, whose last bit may differ.)
#include <algorithm>

#include "wave_gemm.h"

namespace rmoe {
namespace {

constexpr int kPad = 4;  // floats of padding per token row of the partial sums

struct LinMfmaArgs {
  const uint8_t* tiles;
  int M, K, T;
  const uint16_t* x;
  uint16_t* y;
  int n_mt, n_nt;  // token tiles, weight-row tiles
};

// kY8: y is 8-byte aligned (as a branch in one kernel it cost 1 to 6 % at 445 tokens).
template <int kFmt, int MF, int NF, int XI, bool kY8>
__global__ __launch_bounds__(512) void linear_mfma_kernel(LinMfmaArgs a) {
  // Per wave 4096 MF bytes of activation rows, then (after the K loop) its partial sums
  // [16 MF tokens][16 NF + kPad].
  extern __shared__ __attribute__((aligned(16))) float lm_lds[];
  constexpr int kTB = kFmt == RMOE_FMT_BFP16 ? kB16TileBytes : kTileBytes;
  constexpr int kCols = 16 * NF, kStride = kCols + kPad;
  // XCD x takes a contiguous eighth of the tiles, the token tiles of one weight tile back
  // to back, so that they share the weights in one L2.
  const int total = a.n_mt * a.n_nt, per = (total + 7) / 8;
  const int id = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (id >= total) return;
  const int nt = id / a.n_mt, tok0 = (id % a.n_mt) * 16 * MF;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id(), W = blockDim.x >> 6;
  const int l16 = lane & 15, lq = lane >> 4;
  const int nkt = a.K / kTileCols;
  WaveOperands<MF, NF, XI> o;
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int row = nt * kCols + 16 * f;
    o.w[f] = a.tiles + (size_t)(row / kTileRows) * nkt * kTB + (row % kTileRows) * 16;
  }
  o.x = reinterpret_cast<const uint8_t*>(a.x);
  // Rows past T repeat the last token; their results are not stored.
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int i = 0; i < XI; ++i)
      o.xoff[m][i] = (uint32_t)min(tok0 + 16 * m + 4 * i + lq, a.T - 1) * (uint32_t)(2 * a.K) + 16u * (uint32_t)l16;
  o.lds = reinterpret_cast<uint8_t*>(lm_lds) + (size_t)wave * 4096 * MF;
  wg_f32x4 acc[MF][NF];
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[m][f] = wg_f32x4{0.f, 0.f, 0.f, 0.f};
  wave_gemm<kFmt, MF, NF, XI>(o, wave * nkt / W, (wave + 1) * nkt / W, acc);
  __syncthreads();  // the partial sums reuse the waves' activation regions
  float* mine = lm_lds + (size_t)wave * 16 * MF * kStride;
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int i = 0; i < 4; ++i) mine[(16 * m + 4 * lq + i) * kStride + 16 * f + l16] = acc[m][f][i];
  __syncthreads();
  const int nrow = min(16 * MF, a.T - tok0);
  constexpr float kUnit = kFmt == RMOE_FMT_BFP16 ? 4.f : 1.f;  // see wave_gemm.h
  for (int i = tid; i < nrow * (kCols / 4); i += blockDim.x) {
    const int t = i / (kCols / 4), c = 4 * (i % (kCols / 4));
    float4 v = *reinterpret_cast<const float4*>(lm_lds + t * kStride + c);
    for (int w = 1; w < W; ++w) {
      const float4 u = *reinterpret_cast<const float4*>(lm_lds + (size_t)w * 16 * MF * kStride + t * kStride + c);
      v.x += u.x;
      v.y += u.y;
      v.z += u.z;
      v.w += u.w;
    }
    const uint32_t lo = f32_to_bf16(kUnit * v.x) | (f32_to_bf16(kUnit * v.y) << 16);
    const uint32_t hi = f32_to_bf16(kUnit * v.z) | (f32_to_bf16(kUnit * v.w) << 16);
    uint16_t* y = a.y + (size_t)(tok0 + t) * a.M + nt * kCols + c;
    if constexpr (kY8) {
      *reinterpret_cast<uint2*>(y) = make_uint2(lo, hi);
    } else {
      y[0] = (uint16_t)lo;
      y[1] = (uint16_t)(lo >> 16);
      y[2] = (uint16_t)hi;
      y[3] = (uint16_t)(hi >> 16);
    }
  }
}

// Dynamic LDS of W waves: their activation regions, then in the same place their partial sums.
constexpr size_t linear_lds(int MF, int NF, int W) {
  const size_t sums = (size_t)16 * MF * (16 * NF + kPad) * 4, rows = (size_t)4096 * MF;
  return W * (sums > rows ? sums : rows);
}

template <int kFmt, int MF, int NF, int XI>
hipError_t launch(LinMfmaArgs a, hipStream_t st) {
  // Waves per workgroup: four, eight for 64 K tiles and more ([2560, 12032], one token:
  // q4nx 12.1 -> 9.1 us, bfp16 17.0 -> 11.1 us; at K = 2560 eight waves are up to 0.7 us
  // faster for one token and 27 % slower for 445 tokens).
  const int nkt = a.K / kTileCols, W = std::min(nkt, nkt >= 64 ? 8 : 4);
  a.n_mt = (a.T + 16 * MF - 1) / (16 * MF);
  a.n_nt = a.M / (16 * NF);
  const size_t lds = linear_lds(MF, NF, W);
  const size_t total = (size_t)a.n_mt * a.n_nt;
  auto* kernel = (reinterpret_cast<uintptr_t>(a.y) & 7) == 0 ? linear_mfma_kernel<kFmt, MF, NF, XI, true>
                                                             : linear_mfma_kernel<kFmt, MF, NF, XI, false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * ((total + 7) / 8))), dim3(64 * W), lds, st, a);
  return hipGetLastError();
}

// The largest tile that still gives the chip's 256 CUs kFillTiles workgroups: a larger tile
// unpacks the weights for more tokens and reads the tokens for more rows, but fewer
// workgroups than about 1.75 per CU leave CUs idle in the last round ([2176, 2560] q4nx:
// 128 tokens 9.7 us with 16 x 32 tiles (544), 10.3 with 32 x 32 (272); 445 tokens 16.2 us
// with 32 x 64 (476), 17.5 with 32 x 32; [1536, 2048]: 445 tokens 11.1 us with 32 x 32
// (672), 12.7 with 32 x 64 (336)).
constexpr int kFillTiles = 448;

template <int kFmt>
hipError_t pick(const LinMfmaArgs& a, hipStream_t st) {
  auto fills = [&](int mf, int nf) {
    return (size_t)((a.T + 16 * mf - 1) / (16 * mf)) * (size_t)(a.M / (16 * nf)) >= kFillTiles;
  };
  if (a.T <= 4) {  // only the first row quartet of the fragment is loaded
    if (fills(1, 4)) return launch<kFmt, 1, 4, 1>(a, st);
    if (fills(1, 2)) return launch<kFmt, 1, 2, 1>(a, st);
    return launch<kFmt, 1, 1, 1>(a, st);
  }
  if (a.T > 16) {
    if (fills(2, 4)) return launch<kFmt, 2, 4, 4>(a, st);
    if (fills(2, 2)) return launch<kFmt, 2, 2, 4>(a, st);
  } else if (fills(1, 4)) {
    return launch<kFmt, 1, 4, 4>(a, st);
  }
  if (fills(1, 2)) return launch<kFmt, 1, 2, 4>(a, st);
  return launch<kFmt, 1, 1, 4>(a, st);
}

}  // namespace

// 16-byte loads of x rows.
bool linear_mfma_ok(const uint16_t* x) { return (reinterpret_cast<uintptr_t>(x) & 15) == 0; }

// Allow the 32 x 64 tiles of eight waves their 68 KB of dynamic LDS (the others stay under 64).
hipError_t linear_mfma_setup() {
  const void* fns[4] = {(const void*)linear_mfma_kernel<RMOE_FMT_Q4NX, 2, 4, 4, true>,
                        (const void*)linear_mfma_kernel<RMOE_FMT_Q4NX, 2, 4, 4, false>,
                        (const void*)linear_mfma_kernel<RMOE_FMT_BFP16, 2, 4, 4, true>,
                        (const void*)linear_mfma_kernel<RMOE_FMT_BFP16, 2, 4, 4, false>};
  for (const void* f : fns) {
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)linear_lds(2, 4, 8));
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

static_assert((size_t)linear_mfma_max_tokens(65536, 512) / 32 * (65536 / 64) * 256 < ((size_t)1 << 32) &&
                  (size_t)linear_mfma_max_tokens(1 << 22, 8192) / 32 * ((1 << 22) / 64) * 512 < ((size_t)1 << 32),
              "grid within HIP's limit");
static_assert((size_t)linear_mfma_max_tokens(128, 8192) * 8192 * 2 <= ((size_t)1 << 32), "x within 32-bit offsets");

hipError_t launch_linear_mfma(const uint8_t* tiles, int fmt, int M, int K, const uint16_t* x, int T, uint16_t* y,
                              hipStream_t st) {
  // A token's bytes do not depend on its batch: one too large for a launch is several.
  const int rows = linear_mfma_max_tokens(M, K);
  for (int t0 = 0; t0 < T; t0 += std::min(rows, T - t0)) {
    LinMfmaArgs a{tiles, M, K, std::min(rows, T - t0), x + (size_t)t0 * K, y + (size_t)t0 * M, 0, 0};
    const hipError_t e = fmt == RMOE_FMT_BFP16 ? pick<RMOE_FMT_BFP16>(a, st) : pick<RMOE_FMT_Q4NX>(a, st);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace rmoe
