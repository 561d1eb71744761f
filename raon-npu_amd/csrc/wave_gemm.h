// One wave's share of y = x W^T on bf16 MFMA: MF fragments of 16 activation rows times NF
// fragments of 16 weight rows over a range of K tiles.  Weights go from global memory
// into registers; activations pass through an LDS region of the wave's own (each load
// instruction then takes whole 256-byte row pieces; an MFMA's own layout would touch 16
// rows with every 16 lanes).  There is no barrier, so waves with different K ranges or
// weight rows run at their own pace and hide each other's loads.
//
// Exactness: every product is exact and every sum is fp32, as in the GEMV kernels.
//   q4nx:  the MFMA multiplies x by 1 + n/16 (exact in bf16, built by one shift and one
//     v_and_or_b32 per pair) for one 32-column group at a time, D' = S + D/16, and the
//     group's scale enters in fp32: acc += (16 scale) D' + (min - 16 scale) S, S the group
//     sum of x.  S comes from an MFMA with ones as its first operand (every output row of
//     column l16 is S of activation row l16), of which lane (l16, lq) keeps group lq: the
//     operand layout of a bf16 MFMA over the groups.  There S is split exactly into three
//     bf16 parts and multiplied by min and by -16 scale (both exact bf16 values).
//   bfp16: m * 2^(e - 133) has 8 significant bits.  The MFMA multiplies a quarter of it,
//     exact in bf16 for every exponent byte (the largest, -128 * 2^122, would overflow
//     undivided; the smallest, 2^-128, is an exact subnormal); the caller multiplies the
//     sums by 4.
// A row's result depends on its own values and on the K range only, not on MF or NF.
#pragma once

#include "../../include/raon_moe.h"
#include "rmoe_internal.h"

namespace rmoe {

typedef __bf16 wg_bf16x8 __attribute__((ext_vector_type(8)));
typedef float wg_f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ wg_f32x4 wg_mfma(const uint4 a, const uint4 b, wg_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(wg_bf16x8, a), __builtin_bit_cast(wg_bf16x8, b),
                                                 c, 0, 0, 0);
}
// Two fp32 values -> RNE bf16 pair (a | b << 16).
__device__ __forceinline__ uint32_t wg_cvt_pair(float a, float b) {
  typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
  const bf16x2v v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, v);
}

// Codes of one dword -> four bf16 pairs 1 + n/16, as unpack_codes.  The masks come from one
// volatile statement ahead of every MFMA and the unpack itself is plain C++: the compiler
// does not add the wait states that a register just written by an MFMA needs when the next
// writer is an inline assembly statement.
struct Q4Masks {
  uint32_t mask, one;  // 0x00780078, 0x3F803F80, in vector registers
};
__device__ __forceinline__ Q4Masks q4_masks() {
  Q4Masks k;
  asm volatile("v_mov_b32 %0, 0x780078\n\tv_mov_b32 %1, 0x3f803f80" : "=&v"(k.mask), "=&v"(k.one));
  return k;
}
__device__ __forceinline__ uint4 q4_pairs(uint32_t v, const Q4Masks& k) {
  return make_uint4(((v << 3) & k.mask) | k.one, ((v >> 1) & k.mask) | k.one, ((v >> 5) & k.mask) | k.one,
                    ((v >> 9) & k.mask) | k.one);
}

// What a wave multiplies.  Lane (l16, lq) = (lane % 16, lane / 16).
// XI: how many of a fragment's four row quartets are loaded (1 when at most 4 rows live; the
// rows that are not loaded hold arbitrary values, which reach only their own results).
template <int MF, int NF, int XI>
struct WaveOperands {
  const uint8_t* w[NF];   // fragment f's first K tile, advanced to its first row (uniform)
  const uint8_t* x;       // activations (uniform)
  uint32_t xoff[MF][XI];  // byte offset of activation row 16m + 4i + lq, plus 16 l16
  uint8_t* lds;           // 4096 MF bytes of the wave's own
};

template <typename T>
__device__ __forceinline__ T wg_load(const uint8_t* base, uint32_t off) {
  return *reinterpret_cast<const T*>(base + off);
}

// 16 bytes of weights; with kOnce (no other token tile reads them) the non-temporal hint.
template <bool kOnce>
__device__ __forceinline__ uint4 wg_load_weights(const uint8_t* base, uint32_t off) {
  if constexpr (kOnce) return load_stream16(base + off);
  return wg_load<uint4>(base, off);
}

// The activation rows of one K tile: global -> registers -> LDS -> MFMA operands.  In LDS
// the 16-byte chunk c of row r sits at chunk c ^ (r % 16), so that both the writes (16
// lanes on one row) and the reads (one chunk of 16 rows) cover all banks.
template <int MF, int NF, int XI>
struct WaveRows {
  uint4 raw[MF][XI];
  uint32_t wr, rd;
  __device__ __forceinline__ WaveRows() {
    const uint32_t lane = threadIdx.x & 63u, l16 = lane & 15u, lq = lane >> 4;
    wr = 256u * lq + 16u * (l16 ^ lq);
    rd = 256u * l16 + 16u * (l16 ^ lq);
  }
  // live == false: every lane reads the same 16 bytes (the last tile's refill is not used).
  __device__ __forceinline__ void load(const WaveOperands<MF, NF, XI>& o, int kt, bool live) {
    const uint8_t* xb = o.x + (size_t)kt * 256;
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
      for (int i = 0; i < XI; ++i) raw[m][i] = wg_load<uint4>(xb, live ? o.xoff[m][i] : 0u);
  }
  __device__ __forceinline__ void store(uint8_t* lds) const {
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
      for (int i = 0; i < XI; ++i) *reinterpret_cast<uint4*>(lds + 4096 * m + 1024 * i + (wr ^ (64u * i))) = raw[m][i];
  }
  // Chunk 4g + lq of row 16m + l16.
  __device__ __forceinline__ uint4 group(const uint8_t* lds, int m, int g) const {
    return *reinterpret_cast<const uint4*>(lds + 4096 * m + (rd ^ (64u * g)));
  }
};

// The int8 mantissas of two dwords times s (a power of two) as a bf16 operand, exactly: byte
// u = m + 128 becomes the fp32 value 2^15 + u by one v_perm_b32, which minus 2^15 + 128 is
// m.  (v_cvt_f32_i32 issues at a quarter of the rate of these.)
__device__ __forceinline__ uint4 b16_operand(uint32_t v0, uint32_t v1, float s) {
  uint32_t r[4];
  const uint32_t u[2] = {v0 ^ 0x80808080u, v1 ^ 0x80808080u};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = u[i >> 1];
    // Selector bytes: 0x07 = the constant's top byte, 0x0c = 0, 0..3 = the byte of w.
    const uint32_t k = (i & 1) ? 0x0200u : 0u;
    const float lo = __uint_as_float(__builtin_amdgcn_perm(0x47000000u, w, 0x070c000cu + k));
    const float hi = __uint_as_float(__builtin_amdgcn_perm(0x47000000u, w, 0x070c010cu + k));
    r[i] = bf16_pair((lo - 32896.0f) * s, (hi - 32896.0f) * s);
  }
  return make_uint4(r[0], r[1], r[2], r[3]);
}

// acc += this wave's K tiles [kt0, kt1).  acc[m][f] in the MFMA output layout: lane (l16,
// lq) holds activation rows 16m + 4lq + i (i = 0..3) of weight row l16 of fragment f.
// The loads of tile kt + 1 are in flight under the MFMAs of tile kt (two register sets).
// bfp16 sums are a quarter of the product's.
template <int MF, int NF, int XI>
__device__ __forceinline__ void wave_gemm_b16(const WaveOperands<MF, NF, XI>& o, int kt0, int kt1,
                                              wg_f32x4 (&acc)[MF][NF]) {
  const uint32_t lane = threadIdx.x & 63u, l16 = lane & 15u, lq = lane >> 4;
  if (kt0 >= kt1) return;
  // MFMA (j, h) takes block 8j + 2lq + h (8 columns) in lane quarter lq: half h of the
  // 16-byte mantissa chunk 4j + lq, with the activations' chunk of the same number.
  struct W {
    uint4 mt[NF][2], e[NF];
  } wa, wb;
  WaveRows<MF, NF, XI> xr;
  const uint32_t rd = 256u * l16 + 16u * (l16 ^ (2u * lq));
  auto load = [&](int kt, bool live, W& w) {
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const uint8_t* p = o.w[f] + (size_t)kt * kB16TileBytes;
#pragma unroll
      for (int j = 0; j < 2; ++j) w.mt[f][j] = wg_load_weights<XI == 1>(p + 4096 * j, live ? 1024u * lq + 16u * l16 : 0u);
      w.e[f] = wg_load_weights<XI == 1>(p + kB16MantBytes, live ? 16u * l16 : 0u);
    }
    xr.load(o, kt, live);
    asm volatile("" ::: "memory");  // keeps the loads ahead of the MFMAs
  };
  auto step = [&](int kt, const W& w, W& next) {
    xr.store(o.lds);
    load(min(kt + 1, kt1 - 1), kt + 1 < kt1, next);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint4 x[MF];
#pragma unroll
        for (int m = 0; m < MF; ++m)
          x[m] = *reinterpret_cast<const uint4*>(o.lds + 4096 * m + (rd ^ (128u * j + 16u * h)));
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          // Exponent byte 8j + 2lq + h: word 2j + lq / 2, byte (2lq + h) % 4.
          const uint32_t ew = j ? ((lq & 2u) ? w.e[f].w : w.e[f].z) : ((lq & 2u) ? w.e[f].y : w.e[f].x);
          const float sc = 0.25f * exp_scale((ew >> (16u * (lq & 1u) + 8u * h)) & 0xffu);
          const uint4 v = w.mt[f][j];
          const uint4 b = h ? b16_operand(v.z, v.w, sc) : b16_operand(v.x, v.y, sc);
#pragma unroll
          for (int m = 0; m < MF; ++m) acc[m][f] = wg_mfma(x[m], b, acc[m][f]);
        }
      }
  };
  load(kt0, true, wa);
#pragma unroll 1
  for (int kt = kt0; kt < kt1; kt += 2) {
    step(kt, wa, wb);
    if (kt + 1 < kt1) step(kt + 1, wb, wa);
  }
}

// a's upper half and b's lower half trade places (32 lanes each); in the 16-lane form a's
// odd rows of 16 lanes and b's even rows.
__device__ __forceinline__ void wg_swap32(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ void wg_swap16(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

template <int MF, int NF, int XI>
__device__ __forceinline__ void wave_gemm_q4(const WaveOperands<MF, NF, XI>& o, int kt0, int kt1,
                                             wg_f32x4 (&acc)[MF][NF]) {
  const uint32_t lane = threadIdx.x & 63u, l16 = lane & 15u, lq = lane >> 4;
  const Q4Masks masks = q4_masks();
  if (kt0 >= kt1) return;
  const wg_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  const uint4 ones = make_uint4(masks.one, masks.one, masks.one, masks.one);
  struct W {
    uint4 c[NF];   // codes of row l16, group lq
    uint4 sm[NF];  // scale | min words of row l16
  } wa, wb;
  WaveRows<MF, NF, XI> xr;
  auto load = [&](int kt, bool live, W& w) {
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const uint8_t* p = o.w[f] + (size_t)kt * kTileBytes;
      w.c[f] = wg_load_weights<XI == 1>(p, live ? 1024u * lq + 16u * l16 : 0u);
      w.sm[f] = wg_load_weights<XI == 1>(p + kCodeBytes, live ? 16u * l16 : 0u);
    }
    xr.load(o, kt, live);
    asm volatile("" ::: "memory");  // keeps the loads ahead of the MFMAs
  };
  // The words of group lq and the group sums of the last four tiles (newest last): their 16
  // groups make one round of correction MFMAs.
  uint32_t sl[4][NF];
  float gs[4][MF];
  auto clear = [&]() {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int f = 0; f < NF; ++f) sl[s][f] = 0u;
#pragma unroll
      for (int m = 0; m < MF; ++m) gs[s][m] = 0.f;
    }
  };
  clear();
  auto step = [&](int kt, W& wt, W& next) {
    xr.store(o.lds);
    load(min(kt + 1, kt1 - 1), kt + 1 < kt1, next);
    // Codes: lane quarter lq holds the four dwords of group lq; a 4 x 4 transpose over the
    // quarters gives it dword lq of every group.
    uint32_t c[NF][4];
    float s16[NF][4];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      c[f][0] = wt.c[f].x;
      c[f][1] = wt.c[f].y;
      c[f][2] = wt.c[f].z;
      c[f][3] = wt.c[f].w;
      wg_swap32(c[f][0], c[f][2]);
      wg_swap32(c[f][1], c[f][3]);
      wg_swap16(c[f][0], c[f][1]);
      wg_swap16(c[f][2], c[f][3]);
      const uint32_t w[4] = {wt.sm[f].x, wt.sm[f].y, wt.sm[f].z, wt.sm[f].w};
#pragma unroll
      for (int g = 0; g < 4; ++g) s16[f][g] = 16.f * __uint_as_float(w[g] << 16);
#pragma unroll
      for (int s = 0; s < 3; ++s) sl[s][f] = sl[s + 1][f];
      const uint32_t lo = (lq & 1u) ? w[1] : w[0], hi = (lq & 1u) ? w[3] : w[2];
      sl[3][f] = (lq & 2u) ? hi : lo;
    }
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
      for (int s = 0; s < 3; ++s) gs[s][m] = gs[s + 1][m];
    // Up to four tokens: all four groups' operands are read, then all their products formed.
    // Left to itself the compiler takes one group at a time through the same few registers,
    // and the wave waits for each; with more tokens the fragments fill those waits.
    constexpr int GB = XI == 1 ? 4 : 1;
#pragma unroll
    for (int g0 = 0; g0 < 4; g0 += GB) {
      uint4 x[GB][MF];
      wg_f32x4 S[GB][MF], d[GB][NF][MF];
#pragma unroll
      for (int g = 0; g < GB; ++g)
#pragma unroll
        for (int m = 0; m < MF; ++m) {
          x[g][m] = xr.group(o.lds, m, g0 + g);
          if constexpr (GB == 1) S[g][m] = wg_mfma(ones, x[g][m], zero);
        }
      if constexpr (GB > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < GB; ++g) {
        if constexpr (GB > 1) {
#pragma unroll
          for (int m = 0; m < MF; ++m) S[g][m] = wg_mfma(ones, x[g][m], zero);
        }
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const uint4 b = q4_pairs(c[f][g0 + g], masks);
#pragma unroll
          for (int m = 0; m < MF; ++m) d[g][f][m] = wg_mfma(x[g][m], b, zero);
        }
      }
      if constexpr (GB > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int gg = 0; gg < GB; ++gg) {
        const int g = g0 + gg;
#pragma unroll
        for (int m = 0; m < MF; ++m) gs[3][m] = g == 0 ? S[gg][m][0] : (lq == (uint32_t)g ? S[gg][m][0] : gs[3][m]);
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int m = 0; m < MF; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[m][f][i] = fmaf(s16[f][g], d[gg][f][m][i], acc[m][f][i]);
      }
    }
  };
  auto correct = [&]() {
    // Correction over the 16 groups: k index 8 lq + i is (tile i % 4 of the four, group
    // lq); the two halves of an operand carry two of the six products.
    uint4 a_hm[MF], a_ll[MF];
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      uint32_t hi[2], mid[2], lo[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float v0 = gs[2 * h][m], v1 = gs[2 * h + 1][m];
        hi[h] = wg_cvt_pair(v0, v1);
        v0 -= __uint_as_float(hi[h] << 16);
        v1 -= __uint_as_float(hi[h] & 0xffff0000u);
        mid[h] = wg_cvt_pair(v0, v1);
        v0 -= __uint_as_float(mid[h] << 16);
        v1 -= __uint_as_float(mid[h] & 0xffff0000u);
        lo[h] = wg_cvt_pair(v0, v1);
      }
      a_hm[m] = make_uint4(hi[0], hi[1], mid[0], mid[1]);
      a_ll[m] = make_uint4(lo[0], lo[1], lo[0], lo[1]);
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      uint32_t mn[2], sc[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t w0 = sl[2 * h][f], w1 = sl[2 * h + 1][f];
        mn[h] = bf16_pair(__uint_as_float(w0), __uint_as_float(w1));
        sc[h] = bf16_pair(-16.f * __uint_as_float(w0 << 16), -16.f * __uint_as_float(w1 << 16));
      }
      const uint4 b_mn = make_uint4(mn[0], mn[1], mn[0], mn[1]), b_sc = make_uint4(sc[0], sc[1], sc[0], sc[1]);
      const uint4 b_ms = make_uint4(mn[0], mn[1], sc[0], sc[1]);
#pragma unroll
      for (int m = 0; m < MF; ++m) {
        acc[m][f] = wg_mfma(a_ll[m], b_ms, acc[m][f]);
        acc[m][f] = wg_mfma(a_hm[m], b_mn, acc[m][f]);
        acc[m][f] = wg_mfma(a_hm[m], b_sc, acc[m][f]);
      }
    }
    clear();
  };
  load(kt0, true, wa);
  // The pairs of up to four tokens run without a branch around the second step: at the branch's
  // join the compiler copies the weights just requested, which waits for them.  With the groups'
  // order above, one token of [768, 2560] 4.3 -> 3.7 us, of [2176, 2560] 4.9 -> 4.3 us (the GEMV
  // kernel that had served it: 3.8 and 4.4); tiles requested two ahead instead 4.0 and 4.4 us.
  if constexpr (XI == 1) {
    int kt = kt0;
#pragma unroll 1
    for (; kt + 1 < kt1; kt += 2) {
      step(kt, wa, wb);
      step(kt + 1, wb, wa);
      if (((kt - kt0) & 2) || kt + 2 >= kt1) correct();
    }
    if (kt < kt1) {
      step(kt, wa, wb);
      correct();
    }
    return;
  }
#pragma unroll 1
  for (int kt = kt0; kt < kt1; kt += 2) {
    step(kt, wa, wb);
    if (kt + 1 < kt1) step(kt + 1, wb, wa);
    if (((kt - kt0) & 2) || kt + 2 >= kt1) correct();
  }
}

template <int kFmt, int MF, int NF, int XI>
__device__ __forceinline__ void wave_gemm(const WaveOperands<MF, NF, XI>& o, int kt0, int kt1, wg_f32x4 (&acc)[MF][NF]) {
  if constexpr (kFmt == RMOE_FMT_BFP16)
    wave_gemm_b16<MF, NF, XI>(o, kt0, kt1, acc);
  else
    wave_gemm_q4<MF, NF, XI>(o, kt0, kt1, acc);
}

}  // namespace rmoe
