// The grouped GEMM for groups of few rows (included by moe_prefill.hip, which defines the
// operand forms).  Same products in the same order as gemm_tile / gemm_tile_b16, so a row's
// result is the same bytes whichever of the two kernels takes it.
//
// What bounds it: the expert weights, read once per 48 rows, are the traffic; a tile has too
// little MFMA work to hide a load round under.  So instead of one 160 KB workgroup per CU
// with weights and rows in a shared ring, a workgroup here has four waves, each of which
// streams the weights of its own 64 weight rows into registers (one 16-byte load per lane
// and fragment of 16 rows).  Only the tile's activation rows go through LDS, two K tiles of
// them, with a barrier per K step that does not wait for weights.  Two workgroups are
// resident per CU, each hiding the other's prologue and load rounds.
// Of a weight tile's 5 KB, 1 KB are scales and mins, which the correction needs before the K
// loop: their scales stay in LDS from there on (2 KB per K tile, 32 to 40 KB per workgroup;
// reading them again beside the codes cost 3 to 7 % of gate/up) as long as two workgroups fit
// a CU, and the first block of them is requested with the first codes, before the row indices
// are known.
// Kernel times against grouped_gemm_kernel, gate/up and down: H=2048, I=768, 445 tokens 95 ->
// 76 and 57 -> 46 us, which is 3.4 and 2.8 TB/s of expert weights; H=2560, I=1088, 32 tokens
// 108 -> 79 and 61 -> 51 us, 256 tokens 142 -> 105 and (bfp16) 139 -> 99 us, 4.2 and 4.8 TB/s.
// The rest is the workgroups' last round: 828 of them in 512 places at 445 tokens.  Tiles of 32
// rows instead of 48 cost 3 to 8 % at 445 tokens, three workgroups per CU (168 registers,
// spills) 10 to 30 %, the first weight tiles requested after the correction instead of first
// 5 to 45 %, weights three K steps ahead instead of two in the 16-row tiles 2 %.
#pragma once

// A barrier that waits for the wave's LDS accesses only.
__device__ __forceinline__ void few_rows_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

constexpr int kFewStageBytes = 2 * kBMFew * 256;                  // two K tiles of activation rows
constexpr int kFewGateUpOut = 3 * kBMFew * kOutStride * 2;         // gate, up and h of SiTU
constexpr int kFewDownOut = kBMFew * 264 * 2;

// One tile of 16 MF rows by 256 weight rows.  Gate/up: units 128 nt + 32 w .. +31 in wave w
// (fragments 0, 1 gate, 2, 3 up); down: output columns 256 nt + 64 w .. +63.
// kWide: the scales of a K tile come with its codes instead of from LDS (few_rows_wide).
template <int MF, bool kDown, bool kB16, bool kWide>
__device__ __forceinline__ void few_rows_tile(const GemmArgs& a, uint32_t te, int nt, uint8_t* lds, int* rowidx,
                                              int8_t* row_e, int* differ) {
  constexpr int NF = 4;
  constexpr int kTB = kB16 ? kB16TileBytes : kTileBytes;
  const int e = (int)(te & 511u), nrows = (int)((te >> 9) & 63u) + 1, row0 = (int)(te >> 15);
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int l16 = lane & 15, lq = lane >> 4;
  // K tiles that hold live columns (a down input has I of them; the rest are padding).
  const int nkt = kDown ? (a.inter + kTileCols - 1) / kTileCols : a.K / kTileCols;
  const int wkt = a.K / kTileCols;
  const uint8_t* W = a.wbase + (size_t)e * a.wstride;
  const int eso = exp_stride(a.K);

  // First weight row of the wave's fragments.  A wave past I (last gate/up tile when I % 128
  // != 0) has none: all its lanes read the same 16 bytes and nothing of it is stored.
  const bool dead = !kDown && 128 * nt + 32 * wave >= a.inter;
  const uint8_t* wf[NF];
  int wrow[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    wrow[f] = kDown ? 256 * nt + 64 * wave + 16 * f : (f >> 1) * a.inter + 128 * nt + 32 * wave + 16 * (f & 1);
    if (dead) wrow[f] = 0;
    wf[f] = W + (size_t)(wrow[f] / kTileRows) * wkt * kTB + (wrow[f] % kTileRows) * 16;
  }
  // Weights of one K tile.  q4nx: codes of (row l16, group lq), the scales come from LDS or,
  // kWide, the group's scale | min word;
  // bfp16: mantissas of columns 32 lq .. +31 and their four exponents.  The first two tiles
  // depend on the tile entry only: requested before anything else.
  struct WTile {
    uint4 c[NF][kB16 ? 2 : 1];
    uint32_t s[kB16 || kWide ? NF : 1];
  };
  auto load_w = [&](int kt, WTile& w) {
    const bool live = kt < nkt && !dead;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const uint8_t* p = wf[f] + (size_t)min(kt, nkt - 1) * kTB;
      if constexpr (kB16) {
#pragma unroll
        for (int h = 0; h < 2; ++h) w.c[f][h] = wg_load_weights<true>(p, live ? 1024u * (2 * lq + h) + 16u * l16 : 0u);
        w.s[f] = wg_load<uint32_t>(p + kB16MantBytes, live ? 16u * l16 + 4u * lq : 0u);
      } else {
        w.c[f][0] = wg_load_weights<true>(p, live ? 1024u * lq + 16u * l16 : 0u);
        if constexpr (kWide) w.s[f] = wg_load<uint32_t>(p + kCodeBytes, live ? 16u * l16 + 4u * lq : 0u);
      }
    }
    asm volatile("" ::: "memory");  // keeps the loads where they are
  };
  WTile wa, wb, wc;
  // Correction operands of a block of 32 groups: the scale | min words of groups 32 blk +
  // 8 lq .. +7 of weight row l16, and the group sums of activation row l16 for them.
  const int G = a.K / 32, Gp = sum_planes_gp(G), nblk = kB16 ? 0 : (G + 31) / 32;
  struct Coef {
    uint4 c[NF][2];
  };
  struct Sums {
    uint4 s[MF][3];
  };
  auto load_c = [&](int blk, Coef& b) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int kt = 8 * blk + 2 * lq + h;
        b.c[f][h] = wg_load<uint4>(wf[f] + kCodeBytes, (uint32_t)((4 * kt < G ? kt : 0) * kTB + 16 * l16));
      }
    asm volatile("" ::: "memory");
  };
  [[maybe_unused]] Coef ca, cb;

  // Source row of each tile row (rows past the tile repeat its first row and are not
  // stored).  A down tile's rows lie one after another; a gate/up tile's token rows are
  // loaded, with the first weights in flight behind them.  (The barriers here wait for LDS
  // only: __syncthreads() would also wait for the weights.)
  const int my_row = row0 + (tid < nrows ? tid : 0);
  int my_src = my_row;
  if constexpr (!kDown) {
    if (tid < 16 * MF) my_src = e < a.n_routed ? a.order[my_row] : my_row - a.shared_base;
  }
  if constexpr (!kB16) load_c(0, ca);
  load_w(0, wa);
  load_w(1, wb);
  if constexpr (!kDown) {
    if (tid < 16 * MF) rowidx[tid] = my_src = e < a.n_routed ? my_src / a.k_routes : my_src;
    few_rows_barrier();
  }
  auto src_row = [&](int r) { return kDown ? row0 + (r < nrows ? r : 0) : rowidx[r]; };

  // Activation rows: thread t brings 16-byte chunk t % 16 of rows t / 16 + 16 i of a K tile,
  // through registers into LDS chunk (t % 16) ^ (row % 16) of the row (as WaveRows).
  const int xrow = tid >> 4;
  uint32_t xoff[MF];
#pragma unroll
  for (int i = 0; i < MF; ++i)
    xoff[i] = (uint32_t)src_row(xrow + 16 * i) * (uint32_t)(2 * a.K) + 16u * (uint32_t)(tid & 15);
  const uint32_t xwr = 256u * xrow + 16u * (uint32_t)((tid & 15) ^ xrow);
  uint4 xr[MF];
  auto load_x = [&](int kt) {
    const uint8_t* xb = reinterpret_cast<const uint8_t*>(a.src) + (size_t)min(kt, nkt - 1) * 256;
#pragma unroll
    for (int i = 0; i < MF; ++i) xr[i] = wg_load<uint4>(xb, kt < nkt ? xoff[i] : 0u);
  };
  Sums sa;
  [[maybe_unused]] Sums sb;
  uint32_t srow[MF];
#pragma unroll
  for (int m = 0; m < MF; ++m) srow[m] = kB16 ? 0u : (uint32_t)src_row(16 * m + l16) * (uint32_t)(6 * Gp);
  auto load_s = [&](int blk, Sums& b) {
    const int gl = 32 * blk + 8 * lq;
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        b.s[m][p] = wg_load<uint4>(reinterpret_cast<const uint8_t*>(a.ssum + p * Gp),
                                   srow[m] + 2u * (uint32_t)(gl < Gp ? gl : 0));
    asm volatile("" ::: "memory");
  };
  if constexpr (!kB16) load_s(0, sa);
  // What is in flight during the correction, as far as registers go (a spill is never worth
  // it here: the compiler has placed one so that it corrupted row addresses).  236 to 243 of
  // 256 registers with these.
  constexpr bool kCoefAhead = MF <= (kWide ? 1 : 2), kSumsAhead = MF <= 1, kRowsAhead = MF <= 1;
  if constexpr (kRowsAhead) {
    load_x(0);
    asm volatile("" ::: "memory");
  }
  if constexpr (!kB16 && kCoefAhead) {
    if (nblk > 1) load_c(1, cb);
  }
  // Power-of-two exponent of each row; a down row's is the largest of its chunks'.
  int my_e = 0, my_d = 0;
  if (tid < 16 * MF) {
    if constexpr (kDown) {
      int emax = -128, emin = 127;
      for (int c0 = 0; c0 < a.K / 128; c0 += 16) {
        const uint4 v = *reinterpret_cast<const uint4*>(a.hexp + (size_t)my_row * eso + c0);
        const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int c = 0; c < 16; ++c)
          if (c0 + c < a.K / 128) {
            const int ec = (int)(int8_t)(w4[c >> 2] >> (8 * (c & 3)));
            emax = max(emax, ec);
            emin = min(emin, ec);
          }
      }
      my_e = emax;
      my_d = emin != emax ? 1 : 0;
    } else {
      my_e = a.aexp[my_src];
    }
    row_e[tid] = (int8_t)my_e;
  }
  const unsigned long long vote = __ballot(my_d != 0);  // rows are wave 0's: its vote is the tile's
  if (tid == 0) *differ = vote ? 1 : 0;
  few_rows_barrier();
  const bool rescale = kDown && *differ != 0;

  auto h2 = [](uint32_t v) { return __builtin_bit_cast(f16x2_t, v); };
  auto u2 = [](f16x2_t v) { return __builtin_bit_cast(uint32_t, v); };
  auto store_x = [&](int kt) {
    if (rescale && kt < nkt) {  // a chunk below its row's exponent (rare), as h_unify_kernel
#pragma unroll
      for (int i = 0; i < MF; ++i) {
        const int r = xrow + 16 * i, d = (int)a.hexp[(size_t)src_row(r) * eso + kt] - (int)row_e[r];
        if (d == 0) continue;
        uint32_t v[4] = {xr[i].x, xr[i].y, xr[i].z, xr[i].w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f16x2_t x = h2(v[q]);
          v[q] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(__builtin_amdgcn_ldexpf((float)x[0], d),
                                                                         __builtin_amdgcn_ldexpf((float)x[1], d)));
        }
        xr[i] = make_uint4(v[0], v[1], v[2], v[3]);
      }
    }
    uint8_t* st = lds + (kt & 1) * (4096 * MF);
#pragma unroll
    for (int i = 0; i < MF; ++i) *reinterpret_cast<uint4*>(st + 4096 * i + xwr) = xr[i];
  };

  f32x4_t acc[MF][NF];
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[m][f] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // The wave's scales, for the K loop: [K tile][fragment][row][group] bf16 in LDS.
  [[maybe_unused]] uint8_t* wsc = lds + kFewStageBytes + (size_t)wave * wkt * (NF * 128) + 8 * l16;
  int fx[NF];
  [[maybe_unused]] int emax_w[NF];
  {
    if constexpr (kB16) {
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        emax_w[f] = a.rowexp[(size_t)e * a.N_total + wrow[f] + l16];
        fx[f] = emax_w[f] - 141;
      }
    } else {
      // Correction: acc += sum_g (min + 8 scale)[r, g] S[m, g], six products per block of 32
      // groups on bf16 MFMA in gemm_tile's order.
      uint32_t smax[NF] = {0u, 0u, 0u, 0u};
      auto corr_blk = [&](int blk, const Coef& b, const Sums& s) {
        const int gl = 32 * blk + 8 * lq;
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const uint32_t sv[8] = {b.c[f][0].x, b.c[f][0].y, b.c[f][0].z, b.c[f][0].w,
                                  b.c[f][1].x, b.c[f][1].y, b.c[f][1].z, b.c[f][1].w};
#pragma unroll
          for (int h = 0; h < 2; ++h)
            if (!kWide && gl + 4 * h < G)
              *reinterpret_cast<uint2*>(wsc + ((8 * blk + 2 * lq + h) * NF + f) * 128) =
                  make_uint2(__builtin_amdgcn_perm(sv[4 * h + 1], sv[4 * h], 0x05040100u),
                             __builtin_amdgcn_perm(sv[4 * h + 3], sv[4 * h + 2], 0x05040100u));
          uint32_t w[8];
          float s8[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            w[i] = gl + i < G ? sv[i] : 0u;
            smax[f] = max(smax[f], w[i] & 0x7fffu);
            s8[i] = 8.f * bf16_to_f32(w[i] & 0xffffu);
          }
          const uint4 bmin = make_uint4(pack_bf16_top(__uint_as_float(w[0]), __uint_as_float(w[1])),
                                        pack_bf16_top(__uint_as_float(w[2]), __uint_as_float(w[3])),
                                        pack_bf16_top(__uint_as_float(w[4]), __uint_as_float(w[5])),
                                        pack_bf16_top(__uint_as_float(w[6]), __uint_as_float(w[7])));
          const uint4 bsc8 = make_uint4(pack_bf16_top(s8[0], s8[1]), pack_bf16_top(s8[2], s8[3]),
                                        pack_bf16_top(s8[4], s8[5]), pack_bf16_top(s8[6], s8[7]));
#pragma unroll
          for (int p = 0; p < 6; ++p)
#pragma unroll
            for (int m = 0; m < MF; ++m)
              acc[m][f] = mfma16(s.s[m][2 - p / 2], (p & 1) ? bsc8 : bmin, acc[m][f]);
        }
      };
      if constexpr (kCoefAhead) {
#pragma unroll 1
        for (int blk = 0; blk < nblk; blk += 2) {
          if (kSumsAhead && blk + 1 < nblk) load_s(blk + 1, sb);
          corr_blk(blk, ca, sa);
          if (blk + 1 < nblk) {
            if (!kSumsAhead) load_s(blk + 1, sa);
            if (blk + 2 < nblk) load_c(blk + 2, ca);
            if (kSumsAhead && blk + 2 < nblk) load_s(blk + 2, sa);
            corr_blk(blk + 1, cb, kSumsAhead ? sb : sa);
            if (!kSumsAhead && blk + 2 < nblk) load_s(blk + 2, sa);
            if (blk + 3 < nblk) load_c(blk + 3, cb);
          }
        }
      } else {
#pragma unroll 1
        for (int blk = 0; blk < nblk; ++blk) {
          corr_blk(blk, ca, sa);
          if (blk + 1 < nblk) {
            load_c(blk + 1, ca);
            load_s(blk + 1, sa);
          }
        }
      }
      // Weight-row exponents, as in gemm_tile: the largest scale lands in [2^11, 2^12).
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        uint32_t m = smax[f];
        m = max(m, (uint32_t)__shfl_xor((int)m, 16, 64));
        m = max(m, (uint32_t)__shfl_xor((int)m, 32, 64));
        const int be = (int)(m >> 7) & 0xff;
        fx[f] = (m == 0u || be == 0xff) ? 0 : (be == 0 ? -138 : be - 127 - 11);
      }
    }
    auto scale_rows = [&](int sign) {
#pragma unroll
      for (int m = 0; m < MF; ++m) {
        const uint32_t e4 = *reinterpret_cast<const uint32_t*>(row_e + 16 * m + 4 * lq);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int er = (int)(int8_t)(e4 >> (8 * i));
#pragma unroll
          for (int f = 0; f < NF; ++f) acc[m][f][i] = __builtin_amdgcn_ldexpf(acc[m][f][i], sign * (er + fx[f]));
        }
      }
    };
    if constexpr (!kRowsAhead) load_x(0);
    if constexpr (!kB16) scale_rows(-1);

    // K loop: MFMA j takes columns 32 lq + 8j .. +7 from lane quarter lq, the activations'
    // chunk 4 lq + j.  Step kt writes the rows of tile kt + 1, loads those of kt + 2 and the
    // weights of kt + 2, and multiplies tile kt; the barrier waits for LDS only.
    const uint32_t rd = 256u * l16 + 16u * (l16 ^ (4u * lq));
    uint32_t kmask, kmask_hi, kmagic;
    asm volatile("v_mov_b32 %0, 0xf000f\n\tv_mov_b32 %1, 0xf000f0\n\tv_mov_b32 %2, 0x64006400"
                 : "=&v"(kmask), "=&v"(kmask_hi), "=&v"(kmagic));
    const f16x2_t k1032 = {(_Float16)1032.0f, (_Float16)1032.0f}, k1152 = {(_Float16)1152.0f, (_Float16)1152.0f};
    store_x(0);
    load_x(1);
    few_rows_barrier();
    auto step = [&](int kt, const WTile& w, WTile& next) {
      store_x(kt + 1);
      load_x(kt + 2);
      load_w(kt + 2, next);
      const uint8_t* xs = lds + (kt & 1) * (4096 * MF);
      f16x2_t s1[NF], s16[NF];
      if constexpr (!kB16) {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          float sc;
          if constexpr (kWide) sc = bf16_to_f32(w.s[f] & 0xffffu);
          else sc = bf16_to_f32(*reinterpret_cast<const uint16_t*>(wsc + (kt * NF + f) * 128 + 2 * lq));
          const float v1 = __builtin_amdgcn_ldexpf(sc, -fx[f]), v16 = __builtin_amdgcn_ldexpf(sc, -fx[f] - 4);
          s1[f] = __builtin_bit_cast(f16x2_t, __builtin_amdgcn_cvt_pkrtz(v1, v1));
          s16[f] = __builtin_bit_cast(f16x2_t, __builtin_amdgcn_cvt_pkrtz(v16, v16));
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint4 av[MF];
#pragma unroll
        for (int m = 0; m < MF; ++m) av[m] = *reinterpret_cast<const uint4*>(xs + 4096 * m + (rd ^ (16u * j)));
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          uint4 b;
          if constexpr (kB16) {
            const uint4 mq = w.c[f][j >> 1];
            const int ex = (int)((w.s[f] >> (8 * j)) & 0xffu);
            const int pw = min(max(ex, 7) - emax_w[f] + 8, 8);
            const uint32_t hb = pw >= -14 ? (uint32_t)(pw + 15) << 10 : (pw >= -24 ? 1u << (pw + 24) : 0u);
            const f16x2_t sc = h2(hb | (hb << 16));
            const uint32_t u0 = ((j & 1) ? mq.z : mq.x) ^ 0x80808080u, u1 = ((j & 1) ? mq.w : mq.y) ^ 0x80808080u;
            b = make_uint4(u2((h2(__builtin_amdgcn_perm(0x64646464u, u0, 0x04010400u)) - k1152) * sc),
                           u2((h2(__builtin_amdgcn_perm(0x64646464u, u0, 0x04030402u)) - k1152) * sc),
                           u2((h2(__builtin_amdgcn_perm(0x64646464u, u1, 0x04010400u)) - k1152) * sc),
                           u2((h2(__builtin_amdgcn_perm(0x64646464u, u1, 0x04030402u)) - k1152) * sc));
          } else {
            const uint4 cq = w.c[f][0];
            const uint32_t cv = j == 0 ? cq.x : j == 1 ? cq.y : j == 2 ? cq.z : cq.w, cu = cv >> 8;
            b = make_uint4(u2((h2((cv & kmask) | kmagic) - k1032) * s1[f]),
                           u2((h2((cv & kmask_hi) | kmagic) - k1152) * s16[f]),
                           u2((h2((cu & kmask) | kmagic) - k1032) * s1[f]),
                           u2((h2((cu & kmask_hi) | kmagic) - k1152) * s16[f]));
          }
#pragma unroll
          for (int m = 0; m < MF; ++m) acc[m][f] = mfma16h(av[m], b, acc[m][f]);
        }
      }
      few_rows_barrier();
    };
#pragma unroll 1
    for (int kt = 0; kt < nkt; kt += 3) {
      step(kt, wa, wc);
      if (kt + 1 < nkt) step(kt + 1, wb, wa);
      if (kt + 2 < nkt) step(kt + 2, wc, wb);
    }
    scale_rows(1);
  }
  __syncthreads();  // every wave is past its activation region: LDS becomes the output staging

  // The thread's place as a value of its own from here on: derived from tid, the epilogue's
  // indices are the same in the three tile sizes, and the compiler computes them once at the
  // kernel's start and holds them in some ten registers through the K loop.
  int et = tid;
  asm volatile("" : "+v"(et));
  const int el16 = et & 15, elq = (et >> 4) & 3;
  uint16_t* stage = reinterpret_cast<uint16_t*>(lds);
  if constexpr (kDown) {
    // [16 MF rows][256 columns + 8]
    constexpr int kStride = 264;
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
          const uint32_t p2 = cvt_bf16x2(acc[m][f][i], acc[m][f][i + 1]);
          uint16_t* st = stage + (16 * m + 4 * elq + i) * kStride + 64 * wave + 16 * f + el16;
          st[0] = (uint16_t)(p2 & 0xffffu);
          st[kStride] = (uint16_t)(p2 >> 16);
        }
    __syncthreads();
    for (int cid = et; cid < nrows * 32; cid += 256) {
      const int r = cid >> 5, c = cid & 31;
      *reinterpret_cast<uint4*>(a.out + (size_t)(row0 + r) * a.out_ld + 256 * nt + 8 * c) =
          *reinterpret_cast<const uint4*>(stage + r * kStride + 8 * c);
    }
    return;
  }
  // Gate/up: h tile [16 MF][128 units] as in gemm_tile's epilogue.
  const int rows_b = 16 * MF * kOutStride;
  if (!dead) {
    if (a.act == 1) {
#pragma unroll
      for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int i = 0; i < 4; i += 2) {
            const uint32_t gu0 = cvt_bf16x2(acc[m][q][i], acc[m][q + 2][i]);
            const uint32_t gu1 = cvt_bf16x2(acc[m][q][i + 1], acc[m][q + 2][i + 1]);
            const float h0 = swiglu_fast(bf16_to_f32(gu0 & 0xffffu), __uint_as_float(gu0 & 0xffff0000u));
            const float h1 = swiglu_fast(bf16_to_f32(gu1 & 0xffffu), __uint_as_float(gu1 & 0xffff0000u));
            const uint32_t hp = cvt_bf16x2(h0, h1);
            uint16_t* st = stage + (16 * m + 4 * elq + i) * kOutStride + 32 * wave + 16 * q + el16;
            st[0] = (uint16_t)(hp & 0xffffu);
            st[kOutStride] = (uint16_t)(hp >> 16);
          }
    } else {
#pragma unroll
      for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t gu = cvt_bf16x2(acc[m][q][i], acc[m][q + 2][i]);
            const int at = (16 * m + 4 * elq + i) * kOutStride + 32 * wave + 16 * q + el16;
            stage[rows_b + at] = (uint16_t)(gu & 0xffffu);
            stage[2 * rows_b + at] = (uint16_t)(gu >> 16);
          }
    }
  }
  __syncthreads();
  const int units = min(128, a.inter - 128 * nt);  // live units of the tile (a multiple of 64)
  if (a.act != 1) {
    for (int idx = et; idx < nrows * 128; idx += 256) {
      if ((idx & 127) >= units) continue;
      const int at = (idx >> 7) * kOutStride + (idx & 127);
      stage[at] = (uint16_t)cvt_bf16x2(
          act_situ(bf16_to_f32(stage[rows_b + at]), bf16_to_f32(stage[2 * rows_b + at]), a.gb, a.vb), 0.f);
    }
    __syncthreads();
  }
  const int Gpo = sum_planes_gp(a.out_ld / 32), eho = exp_stride(a.out_ld);
  if (et < 64 * MF) {
    const int r = et >> 2, q = et & 3;
    if (r < nrows && 32 * q < units) {
      float hs = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint4 v = *reinterpret_cast<const uint4*>(stage + r * kOutStride + 32 * q + 8 * c);
        const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int d = 0; d < 4; ++d) hs += bf16_to_f32(w4[d] & 0xffffu) + bf16_to_f32(w4[d] >> 16);
      }
      store_split3_planar(a.out_ssum + (size_t)(row0 + r) * 3 * Gpo + 4 * nt + q, Gpo, hs);
    }
  }
#pragma unroll
  for (int q = 0; q < MF; ++q) {
    const int cid = et + 256 * q, r = cid >> 4, c = cid & 15;
    const bool live = 8 * c < units;
    const uint4 v = *reinterpret_cast<const uint4*>(stage + r * kOutStride + 8 * c);
    const float mx = row16_max(live ? max_abs_bf16x8(v) : 0.f);
    const int ex = f16_exp_chunk(mx);
    if (r < nrows && live)
      *reinterpret_cast<uint4*>(a.out + (size_t)(row0 + r) * a.out_ld + 128 * nt + 8 * c) =
          make_uint4(bf16x2_to_f16x2(v.x, ex), bf16x2_to_f16x2(v.y, ex), bf16x2_to_f16x2(v.z, ex),
                     bf16x2_to_f16x2(v.w, ex));
    if (r < nrows && c == 0) a.out_exp[(size_t)(row0 + r) * eho + nt] = (int8_t)ex;
  }
  if (nt == a.n_tiles - 1 && a.inter < a.out_ld)
    for (int r = et >> 4; r < nrows; r += 16) zero_row_padding(a, row0 + r, et & 15, 16);
}

// Dynamic LDS: the stages and, with q4nx weights, the four waves' scales (2 KB per K tile);
// then, in the same place, the epilogue staging.  Two workgroups of it share a CU's 160 KB
// (with 1 KB for what the kernel declares itself): a layer whose scales take more than that
// (K over 3,328) reads them beside the codes instead, at any width.  With one workgroup per CU
// whole layers of 32 experts took, against this form: H = 4096, I = 768, 368 tokens 138.5 /
// 116.6 us, H = I = 4096, 256 tokens 374 / 307 us; batches that fill less than one workgroup per
// CU lose 2 to 6 % by it (H = 3584, I = 768, 32 tokens 65.9 / 70.0 us).
constexpr size_t kFewMaxLds = (size_t)79 << 10;
constexpr size_t few_rows_scales(int K) { return (size_t)4 * (K / kTileCols) * 512; }
constexpr bool few_rows_wide(int K, bool b16) { return !b16 && kFewStageBytes + few_rows_scales(K) > kFewMaxLds; }
static size_t few_rows_lds(const GemmArgs& a, bool b16) {
  const size_t loop = kFewStageBytes + (b16 || few_rows_wide(a.K, b16) ? 0 : few_rows_scales(a.K));
  return std::max(loop, (size_t)(a.mode == 0 ? kFewGateUpOut : kFewDownOut));
}

// Grid: as grouped_gemm_kernel's, 256 threads.  XCD x takes a contiguous eighth of each
// class's tiles, the largest first.
template <bool kDown, bool kB16, bool kWide>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void few_rows_gemm_kernel(GemmArgs a, int cap) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // few_rows_lds() bytes
  __shared__ int rowidx[kBMFew];
  __shared__ __attribute__((aligned(16))) int8_t row_e[kBMFew];
  __shared__ int differ;
  const int xcd = blockIdx.x % 8;
  int j = blockIdx.x / 8;
#pragma unroll
  for (int c = kTileClasses - 1; c >= 0; --c) {
    const int n = a.n_tiles * a.ntiles[c], per = (n + 7) / 8;
    if (j >= per) {
      j -= per;
      continue;
    }
    const int lid = xcd * per + j;
    if (lid >= n) return;
    const uint32_t te = a.tiles[(size_t)c * cap + lid / a.n_tiles];
    const int nt = lid % a.n_tiles;
    if (c == 2) few_rows_tile<3, kDown, kB16, kWide>(a, te, nt, lds, rowidx, row_e, &differ);
    else if (c == 1) few_rows_tile<2, kDown, kB16, kWide>(a, te, nt, lds, rowidx, row_e, &differ);
    else few_rows_tile<1, kDown, kB16, kWide>(a, te, nt, lds, rowidx, row_e, &differ);
    return;
  }
}
