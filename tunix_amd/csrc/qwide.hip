// int4 projections of more than 128 rows: cache fill over prompts, scoring passes, decode steps of many sequences.
// Same weights, rounding and LoRA arithmetic as qlinear.hip (tunix/models/llama3/model.py:216-218, :489-496 with the
// qwix-wrapped projections); reads for the reference's prefill (tunix/generate/sampler.py:601-730).
#include "tmx_kernels.h"

namespace tmx {

// A workgroup is 8 waves = CT column tiles x KW = 8 / CT k-parts over MT row tiles of 32.  A wave multiplies its column
// tile against all MT row tiles (16 MT accumulator registers), so a dequantised weight fragment feeds MT MFMAs.
// Weights come by buffer loads one step ahead, the activation slab of a step (2 k-tiles) by direct-to-LDS loads into
// two buffers: slab rows are 256 bytes (four per 1 KiB transfer), their 16-byte chunks XOR-swizzled by row % 16.  With
// KW = 2 a wave takes one k-tile of every step, and the two halves of a column tile meet through LDS at the end.
constexpr int kWideTS = 2, kWideXS = 128;
// the MFMA of a group behind which part p (1..4) of the next fragment's dequantisation goes
constexpr int wide_slot(int MT, int p) { return p < MT ? p : MT - 1; }
constexpr size_t wide_lds(int MT) { return (size_t)2 * MT * 32 * kWideXS * 2; }

template <int MT, int CT, bool LORA>
__device__ __forceinline__ void gemm_block_wide(const QLinearArgs& a, uint16_t* smem, int bx, int by, int bz) {
  constexpr int TS = kWideTS, XS = kWideXS, ROWS = MT * 32, KW = 8 / CT, TPW = TS / KW;
  static_assert(KW * CT == 8 && TPW >= 1, "8 waves, at least one k-tile of a step each");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ct = wave % CT, kw = wave / CT;
  const int h = lane >> 5, nl = lane & 31;
  const int KT = a.K >> 6;
  const int slice = LORA ? (bx - a.n_main_blocks) + a.lora_blocks_per_split * by : by;
  const int per = LORA ? a.kt_per_lora_split : a.kt_per_split;
  const int kb0 = slice * per;
  const int kb1 = (kb0 + per < KT) ? kb0 + per : KT;
  const int nsteps = (kb1 - kb0) / TS, last_step = nsteps - 1;  // host: whole steps
  if (nsteps <= 0) return;
  const int row0 = bz * ROWS;
  const int rows = a.M - row0 < ROWS ? a.M - row0 : ROWS;  // host: >= 1
  const int gs = __builtin_ctz(a.G >> 6), KG = a.K / a.G;
  const int NT = LORA ? (a.Rpad >> 5) : (a.N >> 5);
  const int nb = LORA ? ct : bx * CT + ct;
  const bool tile_ok = nb < NT;  // waves past the last tile only help with the slab

  const __amdgpu_buffer_rsrc_t rw =
      LORA ? make_rsrc(a.a_t, (uint32_t)KT * NT * 4096u) : make_rsrc(a.qw, (uint32_t)NT * KT * 1024u);
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.scales, LORA ? 0u : (uint32_t)NT * KG * 64u);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x + (size_t)row0 * a.ldx, (uint32_t)rows * a.ldx * 2u);
  const int wv = LORA ? nb * 4096 + lane * 16 : (nb * KT * 64 + lane) * 16;
  const int wstep = LORA ? NT * 4096 : 1024;  // bytes between consecutive k-tiles
  const int sv = (nb * KG * 32 + nl) * 2;
  // slab transfer: MT loads per wave and step; load i moves rows 4 wave + 32 i .. + 3 (16 lanes
  // each), lane l delivering chunk (l % 16) ^ (row % 16) of the step to slot l % 16
  int xoff[MT];  // per-lane byte offset in the row block (rows past the end repeat the last)
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int row_l = 4 * wave + 32 * i + (lane >> 4);
    xoff[i] = (row_l < rows ? row_l : rows - 1) * a.ldx * 2 + (((lane & 15) ^ (row_l & 15)) * 16) + kb0 * 128;
  }

  f32x16_t acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[m][r] = 0.f;
  constexpr int WPT = LORA ? 4 : 1;  // 16-byte words per lane and tile
  u32x4_t wring[TPW][WPT];
  uint16_t sring[TPW];

  auto load_w_tile = [&](int step, auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    step = step < last_step ? step : last_step;
    const int kt = kb0 + step * TS + kw * TPW + j;
#pragma unroll
    for (int t = 0; t < WPT; ++t) wring[j][t] = __builtin_amdgcn_raw_buffer_load_b128(rw, wv + t * 1024, kt * wstep, 0);
    if (!LORA) sring[j] = __builtin_amdgcn_raw_buffer_load_b16(rs, sv, (kt >> gs) * 64, 0);
  };
  auto dma_x = [&](int step, int buf) __attribute__((always_inline)) {
    step = step < last_step ? step : last_step;
    uint16_t* base = smem + (size_t)buf * ROWS * XS + wave * 4 * XS;
#pragma unroll
    for (int i = 0; i < MT; ++i) load_row_to_lds(rx, base + i * 32 * XS, xoff[i], step * (TS * 128));
  };
  // One step: 4 TPW fragment groups g = 4 j + t (k-tile j, 16-wide k-block t) of MT MFMAs, one per row
  // tile.  Between the MFMAs of group g the wave reads the x fragments of group g + 1 (one LDS
  // read per MFMA; chunk 2 g + h of its part of a row sits at that slot ^ (row % 16)) and dequantises its
  // weight fragment a quarter at a time, so the matrix pipe waits neither for LDS nor for the
  // VALU, also when both waves of a SIMD run in phase after a barrier.  The order is pinned.
  auto step_math = [&](int step, int buf) __attribute__((always_inline)) {
    u32x4_t wc[TPW][WPT];
    float s_c[TPW], m8s[TPW];
    static_for<TPW>([&](auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
#pragma unroll
      for (int t = 0; t < WPT; ++t) wc[j][t] = wring[j][t];
      s_c[j] = LORA ? 0.f : bf2f(sring[j]);
      m8s[j] = -8.f * s_c[j];
      load_w_tile(step + 1, jc);  // registers consumed: refill them one step ahead
    });
    const uint16_t* xb = smem + (size_t)buf * ROWS * XS + nl * XS;
    const int c0 = 8 * TPW * kw + h;  // this wave's first chunk of a slab row
    auto word_of = [&](auto gc) __attribute__((always_inline)) {
      constexpr int g = decltype(gc)::value, j = g / 4, t = g % 4;
      return t == 0 ? wc[j][0].x : (t == 1 ? wc[j][0].y : (t == 2 ? wc[j][0].z : wc[j][0].w));
    };
    bf16x8_t xq[2][MT];
    u32x4_t bq[2];
    {
      const int slot = (c0 ^ (nl & 15)) * 8;
#pragma unroll
      for (int m = 0; m < MT; ++m) xq[0][m] = *reinterpret_cast<const bf16x8_t*>(xb + m * 32 * XS + slot);
      if (LORA) bq[0] = wc[0][0];
      else bq[0] = __builtin_bit_cast(u32x4_t, dequant_word(word_of(IC<0>{}), s_c[0], m8s[0]));
    }
    __builtin_amdgcn_sched_barrier(0);
    static_for<4 * TPW>([&](auto gc) __attribute__((always_inline)) {
      constexpr int g = decltype(gc)::value, cur = g & 1, nxt = cur ^ 1;
      constexpr bool more = g + 1 < 4 * TPW;
      constexpr int jn = (g + 1) / 4 % TPW, tn = (g + 1) % 4;
      const int slot = ((c0 + 2 * (g + 1)) ^ (nl & 15)) * 8;
      uint32_t lo = 0, hi = 0;
      static_for<MT>([&](auto mc) __attribute__((always_inline)) {
        constexpr int m = decltype(mc)::value;
        acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xq[cur][m], __builtin_bit_cast(bf16x8_t, bq[cur]), acc[m],
                                                         0, 0, 0);
        if constexpr (more) {
          xq[nxt][m] = *reinterpret_cast<const bf16x8_t*>(xb + m * 32 * XS + slot);
          if (LORA) {
            if (m == 0) bq[nxt] = wc[jn][tn % WPT];
          } else {
            if (m == 0) dequant_masks(word_of(IC<g + 1>{}), lo, hi);
            if (m == wide_slot(MT, 1)) bq[nxt].x = dequant_part<0>(lo, hi, s_c[jn], m8s[jn]);
            if (m == wide_slot(MT, 2)) bq[nxt].y = dequant_part<1>(lo, hi, s_c[jn], m8s[jn]);
            if (m == wide_slot(MT, 3)) bq[nxt].z = dequant_part<2>(lo, hi, s_c[jn], m8s[jn]);
            if (m == wide_slot(MT, 4)) bq[nxt].w = dequant_part<3>(lo, hi, s_c[jn], m8s[jn]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      });
    });
  };
  // loads of a step younger than its slab transfer (in-order counter)
  constexpr int kYounger = TPW * (LORA ? 4 : 2);
  auto wait_slab = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    if (tile_ok) __builtin_amdgcn_s_waitcnt(0x0F70 | (kYounger & 15) | ((kYounger >> 4) << 14));
    else __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
  };

  dma_x(0, 0);
  if (tile_ok) static_for<TPW>([&](auto jc) __attribute__((always_inline)) { load_w_tile(0, jc); });
  wait_slab();
  for (int step = 0; step < nsteps; ++step) {
    const int buf = step & 1;
    dma_x(step + 1, buf ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    if (tile_ok) step_math(step, buf);
    wait_slab();
  }
  // Two k-parts of a tile swap halves of their accumulators (the slab is free: the last step ended with a barrier,
  // and its surplus transfer, a repeat of the last step, has landed): the first finishes registers 0..7, the
  // second 8..15.
  constexpr int NR = 16 / KW;  // accumulator registers this wave finishes
  const int rbase = kw * NR;
  if constexpr (KW == 2) {
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();
    float* hb = reinterpret_cast<float*>(smem);  // [CT][MT][16][64]
    if (tile_ok) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r8 = 0; r8 < 8; ++r8)
          hb[(((ct * MT + m) * 16 + (kw ? r8 : r8 + 8)) << 6) + lane] = kw ? acc[m][r8] : acc[m][r8 + 8];
    }
    __syncthreads();
    if (tile_ok) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r8 = 0; r8 < 8; ++r8) {
          const float mine = kw ? acc[m][r8 + 8] : acc[m][r8];
          const float other = hb[(((ct * MT + m) * 16 + (kw ? r8 + 8 : r8)) << 6) + lane];
          acc[m][r8] = kw ? other + mine : mine + other;  // first half + second half
        }
    }
  }
  if (!tile_ok) return;
  const int col = nb * 32 + nl;
  if (!LORA && a.t16) {
    // LoRA in the epilogue: delta tile [32 rows, 32 columns] = t16 rows . B columns, 16 ranks per
    // MFMA (t rows are the A operand, so the delta lands in the accumulator layout of acc[m]);
    // y = bf16(bf16(base) + bf16(bf16(delta) ls))
    const int seg = nb * 32 >= a.seg_end[0] ? (nb * 32 >= a.seg_end[1] ? 2 : 1) : 0;
    const int tc0 = seg * a.lora_r;
    const int nkb = (a.lora_r + 15) >> 4;  // host: <= 4
    u32x4_t bfr[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      uint32_t w[4] = {0, 0, 0, 0};
      if (kb < nkb) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int rr = kb * 16 + 8 * h + j;
          const uint32_t e = rr < a.lora_r ? a.lora_b[(size_t)rr * a.N + col] : 0u;
          w[j >> 1] |= e << (16 * (j & 1));
        }
      }
      bfr[kb] = u32x4_t{w[0], w[1], w[2], w[3]};
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int trow = row0 + m * 32 + nl;
      const uint16_t* tp = a.t16 + (size_t)(trow < a.M ? trow : a.M - 1) * a.ldt16 + tc0 + 8 * h;
      f32x16_t d;
#pragma unroll
      for (int r = 0; r < 16; ++r) d[r] = 0.f;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
        if (kb < nkb) {
          const bf16x8_t tf = *reinterpret_cast<const bf16x8_t*>(tp + kb * 16);
          d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tf, __builtin_bit_cast(bf16x8_t, bfr[kb]), d, 0, 0, 0);
        }
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int row = row0 + m * 32 + acc_row(rbase + i, lane);
        if (row >= a.M) continue;
        const float dv = KW == 2 ? (kw ? d[(i + 8) & 15] : d[i]) : d[i];
        a.y_bf16[(size_t)row * a.ldy + col] = f2bf(rbf(acc[m][i]) + rbf(rbf(dv) * a.lora_ls));
      }
    }
    return;
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int row = row0 + m * 32 + acc_row(rbase + i, lane);
      if (row >= a.M) continue;
      const float v = acc[m][i];
      if (LORA) a.t_part[((size_t)slice * a.M + row) * a.ldt + col] = v;
      else if (a.y_bf16) a.y_bf16[(size_t)row * a.ldy + col] = f2bf(v);
      else a.y_part[((size_t)slice * a.M + row) * a.N + col] = v;
    }
}

// Workgroups are dispatched round-robin over the 8 XCDs (linear id % 8), each with its own L2.
// The launch is one-dimensional and maps ids so that the workgroups of an XCD share row blocks:
// with S = gcd(row blocks, 8), XCD x works on row blocks x % S, x % S + S, ... in turn, all column
// blocks and K-slices of one before the next, so the activation slab of a step is fetched into
// that L2 once and the other workgroups of the XCD hit it.  Ids past the end do nothing.
template <int MT, int CT>
__global__ __launch_bounds__(512, MT <= 4 && CT == 4 ? 4 : 1) void qlinear_mfma_wide_kernel(QLinearArgs a, int blocks, int row_blocks, int S) {
  extern __shared__ __align__(16) uint16_t smem[];
  const int id = (int)blockIdx.x, xcd = id & 7, idx = id >> 3;
  const int per_rb = blocks * a.nsplit;
  const int p = xcd / S + (8 / S) * idx;
  // an XCD with an even number of row blocks takes them two at a time, the same column block on both in
  // consecutive workgroups, so that a weight tile fetched for one is an L2 hit for the other
  const int R = (row_blocks + S - 1) / S, Gr = (R & 1) ? 1 : 2;
  const int blk = p / (per_rb * Gr), within = p % (per_rb * Gr);
  const int bz = xcd % S + S * (blk * Gr + within % Gr);
  if (bz >= row_blocks) return;
  const int cb = within / Gr, bx = cb % blocks, by = cb / blocks;
  if (bx >= a.n_main_blocks) gemm_block_wide<MT, CT, true>(a, smem, bx, by, bz);
  else gemm_block_wide<MT, CT, false>(a, smem, bx, by, bz);
}

// t16[m][c] = bf16(sum of the planes' values) for c < cols, 0 up to the row stride ldt
__global__ __launch_bounds__(256) void lora_t_reduce_kernel(const float* t_part, int nsplit, int M, int ldt,
                                                            uint16_t* t16, int cols) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= M * ldt) return;
  const int m = i / ldt, c = i - m * ldt;
  float t = 0.f;
  if (c < cols)
    for (int sp = 0; sp < nsplit; ++sp) t += t_part[((size_t)sp * M + m) * ldt + c];
  t16[(size_t)m * ldt + c] = f2bf(t);
}

int lora_t_reduce(hipStream_t st, const float* t_part, int nsplit, int M, uint16_t* t16, int cols) {
  hipLaunchKernelGGL(lora_t_reduce_kernel, dim3((M * TMX_MAX_RPAD + 255) / 256), dim3(256), 0, st, t_part, nsplit, M,
                     TMX_MAX_RPAD, t16, cols);
  return check_launch();
}

template <int MT, int CT>
static int launch_wide(hipStream_t st, QLinearArgs a, int part) {
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&qlinear_mfma_wide_kernel<MT, CT>), hipFuncAttributeMaxDynamicSharedMemorySize,
      (int)wide_lds(MT));
  if (attr != hipSuccess) return TMX_ERR_LAUNCH;
  a.n_main_blocks = part == 1 ? 0 : (a.N + CT * 32 - 1) / (CT * 32);
  const int blocks = a.n_main_blocks + ((a.a_t && part != 2) ? a.lora_blocks_per_split : 0);
  const int row_blocks = (a.M + MT * 32 - 1) / (MT * 32);
  int S = 8;
  while (row_blocks % S) S >>= 1;  // gcd(row_blocks, 8)
  // ids cover 8 / S XCDs x (row_blocks / S) row blocks x blocks x nsplit per residue, rounded up to 8
  const long total = (long)blocks * a.nsplit * row_blocks;
  const int ids = (int)((total + 7) / 8 * 8);
  hipLaunchKernelGGL((qlinear_mfma_wide_kernel<MT, CT>), dim3(ids), dim3(512), wide_lds(MT), st, a, blocks, row_blocks, S);
  return check_launch();
}

// Which tile and how many K-slices.  A launch of at most one workgroup per CU takes (steps of a slice) x (time of a
// step) + a fixed part; a step is 0.24 us + 0.05 us per column tile and row tile (measured, 8B and 1B shapes, 160 to
// 4096 rows: 0.64 us for 2 x 4 tiles, 1.04 for 4 x 4, 1.76 for 8 x 4, 3.37 for 8 x 8), the fixed part 8 us (first slab
// and weights from cold caches, exchange, stores).  More workgroups run in rounds, except that two workgroups of up to
// 4 x 4 tiles share a CU and hide each other's fixed part.  K-slices cost their f32 planes twice, written here and
// read by the consumer.  So the tile is as large as still gives every CU one workgroup: at 256 rows of the 8B shape
// q|k|v runs 4 x 4 tiles in 2 slices (25.6 us with its planes; 8 x 8 in 8 slices 34.3), o 2 x 4 in 2 (19.2; 30.6),
// gate|up 8 x 4 unsplit (65.7; 72.3), down 4 x 4 in 4 (40.7; 50.7); from 4096 rows on 8 x 8 wins everywhere.
static const int kWideTiles[][2] = {{2, 4}, {3, 4}, {4, 4}, {5, 4}, {6, 4}, {7, 4}, {8, 4}, {4, 8}, {5, 8}, {6, 8}, {7, 8}, {8, 8}};

WidePlan wide_plan(int M, int N, int K, int nsplit) {
  const int cus = device_cus(), KT = K >> 6;
  WidePlan best = {8, 8, nsplit > 0 ? nsplit : 1};
  float best_cost = 1e30f;
  for (const auto& t : kWideTiles) {
    const int mt = t[0], ct = t[1];
    const long tiles = (long)((M + 32 * mt - 1) / (32 * mt)) * ((N + 32 * ct - 1) / (32 * ct));
    for (int s = nsplit > 0 ? nsplit : 1; s <= (nsplit > 0 ? nsplit : TMX_MAX_SPLITS); ++s) {
      if (!slices_ok(KT, s)) continue;
      const float loop = (slice_len(KT, s) / kWideTS) * (0.24f + 0.05f * mt * ct);
      const long n = (tiles * s + cus - 1) / cus;  // workgroups of a CU
      const float t_us = mt <= 4 && ct == 4 ? 8.f + (n == 1 ? 1.f : 0.92f) * n * loop : n * (8.f + loop);
      const float cost = t_us + (s > 1 ? 0.3e-6f * s * (float)M * N * 4.f : 0.f);
      if (cost < best_cost) { best_cost = cost; best = {mt, ct, s}; }
    }
  }
  return best;
}

// part: 0 = main blocks and LoRA blocks in one launch, 1 = LoRA blocks only, 2 = main blocks only
int qwide_launch(hipStream_t st, const QLinearArgs& a, int part) {
  const WidePlan p = part == 1 ? WidePlan{8, 8, 1} : wide_plan(a.M, a.N, a.K, a.nsplit);
#define TMX_WIDE_CASE(MM, CC) \
  if (p.mt == MM && p.ct == CC) return launch_wide<MM, CC>(st, a, part);
  TMX_WIDE_CASE(2, 4)
  TMX_WIDE_CASE(3, 4)
  TMX_WIDE_CASE(4, 4)
  TMX_WIDE_CASE(5, 4)
  TMX_WIDE_CASE(6, 4)
  TMX_WIDE_CASE(7, 4)
  TMX_WIDE_CASE(8, 4)
  TMX_WIDE_CASE(4, 8)
  TMX_WIDE_CASE(5, 8)
  TMX_WIDE_CASE(6, 8)
  TMX_WIDE_CASE(7, 8)
  TMX_WIDE_CASE(8, 8)
#undef TMX_WIDE_CASE
  return TMX_ERR_UNSUPPORTED;
}

}  // namespace tmx
