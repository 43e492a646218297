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
constexpr int kWideTiles32 = TMX_MAX_FILL_ROWS / 32;  // words per kind in a hand-over area: arrivals | ready flags
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
// the MFMA of a group behind which part p (1..4) of the next fragment's dequantisation goes
constexpr int wide_slot(int MT, int p) { return p < MT ? p : MT - 1; }
constexpr size_t wide_lds(int MT) { return (size_t)2 * MT * 32 * kWideXS * 2; }

template <int MT, int CT>
__device__ __forceinline__ void gemm_block_wide(const QLinearArgs& a, uint16_t* smem, int bx, int slice, int bz) {
  constexpr int TS = kWideTS, XS = kWideXS, ROWS = MT * 32, KW = 8 / CT, TPW = TS / KW;
  static_assert(KW * CT == 8 && TPW >= 1, "8 waves, at least one k-tile of a step each");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ct = wave % CT, kw = wave / CT;
  const int h = lane >> 5, nl = lane & 31;
  const int KT = a.K >> 6;
  const int per = a.kt_per_split;
  const int kb0 = slice * per;
  const int kb1 = (kb0 + per < KT) ? kb0 + per : KT;
  const int nsteps = (kb1 - kb0) / TS, last_step = nsteps - 1;  // host: whole steps
  if (nsteps <= 0) return;
  const int row0 = bz * ROWS;
  const int rows = a.M - row0 < ROWS ? a.M - row0 : ROWS;  // host: >= 1
  const int gs = __builtin_ctz(a.G >> 6), KG = a.K / a.G;
  const int NT = a.N >> 5, nb = bx * CT + ct;
  const bool tile_ok = nb < NT;  // waves past the last tile only help with the slab

  const __amdgpu_buffer_rsrc_t rw = make_rsrc(a.qw, (uint32_t)NT * KT * 1024u);
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.scales, (uint32_t)NT * KG * 64u);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x + (size_t)row0 * a.ldx, (uint32_t)rows * a.ldx * 2u);
  const int wv = (nb * KT * 64 + lane) * 16;
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
  u32x4_t wring[TPW];
  uint16_t sring[TPW];

  auto load_w_tile = [&](int step, auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    step = step < last_step ? step : last_step;
    const int kt = kb0 + step * TS + kw * TPW + j;
    wring[j] = __builtin_amdgcn_raw_buffer_load_b128(rw, wv, kt * 1024, 0);
    sring[j] = __builtin_amdgcn_raw_buffer_load_b16(rs, sv, (kt >> gs) * 64, 0);
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
    u32x4_t wc[TPW];
    float s_c[TPW], m8s[TPW];
    static_for<TPW>([&](auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      wc[j] = wring[j];
      s_c[j] = bf2f(sring[j]);
      m8s[j] = -8.f * s_c[j];
      load_w_tile(step + 1, jc);  // registers consumed: refill them one step ahead
    });
    const uint16_t* xb = smem + (size_t)buf * ROWS * XS + nl * XS;
    const int c0 = 8 * TPW * kw + h;  // this wave's first chunk of a slab row
    auto word_of = [&](auto gc) __attribute__((always_inline)) {
      constexpr int g = decltype(gc)::value, j = g / 4, t = g % 4;
      return t == 0 ? wc[j].x : (t == 1 ? wc[j].y : (t == 2 ? wc[j].z : wc[j].w));
    };
    bf16x8_t xq[2][MT];
    u32x4_t bq[2];
    {
      const int slot = (c0 ^ (nl & 15)) * 8;
#pragma unroll
      for (int m = 0; m < MT; ++m) xq[0][m] = *reinterpret_cast<const bf16x8_t*>(xb + m * 32 * XS + slot);
      bq[0] = __builtin_bit_cast(u32x4_t, dequant_word(word_of(IC<0>{}), s_c[0], m8s[0]));
    }
    __builtin_amdgcn_sched_barrier(0);
    static_for<4 * TPW>([&](auto gc) __attribute__((always_inline)) {
      constexpr int g = decltype(gc)::value, cur = g & 1, nxt = cur ^ 1;
      constexpr bool more = g + 1 < 4 * TPW;
      constexpr int jn = (g + 1) / 4 % TPW;
      const int slot = ((c0 + 2 * (g + 1)) ^ (nl & 15)) * 8;
      uint32_t lo = 0, hi = 0;
      static_for<MT>([&](auto mc) __attribute__((always_inline)) {
        constexpr int m = decltype(mc)::value;
        acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xq[cur][m], __builtin_bit_cast(bf16x8_t, bq[cur]), acc[m],
                                                         0, 0, 0);
        if constexpr (more) {
          xq[nxt][m] = *reinterpret_cast<const bf16x8_t*>(xb + m * 32 * XS + slot);
          if (m == 0) dequant_masks(word_of(IC<g + 1>{}), lo, hi);
          if (m == wide_slot(MT, 1)) bq[nxt].x = dequant_part<0>(lo, hi, s_c[jn], m8s[jn]);
          if (m == wide_slot(MT, 2)) bq[nxt].y = dequant_part<1>(lo, hi, s_c[jn], m8s[jn]);
          if (m == wide_slot(MT, 3)) bq[nxt].z = dequant_part<2>(lo, hi, s_c[jn], m8s[jn]);
          if (m == wide_slot(MT, 4)) bq[nxt].w = dequant_part<3>(lo, hi, s_c[jn], m8s[jn]);
          __builtin_amdgcn_sched_barrier(0);
        }
      });
    });
  };
  // loads of a step younger than its slab transfer (in-order counter)
  constexpr int kYounger = TPW * 2;
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
  bool t_ready = true;
  if (a.t16 && a.sync) {
    // t of this block's rows comes from the LoRA workgroups of the launch (without a.sync: of a launch before): wait (a
    // bounded number of polls) for the flags of its row tiles
    __shared__ uint32_t s_late;
    if (tid == 0) s_late = 0u;
    __syncthreads();
    if (tid < MT && row0 + tid * 32 < a.M) {
      uint32_t* flag = a.sync + kWideTiles32 + (row0 >> 5) + tid;
      uint32_t ok = 0;
      for (int spin = 0; spin < (1 << 20); ++spin) {
        if (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) { ok = 1; break; }
        __builtin_amdgcn_s_sleep(1);
      }
      if (!ok) {
        s_late = 1u;
        if (a.sync_status) __hip_atomic_store(a.sync_status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();
    t_ready = s_late == 0u;  // false: t is taken as zero (the status word says so)
  }
  if (!tile_ok) return;
  const int col = nb * 32 + nl;
  if (a.t16) {
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
    const __amdgpu_buffer_rsrc_t rt = make_rsrc(a.t16, (uint32_t)a.M * a.ldt16 * 2u);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int trow = row0 + m * 32 + nl;
      const int tp = ((trow < a.M ? trow : a.M - 1) * a.ldt16 + tc0 + 8 * h) * 2;
      f32x16_t d;
#pragma unroll
      for (int r = 0; r < 16; ++r) d[r] = 0.f;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
        if (kb < nkb) {
          // past this XCD's L2: the rows were written during this launch
          u32x4_t tf = {0u, 0u, 0u, 0u};
          if (t_ready) tf = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rt, tp + kb * 32, 0, 0x10));
          d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, tf), __builtin_bit_cast(bf16x8_t, bfr[kb]), d, 0, 0, 0);
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
      if (a.y_bf16) a.y_bf16[(size_t)row * a.ldy + col] = f2bf(v);
      else a.y_part[((size_t)slice * a.M + row) * a.N + col] = v;
    }
}

// t = x . A of one row tile (32 rows) over one K-slice.  The 8 waves are column tiles of A (1, 2 or 4) x k-parts; a wave
// reads its x fragments straight from global memory (32 rows, 64 bytes each per pair of loads; the column tiles of a
// k-part hit the same lines) two k-tiles ahead, the parts meet in LDS.  Every slice leaves its f32 plane; with a
// hand-over area (a.sync) the last slice of the row tile to arrive adds the planes in slice order and writes the
// rounded t: bf16 for the epilogues of this launch (a.t16, then its ready flag), f32 for a consumer behind it
// (a.t_fin).  Stores are write-through and loads go past L2 (sc1), so no cache write-back happens inside the
// launch.  In the projection's launch these workgroups come first in dispatch order and wait for nobody.  What bounds
// them is latency: about 8 us at 256 rows, hidden behind the main workgroups' loop, where a LoRA-only launch and a
// reduction launch in front of the projection took 14 + 5 us (decode step of 256 sequences, 8 layers: 3.43 -> 3.25 ms).
__device__ __forceinline__ void wide_lora_block(const QLinearArgs& a, float* red, int id) {
  const int RT = (a.M + 31) >> 5, rt = id % RT, ks = id / RT;
  if (ks >= a.n_lora_slices) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, nl = lane & 31;
  const int KT = a.K >> 6, NT = a.Rpad >> 5, NP = NT > 2 ? 4 : NT, nk = 8 / NP;
  const int ct = wave % NP, kp = wave / NP;
  const int k0 = ks * a.kt_per_lora_split, k1 = min(k0 + a.kt_per_lora_split, KT);
  if (a.sync_clear && ks == 0 && tid < 2) a.sync_clear[tid * kWideTiles32 + rt] = 0u;  // the next launch's area

  f32x16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  if (ct < NT) {
    const int row = min(rt * 32 + nl, a.M - 1);
    const u32x4_t* xp = reinterpret_cast<const u32x4_t*>(a.x + (size_t)row * a.ldx) + h;
    const u32x4_t* ap = reinterpret_cast<const u32x4_t*>(a.a_t) + (size_t)ct * 256 + lane;
    u32x4_t xr[2][4], ar[2][4];
    auto load = [&](int kt, auto pc) __attribute__((always_inline)) {
      constexpr int p = decltype(pc)::value;
      kt = kt < k1 ? kt : k1 - 1;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        xr[p][t] = xp[kt * 8 + 2 * t];
        ar[p][t] = ap[((size_t)kt * NT) * 256 + t * 64];
      }
    };
    auto math = [&](auto pc) __attribute__((always_inline)) {
      constexpr int p = decltype(pc)::value;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, xr[p][t]),
                                                      __builtin_bit_cast(bf16x8_t, ar[p][t]), acc, 0, 0, 0);
    };
    int kt = k0 + kp;
    if (kt < k1) {
      load(kt, IC<0>{});
      load(kt + nk, IC<1>{});
      for (; kt < k1; kt += 2 * nk) {
        math(IC<0>{});
        load(kt + 2 * nk, IC<0>{});
        if (kt + nk < k1) math(IC<1>{});
        load(kt + 3 * nk, IC<1>{});
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) red[(wave * 16 + r) * 64 + lane] = acc[r];
  __syncthreads();
  // thread: four adjacent columns of a row
  const int quads = a.Rpad >> 2;
  const __amdgpu_buffer_rsrc_t rp = make_rsrc(a.t_part, 0x7FFFFFFFu);
  const bool final_here = a.sync != nullptr;
  auto finish = [&](int row, int c, f32x4_t v) __attribute__((always_inline)) {
    const uint32_t lo = pack_bf2(v[0], v[1]), hi = pack_bf2(v[2], v[3]);
    if (a.t16)
      __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{lo, hi}, make_rsrc(a.t16, (uint32_t)a.M * a.ldt16 * 2u),
                                            (row * a.ldt16 + c) * 2, 0, 0x10);
    if (a.t_fin) *reinterpret_cast<f32x4_t*>(a.t_fin + (size_t)row * a.ldt + c) = f32x4_t{bf_lo(lo), bf_hi(lo), bf_lo(hi), bf_hi(hi)};
  };
  for (int e = tid; e < 32 * quads; e += 512) {
    const int rl = e / quads, c = (e - rl * quads) * 4, row = rt * 32 + rl;
    if (row >= a.M) continue;
    const int r = (rl >> 3) * 4 + (rl & 3), ln = ((rl >> 2) & 1) * 32 + (c & 31);
    f32x4_t v = {0.f, 0.f, 0.f, 0.f};
    for (int p = 0; p < nk; ++p) v += *reinterpret_cast<const f32x4_t*>(red + ((p * NP + (c >> 5)) * 16 + r) * 64 + ln);
    if (final_here && a.n_lora_slices == 1) finish(row, c, v);
    else if (!final_here) *reinterpret_cast<f32x4_t*>(a.t_part + ((size_t)ks * a.M + row) * a.ldt + c) = v;
    else __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), rp, (int)((((size_t)ks * a.M + row) * a.ldt + c) * 4), 0, 0x10);
  }
  if (!final_here) return;
  __builtin_amdgcn_s_waitcnt(0);  // this thread's stores are in memory
  __syncthreads();
  if (a.n_lora_slices > 1) {
    __shared__ uint32_t s_last;
    if (tid == 0)
      s_last = __hip_atomic_fetch_add(a.sync + rt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)(a.n_lora_slices - 1);
    __syncthreads();
    if (!s_last) return;
    for (int e = tid; e < 32 * quads; e += 512) {
      const int rl = e / quads, c = (e - rl * quads) * 4, row = rt * 32 + rl;
      if (row >= a.M) continue;
      f32x4_t t = {0.f, 0.f, 0.f, 0.f};
      for (int p0 = 0; p0 < a.n_lora_slices; p0 += 8) {
        u32x4_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int p = min(p0 + u, a.n_lora_slices - 1);
          v[u] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rp, (int)((((size_t)p * a.M + row) * a.ldt + c) * 4), 0, 0x10));
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (p0 + u < a.n_lora_slices) t += __builtin_bit_cast(f32x4_t, v[u]);
      }
      finish(row, c, t);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  if (tid == 0) __hip_atomic_store(a.sync + kWideTiles32 + rt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Workgroups are dispatched round-robin over the 8 XCDs (linear id % 8), each with its own L2.
// The launch is one-dimensional and maps ids so that the workgroups of an XCD share row blocks:
// with S = gcd(row blocks, 8), XCD x works on row blocks x % S, x % S + S, ... in turn, all column
// blocks and K-slices of one before the next, so the activation slab of a step is fetched into
// that L2 once and the other workgroups of the XCD hit it.  Ids past the end do nothing.
template <int MT, int CT>
__global__ __launch_bounds__(512, MT <= 4 && CT == 4 ? 4 : 1) void qlinear_mfma_wide_kernel(QLinearArgs a, int blocks, int row_blocks, int S) {
  extern __shared__ __align__(16) uint16_t smem[];
  if ((int)blockIdx.x < a.lora_wgs) {
    wide_lora_block(a, reinterpret_cast<float*>(smem), (int)blockIdx.x);
    return;
  }
  const int id = (int)blockIdx.x - a.lora_wgs, xcd = id & 7, idx = id >> 3;  // host: lora_wgs % 8 == 0
  const int per_rb = blocks * a.nsplit;
  const int p = xcd / S + (8 / S) * idx;
  // an XCD with an even number of row blocks takes them two at a time, the same column block on both in
  // consecutive workgroups, so that a weight tile fetched for one is an L2 hit for the other
  const int R = (row_blocks + S - 1) / S, Gr = (R & 1) ? 1 : 2;
  const int blk = p / (per_rb * Gr), within = p % (per_rb * Gr);
  const int bz = xcd % S + S * (blk * Gr + within % Gr);
  if (bz >= row_blocks) return;
  const int cb = within / Gr, bx = cb % blocks, by = cb / blocks;
  gemm_block_wide<MT, CT>(a, smem, bx, by, bz);
}

template <int MT, int CT>
static int launch_wide(hipStream_t st, QLinearArgs a) {
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&qlinear_mfma_wide_kernel<MT, CT>), hipFuncAttributeMaxDynamicSharedMemorySize,
      (int)wide_lds(MT));
  if (attr != hipSuccess) return TMX_ERR_LAUNCH;
  const int blocks = (a.N + CT * 32 - 1) / (CT * 32);
  a.lora_wgs = a.a_t ? ((a.M + 31) / 32 * a.n_lora_slices + 7) / 8 * 8 : 0;
  const int row_blocks = (a.M + MT * 32 - 1) / (MT * 32);
  int S = 8;
  while (row_blocks % S) S >>= 1;  // gcd(row_blocks, 8)
  // ids cover 8 / S XCDs x (row_blocks / S) row blocks x blocks x nsplit per residue, rounded up to 8
  const long total = (long)blocks * a.nsplit * row_blocks;
  const int ids = (int)((total + 7) / 8 * 8);
  hipLaunchKernelGGL((qlinear_mfma_wide_kernel<MT, CT>), dim3(a.lora_wgs + ids), dim3(512), wide_lds(MT), st, a, blocks, row_blocks, S);
  return check_launch();
}

// Which tile and how many K-slices.  A launch of at most one workgroup per CU takes (steps of a slice) x (time of a
// step) + a fixed part; a step is priced at 0.24 us + 0.05 us per column tile and row tile, the fixed part at 8 us (first
// slab and weights from cold caches, exchange, stores).  Measured at K = 4096, fixed part taken off: 0.58 us a step for
// 2 x 4 tiles, 0.95 for 4 x 4, 1.75 for 8 x 4, 3.0 for 8 x 8.  More workgroups run in rounds, except that two workgroups of up to
// 4 x 4 tiles share a CU and hide each other's fixed part.  K-slices cost their f32 planes twice, written here and
// read by the consumer.  So the tile is as large as still gives every CU one workgroup: at 256 rows of the 8B shape (us,
// without LoRA and without the consumer's read) q|k|v runs 4 x 4 tiles in 2 slices, 24.3 (8 x 8 in 8: 25.9 and four times
// the planes), o 2 x 4 in 2, 19.0 (8 x 8 in 8: 25.0), gate|up 8 x 4 unsplit, 64.0 (8 x 8 unsplit: 88.3), down 4 x 4 in 4,
// 38.0 (8 x 8 in 8: 47.9); 4096 rows of gate|up 8 x 8, 771 (4 x 4: 888).  Every tile and slice count timed for ten
// matrices of the 8B, 1B and Qwen3-8B shapes at 13 row counts from 135 to 4096: the choice is 1.4 % slower than the best
// in the mean, more than 5 % in 18 of 130, 13 % at worst (768 rows of 4096 x 28672: 3 x 4 tiles 184, 6 x 8 162).  What it
// prices wrong is several rounds of large tiles, about 10 % too high (2048 rows there: 4 x 4 448, 8 x 8 418).
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

// t in a launch of its own, ordered in front of the projection, for callers that have no word to ask whether a wait ran
// out (tmx_qlora_linear).  It costs the launch, 2 to 7 us: 300 x 4096 x 12288 with rank 16 takes 63 us against 57 with
// the LoRA workgroups inside, 4096 x 4096 x 28672 841 against 840.
int qwide_lora_launch(hipStream_t st, QLinearArgs a) {
  static_assert(wide_lds(2) >= 8 * 16 * 64 * 4, "the accumulators of the 8 waves meet in LDS");
  if (!a.a_t || !a.sync || a.M > TMX_MAX_FILL_ROWS) return TMX_ERR_ARG;
  a.lora_wgs = ((a.M + 31) / 32 * a.n_lora_slices + 7) / 8 * 8;
  hipLaunchKernelGGL((qlinear_mfma_wide_kernel<2, 4>), dim3(a.lora_wgs), dim3(512), wide_lds(2), st, a, 1, 1, 1);
  return check_launch();
}

int qwide_launch(hipStream_t st, const QLinearArgs& a) {
  if (a.sync && a.M > TMX_MAX_FILL_ROWS) return TMX_ERR_SHAPE;  // the hand-over area has a word per row tile
  const WidePlan p = wide_plan(a.M, a.N, a.K, a.nsplit);
#define TMX_WIDE_CASE(MM, CC) \
  if (p.mt == MM && p.ct == CC) return launch_wide<MM, CC>(st, a);
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
