// int4 projections of more than 128 rows: cache fill over prompts, scoring passes, decode steps of many sequences.
// Same weights, rounding and LoRA arithmetic as qlinear.hip (tunix/models/llama3/model.py:216-218, :489-496 with the
// qwix-wrapped projections); reads for the reference's prefill (tunix/generate/sampler.py:601-730).
#include "tmx_kernels.h"

namespace tmx {

// A workgroup is 8 waves = CT column tiles of 32 x KW = 8 / CT k-parts over MT row tiles of 32.  A wave multiplies its
// column tile against all row tiles (16 MT accumulator registers) on the 16 x 16 x 32 MFMA with the weights as A operand,
// so a lane ends up with four consecutive columns of a row, and a dequantised weight fragment feeds 2 MT MFMAs.
// What bounds it: at a thousand rows and more the power of the chip, and the schedule for the rest.  With every CU at work the clock
// falls from 2.39 to 1.8 GHz (4096 x 4096 x 28672: its MFMAs, 16 cycles each, are 0.64 of the launch at that clock), and the same
// launch with zeros for x runs 1.27 times as fast.  Registers only and on
// random bf16 the 16 x 16 x 32 MFMA sustains 2.02 PFLOP/s and the 32 x 32 x 16 one 1.77, so the former, although it takes
// twice the issue slots.  In one round of workgroups it is the schedule: the loop below takes 2.18 us a step of 8 x 8 tiles
// where its MFMAs alone are 1.71.  Before (32 x 32 x 16, the barrier between two steps, the transfers of a slab in one
// burst behind it), us: 4096 x 4096 x 28672 800 -> 715, 4096 x 14336 x 4096 385 -> 338, 256 x 4096 x 28672 64 -> 55.
// A q4t word holds 8 k of a column; lane (h, n) of a tile has those of column n, k-chunk 2 t + h in word t.  Two lane
// swaps of the words of a group leave lane group q of 16 lanes with chunk q of column n % 16 in one and of 16 + n % 16 in
// the other.  In that order of the chunks the MFMA rounds like two 32 x 32 x 16 ones, bit for bit.
// Weights come by buffer loads, the activation slab of a step (2 k-tiles) by direct-to-LDS loads into NB buffers: slab
// rows are 256 bytes (four per 1 KiB transfer), their 16-byte chunks XOR-swizzled by row % 16.  With KW = 2 a wave takes
// one k-tile of every step, and the two halves of a column tile meet through LDS at the end.
// NB is 4 for the smallest tile, whose step is shorter than a load takes (256 x 4096 x 4096 in 2 slices: 19.1 -> 15.9 us), 2
// for the others (3 x 4 in 3 buffers measured the same).
constexpr int kWideTS = 2, kWideXS = 128;
constexpr int kWideTiles32 = TMX_MAX_FILL_ROWS / 32;  // words per kind in a hand-over area: arrivals | ready flags
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
// four bf16 of an output row in one store: rows may begin at any element (a caller's stride or view), and 8-byte stores take
// every address
__device__ __forceinline__ void store8(uint16_t* p, u32x2_t v) { __builtin_memcpy(p, &v, 8); }
constexpr int wide_bufs(int mt) { return mt == 2 ? 4 : 2; }
constexpr size_t wide_lds(int mt) { return (size_t)wide_bufs(mt) * mt * 32 * kWideXS * 2; }

// The product itself: acc[u][r] = rows 16 r .. + 15 of x times columns 16 u .. + 15 of a wave's column tile, over nsteps steps
// from k-tile kb0 on.  wv / sv: byte offsets of this lane's words and scale in the first k-tile (of the tile's columns
// lane % 32; any 16 + 16 columns do); xo(i): of this lane's 16 bytes of the i-th slab transfer.  Every wave of the workgroup
// takes part; one that is not `active` only helps with the slab.
template <int MT, int KW, int NB, class XO>
__device__ __forceinline__ void wide_core(uint16_t* smem, __amdgpu_buffer_rsrc_t rw, int wv, __amdgpu_buffer_rsrc_t rs, int sv,
                                          int gs, __amdgpu_buffer_rsrc_t rx, XO xo, int kb0, int nsteps, int kw, bool active,
                                          f32x4_t (&acc)[2][2 * MT]) {
  constexpr int TS = kWideTS, XS = kWideXS, ROWS = MT * 32, TPW = TS / KW;
  constexpr int WB = NB > 2 ? NB : 1;                      // weight registers (steps on the way)
  constexpr int G = 2 * TPW, RF = 2 * MT;                  // groups of 32 k a step, x fragments (16 rows) of a group
  constexpr int RING = RF <= 4 ? RF : RF / 2;              // x fragments in registers
  constexpr int MEET = RF - RING + 2 < RF ? RF - RING + 2 : RF - 1;  // the fragment of the last group in front of which the waves meet
  constexpr int DS = (G - 1) * RF / MT < 2 ? 1 : 2;        // fragments between two slab transfers
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int q = lane >> 4, nl = lane & 15, last_step = nsteps - 1;
#pragma unroll
  for (int r = 0; r < RF; ++r) acc[0][r] = acc[1][r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  u32x4_t wring[WB][TPW], wc[TPW];
  uint16_t sring[WB][TPW];
  NibbleScale sc[TPW][2];

  auto load_w = [&](int step, auto bc) __attribute__((always_inline)) {
    constexpr int b = decltype(bc)::value;
    step = step < last_step ? step : last_step;
    static_for<TPW>([&](auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      const int kt = kb0 + step * TS + kw * TPW + j;
      wring[b][j] = __builtin_amdgcn_raw_buffer_load_b128(rw, wv, kt * 1024, 0);
      sring[b][j] = __builtin_amdgcn_raw_buffer_load_b16(rs, sv, (kt >> gs) * 64, 0);
    });
  };
  auto take_w = [&](auto bc) __attribute__((always_inline)) {
    constexpr int b = decltype(bc)::value;
    static_for<TPW>([&](auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      wc[j] = WB == 1 ? moved(wring[b][j]) : wring[b][j];
      const uint32_t both = WB == 1 ? moved((uint32_t)sring[b][j]) : (uint32_t)sring[b][j];
      const auto s = __builtin_amdgcn_permlane16_swap(both, both, false, false);
      sc[j][0] = nibble_scale(bf2f((uint16_t)s[0]));
      sc[j][1] = nibble_scale(bf2f((uint16_t)s[1]));
    });
  };
  auto dma_x = [&](int step, int buf, int i) __attribute__((always_inline)) {
    step = step < last_step ? step : last_step;
    uint16_t* base = smem + (size_t)buf * ROWS * XS + wave * 4 * XS;
    load_row_to_lds(rx, base + i * 32 * XS, xo(i), step * (TS * 128));
  };
  // all but the youngest loads of this wave have arrived and its LDS reads are done; then all waves
  auto meet = [&](auto younger) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(decltype(younger)::value) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  bf16x8_t xq[RING];
  u32x4_t bq[2][2];  // weight fragments of two groups
  uint32_t words[2];
  NibblePairs pairs;
  const int c0 = 8 * TPW * kw + q;  // this lane's first chunk of a slab row
  const uint16_t* xlane = smem + nl * XS;
  auto read_x = [&](const uint16_t* xb, auto rc) __attribute__((always_inline)) {
    constexpr int r = decltype(rc)::value;
    xq[r % RING] = *reinterpret_cast<const bf16x8_t*>(xb + r * 16 * XS);
  };
  // an eighth of the weight fragments of group g
  auto dequant = [&](auto gc, auto pc) __attribute__((always_inline)) {
    constexpr int g = decltype(gc)::value, p = decltype(pc)::value, j = g / 2;
    if constexpr (p == 0) {
      const auto x = __builtin_amdgcn_permlane32_swap(wc[j][g % 2 * 2], wc[j][g % 2 * 2 + 1], false, false);
      const auto w = __builtin_amdgcn_permlane16_swap(x[0], x[1], false, false);
      words[0] = w[0]; words[1] = w[1];
    }
    dequant_part<p % 4>(words[p / 4], sc[j][p / 4], pairs, bq[g & 1][p / 4]);
  };
  // A step is G groups of RF fragments of two MFMAs.  Behind the MFMAs of a fragment its register is refilled with the
  // one RING further on, and the weight fragments of the next group are dequantised an eighth at a time, so the matrix pipe
  // waits neither for LDS nor for the VALU; the transfers of a slab are spread over the first fragments of a step
  // (in one burst behind the barrier they hold up all waves: 256 x 14336 x 4096 in 8 x 8 tiles 310 -> 268 us).  The order is pinned.
  // The barrier that hands over the next slab stands inside the last group, where no fragment of this slab is left to
  // read and those in registers keep the pipe busy; the first ones of the next step are read behind it.
  // The wave that is behind goes first (s_setprio falls with the groups done): otherwise the older of the two waves of a
  // SIMD runs ahead and then waits at the barrier, and the other cannot fill the pipe by itself (717 us against 750 at
  // 4096 x 4096 x 28672).
  // buf: the slab's buffer, step % NB; bc: the same as a constant where WB > 1
  auto step_math = [&](int step, int buf, auto bc) __attribute__((always_inline)) {
    constexpr int b = decltype(bc)::value;
    const int next = buf + 1 == NB ? 0 : buf + 1, prev = buf == 0 ? NB - 1 : buf - 1;
    const uint16_t* xs = xlane + (size_t)buf * ROWS * XS;
    const uint16_t* xn = xlane + (size_t)next * ROWS * XS + (c0 ^ nl) * 8;
    static_for<G>([&](auto gc) __attribute__((always_inline)) {
      constexpr int g = decltype(gc)::value;
      constexpr bool last = g == G - 1;
      __builtin_amdgcn_s_setprio(G - 1 - g);
      if constexpr (last) take_w(IC<(b + 1) % WB>{});
      const uint16_t* xb = xs + ((c0 + 4 * g) ^ nl) * 8;
      const uint16_t* xb1 = last ? xn : xs + ((c0 + 4 * (g + 1)) ^ nl) * 8;
      static_for<RF>([&](auto rc) __attribute__((always_inline)) {
        constexpr int r = decltype(rc)::value, f = g * RF + r;
        if constexpr (last && r == MEET) {
          // the next slab was requested NB - 2 slabs and weight loads ago (at least one of the latter in the first steps)
          meet(IC<(NB - 2) * MT + (NB > 2 ? 2 * TPW : 0)>{});
          load_w(step + 1 + WB, IC<(b + 1) % WB>{});
          __builtin_amdgcn_sched_barrier(0);
        }
        static_for<2>([&](auto uc) __attribute__((always_inline)) {
          constexpr int u = decltype(uc)::value;
          acc[u][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, bq[g & 1][u]), xq[r % RING], acc[u][r], 0, 0, 0);
          static_for<8>([&](auto pc) __attribute__((always_inline)) {
            if constexpr (decltype(pc)::value * RF / 4 == 2 * r + u) dequant(IC<last ? 0 : g + 1>{}, pc);
          });
          if constexpr (u == 0) __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (f % DS == 0 && f / DS < MT) dma_x(step + NB - 1, prev, f / DS);
        if constexpr (r + RING < RF) {
          read_x(xb, IC<r + RING>{});
        } else if constexpr (!last) {
          read_x(xb1, IC<r + RING - RF>{});
        } else if constexpr (r >= MEET) {  // two at a time until the two left out in front of the barrier are caught up
          constexpr int n = r - MEET, t0 = n < 2 ? 2 * n : n + 2, t1 = r + 1 == RF ? RING : n < 1 ? 2 : n + 3;
          static_for<t1 - t0>([&](auto nc) __attribute__((always_inline)) { read_x(xb1, IC<t0 + decltype(nc)::value>{}); });
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };

  // (in this order, which the counts of the waits assume)
  static_for<WB>([&](auto bc) __attribute__((always_inline)) { load_w(decltype(bc)::value, bc); });
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < (NB - 1) * MT; ++i) {
    dma_x(i / MT, i / MT, i % MT);
    if (i % MT == MT - 1) __builtin_amdgcn_sched_barrier(0);
  }
  meet(IC<(NB - 2) * MT>{});
  take_w(IC<0>{});
  load_w(WB, IC<0>{});
  __builtin_amdgcn_sched_barrier(0);
  if (active) {
    static_for<RING>([&](auto rc) __attribute__((always_inline)) { read_x(xlane + (c0 ^ nl) * 8, rc); });
    static_for<8>([&](auto pc) __attribute__((always_inline)) { dequant(IC<0>{}, pc); });
    if constexpr (WB == 1) {
      for (int step = 0; step < nsteps; ++step) step_math(step, step & 1, IC<0>{});
    } else {
      for (int step = 0; step < nsteps; step += NB)
        static_for<NB>([&](auto bc) __attribute__((always_inline)) {
          if (step + decltype(bc)::value < nsteps) step_math(step + decltype(bc)::value, decltype(bc)::value, bc);
        });
    }
  } else {
    for (int step = 0; step < nsteps; ++step) {
#pragma unroll
      for (int i = 0; i < MT; ++i) dma_x(step + NB - 1, (step + NB - 1) % NB, i);
      meet(IC<(NB - 2) * MT>{});
    }
  }
  __builtin_amdgcn_s_setprio(0);
}

template <int MT, int CT>
__device__ __forceinline__ void gemm_block_wide(const QLinearArgs& a, uint16_t* smem, int bx, int slice, int bz) {
  constexpr int ROWS = MT * 32, KW = 8 / CT, RF = 2 * MT;
  static_assert(KW * CT == 8, "8 waves");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ct = wave % CT, kw = wave / CT;
  const int q = lane >> 4, nl = lane & 15;
  const int KT = a.K >> 6;
  const int per = a.kt_per_split;
  const int kb0 = slice * per;
  const int kb1 = (kb0 + per < KT) ? kb0 + per : KT;
  const int nsteps = (kb1 - kb0) / kWideTS;  // host: whole steps
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
  const int sv = (nb * KG * 32 + (lane & 31)) * 2;
  // slab transfer: MT loads per wave and step; load i moves rows 4 wave + 32 i .. + 3 (16 lanes each), lane l
  // delivering chunk (l % 16) ^ (row % 16) of the step to slot l % 16.  Rows past the end lie past the descriptor's: zeros.
  const int row_l = 4 * wave + (lane >> 4);
  const int xoff = row_l * a.ldx * 2 + (((lane & 15) ^ (row_l & 15)) * 16) + kb0 * 128;

  f32x4_t acc[2][RF];  // columns 0..15 and 16..31 of the tile
  wide_core<MT, KW, wide_bufs(MT)>(smem, rw, wv, rs, sv, gs, rx, [&](int i) { return xoff + i * 64 * a.ldx; }, kb0, nsteps, kw, tile_ok, acc);
  // Two k-parts of a tile swap halves of their accumulators (the slab is free once the surplus transfers, repeats of
  // the last step, have landed): the first finishes the first half of the rows, the second the other.
  constexpr int NR = RF / KW;  // row tiles of 16 this wave finishes
  if constexpr (KW == 2) {
    __builtin_amdgcn_s_waitcnt(0x0070);
    __syncthreads();
    f32x4_t* hb = reinterpret_cast<f32x4_t*>(smem) + (size_t)ct * RF * 2 * 64 + lane;  // [CT][2 parts][2][NR][64]
    if (tile_ok)
#pragma unroll
      for (int i = 0; i < RF; ++i) {
        f32x4_t(&v)[RF] = acc[i / NR];
        hb[(i + (kw ? 0 : RF)) * 64] = kw ? v[i % NR] : v[i % NR + NR];
      }
    __syncthreads();
    if (tile_ok)
#pragma unroll
      for (int i = 0; i < RF; ++i) {
        f32x4_t(&v)[RF] = acc[i / NR];
        const f32x4_t mine = kw ? v[i % NR + NR] : v[i % NR], other = hb[(i + (kw ? RF : 0)) * 64];
        v[i % NR] = kw ? other + mine : mine + other;  // first half + second half
      }
  }
  const int wrow0 = row0 + kw * NR * 16 + nl;  // this lane's row of the first row tile
  const int tile0 = nb * 32, col0 = tile0 + 4 * q;  // its four columns of the first half of the tile, + 16 of the second
  if (!a.t16) {
    if (tile_ok)
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int row = wrow0 + i * 16;
        if (row >= a.M) continue;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const f32x4_t v = acc[u][i];
          if (a.y_bf16) store8(a.y_bf16 + (size_t)row * a.ldy + col0 + 16 * u, u32x2_t{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])});
          else *reinterpret_cast<f32x4_t*>(a.y_part + ((size_t)slice * a.M + row) * a.N + col0 + 16 * u) = v;
        }
      }
    return;
  }
  // LoRA in the epilogue: delta tile [16 columns, 16 rows] = B columns . t16 rows, 32 ranks per MFMA (in the
  // orientation of acc); y = bf16(bf16(base) + bf16(bf16(delta) ls)).  What it costs is round trips to memory, so the
  // columns of B are requested in front of the wait for t, and the rows of t four row tiles ahead.
  auto lora = [&](auto nkbc) __attribute__((always_inline)) {
    constexpr int NKB = decltype(nkbc)::value, BT = 4, NBT = (NR + BT - 1) / BT;
    const int seg = tile0 >= a.seg_end[0] ? (tile0 >= a.seg_end[1] ? 2 : 1) : 0;
    uint16_t be[2][NKB][8];
#pragma unroll
    for (int i = 0; i < 2 * NKB * 8; ++i) {
      const int u = i / (8 * NKB), kb = i / 8 % NKB, rr = kb * 32 + 8 * q + i % 8;
      be[u][kb][i % 8] = tile_ok && rr < a.lora_r ? a.lora_b[(size_t)rr * a.N + tile0 + u * 16 + nl] : (uint16_t)0;
    }
    bool t_ready = true;
    if (a.sync) {
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
    u32x4_t bfr[2][NKB];
#pragma unroll
    for (int i = 0; i < 2 * NKB; ++i) __builtin_memcpy(&bfr[i / NKB][i % NKB], be[i / NKB][i % NKB], 16);
    const __amdgpu_buffer_rsrc_t rt = make_rsrc(a.t16, (uint32_t)a.M * a.ldt16 * 2u);
    u32x4_t tf[2][BT][NKB];
    auto load_t = [&](auto bc) __attribute__((always_inline)) {
      constexpr int bt = decltype(bc)::value;
#pragma unroll
      for (int i = 0; i < BT; ++i) {
        const int row = wrow0 + (bt * BT + i) * 16;
        const int tp = ((row < a.M ? row : a.M - 1) * a.ldt16 + seg * a.lora_r + 8 * q) * 2;
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) {
          // past this XCD's L2: the rows were written during this launch
          tf[bt & 1][i][kb] = u32x4_t{0u, 0u, 0u, 0u};
          if (bt * BT + i < NR && t_ready && kb * 32 + 8 * q < a.lora_r)
            tf[bt & 1][i][kb] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rt, tp + kb * 64, 0, 0x10));
        }
      }
    };
    load_t(IC<0>{});
    static_for<NBT>([&](auto bc) __attribute__((always_inline)) {
      constexpr int bt = decltype(bc)::value;
      if constexpr (bt + 1 < NBT) load_t(IC<bt + 1>{});
#pragma unroll
      for (int ii = 0; ii < BT; ++ii) {
        const int i = bt * BT + ii, row = wrow0 + i * 16;
        if (i >= NR) break;
        f32x4_t d[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          d[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kb = 0; kb < NKB; ++kb)
            d[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, bfr[u][kb]), __builtin_bit_cast(bf16x8_t, tf[bt & 1][ii][kb]), d[u], 0, 0, 0);
        }
        if (row >= a.M) continue;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          f32x4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = rbf(acc[u][i][e]) + rbf(rbf(d[u][e]) * a.lora_ls);
          store8(a.y_bf16 + (size_t)row * a.ldy + col0 + 16 * u, u32x2_t{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])});
        }
      }
    });
  };
  if (a.lora_r <= 32) lora(IC<1>{});
  else lora(IC<2>{});
}

__host__ __device__ inline int lora_col_waves(const QLinearArgs& a) { return a.Rpad > 64 ? 4 : a.Rpad >> 5; }

// t = x . A of one row tile (32 rows) over one K-slice (or a.lora_par short ones side by side).  The 8 waves are column tiles of
// A (1, 2 or 4) x k-parts; a wave
// reads its x fragments straight from global memory (32 rows, 64 bytes each per pair of loads; the column tiles of a
// k-part hit the same lines) two k-tiles ahead, the parts meet in LDS.  Every slice leaves its f32 plane; with a
// hand-over area (a.sync) the last slice of the row tile to arrive adds the planes in slice order and writes the
// rounded t: bf16 for the epilogues of this launch (a.t16, then its ready flag), f32 for a consumer behind it
// (a.t_fin).  Stores are write-through and loads go past L2 (sc1), so no cache write-back happens inside the
// launch.  In the projection's launch these workgroups come first in dispatch order and wait for nobody.  What bounds
// them is latency: about 8 us at 256 rows, hidden behind the main workgroups' loop, where a LoRA-only launch and a
// reduction launch in front of the projection took 14 + 5 us (decode step of 256 sequences, 8 layers: 3.43 -> 3.25 ms).
__device__ __forceinline__ void wide_lora_block(const QLinearArgs& a, float* red, int id) {
  const int PS = a.lora_par, RT = (a.M + 31) >> 5, rt = id % RT, ks0 = id / RT * PS;
  if (ks0 >= a.n_lora_slices) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, nl = lane & 31;
  const int KT = a.K >> 6, NT = a.Rpad >> 5, NP = lora_col_waves(a), nk = 8 / NP / PS;
  const int ct = wave % NP, kp = wave / NP % nk, ks = ks0 + wave / NP / nk;  // (a slice past the last one has no k-tiles)
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
  for (int e = tid; e < PS * 32 * quads; e += 512) {
    const int rs = e / quads, c = (e - rs * quads) * 4, rl = rs & 31, s = rs >> 5, row = rt * 32 + rl, sl = ks0 + s;
    if (row >= a.M || sl >= a.n_lora_slices) continue;
    const int r = (rl >> 3) * 4 + (rl & 3), ln = ((rl >> 2) & 1) * 32 + (c & 31);
    f32x4_t v = {0.f, 0.f, 0.f, 0.f};
    for (int p = s * nk; p < (s + 1) * nk; ++p) v += *reinterpret_cast<const f32x4_t*>(red + ((p * NP + (c >> 5)) * 16 + r) * 64 + ln);
    if (final_here && a.n_lora_slices == 1) finish(row, c, v);
    else if (!final_here) *reinterpret_cast<f32x4_t*>(a.t_part + ((size_t)sl * a.M + row) * a.ldt + c) = v;
    else __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), rp, (int)((((size_t)sl * a.M + row) * a.ldt + c) * 4), 0, 0x10);
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

// Workgroups of t = x . A, and how many slices each takes: as many as leave every wave a k-tile, where nothing is handed over (the
// f32 planes of a caller may have slices of 4 k-tiles: 844 x 4096 x 1024 with rank 32 in 432 workgroups of one slice 24.3 us, in 216 of two 16.9).
static int lora_workgroups(QLinearArgs& a) {
  a.lora_par = 1;
  if (!a.a_t) return 0;
  if (!a.sync)
    while (8 / lora_col_waves(a) / (2 * a.lora_par) >= a.kt_per_lora_split) a.lora_par *= 2;
  return ((a.M + 31) / 32 * ((a.n_lora_slices + a.lora_par - 1) / a.lora_par) + 7) / 8 * 8;
}

template <int MT, int CT>
static int launch_wide(hipStream_t st, QLinearArgs a) {
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&qlinear_mfma_wide_kernel<MT, CT>), hipFuncAttributeMaxDynamicSharedMemorySize,
      (int)wide_lds(MT));
  if (attr != hipSuccess) return TMX_ERR_LAUNCH;
  const int blocks = (a.N + CT * 32 - 1) / (CT * 32);
  a.lora_wgs = lora_workgroups(a);
  const int row_blocks = (a.M + MT * 32 - 1) / (MT * 32);
  int S = 8;
  while (row_blocks % S) S >>= 1;  // gcd(row_blocks, 8)
  // ids cover 8 / S XCDs x (row_blocks / S) row blocks x blocks x nsplit per residue, rounded up to 8
  const long total = (long)blocks * a.nsplit * row_blocks;
  const int ids = (int)((total + 7) / 8 * 8);
  hipLaunchKernelGGL((qlinear_mfma_wide_kernel<MT, CT>), dim3(a.lora_wgs + ids), dim3(512), wide_lds(MT), st, a, blocks, row_blocks, S);
  return check_launch();
}

// Routed experts with many rows (cache fill and scoring passes of a MoE model): workgroup = (column block, expert), up to 128
// of the expert's rows at a time through the many-rows product, gathered rows in and scattered rows out.  A wave has 32
// columns: a tile of down, or 16 hidden units of gate | up as 16 gate and the matching 16 up columns, so that both meet in
// a lane and SwiGLU needs no exchange.  Sums run over K in the order of moe_stream_kernel: the same bits.
// What bounds it at the 64 rows an expert has in a pass of 1024 tokens (128 experts of 2048 x 768, top-8) is the
// instructions of the dequantisation (32 us of issue) beside those of the MFMAs: 92 + 63 us per layer, in chunks of 32 rows that
// dequantised every matrix two to three times 194 + 145 us.  In this form (156 registers, one workgroup per CU): held to 128
// registers, two per CU, it spills and takes 121 us for gate | up; three or four slab buffers, 101 and 106; chunks
// of 64 rows 125 (an expert with 65 rows streams its matrices twice).  The list of rows is read in one go by every
// workgroup, consecutive pairs by consecutive lanes; 16 pairs per lane instead cost 23 us of down's 80.
constexpr int kMoeRows = 128;  // rows of a chunk
template <bool DOWN, int MT>
__device__ __forceinline__ void moe_chunk(const MoeArgs& m, int e, int bx, const uint16_t* rows_s, int n, uint16_t* smem) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 4, nl = lane & 15, h = lane >> 5, sub = q & 1;
  const int KT = m.K >> 6, KG = m.K / m.G, unit = bx * 8 + wave;
  const bool active = unit * 32 < m.N;
  // the tile and the 16 columns of it that this lane has words of; descriptors begin at the wave's first tile, so 32-bit
  // offsets reach an up tile of every matrix that moe_experts takes
  const int nb = DOWN ? unit : unit >> 1, up = DOWN ? 0 : sub * (m.N >> 6), half = DOWN ? sub : unit & 1;
  const int wv = (up * KT * 64 + 32 * h + 16 * half + nl) * 16, sv = (up * KG * 32 + 16 * half + nl) * 2;
  const uint32_t tiles = active ? (DOWN ? 1u : (uint32_t)(m.N >> 6) + 1u) : 0u;
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(m.qw + (size_t)e * m.qw_stride + (active ? (size_t)nb * KT * 64 : 0), tiles * KT * 1024u);
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(m.scales + (size_t)e * m.sc_stride + (active ? (size_t)nb * KG * 32 : 0), tiles * KG * 64u);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(m.x, (uint32_t)moe_x_bytes(m, DOWN));
  const int row_l = 4 * wave + q;
  int xoff[MT];  // rows past the end: past the descriptor's end, zeros
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int r = row_l + 32 * i, p = rows_s[r < n ? r : 0];
    xoff[i] = r < n ? (DOWN ? p : p / m.top_k) * m.ldx * 2 + ((nl ^ (row_l & 15)) * 16) : (int)kMoeRowsXBytes;
  }
  f32x4_t acc[2][2 * MT];
  wide_core<MT, 1, 2>(smem, rw, wv, rs, sv, __builtin_ctz(m.G >> 6), rx, [&](int i) { return xoff[i]; }, 0, m.K / (64 * kWideTS), 0,
                      active, acc);
  if (!active) return;
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i) {
    const int r = i * 16 + nl;
    if (r >= n) continue;
    uint16_t* out = m.out + (size_t)rows_s[r] * m.ldo + unit * (DOWN ? 32 : 16) + 4 * q;
    if constexpr (DOWN) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
        store8(out + 16 * u, u32x2_t{pack_bf2(acc[u][i][0], acc[u][i][1]), pack_bf2(acc[u][i][2], acc[u][i][3])});
    } else {
      float v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float g = rbf(acc[0][i][k]), up = rbf(acc[1][i][k]);
        v[k] = rbf(g * rbf(1.f / (1.f + expf(-g)))) * up;
      }
      store8(out, u32x2_t{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3])});
    }
  }
}

template <bool DOWN>
__global__ __launch_bounds__(512, 2) void moe_rows_kernel(MoeArgs m, int E, int blocks) {
  extern __shared__ __align__(16) uint16_t smem[];
  __shared__ uint16_t rows_s[TMX_MAX_MOE_PAIRS];
  __shared__ int n_s;
  // the column blocks of an expert on one XCD: its rows are fetched into one L2
  const int xcd = blockIdx.x & 7, idx = (int)blockIdx.x >> 3, e = idx / blocks * 8 + xcd, bx = idx % blocks, tid = threadIdx.x;
  if (e >= E) return;
  if (tid == 0) n_s = 0;
  __syncthreads();
  {  // { p : expert_of[p] == e }, in any order: the rows of a product do not meet
    constexpr int PT = TMX_MAX_MOE_PAIRS / 512;
    int ex[PT];
#pragma unroll
    for (int u = 0; u < PT; ++u) ex[u] = tid + 512 * u < m.P ? m.expert_of[tid + 512 * u] : -1;
#pragma unroll
    for (int u = 0; u < PT; ++u)
      if (ex[u] == e) rows_s[atomicAdd(&n_s, 1)] = (uint16_t)(tid + 512 * u);
  }
  __syncthreads();
  const int n = n_s;
  for (int c0 = 0; c0 < n; c0 += kMoeRows) {
    const int left = n - c0;
    if (left <= 32) moe_chunk<DOWN, 1>(m, e, bx, rows_s + c0, left, smem);
    else if (left <= 64) moe_chunk<DOWN, 2>(m, e, bx, rows_s + c0, left, smem);
    else if (left <= 96) moe_chunk<DOWN, 3>(m, e, bx, rows_s + c0, left, smem);
    else moe_chunk<DOWN, 4>(m, e, bx, rows_s + c0, left < kMoeRows ? left : kMoeRows, smem);
    __builtin_amdgcn_s_waitcnt(0x0070);  // the surplus transfers have landed before the slab is used again
    __syncthreads();
  }
}

template <bool DOWN>
static int launch_moe_rows(hipStream_t st, const MoeArgs& a, int E) {
  constexpr size_t lds = (size_t)2 * kMoeRows * kWideXS * 2;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_rows_kernel<DOWN>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (attr != hipSuccess) return TMX_ERR_LAUNCH;
  const int blocks = (a.N + 255) / 256;
  hipLaunchKernelGGL(moe_rows_kernel<DOWN>, dim3((E + 7) / 8 * 8 * blocks), dim3(512), lds, st, a, E, blocks);
  return check_launch();
}
int moe_rows(hipStream_t st, const MoeArgs& a, int E, bool down) {
  return down ? launch_moe_rows<true>(st, a, E) : launch_moe_rows<false>(st, a, E);
}

// Which tile and how many K-slices.  The slices, which callers make room for, follow prices of their own: a fixed part
// of 8 us and steps of 0.24 us + 0.05 us per column tile and row tile (by the prices below they would be fewer here and there, and
// nothing gained: 256 x 4096 x 6144 unsplit instead of in 2 slices 0.4 % of a decode step slower).  The tile follows what the kernel
// takes: a fixed part (first slab and weights from cold caches, exchange, stores) and a time per step, both linear in the tile;
// fitted to every tile and slice count of twelve matrices of the 8B, 1B, Qwen3-8B and 30B-A3B shapes at 13 row counts from 135 to
// 4096, they are 6 % off in the mean.  More workgroups than CUs run in rounds, whose steps are 1.12 times as long (the clock falls
// with every CU at work) and which hide half of the fixed part; two workgroups of up to 4 x 4 tiles share a CU and hide
// all of it.  K-slices cost their f32 planes, written here and read by the consumer.  At 256 rows of the 8B shape (us,
// without LoRA and without the consumer's read) q|k|v runs 4 x 4 tiles in 2 slices, 20.6 (8 x 4 in 4: 21.6 and
// twice the planes), gate|up 8 x 4 unsplit, 55 (4 x 4: 59, 8 x 8: 81), down 4 x 4 in 4, 33 (8 x 4 in 4: 43); 4096 rows of
// gate|up 8 x 8, 715 (4 x 4: 840); 3606 rows of it 8 x 8, 705 (7 x 4, which the prices of the slices would take, 789), 1024 rows
// 8 x 8, 200 (4 x 4: 226), 400 rows of 4096 x 24576 7 x 8, 82 (7 x 4: 99).
static const int kWideTiles[][2] = {{2, 4}, {3, 4}, {4, 4}, {5, 4}, {6, 4}, {7, 4}, {8, 4}, {4, 8}, {5, 8}, {6, 8}, {7, 8}, {8, 8}};

// The LoRA workgroups of a launch (1 us + 0.25 a k-tile each) come first: where they and the others make more rounds, the last of
// the others start behind them or share a CU.  Left out of the price, tiles that fill the chip by themselves were chosen: 630 x 2048 x
// 16384 with rank 16 in 5 x 8 tiles (256 + 24 workgroups) 54.7 us, in 7 x 8 (192 + 24) 51.0; 200 x 4096 x 2048 in 4 slices and 2 x 4
// tiles (256 + 16) 17.5, in 3 x 4 (192 + 16) 13.4.  Over 16 matrices at 15 row counts with adapters the choice is 0.5 % off the best
// tile in the mean, 13 % at most (4.9 and 31 % without this), without adapters 0.15 and 9 %.

// What a tile in s slices costs, us; `order`: by the prices that fix the slices.
static float wide_price(int M, int N, int KT, int mt, int ct, int s, int cus, int lora_wgs, float lora_us, bool order) {
  const long tiles = (long)((M + 32 * mt - 1) / (32 * mt)) * ((N + 32 * ct - 1) / (32 * ct));
  const long n = (tiles * s + cus - 1) / cus;  // workgroups of a CU
  const bool pairs = mt <= 4 && ct == 4;
  const float steps = (float)(slice_len(KT, s) / kWideTS), planes = s > 1 ? 0.3e-6f * s * (float)M * N * 4.f : 0.f;
  if (order) {
    const float loop = steps * (0.24f + 0.05f * mt * ct);
    return (pairs ? 8.f + (n == 1 ? 1.f : 0.92f) * n * loop : n * (8.f + loop)) + planes;
  }
  const float fixed = ct == 4 ? 3.7f + 0.78f * mt : 5.8f + 0.62f * mt, loop = steps * ((ct == 4 ? 0.4f : 0.56f) + 0.024f * mt * ct);
  auto rounds = [&](long k) { return pairs || k == 1 ? fixed + k * loop : fixed + 1.12f * k * loop + 0.5f * (k - 1) * fixed; };
  const long with = (tiles * s + lora_wgs + cus - 1) / cus;
  const float more = rounds(with), behind = rounds(n) + (with - n) * lora_us;
  return (more < behind ? more : behind) + planes;
}

WidePlan wide_plan(int M, int N, int K, int nsplit, int lora_wgs, int lora_kt) {
  const int cus = device_cus(), KT = K >> 6;
  WidePlan best = {8, 8, nsplit > 0 ? nsplit : 1};
  float best_cost = 1e30f;
  auto offer = [&](int mt, int ct, int s, bool order) {
    const float cost = wide_price(M, N, KT, mt, ct, s, cus, lora_wgs, 1.f + 0.25f * lora_kt, order);
    if (cost < best_cost) { best_cost = cost; best = {mt, ct, s}; }
  };
  for (const auto& t : kWideTiles)
    for (int s = nsplit > 0 ? nsplit : 1; s <= (nsplit > 0 ? nsplit : TMX_MAX_SPLITS); ++s)
      if (slices_ok(KT, s)) offer(t[0], t[1], s, true);
  const int s = best.nsplit;
  best_cost = 1e30f;
  for (const auto& t : kWideTiles) offer(t[0], t[1], s, false);
  return best;
}

// t in a launch of its own, ordered in front of the projection, for callers that have no word to ask whether a wait ran
// out (tmx_qlora_linear).  It costs the launch, 2 to 7 us: 300 x 4096 x 12288 with rank 16 takes 63 us against 57 with
// the LoRA workgroups inside, 4096 x 4096 x 28672 841 against 840.
int qwide_lora_launch(hipStream_t st, QLinearArgs a) {
  static_assert(wide_lds(2) >= 8 * 16 * 64 * 4, "the accumulators of the 8 waves meet in LDS");
  if (!a.a_t || !a.sync || a.M > TMX_MAX_FILL_ROWS) return TMX_ERR_ARG;
  a.lora_wgs = lora_workgroups(a);
  hipLaunchKernelGGL((qlinear_mfma_wide_kernel<2, 4>), dim3(a.lora_wgs), dim3(512), wide_lds(2), st, a, 1, 1, 1);
  return check_launch();
}

int qwide_launch(hipStream_t st, QLinearArgs a) {
  if (a.sync && a.M > TMX_MAX_FILL_ROWS) return TMX_ERR_SHAPE;  // the hand-over area has a word per row tile
  const WidePlan p = wide_plan(a.M, a.N, a.K, a.nsplit, lora_workgroups(a), a.kt_per_lora_split);
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
