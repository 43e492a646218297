// Final projection to the vocabulary fused with log-softmax statistics and token
// selection, so the [B, V] logits never travel through HBM.
//
// Replaces the tail of the model call and Sampler._sample:
//   logits = bf16(x . head) -> f32      tunix/models/llama3/model.py:688-697, :244-246
//                                       tunix/models/qwen3/model.py:1422-1442, :425-429
//   forbidden ids -> -inf               tunix/generate/sampler.py:536-537
//   greedy: argmax, first index on ties tunix/generate/sampler.py:158-168
//   top_p mode with top_p >= 1, no top_k: z = logits / T, token = categorical(
//     fold_in(seed, step), z), logprob = log_softmax(z)[token]
//                                       tunix/generate/sampler.py:112-134, :562
//   token / logprob scatter, done |= isin(token, eos)   tunix/generate/sampler.py:575-581
//
// categorical(key, z) = argmax(z + gumbel), gumbel from threefry2x32 bits over
// the linear index b * V + v (jax's partitionable bit generation).
//
// Mapping: the head matrix [V, D] (bf16, the tied embedding table or the
// transposed lm_head) is the A operand of v_mfma_f32_32x32x16_bf16, the hidden
// states the B operand, so a lane's accumulator registers are 16 vocabulary rows
// of ONE sequence: max / sum-exp / arg-best run down the registers without
// cross-lane traffic.  Workgroup partials are merged by a second tiny kernel.
#include "tmx_kernels.h"
#include "tmx_sampling.h"

namespace tmx {

template <int V>
struct HIC { static constexpr int value = V; };
// Up to here head_kernel spreads the values of a sequence row over the lanes.  Its epilogue is a chain of 16 values a lane however
// many rows there are, 20 threefry rounds and two logarithms each when sampling; spread out, half a value a lane and row, and a
// reduction.  us per launch with finalize, chain / spread: 1024 x 256 head, one row greedy 12.7 / 7.8, sampling 25.5 / 8.3, 9 rows
// 15.5 / 11.0, 16 rows 15.6 / 12.9; 128256 x 2048, one row sampling 104.6 / 91.8, 16 rows 99.7 / 97.5.  More rows would not fit the
// slabs' LDS.
constexpr int kHeadFewRows = 16;
constexpr int kHXStride = 72;  // bf16 elements per LDS row of the activation tile (64 + 8 pad)

// Scoring (tunix/rl/common.py:217-221, selective_log_softmax): a NaN logit counts as -1e9 and
// the others are clipped to [-1e9, 1e9] before the log-softmax, so the result is always finite.
__device__ __forceinline__ float score_clip(float z) {
  return z != z ? -1e9f : fminf(fmaxf(z, -1e9f), 1e9f);
}

// Running statistics of one sequence row: max and sum of exp over the vocabulary rows seen, best candidate by key.
struct RowStat {
  float mx = kNegBig, se = 0.f;
  Best best = {-INFINITY, -INFINITY, 0x7FFFFFFF};
};

// A vocabulary row of sequence row `row`: z, what the log-softmax runs over, and the key the best candidate is found by.
// In sampling with sort_keys the key is z, and sort_key the 16-bit key whose ascending order is the descending order of the logit
// (= of z, T > 0; -0 counts as +0): non-negative values count down from 0x7FFF, negative ones up from 0x8000.
struct HeadValue { float z, key; uint32_t sort_key; };
__device__ __forceinline__ HeadValue head_value(const HeadArgs& a, float acc, int v, int row, int target, uint32_t key0, uint32_t key1) {
  float logit = rbf(acc);
  if (a.logits_out) a.logits_out[(size_t)row * a.V + v] = logit;
  for (int f = 0; f < a.n_forbidden; ++f)
    if (a.forbidden[f] == v) logit = -INFINITY;
  HeadValue c = {logit, logit, 0u};
  if (a.mode == TMX_SAMPLE_SCORE) {
    // the "best" candidate is the given next token: its z is what the log-prob needs
    c.z = score_clip(rbf(logit / a.temperature));  // bf16 logits divided in place stay bf16 (rl/common.py:591-592)
    c.key = (v == target) ? 0.f : -INFINITY;
  } else if (a.mode == TMX_SAMPLE_TOP_P) {
    c.key = c.z = logit / a.temperature;
    if (a.sort_keys) {
      const uint32_t zb = __float_as_uint(logit + 0.0f) >> 16;
      c.sort_key = (zb & 0x8000u) ? zb : (~zb & 0x7FFFu);
    } else {
      uint32_t o0, o1;
      threefry2x32(key0, key1, 0u, (uint32_t)(a.row_off + row) * (uint32_t)a.V + (uint32_t)v, o0, o1);
      c.key = c.z + gumbel_from_bits(o0 ^ o1);
    }
  }
  return c;
}
// exp(z - mx) of a z that is at most mx (the infinite maximum itself counts once, as every maximum does)
__device__ __forceinline__ float head_exp(float z, float mx) { return z == mx ? 1.f : expf(z - mx); }

// Adds the 16 vocabulary rows of an accumulator tile (first row v0) to the statistics of sequence row `row`: their maximum
// first, so that a value takes one exponential and no branch (a running maximum takes both sides of one in most waves).
// 128256 x 4096, greedy / sampling: 64 rows 185.5 / 191.5 -> 183.7 / 189.0 us, 256 rows 331.6 / 397.6 -> 325.9 / 393.3.
__device__ __forceinline__ void head_tile_stats(const HeadArgs& a, const f32x16_t& acc, int v0, int row, int lane, int target,
                                                uint32_t key0, uint32_t key1, RowStat& st) {
  uint64_t packed = 0;
  float z[16], mx = st.mx;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int v = v0 + acc_row(r, lane);
    const HeadValue c = head_value(a, acc[r], v, row, target, key0, key1);
    if (a.sort_keys) {
      // registers 4 q .. 4 q + 3 hold four consecutive vocabulary rows: one 8-byte store
      packed |= (uint64_t)c.sort_key << (16 * (r & 3));
      if ((r & 3) == 3) {
        *reinterpret_cast<uint64_t*>(a.sort_keys + (size_t)row * a.V + v - 3) = packed;
        packed = 0;
      }
    }
    z[r] = c.z;
    mx = fmaxf(mx, c.z);
    Best b = {c.key, c.z, v};
    best_merge(st.best, b);
  }
  st.se *= head_exp(st.mx, mx);
  st.mx = mx;
#pragma unroll
  for (int r = 0; r < 16; ++r) st.se += head_exp(z[r], mx);
}

// Maximum / sum over the lanes of a half-wave, every lane gets it.
__device__ __forceinline__ float half_max(float v) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
  v = fmaxf(v, dpp_f<0x128>(v));  // row_ror:8
  v = fmaxf(v, dpp_f<0x124>(v));  // row_ror:4
  v = fmaxf(v, dpp_f<0x4E>(v));   // quad_perm [2,3,0,1]
  return fmaxf(v, dpp_f<0xB1>(v));  // quad_perm [1,0,3,2]
}
__device__ __forceinline__ float half_sum(float v) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  v += dpp_f<0x128>(v);
  v += dpp_f<0x124>(v);
  v += dpp_f<0x4E>(v);
  return v + dpp_f<0xB1>(v);
}

// The given next token of sequence row `row` of this launch (scoring), or -1.
__device__ __forceinline__ int head_target(const HeadArgs& a, int row) {
  if (a.mode != TMX_SAMPLE_SCORE || row >= a.M) return -1;
  const int2 at = score_row(a, a.row_base + row);
  return a.token_buffer[(size_t)at.x * a.buf_len + min(at.y + 1, a.buf_len - 1)];
}

// The other half-wave holds the other 16 vocabulary rows of the same sequence; one half stores the result.
__device__ __forceinline__ void head_stat_to_lds(RowStat st, int h, float* f, int* idx) {
  const float mx2 = __shfl_xor(st.mx, 32, 64), se2 = __shfl_xor(st.se, 32, 64);
  Best o = {__shfl_xor(st.best.key, 32, 64), __shfl_xor(st.best.z, 32, 64), __shfl_xor(st.best.idx, 32, 64)};
  lse_merge(st.mx, st.se, mx2, se2);
  best_merge(st.best, o);
  if (h == 0) {
    f[0] = st.mx; f[1] = st.se; f[2] = st.best.key; f[3] = st.best.z;
    *idx = st.best.idx;
  }
}

// Partials of this workgroup for row `row`: the `n` waves' statistics at f + 4 * stride * w, idx + stride * w.
__device__ __forceinline__ void head_store_partial(const HeadArgs& a, int row, int wg, const float* f, const int* idx, int n, int stride) {
  float mx = f[0], se = f[1];
  Best best = {f[2], f[3], idx[0]};
  for (int w = 1; w < n; ++w) {
    const float* g = f + (size_t)4 * stride * w;
    lse_merge(mx, se, g[0], g[1]);
    Best o = {g[2], g[3], idx[stride * w]};
    best_merge(best, o);
  }
  float* pf = a.part_f + ((size_t)row * a.nwg + wg) * 4;
  pf[0] = mx; pf[1] = se; pf[2] = best.key; pf[3] = best.z;
  a.part_i[(size_t)row * a.nwg + wg] = best.idx;
}

// Statistics of the rows of a tile when they are at most R: few sequence rows use few lanes of it, 16 vocabulary rows each, one
// after the other, so it is turned over in LDS (tile_s: 4 x 32 x (R + 1) floats), and the half-waves take a sequence row each and a
// lane one vocabulary row of it.  Every thread of the workgroup comes here.
template <int R, int ROWS>
__device__ __forceinline__ void head_few_stats(const HeadArgs& a, const f32x16_t& acc, float* tile_s, int wave, int lane, bool live,
                                               int v0, uint32_t key0, uint32_t key1, float (*s_f)[ROWS][4], int (*s_i)[ROWS]) {
  const int h = lane >> 5, nl = lane & 31;
  tile_s += wave * 32 * (R + 1);
  if (nl < R) {
#pragma unroll
    for (int r = 0; r < 16; ++r) tile_s[acc_row(r, lane) * (R + 1) + nl] = acc[r];
  }
  __syncthreads();
  for (int m0 = 0; m0 < a.M; m0 += 2) {
    const int row = m0 + h;
    RowStat st;
    if (live && row < a.M) {
      const int v = v0 + nl;
      const HeadValue c = head_value(a, tile_s[nl * (R + 1) + row], v, row, head_target(a, row), key0, key1);
      if (a.sort_keys) a.sort_keys[(size_t)row * a.V + v] = (uint16_t)c.sort_key;
      st.mx = fmaxf(st.mx, half_max(c.z));
      st.se = half_sum(head_exp(c.z, st.mx));
      const float key = half_max(c.key);
      const uint32_t ahead = (uint32_t)(__ballot(c.key == key) >> (h * 32));
      if (ahead) {  // (none: every key is NaN)
        const int first = __builtin_ctz(ahead);  // equal keys: the lowest vocabulary row
        st.best = {key, __shfl(c.z, h * 32 + first, 64), v0 + first};
      }
    }
    if (nl == 0 && row < a.M) {
      float* f = s_f[wave][row];
      f[0] = st.mx; f[1] = st.se; f[2] = st.best.key; f[3] = st.best.z;
      s_i[wave][row] = st.best.idx;
    }
  }
}

// Workgroup = 4 waves x 32 vocabulary rows.  The hidden-state k-tile x[0:M, 64 kb : 64 kb + 64]
// is fetched once per workgroup, double-buffered in LDS and shared by the waves (MFMA B
// fragments); head rows stream HBM -> registers through a ring of 4 k-tiles per wave.  Lane
// (row, h) reads the 64 contiguous bytes k = 32 h .. 32 h + 31 of its row, so a k-tile of a row
// is one 128-byte line split between two lanes; MFMA step t pairs them with x[.., 32 h + 8 t ..].
// TILED: the same 16-byte pieces from the tile copy of the matrix (head_tiles_kernel), where the
// piece of (k-tile, step t, lane) sits at ((k-tile * 4 + t) * 64 + lane) * 16 of its row tile:
// a wave's load is 1 KiB of consecutive bytes and its whole share of the matrix one contiguous
// stream, read once (non-temporal).  Row-major, one load touches 32 lines of 32 different DRAM
// pages; measured on the 1.05 GB head at 64 rows: 252 us row-major, 190 us from tiles.
template <int MT, bool TILED>
__global__ __launch_bounds__(256, 2) void head_kernel(HeadArgs a) {
  __shared__ __align__(16) uint16_t xs[2][MT * 32][kHXStride];
  __shared__ float s_f[4][MT * 32][4];
  __shared__ int s_i[4][MT * 32];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int h = lane >> 5, nl = lane & 31;
  const int tile = blockIdx.x * 4 + wave;
  const bool live = tile * 32 < a.V;
  const int v0 = live ? tile * 32 : a.V - 32;  // dead waves recompute the last tile (dropped)
  const int KT = a.D >> 6;

  f32x16_t acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[m][r] = 0.f;

  const u32x4_t* wsrc = TILED ? reinterpret_cast<const u32x4_t*>(a.w_tiles + (size_t)v0 * a.D) + lane
                              : reinterpret_cast<const u32x4_t*>(a.w + (size_t)(v0 + nl) * a.D + h * 32);
  const uint16_t* xsrc[MT];
  int xrow_l[MT], xcol_l[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int c = tid + 256 * i;
    xrow_l[i] = c >> 3;
    xcol_l[i] = (c & 7) * 8;
    const int row = xrow_l[i] < a.M ? xrow_l[i] : a.M - 1;
    xsrc[i] = a.x + (size_t)row * a.D + xcol_l[i];
  }
  constexpr int P = 4;
  u32x4_t wring[P][4];
  u32x4_t xring[P][MT];
  const int klast = KT - 1;
  auto load_w = [&](int kb, auto pc) __attribute__((always_inline)) {
    constexpr int p = decltype(pc)::value;
    kb = kb < klast ? kb : klast;
#pragma unroll
    for (int t = 0; t < 4; ++t)
      wring[p][t] = TILED ? __builtin_nontemporal_load(wsrc + (size_t)kb * 256 + t * 64) : wsrc[(size_t)kb * 8 + t];
  };
  auto load_x = [&](int kb, auto pc) __attribute__((always_inline)) {
    constexpr int p = decltype(pc)::value;
    kb = kb < klast ? kb : klast;
#pragma unroll
    for (int i = 0; i < MT; ++i) xring[p][i] = *reinterpret_cast<const u32x4_t*>(xsrc[i] + kb * 64);
  };
  auto stash_x = [&](int buf, auto pc) __attribute__((always_inline)) {
    constexpr int p = decltype(pc)::value;
#pragma unroll
    for (int i = 0; i < MT; ++i)
      *reinterpret_cast<u32x4_t*>(&xs[buf][xrow_l[i]][xcol_l[i]]) = xring[p][i];
  };
  auto tile_step = [&](int kb, auto pc) __attribute__((always_inline)) {
    constexpr int p = decltype(pc)::value;
    constexpr int p1 = (p + 1) % P;
    bf16x8_t xf[MT][4];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        xf[m][t] = *reinterpret_cast<const bf16x8_t*>(&xs[p & 1][m * 32 + nl][h * 32 + t * 8]);
    u32x4_t wc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) wc[t] = wring[p][t];
    load_w(kb + P, pc);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wc[t]), xf[m][t],
                                                         acc[m], 0, 0, 0);
    stash_x((p + 1) & 1, HIC<p1>{});
    load_x(kb + 1 + P, HIC<p1>{});
    __syncthreads();
  };
  load_x(0, HIC<0>{}); load_x(1, HIC<1>{}); load_x(2, HIC<2>{}); load_x(3, HIC<3>{});
  load_w(0, HIC<0>{}); load_w(1, HIC<1>{}); load_w(2, HIC<2>{}); load_w(3, HIC<3>{});
  stash_x(0, HIC<0>{});
  load_x(P, HIC<0>{});
  __syncthreads();
  const int ngroups = KT / P;
  for (int g = 0; g < ngroups; ++g) {
    const int kb = g * P;
    tile_step(kb + 0, HIC<0>{}); tile_step(kb + 1, HIC<1>{});
    tile_step(kb + 2, HIC<2>{}); tile_step(kb + 3, HIC<3>{});
  }
  {
    const int kb = ngroups * P, rem = KT - ngroups * P;
    if (rem > 0) tile_step(kb + 0, HIC<0>{});
    if (rem > 1) tile_step(kb + 1, HIC<1>{});
    if (rem > 2) tile_step(kb + 2, HIC<2>{});
  }

  // per-step key = fold_in(seed, step)
  uint32_t key0 = 0, key1 = 0;
  if (a.mode == TMX_SAMPLE_TOP_P) threefry2x32(a.k0, a.k1, 0u, (uint32_t)*a.step, key0, key1);
  if (MT == 1 && a.M <= kHeadFewRows) {
    static_assert(4 * 32 * (kHeadFewRows + 1) * 4 <= (int)sizeof(uint16_t) * 2 * 32 * kHXStride, "the tiles of the waves take the place of the slabs");
    head_few_stats<kHeadFewRows, MT * 32>(a, acc[0], reinterpret_cast<float*>(&xs[0][0][0]), wave, lane, live, v0, key0, key1, s_f, s_i);
  } else {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int row = m * 32 + nl;
      RowStat st;
      if (live && row < a.M) head_tile_stats(a, acc[m], v0, row, lane, head_target(a, row), key0, key1, st);
      head_stat_to_lds(st, h, s_f[wave][row], &s_i[wave][row]);
    }
  }
  __syncthreads();
  for (int row = threadIdx.x; row < MT * 32; row += 256)
    if (row < a.M) head_store_partial(a, row, blockIdx.x, s_f[0][row], &s_i[0][row], 4, MT * 32);
}

// The same for at most kHeadRows rows of at most kHeadRowD values: they fit LDS whole, [M][D + 8], so the matrix streams past them
// without a barrier, and the norm in front of the head is taken here, by every workgroup while its first tiles are on the way (the
// bits of row_norm_kernel: the squares of 8 values by a thread, 64 threads by a wave, the waves in order), instead of by a
// launch of its own.  Measured (back to back with finalize, without a norm, head_kernel / this; its launch of 3.5 to 4.7 us goes as
// well), one row and four rows, sampling: 128256 x 4096 167.6 / 160.6 and 168.6 / 162.7 us (6.5 TB/s), 128256 x 2048 92.4 / 88.1 and
// 93.9 / 89.6, 1024 x 256 8.1 / 7.8 and 9.2 / 9.1.
constexpr int kHeadRows = 4, kHeadRowD = 4096;
template <int R, bool TILED>  // M <= R
__global__ __launch_bounds__(256, 3) void head_row_kernel(HeadArgs a) {
  extern __shared__ __align__(16) uint16_t xs[];  // [M][D + 8]
  __shared__ float tile_s[4 * 32 * (R + 1)];
  __shared__ float s_ss[R][8];
  __shared__ float s_f[4][R][4];
  __shared__ int s_i[4][R];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, nl = lane & 31;
  const int tile = blockIdx.x * 4 + wave;
  const bool live = tile * 32 < a.V;
  const int v0 = live ? tile * 32 : a.V - 32;  // dead waves recompute the last tile (dropped)
  const int D = a.D, KT = D >> 6, klast = KT - 1, XS = D + 8;

  // the rows first: they are waited for first.  Loads of rows and columns that are not there fetch nothing.
  constexpr int kNowhere = 0x7FFF0000;
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x, (uint32_t)a.M * D * 2u), rn = make_rsrc(a.norm_w, a.norm_w ? (uint32_t)D * 2u : 0u);
  u32x4_t xq[R][2], nq[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int at = (tid + 256 * i) * 8 < D ? (tid + 256 * i) * 16 : kNowhere;
#pragma unroll
    for (int m = 0; m < R; ++m)
      xq[m][i] = __builtin_amdgcn_raw_buffer_load_b128(rx, at == kNowhere ? at : m * D * 2 + at, 0, 0);
    nq[i] = __builtin_amdgcn_raw_buffer_load_b128(rn, at, 0, 0);
  }
  constexpr int P = 4;
  u32x4_t wring[P][4];
  const u32x4_t* wsrc = TILED ? reinterpret_cast<const u32x4_t*>(a.w_tiles + (size_t)v0 * D) + lane
                              : reinterpret_cast<const u32x4_t*>(a.w + (size_t)(v0 + nl) * D + h * 32);
  auto load_w = [&](int kb, auto pc, auto tc) __attribute__((always_inline)) {
    constexpr int p = decltype(pc)::value, t = decltype(tc)::value;
    kb = kb < klast ? kb : klast;
    wring[p][t] = TILED ? __builtin_nontemporal_load(wsrc + (size_t)kb * 256 + t * 64) : wsrc[(size_t)kb * 8 + t];
  };
  __builtin_amdgcn_sched_barrier(0);
  static_for<P>([&](auto pc) __attribute__((always_inline)) {
    static_for<4>([&](auto tc) __attribute__((always_inline)) { load_w(decltype(pc)::value, pc, tc); });
  });
  __builtin_amdgcn_sched_barrier(0);
  auto unpack = [](const u32x4_t& q, float (&v)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) { v[2 * e] = bf_lo(q[e]); v[2 * e + 1] = bf_hi(q[e]); }
  };
  auto put = [&](int m, int i, u32x4_t q) __attribute__((always_inline)) {
    if ((tid + 256 * i) * 8 < D) *reinterpret_cast<u32x4_t*>(xs + m * XS + (tid + 256 * i) * 8) = q;
  };
  if (a.norm_w) {
#pragma unroll
    for (int m = 0; m < R; ++m)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float ss = 0.f;
        if (m < a.M && wave * 512 + i * 2048 < D) {  // (the whole wave or none of it)
          float v[8];
          unpack(xq[m][i], v);
#pragma unroll
          for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
          ss = wave_sum(ss);
        }
        if (lane == 0) s_ss[m][wave + 4 * i] = ss;
      }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < R; ++m) {
      float t = 0.f;
#pragma unroll
      for (int w = 0; w < 8; ++w) t += s_ss[m][w];
      const float rms = sqrtf(t / (float)D + a.eps);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (m < a.M && wave * 512 + i * 2048 < D) {
          float v[8], w[8], o[8];
          unpack(xq[m][i], v);
          unpack(nq[i], w);
          __builtin_amdgcn_sched_barrier(0);  // (one piece at a time: side by side their divisions take 50 registers)
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = a.family == TMX_FAMILY_LLAMA3 ? rbf(w[e] * v[e]) / rms : w[e] * (v[e] / rms);
          put(m, i, u32x4_t{pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3]), pack_bf2(o[4], o[5]), pack_bf2(o[6], o[7])});
        }
    }
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int m = 0; m < R; ++m)
        if (m < a.M) put(m, i, xq[m][i]);
  }
  __syncthreads();

  f32x16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  const uint16_t* xb = xs + min(nl, a.M - 1) * XS + h * 32;  // lanes past the rows repeat the last one (dropped)
  auto step = [&](int kb, auto pc) __attribute__((always_inline)) {
    constexpr int p = decltype(pc)::value;
    static_for<4>([&](auto tc) __attribute__((always_inline)) {
      constexpr int t = decltype(tc)::value;
      const bf16x8_t xf = *reinterpret_cast<const bf16x8_t*>(xb + kb * 64 + t * 8);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wring[p][t]), xf, acc, 0, 0, 0);
      load_w(kb + P, pc, tc);  // consumed: refill
    });
    __builtin_amdgcn_sched_barrier(0);
  };
  int kb = 0;
  for (; kb + P <= KT; kb += P)
    static_for<P>([&](auto pc) __attribute__((always_inline)) { step(kb + decltype(pc)::value, pc); });
  static_for<P - 1>([&](auto pc) __attribute__((always_inline)) {
    if (kb + decltype(pc)::value < KT) step(kb + decltype(pc)::value, pc);
  });

  uint32_t key0 = 0, key1 = 0;
  if (a.mode == TMX_SAMPLE_TOP_P) threefry2x32(a.k0, a.k1, 0u, (uint32_t)*a.step, key0, key1);
  head_few_stats<R, R>(a, acc, tile_s, wave, lane, live, v0, key0, key1, s_f, s_i);
  __syncthreads();
  if (tid < a.M) head_store_partial(a, tid, blockIdx.x, s_f[0][tid], &s_i[0][tid], 4, R);
}
bool head_row_ok(int M, int D) { return M <= kHeadRows && D <= kHeadRowD; }

// 65 to 256 rows: the matrix still has to stream once, but a wave multiplies up to 256 sequence rows (MT = 4 or 8 tiles),
// so the hidden states go to LDS by direct transfers (no registers) and the weights, from the tile copy, straight to
// registers as MFMA A operands, P steps ahead.  NW waves of 32 vocabulary rows each; slabs of 64 columns in 64 KiB of LDS:
// rows of 128 bytes, 16-byte chunk c of row r at slot c ^ (r / 2 % 8), which spreads a fragment read over all banks.
// Two workgroups share a CU, so that one's epilogue (20 threefry rounds a value when sampling) runs under the other's
// loads.  On the 1.05 GB head, greedy / sampling (trace): 96 rows 196 / 221 us, 128 rows 214 / 245, bound by the stream (64
// rows: 182 / 187); 160 rows 277 / 321, 256 rows 309 / 383, bound by LDS (a fragment read per MFMA) and, sampling, by the
// epilogue's VALU work.  The 256 x 256 blocks of head_wide_kernel take 266 / 369, 277 / 387 (160 rows) and 287 / 414 (256).
// For 256 rows also measured, where this form took 327 / 396: two waves of 64 vocabulary rows on each 128 rows (half the
// LDS reads, every weight read twice) 351 / 418; one workgroup of 8 waves per CU 316 / 412.
template <int MT, int NW, int P>
__global__ __launch_bounds__(NW * 64, NW == 4 ? 2 : 1) void head_mid_kernel(HeadArgs a) {
  constexpr int ROWS = MT * 32, R = 512 / ROWS, DX = ROWS / (8 * NW);
  static_assert(P % R == 0 && NW % 4 == 0, "a ring turn covers whole turns of the slabs; 128 vocabulary rows per partial");
  extern __shared__ __align__(16) uint16_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, nl = lane & 31;
  const int KT = a.D >> 6, klast = KT - 1, vtiles = a.V >> 5;
  const int tile = blockIdx.x * NW + wave;
  const bool live = tile < vtiles;  // waves past the end repeat the last tile (dropped)
  const int v0 = (live ? tile : vtiles - 1) * 32;
  const u32x4_t* wsrc = reinterpret_cast<const u32x4_t*>(a.w_tiles + (size_t)v0 * a.D) + lane;
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x, (uint32_t)a.M * a.D * 2u);
  int xoff[DX];  // transfer i of a wave: rows 8 (wave + NW i) .. + 7, 8 lanes each
#pragma unroll
  for (int i = 0; i < DX; ++i) {
    const int r = 8 * (wave + NW * i) + (lane >> 3);
    xoff[i] = (r < a.M ? r : a.M - 1) * a.D * 2 + (((lane & 7) ^ ((r >> 1) & 7)) * 16);
  }
  f32x16_t acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[m][r] = 0.f;
  u32x4_t wring[P][4];

  auto load_w = [&](int kb, auto pc, auto tc) __attribute__((always_inline)) {
    constexpr int p = decltype(pc)::value, t = decltype(tc)::value;
    kb = kb < klast ? kb : klast;
    wring[p][t] = __builtin_nontemporal_load(wsrc + (size_t)kb * 256 + t * 64);
  };
  auto dma_x = [&](int kb, int buf) __attribute__((always_inline)) {
    kb = kb < klast ? kb : klast;
    uint16_t* base = smem + (size_t)buf * ROWS * 64 + wave * 512;
#pragma unroll
    for (int i = 0; i < DX; ++i) load_row_to_lds(rx, base + i * (NW * 512), xoff[i], kb * 128);
  };
  // in-order counter: waiting for the slab of the next step leaves its step's weights and R - 2 whole steps outstanding
  constexpr int kYounger = 4 + (R - 2) * (DX + 4);
  auto step = [&](int kb, auto pc) __attribute__((always_inline)) {
    constexpr int p = decltype(pc)::value;
    dma_x(kb + R - 1, (p + R - 1) % R);
    __builtin_amdgcn_sched_barrier(0);
    const uint16_t* xb = smem + (size_t)(p % R) * ROWS * 64 + nl * 64;
    static_for<4>([&](auto tc) __attribute__((always_inline)) {
      constexpr int t = decltype(tc)::value;
      const int slot = ((4 * h + t) ^ ((nl >> 1) & 7)) * 8;
      bf16x8_t xf[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) xf[m] = *reinterpret_cast<const bf16x8_t*>(xb + m * 32 * 64 + slot);
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wring[p][t]), xf[m], acc[m], 0, 0, 0);
      load_w(kb + P, pc, tc);  // consumed: refill
    });
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70 | (kYounger & 15) | ((kYounger >> 4) << 14));
    __syncthreads();
  };
  static_for<P>([&](auto pc) __attribute__((always_inline)) {
    static_for<4>([&](auto tc) __attribute__((always_inline)) { load_w(decltype(pc)::value, pc, tc); });
  });
#pragma unroll
  for (int r = 0; r < R - 1; ++r) dma_x(r, r);
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  int kb = 0;
  for (; kb + P <= KT; kb += P)
    static_for<P>([&](auto pc) __attribute__((always_inline)) { step(kb + decltype(pc)::value, pc); });
  static_for<P - 1>([&](auto pc) __attribute__((always_inline)) {
    if (kb + decltype(pc)::value < KT) step(kb + decltype(pc)::value, pc);
  });
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the surplus transfers of the last steps have landed, the slabs are free
  __syncthreads();
  uint32_t key0 = 0, key1 = 0;
  if (a.mode == TMX_SAMPLE_TOP_P) threefry2x32(a.k0, a.k1, 0u, (uint32_t)*a.step, key0, key1);
  float* s_f = reinterpret_cast<float*>(smem);             // [NW][ROWS][4]
  int* s_i = reinterpret_cast<int*>(s_f + NW * ROWS * 4);  // [NW][ROWS]
  // One copy of the epilogue's code for all tiles (unrolled over them it would not fit the instruction cache): a
  // wave-uniform index picks the accumulators.
#pragma unroll 1
  for (int m = 0; m < MT; ++m) {
    const int row = m * 32 + nl;
    RowStat st;
    f32x16_t cur = acc[0];
    static_for<MT>([&](auto qc) __attribute__((always_inline)) {
      if (m == decltype(qc)::value) cur = acc[decltype(qc)::value];
    });
    if (live && row < a.M) head_tile_stats(a, cur, v0, row, lane, head_target(a, row), key0, key1, st);
    head_stat_to_lds(st, h, s_f + (wave * ROWS + row) * 4, s_i + wave * ROWS + row);
  }
  __syncthreads();
  for (int e = tid; e < NW / 4 * ROWS; e += NW * 64) {  // a partial per four waves
    const int row = e % ROWS, q = e / ROWS, wg = blockIdx.x * (NW / 4) + q;
    if (row < a.M && wg < a.nwg) head_store_partial(a, row, wg, s_f + (q * 4 * ROWS + row) * 4, s_i + q * 4 * ROWS + row, 4, ROWS);
  }
}

constexpr size_t kHeadMidLds = 65536;

template <int MT, int NW, int P>
static int launch_head_mid(hipStream_t st, const HeadArgs& a) {
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&head_mid_kernel<MT, NW, P>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kHeadMidLds);
  if (attr != hipSuccess) return TMX_ERR_LAUNCH;
  hipLaunchKernelGGL((head_mid_kernel<MT, NW, P>), dim3((a.nwg + NW / 4 - 1) / (NW / 4)), dim3(NW * 64), kHeadMidLds, st, a);
  return TMX_OK;
}

// The tile copy of the head matrix: row tile vt (32 vocabulary rows) x k-tile kt (64 columns) is 4 KiB at
// (vt * D / 64 + kt) * 4 KiB, and in it the 16 bytes W[32 vt + nl][64 kt + 32 h + 8 t .. + 7] sit at
// (t * 64 + 32 h + nl) * 16: what lane (nl, h) of head_kernel feeds to MFMA step t.  One workgroup per tile.
__global__ __launch_bounds__(256) void head_tiles_kernel(const uint16_t* __restrict__ w, uint16_t* __restrict__ tiles,
                                                         int D) {
  const int kt = blockIdx.x, vt = blockIdx.y, KT = D >> 6;
  const int t = threadIdx.x >> 6, lane = threadIdx.x & 63, h = lane >> 5, nl = lane & 31;
  const u32x4_t v = *reinterpret_cast<const u32x4_t*>(w + (size_t)(32 * vt + nl) * D + 64 * kt + 32 * h + 8 * t);
  reinterpret_cast<u32x4_t*>(tiles)[((size_t)vt * KT + kt) * 256 + t * 64 + lane] = v;
}

int head_tiles_pack(hipStream_t st, const uint16_t* w, uint16_t* tiles, int V, int D) {
  if (V <= 0 || D <= 0 || V % 32 || D % 64 || V / 32 > 65535) return TMX_ERR_SHAPE;
  hipLaunchKernelGGL(head_tiles_kernel, dim3(D / 64, V / 32), dim3(256), 0, st, w, tiles, D);
  return check_launch();
}

// The last workgroup of a launch to come here moves the step on (a launch of its own costs 1 to 4.6 us): all the others have
// read it.  One thread per workgroup; the counter is left at zero.
__device__ __forceinline__ void finalize_advance(const HeadArgs& a, int step) {
  if (!a.advance) return;
  if (gridDim.x > 1) {
    asm volatile("" ::"s"(step) : "memory");
    __builtin_amdgcn_s_waitcnt(0);
    if (__hip_atomic_fetch_add(a.arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != gridDim.x - 1) return;
    __hip_atomic_store(a.arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  *a.advance = step + (a.tpp > 0 ? a.tpp : 1);
}

// One workgroup per sequence: merge the vocabulary-tile partials, emit the token
// and its log-probability into column step + 1, update `done`.
__global__ __launch_bounds__(256) void head_finalize_kernel(HeadArgs a) {
  __shared__ float s_f[4][4];
  __shared__ int s_i[4];
  const int row = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float mx = kNegBig, se = 0.f;
  Best best = {-INFINITY, -INFINITY, 0x7FFFFFFF};
  for (int i = threadIdx.x; i < a.nwg; i += 256) {
    const float* pf = a.part_f + ((size_t)row * a.nwg + i) * 4;
    lse_merge(mx, se, pf[0], pf[1]);
    Best o = {pf[2], pf[3], a.part_i[(size_t)row * a.nwg + i]};
    best_merge(best, o);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float mx2 = __shfl_xor(mx, off, 64), se2 = __shfl_xor(se, off, 64);
    Best o = {__shfl_xor(best.key, off, 64), __shfl_xor(best.z, off, 64), __shfl_xor(best.idx, off, 64)};
    lse_merge(mx, se, mx2, se2);
    best_merge(best, o);
  }
  if (lane == 0) {
    s_f[wave][0] = mx; s_f[wave][1] = se; s_f[wave][2] = best.key; s_f[wave][3] = best.z;
    s_i[wave] = best.idx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    mx = s_f[0][0]; se = s_f[0][1];
    best = {s_f[0][2], s_f[0][3], s_i[0]};
    for (int w = 1; w < 4; ++w) {
      lse_merge(mx, se, s_f[w][0], s_f[w][1]);
      Best o = {s_f[w][2], s_f[w][3], s_i[w]};
      best_merge(best, o);
    }
    if (a.mode == TMX_SAMPLE_SCORE) {  // teacher forcing: the token stays, only its log-prob is written
      const int2 at = score_row(a, a.row_base + row);
      // selective_log_softmax: logit - logsumexp, with logsumexp = max + log(sum exp(z - max))
      const int step = *a.step, scol = at.y + 1;
      if (a.logprobs && scol < a.buf_len) a.logprobs[(size_t)at.x * a.buf_len + scol] = best.z - (mx + logf(se));
      finalize_advance(a, step);
      return;
    }
    const int step = *a.step, col = step + 1;
    finalize_advance(a, step);
    if (col >= a.buf_len) return;  // a caller that steps past the buffer gets no write instead of a stray one
    const int tok = best.idx;
    a.token_buffer[(size_t)row * a.buf_len + col] = tok;
    if (a.logprobs) a.logprobs[(size_t)row * a.buf_len + col] = (best.z - mx) - logf(se);
    bool hit = false;
    for (int e = 0; e < a.n_eos; ++e) hit = hit || (a.eos[e] == tok);
    if (hit) a.done[row] = 1;
  }
}

// ---------------------------------------------------------------------------
// Many rows (scoring passes over whole sequences, decode steps of more than 128 sequences): the same
// product as a matrix-pipe-bound kernel.  A workgroup multiplies 256 vocabulary rows by 256 sequence rows:
// the vocabulary rows are the A operand and come through four LDS slabs filled by
// direct-to-LDS loads (128-byte rows of 64 k, 16-byte chunk c of row r at slot c ^ (r / 2 % 8));
// wave w owns sequence rows 32 w .. 32 w + 31 as the B operand, read straight from global
// memory (lane (row, h) holds k = 32 h .. 32 h + 31 of a k-tile of 64, MFMA step t pairs k = 32 h + 8 t ..
// with the same k of the vocabulary rows), from a copy of the rows in fragment order.  A lane's
// 128 accumulator registers are 128 vocabulary rows of ONE sequence row, so max / sum-exp / the
// target's z run down the registers.  LDS reads of fragment group g + 1 and the refill of the
// B registers are pinned between the MFMAs of group g.  The matrix comes from HBM, so its slabs are short (64 k) and
// requested three ahead; the barrier that hands one over stands inside the last group of the one before, whose fragments
// are in registers, and the wave that is behind goes first (see wide_core in qwide.hip).  Consecutive workgroups take the
// sequence-row blocks of one vocabulary block, so the head matrix leaves HBM once.
// Bound by the matrix pipe and, a tenth of the time, by the epilogue, which nothing runs beside.  Scoring, 4096 rows of the
// 1.05 GB head: 4.67 ms with the rows read in place and two slabs of 128 k, 3.86 ms + 0.01 for the copy (1.11 PF/s); 630 rows
// of the 0.53 GB head 592 -> 501 us.  The four slabs without the copy took 5.0 ms (the address unit, see below), without
// wave priorities 5.2.  Taking the maximum of the accumulators first, then one exponential a value: 3.88 ms, nothing gained.
struct HW {
  static constexpr int MT = 8, ROWS = 256, XS = 64, NB = 4;
  static constexpr size_t LDS = (size_t)NB * ROWS * XS * 2;  // 128 KiB
};

// The rows of x in the order the wide kernel's B fragments take them: 32 rows x 16 k are 1 KiB, lane (row, h) of fragment
// 4 j + t of a step holds k = 64 j + 32 h + 8 t .. + 7.  Read from the rows themselves neighbouring lanes are in different
// rows, and the CU's address unit takes one of them at a time: 64 clocks a fragment, as much as the products of a step.
__global__ __launch_bounds__(512) void head_x_tiles_kernel(const uint16_t* x, uint16_t* tiles, int M, int D) {
  const int row = threadIdx.x >> 4, c = threadIdx.x & 15;  // 16 bytes of a row: k = 8 c of step blockIdx.x
  const u32x4_t v = *reinterpret_cast<const u32x4_t*>(x + (size_t)min((int)blockIdx.y * 32 + row, M - 1) * D + blockIdx.x * 128 + c * 8);
  const int g = (c >> 3) * 4 + (c & 3), h = (c >> 2) & 1;
  reinterpret_cast<u32x4_t*>(tiles)[((size_t)blockIdx.y * (D >> 4) + blockIdx.x * 8 + g) * 64 + 32 * h + row] = v;
}

template <int MODE>  // TMX_SAMPLE_*: the epilogue is compiled per mode
__global__ __launch_bounds__(512, 1) void head_wide_kernel(HeadArgs a, int tok_blocks, int voc_blocks) {
  extern __shared__ __align__(16) uint16_t smem[];
  constexpr int MT = HW::MT, XS = HW::XS, ROWS = HW::ROWS, NB = HW::NB;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, nl = lane & 31;
  const int vb = (int)blockIdx.x / tok_blocks, tb = (int)blockIdx.x % tok_blocks;
  if (vb >= voc_blocks) return;
  const int v0 = vb * ROWS;
  const int vrows = a.V - v0 < ROWS ? a.V - v0 : ROWS;
  const int tok = tb * 256 + wave * 32 + nl;       // sequence row of this lane's accumulator column
  const int tok_l = tok < a.M ? tok : a.M - 1;
  const int nsteps = a.D >> 7, last_step = nsteps - 1;  // steps of two slabs

  const __amdgpu_buffer_rsrc_t rw = make_rsrc(a.w + (size_t)v0 * a.D, (uint32_t)vrows * a.D * 2u);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x_tiles, (uint32_t)(a.M + 31) / 32 * 32 * a.D * 2u);
  constexpr int XR = ROWS / 64;
  int woff[XR];  // slab transfer: load i moves vocabulary rows 8 wave + 64 i .. + 7, 8 lanes each
#pragma unroll
  for (int i = 0; i < XR; ++i) {
    const int row_l = 8 * wave + 64 * i + (lane >> 3);
    woff[i] = (row_l < vrows ? row_l : vrows - 1) * a.D * 2 + (((lane & 7) ^ ((row_l >> 1) & 7)) * 16);
  }
  const int xv = (tb * 8 + wave) * (a.D >> 4) * 1024 + lane * 16;  // B fragments: 1 KiB each

  f32x16_t acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[m][r] = 0.f;
  constexpr int G = 8;  // fragment groups of a step, 16 k each
  u32x4_t breg[G];      // B fragments of a step, refilled for the next one after use

  auto load_b = [&](int step, auto gc) __attribute__((always_inline)) {
    constexpr int g = decltype(gc)::value;
    step = step < last_step ? step : last_step;
    breg[g] = __builtin_amdgcn_raw_buffer_load_b128(rx, xv, (step * G + g) * 1024, 0);
  };
  auto dma_w = [&](int slab, int i) __attribute__((always_inline)) {
    uint16_t* base = smem + (size_t)(slab & (NB - 1)) * ROWS * XS + wave * 8 * XS;
    load_row_to_lds_nt(rw, base + i * 64 * XS, woff[i], min(slab, 2 * nsteps - 1) * 128);
  };
  // all but the youngest loads of this wave have arrived and its LDS reads are done; then all waves
  auto meet = [&](auto younger) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(decltype(younger)::value) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int MEET = 2;  // the MFMA of a slab's last group in front of which the waves meet
  // younger than a slab when the next one is handed over: the B fragments behind its transfer (4), a slab and its B
  // fragments (XR + 4), and of the current one the transfer and three B fragments
  constexpr int kYounger = 4 + XR + 4 + XR + 3;
  bf16x8_t wq[2][MT];
  const uint16_t* wlane = smem + nl * XS;
  // group g = 4 j + t needs k = 64 j + 32 h + 8 t ..: chunk 4 h + t of slab j's row, at that slot ^ (row / 2 % 8)
  auto slot_of = [&](int g) __attribute__((always_inline)) { return ((4 * h + (g & 3)) ^ ((nl >> 1) & 7)) * 8; };
  auto step_math = [&](int step) __attribute__((always_inline)) {
    static_for<G>([&](auto gc) __attribute__((always_inline)) {
      constexpr int g = decltype(gc)::value, cur = g & 1, nxt = cur ^ 1;
      constexpr bool last = g % 4 == 3;
      const int slab = 2 * step + g / 4;
      const uint16_t* wb = wlane + (size_t)((last ? slab + 1 : slab) & (NB - 1)) * ROWS * XS + slot_of(g + 1);
      const bf16x8_t b = __builtin_bit_cast(bf16x8_t, breg[g]);
      __builtin_amdgcn_s_setprio(3 - g % 4);
      static_for<MT>([&](auto mc) __attribute__((always_inline)) {
        constexpr int m = decltype(mc)::value;
        if constexpr (last && m == MEET) meet(IC<kYounger>{});
        acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wq[cur][m], b, acc[m], 0, 0, 0);
        if constexpr (!last) {
          wq[nxt][m] = *reinterpret_cast<const bf16x8_t*>(wb + m * 32 * XS);
        } else if constexpr (m >= MEET) {  // two at a time until the two left out in front of the barrier are caught up
          constexpr int n = m - MEET, t0 = n < 2 ? 2 * n : n + 2, t1 = n < 1 ? 2 : n + 3;
          static_for<t1 - t0>([&](auto nc) __attribute__((always_inline)) {
            constexpr int r = t0 + decltype(nc)::value;
            wq[nxt][r] = *reinterpret_cast<const bf16x8_t*>(wb + r * 32 * XS);
          });
        }
        if constexpr (g % 4 == 0 && m % 2 == 0 && m / 2 < XR) dma_w(slab + NB - 1, m / 2);
        __builtin_amdgcn_sched_barrier(0);
      });
      load_b(step + 1, gc);  // fragment consumed: refill it for the next step
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  // (in this order, which the counts of the waits assume)
#pragma unroll
  for (int i = 0; i < (NB - 1) * XR; ++i) {
    dma_w(i / XR, i % XR);
    if (i % XR == XR - 1) __builtin_amdgcn_sched_barrier(0);
  }
  static_for<G>([&](auto gc) __attribute__((always_inline)) { load_b(0, gc); });
  meet(IC<(NB - 2) * XR + G>{});
#pragma unroll
  for (int m = 0; m < MT; ++m) wq[0][m] = *reinterpret_cast<const bf16x8_t*>(wlane + slot_of(0) + m * 32 * XS);
  for (int step = 0; step < nsteps; ++step) step_math(step);
  __builtin_amdgcn_s_setprio(0);

  // per sequence row: running max and sum of exp over this block's vocabulary rows and the best
  // candidate by key, as in head_kernel: greedy key = logit; sampling key = z + Gumbel noise of the
  // counter row * V + v; scoring: the given next token (key 0 marks it)
  constexpr bool score = MODE == TMX_SAMPLE_SCORE, sampling = MODE == TMX_SAMPLE_TOP_P;
  uint32_t key0 = 0, key1 = 0;
  if (sampling) threefry2x32(a.k0, a.k1, 0u, (uint32_t)*a.step, key0, key1);
  const int2 at = score ? score_row(a, tok_l) : make_int2(0, 0);
  const int target = score ? a.token_buffer[(size_t)at.x * a.buf_len + min(at.y + 1, a.buf_len - 1)] : -1;
  float mx = kNegBig, se = 0.f;
  Best best = {-INFINITY, -INFINITY, 0x7FFFFFFF};
  uint64_t packed = 0;  // sorting branch: the 16-bit keys of four consecutive vocabulary rows
  const bool keys_out = sampling && a.sort_keys != nullptr && tok < a.M;
  // (unrolled by construction: a loop the compiler declines to unroll would index the accumulators
  // dynamically and move them to scratch memory)
  static_for<MT * 16>([&](auto ic) __attribute__((always_inline)) {
      constexpr int m = decltype(ic)::value / 16, r = decltype(ic)::value % 16;
      const int v = v0 + m * 32 + acc_row(r, lane);
      if (v >= a.V) return;  // (V % 32 == 0 where keys are written: a group of four rows is in or out as one)
      const float logit = rbf(acc[m][r]);
      float z = logit, key = logit;
      if (score) {
        z = score_clip(rbf(logit / a.temperature));  // bf16 logits divided in place stay bf16 (rl/common.py:591-592)
        key = (v == target) ? 0.f : -INFINITY;
      } else if (sampling) {
        z = logit / a.temperature;
        if (a.sort_keys) {
          // the same 16-bit descending key as head_kernel writes (selection happens in nucleus.hip)
          if (keys_out) {
            const uint32_t zb = __float_as_uint(logit + 0.0f) >> 16;
            packed |= (uint64_t)((zb & 0x8000u) ? zb : (~zb & 0x7FFFu)) << (16 * (r & 3));
            if constexpr ((r & 3) == 3) {
              *reinterpret_cast<uint64_t*>(a.sort_keys + (size_t)tok * a.V + v - 3) = packed;
              packed = 0;
            }
          }
          key = z;
        } else {
          uint32_t o0, o1;
          threefry2x32(key0, key1, 0u, (uint32_t)tok_l * (uint32_t)a.V + (uint32_t)v, o0, o1);
          key = z + gumbel_from_bits(o0 ^ o1);
        }
      }
      if (z > mx) {
        se = se * expf(mx - z) + 1.f;
        mx = z;
      } else {
        se += expf(z - mx);
      }
      if (score) {
        if (v == target) best = {0.f, z, v};  // at most one vocabulary row is the target
      } else {
        Best c = {key, z, v};
        best_merge(best, c);
      }
  });
  {
    const float mx2 = __shfl_xor(mx, 32, 64), se2 = __shfl_xor(se, 32, 64);
    Best o = {__shfl_xor(best.key, 32, 64), __shfl_xor(best.z, 32, 64), __shfl_xor(best.idx, 32, 64)};
    lse_merge(mx, se, mx2, se2);
    best_merge(best, o);
  }
  if (h == 0 && tok < a.M) {
    float* pf = a.part_f + ((size_t)tok * a.nwg + vb) * 4;
    pf[0] = mx; pf[1] = se; pf[2] = best.key; pf[3] = best.z;
    a.part_i[(size_t)tok * a.nwg + vb] = best.idx;
  }
}

// M rows (any count) with the wide kernel + the finalize kernel: greedy, sampling without the sorting
// branch, or scoring; the caller has checked: no forbidden ids, no logits output, D % 128 == 0.
template <int MODE>
static int launch_head_wide(hipStream_t st, const HeadArgs& a, int tok_blocks, int voc_blocks) {
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&head_wide_kernel<MODE>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)HW::LDS);
  if (attr != hipSuccess) return TMX_ERR_LAUNCH;
  hipLaunchKernelGGL(head_wide_kernel<MODE>, dim3(tok_blocks * voc_blocks), dim3(512), HW::LDS, st, a, tok_blocks,
                     voc_blocks);
  return TMX_OK;
}

// With a tile copy, up to 256 rows are faster from it (head_logits): both read the matrix once, and on the 1.05 GB head the
// 256 x 256 blocks take 266 us at 96 rows and 287 at 256, greedy, where the stream takes 196 and 309 (sampling 369 and 414
// against 221 and 383; at 160 rows 277 each and 387 against 321): one line for all, although greedy alone it would lie at
// 160.  More rows would be several passes over the tile copy.
bool head_wide_ok(const HeadArgs& a) {
  return (a.M > 256 || (a.M > 64 && !a.w_tiles)) && a.D % 128 == 0 && a.M > 0 && (size_t)a.M * a.D * 2 < (1u << 31) && (size_t)256 * a.D * 2 < (1u << 31) &&
         a.n_forbidden == 0 && !a.logits_out;
}

size_t head_x_tiles_bytes(int M, int D) { return M > 64 ? (size_t)(M + 31) / 32 * 32 * D * 2 : 0; }

// The wide kernel alone: partials (and, in the sorting branch, keys) of every row; sets a.nwg.
int head_wide_logits(hipStream_t st, HeadArgs& a) {
  if (!head_wide_ok(a)) return TMX_ERR_SHAPE;
  if (!a.x_tiles) return TMX_ERR_ARG;
  const int tok_blocks = (a.M + 255) / 256, voc_blocks = (a.V + HW::ROWS - 1) / HW::ROWS;
  hipLaunchKernelGGL(head_x_tiles_kernel, dim3(a.D / 128, (a.M + 31) / 32), dim3(512), 0, st, a.x, a.x_tiles, a.M, a.D);
  const int rc = check_launch();
  if (rc != TMX_OK) return rc;
  a.nwg = voc_blocks;
  a.row_base = 0;
  int lrc;
  if (a.mode == TMX_SAMPLE_SCORE) lrc = launch_head_wide<TMX_SAMPLE_SCORE>(st, a, tok_blocks, voc_blocks);
  else if (a.mode == TMX_SAMPLE_TOP_P) lrc = launch_head_wide<TMX_SAMPLE_TOP_P>(st, a, tok_blocks, voc_blocks);
  else lrc = launch_head_wide<TMX_SAMPLE_GREEDY>(st, a, tok_blocks, voc_blocks);
  if (lrc != TMX_OK) return lrc;
  return check_launch();
}

int head_wide(hipStream_t st, HeadArgs a) {
  int rc = head_wide_logits(st, a);
  if (rc != TMX_OK) return rc;
  hipLaunchKernelGGL(head_finalize_kernel, dim3(a.M), dim3(256), 0, st, a);
  return check_launch();
}

int head_logits(hipStream_t st, HeadArgs& a) {
  if (a.V % 32 || a.D % 64 || a.M <= 0 || a.M > TMX_MAX_FILL_ROWS) return TMX_ERR_SHAPE;
  a.nwg = (a.V + 127) / 128;
  // One pass over the head matrix per chunk of rows: up to 256 from the tile copy, 64 from the rows themselves.  The
  // partials of every chunk sit where one finalize launch over all rows expects them.
  const int chunk = a.w_tiles ? 256 : 64;
  for (int r0 = 0; r0 < a.M; r0 += chunk) {
    HeadArgs c = a;
    c.M = a.M - r0 < chunk ? a.M - r0 : chunk;
    c.x = a.x + (size_t)r0 * a.D;
    c.row_base = a.row_base + r0;
    c.row_off = a.row_off + r0;
    if (a.logits_out) c.logits_out = a.logits_out + (size_t)r0 * a.V;
    if (a.sort_keys) c.sort_keys = a.sort_keys + (size_t)r0 * a.V;
    c.part_f = a.part_f + (size_t)r0 * a.nwg * 4;
    c.part_i = a.part_i + (size_t)r0 * a.nwg;
    int rc = TMX_OK;
    if (head_row_ok(c.M, c.D)) {
      const size_t lds = (size_t)c.M * (c.D + 8) * 2;
#define TMX_HEAD_ROW(R) \
  if (c.w_tiles) hipLaunchKernelGGL((head_row_kernel<R, true>), dim3(a.nwg), dim3(256), lds, st, c); \
  else hipLaunchKernelGGL((head_row_kernel<R, false>), dim3(a.nwg), dim3(256), lds, st, c)
      if (c.M == 1) { TMX_HEAD_ROW(1); } else if (c.M == 2) { TMX_HEAD_ROW(2); } else { TMX_HEAD_ROW(4); }
#undef TMX_HEAD_ROW
    } else if (c.w_tiles) {
      if (c.M <= 32) hipLaunchKernelGGL((head_kernel<1, true>), dim3(a.nwg), dim3(256), 0, st, c);
      else if (c.M <= 64) hipLaunchKernelGGL((head_kernel<2, true>), dim3(a.nwg), dim3(256), 0, st, c);
      else rc = c.M <= 128 ? launch_head_mid<4, 4, 4>(st, c) : launch_head_mid<8, 4, 4>(st, c);
    } else {
      if (c.M <= 32) hipLaunchKernelGGL((head_kernel<1, false>), dim3(a.nwg), dim3(256), 0, st, c);
      else hipLaunchKernelGGL((head_kernel<2, false>), dim3(a.nwg), dim3(256), 0, st, c);
    }
    if (rc != TMX_OK) return rc;
  }
  return check_launch();
}

int head_sample(hipStream_t st, HeadArgs a) {
  int rc = head_logits(st, a);
  if (rc != TMX_OK) return rc;
  hipLaunchKernelGGL(head_finalize_kernel, dim3(a.M), dim3(256), 0, st, a);
  return check_launch();
}

size_t head_partial_bytes(int M, int V) {
  const size_t nwg = (V + 127) / 128;
  return (size_t)M * nwg * 5 * sizeof(float);
}

}  // namespace tmx

using namespace tmx;

extern "C" size_t tmx_head_sample_workspace_bytes(int M, int V) { return head_partial_bytes(M, V); }

static int head_sample_entry(void* stream, const void* x, const void* head_w, const void* head_tiles, int M, int D,
                             int V, int mode, float temperature, uint32_t seed_hi, uint32_t seed_lo,
                             const int32_t* step, const int32_t* forbidden, int n_forbidden,
                             const int32_t* eos, int n_eos, int32_t* token_buffer, float* logprobs,
                             uint8_t* done, int buf_len, float* logits_out, void* workspace) {
  if (!x || (!head_w && !head_tiles) || !step || !token_buffer || !done || !workspace) return TMX_ERR_ARG;
  if ((n_forbidden > 0 && !forbidden) || (n_eos > 0 && !eos)) return TMX_ERR_ARG;
  if (mode != TMX_SAMPLE_GREEDY && mode != TMX_SAMPLE_TOP_P && mode != TMX_SAMPLE_SCORE) return TMX_ERR_UNSUPPORTED;
  HeadArgs a = {};
  a.x = (const uint16_t*)x;
  a.w = (const uint16_t*)head_w;
  a.w_tiles = (const uint16_t*)head_tiles;
  a.M = M; a.D = D; a.V = V;
  a.mode = mode;
  a.temperature = temperature;
  a.k0 = seed_hi; a.k1 = seed_lo;
  a.step = step;
  a.forbidden = forbidden; a.n_forbidden = n_forbidden;
  a.logits_out = logits_out;
  const size_t nwg = (V + 127) / 128;
  a.part_f = (float*)workspace;
  a.part_i = (int32_t*)((float*)workspace + (size_t)M * nwg * 4);
  a.token_buffer = token_buffer;
  a.logprobs = logprobs;
  a.done = done;
  a.eos = eos; a.n_eos = n_eos;
  a.buf_len = buf_len;
  return head_sample((hipStream_t)stream, a);
}

extern "C" int tmx_head_sample(void* stream, const void* x, const void* head_w, int M, int D, int V,
                               int mode, float temperature, uint32_t seed_hi, uint32_t seed_lo,
                               const int32_t* step, const int32_t* forbidden, int n_forbidden,
                               const int32_t* eos, int n_eos, int32_t* token_buffer, float* logprobs,
                               uint8_t* done, int buf_len, float* logits_out, void* workspace) {
  return head_sample_entry(stream, x, head_w, nullptr, M, D, V, mode, temperature, seed_hi, seed_lo, step, forbidden,
                           n_forbidden, eos, n_eos, token_buffer, logprobs, done, buf_len, logits_out, workspace);
}

extern "C" int tmx_head_sample_tiles(void* stream, const void* x, const void* head_tiles, int M, int D, int V,
                                     int mode, float temperature, uint32_t seed_hi, uint32_t seed_lo,
                                     const int32_t* step, const int32_t* forbidden, int n_forbidden,
                                     const int32_t* eos, int n_eos, int32_t* token_buffer, float* logprobs,
                                     uint8_t* done, int buf_len, float* logits_out, void* workspace) {
  if (!head_tiles) return TMX_ERR_ARG;
  return head_sample_entry(stream, x, nullptr, head_tiles, M, D, V, mode, temperature, seed_hi, seed_lo, step,
                           forbidden, n_forbidden, eos, n_eos, token_buffer, logprobs, done, buf_len, logits_out,
                           workspace);
}

extern "C" int tmx_head_tiles_pack(void* stream, const void* head_w, void* head_tiles, int V, int D) {
  if (!head_w || !head_tiles) return TMX_ERR_ARG;
  return head_tiles_pack((hipStream_t)stream, (const uint16_t*)head_w, (uint16_t*)head_tiles, V, D);
}
