// The decode step for one to four sequences (single-sequence latency regime): five launches per
// layer instead of eight.
//
// At this size a projection is a matrix-vector product: the activations of all rows are a few KiB,
// so every workgroup keeps ALL of them in LDS and can afford to redo the cheap row work itself.
// That removes the launches whose only job was a cross-workgroup reduction:
//   * RMSNorm (tunix/models/llama3/model.py:290-297) runs in the prologue of the projection that
//     consumes it (q|k|v and gate|up): every workgroup normalises the residual stream itself;
//   * the LoRA projection t = x . A (qwix LoRA on tunix/models/llama3/model.py:216-218, :461-487)
//     is computed by every workgroup over the full K (A comes from L2), so the delta
//     bf16(bf16(t . B) * alpha / r) and, for o and down, the residual add
//     (llama3/model.py:546-564) happen in the projection's own epilogue; for the down projection
//     t comes from partial products the gate|up workgroups leave behind (each owns 32 hidden units);
//   * SwiGLU (llama3/model.py:489-496) is the epilogue of gate|up (a workgroup owns a gate tile and
//     the matching up tile);
//   * RoPE and the KV-cache write (llama3/model.py:249-270, :367-377) are the prologue of the
//     attention kernel, and the merge of its context splits is the prologue of the o projection.
// Weights stream HBM -> registers in the packed tile format (one coalesced 1 KiB load per tile and
// wave), every tile load of a wave is issued before the first use, dequantisation is the same
// bit-exact bf16((u - 8) * s), and the product runs on v_mfma_f32_32x32x16_bf16 with the rows
// beyond the batch ignored: at one row the VALU dequantisation, not the matrix pipe, is what a
// tile costs.  A workgroup is 8 waves = column tiles x K-slices; the K-slices meet in LDS.  (The projections without
// SwiGLU take 16 columns per workgroup instead: sb_linear16_kernel.)
#include "tmx_kernels.h"

namespace tmx {

constexpr int kSbThreads = 512, kSbWaves = 8;
constexpr int kSbMaxRows = 4;

// A lane offset past the end of every descriptor here: the load fetches nothing and gives zero.  Loads that some threads, or some
// launches, have no use for take it instead of a branch: behind one the compiler no longer knows how many loads are on the way.
constexpr int kSbNowhere = 0x7FFF0000;

enum { SB_PRO_PLAIN = 0, SB_PRO_NORM = 1, SB_PRO_ATTN = 2 };
enum { SB_EPI_PLAIN = 0, SB_EPI_RESIDUAL = 1, SB_EPI_SWIGLU = 2 };

// LDS carve of sb_linear_kernel (bytes): x [M][K + 8] bf16 | red [8 waves][4][32] f32 |
// red_t [8][4][64] f32 | t [4][64] f32 | act [4][32] f32 | row scratch [4 + 8 * 4] f32 | B [2][16][32] bf16 | A_next [4][32][8] bf16
__host__ __device__ inline size_t sb_x_bytes(int M, int K) { return ((size_t)M * (K + 8) * 2 + 15) & ~(size_t)15; }
constexpr size_t kSbTailFloats = kSbWaves * kSbMaxRows * 32 + kSbWaves * kSbMaxRows * 64 + kSbMaxRows * 64 +
                                 kSbMaxRows * 32 + 4 + kSbWaves * 4 + 2 * 16 * 32 / 2 + 4 * 32 * 4;

// t handed over as parts by the launch before: a thread adds a run of parts of four adjacent columns of a row (columns
// 0 .. 4 nq - 1), in up to 32 runs; the runs meet in red_t [run][m][4 nq] and are added in run order.
struct SbParts {
  int nq, lanes, groups;  // groups 0: nothing handed over
  f32x4_t pv[8];
  __device__ __forceinline__ void load(const SbLinearArgs& a, int pb) {
    const int rest = (int)threadIdx.x % lanes, m = rest / nq, c = (rest - m * nq) * 4;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      pv[u] = *reinterpret_cast<const f32x4_t*>(a.t_parts + ((size_t)min(pb + u, a.t_nparts - 1) * a.M + m) * 32 + c);
  }
  __device__ __forceinline__ void request(const SbLinearArgs& a) {
    groups = 0;
    if (!a.t_parts) return;
    nq = (a.lora_r + 3) >> 2;
    lanes = nq * a.M;
    groups = min(kSbThreads / lanes, 32);
    const int grp = (int)threadIdx.x / lanes;
    if (grp < groups) load(a, grp * ((a.t_nparts + groups - 1) / groups));
  }
  __device__ __forceinline__ void finish(const SbLinearArgs& a, float* red_t) {
    if (!groups) return;
    const int grp = (int)threadIdx.x / lanes, rest = (int)threadIdx.x - grp * lanes;
    if (grp >= groups) return;
    const int run = (a.t_nparts + groups - 1) / groups;
    const int b0 = grp * run, b1 = min(b0 + run, a.t_nparts);
    f32x4_t t = {0.f, 0.f, 0.f, 0.f};
    for (int pb = b0; pb < b1; pb += 8) {
      if (pb > b0) load(a, pb);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (pb + u < b1) t += pv[u];
    }
    *reinterpret_cast<f32x4_t*>(red_t + (grp * lanes + rest) * 4) = t;
  }
};
__device__ __forceinline__ float sb_parts_total(const SbParts& p, const float* red_t, int m, int cc) {
  if (cc >= p.nq * 4) return 0.f;
  float t = 0.f;
  for (int g = 0; g < p.groups; ++g) t += red_t[(g * p.lanes + m * p.nq) * 4 + cc];
  return t;
}
__device__ __forceinline__ float sb_rms(const SbLinearArgs& a, const float* rms_s, int m) {
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < kSbWaves; ++w) t += rms_s[4 + w * 4 + m];
  return sqrtf(t / (float)a.K + a.eps);
}

// The prologues: the activations of every row into LDS [M][XS] bf16, in two halves: request() before anything of the
// launch is waited for, finish() afterwards.  Loads return in order, so a load requested behind a wait costs a whole
// further round trip to memory.

// merge of the context splits of the attention kernel: out = sum_s o_s exp(m_s - m) / sum_s l_s exp(m_s - m); a thread
// owns four adjacent values of a head at a time, of up to 8 splits
struct SbMerge {
  f32x4_t po[8];
  f32x2_t pm[8];
  __device__ __forceinline__ void load(const SbLinearArgs& a, int e) {
    const int H = a.attn_h, ns = a.attn_ns, G = a.attn_g, heads = a.attn_kh * G, per_row = heads * H / 4;
    const float* ml = a.attn_part + (size_t)a.M * heads * ns * H;  // (max, sum) behind the outputs
    if (e >= a.M * per_row) return;
    const int m = e / per_row, rest = (e - m * per_row) * 4, head = rest / H, d = rest - head * H;
    const size_t first = ((size_t)(m * a.attn_kh + head / G) * ns) * G + head % G;  // split 0 of this head; + G per split
#pragma unroll
    for (int sp = 0; sp < 8; ++sp)
      if (sp < ns) {
        const size_t i = first + (size_t)sp * G;
        po[sp] = *reinterpret_cast<const f32x4_t*>(a.attn_part + i * H + d);
        pm[sp] = *reinterpret_cast<const f32x2_t*>(ml + i * 2);
      }
  }
  __device__ __forceinline__ void store(const SbLinearArgs& a, int e, uint16_t* xs, int XS) const {
    const int ns = a.attn_ns, per_row = a.attn_kh * a.attn_g * a.attn_h / 4;
    if (e >= a.M * per_row) return;
    float mm = -1e30f;
#pragma unroll
    for (int sp = 0; sp < 8; ++sp)
      if (sp < ns) mm = fmaxf(mm, pm[sp].x);
    float ls = 0.f;
    f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int sp = 0; sp < 8; ++sp)
      if (sp < ns) {
        const float w = __expf(pm[sp].x - mm);
        ls += pm[sp].y * w;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] += po[sp][i] * w;
      }
    uint2 p = {0u, 0u};
    if (ls > 0.f) {
      p.x = pack_bf2(o[0] / ls, o[1] / ls);
      p.y = pack_bf2(o[2] / ls, o[3] / ls);
    }
    const int m = e / per_row;
    *reinterpret_cast<uint2*>(xs + m * XS + (e - m * per_row) * 4) = p;
  }
  __device__ __forceinline__ void request(const SbLinearArgs& a) { load(a, threadIdx.x); }
  __device__ __forceinline__ void finish(const SbLinearArgs& a, uint16_t* xs, int XS, float*) {
    const int items = a.M * a.attn_kh * a.attn_g * a.attn_h / 4;
    store(a, threadIdx.x, xs, XS);
    for (int e = (int)threadIdx.x + kSbThreads; e < items; e += 2 * kSbThreads) {  // more rows: two at a time
      SbMerge second;
      load(a, e);
      second.load(a, e + kSbThreads);
      store(a, e, xs, XS);
      second.store(a, e + kSbThreads, xs, XS);
    }
  }
};

struct SbCopy {
  // host: at most 8 chunks per thread.  (As an array of HIP's uint4 it lived in scratch memory, which the data had to reach
  // and come back from: down of the 1B shape at one row 9.9 -> 9.1 us, at three rows 13.1 -> 10.2.)
  u32x4_t v[8];
  __device__ __forceinline__ void request(const SbLinearArgs& a) {
    const int cpr = a.K >> 3, nchunks = a.M * cpr;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int ch = (int)threadIdx.x + kSbThreads * i, m = ch / cpr;
      if (ch < nchunks) v[i] = *reinterpret_cast<const u32x4_t*>(a.x + (size_t)m * a.ldx + (ch - m * cpr) * 8);
    }
  }
  __device__ __forceinline__ void finish(const SbLinearArgs& a, uint16_t* xs, int XS, float*) {
    const int cpr = a.K >> 3, nchunks = a.M * cpr;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int ch = (int)threadIdx.x + kSbThreads * i, m = ch / cpr;
      if (ch < nchunks) *reinterpret_cast<u32x4_t*>(xs + m * XS + (ch - m * cpr) * 8) = v[i];
    }
  }
};

// RMSNorm of every row: up to 4 chunks of 8 elements per thread (M K <= 16384); rms_s: [4] + per-wave sums [8][4]
struct SbNorm {
  uint4 xq[4], wq[4];
  __device__ __forceinline__ void request(const SbLinearArgs& a) {
    const int cpr = a.K >> 3, nchunks = a.M * cpr;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ch = (int)threadIdx.x + kSbThreads * i, m = ch / cpr, cc = ch - m * cpr;
      if (ch < nchunks) {
        xq[i] = *reinterpret_cast<const uint4*>(a.x + (size_t)m * a.ldx + cc * 8);
        wq[i] = *reinterpret_cast<const uint4*>(a.norm_w + cc * 8);
      }
    }
  }
  __device__ __forceinline__ void finish(const SbLinearArgs& a, uint16_t* xs, int XS, float* rms_s) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int cpr = a.K >> 3, nchunks = a.M * cpr;
    auto unpack = [](const uint4& q, float (&v)[8]) __attribute__((always_inline)) {
      v[0] = bf_lo(q.x); v[1] = bf_hi(q.x); v[2] = bf_lo(q.y); v[3] = bf_hi(q.y);
      v[4] = bf_lo(q.z); v[5] = bf_hi(q.z); v[6] = bf_lo(q.w); v[7] = bf_hi(q.w);
    };
    float ss[kSbMaxRows] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ch = tid + kSbThreads * i;
      if (ch < nchunks) {
        const int m = ch / cpr;
        float v[8], sq = 0.f;
        unpack(xq[i], v);
#pragma unroll
        for (int e = 0; e < 8; ++e) sq += v[e] * v[e];
#pragma unroll
        for (int r = 0; r < kSbMaxRows; ++r) ss[r] += (m == r) ? sq : 0.f;
      }
    }
    // sum of squares of each row over the workgroup, in a fixed order
#pragma unroll
    for (int r = 0; r < kSbMaxRows; ++r)
      if (r < a.M) ss[r] = wave_sum(ss[r]);
    if (lane == 0) {
#pragma unroll
      for (int r = 0; r < kSbMaxRows; ++r) rms_s[4 + wave * 4 + r] = ss[r];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ch = tid + kSbThreads * i;
      if (ch < nchunks) {
        const int m = ch / cpr, cc = ch - m * cpr;
        const float rms = sb_rms(a, rms_s, m);
        float v[8], w[8], o[8];
        unpack(xq[i], v);
        unpack(wq[i], w);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          o[e] = a.family == TMX_FAMILY_LLAMA3 ? rbf(w[e] * v[e]) / rms : w[e] * (v[e] / rms);
        uint4 pk;
        pk.x = pack_bf2(o[0], o[1]); pk.y = pack_bf2(o[2], o[3]);
        pk.z = pack_bf2(o[4], o[5]); pk.w = pack_bf2(o[6], o[7]);
        *reinterpret_cast<uint4*>(xs + m * XS + cc * 8) = pk;
      }
    }
  }
};

template <int PRO> struct SbPrologue { using type = SbMerge; };
template <> struct SbPrologue<SB_PRO_PLAIN> { using type = SbCopy; };
template <> struct SbPrologue<SB_PRO_NORM> { using type = SbNorm; };

// Loads return in the order they are requested, and a wait counts the ones behind: what is waited for first, the rows, is
// requested in front of the weights, whose number NT (at least a wave's k-tiles, up to 8 at once) is a constant, as is the
// number NA of the tiles of A, so that the wait for the rows leaves the others on the way.  Requested behind the weights ("they
// come from farther") the norm began when the last weight had arrived.  A, which every workgroup reads whole, is 128 KiB a CU
// beside 64 KiB of weights in gate|up of the 1B shape: requested with the weights it holds them up (11.7 us a launch at one
// row), a k-tile at a time behind them it costs a round trip each (10.6); requested at once when half the weights are used up:
// 9.9 (8.2 without an adapter; four rows 12.1 -> 11.3).
template <int PRO, int EPI, int NT, int NA>
__global__ __launch_bounds__(kSbThreads) void sb_linear_kernel(SbLinearArgs a) {
  extern __shared__ __align__(16) unsigned char sb_smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, nl = lane & 31;
  const int M = a.M, K = a.K, KT = K >> 6, XS = K + 8;
  constexpr int CT = EPI == SB_EPI_SWIGLU ? 2 : 1;  // column tiles per workgroup
  constexpr int KS = kSbWaves / CT;                  // K-slices
  const int c = wave % CT, s = wave / CT;
  uint16_t* xs = reinterpret_cast<uint16_t*>(sb_smem);
  float* red = reinterpret_cast<float*>(sb_smem + sb_x_bytes(M, K));
  float* red_t = red + kSbWaves * kSbMaxRows * 32;
  float* t_s = red_t + kSbWaves * kSbMaxRows * 64;
  float* act_s = t_s + kSbMaxRows * 64;
  float* rms_s = act_s + kSbMaxRows * 32;  // [4] + per-wave sums [8][4]
  uint16_t* b_s = reinterpret_cast<uint16_t*>(rms_s + 4 + kSbWaves * 4);  // [CT][16][32]
  u32x4_t* an_s = reinterpret_cast<u32x4_t*>(b_s + 2 * 16 * 32);          // [4][32]

  // what the epilogue needs that depends on no other launch: the B values of the column tile(s) (rows 0..15 of B; a larger
  // rank reads the rest in the epilogue), the residual, and the rows of the next projection's A
  const bool epi_thread = tid < kSbMaxRows * 32 && (tid >> 5) < M;
  const int em = tid >> 5, ej = tid & 31;
  // (one 16-byte load of a wave: column tile q of B by wave q, lane (row, piece); the 32 rows of A_next by waves 2 and 3; they
  // meet the threads that use them in LDS.  As 16 or 32 values of two bytes a thread they held up the loads behind them)
  uint32_t res_v = 0;
  u32x4_t aux;
  {
    const bool of_b = wave < CT;
    const int n0 = ((int)blockIdx.x + wave * (EPI == SB_EPI_SWIGLU ? a.pair_off : 0)) * 32;
    // rows k .. k + 7 of column j are 8 consecutive values in fragment order (r_pad 32): ((kb * 4 + t) * 64 + 32 h + j) * 8 with
    // k = 64 kb + 16 t + 8 h, so the 32 rows from 32 blockIdx.x on are 2 KiB
    const bool of_next = EPI == SB_EPI_SWIGLU && (wave >> 1) == 1 && a.a_next;
    const void* src = of_b ? (const void*)a.lora_b : (const void*)a.a_next;
    const uint32_t bytes = of_b ? (a.lora_b ? (uint32_t)a.lora_r * a.N * 2u : 0u) : of_next ? (uint32_t)gridDim.x * 2048u : 0u;
    aux = __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(src, bytes), of_b ? ((lane >> 2) * a.N + n0) * 2 + (lane & 3) * 16 : lane * 16,
                                                of_b ? 0 : (int)blockIdx.x * 2048 + (wave & 1) * 1024, 0);
    if constexpr (EPI == SB_EPI_RESIDUAL)
      res_v = __builtin_amdgcn_raw_buffer_load_b16(make_rsrc(a.residual, (uint32_t)M * a.ldy * 2u),
                                                   epi_thread ? (em * a.ldy + (int)blockIdx.x * 32 + ej) * 2 : kSbNowhere, 0, 0);
  }
  // parts of t and the rows
  SbParts parts;
  parts.request(a);  // handed over for single matrices only (down projection)
  typename SbPrologue<PRO>::type pro;
  pro.request(a);
  __builtin_amdgcn_sched_barrier(0);

  // column tile of this wave: its first weight tiles and scales
  const int nb = EPI == SB_EPI_SWIGLU ? (int)blockIdx.x + c * a.pair_off : (int)blockIdx.x;
  const int per = (KT + KS - 1) / KS;  // k-tiles per slice
  const int kt0 = s * per, kt1 = min(kt0 + per, KT);
  const int gs = __builtin_ctz(a.G >> 6), KG = K / a.G;
  const u32x4_t* wsrc = reinterpret_cast<const u32x4_t*>(a.qw) + (size_t)nb * KT * 64 + lane;
  const uint16_t* ssrc = a.scales + (size_t)nb * KG * 32 + nl;
  u32x4_t wr[NT];
  uint32_t sr[NT];
  auto load_w = [&](int kt, int slot) __attribute__((always_inline)) {
    kt = min(kt, KT - 1);
    wr[slot] = __builtin_nontemporal_load(wsrc + (size_t)kt * 64);  // every tile is read once, by this wave
    sr[slot] = ssrc[(size_t)(kt >> gs) * 32];
  };
#pragma unroll
  for (int i = 0; i < NT; ++i) load_w(kt0 + i, i);
  // x . A: wave w takes the w-th eighth of K, i.e. the c-th part of its own slice
  constexpr int LT = NT < 4 / (NA ? NA : 1) ? NT : 4 / (NA ? NA : 1);  // k-tiles of A per wave requested at once
  const int lpart = (per + CT - 1) / CT, l0 = kt0 + c * lpart, nk = min(lpart, kt1 - l0);
  u32x4_t ab[LT][NA ? NA : 1][4];  // [slot][tile of A][step]
  // the epilogue uses the t columns of its own segment(s) only: the tiles of A that hold them
  const int RT = a.Rpad >> 5;  // 32-column tiles of A (<= 2)
  int q0 = 0;
  if (NA && CT == 1) {
    const int n0 = blockIdx.x * 32;
    const int seg = n0 >= a.seg_end[0] ? (n0 >= a.seg_end[1] ? 2 : 1) : 0;
    q0 = min((seg * a.lora_r) >> 5, RT - NA);
  }
  auto load_a = [&](int k, int slot) __attribute__((always_inline)) {
    const u32x4_t* ap = reinterpret_cast<const u32x4_t*>(a.a_t) + ((size_t)min(l0 + k, KT - 1) * RT + q0) * 256 + lane;
#pragma unroll
    for (int i = 0; i < NA * 4; ++i) ab[slot][i / 4][i % 4] = ap[i * 64];
  };
  __builtin_amdgcn_sched_barrier(0);

  // ---- prologue: the activations of every row into LDS ----
  parts.finish(a, red_t);
  pro.finish(a, xs, XS, rms_s);
  __syncthreads();

  // ---- the K-slice of this wave: its column tile, and its share of x . A ----
  const int xrow = min(nl, M - 1);  // rows beyond the batch repeat the last one (their results are dropped)
  const uint16_t* xb = xs + xrow * XS + h * 8;
  f32x16_t acc, tacc[2];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = tacc[0][r] = tacc[1][r] = 0.f;
  for (int base = 0; base < per; base += NT) {
    static_for<NT>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      if constexpr (NA > 0 && i == NT / 2) {
        if (base == 0) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int d = 0; d < LT; ++d) load_a(d, d);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      const int kt = kt0 + base + i;
      if (kt < kt1) {
        bf16x8_t xa[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) xa[t] = *reinterpret_cast<const bf16x8_t*>(xb + kt * 64 + t * 16);
        const NibbleScale sc = nibble_scale(bf2f((uint16_t)sr[i]));
        const uint32_t wd[4] = {wr[i].x, wr[i].y, wr[i].z, wr[i].w};
        if (base + i + NT < per) load_w(kt + NT, i);  // slot consumed: refill it for the tile NT further on
#pragma unroll
        for (int t = 0; t < 4; ++t)
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[t], dequant_word(wd[t], sc), acc, 0, 0, 0);
      }
    });
  }
  if constexpr (NA > 0) {
    for (int k0 = 0; k0 < nk; k0 += LT)
      static_for<LT>([&](auto dc) __attribute__((always_inline)) {
        constexpr int d = decltype(dc)::value;
        const int k = k0 + d;
        if (k < nk) {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const bf16x8_t xa = *reinterpret_cast<const bf16x8_t*>(xb + (l0 + k) * 64 + t * 16);
#pragma unroll
            for (int u = 0; u < NA; ++u)
              tacc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa, __builtin_bit_cast(bf16x8_t, ab[d][u][t]), tacc[u], 0, 0, 0);
          }
          if (k + LT < nk) load_a(k + LT, d);
        }
      });
  }
  if (wave < CT) reinterpret_cast<u32x4_t*>(b_s)[wave * 64 + lane] = aux;
  else if (EPI == SB_EPI_SWIGLU && (wave >> 1) == 1) an_s[(wave & 1) * 64 + lane] = aux;
  // rows 0..3 of a tile are accumulator registers 0..3 of the lanes with h == 0
  if (h == 0) {
#pragma unroll
    for (int r = 0; r < kSbMaxRows; ++r) {
      red[(wave * kSbMaxRows + r) * 32 + nl] = acc[r];
      if constexpr (NA > 0) {
#pragma unroll
        for (int u = 0; u < NA; ++u) red_t[(wave * kSbMaxRows + r) * 64 + (q0 + u) * 32 + nl] = tacc[u][r];
      }
    }
  }
  __syncthreads();
  // t = bf16(sum over the waves, in wave order), or bf16(sum of the runs of handed-over parts, in run order)
  if (tid < kSbMaxRows * 64) {
    const int m = tid >> 6, cc = tid & 63;
    float t = 0.f;
    if (m < M) {
      if (a.t_parts) {
        t = sb_parts_total(parts, red_t, m, cc);
      } else if (NA && (cc >> 5) >= q0 && (cc >> 5) < q0 + NA) {
#pragma unroll
        for (int w = 0; w < kSbWaves; ++w) t += red_t[(w * kSbMaxRows + m) * 64 + cc];
      }
    }
    t_s[m * 64 + cc] = rbf(t);
  }
  __syncthreads();

  // ---- epilogue: thread (row m, column j of the tile) ----
  const bool lora = a.lora_b != nullptr;
  if (epi_thread) {
    const int m = em, j = ej;
    float yv[CT];
#pragma unroll
    for (int q = 0; q < CT; ++q) {
      const int tile = EPI == SB_EPI_SWIGLU ? (int)blockIdx.x + q * a.pair_off : (int)blockIdx.x;
      const int n = tile * 32 + j;
      float b = 0.f;
      for (int sl = 0; sl < KS; ++sl) b += red[((sl * CT + q) * kSbMaxRows + m) * 32 + j];
      b = rbf(b);
      if (lora) {
        const int seg = n >= a.seg_end[0] ? (n >= a.seg_end[1] ? 2 : 1) : 0;
        const float* tp = t_s + m * 64 + seg * a.lora_r;
        float d = 0.f;
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) d = fmaf(rr < a.lora_r ? tp[rr] : 0.f, bf2f(b_s[(q * 16 + rr) * 32 + j]), d);
        for (int rr = 16; rr < a.lora_r; ++rr) d = fmaf(tp[rr], bf2f(a.lora_b[(size_t)rr * a.N + n]), d);
        b = rbf(b + rbf(rbf(d) * a.lora_ls));
      }
      yv[q] = b;
    }
    if constexpr (EPI == SB_EPI_SWIGLU) {
      const float g = yv[0], u = yv[CT - 1];
      const float sg = rbf(1.f / (1.f + expf(-g)));
      const float av = rbf(rbf(g * sg) * u);
      a.y[(size_t)m * a.ldy + blockIdx.x * 32 + j] = f2bf(av);
      act_s[m * 32 + j] = av;
    } else {
      const int n = blockIdx.x * 32 + j;
      float v = yv[0];
      if constexpr (EPI == SB_EPI_RESIDUAL) v = rbf(v + bf2f((uint16_t)res_v));
      a.y[(size_t)m * a.ldy + n] = f2bf(v);
    }
  }
  if constexpr (EPI == SB_EPI_SWIGLU) {
    if (a.a_next) {
      // this workgroup's 32 hidden units times their rows of the next projection's A: one part of its t
      __syncthreads();
      if (epi_thread) {
        float t = 0.f;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const u32x4_t w = an_s[u * 32 + ej];
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) {
            t = fmaf(act_s[em * 32 + u * 8 + 2 * jj], bf_lo(w[jj]), t);
            t = fmaf(act_s[em * 32 + u * 8 + 2 * jj + 1], bf_hi(w[jj]), t);
          }
        }
        a.t_parts_out[((size_t)blockIdx.x * M + em) * 32 + ej] = t;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The projections without SwiGLU (q|k|v, o, down) with 16 columns per workgroup.  At one row such a launch is bound by
// the bytes it has in flight and by its chain of round trips, not by HBM: 32 columns of a 2048-wide matrix were 64
// workgroups on 256 CUs, each pulling a 128 KB column stream of the down projection (1B shape) at what one CU can keep
// in flight.  16 columns are twice as many workgroups with half the stream each, and every load a wave makes (its whole
// K-slice of weights, its tiles of A, its share of the handed-over results) is requested before the first is used.
// The 16 x 16 x 32 MFMA takes them: lane (n = l % 16, q = l / 16) holds column n of k-tile 2 p + q / 2, half q % 2, so a
// wave's load is two half tiles, and word t of the four lanes of a column is 32 consecutive steps of the contraction
// (the x operand reads the same k).  Measured on the 1B shape at one row / three rows (trace, us per launch,
// 32 columns -> 16): q|k|v 8.0 / 9.1 -> 8.0 / 9.0, o 9.3 / 15.6 -> 7.4 / 9.6, down 11.8 / 14.4 -> 9.8 / 13.0 (see
// also SbCopy); with the rows requested before the weights, and the numbers of loads constants (see sb_linear_kernel), at one row
// 6.7 -> 6.1, 6.4 -> 5.9 and, without the x . A that is handed over, 9.0 -> 7.6.

// LDS: x [M][K + 8] bf16 | red [8 waves][4][16] f32 | red_t [8][4][64] f32 | t [4][64] f32 | row scratch [4 + 8 * 4] f32 | B [16][16] bf16
constexpr size_t kSb16TailFloats = kSbWaves * kSbMaxRows * 16 + kSbWaves * kSbMaxRows * 64 + kSbMaxRows * 64 + 4 + kSbWaves * 4 + 16 * 16 / 2;

template <int PRO, int EPI, int NT, int NQ>  // pairs of k-tiles per wave requested at once (1 to 8), tiles of 16 columns of A (0 to 2)
__global__ __launch_bounds__(kSbThreads) void sb_linear16_kernel(SbLinearArgs a) {
  extern __shared__ __align__(16) unsigned char sb_smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15, q = lane >> 4, h = q & 1, par = q >> 1;
  const int M = a.M, K = a.K, KT = K >> 6, KP = KT >> 1, XS = K + 8;
  uint16_t* xs = reinterpret_cast<uint16_t*>(sb_smem);
  float* red = reinterpret_cast<float*>(sb_smem + sb_x_bytes(M, K));
  float* red_t = red + kSbWaves * kSbMaxRows * 16;
  float* t_s = red_t + kSbWaves * kSbMaxRows * 64;
  float* rms_s = t_s + kSbMaxRows * 64;  // [4] + per-wave sums [8][4]
  uint16_t* b_s = reinterpret_cast<uint16_t*>(rms_s + 4 + kSbWaves * 4);  // [16][16]

  // what the epilogue needs and no other launch makes
  const bool epi_thread = tid < kSbMaxRows * 16 && (tid >> 4) < M;
  const int em = tid >> 4, n = (int)blockIdx.x * 16 + (tid & 15);
  uint32_t res_v = 0;
  u32x4_t aux;  // rows 0..15 of B, by the first 32 threads (see sb_linear_kernel)
  {
    aux = __builtin_amdgcn_raw_buffer_load_b128(make_rsrc(a.lora_b, a.lora_b ? (uint32_t)a.lora_r * a.N * 2u : 0u),
                                                tid < 32 ? ((tid >> 1) * a.N + (int)blockIdx.x * 16) * 2 + (tid & 1) * 16 : kSbNowhere, 0, 0);
    if constexpr (EPI == SB_EPI_RESIDUAL)
      res_v = __builtin_amdgcn_raw_buffer_load_b16(make_rsrc(a.residual, (uint32_t)M * a.ldy * 2u),
                                                   epi_thread ? (em * a.ldy + n) * 2 : kSbNowhere, 0, 0);
  }

  // parts of t and the rows: in front of the weights, see sb_linear_kernel
  SbParts parts;
  parts.request(a);  // handed over for single matrices only (down projection)
  typename SbPrologue<PRO>::type pro;
  pro.request(a);
  __builtin_amdgcn_sched_barrier(0);

  // weights and scales of this wave's pairs
  const int nb = (int)blockIdx.x >> 1, half16 = ((int)blockIdx.x & 1) * 16;
  const int per = (KP + kSbWaves - 1) / kSbWaves, p0 = wave * per, p1 = min(p0 + per, KP);
  const int gs = __builtin_ctz(a.G >> 6), KG = K / a.G;
  const u32x4_t* wsrc = reinterpret_cast<const u32x4_t*>(a.qw) + ((size_t)nb * KT + par) * 64 + 32 * h + half16 + n16;
  const uint16_t* ssrc = a.scales + (size_t)nb * KG * 32 + half16 + n16;
  u32x4_t wr[NT];
  uint32_t sr[NT];
  auto load_w = [&](int p, int slot) __attribute__((always_inline)) {
    p = min(p, KP - 1);
    wr[slot] = __builtin_nontemporal_load(wsrc + (size_t)p * 128);
    sr[slot] = ssrc[(size_t)((2 * p + par) >> gs) * 32];
  };
#pragma unroll
  for (int i = 0; i < NT; ++i) load_w(p0 + i, i);

  // x . A of this wave's eighth of K, for the tiles of 16 columns of A that hold this workgroup's segment (of a rank of 16
  // half of what lies in a tile of 32 is another segment's or padding: 64 KB instead of 128 KB of A per workgroup on the 1B
  // shape, one row / three rows: q|k|v 8.0 / 9.1 -> 7.0 / 7.8 us, o 7.5 / 9.8 -> 6.4 / 8.7), the first of them requested now.
  // The four lane groups of a load hold 32 consecutive steps of the contraction.
  constexpr int LT = NT == 1 ? 2 : 4;  // k-tiles of A per wave requested at once
  int q0 = 0;
  if constexpr (NQ > 0) {
    const int n0 = (int)blockIdx.x * 16;
    const int seg = n0 >= a.seg_end[0] ? (n0 >= a.seg_end[1] ? 2 : 1) : 0;
    q0 = min((seg * a.lora_r) >> 4, (a.Rpad >> 4) - NQ);
  }
  const int RT = a.Rpad >> 5;
  const int lper = (KT + kSbWaves - 1) / kSbWaves, l0 = wave * lper, nk = min(lper, KT - l0);
  u32x4_t ab[LT][NQ ? NQ : 1][2];
  auto load_a = [&](int k, int slot) __attribute__((always_inline)) {
    const u32x4_t* ap = reinterpret_cast<const u32x4_t*>(a.a_t) + ((size_t)min(l0 + k, KT - 1) * RT * 4 + par) * 64 + 32 * h + n16;
#pragma unroll
    for (int i = 0; i < 2 * NQ; ++i) ab[slot][i / 2][i % 2] = ap[((q0 + i / 2) >> 1) * 256 + ((q0 + i / 2) & 1) * 16 + i % 2 * 128];
  };
  if constexpr (NQ > 0) {
#pragma unroll
    for (int i = 0; i < LT; ++i) load_a(i, i);
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- prologue: the activations of every row into LDS ----
  parts.finish(a, red_t);
  pro.finish(a, xs, XS, rms_s);
  __syncthreads();

  // ---- this wave's pairs of k-tiles ----
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  const uint16_t* xb = xs + min(n16, M - 1) * XS + par * 64 + h * 8;  // rows beyond the batch repeat the last one
  for (int base = 0; base < per; base += NT) {
    static_for<NT>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      const int p = p0 + base + i;
      if (p < p1) {
        bf16x8_t xa[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) xa[t] = *reinterpret_cast<const bf16x8_t*>(xb + p * 128 + t * 16);
        const NibbleScale sc = nibble_scale(bf2f((uint16_t)sr[i]));
        const uint32_t wd[4] = {wr[i].x, wr[i].y, wr[i].z, wr[i].w};
        if (base + i + NT < per) load_w(p + NT, i);
#pragma unroll
        for (int t = 0; t < 4; ++t)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[t], dequant_word(wd[t], sc), acc, 0, 0, 0);
      }
    });
  }
  if constexpr (NQ > 0) {
    f32x4_t tacc[NQ];
#pragma unroll
    for (int u = 0; u < NQ; ++u) tacc[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const uint16_t* lb = xs + min(n16, M - 1) * XS + l0 * 64 + par * 16 + h * 8;
    for (int k0 = 0; k0 < nk; k0 += LT)
      static_for<LT>([&](auto dc) __attribute__((always_inline)) {
        constexpr int d = decltype(dc)::value;
        const int k = k0 + d;
        if (k < nk) {
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const bf16x8_t xa = *reinterpret_cast<const bf16x8_t*>(lb + k * 64 + s * 32);
#pragma unroll
            for (int u = 0; u < NQ; ++u)
              tacc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa, __builtin_bit_cast(bf16x8_t, ab[d][u][s]), tacc[u], 0, 0, 0);
          }
          if (k + LT < nk) load_a(k + LT, d);
        }
      });
    if (q == 0) {
#pragma unroll
      for (int u = 0; u < NQ; ++u)
#pragma unroll
        for (int r = 0; r < kSbMaxRows; ++r) red_t[(wave * kSbMaxRows + r) * 64 + (q0 + u) * 16 + n16] = tacc[u][r];
    }
  }
  if (tid < 32) reinterpret_cast<u32x4_t*>(b_s)[tid] = aux;
  if (q == 0) {  // rows 0..3 of the 16 x 16 tile: registers 0..3 of lanes 0..15
#pragma unroll
    for (int r = 0; r < kSbMaxRows; ++r) red[(wave * kSbMaxRows + r) * 16 + n16] = acc[r];
  }
  __syncthreads();
  // t = bf16(sum over the waves, in wave order), or bf16(sum of the runs, in run order)
  if (tid < kSbMaxRows * 64) {
    const int m = tid >> 6, cc = tid & 63;
    float t = 0.f;
    if (m < M) {
      if (a.t_parts) {
        t = sb_parts_total(parts, red_t, m, cc);
      } else if (NQ && (cc >> 4) >= q0 && (cc >> 4) < q0 + NQ) {
#pragma unroll
        for (int w = 0; w < kSbWaves; ++w) t += red_t[(w * kSbMaxRows + m) * 64 + cc];
      }
    }
    t_s[m * 64 + cc] = rbf(t);
  }
  __syncthreads();
  if (epi_thread) {
    float b = 0.f;
#pragma unroll
    for (int w = 0; w < kSbWaves; ++w) b += red[(w * kSbMaxRows + em) * 16 + (tid & 15)];
    b = rbf(b);
    if (a.lora_b) {
      const int seg = n >= a.seg_end[0] ? (n >= a.seg_end[1] ? 2 : 1) : 0;
      const float* tp = t_s + em * 64 + seg * a.lora_r;
      float d = 0.f;
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) d = fmaf(rr < a.lora_r ? tp[rr] : 0.f, bf2f(b_s[rr * 16 + (tid & 15)]), d);
      for (int rr = 16; rr < a.lora_r; ++rr) d = fmaf(tp[rr], bf2f(a.lora_b[(size_t)rr * a.N + n]), d);
      b = rbf(b + rbf(rbf(d) * a.lora_ls));
    }
    if constexpr (EPI == SB_EPI_RESIDUAL) b = rbf(b + bf2f((uint16_t)res_v));
    a.y[(size_t)em * a.ldy + n] = f2bf(b);
  }
}

size_t sb_linear_lds(int M, int K) { return sb_x_bytes(M, K) + kSbTailFloats * 4; }

template <int PRO, int EPI, int NT, int NA>
static int launch_sb(hipStream_t st, const SbLinearArgs& a, int blocks) {
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&sb_linear_kernel<PRO, EPI, NT, NA>), hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
  if (attr != hipSuccess) return TMX_ERR_LAUNCH;
  hipLaunchKernelGGL((sb_linear_kernel<PRO, EPI, NT, NA>), dim3(blocks), dim3(kSbThreads), sb_linear_lds(a.M, a.K), st, a);
  return check_launch();
}
// tiles of A that hold the columns of any workgroup's segment
static int sb_a_tiles(const SbLinearArgs& a, bool pairs, int width) {
  if (!a.a_t) return 0;
  if (pairs) return a.Rpad / width;  // gate and up columns meet in a workgroup
  int n = 1;
  for (int seg = 0; seg < (a.seg_end[0] < a.N ? (a.seg_end[1] < a.N ? 3 : 2) : 1); ++seg) {
    const int q0 = seg * a.lora_r / width, q1 = ((seg + 1) * a.lora_r - 1) / width;
    if (q1 - q0 + 1 > n) n = q1 - q0 + 1;
  }
  return n < a.Rpad / width ? n : a.Rpad / width;
}
template <int PRO, int EPI, int NT>
static int launch_sb_a(hipStream_t st, const SbLinearArgs& a, int blocks) {
  switch (sb_a_tiles(a, EPI == SB_EPI_SWIGLU, 32)) {
    case 0: return launch_sb<PRO, EPI, NT, 0>(st, a, blocks);
    case 1: return launch_sb<PRO, EPI, NT, 1>(st, a, blocks);
    default: return launch_sb<PRO, EPI, NT, 2>(st, a, blocks);
  }
}

size_t sb_linear16_lds(int M, int K) { return sb_x_bytes(M, K) + kSb16TailFloats * 4; }

template <int PRO, int EPI, int NT, int NQ>
static int launch_sb16(hipStream_t st, const SbLinearArgs& a) {
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&sb_linear16_kernel<PRO, EPI, NT, NQ>), hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
  if (attr != hipSuccess) return TMX_ERR_LAUNCH;
  hipLaunchKernelGGL((sb_linear16_kernel<PRO, EPI, NT, NQ>), dim3(a.N / 16), dim3(kSbThreads), sb_linear16_lds(a.M, a.K), st, a);
  return check_launch();
}
template <int PRO, int EPI, int NT>
static int launch_sb16_a(hipStream_t st, const SbLinearArgs& a) {
  switch (sb_a_tiles(a, false, 16)) {
    case 0: return launch_sb16<PRO, EPI, NT, 0>(st, a);
    case 1: return launch_sb16<PRO, EPI, NT, 1>(st, a);
    default: return launch_sb16<PRO, EPI, NT, 2>(st, a);
  }
}
// as many requests at once as a wave has k-tiles (pairs), at most 8
template <int PRO, int EPI>
static int launch_sb16_t(hipStream_t st, const SbLinearArgs& a) {
  const int per = ((a.K >> 7) + kSbWaves - 1) / kSbWaves;
  if (per <= 1) return launch_sb16_a<PRO, EPI, 1>(st, a);
  if (per <= 2) return launch_sb16_a<PRO, EPI, 2>(st, a);
  if (per <= 4) return launch_sb16_a<PRO, EPI, 4>(st, a);
  return launch_sb16_a<PRO, EPI, 8>(st, a);
}

bool sb_linear_ok(int M, int K, int N, int G, int rank, int rpad, bool norm) {
  if (M < 1 || M > kSbMaxRows || K % 64 || N % 32 || G % 64 || (G & (G - 1)) || K % G) return false;
  if ((size_t)M * K > (norm ? 16384u : 32768u) || sb_linear_lds(M, K) > 96 * 1024) return false;
  if (rpad > 64 || rank > 32) return false;
  return true;
}

int sb_linear(hipStream_t st, const SbLinearArgs& a, int pro, int epi) {
  if (!a.qw || !a.scales || !a.y) return TMX_ERR_ARG;
  if (!sb_linear_ok(a.M, a.K, a.N, a.G, a.lora_r, a.Rpad, pro == SB_PRO_NORM)) return TMX_ERR_SHAPE;
  if (epi == SB_EPI_SWIGLU) {
    if (pro != SB_PRO_NORM || a.N % 64) return TMX_ERR_UNSUPPORTED;
    const int per = ((a.K >> 6) + kSbWaves / 2 - 1) / (kSbWaves / 2);
    if (per <= 1) return launch_sb_a<SB_PRO_NORM, SB_EPI_SWIGLU, 1>(st, a, a.N / 64);
    if (per <= 2) return launch_sb_a<SB_PRO_NORM, SB_EPI_SWIGLU, 2>(st, a, a.N / 64);
    if (per <= 4) return launch_sb_a<SB_PRO_NORM, SB_EPI_SWIGLU, 4>(st, a, a.N / 64);
    return launch_sb_a<SB_PRO_NORM, SB_EPI_SWIGLU, 8>(st, a, a.N / 64);
  }
  // whole pairs of k-tiles and segment ends on 16 columns: 16 columns per workgroup
  if (a.K % 128 == 0 && a.seg_end[0] % 16 == 0 && a.seg_end[1] % 16 == 0) {
    if (pro == SB_PRO_NORM && epi == SB_EPI_PLAIN) return launch_sb16_t<SB_PRO_NORM, SB_EPI_PLAIN>(st, a);
    if (pro == SB_PRO_ATTN && epi == SB_EPI_RESIDUAL) return launch_sb16_t<SB_PRO_ATTN, SB_EPI_RESIDUAL>(st, a);
    if (pro == SB_PRO_PLAIN && epi == SB_EPI_RESIDUAL) return launch_sb16_t<SB_PRO_PLAIN, SB_EPI_RESIDUAL>(st, a);
    if (pro == SB_PRO_PLAIN && epi == SB_EPI_PLAIN) return launch_sb16_t<SB_PRO_PLAIN, SB_EPI_PLAIN>(st, a);
  }
  const int blocks = a.N / 32;
  if (pro == SB_PRO_NORM && epi == SB_EPI_PLAIN) return launch_sb_a<SB_PRO_NORM, SB_EPI_PLAIN, 8>(st, a, blocks);
  if (pro == SB_PRO_ATTN && epi == SB_EPI_RESIDUAL) return launch_sb_a<SB_PRO_ATTN, SB_EPI_RESIDUAL, 8>(st, a, blocks);
  if (pro == SB_PRO_PLAIN && epi == SB_EPI_RESIDUAL) return launch_sb_a<SB_PRO_PLAIN, SB_EPI_RESIDUAL, 8>(st, a, blocks);
  if (pro == SB_PRO_PLAIN && epi == SB_EPI_PLAIN) return launch_sb_a<SB_PRO_PLAIN, SB_EPI_PLAIN, 8>(st, a, blocks);
  return TMX_ERR_UNSUPPORTED;
}

// ---------------------------------------------------------------------------
// Attention of the small-batch step: gqa_decode_kernel's walk over the cache with RoPE and the
// cache write in front.  Workgroup (kv head, row, context split); the q | k | v row comes from the
// projection with its LoRA deltas applied.  Every workgroup rotates the G query heads of its kv
// head into LDS; the one whose split ends at the newest slot also rotates k, writes k and v into
// that slot and reads them back after a barrier with the rest of its positions.  Every split
// leaves (unnormalised output, max, sum) for the o projection's prologue to merge.
template <int H, int G>
__global__ __launch_bounds__(256) void sb_attn_kernel(SbAttnArgs a) {
  constexpr int NW = 4, LPP = H / 8, PPW = 64 / LPP, U = 4, NG = NW * PPW;
  __shared__ float s_m[NG][G], s_l[NG][G];
  __shared__ float s_acc[NG][G][H];
  __shared__ __align__(16) uint16_t q_s[G][H];
  const int kvh = blockIdx.x, b = blockIdx.y, split = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int pg = lane / LPP, dl = lane % LPP;
  const int step = min(*a.step, min(a.C, a.buf_len) - 1);
  const int chunk = (((step + a.nsplit) / a.nsplit) + 31) & ~31;
  const int s_begin = split * chunk;
  int s_end = s_begin + chunk;
  if (s_end > step + 1) s_end = step + 1;
  constexpr int half = H / 2;
  const int ntot = (a.N + 2 * a.Kh) * H;
  const uint16_t* row = a.qkv + (size_t)b * ntot;
  const float* tab = a.rope_tab + (size_t)b * half * 2;
  // Per-head RMSNorm (Qwen3 q_norm / k_norm: f32 with one cast, qwen3/model.py:478-484) of a head vector held as
  // one (x1, x2) pair per lane by `half` consecutive lanes, then the rotation: f32 throughout with one cast for
  // Llama3 (llama3/model.py:249-270); sin / cos and every product rounded to bf16 for Qwen3 (qwen3/model.py:432-453).
  const bool qwen = a.family == TMX_FAMILY_QWEN3;
  auto norm_rotate = [&](float x1, float x2, const uint16_t* nw, int i, float& o1, float& o2) __attribute__((always_inline)) {
    if (nw) {
      float ss = x1 * x1 + x2 * x2;
#pragma unroll
      for (int off = half / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
      const float rms = sqrtf(ss / (float)H + a.eps);
      x1 = rbf(bf2f(nw[i]) * (x1 / rms));
      x2 = rbf(bf2f(nw[i + half]) * (x2 / rms));
    }
    float sn = tab[i * 2], cs = tab[i * 2 + 1];
    if (qwen) {
      sn = rbf(sn);
      cs = rbf(cs);
      o1 = rbf(x1 * cs) - rbf(x2 * sn);
      o2 = rbf(x2 * cs) + rbf(x1 * sn);
    } else {
      o1 = x1 * cs - x2 * sn;
      o2 = x2 * cs + x1 * sn;
    }
  };
  static_assert(G * (H / 2) <= 256, "one (x1, x2) pair of the query heads per thread");
  {  // the G query heads: thread (g, i); the `half` lanes of a head are consecutive and aligned
    const bool act = tid < G * half;
    const int g = act ? tid / half : 0, i = tid % half;
    const uint16_t* qh = row + (size_t)(kvh * G + g) * H;
    float o1, o2;
    norm_rotate(act ? bf2f(qh[i]) : 0.f, act ? bf2f(qh[i + half]) : 0.f, a.q_norm_w, i, o1, o2);
    if (act) {
      q_s[g][i] = f2bf(o1);
      q_s[g][i + half] = f2bf(o2);
    }
  }
  uint16_t* kc = a.kcache + ((size_t)b * a.C * a.Kh + kvh) * H;
  uint16_t* vc = a.vcache + ((size_t)b * a.C * a.Kh + kvh) * H;
  const size_t row_stride = (size_t)a.Kh * H;
  if (s_begin <= step && step < s_end) {  // this split holds the newest slot: write it
    const int slot = step % a.C;
    if (tid < half) {
      const uint16_t* kh = row + (size_t)(a.N + kvh) * H;
      float o1, o2;
      norm_rotate(bf2f(kh[tid]), bf2f(kh[tid + half]), a.k_norm_w, tid, o1, o2);
      kc[(size_t)slot * row_stride + tid] = f2bf(o1);
      kc[(size_t)slot * row_stride + tid + half] = f2bf(o2);
    } else if (tid >= 128 && tid < 128 + H) {
      vc[(size_t)slot * row_stride + (tid - 128)] = row[(size_t)(a.N + a.Kh + kvh) * H + (tid - 128)];
    }
  }
  __syncthreads();  // q in LDS; the new cache row is visible to this workgroup's loads

  uint32_t qf[G][4];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const uint4 v = *reinterpret_cast<const uint4*>(&q_s[g][dl * 8]);
    qf[g][0] = v.x; qf[g][1] = v.y; qf[g][2] = v.z; qf[g][3] = v.w;
  }
  float m[G], l[G], acc[G][8];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = -1e30f;
    l[g] = 0.f;
#pragma unroll
    for (int d = 0; d < 8; ++d) acc[g][d] = 0.f;
  }
  const uint16_t* kbase = kc + dl * 8;
  const uint16_t* vbase = vc + dl * 8;
  const uint8_t* mrow = a.input_mask + (size_t)b * a.buf_len;
  for (int p0 = s_begin + (wave * PPW + pg) * U; p0 < s_end; p0 += NG * U) {
    uint4 kr[U], vr[U];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + u;
      ok[u] = p < s_end;
      const int pc = ok[u] ? p : p0;
      kr[u] = *reinterpret_cast<const uint4*>(kbase + (size_t)pc * row_stride);
      vr[u] = *reinterpret_cast<const uint4*>(vbase + (size_t)pc * row_stride);
      ok[u] = ok[u] && mrow[pc] != 0;
    }
    float sc[U][G];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t kw[4] = {kr[u].x, kr[u].y, kr[u].z, kr[u].w};
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float d = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          d = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, qf[g][j]),
                                              __builtin_bit_cast(bf16x2_t, kw[j]), d, false);
        d = group_sum<LPP>(d);
        sc[u][g] = ok[u] ? d * a.scale : -1e30f;
      }
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float mn = m[g];
#pragma unroll
      for (int u = 0; u < U; ++u) mn = fmaxf(mn, sc[u][g]);
      const float alpha = __expf(m[g] - mn);
      m[g] = mn;
      float pw[U], ps = 0.f;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        pw[u] = ok[u] ? __expf(sc[u][g] - mn) : 0.f;
        ps += pw[u];
      }
      l[g] = l[g] * alpha + ps;
#pragma unroll
      for (int d = 0; d < 8; ++d) acc[g][d] *= alpha;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t vw[4] = {vr[u].x, vr[u].y, vr[u].z, vr[u].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc[g][2 * j] = fmaf(pw[u], bf_lo(vw[j]), acc[g][2 * j]);
          acc[g][2 * j + 1] = fmaf(pw[u], bf_hi(vw[j]), acc[g][2 * j + 1]);
        }
      }
    }
  }
  const int gi = wave * PPW + pg;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    if (dl == 0) {
      s_m[gi][g] = m[g];
      s_l[gi][g] = l[g];
    }
#pragma unroll
    for (int d = 0; d < 8; ++d) s_acc[gi][g][dl * 8 + d] = acc[g][d];
  }
  __syncthreads();
  for (int e = tid; e < G * H; e += 256) {
    const int g = e / H, d = e % H;
    float mm = -1e30f;
#pragma unroll
    for (int i = 0; i < NG; ++i) mm = fmaxf(mm, s_m[i][g]);
    float ls = 0.f, o = 0.f;
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      const float w = __expf(s_m[i][g] - mm);
      ls += s_l[i][g] * w;
      o += s_acc[i][g][d] * w;
    }
    const size_t i = (((size_t)b * a.Kh + kvh) * a.nsplit + split) * G + g;
    a.partial[i * H + d] = o;
    if (d == 0) *reinterpret_cast<f32x2_t*>(a.partial + (size_t)a.B * a.Kh * a.nsplit * G * H + i * 2) = f32x2_t{mm, ls};
  }
}

int sb_attn_splits(int B, int Kh, int C) {
  // enough workgroups to spread the cache walk, few enough parts for the o projection to merge
  int ns = 64 / (B * Kh);
  const int by_len = (C + 127) / 128;
  if (ns > by_len) ns = by_len;
  if (ns > 8) ns = 8;
  return ns < 1 ? 1 : ns;
}

size_t sb_attn_partial_bytes(int B, int N, int Kh, int H, int C) {
  return (size_t)B * N * sb_attn_splits(B, Kh, C) * (H + 2) * sizeof(float);
}

bool sb_attn_ok(int N, int Kh, int H) {
  const int G = Kh > 0 ? N / Kh : 0;
  return Kh > 0 && N % Kh == 0 && (H == 64 || H == 128) && (G == 1 || G == 2 || G == 4);
}

int sb_attn(hipStream_t st, SbAttnArgs a, int H) {
  if (!a.qkv || !a.rope_tab || !a.kcache || !a.vcache || !a.input_mask || !a.step || !a.partial) return TMX_ERR_ARG;
  if (!sb_attn_ok(a.N, a.Kh, H)) return TMX_ERR_UNSUPPORTED;
  const int G = a.N / a.Kh;
  const dim3 grid(a.Kh, a.B, a.nsplit);
#define TMX_SB_ATTN_CASE(HH, GG) \
  if (H == HH && G == GG) { hipLaunchKernelGGL((sb_attn_kernel<HH, GG>), grid, dim3(256), 0, st, a); return check_launch(); }
  TMX_SB_ATTN_CASE(64, 1)
  TMX_SB_ATTN_CASE(64, 2)
  TMX_SB_ATTN_CASE(64, 4)
  TMX_SB_ATTN_CASE(128, 1)
  TMX_SB_ATTN_CASE(128, 2)
  TMX_SB_ATTN_CASE(128, 4)
#undef TMX_SB_ATTN_CASE
  return TMX_ERR_UNSUPPORTED;
}

}  // namespace tmx

using namespace tmx;

extern "C" int tmx_small_linear(void* stream, const void* x, const void* norm_w, float eps, int family,
                                const void* qweight, const void* scales, const void* lora_a_t, const void* lora_b,
                                const void* residual, void* y, int M, int K, int N, int G, int r, int r_pad,
                                float lora_scale, int swiglu) {
  if (!x || !qweight || !scales || !y) return TMX_ERR_ARG;
  if (lora_a_t && (!lora_b || r <= 0 || r_pad < r)) return TMX_ERR_ARG;
  if (swiglu && (!norm_w || residual || (lora_a_t && (r_pad != 32 || 2 * r > 32)))) return TMX_ERR_UNSUPPORTED;
  if (norm_w && residual) return TMX_ERR_UNSUPPORTED;
  SbLinearArgs a = {};
  a.M = M;
  a.x = (const uint16_t*)x; a.ldx = K;
  a.norm_w = (const uint16_t*)norm_w; a.eps = eps; a.family = family;
  a.qw = (const uint4*)qweight; a.scales = (const uint16_t*)scales;
  a.K = K; a.N = N; a.G = G;
  a.seg_end[0] = swiglu ? N / 2 : N; a.seg_end[1] = a.seg_end[2] = N;
  if (lora_a_t) {
    a.a_t = (const uint16_t*)lora_a_t; a.Rpad = r_pad;
    a.lora_b = (const uint16_t*)lora_b; a.lora_r = r; a.lora_ls = lora_scale;
  }
  a.residual = (const uint16_t*)residual;
  a.y = (uint16_t*)y;
  a.ldy = swiglu ? N / 2 : N;
  a.pair_off = swiglu ? N / 64 : 0;
  return sb_linear((hipStream_t)stream, a, norm_w ? 1 : 0, swiglu ? 2 : (residual ? 1 : 0));
}
