// Routing of one token by one workgroup of kRouterThreads threads (shared by the stand-alone router kernel
// and the row kernel that produces the router's input).
//
// tunix/models/qwen3/model.py:895-902:
//   scores = bf16(x . router)  -> f32;  p = softmax(scores)
//   weights, experts = lax.top_k(p, k)        (ties: lower expert id first)
//   weights = bf16(weights / sum(weights))
#pragma once
#include "tmx_kernels.h"

namespace tmx {

constexpr int kRouterThreads = 512, kRouterWaves = kRouterThreads / 64;

// What the routing of a token was first given: fixes which shapes are taken.
inline size_t moe_router_floats(int D, int E) { return (size_t)D + 33 * (size_t)E; }
inline bool moe_router_ok(int D, int E) { return moe_router_floats(D, E) * sizeof(float) <= 60000; }
// Bytes of LDS the routing of a token needs: x row, whole steps | probabilities [E] | partial scores [kRouterWaves][E]
__host__ __device__ inline int moe_router_steps(int D) { return (D + 511) / 512 * 2; }  // of 256 rows, in pairs
inline size_t moe_router_lds(int D, int E) { return (size_t)moe_router_steps(D) * 512 + (size_t)(1 + kRouterWaves) * E * 4; }

// scores = x . router on the 16 x 16 x 32 MFMA, 256 rows of the router a step: a wave takes 32 of them for 128 experts.  Lane (n, q)
// loads rows 8 q .. + 7 of experts 8 n .. + 7, 16 bytes each; 32 permutes pair the rows up, and the eight words of expert 8 n + j are
// the B operand of MFMA j.  So the router is read as it lies, and up to 16 tokens share it.  As products of pairs
// on the vector ALU, unpacking, it was 2.8 us of issue for 2048 x 128 and one token, here 1.2; the launch by itself 11.7 -> 9.7 us,
// 8 layers and 48 steps at 32 tokens with their prompts 72.5 -> 70.6 ms.
struct RouterStep { u32x4_t w[8]; };
__device__ __forceinline__ void router_load(const RouterArgs& a, int step, int e0, RouterStep& s) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int e = e0 + (lane & 15) * 8, d0 = step * 256 + wave * 32 + (lane >> 4) * 8;
  const uint16_t* src = a.w + (e < a.E ? e : 0);
#pragma unroll
  for (int i = 0; i < 8; ++i)  // rows past D: the last one, times zero
    s.w[i] = *reinterpret_cast<const u32x4_t*>(src + (size_t)min(d0 + i, a.D - 1) * a.E);
}
// acc[j][r] += token 4 q + r of the tile times expert 8 n + j; x: this lane's fragment (token n, rows 8 q .. + 7 of the wave's)
__device__ __forceinline__ void router_step(const RouterStep& s, bf16x8_t x, f32x4_t (&acc)[8]) {
  static_for<8>([&](auto jc) __attribute__((always_inline)) {
    constexpr int j = decltype(jc)::value;
    u32x4_t b;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      b[r] = __builtin_amdgcn_perm(s.w[2 * r + 1][j / 2], s.w[2 * r][j / 2], j % 2 ? 0x07060302u : 0x05040100u);
    acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, __builtin_bit_cast(bf16x8_t, b), acc[j], 0, 0, 0);
  });
}

// scores -> probabilities of one token, by one wave
__device__ __forceinline__ void router_softmax(float* prob, int E, int lane) {
  float mx = -INFINITY;
  for (int e = lane; e < E; e += 64) mx = fmaxf(mx, prob[e]);
  mx = wave_max(mx);
  float se = 0.f;
  for (int e = lane; e < E; e += 64) {
    const float ex = expf(prob[e] - mx);
    prob[e] = ex;
    se += ex;
  }
  se = wave_sum(se);
  for (int e = lane; e < E; e += 64) prob[e] = prob[e] / se;
}
// How many of experts j .. j + 3 come in front of expert e of probability v
__device__ __forceinline__ int router_ahead(const float* prob, int j, float v, int e) {
  const float4 u = *reinterpret_cast<const float4*>(prob + j);
  return ((u.x > v || (u.x == v && j < e)) ? 1 : 0) + ((u.y > v || (u.y == v && j + 1 < e)) ? 1 : 0) +
         ((u.z > v || (u.z == v && j + 2 < e)) ? 1 : 0) + ((u.w > v || (u.w == v && j + 3 < e)) ? 1 : 0);
}

// sm: moe_router_lds(D, E) bytes that begin with the token's normed hidden state (bf16, zeros up to a whole step),
// visible to every thread (the caller has synchronised).  Writes expert_of / weight_of of token b.  ring: the first two
// steps of the router for experts 0 .. 127, which the caller has requested.
__device__ __forceinline__ void moe_route_token(const RouterArgs& a, float* sm, const int b, RouterStep (&ring)[2]) {
  const uint16_t* xrow = reinterpret_cast<const uint16_t*>(sm);
  const int steps = moe_router_steps(a.D);
  float* prob = sm + steps * 128;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float* part = prob + a.E;  // [kRouterWaves][E]
  for (int e0 = 0; e0 < a.E; e0 += 128) {
    if (e0) {
      router_load(a, 0, e0, ring[0]);
      router_load(a, 1, e0, ring[1]);
    }
    f32x4_t acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < steps; s0 += 2)
      static_for<2>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        u32x4_t x = *reinterpret_cast<const u32x4_t*>(xrow + (s0 + i) * 256 + wave * 32 + (lane >> 4) * 8);
        if (lane & 15) x = u32x4_t{0u, 0u, 0u, 0u};
        router_step(ring[i], __builtin_bit_cast(bf16x8_t, x), acc);
        router_load(a, s0 + i + 2, e0, ring[i]);  // (past the last step: the router's last row)
      });
    if (lane < 16 && e0 + lane * 8 < a.E)
#pragma unroll
      for (int j = 0; j < 8; ++j) part[wave * a.E + e0 + lane * 8 + j] = acc[j][0];
  }
  __syncthreads();
  for (int e = tid; e < a.E; e += kRouterThreads) {
    float s = 0.f;
#pragma unroll
    for (int g = 0; g < kRouterWaves; ++g) s += part[g * a.E + e];
    prob[e] = rbf(s);
  }
  __syncthreads();
  // softmax by the first wave alone (E / 64 values per lane; the sums run over the experts in the same fixed
  // order on every call)
  if (wave == 0) router_softmax(prob, a.E, lane);
  __syncthreads();
  // top-k by rank: expert e comes after every expert with a larger probability and after the equal ones with a
  // lower id (lax.top_k's order), so its place is the count of those; four threads per expert count over a quarter of the
  // probabilities each -- no round depends on the one before, as k repeated arg-max searches would
  float* sel = part;  // [top_k] the chosen probabilities by place (the partial scores are spent)
  for (int i = tid; i < (a.E * 4 + 63) / 64 * 64; i += kRouterThreads) {  // (whole waves: E % 8 == 0)
    const int e = min(i >> 2, a.E - 1), quarter = i & 3;
    const float v = prob[e];
    int place = 0;
    for (int j = quarter * 4; j < a.E; j += 16) place += router_ahead(prob, j, v, e);
    place += __shfl_xor(place, 1, 64);
    place += __shfl_xor(place, 2, 64);
    if (quarter == 0 && i >> 2 < a.E && place < a.top_k) {
      a.expert_of[(size_t)b * a.top_k + place] = e;
      sel[place] = v;
    }
  }
  __syncthreads();
  if (tid < a.top_k) {
    float wsum = 0.f;
    for (int j = 0; j < a.top_k; ++j) wsum += sel[j];  // in the order of the places
    a.weight_of[(size_t)b * a.top_k + tid] = rbf(sel[tid] / wsum);
  }
}

}  // namespace tmx
