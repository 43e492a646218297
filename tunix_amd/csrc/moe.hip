// Mixture-of-experts routing for decode (Qwen3 MoE).
//
// Replaces MoELayer.__call__'s routing, tunix/models/qwen3/model.py:895-902:
//   scores = bf16(x . router)  -> f32;  p = softmax(scores)
//   weights, experts = lax.top_k(p, k)        (ties: lower expert id first)
//   weights = bf16(weights / sum(weights))
// One workgroup per token, or per 16 where there are many.  The expert matrices themselves are multiplied by
// moe_stream_kernel (qlinear.hip); the weighted sum over a token's experts is taken by the
// row kernel that also adds the residual and normalises (glue.hip).
#include "tmx_router.h"

namespace tmx {

__global__ __launch_bounds__(kRouterThreads) void moe_router_kernel(RouterArgs a) {
  extern __shared__ __align__(16) float sm[];
  const int b = blockIdx.x;
  RouterStep ring[2];
  router_load(a, 0, 0, ring[0]);
  router_load(a, 1, 0, ring[1]);
  uint16_t* xs = reinterpret_cast<uint16_t*>(sm);
  for (int d = threadIdx.x; d < moe_router_steps(a.D) * 256; d += kRouterThreads) xs[d] = d < a.D ? a.x[(size_t)b * a.D + d] : (uint16_t)0;
  __syncthreads();
  moe_route_token(a, sm, b, ring);
}

// The same for 16 tokens a workgroup (many rows): the router leaves L2 once for all of them.  A wave adds up its share of the
// rows of the router for all 16, the shares meet in LDS, and every wave finishes two tokens.
constexpr int kRouterTile = 16;
inline size_t moe_router_rows_lds(int E) { return (size_t)4 * kRouterTile * E * 4 + (size_t)kRouterTile * E * 4; }
__global__ __launch_bounds__(kRouterThreads) void moe_router_rows_kernel(RouterArgs a, int B) {
  extern __shared__ __align__(16) float sm[];
  float* prob = sm;                        // [16][E]
  float* part = sm + kRouterTile * a.E;    // [4][16][E]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4;
  const int b0 = blockIdx.x * kRouterTile, steps = moe_router_steps(a.D);
  const uint16_t* xrow = a.x + (size_t)min(b0 + (lane & 15), B - 1) * a.D;
  for (int e0 = 0; e0 < a.E; e0 += 128) {
    RouterStep ring[2];
    u32x4_t x[2];
    auto load = [&](int step, auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      router_load(a, step, e0, ring[i]);
      x[i] = *reinterpret_cast<const u32x4_t*>(xrow + min(step * 256 + wave * 32 + q * 8, a.D - 8));
    };
    f32x4_t acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    load(0, IC<0>{});
    load(1, IC<1>{});
    for (int s0 = 0; s0 < steps; s0 += 2)
      static_for<2>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        if ((s0 + i) * 256 + wave * 32 + q * 8 >= a.D) x[i] = u32x4_t{0u, 0u, 0u, 0u};  // (a select, not a branch)
        router_step(ring[i], __builtin_bit_cast(bf16x8_t, x[i]), acc);
        load(s0 + i + 2, ic);
      });
    // waves 4..7 leave theirs, waves 0..3 add their own and leave the sum
    const int e = e0 + (lane & 15) * 8;
    for (int turn = 0; turn < 2; ++turn) {
      if (wave / 4 == 1 - turn && e < a.E)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          f32x4_t* d = reinterpret_cast<f32x4_t*>(part + ((size_t)(wave & 3) * kRouterTile + 4 * q + r) * a.E + e);
          f32x4_t lo = {acc[0][r], acc[1][r], acc[2][r], acc[3][r]}, hi = {acc[4][r], acc[5][r], acc[6][r], acc[7][r]};
          if (turn) { lo += d[0]; hi += d[1]; }
          d[0] = lo; d[1] = hi;
        }
      __syncthreads();
    }
  }
  for (int i = tid; i < kRouterTile * a.E; i += kRouterThreads) {
    float s = 0.f;
#pragma unroll
    for (int g = 0; g < 4; ++g) s += part[(size_t)g * kRouterTile * a.E + i];
    prob[i] = rbf(s);
  }
  __syncthreads();
  float* sel = part + wave * 64;  // [top_k] (the partial scores are spent)
  for (int t = wave; t < kRouterTile && b0 + t < B; t += kRouterWaves) {
    float* p = prob + t * a.E;
    router_softmax(p, a.E, lane);
    const int b = b0 + t;
    // the place of expert e: larger probabilities, and equal ones of a lower id.  As integers (they are not negative), those are
    // the ones above v - 1 in front of its group of four, above v behind, and in the group the equal ones are looked up.  Two
    // experts of a lane at a time share the broadcast reads, whose latency is what this takes
    auto bits = [](float v) { return __float_as_int(v); };
    for (int e1 = lane; e1 < (a.E + 63) / 64 * 64; e1 += 128) {
      const int ee[2] = {min(e1, a.E - 1), min(e1 + 64, a.E - 1)}, v[2] = {bits(p[ee[0]]), bits(p[ee[1]])};
      int place[2] = {0, 0};
#pragma unroll 8
      for (int j = 0; j < a.E; j += 4) {
        const f32x4_t u = *reinterpret_cast<const f32x4_t*>(p + j);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int t = v[k] - (j + 3 < ee[k] ? 1 : 0);
          place[k] += (bits(u[0]) > t) + (bits(u[1]) > t) + (bits(u[2]) > t) + (bits(u[3]) > t);
        }
      }
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        for (int j = ee[k] & ~3; j < ee[k]; ++j) place[k] += bits(p[j]) == v[k];
        if (e1 + 64 * k < a.E && place[k] < a.top_k) {
          a.expert_of[(size_t)b * a.top_k + place[k]] = ee[k];
          sel[place[k]] = p[ee[k]];
        }
      }
    }
    // (one wave: its LDS writes are read in order)
    if (lane < a.top_k) {
      float wsum = 0.f;
      for (int j = 0; j < a.top_k; ++j) wsum += sel[j];
      a.weight_of[(size_t)b * a.top_k + lane] = rbf(sel[lane] / wsum);
    }
  }
}

// More tokens than CUs: 16 a workgroup, in a launch of their own.  2048 x 128, us with a launch each: 256 tokens 12.4 one a workgroup,
// 16.8 so; 512 19 and 16.9; 1024 33 and 16.9 (and the row kernel in front is the one for finished rows).
bool moe_route_rows_ok(const RouterArgs& a, int B) {
  return B > 256 && a.D % 8 == 0 && moe_router_rows_lds(a.E) <= 60000 && moe_router_ok(a.D, a.E);
}

int moe_route(hipStream_t st, const RouterArgs& a, int B) {
  if (!a.x || !a.w || !a.expert_of || !a.weight_of) return TMX_ERR_ARG;
  if (B <= 0 || a.D <= 0 || a.D % 4 || a.E <= 0 || a.E % 8 || a.top_k <= 0 || a.top_k > 64 || a.top_k > a.E)
    return TMX_ERR_SHAPE;
  if (!moe_router_ok(a.D, a.E)) return TMX_ERR_SHAPE;
  if (moe_route_rows_ok(a, B)) {
    hipLaunchKernelGGL(moe_router_rows_kernel, dim3((B + kRouterTile - 1) / kRouterTile), dim3(kRouterThreads),
                       moe_router_rows_lds(a.E), st, a, B);
    return check_launch();
  }
  hipLaunchKernelGGL(moe_router_kernel, dim3(B), dim3(kRouterThreads), moe_router_lds(a.D, a.E), st, a);
  return check_launch();
}

}  // namespace tmx

using namespace tmx;

extern "C" int tmx_moe_route(void* stream, const void* x, const void* router_w, int B, int D, int E,
                             int top_k, int32_t* expert_of, float* weight_of) {
  RouterArgs a = {};
  a.x = (const uint16_t*)x;
  a.w = (const uint16_t*)router_w;
  a.D = D; a.E = E; a.top_k = top_k;
  a.expert_of = expert_of;
  a.weight_of = weight_of;
  return moe_route((hipStream_t)stream, a, B);
}

extern "C" int tmx_moe_experts(void* stream, const void* x, int ldx, const void* qweight, const void* scales,
                               const int32_t* expert_of, int P, int top_k, int E, int K, int N, int G,
                               int down, void* out, int ldo) {
  MoeArgs a = {};
  a.x = (const uint16_t*)x;
  a.ldx = ldx;
  a.qw = (const uint4*)qweight;
  a.scales = (const uint16_t*)scales;
  a.qw_stride = (size_t)K * N / 32;            // 16-byte words of one expert's q4t matrix
  a.sc_stride = (size_t)(K / (G > 0 ? G : 1)) * N;
  a.expert_of = expert_of;
  a.P = P; a.top_k = top_k;
  a.K = K; a.N = N; a.G = G;
  a.out = (uint16_t*)out;
  a.ldo = ldo;
  if (G <= 0) return TMX_ERR_SHAPE;
  return moe_experts((hipStream_t)stream, a, E, down != 0);
}
