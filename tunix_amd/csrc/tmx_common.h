// Device-side helpers shared by the gfx950 kernels: bf16 bit handling, wave64
// reductions, MFMA fragment types and the status codes of the C ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tmx.h"

namespace tmx {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr float kMask = -2.3819763e38f;  // the reference's K_MASK

__device__ __forceinline__ float bf2f(uint16_t b) {
  return __uint_as_float(((uint32_t)b) << 16);
}
__device__ __forceinline__ float bf_lo(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf_hi(uint32_t p) { return __uint_as_float(p & 0xFFFF0000u); }

// float -> bf16, round to nearest even (hardware conversion on gfx950).
__device__ __forceinline__ uint16_t f2bf(float f) {
  return __builtin_bit_cast(uint16_t, (__bf16)f);
}
// Round a float to the nearest bf16 and return it widened again.
__device__ __forceinline__ float rbf(float f) { return bf2f(f2bf(f)); }

__device__ __forceinline__ uint32_t pack_bf2(float lo, float hi) {
  f32x2_t v = {lo, hi};
  bf16x2_t b = __builtin_convertvector(v, bf16x2_t);
  return __builtin_bit_cast(uint32_t, b);
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
// Butterfly sum over the wave (lane distances 32, 16, 8, 4, 2, 1), every lane gets the total.  Six vector instructions
// and adds instead of six trips through the LDS permute unit (about 0.3 us per sum at one wave per SIMD): half-wave and
// row swaps, then rotations within rows of 16, which are the distance-8 and -4 partners once the sums repeat with period
// 16 and 8.  Same pairs in the same order as the shuffle form.
__device__ __forceinline__ float wave_sum(float v) {
  {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
  {
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
  v += dpp_f<0x128>(v);  // row_ror:8
  v += dpp_f<0x124>(v);  // row_ror:4
  v += dpp_f<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_f<0xB1>(v);   // quad_perm [1,0,3,2]
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// Sum over aligned groups of LPP (8 or 16) lanes; every lane gets the total.
template <int LPP>
__device__ __forceinline__ float group_sum(float v) {
  v += dpp_f<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_f<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_f<0x141>(v);  // row_half_mirror
  if (LPP == 16) v += dpp_f<0x140>(v);  // row_mirror
  return v;
}

// Sum over a workgroup of NW waves; every thread receives the total.
template <int NW>
__device__ __forceinline__ float block_sum(float v, float* smem /* >= NW floats */) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) smem[w] = v;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < NW; ++i) t += smem[i];
  return t;
}

// Row of MFMA 32x32 accumulator register r held by `lane` (column = lane % 32).
__device__ __forceinline__ int acc_row(int r, int lane) {
  return (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
}

// Expand one 32-bit word (8 nibbles, element j = 2 (i % 4) + i / 4 for nibble i) into the 8 bf16 B-operand values of
// one MFMA step: bf16((u - 8) * s), (4 + 8 significant bits) exact as a float and rounded once, for every scale whose -8 s is
// finite.  A byte 0x0U read as an fp8 number (E4M3, bias 7) is U * 2^-9 for every U in 0..15 (below 8 subnormal, from 8 on
// with exponent field 1), so one v_cvt_scalef32_pk_f32_fp8 with the scale 2^9 widens two nibbles of a masked word: 19
// instructions per word.  Widening and scaling masked nibbles as f16 subnormals by v_fma_mix_f32 takes 17, but needs s * 2^24
// finite; it is 0.4 to 0.8 % of a decode step faster (64 rows of the 8B shape, 8 layers, 64 tokens: 74.6 against 75.0 ms, 23 rows 42.0
// against 42.4), and a branch per tile for the scales it cannot take costs more than it gains (77.8, 43.6 ms).
struct NibbleScale { float s, m8s; };  // s, -8 s
__device__ __forceinline__ NibbleScale nibble_scale(float s) { return {s, -8.f * s}; }
typedef float f32x2_t __attribute__((ext_vector_type(2)));
// The four registers of the B operand (register p: elements 2 p, 2 p + 1 = nibbles p, p + 4 of word d) in four parts, for loops
// that spread them between MFMAs: part 0 widens the even nibbles and makes register 0, part 1 register 2, part 2 widens the
// odd ones and makes register 1, part 3 register 3.
struct NibblePairs { f32x2_t a, b; };
template <int P>
__device__ __forceinline__ void dequant_part(uint32_t d, const NibbleScale& sc, NibblePairs& n, u32x4_t& r) {
  if constexpr (P % 2 == 0) {
    const uint32_t w = (P ? d >> 4 : d) & 0x0F0F0F0Fu;
    n.a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w, 512.f, false);
    n.b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w, 512.f, true);
    r[P / 2] = pack_bf2(fmaf(n.a.x, sc.s, sc.m8s), fmaf(n.b.x, sc.s, sc.m8s));
  } else {
    r[P / 2 + 2] = pack_bf2(fmaf(n.a.y, sc.s, sc.m8s), fmaf(n.b.y, sc.s, sc.m8s));
  }
}
__device__ __forceinline__ bf16x8_t dequant_word(uint32_t d, const NibbleScale& sc) {
  NibblePairs n;
  u32x4_t r;
  dequant_part<0>(d, sc, n, r);
  dequant_part<1>(d, sc, n, r);
  dequant_part<2>(d, sc, n, r);
  dequant_part<3>(d, sc, n, r);
  return __builtin_bit_cast(bf16x8_t, r);
}

// A copy the compiler does not see through: it happens here, so the registers of v are free for the load that follows
// (otherwise the copy moves to the end of the loop, behind that load, and waits for it).
__device__ __forceinline__ uint32_t moved(uint32_t v) {
  uint32_t r;
  asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}
__device__ __forceinline__ u32x4_t moved(u32x4_t v) { return u32x4_t{moved(v.x), moved(v.y), moved(v.z), moved(v.w)}; }

template <int V>
struct IC { static constexpr int value = V; };

// f(IC<0>{}), ..., f(IC<N - 1>{}): a loop whose index is a compile-time constant
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(IC<I>{});
    static_for<N, I + 1>(f);
  }
}

// Raw buffer descriptor over `bytes` bytes at p (loads take a per-lane and a scalar byte offset).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}

// 1 KiB from global memory straight into LDS (buffer_load ... lds): lane i's 16 bytes at byte
// offset voffset + soffset of the buffer land at dst + 16 i; dst and soffset are wave-uniform.
// Counted by vmcnt like any other load.
__device__ __forceinline__ void load_row_to_lds(__amdgpu_buffer_rsrc_t r, void* dst, int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voffset, soffset, 0, 0);
}
// the same with the non-temporal cache policy, for data that is read once
__device__ __forceinline__ void load_row_to_lds_nt(__amdgpu_buffer_rsrc_t r, void* dst, int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voffset, soffset, 0, 2);
}


inline int check_launch() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? TMX_OK : TMX_ERR_LAUNCH;
}

}  // namespace tmx
