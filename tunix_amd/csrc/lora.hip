// LoRA weight sync between rollouts: the trainer's adapters (row-major, the trainer's precision) into the layout
// the projection kernels read, 64 tensors per launch.
//
// Stands where the reference merges the new nnx.LoRAParam leaves into the sampler's state
// (tunix/generate/sampler.py:361-392: cast to the rollout precision, then replace).
#include "tmx_kernels.h"

namespace tmx {

constexpr int kLoraBatch = 64;       // tensors per launch: their descriptors travel as kernel arguments
constexpr int kLoraPerBlock = 2048;  // elements per workgroup: 8 per thread

struct LoraPackArgs {
  tmx_lora_pack_desc d[kLoraBatch];
  int first_block[kLoraBatch + 1];
  int n;
};

__device__ __forceinline__ float lora_value(const void* src, int dtype, size_t i) {
  if (dtype == TMX_DTYPE_F32) return reinterpret_cast<const float*>(src)[i];
  if (dtype == TMX_DTYPE_BF16) return bf2f(reinterpret_cast<const uint16_t*>(src)[i]);
  return (float)reinterpret_cast<const _Float16*>(src)[i];
}

// A sync moves a few KB to a few MB per tensor, so what it costs is launches and the host's work per tensor, not
// bytes.  A workgroup finds its tensor in the descriptors (6 comparisons) and moves 2048 elements; a thread owns 8
// elements that are adjacent in the destination: 8 rows of one column of A (16 bytes of a fragment), or 8 consecutive
// columns of B, whose stores are 16 bytes wide where the widths allow it.
__global__ __launch_bounds__(256) void lora_pack_kernel(LoraPackArgs a) {
  int lo = 0, hi = a.n;  // first_block[lo] <= blockIdx.x < first_block[lo + 1]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if ((int)blockIdx.x >= a.first_block[mid]) lo = mid;
    else hi = mid;
  }
  const tmx_lora_pack_desc& d = a.d[lo];
  const int i0 = ((int)blockIdx.x - a.first_block[lo]) * kLoraPerBlock + threadIdx.x * 8;  // host: rows * cols < 2^30
  const int rows = d.rows, cols = d.cols, col0 = d.col0, dtype = d.dtype;
  uint16_t* dst = reinterpret_cast<uint16_t*>(d.dst);
  float v[8];
  uint4 p;
  if (d.is_a) {
    // [K, r] -> fragment order (see tmx_qlora_linear): rows k .. k + 7, k a multiple of 8, of a column are adjacent
    const int k = (i0 >> 3) / cols * 8, c = (i0 >> 3) % cols;
    if (k >= rows) return;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = lora_value(d.src, dtype, (size_t)(k + j) * cols + c);
    p.x = pack_bf2(v[0], v[1]); p.y = pack_bf2(v[2], v[3]);
    p.z = pack_bf2(v[4], v[5]); p.w = pack_bf2(v[6], v[7]);
    const int col = col0 + c, kb = k >> 6, t = (k & 63) >> 4, h = (k & 15) >> 3;
    *reinterpret_cast<uint4*>(dst + ((((size_t)kb * (d.ld >> 5) + (col >> 5)) * 4 + t) * 64 + 32 * h + (col & 31)) * 8) = p;
    return;
  }
  // [r, n] -> columns col0 .. col0 + n - 1 of [r, ld]
  const int total = rows * cols;
  if (i0 >= total) return;
  if (((cols | col0 | d.ld) & 7) == 0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = lora_value(d.src, dtype, (size_t)i0 + j);
    p.x = pack_bf2(v[0], v[1]); p.y = pack_bf2(v[2], v[3]);
    p.z = pack_bf2(v[4], v[5]); p.w = pack_bf2(v[6], v[7]);
    *reinterpret_cast<uint4*>(dst + (size_t)(i0 / cols) * d.ld + col0 + i0 % cols) = p;
    return;
  }
  for (int i = i0; i < i0 + 8 && i < total; ++i)
    dst[(size_t)(i / cols) * d.ld + col0 + i % cols] = f2bf(lora_value(d.src, dtype, i));
}

}  // namespace tmx

using namespace tmx;

extern "C" int tmx_lora_pack(void* stream, const tmx_lora_pack_desc* descs_host, int n) {
  if (n < 0 || (n > 0 && !descs_host)) return TMX_ERR_ARG;
  for (int i = 0; i < n; ++i) {
    const tmx_lora_pack_desc& d = descs_host[i];
    if (!d.src || !d.dst) return TMX_ERR_ARG;
    if (d.dtype != TMX_DTYPE_F32 && d.dtype != TMX_DTYPE_BF16 && d.dtype != TMX_DTYPE_F16) return TMX_ERR_UNSUPPORTED;
    if (d.rows <= 0 || d.cols <= 0 || d.col0 < 0 || (size_t)d.col0 + d.cols > (size_t)d.ld ||
        (size_t)d.rows * d.cols >= (1u << 30))
      return TMX_ERR_SHAPE;
    if (d.is_a && (d.rows % 64 || d.ld % 32)) return TMX_ERR_SHAPE;
  }
  for (int i0 = 0; i0 < n; i0 += kLoraBatch) {
    LoraPackArgs a;
    a.n = n - i0 < kLoraBatch ? n - i0 : kLoraBatch;
    int blocks = 0;
    for (int i = 0; i < a.n; ++i) {
      a.d[i] = descs_host[i0 + i];
      a.first_block[i] = blocks;
      blocks += (a.d[i].rows * a.d[i].cols + kLoraPerBlock - 1) / kLoraPerBlock;
    }
    a.first_block[a.n] = blocks;
    hipLaunchKernelGGL(lora_pack_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, a);
    const int rc = check_launch();
    if (rc != TMX_OK) return rc;
  }
  return TMX_OK;
}
