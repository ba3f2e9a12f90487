// Device helpers shared by the flash attention kernels (k_flash.hip on the
// FP32 MFMA, k_flash_planes.hip on the bf16 MFMA).
#pragma once

#include "common.h"
#include "k_split.h"

namespace malus {
namespace k {

// The kernels of k_flash_planes.hip.  planes: 3, f32 products as split bf16
// pieces; 1, operands rounded to bf16 (autocast).  qkv_bf16: Q, K, V and
// their gradients stored in bf16 (planes 1 only).
void flash_planes_fwd(size_t hs, bool causal, int planes, bool qkv_bf16, const float* Q, const float* K, const float* V,
                      const float* scale, float* O, int ldo, int H, float* lse, int T, int BH, hipStream_t s);
void flash_planes_bwd(size_t hs, bool causal, int planes, bool qkv_bf16, const FlashBwd& a, int ldo, int H, int T, int BH,
                      hipStream_t s);

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

// Bits 2 and 3 of a row swapped, and the row that register r of lane half
// lk then holds: the row order that feeds an accumulator to the next product.
__device__ __forceinline__ int perm_row(int x) { return x ^ ((((x >> 2) ^ (x >> 3)) & 1) * 12); }
__device__ __forceinline__ int perm_index(int r, int lk) { return 16 * (r >> 3) + 8 * lk + (r & 7); }

// 8 consecutive floats (16-byte aligned)
__device__ __forceinline__ void load8(const float* __restrict__ p, float (&v)[8]) {
  const v4f a = *reinterpret_cast<const v4f*>(p), b = *reinterpret_cast<const v4f*>(p + 4);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = a[e];
    v[4 + e] = b[e];
  }
}

// A head's row `row` of a [B*T, H*HS] tensor (O, dO) or of [B*H, T, HS].
__device__ __forceinline__ const float* head_row(const float* base, int bh, int H, int T, int ld, int hs, int row) {
  return base + (size_t)(bh / H) * T * ld + (size_t)(bh % H) * hs + (size_t)row * ld;
}

}  // namespace
}  // namespace k
}  // namespace malus
