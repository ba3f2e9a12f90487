// The split-product f32 GEMM for products that leave most of the chip idle
// (k_split.h: six bf16 piece products per slab).
//
// What bounds them: latency.  A tile of a small product walks its K slabs
// one after the other, each with a barrier and the round trip through LDS
// (0.33 us a slab on a 64 x 64 tile: 8 us for K = 384, of which the MFMAs
// take 0.7).  Here the waves of a workgroup split the tile's K range between
// them: every wave computes the whole 32 x 64 tile over its own slabs, with
// its operands loaded straight into fragment layout (no LDS and no barrier
// in the loop, the next slabs in flight), and the waves' partial sums are
// added through LDS, in wave order, at the end.  Each wave splits all the
// values it reads (528 VALU beside 384 MFMA cycles a slab), which a filled
// chip would pay for; here a K = 384 product has 3 slabs per wave.
#pragma once

#include "k_gemm_x3.h"

namespace malus {
namespace k {
namespace {

// One operand's fragments: 32 T rows of its free dimension, 16 k a slab.  A
// lane (i, h) holds k = 8 h .. 8 h + 7 of rows i, 32 + i, ...: two 16-byte
// loads for a k-contiguous operand, eight 4-byte loads for the other.  Rows past
// the operand read its last one.
template <int T, bool KC>
struct DirectFrag {
  int off[T];  // byte offset at k = 0
  template <bool MAP>
  __device__ __forceinline__ void init(int x0, int X, const GemmMap& fx, const GemmMap& fk, int li, int lk) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int x = min(x0 + 32 * t + li, X - 1);
      off[t] = 4 * (map_at<MAP>(fx, x) + 8 * lk * (KC ? 1 : fk.s0));
    }
  }
#if defined(__HIP_DEVICE_COMPILE__)
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, int dk, int ks, float (&f)[T][8]) const {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      if constexpr (KC) {
        const v4f a = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, off[t], dk, 0));
        const v4f b = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, off[t] + 16, dk, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f[t][e] = a[e];
          f[t][4 + e] = b[e];
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          f[t][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off[t], dk + e * ks, 0));
      }
    }
  }
#endif
};

// C = op(A) op(B) with the operand maps and epilogues of k_gemm_x3, no split
// partials.  Tile 32 TM x 32 TN, NW waves.
template <int NW, int TM, int TN, bool TA, bool TB, bool MAP, int EPI>
__global__ __launch_bounds__(64 * NW, 2) void k_gemm_x3k(const float* __restrict__ A, const float* __restrict__ B,
                                                      float* __restrict__ C, int M, int N, int K, GemmLayouts L,
                                                      int tiles_n, const float* __restrict__ D, float* __restrict__ E) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int BM = 32 * TM, BN = 32 * TN, G = 3, R = TM * TN * 16, Q = R / NW;
  static_assert(R % NW == 0, "whole registers per wave in the final sum");
  __shared__ float part[NW][R][64];

  const int tile_m = __builtin_amdgcn_readfirstlane((int)blockIdx.x / tiles_n);
  const int m0 = tile_m * BM, n0 = ((int)blockIdx.x - tile_m * tiles_n) * BN;
  const bool grouped = MAP && L.ngroup > 1;
  const int b = grouped ? 0 : blockIdx.z;
  if (grouped && EPI != 3) {
    A = L.ga[blockIdx.z];
    B = L.gb[blockIdx.z];
    C = L.gc[blockIdx.z];
  }
  const int ba = map_at<MAP>(L.a.b, b), bb = map_at<MAP>(L.b.b, b), coff = map_at<MAP>(L.c.b, b);
  const int lane = threadIdx.x & 63, li = lane & 31, lk = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const GemmMap& fak = TA ? L.a.r : L.a.c;
  const GemmMap& fbk = TB ? L.b.c : L.b.r;
  DirectFrag<TM, !TA> da;
  DirectFrag<TN, TB> db;
  da.template init<MAP>(m0, M, TA ? L.a.c : L.a.r, fak, li, lk);
  db.template init<MAP>(n0, N, TB ? L.b.r : L.b.c, fbk, li, lk);
  const int ksa = 4 * fak.s0, ksb = 4 * fbk.s0;
  const int nk = K / BK, first = nk * wave / NW, last = nk * (wave + 1) / NW;  // this wave's slabs

  // this wave's share of the tile's sum, then registers [wave Q, (wave + 1) Q)
  // of all waves' in v
  float v[Q];
  auto product = [&](const float* Ap, const float* Bp) {
    const __amdgpu_buffer_rsrc_t ra = buffer_rsrc(Ap + ba, (unsigned)((L.ext_a - ba) * 4));
    const __amdgpu_buffer_rsrc_t rb = buffer_rsrc(Bp + bb, (unsigned)((L.ext_b - bb) * 4));
    v16f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = v16f{0};
    KCursor<MAP> ka, kb;
    ka.init(fak, min(first, nk - 1) * BK);
    kb.init(fbk, min(first, nk - 1) * BK);
    float fa[G][TM][8], fb[G][TN][8];
    int slab = first;
    auto load = [&](int g) {  // past the last slab: that one again (values no product uses)
      da.load(ra, ka.bytes(fak), ksa, fa[g]);
      db.load(rb, kb.bytes(fbk), ksb, fb[g]);
      if (++slab < last) {
        ka.advance(fak);
        kb.advance(fbk);
      }
    };
#pragma unroll
    for (int g = 0; g < G; ++g) load(g);
    for (int s = first; s < last; s += G) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if (s + g < last) {
          Split3 a[TM], bs[TN];
#pragma unroll
          for (int i = 0; i < TM; ++i) a[i] = split3(fa[g][i]);
#pragma unroll
          for (int j = 0; j < TN; ++j) bs[j] = split3(fb[g][j]);
          load(g);
          x3_slab<false, TM, TN>(a, bs, acc);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) part[wave][(i * TN + j) * 16 + r][lane] = acc[i][j][r];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q) v[q] = part[0][wave * Q + q][lane];
#pragma unroll
    for (int w = 1; w < NW; ++w)
#pragma unroll
      for (int q = 0; q < Q; ++q) v[q] += part[w][wave * Q + q][lane];
    if (EPI == 3) __syncthreads();  // the next group's partials go to the same place
  };
  // f(q, live, offset in C) for this wave's registers
  auto for_each = [&](auto&& f) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int reg = wave * Q + q, ij = reg >> 4, r = reg & 15;
      const int m = m0 + 32 * (ij / TN) + 8 * (r >> 2) + 4 * lk + (r & 3), n = n0 + 32 * (ij % TN) + li;
      f(q, m < M && n < N, coff + map_at<MAP>(L.c.r, m) + map_at<MAP>(L.c.c, n));
    }
  };
  if constexpr (EPI == 3) {
    float tot[Q];
    for (int g = 0; g < L.ngroup; ++g) {
      product(L.ga[g], L.gb[g]);
      for_each([&](int q, bool live, int o) {
        tot[q] = g == 0 ? (D && live ? D[o] + v[q] : v[q]) : tot[q] + v[q];
      });
    }
    for_each([&](int q, bool live, int o) {
      if (live) C[o] = tot[q];
    });
  } else {
    product(A, B);
    for_each([&](int q, bool live, int o) {
      if (!live) return;
      float x = v[q];
      if (EPI == 2) x = gelu_bwd(E[o], x);
      C[o] = D ? D[o] + x : x;
      if (EPI == 1) E[o] = gelu_fwd(x);
    });
  }
#endif
}

}  // namespace
}  // namespace k
}  // namespace malus
