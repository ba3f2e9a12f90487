// The bf16 GEMM (autocast) on f32 operands with each value rounded once per
// workgroup and stored in LDS as bf16.
//
// What bounds it: moving the f32 operands.  A kernel that stages f32 in LDS
// reads every fragment back at 4 bytes a value and rounds it in each wave;
// at one MFMA per 32 x 32 x 16 block the LDS reads then take several times
// the matrix time.  Here a 32-deep stage is loaded into registers, rounded
// and stored as bf16: half the LDS bytes, read as fragments ready for the
// MFMA by wide wave tiles.  What is left at the limit are the f32 loads (64 B
// per clock and CU for a 256 x 256 tile at the MFMA rate, the most the CU's
// cache gives) and the LDS (130 KB per stage and 1024 MFMA cycles).
// Measured, 8192 x 4096 x 1024 (256 x 256): 214 -> 121 us; 8192 x 1024 x
// 4096, B transposed (256 x 128): 251 -> 116 us; four waves of 128 x 128 instead
// of eight of 128 x 64: the same with spills; 128 x 128 tiles: 191 and 156 us.
//
// Schedule of one 32-deep stage s (three LDS stages, one barrier each): while the
// MFMAs of its first 16-deep slab run, the second slab's fragments are read;
// during the second slab's, the next stage's first fragments (that stage
// was written a stage ago).  Between the MFMAs the wave rounds and stores
// stage s + 2 from its staging registers and loads stage s + 2 + G into them.
// The sums run over the k slabs upwards in one MFMA each, as in
// k_sgemm_dma, so the values are the same for the same K split.
#pragma once

#include "k_gemm_x3.h"

namespace malus {
namespace k {
namespace {

// Dense operands (C = op(A) op(B) (+ D) or split-K partials); the host
// guarantees K % 16 == 0, 16-byte aligned k-contiguous rows and byte offsets
// below 2^31.  WM x WN waves of TM x TN accumulators.
template <int WM, int WN, int TM, int TN, bool TA, bool TB, int G>
__global__ __launch_bounds__(64 * WM * WN, 2) void k_gemm_bf(const float* __restrict__ A, const float* __restrict__ B,
                                                         float* __restrict__ C, int M, int N, int K, GemmLayouts L,
                                                         int k_chunk, int tiles_n, long split_stride,
                                                         const float* __restrict__ D) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NT = 64 * WM * WN, BM = 32 * WM * TM, BN = 32 * WN * TN;
  using StA = X3Stage<BM, NT, !TA, 1>;
  using StB = X3Stage<BN, NT, TB, 1>;
  constexpr int UA = StA::U, UB = StB::U, U = UA + UB;
  constexpr int PA = StA::PLANE, PB = StB::PLANE, SLAB = PA + PB, STAGE = 2 * SLAB;
  __shared__ __attribute__((aligned(1024))) char lds[3 * STAGE];

  // XCD-contiguous work, as in k_sgemm_dma
  const int nt = gridDim.x, ns = gridDim.y;
  int tile, split;
  if (ns == 1) {
    tile = blockIdx.x;
    if ((nt & 7) == 0) tile = (tile & 7) * (nt >> 3) + (tile >> 3);
    split = 0;
  } else {
    const int w = xcd_range(blockIdx.x + nt * blockIdx.y, nt * ns);
    split = __builtin_amdgcn_readfirstlane(w / nt);
    tile = w - split * nt;
  }
  const int tile_m = __builtin_amdgcn_readfirstlane(tile / tiles_n);
  const int m0 = tile_m * BM, n0 = (tile - tile_m * tiles_n) * BN;
  C += (long)split * split_stride;
  const int kbeg = split * k_chunk, kend = min(K, kbeg + k_chunk);
  const int nk = kend > kbeg ? (kend - kbeg) / BK : 0;  // 16-deep slabs
  const int nst = (nk + 1) / 2;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave / WN) * 32 * TM, wn = (wave % WN) * 32 * TN;
  const int li = lane & 31, lk = lane >> 5;
  const GemmMap& fam = TA ? L.a.c : L.a.r;
  const GemmMap& fak = TA ? L.a.r : L.a.c;
  const GemmMap& fbn = TB ? L.b.r : L.b.c;
  const GemmMap& fbk = TB ? L.b.c : L.b.r;
  StA sa;
  StB sb;
  sa.template init<false>(m0, M, fam, fak);
  sb.template init<false>(n0, N, fbn, fbk);
  const int ksa = 4 * fak.s0, ksb = 4 * fbk.s0;
  const int frag_lane = li * 32 + ((lk ^ ((li >> 3) & 1)) << 4);
  const char* fra = lds + wm * 32 + frag_lane;
  const char* frb = lds + PA + wn * 32 + frag_lane;

  v16f acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = v16f{0};
  const __amdgpu_buffer_rsrc_t ra = buffer_rsrc(A, (unsigned)(L.ext_a * 4));
  const __amdgpu_buffer_rsrc_t rb = buffer_rsrc(B, (unsigned)(L.ext_b * 4));
  // the next stage to load: the k offsets of its two slabs; past the last
  // slab they stay there (values no product uses)
  KCursor<false> ka, kb;
  ka.init(fak, kbeg);
  kb.init(fbk, kbeg);
  int slab = 0, dka[2], dkb[2];
  auto next_offsets = [&]() {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      dka[h] = ka.bytes(fak);
      dkb[h] = kb.bytes(fbk);
      if (++slab < nk) {
        ka.advance(fak);
        kb.advance(fbk);
      }
    }
  };
  v4f st[G][2][U];  // G stages' units, slab by slab
  auto load_unit = [&](int g, int h, int u) {
    st[g][h][u] = u < UA ? sa.load(ra, u, dka[h], ksa) : sb.load(rb, u - UA, dkb[h], ksb);
  };
  auto store_unit = [&](char* S, int g, int h, int u) {
    if (u < UA) sa.store(S + h * SLAB, u, st[g][h][u]);
    else sb.store(S + h * SLAB + PA, u - UA, st[g][h][u]);
  };
  auto sync = [&]() {  // this wave's LDS operations are done, then everyone's
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (nk > 0) {
    auto load_stage = [&](int g) {
      next_offsets();
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int u = 0; u < U; ++u) load_unit(g, h, u);
    };
#pragma unroll
    for (int s = 0; s < 2; ++s) {  // stages 0 and 1 into LDS
      load_stage(s % G);
      if (G == 1 || s == 1) {
#pragma unroll
        for (int t = G == 1 ? s : 0; t <= s; ++t)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int u = 0; u < U; ++u) store_unit(lds + t * STAGE, t % G, h, u);
      }
    }
#pragma unroll
    for (int g = 0; g < G; ++g) load_stage(g);  // stages 2 .. 1 + G
    sync();
    bf16x8 fa[2][TM], fb[2][TN];
    auto read = [&](int set, int at) {
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[set][i] = *reinterpret_cast<const bf16x8*>(fra + at + i * 1024);
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[set][j] = *reinterpret_cast<const bf16x8*>(frb + at + j * 1024);
    };
    read(0, 0);
    int cur = 0, nxt = STAGE, wr = 2 * STAGE;  // LDS offsets of stages s, s + 1 and s + 2
    auto half = [&](auto gc, auto hc, int at) {
      constexpr int P = decltype(gc)::value, H = decltype(hc)::value;
      read(H ^ 1, at);  // the next slab's fragments
#pragma unroll
      for (int u = 0; u < U; ++u) {
        store_unit(lds + wr, P, H, u);
        load_unit(P, H, u);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[H][i], fb[H][j], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int q = 0; q < TM * TN; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (2 * U + TM * TN - 1) / (TM * TN) + 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto body = [&](auto gc, int s) {
      next_offsets();
      half(gc, std::integral_constant<int, 0>{}, cur + SLAB);
      // an odd slab count: the last stage's second slab repeats the last one
      if (2 * s + 1 < nk) half(gc, std::integral_constant<int, 1>{}, nxt);
      sync();
      const int t = cur;
      cur = nxt;
      nxt = wr;
      wr = t;
    };
    for (int s = 0; s < nst; s += G) {
      body(std::integral_constant<int, 0>{}, s);
      if (G == 2 && s + 1 < nst) body(std::integral_constant<int, G - 1>{}, s + 1);
    }
  }

  const TileOut<TM, TN, false> out{L.c, M, N, m0 + wm, n0 + wn, li, lk, m0 + BM <= M && n0 + BN <= N};
  out.for_each([&](int i, int j, auto&& live, auto&& off) {
    write16(C, D ? read16(D, live, off) + acc[i][j] : acc[i][j], live, off);
  });
#endif
}

}  // namespace
}  // namespace k
}  // namespace malus
