// The f32 GEMM on the bf16 MFMA with each operand value split once per
// workgroup (k_split.h: three exact bf16 pieces, six piece products).
//
// What bounds it: six v_mfma_f32_32x32x16_bf16 per 32 x 32 accumulator and
// 16-deep k slab.  A kernel whose waves split their own fragments repeats
// each split once per wave that reads the value, and the split's 5.5 VALU
// instructions per value then take longer than the MFMAs (528 against 384
// cycles per slab for a 64 x 32 wave tile).  Here a slab's f32 values are
// loaded into registers, split once and stored in LDS as three bf16 planes,
// which the waves read as MFMA fragments; on a 128 x 192 tile of four waves
// the split is 440 VALU cycles beside 1152 MFMA cycles per wave and slab.
//
// Schedule of one slab s (one workgroup barrier): its six piece products run
// as six phases, and between the MFMAs of phase p the wave
//   splits the p-th unit of slab s + 2 from its staging registers into the
//   LDS stage slab s left, reloads those registers with slab s + 2 + G, and
//   reads slab s + 1's fragments into the registers whose piece product has
//   just been issued for the last time (only the two h planes, which are
//   used first and last, need a second set).
// So global latency has G slabs and LDS latency a phase or more to hide
// under MFMAs, with one barrier per slab at a point where the wave has
// nothing outstanding.
//
// The accumulators round the same sums in the same order as any kernel that
// walks the k slabs upwards with x3_slab, so the values equal those of the
// per-wave split for the same K split.
#pragma once

#include "k_gemm_dma.h"

namespace malus {
namespace k {
namespace {

// One operand's staging: BX rows of its free dimension by 16 k.  The slab in
// LDS is, per plane, [BX rows][16 k] bf16 (32 bytes a row), the 16-byte chunk
// c of row r at c ^ ((r >> 3) & 1): the 16 lanes of a 128-bit fragment read
// then cover the 64 banks once.  A unit is 4 k of one row, 8 bytes per
// plane.  KC operands load a unit as one 16-byte load (4 lanes per row); XC
// operands as four 4-byte loads, 64 consecutive rows per wave, with the two
// 8-byte halves of a chunk dealt to alternate 16-row groups so that the
// 8-byte stores of a half-wave do not meet in one bank.
// NP: 3 planes, or one of the values rounded to bf16 (k_gemm_bf.h).
template <int BX, int NT, bool KC, int NP = 3>
struct X3Stage {
  static constexpr int U = BX * 4 / NT;    // units per thread
  static constexpr int PLANE = BX * 32;    // bytes
  static_assert(BX * 4 % NT == 0 && BX % 64 == 0, "whole units per thread, whole waves per row group");
  int goff[U];  // byte offset of the unit's first value at k = 0
  int loff[U];  // byte offset in a plane

  // Rows past the operand's X read row X - 1 (their products are never
  // stored), so every load is in bounds.
  template <bool MAP>
  __device__ __forceinline__ void init(int x0, int X, const GemmMap& fx, const GemmMap& fk) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int idx = u * NT + (int)threadIdx.x;
      const int r = KC ? idx / 4 : idx % BX;
      const int q = KC ? idx % 4 : (idx / BX) ^ ((r >> 4) & 1);
      const int x = min(x0 + r, X - 1);
      goff[u] = 4 * (map_at<MAP>(fx, x) + 4 * q * (KC ? 1 : fk.s0));
      loff[u] = r * 32 + (((q >> 1) ^ ((r >> 3) & 1)) << 4) + ((q & 1) << 3);
    }
  }
#if defined(__HIP_DEVICE_COMPILE__)
  // unit u of the slab whose k offset is dk bytes; ks: bytes between k rows
  __device__ __forceinline__ v4f load(__amdgpu_buffer_rsrc_t rs, int u, int dk, int ks) const {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    if constexpr (KC) {
      return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, goff[u], dk, 0));
    } else {
      u32x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = __builtin_amdgcn_raw_buffer_load_b32(rs, goff[u], dk + j * ks, 0);
      return __builtin_bit_cast(v4f, v);
    }
  }
  // splits (rounds) unit u's values into the planes at S
  __device__ __forceinline__ void store(char* S, int u, v4f f) const {
    store_planes<NP>(S + loff[u], PLANE, {f[0], f[1], f[2], f[3]});
  }
#endif
};

// The C elements of a wave's accumulators: register r of (i, j) is C at
// cn(i, j) + dm(r) * row stride.  f(i, j, live(r), offset(r)) runs once per
// accumulator; a tile inside C skips the edge tests.
template <int TM, int TN, bool MAP>
struct TileOut {
  const GemmLayout& c;
  int M, N, m0, n0, li, lk;
  bool inside;
  template <class F>
  __device__ __forceinline__ void for_each(F&& f) const {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int rbase = map_at<MAP>(c.r, m0 + 32 * i) + 4 * lk * c.r.s0;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + 32 * j + li, m = m0 + 32 * i + 4 * lk;
        const int cn = map_at<MAP>(c.c, n) + rbase;
        auto off = [&](int r) { return cn + (8 * (r >> 2) + (r & 3)) * c.r.s0; };
        if (inside) f(i, j, [](int) { return true; }, off);
        else f(i, j, [&](int r) { return n < N && m + 8 * (r >> 2) + (r & 3) < M; }, off);
      }
    }
  }
};

template <class Live, class Off>
__device__ __forceinline__ v16f read16(const float* P, Live&& live, Off&& off) {
  v16f v = v16f{0};
#pragma unroll
  for (int r = 0; r < 16; ++r)
    if (live(r)) v[r] = P[off(r)];
  return v;
}
template <class Live, class Off>
__device__ __forceinline__ void write16(float* P, const v16f& v, Live&& live, Off&& off) {
#pragma unroll
  for (int r = 0; r < 16; ++r)
    if (live(r)) P[off(r)] = v[r];
}

// C = op(A) op(B) (+ D) as k_sgemm_dma computes it with X3 (the same
// operand maps, epilogues EPI 0..3 and split-K partials); the host
// guarantees K % 16 == 0, k maps whose div is a multiple of 16, C row maps
// whose div is a multiple of 32, 16-byte aligned k-contiguous rows, and byte
// offsets below 2^31.  WM x WN waves of TM x TN accumulators.
template <int WM, int WN, int TM, int TN, bool TA, bool TB, bool MAP, int EPI, int G = 1>
__global__ __launch_bounds__(64 * WM * WN, WM * WN == 4 && EPI == 3 ? 1 : 2) void k_gemm_x3(const float* __restrict__ A,
                                                                         const float* __restrict__ B,
                                                                         float* __restrict__ C, int M, int N, int K,
                                                                         GemmLayouts L, int k_chunk, int tiles_n,
                                                                         long split_stride, const float* __restrict__ D,
                                                                         float* __restrict__ E) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NT = 64 * WM * WN, BM = 32 * WM * TM, BN = 32 * WN * TN;
  using StA = X3Stage<BM, NT, !TA>;
  using StB = X3Stage<BN, NT, TB>;
  constexpr int UA = StA::U, UB = StB::U, U = UA + UB;
  constexpr int PA = StA::PLANE, PB = StB::PLANE, STAGE = 3 * (PA + PB);
  __shared__ __attribute__((aligned(1024))) char lds[2 * STAGE];

  // XCD-contiguous work, as in k_sgemm_dma: consecutive tiles of one output
  // row without a K split, a contiguous range of the split-major list with one
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
  const bool grouped = MAP && L.ngroup > 1;
  const int b = grouped ? 0 : blockIdx.z;
  if (grouped && EPI != 3) {
    A = L.ga[blockIdx.z];
    B = L.gb[blockIdx.z];
    C = L.gc[blockIdx.z];
  }
  const int ba = map_at<MAP>(L.a.b, b), bb = map_at<MAP>(L.b.b, b);
  const long coff = map_at<MAP>(L.c.b, b);
  float* __restrict__ Cf = C + coff + (long)split * split_stride;
  if (D) D += coff;
  float* __restrict__ Ef = (EPI == 1 || EPI == 2) ? E + coff : E;
  const int kbeg = split * k_chunk, kend = min(K, kbeg + k_chunk);
  const int nk = kend > kbeg ? (kend - kbeg) / BK : 0;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave / WN) * 32 * TM, wn = (wave % WN) * 32 * TN;
  const int li = lane & 31, lk = lane >> 5;
  const GemmMap& fam = TA ? L.a.c : L.a.r;
  const GemmMap& fak = TA ? L.a.r : L.a.c;
  const GemmMap& fbn = TB ? L.b.r : L.b.c;
  const GemmMap& fbk = TB ? L.b.c : L.b.r;
  StA sa;
  StB sb;
  sa.template init<MAP>(m0, M, fam, fak);
  sb.template init<MAP>(n0, N, fbn, fbk);
  const int ksa = 4 * fak.s0, ksb = 4 * fbk.s0;
  const int frag_lane = li * 32 + ((lk ^ ((li >> 3) & 1)) << 4);
  const char* fra = lds + wm * 32 + frag_lane;
  const char* frb = lds + 3 * PA + wn * 32 + frag_lane;

  v16f acc[TM][TN];
  auto run_k = [&](const float* Ap, const float* Bp) {
    const __amdgpu_buffer_rsrc_t ra = buffer_rsrc(Ap + ba, (unsigned)((L.ext_a - ba) * 4));
    const __amdgpu_buffer_rsrc_t rb = buffer_rsrc(Bp + bb, (unsigned)((L.ext_b - bb) * 4));
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = v16f{0};
    if (nk == 0) return;
    // next slab to load; past the last one it stays there (a repeated load
    // whose values no product uses)
    KCursor<MAP> ka, kb;
    ka.init(fak, kbeg);
    kb.init(fbk, kbeg);
    int slab = 0;
    int dka = ka.bytes(fak), dkb = kb.bytes(fbk);
    auto advance = [&]() {
      if (++slab < nk) {
        ka.advance(fak);
        kb.advance(fbk);
        dka = ka.bytes(fak);
        dkb = kb.bytes(fbk);
      }
    };
    v4f st[G][U];
    auto load_unit = [&](int g, int u) {
      st[g][u] = u < UA ? sa.load(ra, u, dka, ksa) : sb.load(rb, u - UA, dkb, ksb);
    };
    auto store_unit = [&](int stage, const v4f& f, int u) {
      char* S = lds + stage * STAGE;
      if (u < UA) sa.store(S, u, f);
      else sb.store(S + 3 * PA, u - UA, f);
    };
    bf16x8 al[TM], am[TM], ah[2][TM], bl[TN], bm[TN], bh[2][TN];
    auto fa = [&](int stage, int p, int i) {
      return *reinterpret_cast<const bf16x8*>(fra + stage * STAGE + p * PA + i * 1024);
    };
    auto fb = [&](int stage, int p, int j) {
      return *reinterpret_cast<const bf16x8*>(frb + stage * STAGE + p * PB + j * 1024);
    };
    auto sync = [&]() {  // this wave's LDS operations are done, then everyone's
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
    {  // slabs 0 and 1 into the two stages, slabs 2 .. 1 + G into registers
      v4f t[2][U];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          t[g][u] = u < UA ? sa.load(ra, u, dka, ksa) : sb.load(rb, u - UA, dkb, ksb);
        advance();
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int u = 0; u < U; ++u) load_unit(g, u);
        advance();
      }
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int u = 0; u < U; ++u) store_unit(g, t[g][u], u);
    }
    sync();
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      ah[0][i] = fa(0, 0, i);
      am[i] = fa(0, 1, i);
      al[i] = fa(0, 2, i);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      bh[0][j] = fb(0, 0, j);
      bm[j] = fb(0, 1, j);
      bl[j] = fb(0, 2, j);
    }
    sync();

    auto mfma = [&](const bf16x8(&a)[TM], const bf16x8(&bb_)[TN]) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], bb_[j], acc[i][j], 0, 0, 0);
    };
    // phase p's share of the next slabs' staging, and its instruction mix:
    // every MFMA followed by a few VALU instructions
    auto stage_unit = [&](auto par, int p) {
      constexpr int P = decltype(par)::value;
#pragma unroll
      for (int u = p; u < U; u += 6) {
        store_unit(P & 1, st[P % G][u], u);
        load_unit(P % G, u);
      }
    };
    auto mix = [&]() {
#pragma unroll
      for (int q = 0; q < TM * TN; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (U > 6 ? 48 : 24) / (TM * TN) + 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto body = [&](auto par) {
      constexpr int P = decltype(par)::value & 1, Q = P ^ 1;
      stage_unit(par, 0);
      mfma(al, bh[P]);
      mix();
#pragma unroll
      for (int i = 0; i < TM; ++i) al[i] = fa(Q, 2, i);
      stage_unit(par, 1);
      mfma(ah[P], bl);
      mix();
#pragma unroll
      for (int j = 0; j < TN; ++j) bl[j] = fb(Q, 2, j);
      stage_unit(par, 2);
      mfma(am, bm);
      mix();
#pragma unroll
      for (int i = 0; i < TM; ++i) ah[Q][i] = fa(Q, 0, i);
#pragma unroll
      for (int j = 0; j < TN; ++j) bh[Q][j] = fb(Q, 0, j);
      stage_unit(par, 3);
      mfma(am, bh[P]);
      mix();
#pragma unroll
      for (int i = 0; i < TM; ++i) am[i] = fa(Q, 1, i);
      stage_unit(par, 4);
      mfma(ah[P], bm);
      mix();
#pragma unroll
      for (int j = 0; j < TN; ++j) bm[j] = fb(Q, 1, j);
      stage_unit(par, 5);
      advance();
      mfma(ah[P], bh[P]);
      mix();
      sync();
    };
    constexpr int UNR = G > 2 ? G : 2;  // bodies per turn: the stage and register sets are compile-time
    static_assert(UNR % G == 0 && UNR % 2 == 0 && UNR <= 4, "");
    int s = 0;
    for (; s + UNR <= nk; s += UNR) {
      body(std::integral_constant<int, 0>{});
      body(std::integral_constant<int, 1>{});
      if constexpr (UNR == 4) {
        body(std::integral_constant<int, 2>{});
        body(std::integral_constant<int, 3>{});
      }
    }
    if (s < nk) body(std::integral_constant<int, 0>{});
    if (s + 1 < nk) body(std::integral_constant<int, 1>{});
    if (UNR == 4 && s + 2 < nk) body(std::integral_constant<int, 2>{});
  };

  const TileOut<TM, TN, MAP> out{L.c, M, N, m0 + wm, n0 + wn, li, lk, m0 + BM <= M && n0 + BN <= N};
  if constexpr (EPI == 3) {
    v16f tot[TM][TN];
    for (int g = 0; g < L.ngroup; ++g) {
      run_k(L.ga[g], L.gb[g]);
      if (g == 0) {
        out.for_each([&](int i, int j, auto&& live, auto&& off) {
          tot[i][j] = D ? read16(D, live, off) + acc[i][j] : acc[i][j];
        });
      } else {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) tot[i][j] = tot[i][j] + acc[i][j];
      }
    }
    out.for_each([&](int i, int j, auto&& live, auto&& off) { write16(Cf, tot[i][j], live, off); });
  } else {
    run_k(A, B);
    out.for_each([&](int i, int j, auto&& live, auto&& off) {
      v16f v = acc[i][j];
      if constexpr (EPI == 2) {
        const v16f e = read16(Ef, live, off);
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = gelu_bwd(e[r], v[r]);
      }
      if (D) v = read16(D, live, off) + v;
      write16(Cf, v, live, off);
      if constexpr (EPI == 1) {
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = gelu_fwd(v[r]);
        write16(Ef, v, live, off);
      }
    });
  }
#endif
}

}  // namespace
}  // namespace k
}  // namespace malus
