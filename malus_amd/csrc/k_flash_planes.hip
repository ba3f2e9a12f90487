// Flash attention on the bf16 MFMA (the algorithm and the lane layout are
// k_flash.hip's): f32 products as split bf16 pieces (NP = 3 planes,
// k_split.h), or operands rounded to bf16 under autocast (NP = 1).
//
// What bounds it: a wave that owns a 32-row tile and streams the other
// operand's tiles spends more VALU cycles on splitting the streamed values
// (5.5 instructions each, in both orientations) than its MFMAs take: in the
// forward 3.2k VALU beside 1.5k MFMA cycles per 32 x 32 block at head size
// 64.  Here W waves of one head, one 32-row tile each, share every streamed
// tile: its f32 values are loaded once per workgroup, split once and kept in
// LDS as bf16 planes.  With four waves (AHEAD) the planes are double buffered,
// the next tile's loads are in flight during the current tile's products and a
// tile takes one barrier.  Workgroups of one or two waves keep one buffer and
// load between the products: the registers and the LDS of the second stage cost
// them more waves per CU than it hides (dkv at head size 64 spilled 31
// registers; the times stand at group_waves).  Both orientations are read from the same planes: rows with 128-bit reads,
// columns with gfx950's transposing read (ds_read_b64_tr_b16).
// The products run in the order of the per-wave form; only exp differs (exp_of).
#include "k_flash.h"

namespace malus {
namespace k {
namespace {

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// NP planes of 8 fragment values
template <int NP>
struct Frag {
  bf16x8 p[NP];
};

template <int NP>
__device__ __forceinline__ Frag<NP> make_frag(const float (&f)[8]) {
  Frag<NP> r;
  if constexpr (NP == 3) {
    const Split3 s = split3(f);
    r.p[0] = s.h;
    r.p[1] = s.m;
    r.p[2] = s.l;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) r.p[0][e] = (__bf16)f[e];
  }
  return r;
}

template <int NP>
__device__ __forceinline__ v16f mul(const Frag<NP>& a, const Frag<NP>& b, v16f c) {
  if constexpr (NP == 3) return x3_one<false>(Split3{a.p[0], a.p[1], a.p[2]}, Split3{b.p[0], b.p[1], b.p[2]}, c);
  else return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[0], b.p[0], c, 0, 0, 0);
}

// exp(x) = 2^n 2^f, n the integer nearest x log2(e) and f the rest from two
// fused multiply-adds (log2(e) = 1.44269502 + 1.92596299e-8): 8 instructions
// where expf takes 13, and its accuracy (rms 2.67e-8 of the value and at most 8.6e-8
// over x = -80 .. 0, expf 2.63e-8 and 8.4e-8; both are v_exp_f32's own error).
// Under autocast too: the f32 row sums and the log-sum-exp are made of these
// values.  Shorter forms measured worse: 2^(x log2(e)) in two instructions 4.2e-7
// at x = -20 .. -10 and 1.7e-6 at -80 .. -40, the same corrected behind v_exp_f32 in
// six 3.6e-8 and 1.4e-7 at most.  48 heads, T = 2048, autocast, forward + backward:
// 219 us with two instructions, 250 with six, 263 here, 296 with expf; 384 heads,
// T = 256, f32: 150.2 with six, 150.4 here, 153.8 with expf.  The clamp keeps n an
// integer that ldexp takes; f is then infinite where x is, and NaN where x is.
__device__ __forceinline__ float exp_of(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const float n = __builtin_rintf(__builtin_amdgcn_fmed3f(x * 1.44269504f, -160.0f, 160.0f));
  const float f = __builtin_fmaf(x, 1.92596299e-8f, __builtin_fmaf(x, 1.44269504f, -n));
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), (int)n);
#else
  return x;
#endif
}

// 8 values of a tensor stored in f32 or, S16, in bf16 (a bf16 value is its
// own h plane)
template <int NP, bool S16>
__device__ __forceinline__ Frag<NP> load_frag(const float* __restrict__ base, size_t i) {
  if constexpr (S16) {
    return Frag<NP>{{*reinterpret_cast<const bf16x8*>(reinterpret_cast<const __bf16*>(base) + i)}};
  } else {
    float f[8];
    load8(base + i, f);
    return make_frag<NP>(f);
  }
}

template <bool S16>
__device__ __forceinline__ void st4(float* __restrict__ base, size_t i, v4f w) {
  if constexpr (S16)
    *reinterpret_cast<bf16x4*>(reinterpret_cast<__bf16*>(base) + i) =
        bf16x4{(__bf16)w[0], (__bf16)w[1], (__bf16)w[2], (__bf16)w[3]};
  else *reinterpret_cast<v4f*>(base + i) = w;
}
template <bool S16>
__device__ __forceinline__ void st1(float* __restrict__ base, size_t i, float w) {
  if constexpr (S16) reinterpret_cast<__bf16*>(base)[i] = (__bf16)w;
  else base[i] = w;
}

// A 32-row tile of [T, HS] in LDS: per plane [32][HS] bf16, the 16-byte chunk
// c of row r at c ^ swz(r).  swz spreads the 16 rows of a 128-bit row read
// over the 64 banks, and keeps the four consecutive rows that a transposing
// read touches (64 bytes each) apart: at HS = 64 two rows fill the banks
// once, so rows two apart get the chunks of the other half.
template <int HS, int NP>
struct Tile {
  static constexpr int ROW = 2 * HS, PLANE = 32 * ROW, SIZE = NP * PLANE;
  __device__ __forceinline__ static int swz(int r) {
    return HS == 64 ? (((r >> 1) & 1) << 2) | (((r >> 2) & 1) << 1) | ((r >> 3) & 1) : (r >> 2) & 3;
  }
  // 4 values (columns 4 c4 ..) of row r
  __device__ __forceinline__ static void store(char* S, int r, int c4, v4f f) {
    store_planes<NP>(S + r * ROW + (((c4 >> 1) ^ swz(r)) << 4) + ((c4 & 1) << 3), PLANE, {f[0], f[1], f[2], f[3]});
  }
  // columns 16 kb + 8 lk .. of row r (the lane's own lk)
  __device__ __forceinline__ static Frag<NP> row(const char* S, int r, int kb, int lk) {
    Frag<NP> f;
    const char* at = S + r * ROW + (((2 * kb + lk) ^ swz(r)) << 4);
#pragma unroll
    for (int p = 0; p < NP; ++p) f.p[p] = *reinterpret_cast<const bf16x8*>(at + p * PLANE);
    return f;
  }
  // rows 16 h + 8 lk .. + 7 of column 32 n + x: lane 16 g + 4 e + a of a
  // transposing read addresses 4 columns (run a) of row e and receives, as
  // value e, its own column of row e
  __device__ __forceinline__ static Frag<NP> col(const char* S, int n, int h) {
    Frag<NP> f;
#if defined(__HIP_DEVICE_COMPILE__)
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    const int lane = threadIdx.x & 63, g = lane >> 4, e = (lane >> 2) & 3, a = lane & 3;
    const int c = 32 * n + 16 * (g & 1) + 4 * a;
    const int r0 = 16 * h + 8 * (g >> 1) + e, r1 = r0 + 4;
    const char* p0 = S + r0 * ROW + (((c >> 3) ^ swz(r0)) << 4) + (c & 7) * 2;
    const char* p1 = S + r1 * ROW + (((c >> 3) ^ swz(r1)) << 4) + (c & 7) * 2;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const s16x4 u = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p0 + p * PLANE));
      const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p1 + p * PLANE));
      f.p[p] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(u, v, 0, 1, 2, 3, 4, 5, 6, 7));
    }
#endif
    return f;
  }
};

// One streamed tile in registers: rows 32 j .. of a [T, HS] matrix whose rows
// are ld apart, 4 values per unit, NT threads.
template <int HS, int NT, bool S16>
struct Stream {
  static constexpr int Q4 = HS / 4, PER = 32 * Q4 / NT;
  v4f v[PER];
  __device__ __forceinline__ void fetch(const float* __restrict__ base, int ld, int j) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int f = (int)threadIdx.x + NT * u;
      const size_t i = (size_t)(32 * j + f / Q4) * ld + 4 * (f % Q4);
      if constexpr (S16) {
        const bf16x4 h = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const __bf16*>(base) + i);
        v[u] = v4f{(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
      } else {
        v[u] = *reinterpret_cast<const v4f*>(base + i);
      }
    }
  }
  template <int NP>
  __device__ __forceinline__ void store(char* S) const {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int f = (int)threadIdx.x + NT * u;
      Tile<HS, NP>::store(S, f / Q4, f % Q4, v[u]);
    }
  }
};

template <bool S16>
__device__ __forceinline__ const float* at(const float* base, size_t i) {
  return S16 ? reinterpret_cast<const float*>(reinterpret_cast<const __bf16*>(base) + i) : base + i;
}

// Forward: query tiles W g .. W g + W - 1 of head bh, one per wave.
template <int HS, bool CAUSAL, int NP, bool S16, int W>
__global__ __launch_bounds__(64 * W, 2) void k_flash_planes_fwd(const float* __restrict__ Q, const float* __restrict__ K,
                                                             const float* __restrict__ V,
                                                             const float* __restrict__ scale, float* __restrict__ O,
                                                             int ldo, int H, float* __restrict__ lse, int T, int BH) {
  constexpr int NKB = HS / 16, NN = HS / 32, NT = 64 * W;
  constexpr bool AHEAD = W == 4 || (W == 2 && HS == 32);
  constexpr int NB = AHEAD ? 2 : 1;
  using Tl = Tile<HS, NP>;
  __shared__ __attribute__((aligned(1024))) char Ks[NB][Tl::SIZE], Vs[NB][W == 1 ? 16 : Tl::SIZE];
  const int tiles = T / 32, groups = (tiles + W - 1) / W;
  const int grp = groups - 1 - (int)(blockIdx.x / BH), bh = (int)(blockIdx.x % BH);  // the longest first
  const int lane = threadIdx.x & 63, x = lane & 31, lk = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);  // uniform: the tile tests are scalar
  const int qt = W * grp + wave;
  const bool live = qt < tiles;  // past the last tile: this wave only helps staging
  const size_t head = (size_t)bh * T * HS;
  const float *Kh = at<S16>(K, head), *Vh = at<S16>(V, head);
  const int i0 = 32 * qt;
  const float sc = scale[0];
  const int jmax = W == 1 ? 0 : CAUSAL ? min(W * grp + W, tiles) - 1 : tiles - 1;  // W = 1: the only tile
  const int last = !live ? -1 : CAUSAL ? qt : tiles - 1;

  Stream<HS, NT, S16> kst, vst;
  kst.fetch(Kh, HS, 0);
  vst.fetch(Vh, HS, 0);
  Frag<NP> q[NKB];  // B of S^T = K Q^T
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb)
    q[kb] = load_frag<NP, S16>(Q, head + (size_t)(live ? i0 + x : 0) * HS + 16 * kb + 8 * lk);
  v16f o[NN];
#pragma unroll
  for (int n = 0; n < NN; ++n) o[n] = v16f{0};
  float m = -INFINITY, l = 0.0f;
  kst.template store<NP>(Ks[0]);
  if (W > 1) vst.template store<NP>(Vs[0]);
  __syncthreads();
  for (int j = 0; j <= jmax; ++j) {
    const int cur = AHEAD ? j & 1 : 0;
    if (AHEAD && j < jmax) {
      kst.fetch(Kh, HS, j + 1);
      vst.fetch(Vh, HS, j + 1);
    }
    if (j <= last) {
      v16f st = v16f{0};
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) st = mul<NP>(Tl::row(Ks[cur], perm_row(x), kb, lk), q[kb], st);
      // lane = query i0 + x, register r = key 32 j + perm_index(r, lk)
      float mt = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; ++r) st[r] = st[r] * sc;
      if (CAUSAL && j == qt) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (perm_index(r, lk) > x) st[r] = -INFINITY;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) mt = fmaxf(mt, st[r]);
      mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
      const float mn = fmaxf(m, mt);
      const float alpha = expf(m - mn);  // 0 on the first tile (m = -inf)
      float ls = 0.0f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = exp_of(st[r] - mn);
        st[r] = p;
        ls += p;
      }
      ls += __shfl_xor(ls, 32, 64);
      l = l * alpha + ls;
      m = mn;
#pragma unroll
      for (int n = 0; n < NN; ++n) o[n] *= alpha;
      const char* vs = Vs[cur];
      if constexpr (W == 1) {  // V takes K's place: half the LDS, twice the waves
        __syncthreads();
        vst.template store<NP>(Ks[0]);
        __syncthreads();
        vs = Ks[0];
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float pb[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) pb[e] = st[8 * h + e];
        const Frag<NP> p = make_frag<NP>(pb);
#pragma unroll
        for (int n = 0; n < NN; ++n) o[n] = mul<NP>(Tl::col(vs, n, h), p, o[n]);
      }
    }
    if (W > 1 && j < jmax) {
      if (!AHEAD) {
        kst.fetch(Kh, HS, j + 1);
        vst.fetch(Vh, HS, j + 1);
        __syncthreads();  // tile j is read
      }
      kst.template store<NP>(Ks[AHEAD ? cur ^ 1 : 0]);
      vst.template store<NP>(Vs[AHEAD ? cur ^ 1 : 0]);
    }
    __syncthreads();  // tile j is read, tile j + 1 is staged
  }
  if (!live) return;
  // O[i0 + x][32 n + 8 g + 4 lk + c] = o[n][4 g + c] / l
  float* orow = O + (size_t)(bh / H) * T * ldo + (size_t)(bh % H) * HS + (size_t)(i0 + x) * ldo;
#pragma unroll
  for (int n = 0; n < NN; ++n)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      v4f w;
#pragma unroll
      for (int c = 0; c < 4; ++c) w[c] = o[n][4 * g + c] / l;
      *reinterpret_cast<v4f*>(orow + 32 * n + 8 * g + 4 * lk) = w;
    }
  if (lk == 0) lse[(size_t)bh * T + i0 + x] = m + logf(l);
}

// Backward, query-centric: dQ (+ Dq) of query tiles W g .., one per wave, and
// D = rowsum(dO * O) of their rows into dsum for the key-centric pass.
template <int HS, bool CAUSAL, int NP, bool S16, int W>
__global__ __launch_bounds__(64 * W, 2) void k_flash_planes_dq(const float* __restrict__ Q, const float* __restrict__ K,
                                                            const float* __restrict__ V, const float* __restrict__ O,
                                                            const float* __restrict__ dO, int ldo, int H,
                                                            const float* __restrict__ lse,
                                                            const float* __restrict__ scale, float* __restrict__ dQ,
                                                            const float* __restrict__ Dq, float* __restrict__ dsum,
                                                            int T, int BH) {
  constexpr int NKB = HS / 16, NN = HS / 32, NT = 64 * W;
  constexpr bool AHEAD = W == 4;
  constexpr int NB = AHEAD ? 2 : 1;
  using Tl = Tile<HS, NP>;
  __shared__ __attribute__((aligned(1024))) char Ks[NB][Tl::SIZE], Vs[NB][Tl::SIZE];
  const int tiles = T / 32, groups = (tiles + W - 1) / W;
  const int grp = groups - 1 - (int)(blockIdx.x / BH), bh = (int)(blockIdx.x % BH);
  const int lane = threadIdx.x & 63, x = lane & 31, lk = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);  // uniform: the tile tests are scalar
  const int qt = W * grp + wave;
  const bool live = qt < tiles;
  const size_t head = (size_t)bh * T * HS;
  const float *Kh = at<S16>(K, head), *Vh = at<S16>(V, head);
  const int i0 = 32 * qt, i = live ? i0 + x : 0;
  const float sc = scale[0];
  const int jmax = W == 1 ? 0 : CAUSAL ? min(W * grp + W, tiles) - 1 : tiles - 1;
  const int last = !live ? -1 : CAUSAL ? qt : tiles - 1;

  Stream<HS, NT, S16> kst, vst;
  kst.fetch(Kh, HS, 0);
  vst.fetch(Vh, HS, 0);
  Frag<NP> q[NKB], og[NKB];  // B of S^T = K Q^T and of dP^T = V dO^T
  const float* dorow = head_row(dO, bh, H, T, ldo, HS, i);
  const float* orow = head_row(O, bh, H, T, ldo, HS, i);
  float d = 0.0f;
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb) {
    q[kb] = load_frag<NP, S16>(Q, head + (size_t)i * HS + 16 * kb + 8 * lk);
    float ob[8], ov[8];
    load8(dorow + 16 * kb + 8 * lk, ob);
    load8(orow + 16 * kb + 8 * lk, ov);
#pragma unroll
    for (int e = 0; e < 8; ++e) d += ob[e] * ov[e];
    og[kb] = make_frag<NP>(ob);
  }
  d += __shfl_xor(d, 32, 64);
  if (live && lk == 0) dsum[(size_t)bh * T + i] = d;
  const float L = lse[(size_t)bh * T + i];

  v16f dq[NN];
#pragma unroll
  for (int n = 0; n < NN; ++n) dq[n] = v16f{0};
  kst.template store<NP>(Ks[0]);
  vst.template store<NP>(Vs[0]);
  __syncthreads();
  for (int j = 0; j <= jmax; ++j) {
    const int cur = AHEAD ? j & 1 : 0;
    if (AHEAD && j < jmax) {
      kst.fetch(Kh, HS, j + 1);
      vst.fetch(Vh, HS, j + 1);
    }
    if (j <= last) {
      v16f st = v16f{0}, dp = v16f{0};
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        st = mul<NP>(Tl::row(Ks[cur], perm_row(x), kb, lk), q[kb], st);
        dp = mul<NP>(Tl::row(Vs[cur], perm_row(x), kb, lk), og[kb], dp);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) st[r] = exp_of(st[r] * sc - L);
      if (CAUSAL && j == qt) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (perm_index(r, lk) > x) st[r] = 0.0f;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float diff = dp[r] - d;
        const float dx = st[r] * diff;
        st[r] = dx * sc;
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float ab[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) ab[e] = st[8 * h + e];
        const Frag<NP> ds = make_frag<NP>(ab);
#pragma unroll
        for (int n = 0; n < NN; ++n) dq[n] = mul<NP>(ds, Tl::col(Ks[cur], n, h), dq[n]);
      }
    }
    if (W > 1 && j < jmax) {
      if (!AHEAD) {
        kst.fetch(Kh, HS, j + 1);
        vst.fetch(Vh, HS, j + 1);
        __syncthreads();  // tile j is read
      }
      kst.template store<NP>(Ks[AHEAD ? cur ^ 1 : 0]);
      vst.template store<NP>(Vs[AHEAD ? cur ^ 1 : 0]);
    }
    __syncthreads();
  }
  if (!live) return;
  // dQ[i0 + 8 (r >> 2) + 4 lk + (r & 3)][32 n + x] (+ Dq: every addend loaded
  // before the first add; f32 storage only)
  auto off = [&](int n, int r) { return head + (size_t)(i0 + 8 * (r >> 2) + 4 * lk + (r & 3)) * HS + 32 * n + x; };
  if (!S16 && Dq) {
    float a[NN][16];
#pragma unroll
    for (int n = 0; n < NN; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) a[n][r] = Dq[off(n, r)];
#pragma unroll
    for (int n = 0; n < NN; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) dQ[off(n, r)] = a[n][r] + dq[n][r];
  } else {
#pragma unroll
    for (int n = 0; n < NN; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) st1<S16>(dQ, off(n, r), dq[n][r]);
  }
}

// Backward, key-centric: dK (+ Dk) and dV (+ Dv) of key tiles W g .., one
// per wave; the query tiles of Q and dO stream.
template <int HS, bool CAUSAL, int NP, bool S16, int W>
__global__ __launch_bounds__(64 * W, 2) void k_flash_planes_dkv(
    const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V, const float* __restrict__ dO,
    int ldo, int H, const float* __restrict__ lse, const float* __restrict__ dsum, const float* __restrict__ scale,
    float* __restrict__ dK, const float* __restrict__ Dk, float* __restrict__ dV, const float* __restrict__ Dv, int T,
    int BH) {
  constexpr int NKB = HS / 16, NN = HS / 32, NT = 64 * W;
  constexpr bool AHEAD = W == 4;
  constexpr int NB = AHEAD ? 2 : 1;
  using Tl = Tile<HS, NP>;
  __shared__ __attribute__((aligned(1024))) char Qs[NB][Tl::SIZE], Os[NB][Tl::SIZE];
  __shared__ __attribute__((aligned(16))) float Ls[NB][2][32];  // lse and dsum of the tile's rows
  const int tiles = T / 32;
  const int grp = (int)(blockIdx.x / BH), bh = (int)(blockIdx.x % BH);
  const int lane = threadIdx.x & 63, x = lane & 31, lk = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);  // uniform: the tile tests are scalar
  const int kt = W * grp + wave;
  const bool live = kt < tiles;
  const size_t head = (size_t)bh * T * HS;
  const float* Qh = at<S16>(Q, head);
  const float* dOh = head_row(dO, bh, H, T, ldo, HS, 0);
  const int j0 = 32 * kt, key = live ? j0 + x : 0;
  const float sc = scale[0];
  // threads 0 .. 63 stage a tile's row values
  const float* rowv = (threadIdx.x & 32 ? dsum : lse) + (size_t)bh * T + (threadIdx.x & 31);
  float rv = 0.0f;
  auto fetch_rows = [&](int it) {
    if (threadIdx.x < 64) rv = rowv[32 * it];
  };
  auto store_rows = [&](int stage) {
    if (threadIdx.x < 64) Ls[stage][threadIdx.x >> 5][threadIdx.x & 31] = rv;
  };
  const int wg_first = CAUSAL ? W * grp : 0;
  const int first = !live ? tiles : CAUSAL ? kt : 0;

  Stream<HS, NT, S16> qst;
  Stream<HS, NT, false> ost;
  qst.fetch(Qh, HS, wg_first);
  ost.fetch(dOh, ldo, wg_first);
  fetch_rows(wg_first);
  Frag<NP> kf[NKB], vf[NKB];  // B of S = Q K^T and of dP = dO V^T
#pragma unroll
  for (int kb = 0; kb < NKB; ++kb) {
    kf[kb] = load_frag<NP, S16>(K, head + (size_t)key * HS + 16 * kb + 8 * lk);
    vf[kb] = load_frag<NP, S16>(V, head + (size_t)key * HS + 16 * kb + 8 * lk);
  }
  v16f dvt[NN], dkt[NN];  // dV^T, dK^T: lane = key, rows = head dims
#pragma unroll
  for (int n = 0; n < NN; ++n) {
    dvt[n] = v16f{0};
    dkt[n] = v16f{0};
  }
  qst.template store<NP>(Qs[0]);
  ost.template store<NP>(Os[0]);
  store_rows(0);
  __syncthreads();
  for (int it = wg_first; it < tiles; ++it) {
    const int cur = AHEAD ? (it - wg_first) & 1 : 0;
    if (AHEAD && it + 1 < tiles) {
      qst.fetch(Qh, HS, it + 1);
      ost.fetch(dOh, ldo, it + 1);
      fetch_rows(it + 1);
    }
    if (it >= first) {
      v16f s = v16f{0}, dp = v16f{0};
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        s = mul<NP>(Tl::row(Qs[cur], perm_row(x), kb, lk), kf[kb], s);
        dp = mul<NP>(Tl::row(Os[cur], perm_row(x), kb, lk), vf[kb], dp);
        if (NP == 3 && kb % 2) __builtin_amdgcn_sched_barrier(0);  // hold the fragment reads to what 256 VGPRs take
      }
      // lane = key j0 + x, register r = query i0 + perm_index(r, lk)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = exp_of(s[r] * sc - Ls[cur][0][perm_index(r, lk)]);
      if (CAUSAL && it == kt) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (x > perm_index(r, lk)) s[r] = 0.0f;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float diff = dp[r] - Ls[cur][1][perm_index(r, lk)];
        const float dx = s[r] * diff;
        dp[r] = dx * sc;
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float pb[8], db[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          pb[e] = s[8 * h + e];
          db[e] = dp[8 * h + e];
        }
        const Frag<NP> p = make_frag<NP>(pb), ds = make_frag<NP>(db);
#pragma unroll
        for (int n = 0; n < NN; ++n) {
          dvt[n] = mul<NP>(Tl::col(Os[cur], n, h), p, dvt[n]);
          dkt[n] = mul<NP>(Tl::col(Qs[cur], n, h), ds, dkt[n]);
          if (NP == 3) __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (W > 1 && it + 1 < tiles) {
      if (!AHEAD) {
        qst.fetch(Qh, HS, it + 1);
        ost.fetch(dOh, ldo, it + 1);
        fetch_rows(it + 1);
        __syncthreads();  // tile it is read
      }
      qst.template store<NP>(Qs[AHEAD ? cur ^ 1 : 0]);
      ost.template store<NP>(Os[AHEAD ? cur ^ 1 : 0]);
      store_rows(AHEAD ? cur ^ 1 : 0);
    }
    __syncthreads();
  }
  if (!live) return;
  // dV[j0 + x][32 n + 8 g + 4 lk + c] = dvt[n][4 g + c] (+ Dv), dK likewise
  // (the addends, where given, are all loaded before the first add)
  v4f av[NN][4], ak[NN][4];
#pragma unroll
  for (int n = 0; n < NN; ++n)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const size_t off = head + (size_t)key * HS + 32 * n + 8 * g + 4 * lk;
      if (!S16 && Dv) av[n][g] = *reinterpret_cast<const v4f*>(Dv + off);
      if (!S16 && Dk) ak[n][g] = *reinterpret_cast<const v4f*>(Dk + off);
    }
#pragma unroll
  for (int n = 0; n < NN; ++n)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const size_t off = head + (size_t)key * HS + 32 * n + 8 * g + 4 * lk;
      v4f wv, wk;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        wv[c] = dvt[n][4 * g + c];
        wk[c] = dkt[n][4 * g + c];
      }
      if (!S16 && Dv) wv = av[n][g] + wv;
      if (!S16 && Dk) wk = ak[n][g] + wk;
      st4<S16>(dV, off, wv);
      st4<S16>(dK, off, wk);
    }
}

template <int HS, bool CAUSAL, int NP, bool S16, int W>
void fwd_launch(const float* Q, const float* K, const float* V, const float* scale, float* O, int ldo, int H, float* lse,
                int T, int BH, hipStream_t s) {
  k_flash_planes_fwd<HS, CAUSAL, NP, S16, W>
      <<<(unsigned)((T / 32 + W - 1) / W * BH), 64 * W, 0, s>>>(Q, K, V, scale, O, ldo, H, lse, T, BH);
}

template <int HS, bool CAUSAL, int NP, bool S16, int W>
void bwd_launch(const FlashBwd& a, int ldo, int H, int T, int BH, hipStream_t s) {
  const unsigned grid = (unsigned)((T / 32 + W - 1) / W * BH);
  k_flash_planes_dq<HS, CAUSAL, NP, S16, W><<<grid, 64 * W, 0, s>>>(a.Q, a.K, a.V, a.O, a.dO, ldo, H, a.lse, a.scale,
                                                                   a.dQ, a.Dq, a.dsum, T, BH);
  k_flash_planes_dkv<HS, CAUSAL, NP, S16, W><<<grid, 64 * W, 0, s>>>(a.Q, a.K, a.V, a.dO, ldo, H, a.lse, a.dsum,
                                                                    a.scale, a.dK, a.Dk, a.dV, a.Dv, T, BH);
}

// Waves per workgroup: one per 32-row tile up to two tiles, then four, which
// read each streamed tile least often.  A causal group of four also waits for
// its longest wave, and a last group of one or two tiles runs as few waves in
// the LDS of four; with split products, where LDS and registers hold a CU to
// two groups of four waves, two waves are then the faster group.  us at 98304 / T
// heads, one wave a tile without shared planes / two waves / four:
// - T = 32: forward at head size 64 20.1 / 23.5 / 28.9, one wave 18.9; backward
//   63.5 / 64.3 / 87.2, one wave 59.5
// - causal forward, head size 64: T = 128 31.0 / 24.8 / 29.7, 160 35.2 / 34.1 /
//   39.5, 224 42.5 / 40.2 / 42.4, 256 42.7 / 37.6 / 35.8, 448 66.4 / 57.7 / 67.7, 512
//   71.2 / 62.2 / 59.6; head size 32: T = 96 15.3 / 17.3 / 15.5, 128 19.3 / 16.0 /
//   18.1, 160 21.9 / 22.1 / 23.5
// - causal backward: T = 128 93.3 / 82.4 / 96.7, 256 133 / 111 / 123, 512 229 / 176 / 181,
//   1024 405 / 328 / 290; head size 32: T = 256 79.2 / 63.4 / 66.2, 384 104 / 79.5 / 77.6
// - the whole square: four at T = 96 already (backward 105 / 96.6 / 93.5)
int group_waves(bool backward, bool causal, int planes, int hs, int T) {
  const int tiles = T / 32, last = tiles % 4;
  if (tiles <= 2) return tiles;
  if (!causal || planes != 3) return 4;
  if (backward) return T <= 8 * hs ? 2 : 4;
  if (T >= 512) return 4;
  return last == 1 || last == 2 || tiles == 4 || (tiles == 3 && hs == 64) ? 2 : 4;
}

// f(HS, CAUSAL, NP, S16, W) as integral constants
template <class F>
void dispatch(bool backward, size_t hs, bool causal, int planes, bool s16, int T, F f) {
  auto waves = [&](auto HS, auto CA, auto NP, auto S) {
    const int w = group_waves(backward, causal, planes, (int)hs, T);
    if (w == 4) f(HS, CA, NP, S, std::integral_constant<int, 4>{});
    else if (w == 2) f(HS, CA, NP, S, std::integral_constant<int, 2>{});
    else f(HS, CA, NP, S, std::integral_constant<int, 1>{});
  };
  auto store = [&](auto HS, auto CA) {
    if (planes == 3) waves(HS, CA, std::integral_constant<int, 3>{}, std::false_type{});
    else if (s16) waves(HS, CA, std::integral_constant<int, 1>{}, std::true_type{});
    else waves(HS, CA, std::integral_constant<int, 1>{}, std::false_type{});
  };
  auto mask = [&](auto HS) {
    if (causal) store(HS, std::true_type{});
    else store(HS, std::false_type{});
  };
  if (hs == 64) mask(std::integral_constant<int, 64>{});
  else mask(std::integral_constant<int, 32>{});
}

}  // namespace

void flash_planes_fwd(size_t hs, bool causal, int planes, bool qkv_bf16, const float* Q, const float* K, const float* V,
                      const float* scale, float* O, int ldo, int H, float* lse, int T, int BH, hipStream_t s) {
  dispatch(false, hs, causal, planes, qkv_bf16, T, [&](auto HS, auto CA, auto NP, auto S, auto W) {
    fwd_launch<decltype(HS)::value, decltype(CA)::value, decltype(NP)::value, decltype(S)::value, decltype(W)::value>(
        Q, K, V, scale, O, ldo, H, lse, T, BH, s);
  });
}

void flash_planes_bwd(size_t hs, bool causal, int planes, bool qkv_bf16, const FlashBwd& a, int ldo, int H, int T, int BH,
                      hipStream_t s) {
  dispatch(true, hs, causal, planes, qkv_bf16, T, [&](auto HS, auto CA, auto NP, auto S, auto W) {
    bwd_launch<decltype(HS)::value, decltype(CA)::value, decltype(NP)::value, decltype(S)::value, decltype(W)::value>(
        a, ldo, H, T, BH, s);
  });
}

}  // namespace k
}  // namespace malus
