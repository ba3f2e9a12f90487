// The instances of k_gemm_x3.h, k_gemm_x3k.h and k_gemm_bf.h, in their own translation unit
// so the GEMM units build in parallel.
#include "k_gemm_bf.h"
#include "k_gemm_x3.h"
#include "k_gemm_x3k.h"

namespace malus {
namespace k {
namespace {

// Variant bits as in k_gemm.hip: 8 transA, 4 transB (the planner sends no
// product with both here), 32 mapped operands, 64 GELU epilogues, 128 grouped
// accumulation.
template <int WM, int WN, int TM, int TN, int G>
const void* x3_instance(int v) {
#define MALUS_X3(TA, TB, MAP, EPI) reinterpret_cast<const void*>(&k_gemm_x3<WM, WN, TM, TN, TA, TB, MAP, EPI, G>)
  const bool ta = v & 8, tb = v & 4, mapped = v & 32;
  if (v & 128) return !ta && tb ? MALUS_X3(false, true, true, 3) : nullptr;
  if (v & 64) return ta ? nullptr : tb ? MALUS_X3(false, true, false, 2) : MALUS_X3(false, false, false, 1);
  if (mapped) {
    if (ta) return MALUS_X3(true, false, true, 0);
    return tb ? MALUS_X3(false, true, true, 0) : MALUS_X3(false, false, true, 0);
  }
  if (ta) return MALUS_X3(true, false, false, 0);
  return tb ? MALUS_X3(false, true, false, 0) : MALUS_X3(false, false, false, 0);
#undef MALUS_X3
}

}  // namespace

const void* gemm_x3_kernel(int tile, int v) {
  switch (tile) {
    case 0: return x3_instance<2, 2, 2, 3, 2>(v);
    case 1: return x3_instance<2, 2, 2, 2, 2>(v);
    case 2: return x3_instance<4, 2, 2, 2, 2>(v);
    default: return x3_instance<2, 2, 1, 1, 4>(v);
  }
}

const void* gemm_x3k_kernel(int v) {
#define MALUS_X3K(TA, TB, MAP, EPI) reinterpret_cast<const void*>(&k_gemm_x3k<8, 1, 2, TA, TB, MAP, EPI>)
  const bool ta = v & 8, tb = v & 4, mapped = v & 32;
  if (v & 128) return !ta && tb ? MALUS_X3K(false, true, true, 3) : nullptr;
  if (v & 64) return ta ? nullptr : tb ? MALUS_X3K(false, true, false, 2) : MALUS_X3K(false, false, false, 1);
  if (mapped) {
    if (ta) return MALUS_X3K(true, false, true, 0);
    return tb ? MALUS_X3K(false, true, true, 0) : MALUS_X3K(false, false, true, 0);
  }
  if (ta) return MALUS_X3K(true, false, false, 0);
  return tb ? MALUS_X3K(false, true, false, 0) : MALUS_X3K(false, false, false, 0);
#undef MALUS_X3K
}

template <int WM, int WN, int TM, int TN, int G>
const void* bf_instance(int v) {
  const bool ta = v & 8, tb = v & 4;
  if (ta) return reinterpret_cast<const void*>(&k_gemm_bf<WM, WN, TM, TN, true, false, G>);
  return tb ? reinterpret_cast<const void*>(&k_gemm_bf<WM, WN, TM, TN, false, true, G>)
            : reinterpret_cast<const void*>(&k_gemm_bf<WM, WN, TM, TN, false, false, G>);
}

const void* gemm_bf_kernel(int tile, int v) {
  return tile == 0 ? bf_instance<2, 4, 4, 2, 1>(v) : bf_instance<4, 2, 2, 2, 2>(v);
}

}  // namespace k
}  // namespace malus
