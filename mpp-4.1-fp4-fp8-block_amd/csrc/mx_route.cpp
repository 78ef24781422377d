// mx_route.cpp - which kernel a GEMM runs on.
#include <cstdint>

#include "mx_internal.h"

namespace mx {

static bool at(uintptr_t align, const void* a, const void* b, const void* c = nullptr) {
  return ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(c)) & (align - 1)) == 0;
}

int gemm_kernel(int ak, int bk, int epi, const QGemmArgs& g) {
  const int m = g.m, n = g.n, k = g.k;
  auto tile = [](int side) { return side == 256 ? GEMM_TILE256 : GEMM_TILE128; };
  if (!gemm_q_ok(ak, bk, epi, m, n, k)) {
    if (const int side = tile_aligned(bk, g) ? tile_side_off_grid(ak, bk, epi, m, n, k) : 0) return tile(side);
    return stream_wins_off_grid(ak, bk, epi, m, n, k) ? GEMM_STREAM : GEMM_H;
  }
  // few tiles (C0): one small tile per CU, operands requested up front
  // (its scale loads are dwords: planes at a 4-byte boundary)
  // from 33 rows on (plain GEMMs 17: their 16-row tiles): 16 rows, 1024 -> 2 x
  // 4096 -> 1024, streaming 4.1 + 5.5 us against 4.7 + 7.5; 64 rows 7.0 + 6.6
  // against 6.7 + 5.1
  const bool gate_up = epi == EPI_SWIGLU_F16 || epi == EPI_SWIGLU_HALF;
  if (ak == AK_F16 && bk == BK_MXFP4 && small_gemm_ok(epi, m, n, k) && m > (gate_up ? 32 : 16) && at(4, g.s0, g.s1)) return GEMM_SMALL;
  if (stream_wins(ak, bk, epi, m, n, k)) return GEMM_STREAM;
  // about one 64 x 64-channel gate/up tile per CU over a long K (C2): K
  // split between the waves of a workgroup, no split-K partials
  if (bk == BK_MXFP4 && kq_gemm_ok(ak, epi, m, n, k) && at(16, g.a, g.b0, g.b1) && at(4, g.s0, g.s1, ak == AK_F8X2 ? g.a_e8 : nullptr))
    return GEMM_KQ;
  if (const int side = tile_aligned(bk, g) ? tile_side(ak, bk, epi, m, n, k) : 0) return tile(side);
  return GEMM_Q;
}

}  // namespace mx
