// mx_tile.cpp - which GEMMs the prefill tile kernel (mx_gemm_tile.h) takes, and
// with which tile.
#include "mx_tile.h"

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace mx {

namespace {

long ceil_div(long a, long b) { return (a + b - 1) / b; }

// What the kernel can run: a whole group of scales, offsets in 32 bits.
bool can(int ak, int bk, int epi, int k) {
  if (k > (1 << 20) || epi == EPI_SWIGLU_F8X2) return false;
  if (ak == AK_I8) return bk == BK_I8 && k % 128 == 0;
  if (ak != AK_F16 || bk == BK_I8 || epi == EPI_SWIGLU_F32 || epi == EPI_STORE_I32) return false;
  return k % 32 == 0 && k >= 256;
}

// Times of the three kernels, us, per K stage (64 K; int8 128) and for the
// launch with its first loads and last stores.  The 256-tile runs one workgroup
// a CU: a full round of 256 costs `full` a stage (the card's matrix rate), one
// of few tiles `part` (a CU's own).  The 128-tile runs two a CU, so tiles count
// as fractions of a round, from one tile's own time on.  `tiled`: the 128-row
// tiles of mx_gemm_q.hip (`start` + `tiled` a stage and round; `deep` at 192 to
// 256 tiles, where most formats have their deep ring).
struct Rates {
  double start256, part, full;
  double own128, round128;
  double start, tiled, deep;
};
const Rates& rates(int ak, int bk) {
  static const Rates mxfp4{8, 1.0, 1.46, 0.42, 0.46, 8, 0.535, 0.54};
  static const Rates int4{10, 1.05, 1.82, 0.55, 0.565, 8, 0.59, 0.6};
  static const Rates bits8{14, 0.9, 1.54, 0.48, 0.456, 7, 0.5, 0.45};
  static const Rates f16{8, 0.95, 1.65, 0.58, 0.47, 12, 0.535, 0.55};
  static const Rates w8a8{19, 1.35, 1.95, 0, 0, 16, 0.61, 0.61};
  return ak == AK_I8 ? w8a8 : bk == BK_MXFP4 ? mxfp4 : bk == BK_INT4G32 ? int4 : bk == BK_F16 ? f16 : bits8;
}

struct Times {
  long t128;
  double us256, us128;
};
Times times(int ak, int bk, int epi, int m, int n, int k) {
  const long n_rows = (long)n * (is_gate_up(epi) ? 2 : 1);
  const long t256 = ceil_div(m, 256) * ceil_div(n_rows, 256), t128 = ceil_div(m, 128) * ceil_div(n_rows, 128);
  const double kt = k / (ak == AK_I8 ? 128.0 : 64.0), last = (t256 % 256) / 256.0;
  const Rates& r = rates(ak, bk);
  const double us256 = r.start256 + kt * (t256 / 256 * r.full + (last > 0 ? r.part + (r.full - r.part) * last : 0));
  return {t128, us256, ak == AK_I8 ? us256 + 1 : 7 + kt * std::max(r.own128, r.round128 * t128 / 256)};
}

}  // namespace

// Tile side, 0 where the 128-row tiled family is the faster one.  By the times
// above, fitted to 200 GEMMs of 256 to 4096 rows (5 formats, 4 MLP sizes), which
// they get right to 10 % or where the sides differ less.  Some of them, us,
// tiled / 256 / 128:
//   MXFP4  4096 -> 2 x 14336   500 rows 139 / 105 / 114   1000 257 / 197 / 205   4096 951 / 670 / 801
//          14336 -> 4096       500 rows 67 / 237 / 92     1000 152 / 238 / 105   4096 484 / 330 / 398
//          2048 -> 2 x 5632    1000 rows 54 / 48 / 47     2048 92 / 93 / 89      4096 181 / 153 / 168
//   FP8    2048 -> 2 x 5632    256 rows 35 / 45 / 22      1000 56 / 56 / 53      4096 186 / 168 / 174
//          5632 -> 2048        1000 rows 35 / 98 / 44     2048 47 / 100 / 50     4096 95 / 109 / 86
//   INT4   4096 -> 2 x 14336   500 rows 157 / 123 / 148   1000 284 / 231 / 265   4096 1065 / 820 / 1034
//   f16    4096 -> 14336       256 rows 40 / 76 / 44      500 103 / 79 / 60      4096 486 / 386 / 432
//   W8A8   4096 -> 2 x 14336   256 rows 52 / 68           500 110 / 72           4096 563 / 478
//          14336 -> 4096       1000 rows 78 / 175         2048 139 / 181         4096 262 / 200
// Below 150 tiles of 128 the split-K launches keep more CUs busy than either
// tile does; from there to 192 they pay for a second launch and the partials.
int tile_side(int ak, int bk, int epi, int m, int n, int k) {
  if (!can(ak, bk, epi, k)) return 0;
  const Times t = times(ak, bk, epi, m, n, k);
  if (t.t128 < 150) return 0;
  const double kt = k / (ak == AK_I8 ? 128.0 : 64.0);
  // MXFP4, a plain store, one round of tiles, up to 2048 K: level with the tiled
  // family's deep ring as a kernel (0.8 us faster to 0.8 slower), behind it or
  // level in a pass.  Down GEMMs of MLP passes, us a pass, deep ring / here: 512
  // rows, 7168 wide, K = 1024 34.9 / 35.9, 1536 44.4 / 44.9, 2048 50.9 / 51.1, 2560
  // 79.0 / 79.7; 6656, 1024 38.8 / 40.0; 8192, 1024 38.1 / 39.0; 768 rows, 4608, 1024
  // 32.3 / 32.8; 1024 rows, 4096, 1024 35.1 / 35.9; 1500 rows, 2304, 2048 47.9 / 48.3;
  // 1792 rows, 2048, 1536 40.9 / 41.8; 2048 rows, 2048, 2048 50.6 / 51.0; past it 1024
  // rows, 4096, K = 2560 84.8 / 84.7, 3584 85.9 / 85.7.  Gate/up GEMMs of the same
  // tiles and K are faster here: 1024 rows, 2048 -> 2 x 2048 41.1 / 39.5, 768 rows,
  // 2048 -> 2 x 2304 39.1 / 38.2, 900 rows, 2048 -> 2 x 1792 39.7 / 38.7, 512 rows, 2048
  // -> 2 x 3584 36.6 / 36.0, K = 1024 level.
  if (bk == BK_MXFP4 && !is_gate_up(epi) && t.t128 >= 192 && t.t128 <= 256 && kt <= 32) return 0;
  const Rates& r = rates(ak, bk);
  const double tiled = t.t128 < 192 ? 17 + kt * 0.32 : t.t128 <= 256 ? 7 + kt * r.deep : r.start + kt * r.tiled * t.t128 / 256;
  return tiled <= std::min(t.us256, t.us128) ? 0 : t.us256 <= t.us128 ? 256 : 128;
}

// Sizes off the 64-wide grid: against streaming and the K-step-32 kernel
// (mx_stream.cpp).  us, the faster of those -> here: MXFP4 MLPs of 1374 tokens,
// 2336 -> 13472, 711 -> 282; 1126 tokens, 1888 -> 5248, 139 -> 83; 2685 tokens, 2144
// -> 4736, 361 -> 168; FP8 455 tokens, 5920 -> 6048, 294 -> 147; 1796 x 2560 x 2208
// 69 -> 36.
int tile_side_off_grid(int ak, int bk, int epi, int m, int n, int k) {
  if (ak != AK_F16 || !can(ak, bk, epi, k)) return 0;
  const Times t = times(ak, bk, epi, m, n, k);
  const double other = std::min(stream_time(ak, bk, epi, m, n, k), k32_time(ak, epi, m, n, k));
  return other <= std::min(t.us256, t.us128) ? 0 : t.us256 <= t.us128 ? 256 : 128;
}

bool tile_aligned(int bk, const QGemmArgs& g) {
  const uintptr_t p = reinterpret_cast<uintptr_t>(g.a) | reinterpret_cast<uintptr_t>(g.b0) | reinterpret_cast<uintptr_t>(g.b1);
  const uintptr_t s = reinterpret_cast<uintptr_t>(g.s0) | reinterpret_cast<uintptr_t>(g.s1);
  return p % 16 == 0 && s % (bk == BK_MXFP4 ? 1 : bk == BK_INT4G32 ? 2 : 4) == 0;
}

hipError_t launch_tile(int side, int ak, int bk, int epi, const QGemmArgs& g, hipStream_t st) {
  using namespace tile;
  if (ak == AK_I8) return launch_i8(epi, g, st);
  switch (bk) {
    case BK_MXFP4: return launch_mxfp4(side, epi, g, st);
    case BK_INT4G32: return launch_int4(side, epi, g, st);
    case BK_E4M3: return launch_e4m3(side, epi, g, st);
    case BK_E5M2: return launch_e5m2(side, epi, g, st);
    case BK_INT8: return launch_int8(side, epi, g, st);
    case BK_F16: return launch_f16(side, epi, g, st);
  }
  return hipErrorInvalidValue;
}

double tile_gemm_time(int ak, int bk, int epi, int m, int n, int k) {
  if (!tile_side(ak, bk, epi, m, n, k)) return HUGE_VAL;
  const Times t = times(ak, bk, epi, m, n, k);
  return std::min(t.us256, t.us128);
}

}  // namespace mx
