// mx_stream.cpp - which shapes the weight-streaming GEMM (mx_gemm_stream.h)
// takes, and with which tile.
#include "mx_stream.h"

#include <algorithm>
#include <cmath>

namespace mx {

using namespace stream;

namespace {

// Bytes of a workgroup's scale copy.
size_t scale_bytes(int bk, int ng, int k) {
  return bits4(bk) ? (size_t)16 * ng * (k / 32) * (bk == BK_INT4G32 ? 2 : 1) : 0;
}

// Megabytes of weight codes of the launch.
double weight_mb(int bk, int epi, int n, int k) {
  return (double)n * (is_gate_up(epi) ? 2 : 1) * k * (bits4(bk) ? 0.5 : bk == BK_F16 ? 2.0 : 1.0) * 1e-6;
}

// Rows of a tile.  32 at most: larger tiles leave one workgroup per CU, and a
// CU with two hides their start and end (40 tokens, 7168 -> 2 x 2048 channels:
// 11.9 us as two 32-row tiles, 13.6 as one of 48 rows; 257 tokens, 2080 -> 2 x
// 5536: 36 us against 47 with 64-row tiles).  f32 rows take twice the LDS.
int tile_rows(int ak, int m) { return m <= 4 && ak != AK_I8 ? 4 : m <= 8 ? 8 : m <= 16 || ak == AK_F32 ? 16 : 32; }

// Workgroups of a launch over the CUs of its fullest XCD (32 CUs each, weight
// tiles dealt out round robin, `tiles` row tiles to each).
double fill(int epi, int n, int ng, long tiles) {
  const int per = (is_gate_up(epi) ? 8 : 16) * ng, nt = (n + per - 1) / per;
  return (nt + 7) / 8 * tiles / 32.0;
}

// Time of a launch of 32-row (f32: 16-row) tiles, us, where the activations'
// way from L2 sets it: 3 for the launch and the last sums, and for each
// workgroup of a CU 2.4 to fill its ring and 0.043 a step and KB (8 of
// activations, 2 of 4-bit weights a group); two workgroups share a CU, a third
// starts as one ends.  Measured against it, K = 7168, 2048 channels, 40 tokens:
// 1 / 2 / 4 groups 17.4 / 11.8 / 16.3 (model 19.8 / 12.6 / 15.0); K = 5536, N =
// 2080, 64 tokens: 14.9 / 11.5 / 17.7 (17.3 / 11.1 / 13.0); 130 tokens, 1024 ->
// 2 x 4096: 19.5 / 14.4 / 12.6 (23.6 / 14.2 / 9.4).
double tile_time(int bk, int epi, int n, int k, int ng, long tiles) {
  const double f = fill(epi, n, ng, tiles), kb = 8 + ng * (bits4(bk) ? 2 : bk == BK_F16 ? 8 : 4);
  const double work = 0.043 * (k / 128.0 / 4) * kb;
  return 3.0 + (f > 2 ? f * (1.2 + work) : (f > 1 ? 2 : 1) * (2.4 + work));
}

// Groups of 16 weight rows of a workgroup: the activations are read once per
// workgroup, so more groups as long as enough workgroups remain.  32-row tiles:
// by tile_time.  Below, the weights are most of the traffic and more workgroups
// keep more of them in flight; measured (us, MXFP4, 1 / 2 / 4 groups): 8
// tokens, 4096 -> 2 x 14336 (3584 groups in all) 20.0 / 17.9 / 16.4, its down
// pass (256 groups) 11.4 / 14.4 / -; 16 tokens, 2048 -> 7168 (448) 6.1 / 5.4 /
// 7.4; 1 token, 2080 -> 2 x 5536 (692) 7.9 / 8.4 / 9.3.
int groups_of(int ak, int bk, int epi, int rows, int n, int k, long tiles) {
  const int per = is_gate_up(epi) ? 8 : 16, most = bk == BK_F16 ? 2 : 4;
  int ng = 1;
  for (int c = 2; c <= most && scale_bytes(bk, c, k) <= kScales; c *= 2) {
    if (rows == (ak == AK_F32 ? 16 : 32)) {
      if (tile_time(bk, epi, n, k, c, tiles) < tile_time(bk, epi, n, k, ng, tiles)) ng = c;
    } else if ((n + per * c - 1) / (per * c) * tiles >= (rows == 4 || c == 4 ? 400 : 200)) {
      ng = c;
    }
  }
  return ng;
}

Args args_of(int epi, const QGemmArgs& q) {
  auto u8 = [](const void* p) { return static_cast<const uint8_t*>(p); };
  return Args{q.a, q.a_scale, u8(q.b0), u8(q.b1), u8(q.s0), u8(q.s1), q.c, q.m, q.n, q.k, epi, 0, 0};
}

// What the kernel can run: its scale copy, and offsets in 32 bits.
bool can(int ak, int bk, int epi, int n, int k) {
  if (k % 32 || k > (1 << 20) || (size_t)n * (is_gate_up(epi) ? 2 : 1) > (1u << 30) || scale_bytes(bk, 1, k) > kScales) return false;
  const bool store = epi == EPI_STORE_F32 || epi == EPI_STORE_F16;
  if (ak == AK_I8) return bk == BK_I8 && k % 128 == 0 && (store || epi == EPI_STORE_I32 || epi == EPI_SWIGLU_F32);
  if (ak == AK_F32) return (bk == BK_F16 || bk == BK_MXFP4) && store;
  return ak == AK_F16 && bk != BK_I8 && (store || epi == EPI_SWIGLU_F16 || epi == EPI_SWIGLU_HALF);
}

}  // namespace

// Time of a launch, us: 2 for it, its first loads and its sums, and for each
// workgroup of a CU 0.055 a step and KB and 0.65 (4-bit weights) to 1.5 a group
// of weight rows for its scales and its outputs; two share a CU, further ones
// start as one ends.  Or, if that is more, each row tile's read of the weights
// at 4.6 TB/s.  Fitted to 1700 GEMMs of 17 to 4097 rows, K of 64 to 16384; half
// of them are within 5 %, nine in ten within 17 %.
double stream_time(int ak, int bk, int epi, int m, int n, int k) {
  if (!can(ak, bk, epi, n, k)) return HUGE_VAL;
  struct Rate { double start, wg, kb, group; };
  const Rate r = ak == AK_I8 ? Rate{2.8, -1.8, 0.05, 1.45} : ak == AK_F32 ? Rate{1.9, 0.3, 0.055, 0.9}
                 : bits4(bk) ? Rate{2.3, 0, 0.055, 0.65} : bk == BK_F16 ? Rate{1.5, 0.3, 0.052, 1.2} : Rate{2.1, 0, 0.058, 0.9};
  const int rows = tile_rows(ak, m), tiles = (m + rows - 1) / rows;
  const int ng = groups_of(ak, bk, epi, rows, n, k, tiles);
  const double f = fill(epi, n, ng, tiles), kb = 8 + ng * (bits4(bk) ? 2 : bk == BK_F16 ? 8 : 4);
  const double wg = r.wg + r.kb * (k / 512.0) * kb + r.group * ng;
  const double rounds = f > 2 ? (f + std::ceil(f)) / 2 : f > 1 ? 1.84 : 0.92;
  return std::max(2.5 + tiles * weight_mb(bk, epi, n, k) / 4.6, r.start + std::max(0.3, rounds * wg));
}

// Rounds that workgroups filling the chip x > 1 times take: between x (they start
// as others end) and whole ones.
static double rounds_of(double x) { return x > 1 ? (x + std::ceil(x)) / 2 : x; }

// Time of `stages` K stages of the 64-K-stage family, us: a workgroup's own
// latency a stage, or where more, the rate of a full chip.  Narrow: 64 weight rows
// a workgroup, else 128.  Fitted to 2400 GEMMs with tiled_time, half of them
// within 6 %, nine in ten within 19 %.
static double stages_time(int ak, int bk, bool narrow, double stages, double workgroups) {
  struct Rate { double own, full; };
  struct Rates { double start; Rate narrow, wide; };
  const Rates r = ak == AK_F32 ? Rates{3.5, {1.21, 1.11}, {1.48, 1.79}} : ak == AK_I8 ? Rates{5.6, {0.49, 0.7}, {0.49, 0.7}}
                  : bk == BK_F16 ? Rates{2.8, {0.28, 0.38}, {0.5, 0.62}} : bk == BK_INT4G32 ? Rates{3.5, {0.42, 0.41}, {0.65, 0.67}}
                  : bk == BK_MXFP4 ? Rates{3.25, {0.41, 0.37}, {0.56, 0.56}} : Rates{4.7, {0.3, 0.39}, {0.52, 0.55}};
  const Rate& w = narrow ? r.narrow : r.wide;
  return r.start + stages * std::max(w.own, w.full * rounds_of(workgroups / 256));
}

// Time of the 64-K-stage family, us: its stages, a split's partials at 2.3 MB a us
// and their sum, or the weights at 3.3 TB/s (W8A8 4.6).
static double tiled_time(int ak, int bk, int epi, int m, int n, int k) {
  const int s = gemm_q_splits(ak, bk, epi, m, n, k);
  const bool narrow = !is_gate_up(epi) && (n % 128 != 0 || (bk == BK_MXFP4 && n / 128 < 16));  // as wide_tiles of mx_gemm_q.hip
  const long tiles = (long)((m + 127) / 128) * (is_gate_up(epi) || narrow ? n / 64 : n / 128);
  double t = stages_time(ak, bk, narrow, (double)k / (ak == AK_I8 ? 128 : 64) / s, (double)tiles * s);
  const bool bytes = bk == BK_E4M3 || bk == BK_E5M2 || bk == BK_INT8 || bk == BK_I8;
  if (s > 1) t += (bytes ? 0.4 : 1.5) + 0.25 * s + 0.43 * s * (is_gate_up(epi) ? 2 : 1) * m * n * 4e-6;
  // one 64 x 64-channel gate/up tile per CU (34 rows, 2560 -> 2 x 12416: 14.1
  // us against 26.0 streaming; 512 rows, 7168 -> 2 x 2048: 31)
  if (bk == BK_MXFP4 && kq_gemm_ok(ak, epi, m, n, k)) t = std::min(t, 4.7 + 0.0037 * k);
  return std::max(t, weight_mb(bk, epi, n, k) / (ak == AK_I8 ? 4.6 : 3.3));
}

// Time of the K-step-32 kernel, us, of 64 columns x 64 rows a workgroup, or 128
// rows from 256 such workgroups on: a serial loop over K of 0.009 to 0.017 us a K
// (f32 rows 0.0126 to 0.02), the same for sizes that look alike.  Taken at 1.3
// times the low end, the choice between it, streaming and the tile kernel is 1.2 %
// from the fastest on average over 490 GEMMs off the grid (2 to 4000 rows); with
// a fixed rate for streaming instead of its estimate it was 10.5 %.
double k32_time(int ak, int epi, int m, int n, int k) {
  const long cols = (n + 63) / 64, w128 = cols * ((m + 127) / 128);
  const bool big = m > 64 && w128 >= 256;
  const double a_k = (ak == AK_F32 ? 0.0164 : 0.0117) * (is_gate_up(epi) ? 1.42 : 1) * (big ? ak == AK_F32 ? 1.44 : 1.08 : 1);
  const double x = (big ? w128 : cols * ((m + 63) / 64)) / 256.0;
  return (2.9 + a_k * k) * std::max(1.0, 0.6 * x + 0.4 * std::ceil(x));
}

// Up to 16 rows streaming wins for any K that a model has; from there the
// faster estimate.  Both sides measured, us, tiled -> streaming:
//   MXFP4  4096 -> 2 x 14336  16: 22.6 -> 18.4  32: 23.4 -> 22.2  64: 26.5 -> 36.4
//          7168 -> 2 x 2048   16: 18.7 -> 9.2   64: 21.0 -> 12.4  128: 21.2 -> 21.3
//          2048 -> 2 x 5632   16: 16.0 -> 7.7   128: 21.5 -> 17.6 256: 31.5 -> 31.0
//          512 -> 3648        1001: 9.2 -> 24.7
//   FP8    4096 -> 2 x 14336  16: 34.1 -> 27.7  32: 35.8 -> 32.4  48: 36.0 -> 56.4
//          7168 -> 2 x 2048   16: 19.8 -> 10.4  64: 20.8 -> 17.6  96: 20.9 -> 30.1
//          2048 -> 7168       64: 16.0 -> 12.5  96: 17.9 -> 19.0
//          256 -> 2 x 1408    385: 4.8 -> 15.6
//   INT4   4096 -> 2 x 14336  16: 42.5 -> 20.0  64: 44.9 -> 40.6  96: 46.7 -> 57.5
//   W8A8   7168 -> 2 x 2048   16: 17.9 -> 10.3  64: 18.6 -> 14.3  128: 19.5 -> 23.9
//          2048 -> 2 x 5632   32: 13.4 -> 11.4  48: 14.1 -> 17.7
//   f16    4096 -> 4096       16: 14.6 -> 9.6   32: 14.6 -> 11.6  128: 17.9 -> 27.3
//   f32 rows x MXFP4  4096 -> 4096  64: 24.7 -> 15.4  256: 43.4 -> 40.0  1024: 125 -> 169
// Over the measured GEMMs this is 0.5 % from the faster side on average.  With a
// flat time for the tiled family, whatever its K, it was 6.5 %, and below 1024 K up
// to 6 times the tiled time.
bool stream_wins(int ak, int bk, int epi, int m, int n, int k) {
  if (!can(ak, bk, epi, n, k)) return false;
  return m <= 16 || stream_time(ak, bk, epi, m, n, k) <=
                        std::min(tiled_time(ak, bk, epi, m, n, k), tile_gemm_time(ak, bk, epi, m, n, k));
}

// Against the K-step-32 kernel (sizes off the 64-wide grid).  Measured, us,
// K-step-32 -> streaming: MXFP4 257 tokens 2080 -> 2 x 5536 81 -> 36, 5536 -> 2080
// 125 -> 23; 1024 tokens 95 -> 117 and 165 -> 77; 1 x 5536 -> 2080 108 -> 5.9; 1078
// tokens, 96 -> 3360 6.3 -> 20.6; f32 rows 1536 x 864 x 128 4.8 -> 31.7.
bool stream_wins_off_grid(int ak, int bk, int epi, int m, int n, int k) {
  return can(ak, bk, epi, n, k) && stream_time(ak, bk, epi, m, n, k) <= k32_time(ak, epi, m, n, k);
}

hipError_t launch_stream(int ak, int bk, int epi, const QGemmArgs& q, hipStream_t st) {
  const int rows = tile_rows(ak, q.m);
  const int ng = groups_of(ak, bk, epi, rows, q.n, q.k, (q.m + rows - 1) / rows);
  const Args g = args_of(epi, q);
  if (ak == AK_I8) return launch_i8(g, rows, ng, st);
  if (ak == AK_F32) return bk == BK_F16 ? launch_f32_f16(g, rows, ng, st) : launch_f32_mxfp4(g, rows, ng, st);
  switch (bk) {
    case BK_F16: return launch_f16(g, rows, ng, st);
    case BK_MXFP4: return launch_mxfp4(g, rows, ng, st);
    case BK_E4M3: return launch_e4m3(g, rows, ng, st);
    case BK_E5M2: return launch_e5m2(g, rows, ng, st);
    case BK_INT8: return launch_int8(g, rows, ng, st);
    case BK_INT4G32: return launch_int4(g, rows, ng, st);
  }
  return hipErrorInvalidValue;
}

namespace {

// MoE: tile rows and groups of weight rows of a launch over experts of uneven
// sizes.  16-row tiles leave three workgroups per CU: better while most experts
// have fewer rows than that (64 experts, 256 tokens, 7168 -> 2048, largest 25: 281
// us, 304 with 32-row tiles; 64 experts with 1024 tokens 444 against 403).
struct Grouped {
  int rows, ng;
  long active;
};
Grouped grouped_of(int epi, int n, int k, const GroupTable& gt, int groups) {
  int most = 0;
  long active = 0;
  for (int e = 0; e < groups; e++) {
    most = std::max(most, gt.off[e + 1] - gt.off[e]);
    active += gt.off[e + 1] > gt.off[e];
  }
  int rows = tile_rows(AK_F16, most);
  if (rows == 32 && gt.off[groups] < 16 * active) rows = 16;
  return {rows, groups_of(AK_F16, BK_MXFP4, epi, rows, n, k, active), active};
}

// stream_time's and tiled_time's terms over experts: an expert's last row tile
// costs its own body's activations, and the 128-row family pays a whole tile for
// it.  The weights once, at 4.6 and 3.3 TB/s.
double grouped_stream_time(int epi, int n, int k, const GroupTable& gt, int groups) {
  const Grouped l = grouped_of(epi, n, k, gt, groups);
  auto workgroup = [&](int rows) {
    const int kb = rows > 16 ? 8 : rows > 8 ? 4 : 2;
    return 0.055 * (k / 512.0) * (kb + 2 * l.ng) + 0.65 * l.ng;
  };
  double per_cu = 0;  // for one weight tile of every CU
  for (int e = 0; e < groups; e++) {
    const int t = gt.off[e + 1] - gt.off[e], full = t / l.rows, rest = t % l.rows;
    per_cu += full * workgroup(l.rows) + (rest ? workgroup(rest) : 0);
  }
  per_cu *= fill(epi, n, l.ng, 1);
  return std::max(2.3 + std::max(per_cu, workgroup(32)), 2.5 + l.active * weight_mb(BK_MXFP4, epi, n, k) / 4.6);
}
double grouped_tiled_time(int epi, int n, int k, const GroupTable& gt, int groups) {
  long tiles = 0, active = 0;
  for (int e = 0; e < groups; e++) {
    const int t = gt.off[e + 1] - gt.off[e];
    tiles += (t + 127) / 128;
    active += t > 0;
  }
  const bool narrow = !is_gate_up(epi) && n % 128 != 0;
  tiles *= is_gate_up(epi) || narrow ? n / 64 : n / 128;
  return std::max(stages_time(AK_F16, BK_MXFP4, narrow, k / 64.0, (double)tiles), active * weight_mb(BK_MXFP4, epi, n, k) / 3.3);
}

}  // namespace

// From 1024 K on, below 20 rows an expert (72 from 4096 K on): the 128-row tiles are
// mostly padding, and the weights, read from HBM, are most of the time.  us a pass,
// tiled -> streaming: 64 experts, 256 tokens, 7168 -> 2048, largest 25: 712 -> 281; 32
// experts, 2000 tokens, 4096 -> 1408: 276 -> 219; 8 experts, 512 tokens, 7168 -> 2048:
// 166 -> 130.  Of 374 GEMMs of at least 1024 x 1024, 2 are over 5 % of a pass faster
// on the other side of that line; below it, shorter K (64 experts, 878 tokens, 448 ->
// 320: 18 -> 31) and above it the estimates decide, with a fifth for what they miss:
// 8 experts, 1024 tokens, 4096 -> 1408: 90 -> 104; 32 experts, 838 tokens, 1408 ->
// 1792: 73 -> 82; 886 tokens, 1408 -> 1664: 67 -> 76; 3005 tokens, 2304 -> 1024: 101
// -> 153.  Over 590 MoE shapes (2 to 128 experts, K of 64 to 7168) a GEMM is 1.5 %
// of a pass from the faster side on average; the line in rows alone, for any K,
// was 12 %.
bool stream_wins_grouped(int epi, int n, int k, const GroupTable& gt, int groups) {
  if (!can(AK_F16, BK_MXFP4, epi, n, k)) return false;
  if (k >= 1024 && gt.off[groups] < (k >= 4096 ? 72L : 20L) * grouped_of(epi, n, k, gt, groups).active) return true;
  return 1.2 * grouped_stream_time(epi, n, k, gt, groups) <= grouped_tiled_time(epi, n, k, gt, groups);
}

hipError_t launch_stream_grouped(int epi, const QGemmArgs& q, const GroupTable& gt, int groups, hipStream_t st) {
  const Grouped l = grouped_of(epi, q.n, q.k, gt, groups);
  return launch_mxfp4_grouped(args_of(epi, q), gt, groups, l.rows, l.ng, st);
}

}  // namespace mx
