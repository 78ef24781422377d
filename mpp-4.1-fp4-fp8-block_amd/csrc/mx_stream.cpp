// mx_stream.cpp - which shapes the weight-streaming GEMM (mx_gemm_stream.h)
// takes, and with which tile.
#include "mx_stream.h"

#include <algorithm>

namespace mx {

using namespace stream;

namespace {

bool bits4(int bk) { return bk == BK_MXFP4 || bk == BK_INT4G32; }

// Bytes of a workgroup's scale copy.
size_t scale_bytes(int bk, int ng, int k) {
  return bits4(bk) ? (size_t)16 * ng * (k / 32) * (bk == BK_INT4G32 ? 2 : 1) : 0;
}

// Megabytes of weight codes of the launch.
double weight_mb(int bk, int epi, int n, int k) {
  return (double)n * (is_dual(epi) ? 2 : 1) * k * (bits4(bk) ? 0.5 : bk == BK_F16 ? 2.0 : 1.0) * 1e-6;
}

// Rows of a tile.  32 at most: larger tiles leave one workgroup per CU, and a
// CU with two hides their start and end (40 tokens, 7168 -> 2 x 2048 channels:
// 11.9 us as two 32-row tiles, 13.6 as one of 48 rows; 257 tokens, 2080 -> 2 x
// 5536: 36 us against 47 with 64-row tiles).  f32 rows take twice the LDS.
int tile_rows(int ak, int m) { return m <= 4 && ak != AK_I8 ? 4 : m <= 8 ? 8 : m <= 16 || ak == AK_F32 ? 16 : 32; }

// Workgroups of a launch over the CUs of its fullest XCD (32 CUs each, weight
// tiles dealt out round robin, `tiles` row tiles to each).
double fill(int epi, int n, int ng, long tiles) {
  const int per = (is_dual(epi) ? 8 : 16) * ng, nt = (n + per - 1) / per;
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
  const int per = is_dual(epi) ? 8 : 16, most = bk == BK_F16 ? 2 : 4;
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
  if (k % 32 || k > (1 << 20) || (size_t)n * (is_dual(epi) ? 2 : 1) > (1u << 30) || scale_bytes(bk, 1, k) > kScales) return false;
  const bool store = epi == EPI_STORE_F32 || epi == EPI_STORE_F16;
  if (ak == AK_I8) return bk == BK_I8 && k % 128 == 0 && (store || epi == EPI_STORE_I32 || epi == EPI_SWIGLU_F32);
  if (ak == AK_F32) return (bk == BK_F16 || bk == BK_MXFP4) && store;
  return ak == AK_F16 && bk != BK_I8 && (store || epi == EPI_SWIGLU_F16 || epi == EPI_SWIGLU_HALF);
}

}  // namespace

// The tiled family's time is almost flat up to 128 rows (its tile) and set by
// the latency of its K stages; this kernel's grows with row tiles x weight
// bytes.  Both sides measured at 1 to 256 rows, us, tiled -> streaming:
//   MXFP4  4096 -> 2 x 14336  16: 22.6 -> 18.4  32: 23.4 -> 22.2  64: 26.5 -> 36.4
//          7168 -> 2 x 2048   16: 18.7 -> 9.2   64: 21.0 -> 12.4  128: 21.2 -> 21.3
//          2048 -> 2 x 5632   16: 16.0 -> 7.7   128: 21.5 -> 17.6 256: 31.5 -> 31.0
//   FP8    4096 -> 2 x 14336  16: 34.1 -> 27.7  32: 35.8 -> 32.4  48: 36.0 -> 56.4
//          7168 -> 2 x 2048   16: 19.8 -> 10.4  64: 20.8 -> 17.6  96: 20.9 -> 30.1
//          5632 -> 2048       128: 17.5 -> 14.2 256: 18.3 -> 23.6
//          2048 -> 7168       64: 16.0 -> 12.5  96: 17.9 -> 19.0
//   INT4   4096 -> 2 x 14336  16: 42.5 -> 20.0  64: 44.9 -> 40.6  96: 46.7 -> 57.5
//   W8A8   7168 -> 2 x 2048   16: 17.9 -> 10.3  64: 18.6 -> 14.3  128: 19.5 -> 23.9
//          2048 -> 2 x 5632   32: 13.4 -> 11.4  48: 14.1 -> 17.7
//   f16    4096 -> 4096       16: 14.6 -> 9.6   32: 14.6 -> 11.6  128: 17.9 -> 27.3
//   f32 rows x MXFP4  4096 -> 4096  64: 24.7 -> 15.4  256: 43.4 -> 40.0  1024: 125 -> 169
//   FP8, K stages that do not split (167): 10688 -> 7168, 40 rows, 97 us tiled
// Up to 16 rows it always wins.  From there both sides are estimated: this
// kernel at 5 us + row tiles x weight bytes at 4.6 TB/s, or tile_time if that
// is more; the tiled family at its flat time (19 us; single GEMMs with 8-bit
// weights and short W8A8 passes 14, f32 rows 34), the weights at 3.3 TB/s (W8A8
// 4.6), or half a us for each K stage of a split.
bool stream_wins(int ak, int bk, int epi, int m, int n, int k) {
  if (!can(ak, bk, epi, n, k)) return false;
  if (m <= 16) return true;
  const int rows = tile_rows(ak, m), tiles = (m + rows - 1) / rows;
  const int ng = groups_of(ak, bk, epi, rows, n, k, tiles);
  const double mb = weight_mb(bk, epi, n, k);
  const double here = std::max(5.0 + tiles * mb / 4.6, tile_time(bk, epi, n, k, ng, tiles));
  const double flat = ak == AK_F32 ? 34.0 : ak == AK_I8 ? (k >= 4096 ? 19.0 : 14.0)
                      : !bits4(bk) && !is_dual(epi) ? 14.0 : 19.0;
  const int stages = k / (ak == AK_I8 ? 128 : 64) / gemm_q_splits(ak, bk, epi, m, n, k);
  return here <= std::max({flat, mb / (ak == AK_I8 ? 4.6 : 3.3), 0.5 * stages});
}

// Against the K-step-32 kernel (sizes off the 64-wide grid), whose time is at
// least about 0.0225 us per K (one tile's serial loop) and else its rate:
// streaming runs these shapes at about 330 (4-bit) or 250 TFLOP/s (f32 rows:
// 180).  Measured, us, K-step-32 -> streaming: MXFP4 257 tokens 2080 -> 2 x
// 5536 81 -> 36, 5536 -> 2080 125 -> 23; 1024 tokens 95 -> 117 and 165 -> 77;
// 4096 tokens 338 -> 476 and 233 -> 286; 1 x 5536 -> 2080 108 -> 5.9.
bool stream_wins_off_grid(int ak, int bk, int epi, int m, int n, int k) {
  if (!can(ak, bk, epi, n, k)) return false;
  const double rate = ak == AK_F32 ? 1.8e8 : bits4(bk) ? 3.3e8 : 2.5e8;  // flop per us
  return 2.0 * m * n * (is_dual(epi) ? 2 : 1) * k <= rate * (0.0225 * k + 10.0);
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

// MoE: experts of uneven sizes.  Below about 72 rows an expert on average (20
// for a short K) the 128-row tiles of the tiled family are mostly padding (us,
// tiled -> streaming: 64 experts, 256 tokens, 7168 -> 2048, largest 25: 712 ->
// 281; 32 experts, 2000 tokens, 4096 -> 1408: 276 -> 219; 8 experts, 512
// tokens, 7168 -> 2048: 166 -> 130; 8 experts, 1024 tokens, 4096 -> 1408: 90 ->
// 104; 32 experts, 838 tokens, 1408 -> 1792: 73 -> 82; 3005 tokens, 2304 ->
// 1024: 101 -> 153; 8 experts, 286 tokens, 3328 -> 1792: 49 -> 51; 64
// experts, 1470 tokens, 1408 -> 1664: 125 -> 137).
// 16-row tiles leave three workgroups per CU: better while most experts have
// fewer rows than that (the first of these 304 us with 32-row tiles, 64
// experts with 1024 tokens 444 against 403).
bool stream_wins_grouped(int epi, int n, int k, const GroupTable& gt, int groups) {
  int active = 0;
  for (int e = 0; e < groups; e++) active += gt.off[e + 1] > gt.off[e];
  return can(AK_F16, BK_MXFP4, epi, n, k) && gt.off[groups] < (k >= 4096 ? 72L : 20L) * active;
}

hipError_t launch_stream_grouped(int epi, const QGemmArgs& q, const GroupTable& gt, int groups, hipStream_t st) {
  long active = 0;
  for (int e = 0; e < groups; e++) active += gt.off[e + 1] > gt.off[e];
  int rows = tile_rows(AK_F16, q.m);
  if (rows == 32 && gt.off[groups] < 16 * active) rows = 16;
  return launch_mxfp4_grouped(args_of(epi, q), gt, groups, rows, groups_of(AK_F16, BK_MXFP4, epi, rows, q.n, q.k, active), st);
}

}  // namespace mx
