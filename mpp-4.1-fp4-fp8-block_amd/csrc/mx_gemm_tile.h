// mx_gemm_tile.h - prefill GEMMs: 256 x 256 and 128 x 128 output tiles, f16 or
// int8 activations against any weight format.
//
//   C[m][n] = sum_k A[m][k] * W[n][k]   (epilogue: store, SwiGLU, row scales)
//
// Bound: the f16 matrix cores, busy 83 to 89 %.  4096 tokens, 4096 -> 2 x 14336 ->
// 4096 with MXFP4 weights run at 1.45 PFLOP/s; on a card where they run at 1.33,
// library products of 16384 reach 1.23 in f16 and 1.31 in bf16.  Per K stage a
// CU's four SIMDs need 2048 clocks for a 256-tile's MFMAs and the rest has to fit
// beneath them:
//   LDS read    a wave owns 128 x 64 of the tile (T = 128: 64 x 64), 192 rows
//               of fragments for 8192 outputs; four waves of 128 x 128 read a
//               third less but leave one wave a SIMD, whose waits then show
//               (692 against 670 us gate/up, 338 against 332 down).
//   L2 -> LDS   a CU takes in 50 to 70 bytes a ns by DMA, whatever the ring's
//               depth or the cache policy: 40 KB a stage for the 256-tile
//               (0.6 us of 1.06), 20 KB for a quarter of the work with the
//               128-tile (0.35 of 0.41, its bound).  With int8 activations
//               (64 KB stages of 128 K, two slots) the matrix cores are busy 52 %
//               at 28 bytes a ns: waves wait at the barrier for a stage's last
//               loads, and four slots of half a stage were no faster.
//   widening    in registers, one k-step ahead of its MFMAs, spread between
//               them (sched_group_barrier; 1017 -> 1000 us for the MLP).
// The weights stay in their stored form up to the registers: a 64-K stage of a
// 256-tile is 32 KB of f16 activations and 8 (4-bit), 16 (8-bit) or 32 KB of
// weights, so 4, 3 or 2 stages fit the 160 KB of LDS; T = 128 has the same
// ring in 80 KB, two workgroups a CU.  One barrier a stage, before its last
// k-step: by then every fragment of the stage is in registers, so its slot is
// free, and the next stage's fragments are read past it.  Each slot is an array
// of its own, which is how the compiler's waits tell them apart.  Any n, and K in
// steps of 32: what lies past a row or past K reads as zero, by the DMA's range
// check.
//
// Measured, us, gate/up + down, 128-row tiles of mx_gemm_q.hip -> here, 4096
// tokens 4096 -> 2 x 14336 -> 4096: MXFP4 951 + 484 -> 670 + 330, E4M3 889 + 450
// -> 706 + 347, INT4 1061 + 534 -> 827 + 411, W8A8 568 + 264 -> 472 + 200.  1000
// tokens, MXFP4, T = 128: down 152 -> 105.
#pragma once

#include <type_traits>

#include "mx_device.h"
#include "mx_dma.h"
#include "mx_internal.h"
#include "mx_tile.h"
#include "mx_widen.h"

namespace mx {
namespace tile {

// bytes of a weight row per stage (64 K; int8 activations 128)
constexpr int rb_of(int bk) { return bk == BK_F16 || bk == BK_I8 ? 128 : bits4(bk) ? 32 : 64; }
constexpr int slots_of(int bk) { return rb_of(bk) == 128 ? 2 : bits4(bk) ? 4 : 3; }
constexpr int wait_lgkm0_vm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4); }

// Scales by which the load of scale group g starts early, so that it ends with
// the row's n scales (n >= 8).  Groups past the row (read ahead, never used)
// stay at 7: a shift below the group's width.
__host__ __device__ constexpr int late_scales(int g, int n) {
  const int late = g * 8 - (n - 8);
  return late < 0 ? 0 : late > 7 ? 7 : late;
}
static_assert(late_scales(0, 8) == 0 && late_scales(1, 16) == 0 && late_scales(1, 9) == 7 && late_scales(1, 15) == 1, "last group");
static_assert(late_scales(1, 8) == 7 && late_scales(2, 9) == 7, "past the last group");

// 16-byte chunks of a row are stored at chunk ^ swz(row): the 32 lanes of a
// fragment read, one row each, then cover all banks.
template <int R>
__device__ __forceinline__ int swz(int row) {
  constexpr int C = R / 16, RPL = 16 / C;
  return (row / RPL) % C;
}

template <int AK, int BK, int EPI, int T>
__global__ __launch_bounds__(T * 2, 2) void k_tile(QGemmArgs g, int n_tiles) {
  static_assert(T == 256 || T == 128, "tile side");
  constexpr bool DUAL = is_gate_up(EPI), S4 = bits4(BK);
  constexpr int KS = AK == AK_I8 ? 128 : 64, RA = 128, RB = rb_of(BK), NS = slots_of(BK);
  constexpr int NW = T / 32;
  constexpr int SLOT = T * (RA + RB), BO = T * RA;
  constexpr int NA = T * RA / 1024 / NW, NBI = T * RB / 1024 / NW, PER = NA + NBI;
  constexpr int NJ = 2, MI = T / 64, RW = 32;  // a wave: 32 MI rows x 64 weight rows; it moves 32 rows of each
  constexpr int BR = RB / 32;               // 16-byte reads of a weight row per lane and stage
  constexpr int ESZ = BK == BK_INT4G32 ? 2 : 1;
  using Acc = typename std::conditional<AK == AK_I8, v16i, v16f>::type;
  __shared__ __attribute__((aligned(16))) uint8_t r0[SLOT];
  __shared__ __attribute__((aligned(16))) uint8_t r1[SLOT];
  __shared__ __attribute__((aligned(16))) uint8_t r2[NS > 2 ? SLOT : 16];
  __shared__ __attribute__((aligned(16))) uint8_t r3[NS > 3 ? SLOT : 16];

  const int tid = threadIdx.x, lane = tid & 63, r32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int M = g.m, N = g.n, K = g.k, KT = (K + KS - 1) / KS;
  const int MT = g.tiles_m;
  // an XCD takes a contiguous run of tiles, walked as 8 weight tiles x all row tiles
  const int tiles = MT * n_tiles, bid = blockIdx.x;
  const int per = tiles / 8, rem = tiles % 8, x = bid & 7;
  const int tile = (x * per + min(x, rem)) + (bid >> 3);
  const int grp = tile / (8 * MT), in = tile % (8 * MT), gw = min(8, n_tiles - grp * 8);
  const int m0 = __builtin_amdgcn_readfirstlane(in / gw * T), nt = __builtin_amdgcn_readfirstlane(grp * 8 + in % gw);
  const int n0 = nt * (DUAL ? T / 2 : T);
  const int a_row = K * (AK == AK_I8 ? 1 : 2);
  const int b_row = AK == AK_I8 || !(S4 || BK == BK_F16) ? K : S4 ? K / 2 : K * 2;

  // ---- DMA: wave w moves tile rows [32 w, +32) of A and of B, whole rows of
  // a stage per instruction; rows past the end read as zero
  const v4i ars = rsrc_of<true>(reinterpret_cast<const uint8_t*>(g.a) + (size_t)m0 * a_row, (uint32_t)min(T, M - m0) * a_row);
  const int bfirst = DUAL ? n0 + (wave & (NW / 2 - 1)) * RW : n0 + wave * RW;
  const uint8_t* bsrc = reinterpret_cast<const uint8_t*>(DUAL && wave >= NW / 2 ? g.b1 : g.b0) + (size_t)min(bfirst, N - 1) * b_row;
  const v4i brs = rsrc_of<true>(bsrc, (uint32_t)max(0, min(RW, N - bfirst)) * (uint32_t)b_row);
  // (K % 64 == 32: the upper half of the last stage reads as zero too)
  constexpr int kPast = 0x40000000;  // past every row range
  const int half_stage = K % KS ? KT - 1 : -1;
  int a_off[NA], b_off[NBI], a_up[NA], b_up[NBI];
#pragma unroll
  for (int q = 0; q < NA; q++) {
    const int r = wave * RW + q * 8 + lane / 8;
    const int c = (lane % 8) ^ swz<RA>(r);
    a_off[q] = r * a_row + (c << 4);
    a_up[q] = c >= 4 ? kPast : 0;
  }
  constexpr int CB = RB / 16;
#pragma unroll
  for (int q = 0; q < NBI; q++) {
    const int r = q * (1024 / RB) + lane / CB;   // within the wave's rows
    const int c = (lane % CB) ^ swz<RB>(wave * RW + r);
    b_off[q] = r * b_row + (c << 4);
    b_up[q] = c >= CB / 2 ? kPast : 0;
  }
  auto slot = [&](auto u) -> uint8_t* {
    constexpr int U = decltype(u)::value;
    if constexpr (U == 0) return r0;
    else if constexpr (U == 1) return r1;
    else if constexpr (U == 2) return r2;
    else return r3;
  };
  auto issue = [&](int k, auto u) {
    uint8_t* s = slot(u);
    const int ao = k < KT ? k * RA : kPast, bo = k < KT ? k * RB : kPast, up = k == half_stage ? kPast : 0;
#pragma unroll
    for (int q = 0; q < NA; q++)
      buffer_dma16(ars, s + (wave * NA + q) * 1024, a_off[q] + ao + (a_up[q] & up));
#pragma unroll
    for (int q = 0; q < NBI; q++)
      buffer_dma16(brs, s + BO + (wave * NBI + q) * 1024, b_off[q] + bo + (b_up[q] & up));
  };

  // ---- fragments
  // block j of a wave: 32 weight rows (SwiGLU: the first half gate channels,
  // the second half the same up channels)
  constexpr int NC = DUAL ? NJ / 2 : NJ;           // column blocks of a wave's output
  auto blk = [&](int j) { return (wn * NC + j % NC) * 32 + (DUAL && j >= NC ? T / 2 : 0); };
  const uint8_t* sc_src[NJ];
  if constexpr (S4) {
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      const int row = min(n0 + (wn * NC + j % NC) * 32 + r32, N - 1);
      sc_src[j] = reinterpret_cast<const uint8_t*>(DUAL && j >= NC ? g.s1 : g.s0) + (size_t)row * (K / 32) * ESZ;
    }
  }
  constexpr int SW = ESZ * 2;  // dwords of a group's scales
  uint32_t scv[NJ][SW], scn[NJ][SW];  // this group's and the next's, by block
  // (rows of K / 32 scales start at any byte; the last group's load ends with
  // the row and is shifted down where it is first used: here it would be waited
  // for)
  auto scales = [&](int grp4, uint32_t (*d)[SW]) {
    if constexpr (S4) {
#pragma unroll
      for (int j = 0; j < NJ; j++) __builtin_memcpy(d[j], sc_src[j] + min(grp4 * (8 * ESZ), K / 32 * ESZ - 8 * ESZ), 8 * ESZ);
    }
  };
  auto to_scv = [&](int grp4) {
    const int sh = late_scales(grp4, K / 32) * (8 * ESZ);
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      uint64_t v[ESZ];
      __builtin_memcpy(v, scn[j], 8 * ESZ);
      if constexpr (ESZ == 2) {
        if (sh) {
          v[0] = sh >= 64 ? v[ESZ - 1] >> (sh & 63) : v[0] >> sh | v[ESZ - 1] << (64 - sh);
          v[ESZ - 1] = sh >= 64 ? 0 : v[ESZ - 1] >> sh;
        }
      } else {
        v[0] >>= sh;
      }
      __builtin_memcpy(scv[j], v, 8 * ESZ);
    }
  };
  // (the swizzles depend on row % 32 only: one lane part per k-step, constants
  // for the blocks)
  int la[4], lb[BR];
#pragma unroll
  for (int q = 0; q < 4; q++) la[q] = wm * (T / 2) * RA + r32 * RA + (((4 * h + q) ^ swz<RA>(r32)) << 4);
#pragma unroll
  for (int u = 0; u < BR; u++) lb[u] = blk(0) * RB + r32 * RB + (((BR * h + u) ^ swz<RB>(r32)) << 4);
  auto read_a = [&](const uint8_t* s, int ks, v4i* a) {
#pragma unroll
    for (int i = 0; i < MI; i++) a[i] = *reinterpret_cast<const v4i*>(s + la[ks] + i * 32 * RA);
  };
  auto read_b = [&](const uint8_t* s, v4i (*b)[BR]) {
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int u = 0; u < BR; u++) b[j][u] = *reinterpret_cast<const v4i*>(s + BO + lb[u] + (j % NC * 32 + (j >= NC ? T / 2 : 0)) * RB);
  };

  Acc acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0;

  issue(0, std::integral_constant<int, 0>{});
  __builtin_amdgcn_sched_barrier(0);
  scales(0, scn);
  __builtin_amdgcn_sched_barrier(0);
  issue(1, std::integral_constant<int, 1>{});
  if constexpr (NS > 2) issue(2, std::integral_constant<int, 2>{});
  if constexpr (NS > 3) issue(3, std::integral_constant<int, 3>{});
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(wait_lgkm0_vm((NS - 1) * PER));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  // One k-step's weights of block j, widened.
  auto widen = [&](const v4i* w, int ks, uint32_t sv) -> v8h {
    if constexpr (BK == BK_F16) {
      return __builtin_bit_cast(v8h, w[ks < BR ? ks : 0]);
    } else if constexpr (BK == BK_MXFP4) {
      return fp4x8_to_f16x8((uint32_t)w[0][ks], e8m0_as_cvt_scale(sv));
    } else if constexpr (BK == BK_INT4G32) {
      return i4x8_to_f16((uint32_t)w[0][ks], __builtin_bit_cast(_Float16, (uint16_t)sv));
    } else {
      const uint32_t lo = (uint32_t)w[BR > 1 ? ks >> 1 : 0][2 * (ks & 1)], hi = (uint32_t)w[BR > 1 ? ks >> 1 : 0][2 * (ks & 1) + 1];
      if constexpr (BK == BK_INT8) return i8x8_to_f16(lo, hi);
      else return fp8x8_to_f16<BK>(lo, hi);
    }
  };
  // scale of stage e of the group, block j
  auto scale_of = [&](auto ee, int j) -> uint32_t {
    constexpr int e = decltype(ee)::value * 2 * ESZ;
    if constexpr (S4) return scv[j][e / 4] >> (8 * (e % 4) + 8 * ESZ * h);
    else return 0u;
  };
  // A fragments and widened weights one k-step ahead of their MFMAs
  v4i af[2][MI], bf[NJ][BR];
  v8h bw[2][NJ];
  read_a(r0, 0, af[0]);
  if constexpr (S4) to_scv(0);
  read_b(r0, bf);
  if constexpr (AK != AK_I8) {
#pragma unroll
    for (int j = 0; j < NJ; j++) bw[0][j] = widen(bf[j], 0, scale_of(std::integral_constant<int, 0>{}, j));
  }
  auto stage = [&](int k, auto uu) {
    constexpr int U = decltype(uu)::value;
    const uint8_t* s = slot(std::integral_constant<int, U % NS>{});
    const uint8_t* sn = slot(std::integral_constant<int, (U + 1) % NS>{});
    v4i bn[NJ][BR];
    uint32_t sv[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) sv[j] = scale_of(std::integral_constant<int, S4 ? U : 0>{}, j);
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
      __builtin_amdgcn_sched_barrier(0);
      if (ks == 3) {
        // every fragment of stage k is in registers, stage k + 1 has landed:
        // slot k is free and slot k + 1 readable past the barrier
        __builtin_amdgcn_s_waitcnt(wait_lgkm0_vm((NS - 2) * PER));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        read_b(sn, bn);
      }
      read_a(ks < 3 ? s : sn, (ks + 1) & 3, af[(ks + 1) & 1]);
      if (ks == 3) {
        issue(k + NS, std::integral_constant<int, U % NS>{});
        if constexpr (S4 && U == 0) scales(k / 4 + 1, scn);
      }
      if (ks < 3) {
        if constexpr (AK != AK_I8) {
#pragma unroll
          for (int j = 0; j < NJ; j++) bw[(ks + 1) & 1][j] = widen(bf[j], ks + 1, sv[j]);
        }
      }
      const v4i* a = af[ks & 1];
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int i = 0; i < MI; i++) {
          if constexpr (AK == AK_I8)
            acc[i][j] = (Acc)__builtin_amdgcn_mfma_i32_32x32x32_i8(a[i], bf[j][ks < BR ? ks : 0], (v16i)acc[i][j], 0, 0, 0);
          else
            acc[i][j] = (Acc)mfma_f16_32x32x16(__builtin_bit_cast(v8h, a[i]), bw[ks & 1][j], (v16f)acc[i][j]);
        }
      if (ks == 3) {
        if constexpr (S4 && U == 3) to_scv(k / 4 + 1);
#pragma unroll
        for (int j = 0; j < NJ; j++) {
#pragma unroll
          for (int u = 0; u < BR; u++) bf[j][u] = bn[j][u];
          if constexpr (AK != AK_I8) bw[0][j] = widen(bf[j], 0, scale_of(std::integral_constant<int, S4 ? (U + 1) % 4 : 0>{}, j));
        }
      }
      // spread the k-step's reads, loads and widening over its MFMAs
#pragma unroll
      for (int t = 0; t < MI * NJ; t++) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if (ks == 3) __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, MI == 4 ? 2 : 4, 0);
      }
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  int k = 0;
  for (; k + NS <= KT; k += NS) {
    stage(k, I0{});
    stage(k + 1, I1{});
    if constexpr (NS > 2) stage(k + 2, I2{});
    if constexpr (NS > 3) stage(k + 3, I3{});
  }
  if (k < KT) {
    stage(k, I0{});
    if constexpr (NS > 2) {
      if (k + 1 < KT) {
        stage(k + 1, I1{});
        if constexpr (NS > 3) {
          if (k + 2 < KT) stage(k + 2, I2{});
        }
      }
    }
  }

  if constexpr (BK == BK_MXFP4) {
    // E8M0 byte 255 (+inf to the reference, NaN to the decode above) makes the
    // sums that it reaches NaN.  A wave with a NaN and such a byte among its
    // weight rows runs its K loop again from global memory, decoded as the
    // reference does; a NaN from x alone stands.
    bool nan = false;
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int v = 0; v < 16; v++) nan |= acc[i][j][v] != acc[i][j][v];
    if (__builtin_expect(__ballot(nan) != 0, 0)) {
      uint32_t hit = 0;
#pragma unroll
      for (int j = 0; j < NJ; j++)
        for (int t = 0; t < K / 32; t++) hit |= sc_src[j][t] == 255u;
      if (__ballot(hit != 0) != 0) {
        const uint8_t* ap[MI];
        const uint8_t* bp[NJ];
#pragma unroll
        for (int i = 0; i < MI; i++)
          ap[i] = reinterpret_cast<const uint8_t*>(g.a) + (size_t)min(m0 + wm * (T / 2) + i * 32 + r32, M - 1) * a_row + h * 64;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
          bp[j] = reinterpret_cast<const uint8_t*>(DUAL && j >= NC ? g.b1 : g.b0) +
                  (size_t)min(n0 + (wn * NC + j % NC) * 32 + r32, N - 1) * b_row + h * 16;
#pragma unroll
          for (int i = 0; i < MI; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0;
        }
#pragma unroll 1
        for (int t = 0; t < KT * 4; t++) {  // k-step t % 4 of stage t / 4
          const bool in = (t >> 2) * 64 + h * 32 < K;
          v4i a[MI];
#pragma unroll
          for (int i = 0; i < MI; i++) {
            a[i] = v4i{0, 0, 0, 0};
            if (in) a[i] = *reinterpret_cast<const v4i*>(ap[i] + (t >> 2) * RA + (t & 3) * 16);
          }
#pragma unroll
          for (int j = 0; j < NJ; j++) {
            uint32_t w = 0, sb = 0;
            if (in) {
              w = *reinterpret_cast<const uint32_t*>(bp[j] + t / 4 * RB + t % 4 * 4);
              sb = sc_src[j][t / 4 * 2 + h];
            }
            const v8h b = fp4x8_dequant_f16(w, sb);
#pragma unroll
            for (int i = 0; i < MI; i++) acc[i][j] = mfma_f16_32x32x16(__builtin_bit_cast(v8h, a[i]), b, acc[i][j]);
          }
        }
      }
    }
  }

  // ---- epilogue
  float cs[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    cs[j] = 1.0f;
    if constexpr (!S4 && BK != BK_F16 && EPI != EPI_STORE_I32)
      cs[j] = reinterpret_cast<const float*>(DUAL && j >= NC ? g.s1 : g.s0)[min(n0 + (wn * NC + j % NC) * 32 + r32, N - 1)];
  }
#pragma unroll
  for (int i = 0; i < MI; i++) {
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int row = m0 + wm * (T / 2) + i * 32 + acc32_row(lane, v);
      if (row >= M) continue;
      const float rs = AK == AK_I8 && EPI != EPI_STORE_I32 ? g.a_scale[row] : 1.0f;
#pragma unroll
      for (int j = 0; j < NC; j++) {
        const int col = n0 + (wn * NC + j) * 32 + r32;
        if (col >= N) continue;
        const size_t o = (size_t)row * N + col;
        if constexpr (EPI == EPI_STORE_I32) {
          reinterpret_cast<int*>(g.c)[o] = (int)acc[i][j][v];
        } else {
          // sum x row scale x column scale, in this order
          float x = (float)acc[i][j][v];
          if (AK == AK_I8) x = x * rs;
          x = x * cs[j];
          if constexpr (DUAL) {
            float u = (float)acc[i][j + NC][v];
            if (AK == AK_I8) u = u * rs;
            u = u * cs[j + NC];
            if constexpr (EPI == EPI_SWIGLU_F32) reinterpret_cast<float*>(g.c)[o] = (x / (1.0f + expf(-x))) * u;
            else if constexpr (EPI == EPI_SWIGLU_F16) reinterpret_cast<uint16_t*>(g.c)[o] = f32_to_f16_bits(silu(x) * u);
            else {  // EPI_SWIGLU_HALF: silu(clamp(g/16, +-20)) * u/16
              const float gg = fminf(fmaxf(x * 0.0625f, -20.0f), 20.0f);
              reinterpret_cast<uint16_t*>(g.c)[o] = f32_to_f16_bits((gg / (1.0f + expf(-gg))) * (u * 0.0625f));
            }
          } else if constexpr (EPI == EPI_STORE_F32) {
            reinterpret_cast<float*>(g.c)[o] = x;
          } else {
            reinterpret_cast<uint16_t*>(g.c)[o] = f32_to_f16_bits(x);
          }
        }
      }
    }
  }
}

template <int AK, int BK, int EPI, int T>
hipError_t launch_one(const QGemmArgs& g0, hipStream_t st) {
  QGemmArgs g = g0;
  g.tiles_m = (g.m + T - 1) / T;
  const int per = is_gate_up(EPI) ? T / 2 : T, n_tiles = (g.n + per - 1) / per;
  hipLaunchKernelGGL((k_tile<AK, BK, EPI, T>), dim3(g.tiles_m * n_tiles), dim3(2 * T), 0, st, g, n_tiles);
  return hipGetLastError();
}

template <int BK, int T>
hipError_t launch_epi(int epi, const QGemmArgs& g, hipStream_t st) {
  switch (epi) {
    case EPI_STORE_F32: return launch_one<AK_F16, BK, EPI_STORE_F32, T>(g, st);
    case EPI_STORE_F16: return launch_one<AK_F16, BK, EPI_STORE_F16, T>(g, st);
    case EPI_SWIGLU_F16: return launch_one<AK_F16, BK, EPI_SWIGLU_F16, T>(g, st);
    case EPI_SWIGLU_HALF: return launch_one<AK_F16, BK, EPI_SWIGLU_HALF, T>(g, st);
    default: return hipErrorInvalidValue;
  }
}

template <int BK>
hipError_t launch_f16a(int side, int epi, const QGemmArgs& g, hipStream_t st) {
  return side == 256 ? launch_epi<BK, 256>(epi, g, st) : launch_epi<BK, 128>(epi, g, st);
}

}  // namespace tile
}  // namespace mx
