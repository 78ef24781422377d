#pragma once
// mx_gemm_stream.h - weight-streaming GEMM for few activation rows and for
// sizes off the 64-wide tile grid.
//
//   C[m][n] = sum_k A[m][k] * W[n][k]   (epilogue: store, SwiGLU, row scales)
//
// The same products as mx_gemm_q.hip (MXFP4Kernels.metal:138-173, 264-286;
// MPPMLPKernels.metal:14-125), for any n and any k % 32 == 0.
//
// Bound: HBM while the weights are read once; from about 24 rows on the
// activations' way from L2, which every workgroup reads whole.
//
//   workgroup = 16 NG weight rows (SwiGLU: 8 NG gate and the same 8 NG up
//               channels, 8 + 8 in each group of 16) x one tile of at most 32
//               activation rows x all of K.  Its 4 waves split K, each with a
//               contiguous run of 128-K steps, so an activation element is
//               used by one wave only and no wave waits for another before
//               the final sum.  At most 80 KB of LDS: two or more workgroups
//               per CU, one's start and end under the others' stream.
//   weights   = global -> registers, one whole 128-byte line of 8 rows per
//               load, the halves swapped between lanes by DPP.  Half lines of
//               16 rows (no swap) measured 20.5 -> 26 us on 62 MB of weights.
//   A         = global -> LDS by buffer DMA into the wave's own part of a ring,
//               whole rows of a step per instruction (a 64-lane load of 16
//               rows x 64 B costs the CU's memory path twice the cycles of one
//               of whole 128-byte lines), chunks XOR-swizzled by row so that a
//               fragment read (16 rows x one chunk) hits distinct banks.  Rows
//               past the tile's end read as zero (the resource's range).
//   K order   = the MFMA sums over k in any order that both operands share.
//               A lane keeps its 16 bytes together: 4-bit lane group lg holds
//               block lg of the step (one scale), 8-bit bytes [64 h + 16 lg,
//               +16) for h = 0, 1, f16 chunk 4 q + lg.
//   scales    = the E8M0 / f16 scales of the workgroup's rows are copied to
//               LDS first.  E8M0 byte 255 (+inf to the reference, NaN to the
//               converter) is noted while streaming; a wave that met one runs
//               its K range again with the exact decode.
//   sum       = the 4 waves' partial tiles are added in LDS in wave order.
//
// Measured (us a launch, weights from HBM; before: the 128-row tiles, or the
// K-step-32 kernel where a size is off their grid): 62 MB gate/up pass at 8
// rows 22.0 -> 17.7 (3.5 TB/s), 15.6 MB at 16 rows 18.7 -> 9.2, 117 MB of FP8
// weights at 1 row 37.1 -> 25.7 (4.6 TB/s), one 4096 x 4096 MXFP4 matrix at 1
// row 13.4 -> 4.9, 2080 x 5536 at 1 row 108 -> 5.9, 64 experts of 7168 x 2048
// with 256 uneven tokens 712 -> 281 (5.0 TB/s, both passes).
#include <type_traits>

#include "mx_device.h"
#include "mx_dma.h"
#include "mx_internal.h"
#include "mx_stream.h"
#include "mx_widen.h"

namespace mx {
namespace stream {

constexpr int kStep = 128;   // K per step
constexpr int kNW = 4;       // waves of a workgroup, splitting K

constexpr int a_elem(int ak) { return ak == AK_I8 ? 1 : ak == AK_F32 ? 4 : 2; }
constexpr int b_bits(int bk) { return bk == BK_F16 ? 16 : (bk == BK_MXFP4 || bk == BK_INT4G32) ? 4 : 8; }
// Ring slots of a launch for tiles of `rows` activation rows.
constexpr int slots(int rows) { return rows <= 8 ? 3 : 2; }
constexpr int wait_vm(int n) { return ((n > 63 ? 63 : n) & 15) | (((n > 63 ? 63 : n) >> 4) << 14) | (7 << 4) | (15 << 8); }

constexpr int lcm(int a, int b) {
  int l = a;
  while (l % b) l += a;
  return l;
}

// Loads that may still be in flight when step i (phase = i % ps) is used.
// The order of issue is: iteration j issues A of step j + d (xi loads), waits,
// then, where j % ps == 0, weights j / ps + dw (wl loads).  Step i needs its A,
// issued in iteration i - d, and (phase 0) its weights, issued in i - dw ps.
constexpr int wait_count(int xi, int wl, int d, int dw, int ps, int phase) {
  const int i = 1000 * ps + phase;  // any iteration of this phase, far from the start
  auto after = [&](int j, bool w) {  // loads issued after iteration j's A (or weights), up to i's A
    int n = 0;
    for (int t = j; t <= i; t++) {
      if (t > j) n += xi;
      if (t % ps == 0 && t < i && (t > j || !w)) n += wl;
    }
    return n;
  };
  const int a = after(i - d, false);
  if (phase) return a;
  const int b = after(i - dw * ps, true);
  return a < b ? a : b;
}

__device__ __forceinline__ void dma16(const void* src, void* lds) { __builtin_amdgcn_global_load_lds(src, lds, 16, 0, 0); }

template <int I, int N, typename F>
__device__ __forceinline__ void unroll(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unroll<I + 1, N>(f);
  }
}

// As unroll, ended by the first f that returns false; false then.
template <int I, int N, typename F>
__device__ __forceinline__ bool unroll_while(F&& f) {
  if constexpr (I < N) {
    if (!f(std::integral_constant<int, I>{})) return false;
    return unroll_while<I + 1, N>(f);
  } else {
    return true;
  }
}

// Ring pieces in LDS: 16 activation rows of one step for every wave (all of a
// tile's rows below 16).  Separate arrays, so that the compiler's waits tell a
// DMA into one from the fragment reads of another.  The first also takes the
// final sums, 4 KB a wave.
struct Lds {
  uint8_t *p0, *p1, *p2, *p3, *sc;
};

// One tile of ROWS activation rows, in a launch whose LDS is sized for tiles
// of MAXR rows.
template <int AK, int BK, int NG, int ROWS, int MAXR>
__device__ __forceinline__ void tile(const Args& g, int m0, int nt, const Lds& lds) {
  constexpr int RB = kStep * a_elem(AK), RPI = 1024 / RB, CH = RB / 16;  // A row bytes, rows per DMA, chunks
  constexpr int XI = ROWS / RPI, MT = (ROWS + 15) / 16;                  // DMAs per step, row tiles of 16
  constexpr int PR = MAXR < 16 ? MAXR : 16, PB_ = PR * RB;                // rows and bytes of a wave's piece
  constexpr int XP = XI < 16 / RPI ? XI : 16 / RPI;                      // DMAs per piece
  constexpr int PIECES = slots(MAXR) * ((MAXR + 15) / 16);
  constexpr int NS = PIECES / MT, D = NS - 1;
  constexpr int NB = b_bits(BK) * kStep / 8 / 64;   // 16-byte pieces of a lane's weights per step
  constexpr bool S4 = BK == BK_MXFP4 || BK == BK_INT4G32;
  constexpr int ESZ = BK == BK_INT4G32 ? 2 : 1;
  constexpr int PS = b_bits(BK) == 4 ? 2 : 1;       // steps per 128-byte line of a weight row
  constexpr int WL = b_bits(BK) == 16 ? 4 : 2;      // weight loads per group and issue
  constexpr int DW = (D + PS) / PS;                 // issues in flight
  constexpr int UN = lcm(lcm(NS, PS * DW), PS);
  constexpr int PG = NG < 4 / MT ? NG : 4 / MT;     // groups a pass of the final sums
  static_assert(ROWS % RPI == 0 && ROWS <= MAXR && PIECES <= 4 && NS >= 1 && NG % PG == 0, "tile shape");
  using Acc = typename std::conditional<AK == AK_I8, v4i, v4f>::type;

  const int T = min(ROWS, g.m - m0);
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = g.k, N = g.n, KB = K / 32;
  const bool dual = is_gate_up(g.epi);
  const int PB = dual ? 8 : 16;                     // output channels per group
  const int n0 = nt * NG * PB;
  const int row_b = K / 8 * b_bits(BK);             // bytes of a weight row

  // first weight row of 8-row block b (two per group) and its matrix
  auto block_row = [&](int b) { return dual ? n0 + (b >> 1) * 8 : n0 + b * 8; };
  auto second = [&](int b) { return dual && (b & 1); };

  // ---- 1) the scales, requested before any load that the loop waits for:
  // by 16-byte DMA, or (odd K / 32, planes at a 4-byte boundary) by 8-byte
  // pieces through registers that are written to LDS once the first operands
  // are on their way (257 tokens, 2080 -> 2 x 5536: written at once, 3 us more)
  constexpr int SP = kScales / 8 / (64 * kNW);
  uint2 sreg[S4 ? SP : 1];
  const int bb = 8 * KB * ESZ;                      // bytes of a block's scales
  const int n_sp = 2 * NG * (bb / 8);               // 8-byte pieces
  int s_path = 0;                                   // workgroup-uniform
  if constexpr (S4) {
    const bool whole = (dual ? n0 + NG * 8 : n0 + NG * 16) <= N;
    const uintptr_t al = reinterpret_cast<uintptr_t>(g.s0) | (dual ? reinterpret_cast<uintptr_t>(g.s1) : 0);
    auto src = [&](int b) { return (second(b) ? g.s1 : g.s0) + (size_t)block_row(b) * KB * ESZ; };
    s_path = !whole || al % 4 ? 2 : bb % 16 || al % 16 ? 1 : 0;
    if (s_path == 0) {
      const int q = bb / 16, np = 2 * NG * q;
      for (int j0 = wave * 64; j0 < np; j0 += 64 * kNW) {
        const int j = j0 + lane;
        if (j < np) dma16(src(j / q) + (j % q) * 16, lds.sc + (size_t)j0 * 16);
      }
    } else if (s_path == 1) {
#pragma unroll
      for (int p = 0; p < SP; p++) {
        if (p * 64 * kNW >= n_sp) break;
        const int j = min(p * 64 * kNW + tid, n_sp - 1), q = bb / 8;
        sreg[p] = *reinterpret_cast<const uint2*>(src(j / q) + (j % q) * 8);
      }
    } else {                                        // rows past the end repeat the last one
      const int rb = KB * ESZ;
#pragma clang loop vectorize(disable) unroll_count(4)
      for (int j = tid; j < 16 * NG * rb; j += 64 * kNW) {
        const int row = j / rb, b = row >> 3;
        const int wr = min(block_row(b) + (row & 7), N - 1);
        lds.sc[j] = ((second(b) ? g.s1 : g.s0) + (size_t)wr * rb)[j % rb];
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  // ---- 2) operand addresses.  A whole line of 8 weight rows per load: load
  // A covers rows 0-7 of a group, load B rows 8-15; lane (r, lg) takes chunk
  // lg of its own row from the load that holds the row and chunk 4 + lg of
  // row r ^ 8 from the other, so the first half line is a select of A / B and
  // the second the other select rotated by 8 lanes.
  const uint8_t *wa[NG], *wb[NG];
#pragma unroll
  for (int i = 0; i < NG; i++) {
    wa[i] = (second(2 * i) ? g.b1 : g.b0) + (size_t)min(block_row(2 * i) + (r & 7), N - 1) * row_b;
    wb[i] = (second(2 * i + 1) ? g.b1 : g.b0) + (size_t)min(block_row(2 * i + 1) + (r & 7), N - 1) * row_b;
  }
  const int ca = lg * 16 + (r >= 8 ? 64 : 0), cb = lg * 16 + (r < 8 ? 64 : 0);
  constexpr int SW = CH < 16 ? CH - 1 : 15;  // chunk swizzle of a row
  const int a_row = K * a_elem(AK);
  const uint8_t* ab = reinterpret_cast<const uint8_t*>(g.a) + (size_t)m0 * a_row;
  const v4i ars = rsrc_of<false>(ab, (uint32_t)T * (uint32_t)a_row);
  int a_off[XI];
#pragma unroll
  for (int i = 0; i < XI; i++) {
    const int row = i * RPI + lane / CH;
    a_off[i] = row * a_row + (((lane % CH) ^ (row & SW)) << 4);
  }
  // The wave's steps: a contiguous run of line columns (PS steps each).
  const int L = (K + kStep * PS - 1) / (kStep * PS);
  const int c0 = L * wave / kNW, n_c = L * (wave + 1) / kNW - c0;
  const int st0 = c0 * PS, n_st = min(n_c * PS, (K + kStep - 1) / kStep - st0);

  auto piece = [&](auto u) -> uint8_t* {
    constexpr int U = decltype(u)::value;
    if constexpr (U == 0) return lds.p0 + wave * (PB_ > 4096 ? PB_ : 4096);
    else if constexpr (U == 1) return lds.p1 + wave * PB_;
    else if constexpr (U == 2) return lds.p2 + wave * PB_;
    else return lds.p3 + wave * PB_;
  };
  // A of step i into slot u.  Past the wave's last step (never used; the
  // wait counts stay constant) the offset is out of the resource's range,
  // which fetches nothing.
  auto issue_a = [&](int i, auto u) {
    const int o = i < n_st ? (st0 + i) * RB : 0x40000000;
    unroll<0, XI>([&](auto qq) {
      constexpr int q = decltype(qq)::value, U = decltype(u)::value;
      uint8_t* dst = piece(std::integral_constant<int, U * MT + q / XP>{}) + (q % XP) * 1024;
      buffer_dma16(ars, dst, a_off[q] + o);
    });
    __builtin_amdgcn_sched_barrier(0);
  };
  // Weights of line column (4-bit) or step i into register set u; past the
  // end the last one again.
  v4i wv[DW][NG][WL];
  auto issue_w = [&](int i, auto u) {
    constexpr int U = decltype(u)::value;
    const int c = (c0 + max(min(i, n_c - 1), 0)) * (WL / 2);
#pragma unroll
    for (int h = 0; h < WL / 2; h++) {
      const int oa = min((c + h) * 128 + ca, row_b - 16), ob = min((c + h) * 128 + cb, row_b - 16);
#pragma unroll
      for (int gi = 0; gi < NG; gi++) {
        const v4i va = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(wa[gi] + oa));
        const v4i vb = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(wb[gi] + ob));
        wv[U][gi][2 * h] = va;
        wv[U][gi][2 * h + 1] = vb;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  Acc acc[NG][MT];
#pragma unroll
  for (int i = 0; i < NG; i++)
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
      for (int v = 0; v < 4; v++) acc[i][t][v] = 0;

  // A chunk of MFMA q (of NQ) for this lane
  constexpr int NQ = AK == AK_I8 ? 2 : 4;
  constexpr int AW = AK == AK_F32 ? 2 : 1;  // chunks per operand
  auto a_chunk = [&](int q) {
    return AW * (AK == AK_I8 ? q * 4 + lg : b_bits(BK) == 4 ? lg * 4 + q : b_bits(BK) == 8 ? (q >> 1) * 8 + lg * 2 + (q & 1) : q * 4 + lg);
  };
  // 8 weights of MFMA q from the step's half lines, and their group scale
  auto widen = [&](const v4i* w, int q, uint32_t s) -> v8h {
    if constexpr (BK == BK_MXFP4) {
      return fp4x8_to_f16x8((uint32_t)w[0][q], e8m0_as_cvt_scale(s));
    } else if constexpr (BK == BK_INT4G32) {
      return i4x8_to_f16((uint32_t)w[0][q], __builtin_bit_cast(_Float16, (uint16_t)s));
    } else if constexpr (BK == BK_F16) {
      return __builtin_bit_cast(v8h, w[NB == 4 ? q : 0]);
    } else {
      const uint32_t lo = (uint32_t)w[NB == 2 ? q >> 1 : 0][2 * (q & 1)], hi = (uint32_t)w[NB == 2 ? q >> 1 : 0][2 * (q & 1) + 1];
      if constexpr (BK == BK_INT8) return i8x8_to_f16(lo, hi);
      else return fp8x8_to_f16<BK>(lo, hi);
    }
  };
  // scale of (group row, 32-K block)
  auto scale_at = [&](int gi, int blk) -> uint32_t {
    if constexpr (!S4) return 0u;
    else if constexpr (ESZ == 2) return reinterpret_cast<const uint16_t*>(lds.sc)[(gi * 16 + r) * KB + blk];
    else return lds.sc[(gi * 16 + r) * KB + blk];
  };

  // The prologue issues in the loop's order (the wait counts rely on it).
  constexpr int J = D > DW * PS ? D : DW * PS;
  unroll<0, J>([&](auto jj) {
    constexpr int j = decltype(jj)::value - J;  // iteration, negative
    if constexpr (j + D >= 0) issue_a(j + D, std::integral_constant<int, j + D >= 0 ? (j + D) % NS : 0>{});
    if constexpr (j % PS == 0 && j / PS + DW >= 0) issue_w(j / PS + DW, std::integral_constant<int, j / PS + DW >= 0 ? (j / PS + DW) % DW : 0>{});
  });
  if constexpr (S4) {
    // the scales (older than those loads) have landed everywhere
    __builtin_amdgcn_s_waitcnt(wait_vm(D * XI + DW * WL * NG));
    if (s_path == 1) {
#pragma unroll
      for (int p = 0; p < SP; p++) {
        if (p * 64 * kNW >= n_sp) break;
        if (p * 64 * kNW + tid < n_sp) reinterpret_cast<uint2*>(lds.sc)[p * 64 * kNW + tid] = sreg[p];
      }
    }
    __builtin_amdgcn_s_waitcnt(wait_vm(63) & ~(15 << 8));  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  }
  uint32_t bad = 0;    // an E8M0 byte 255 among the lane's blocks
  v4i w2[NG][NB * PS];  // the half lines of the line column (4-bit) or step in use
  for (int i0 = 0;; i0 += UN) {
    const bool more = unroll_while<0, UN>([&](auto uu) -> bool {
      constexpr int U = decltype(uu)::value;
      const int i = i0 + U, st = st0 + i;
      if (i >= n_st) return false;
      issue_a(i + D, std::integral_constant<int, (U + D) % NS>{});
      __builtin_amdgcn_s_waitcnt(wait_vm(wait_count(XI, WL * NG, D, DW, PS, U % PS)));
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (U % PS == 0) {
        constexpr int V = U / PS % DW;
#pragma unroll
        for (int gi = 0; gi < NG; gi++)
#pragma unroll
          for (int h = 0; h < WL / 2; h++) {
            // element by element: a select of whole vectors went through memory
#pragma unroll
            for (int e = 0; e < 4; e++) {
              const int a = wv[V][gi][2 * h][e], b = wv[V][gi][2 * h + 1][e];
              w2[gi][2 * h][e] = r < 8 ? a : b;
              w2[gi][2 * h + 1][e] = __builtin_amdgcn_mov_dpp(r < 8 ? b : a, 0x128, 0xf, 0xf, false);
            }
          }
        issue_w(i / PS + DW, std::integral_constant<int, V>{});
      }
      v4i af[NQ][MT][AW];
      unroll<0, MT>([&](auto tt) {
        constexpr int t = decltype(tt)::value;
        const uint8_t* as = piece(std::integral_constant<int, (U % NS) * MT + t>{}) + (ROWS < 16 ? r & (ROWS - 1) : r) * RB;
#pragma unroll
        for (int q = 0; q < NQ; q++)
#pragma unroll
          for (int c = 0; c < AW; c++)
            af[q][t][c] = *reinterpret_cast<const v4i*>(as + (((a_chunk(q) + c) ^ ((ROWS < 16 ? r & (ROWS - 1) : r) & SW)) << 4));
      });
      uint32_t s[NG];
#pragma unroll
      for (int gi = 0; gi < NG; gi++) s[gi] = scale_at(gi, min(st * 4 + lg, KB - 1));
      v4i w[NG][NB];
#pragma unroll
      for (int gi = 0; gi < NG; gi++)
#pragma unroll
        for (int h = 0; h < NB; h++) w[gi][h] = w2[gi][PS == 2 ? U % PS : h];
      if ((st + 1) * kStep > K) {  // a last step of less than 128 K: zero what is past the end
        // (the scales too: an infinite one of the row's last block makes a zero code NaN)
#pragma unroll
        for (int gi = 0; gi < NG; gi++) s[gi] = st * 4 + lg < KB ? s[gi] : 0u;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
          const bool in = st * RB + a_chunk(q) * 16 < a_row;
#pragma unroll
          for (int t = 0; t < MT; t++)
#pragma unroll
            for (int c = 0; c < AW; c++) {
              if (!in) af[q][t][c] = (v4i){0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int h = 0; h < NB; h++) {
          const bool in = st * (64 * NB) + h * 64 + lg * 16 < row_b;
#pragma unroll
          for (int gi = 0; gi < NG; gi++) {
            if (!in) w[gi][h] = (v4i){0, 0, 0, 0};
          }
        }
      }
      v8h ah[NQ][MT], al[NQ][MT];  // f16 operands (f32 activations: x = hi + lo)
      if constexpr (AK != AK_I8) {
#pragma unroll
        for (int q = 0; q < NQ; q++)
#pragma unroll
          for (int t = 0; t < MT; t++) {
            if constexpr (AK == AK_F16) ah[q][t] = __builtin_bit_cast(v8h, af[q][t][0]);
            else split_f32(__builtin_bit_cast(v4f, af[q][t][0]), __builtin_bit_cast(v4f, af[q][t][AW - 1]), ah[q][t], al[q][t]);
          }
      }
#pragma unroll
      for (int gi = 0; gi < NG; gi++) {
        if (BK == BK_MXFP4) bad |= s[gi] == 255u;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
          if constexpr (AK == AK_I8) {
            const v4i b = w[gi][q];
#pragma unroll
            for (int t = 0; t < MT; t++) acc[gi][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[q][t][0], b, acc[gi][t], 0, 0, 0);
          } else {
            const v8h b = widen(w[gi], q, s[gi]);
#pragma unroll
            for (int t = 0; t < MT; t++) {
              acc[gi][t] = mfma_f16_16x16x32(ah[q][t], b, acc[gi][t]);
              if constexpr (AK == AK_F32) acc[gi][t] = mfma_f16_16x16x32(al[q][t], b, acc[gi][t]);
            }
          }
        }
      }
      return true;
    });
    if (!more) break;
  }

  if constexpr (BK == BK_MXFP4) {
    // E8M0 byte 255 in this wave's blocks: its K range again, decoded as the
    // reference does (rare; straight from global memory)
    if (__builtin_expect(__ballot(bad != 0) != 0, 0)) {
#pragma unroll
      for (int i = 0; i < NG; i++)
#pragma unroll
        for (int t = 0; t < MT; t++) acc[i][t] = (Acc){0, 0, 0, 0};
#pragma nounroll
      for (int i = 0; i < n_st; i++) {
        const int blk = (st0 + i) * 4 + lg;
        const bool in = blk < KB;
        const int bc = min(blk, KB - 1);
#pragma unroll
        for (int gi = 0; gi < NG; gi++) {
          const int row = min(block_row(2 * gi + (r >> 3)) + (r & 7), N - 1);
          const uint8_t* wp = (second(2 * gi + (r >> 3)) ? g.b1 : g.b0) + (size_t)row * row_b;
          const uint4 w = *reinterpret_cast<const uint4*>(wp + (size_t)bc * 16);
          const uint32_t d[4] = {in ? w.x : 0u, in ? w.y : 0u, in ? w.z : 0u, in ? w.w : 0u};
          const uint32_t sb = in ? scale_at(gi, bc) : 127u;
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const v8h b = fp4x8_dequant_f16(d[q], sb);
#pragma unroll
            for (int t = 0; t < MT; t++) {
              const uint8_t* xp = ab + (size_t)min(t * 16 + r, T - 1) * a_row + ((size_t)bc * 32 + q * 8) * a_elem(AK);
              v4i x0 = *reinterpret_cast<const v4i*>(xp), x1 = *reinterpret_cast<const v4i*>(xp + (AW - 1) * 16);
              if (!in) x0 = x1 = (v4i){0, 0, 0, 0};
              if constexpr (AK == AK_F16) {
                acc[gi][t] = mfma_f16_16x16x32(__builtin_bit_cast(v8h, x0), b, acc[gi][t]);
              } else {
                v8h hi, lo;
                split_f32(__builtin_bit_cast(v4f, x0), __builtin_bit_cast(v4f, x1), hi, lo);
                acc[gi][t] = mfma_f16_16x16x32(hi, b, acc[gi][t]);
                acc[gi][t] = mfma_f16_16x16x32(lo, b, acc[gi][t]);
              }
            }
          }
        }
      }
    }
  }

  // ---- 3) sum over the waves and epilogue, PG groups a pass.  A wave's
  // partial of (group, row tile) is 1 KB, [column][4 chunks of 4 rows], the
  // chunks XORed by column / 4 so that the column reads spread over the banks.
  __builtin_amdgcn_s_waitcnt(wait_vm(0) & ~(15 << 8));  // no DMA of past-the-end steps may land on the sums
  const int cw = PG * PB;  // channels a pass
#pragma unroll
  for (int p = 0; p < NG; p += PG) {
    if (p) __syncthreads();
    uint8_t* own = lds.p0 + wave * (PB_ > 4096 ? PB_ : 4096);
#pragma unroll
    for (int gi = 0; gi < PG; gi++)
#pragma unroll
      for (int t = 0; t < MT; t++)
        *reinterpret_cast<v4i*>(own + (gi * MT + t) * 1024 + r * 64 + ((lg ^ (r >> 2)) << 4)) =
            __builtin_bit_cast(v4i, acc[p + gi][t]);
    __syncthreads();
    auto sum = [&](int gi, int tok, int col) -> float {
      const int o = (gi * MT + (tok >> 4)) * 1024 + col * 64 + ((((tok >> 2) & 3) ^ (col >> 2)) << 4) + (tok & 3) * 4;
      if constexpr (AK == AK_I8) {
        int v = 0;
#pragma unroll
        for (int w = 0; w < kNW; w++) v += *reinterpret_cast<const int*>(lds.p0 + w * (PB_ > 4096 ? PB_ : 4096) + o);
        return g.epi == EPI_STORE_I32 ? __builtin_bit_cast(float, v) : (float)v * g.a_scale[m0 + tok];
      } else {
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < kNW; w++) v += *reinterpret_cast<const float*>(lds.p0 + w * (PB_ > 4096 ? PB_ : 4096) + o);
        return v;
      }
    };
    for (int j = tid; j < T * cw; j += 64 * kNW) {
      const int tok = j / cw, ch = j % cw, n = n0 + p * PB + ch;
      if (n >= N) continue;
      const size_t o = (size_t)(m0 + tok) * N + n;
      float v = sum(ch / PB, tok, ch % PB);
      if constexpr (!S4 && BK != BK_F16) {
        if (g.epi != EPI_STORE_I32) v *= reinterpret_cast<const float*>(g.s0)[n];
      }
      if (dual) {
        float u = sum(ch / PB, tok, ch % PB + 8);
        if constexpr (!S4 && BK != BK_F16) u *= reinterpret_cast<const float*>(g.s1)[n];
        if (g.epi == EPI_SWIGLU_F16) {
          reinterpret_cast<uint16_t*>(g.c)[o] = f32_to_f16_bits(silu(v) * u);
        } else if (g.epi == EPI_SWIGLU_F32) {
          reinterpret_cast<float*>(g.c)[o] = (v / (1.0f + expf(-v))) * u;
        } else {  // swiglu_half (MPPMLPKernels.metal:204-220)
          const float gg = fminf(fmaxf(v * 0.0625f, -20.0f), 20.0f);
          reinterpret_cast<uint16_t*>(g.c)[o] = f32_to_f16_bits((gg / (1.0f + expf(-gg))) * (u * 0.0625f));
        }
      } else if (g.epi == EPI_STORE_F16) {
        reinterpret_cast<uint16_t*>(g.c)[o] = f32_to_f16_bits(v);
      } else {
        reinterpret_cast<float*>(g.c)[o] = v;  // f32, or the bits of an i32
      }
    }
  }
}

template <int AK, int BK, int NG, int MAXR, bool GROUPED>
__global__ __launch_bounds__(64 * kNW) void k_stream(Args g, typename std::conditional<GROUPED, GroupTable, int>::type gt) {
  constexpr int PB = (MAXR < 16 ? MAXR : 16) * kStep * a_elem(AK) * kNW;  // bytes of a piece
  constexpr int PIECES = slots(MAXR) * ((MAXR + 15) / 16);
  __shared__ __attribute__((aligned(16))) uint8_t p0[PB > 4096 * kNW ? PB : 4096 * kNW];
  __shared__ __attribute__((aligned(16))) uint8_t p1[PIECES > 1 ? PB : 16];
  __shared__ __attribute__((aligned(16))) uint8_t p2[PIECES > 2 ? PB : 16];
  __shared__ __attribute__((aligned(16))) uint8_t p3[PIECES > 3 ? PB : 16];
  __shared__ __attribute__((aligned(16))) uint8_t sc[BK == BK_MXFP4 || BK == BK_INT4G32 ? kScales : 16];
  const Lds lds{p0, p1, p2, p3, sc};
  // Workgroup ids 8 apart share an XCD.  One matrix: the row tiles of a weight
  // tile run there one after another and meet its weights in L2.  Groups: row
  // tiles outermost, since most groups lack the later ones, and workgroups
  // that exit at once in a regular pattern leave whole shader engines idle (64
  // experts x 4 tokens, largest 25, tiles of 8 rows: 804 us interleaved).
  const int bid = blockIdx.x, ix = bid >> 3, nt8 = (g.n_tiles + 7) & ~7;
  const int m0 = (GROUPED ? bid / nt8 : ix % g.m_tiles) * MAXR;
  const int nt = GROUPED ? bid % nt8 : ix / g.m_tiles * 8 + (bid & 7);
  if (nt >= g.n_tiles) return;
  if constexpr (GROUPED) {
    const int e = blockIdx.y, t0 = gt.off[e];
    g.m = gt.off[e + 1] - t0;
    g.a = reinterpret_cast<const uint8_t*>(g.a) + (size_t)t0 * g.k * a_elem(AK);
    g.c = reinterpret_cast<uint8_t*>(g.c) + (size_t)t0 * g.n * 2;
    g.b0 += e * gt.b_stride;
    g.s0 += e * gt.s_stride;
    if (is_gate_up(g.epi)) {
      g.b1 += e * gt.b_stride;
      g.s1 += e * gt.s_stride;
    }
    const int t = g.m - m0;
    if (t <= 0) return;  // workgroup-uniform, before any barrier
    // a group's own rows choose the tile body
    if constexpr (MAXR > 8) {
      if (t <= 8) return tile<AK, BK, NG, 8, MAXR>(g, m0, nt, lds);
    }
    if constexpr (MAXR > 16) {
      if (t <= 16) return tile<AK, BK, NG, 16, MAXR>(g, m0, nt, lds);
    }
  }
  tile<AK, BK, NG, MAXR, MAXR>(g, m0, nt, lds);
}

template <int AK, int BK, int NG, int MAXR, bool GROUPED>
hipError_t launch_ng(const Args& g0, const GroupTable* gt, int groups, hipStream_t st) {
  Args g = g0;
  const int pb = (is_gate_up(g.epi) ? 8 : 16) * NG;
  g.m_tiles = (g.m + MAXR - 1) / MAXR;
  g.n_tiles = (g.n + pb - 1) / pb;
  const dim3 grid((unsigned)((g.n_tiles + 7) / 8 * 8 * g.m_tiles), groups);
  if constexpr (GROUPED) hipLaunchKernelGGL((k_stream<AK, BK, NG, MAXR, true>), grid, dim3(64 * kNW), 0, st, g, *gt);
  else hipLaunchKernelGGL((k_stream<AK, BK, NG, MAXR, false>), grid, dim3(64 * kNW), 0, st, g, 0);
  return hipGetLastError();
}

template <int AK, int BK, int MAXR, bool GROUPED>
hipError_t launch_rows(const Args& g, const GroupTable* gt, int groups, int ng, hipStream_t st) {
  switch (ng) {
    case 1: return launch_ng<AK, BK, 1, MAXR, GROUPED>(g, gt, groups, st);
    case 2: return launch_ng<AK, BK, 2, MAXR, GROUPED>(g, gt, groups, st);
    case 4:  // f16 weights: too many registers for two waves per SIMD
      if constexpr (BK != BK_F16) return launch_ng<AK, BK, 4, MAXR, GROUPED>(g, gt, groups, st);
  }
  return hipErrorInvalidValue;
}

// One weight format: tile rows and groups as launch_stream chose them.
template <int AK, int BK, bool GROUPED>
hipError_t launch_bk(const Args& g, const GroupTable* gt, int groups, int rows, int ng, hipStream_t st) {
  switch (rows) {
    case 4:
      if constexpr (AK != AK_I8) return launch_rows<AK, BK, 4, GROUPED>(g, gt, groups, ng, st);
      else break;
    case 8: return launch_rows<AK, BK, 8, GROUPED>(g, gt, groups, ng, st);
    case 16: return launch_rows<AK, BK, 16, GROUPED>(g, gt, groups, ng, st);
    case 32:
      if constexpr (AK != AK_F32) return launch_rows<AK, BK, 32, GROUPED>(g, gt, groups, ng, st);
      else break;
  }
  return hipErrorInvalidValue;
}

}  // namespace stream
}  // namespace mx
