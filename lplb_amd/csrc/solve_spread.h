// LP solver, one LP per wave, groups of up to 32 ranks: the group's G x G system spread over all 64
// lanes.  Same problem, method and arithmetic as solve_kernel.h (read that first); what differs is who
// holds what.
//
// A lone wave issues one instruction every 2.3 ns (3.5 ns if it needs the one before), whatever the
// instruction does for how many lanes, so the time of an LP is the number of instructions on its path
// and the round trips through LDS in it.
// With one lane per rank and one lane per edge (solve_kernel.h) 48 or 56 of the 64 lanes idle, every
// lane carries a whole row of S through assembly and elimination, and what goes from edges to ranks and
// back goes through ten ds_bpermute per step.  Here
//   * wave lane l belongs to rank l / TS (TS = 64 / GM lanes per rank) and holds the columns
//     k * TS + l % TS, k < KC = GM / TS, of that rank's row of S: 1 column at 8 ranks, 4 at 16, 16 at 32;
//   * a rank's lanes also hold the rank's replica edges, both those it is the original of and those whose
//     copy it hosts ("edge ends": end e = 2 d is the rank's own edge in slot d, e = 2 d + 1 the edge
//     copied into slot d; lane l holds ends l % TS + TS * p).  Every edge lives twice, at its two ends,
//     with the same values computed twice; a rank's sums over its edges are DPP adds inside its lanes,
//     and the only value that has to travel is the solution y of the other end's rank.
// Measured per affine-scaling step (in-kernel clock; one lane per rank and edge before): (8, 2) 1.15 -> 0.70 us,
// of which the elimination is 0.48 (a pivot is one round trip through LDS), assembly 0.15 and the rest 0.2;
// (16, 2) 1.8 -> 1.3 us; (32, 2) 3.1 -> 2.9 us, nearly all of it elimination.
// (A form in which rank i is lane i of every 16-lane row and holds its whole row, the elimination made of
// fp64 multiply-adds with a row_newbcast operand, has pivots of 40 instead of 60 ns and no LDS in them; but
// getting the rows into that shape costs 0.25 us a step more than it gains at 8 ranks.)
#pragma once
#include "solve_kernel.h"

namespace lplb {

// Which instantiations take this form (one LP per wave, one edge per lane in the other form).
constexpr bool spread_shape(int gm, int dm) { return gm <= 32 && gm * dm <= 128 && dm <= 8; }

// LDS per wave: the pivot columns in flight (two buffers) and, except at 8 ranks with at most two slots,
// the tile in which the rows of S are put together, followed by a copy of v.
constexpr int spread_row_doubles = 9;   // 8 ranks: rows of S, padded so that a column is in distinct banks
constexpr int spread_pivot_doubles(int gm) { return gm <= 8 ? 2 * 8 * spread_row_doubles : 2 * kWave; }
constexpr bool spread_uses_tile(int gm, int dm) { return gm > 8 || dm > 2; }
constexpr int spread_tile_floats(int gm, int dm) { return spread_uses_tile(gm, dm) ? gm * (gm + 4) + 2 * gm : 4; }

// v of the lane that CTRL names, for controls in which every lane has a source.
template <int CTRL> __device__ inline float dpp_all(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
constexpr int kRowRor8 = 0x128;
template <int LANE> __device__ inline float quad_bcast(float v) { return dpp_all<LANE * 0x55>(v); }

// Sums and maxima across the four 16-lane rows (complete in the last row) and, for maxima, inside them.
// Written out because the compiler splits a DPP operand with a row mask, or one of a maximum, into two to
// four instructions.  (A DPP operand must be two wait states old.)
#define LPLB_DPP(OP, CTRL, ROWS) "s_nop 1\n\t" OP "_dpp %0, %0, %0 " CTRL " row_mask:" ROWS " bank_mask:0xf\n\t"
#define LPLB_ROWS(OP) LPLB_DPP(OP, "row_bcast:15", "0xa") LPLB_DPP(OP, "row_bcast:31", "0xc")
__device__ inline float rows_sum(float v) {
  asm(LPLB_ROWS("v_add_f32") : "+v"(v));
  return readlane(v, kWave - 1);
}
template <bool Q1, bool Q2, bool H> __device__ inline float wave_max_of_groups(float v) {
  if (Q1) asm(LPLB_DPP("v_max_f32", "quad_perm:[1,0,3,2]", "0xf") : "+v"(v));
  if (Q2) asm(LPLB_DPP("v_max_f32", "quad_perm:[2,3,0,1]", "0xf") : "+v"(v));
  if (H) asm(LPLB_DPP("v_max_f32", "row_half_mirror", "0xf") : "+v"(v));
  asm(LPLB_DPP("v_max_f32", "row_ror:8", "0xf") LPLB_ROWS("v_max_f32") : "+v"(v));
  return readlane(v, kWave - 1);
}
#undef LPLB_ROWS
#undef LPLB_DPP

// Over the ranks: v is the same in the TS lanes of each rank; the result is wave-uniform.
template <int TS> __device__ inline float over_ranks_sum(float v) {
  if (TS <= 2) v += dpp_all<kQuadSwap2>(v);
  if (TS <= 4) v += dpp_all<kHalfMirror>(v);
  v += dpp_all<kRowRor8>(v);
  return rows_sum(v);
}
// Over a rank's edge ends (NE of them, E per lane); every lane of the rank gets the result.
template <int TS, int NE, int E> __device__ inline float over_ends_sum(const float (&v)[E]) {
  float t = v[0] + dpp_all<kQuadSwap1>(v[0]);
#pragma unroll
  for (int p = 1; p < E; ++p)
    t += v[p] + dpp_all<kQuadSwap1>(v[p]);
  if (NE > 2 && TS >= 4) t += dpp_all<kQuadSwap2>(t);
  if (NE > 4 && TS >= 8) t += dpp_all<kHalfMirror>(t);
  return t;
}
// Maximum over the wave (a NaN operand is ignored); lanes that only repeat other lanes' edge ends are skipped.
template <int TS, int NE> __device__ inline float over_all_max(float v) {
  return wave_max_of_groups<true, (TS <= 2 || NE > 2), (TS <= 4 || NE > 4)>(v);
}

// `old` with the lanes of rank RANK replaced by those of v, which is the same in all lanes of a 16-lane row:
// one instruction (DPP row_newbcast with row and bank masks; a bank is four lanes).  With two lanes per rank
// the other rank of the bank is overwritten as well.
template <int TS, int RANK> __device__ inline double set_rank(double old, double v) {
  constexpr int row = RANK * TS / 16, bank = RANK * TS % 16 / 4, banks = TS == 8 ? 3 << bank : 1 << bank;
  const long long o = __builtin_bit_cast(long long, old), w = __builtin_bit_cast(long long, v);
  const long long r = __builtin_amdgcn_update_dpp(o, w, 0x150, 1 << row, banks, false);
  return __builtin_bit_cast(double, r);
}

// 0.999 / d_max in fp64, rounded to fp32 by the caller: estimate, Newton step, one correction of the
// quotient (error below one fp64 ulp; the compiler's full division takes twice the instructions, all of
// them in the chain from one step to the next).  d_max = 0 or infinite gives NaN where the division gives
// infinity or 0: either way the step leaves the artificial variable without a number below the
// feasibility limit, so the LP is reported infeasible and its shares are the neutral ones.
__device__ inline double step_length(double d_max) {
  const double r = rcp_f64(d_max);
  const double q = 0.999 * r;
  return __builtin_fma(__builtin_fma(-d_max, q, 0.999), r, q);
}

// Arguments, LDS contracts and the returned value as for solve_lp; pivot_rows has spread_pivot_doubles(GM)
// doubles, tile spread_tile_floats(GM, DM) floats, both 16-byte aligned; rep_of_edge kWave ints, or twice
// that if GM * DM > kWave.
// counts_have_come: called once the wave's table loads have been issued if a.counts_by_caller; returns when the
// counts are in staged_counts (true), or when they will not come: then -1 is returned, nothing solved or stored.
template <int GM, int DM, bool EXACT, typename Counts>
__device__ inline int solve_lp_spread(const SolveArgs &a, int unit, float *staged_counts, int *rep_of_edge,
                                      double *pivot_rows, float *tile, Counts counts_have_come) {
  static_assert(spread_shape(GM, DM) && (GM == 8 || GM == 16 || GM == 32), "a lane holds GM * GM / 64 entries of S");
  constexpr int TS = kWave / GM, KC = GM / TS;
  constexpr int NE = 2 * DM, E = NE > TS ? NE / TS : 1;
  constexpr bool kTile = spread_uses_tile(GM, DM);
  constexpr int KB = 4;   // counts of experts that cannot move a lane prefetches
  constexpr int KG = 4;   // normalised counts a lane prefetches for the output (and loop unrolling)
  const int lane = threadIdx.x % kWave;
  const int rank = lane / TS, sub = lane % TS;
  const int G = EXACT ? GM : a.G, D = EXACT ? DM : a.D;
  const int C = a.C, n = G * D, n_fixed = a.n_fixed;
  const int L = D * C + n_fixed, P = L + D * C;
  const int grp = unit % a.n_group, inst = unit / a.n_group;
  const int32_t *__restrict__ wl = a.workload + (int64_t)inst * a.n_experts;
  const int32_t *__restrict__ p2l = a.phy2log + (int64_t)grp * G * P;
  const bool is_rank = EXACT || rank < G;
  const bool staged = a.staged_stride > 0 || a.counts_by_caller;
  auto count_of = [&](int e) -> float {
    if (e < 0 || e >= a.n_experts)
      return 0.0f;
    return staged ? staged_counts[e] : (float)wl[e];
  };
  // my edge ends
  const bool is_copy = sub & 1;
  int slot[E];
  bool on[E];
#pragma unroll
  for (int p = 0; p < E; ++p) {
    slot[p] = ((sub + TS * p) % NE) >> 1;
    on[p] = EXACT || (is_rank && slot[p] < D);
  }

  LPLB_STAMP(0);
  // ---- all global reads up front, as independent loads ----
  int e_first[E], orig_rank[E];
#pragma unroll
  for (int p = 0; p < E; ++p) {
    e_first[p] = (on[p] && C > 0) ? p2l[rank * P + slot[p]] : -1;
    const int k = on[p] ? a.r2o[rank * D + slot[p]] : 0;
    orig_rank[p] = k < 0 ? 0 : (k >= G ? G - 1 : k);
  }
  int fixed_e[KB];
#pragma unroll
  for (int u = 0; u < KB; ++u) {
    const int j = sub + u * TS;
    fixed_e[u] = (is_rank && j < n_fixed) ? p2l[rank * P + D * C + j] : -1;
  }
  float wmax = 0.0f;
  float out_cnt[KG];
  if (a.counts_by_caller) {
    if (!counts_have_come())
      return -1;
    for (int i = lane; i < a.n_experts; i += kWave)
      wmax = fmaxf(wmax, staged_counts[i]);
#pragma unroll
    for (int u = 0; u < KG; ++u) {
      const int i = lane + u * kWave;
      out_cnt[u] = (a.gw_out && i < G * L) ? staged_counts[grp * G * L + i] : 0.0f;
    }
  } else {
#pragma unroll KG
    for (int i = lane; i < a.n_experts; i += kWave) {
      const float cnt = (float)wl[i];
      wmax = fmaxf(wmax, cnt);
      if (staged)
        staged_counts[i] = cnt;
    }
#pragma unroll
    for (int u = 0; u < KG; ++u) {
      const int i = lane + u * kWave;
      out_cnt[u] = (a.gw_out && i < G * L) ? (float)wl[grp * G * L + i] : 0.0f;
    }
  }
  __builtin_amdgcn_wave_barrier();   // staged counts are visible to the whole wave
  float w_first[E], fixed_cnt[KB];
#pragma unroll
  for (int p = 0; p < E; ++p)
    w_first[p] = count_of(e_first[p]);
#pragma unroll
  for (int u = 0; u < KB; ++u)
    fixed_cnt[u] = count_of(fixed_e[u]);
  wmax = reduce_max<kWave>(wmax);

  LPLB_STAMP(1);
  // ---- weights and other ends of my edge ends (minilp.cu:203-221) ----
  float w[E];          // tokens of the edge's expert set over the largest count
  int edge[E], other[E];
#pragma unroll
  for (int p = 0; p < E; ++p) {
    float own = on[p] && C > 0 ? w_first[p] / wmax : 0.0f;
    if (on[p])
      for (int c = 1; c < C; ++c)
        own += count_of(p2l[rank * P + c * D + slot[p]]) / wmax;
    // a copied edge's weight is its original's, found at the even lane of that rank
    const float copied = bpermute(own, orig_rank[p] * TS + (sub & ~1));
    w[p] = on[p] ? (is_copy ? copied : own) : 0.0f;
    edge[p] = (is_copy ? orig_rank[p] : rank) * D + slot[p];
    if (on[p] && !is_copy)
      rep_of_edge[edge[p]] = rank;
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int p = 0; p < E; ++p)
    if (on[p] && is_copy)
      rep_of_edge[edge[p]] = rank;
  __builtin_amdgcn_wave_barrier();
  float w_lap[E];      // ... zero where the edge is no edge of the Laplacian (inactive, or a loop)
#pragma unroll
  for (int p = 0; p < E; ++p) {
    const int rep = on[p] && !is_copy ? rep_of_edge[edge[p]] : rank;
    other[p] = on[p] ? (is_copy ? orig_rank[p] : rep) : rank;
    w_lap[p] = other[p] == rank ? 0.0f : w[p];
  }

  LPLB_STAMP(2);
  // ---- per-rank constants, the same in all lanes of a rank ----
  // b = -(load of the experts that cannot move), minilp.cu:223-234
  float part = 0.0f;
#pragma unroll
  for (int u = 0; u < KB; ++u)
    part += fixed_cnt[u] / wmax;
  if (is_rank)
    for (int j0 = sub + KB * TS; j0 < n_fixed; j0 += KB * TS) {
      int more_e[KB];
#pragma unroll
      for (int u = 0; u < KB; ++u)
        more_e[u] = j0 + u * TS < n_fixed ? p2l[rank * P + D * C + j0 + u * TS] : -1;
#pragma unroll
      for (int u = 0; u < KB; ++u)
        if (j0 + u * TS < n_fixed)
          part += count_of(more_e[u]) / wmax;
    }
  part += dpp<kQuadSwap1>(part);
  if (TS >= 4) part += dpp<kQuadSwap2>(part);
  if (TS >= 8) part += dpp<kHalfMirror>(part);
  const float b = is_rank ? -part : 0.0f;
  // Big-M column, minilp.cu:275-281: b minus the weights of the rank's ends, own edges first
  float m = b;
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    constexpr int half = DM;
    const int end = e < half ? 2 * e : 2 * (e - half) + 1;
    m -= bpermute(w[end / TS], rank * TS + end % TS);
  }
  m = is_rank ? (m - 1.0f) + 1.0f : 0.0f;

  // ---- where my part of S comes from ----
  // 8 ranks, at most two slots: entry (rank, sub) is the rank's diagonal or minus the edges whose other
  // end is rank `sub`; the rank's ends are spread over every four of its lanes, a DPP operand away.
  float sel[kTile ? 1 : NE];
  const bool diagonal = KC == 1 && sub == rank;
  if constexpr (!kTile) {
#pragma unroll
    for (int e = 0; e < NE; ++e)
      sel[e] = bpermute(other[0], rank * TS + e) == sub && !diagonal ? -1.0f : 0.0f;
  }
  // Else: rows in LDS, a lane's columns adjacent (column r at (r % TS) * KC + r / TS); row stride GM + 4.
  auto tile_pos = [](int r) { return (r % TS) * KC + r / TS; };
  float *row_in_tile = tile + rank * (GM + 4);
  float *my_tile = row_in_tile + sub * KC;
  double *v_copy = reinterpret_cast<double *>(tile + GM * (GM + 4)), *my_v = v_copy + sub * KC;
  int other_at[E];
#pragma unroll
  for (int p = 0; p < E; ++p)
    other_at[p] = tile_pos(other[p]);
  const int own_at = tile_pos(rank);
  const f32x4 zero4{0.0f, 0.0f, 0.0f, 0.0f};
  auto clear_my_tile = [&]() {
    if constexpr (KC == 1) {
      *my_tile = 0.0f;
    } else {
#pragma unroll
      for (int k4 = 0; k4 < KC / 4; ++k4)
        reinterpret_cast<f32x4 *>(my_tile)[k4] = zero4;
    }
  };
  if constexpr (kTile)
    clear_my_tile();

  LPLB_STAMP(4);
  // ---- affine scaling ----
  float xo[E], xr[E], xs = 1.0f, xt = 1.0f, xM = 1.0f;
  float d_max = 0.0f;
  const int NV = 2 * n + G + 2;
  const int win_lo = a.step_rule == LPLB_STEP_REFERENCE_WINDOW ? (NV > 32 ? NV - 32 : 0) : 0;
  const bool with_zero = a.step_rule != LPLB_STEP_REFERENCE_WINDOW || NV < 32;
  bool win_o[E], win_r[E];
#pragma unroll
  for (int p = 0; p < E; ++p) {
    xo[p] = xr[p] = 1.0f;
    win_o[p] = on[p] && edge[p] >= win_lo;
    win_r[p] = on[p] && n + edge[p] >= win_lo;
  }
  const bool win_s = is_rank && 2 * n + rank >= win_lo;

  for (int step = 0; step < a.n_steps; ++step) {
    const float ss = xs * xs, st = xt * xt, sM = xM * xM;
    float so[E], sr[E], u[E], u_own[E], lam[E], mine[E];
#pragma unroll
    for (int p = 0; p < E; ++p) {
      so[p] = xo[p] * xo[p];
      sr[p] = xr[p] * xr[p];
      u[p] = on[p] ? __builtin_amdgcn_rcpf(so[p] + sr[p]) : 0.0f;
      const float wu = w[p] * u[p];
      const float ao = wu * so[p], ar = wu * sr[p];
      lam[p] = w_lap[p] * ao * sr[p];            // w^2 so sr / (so + sr)
      mine[p] = is_copy ? ar : ao;               // what the edge adds to q of this end's rank
      u_own[p] = is_copy ? 0.0f : u[p];          // every edge once
    }
    const float sigma = over_ranks_sum<TS>(over_ends_sum<TS, NE, E>(u_own));
    const float kappa = sM * __builtin_amdgcn_rcpf(1.0f + sM * sigma);
    const float v = is_rank ? m + over_ends_sum<TS, NE, E>(mine) : 0.0f;
    // the Laplacian's diagonal, added up slot by slot
    float lam_sum = ss;
    if constexpr (TS >= 4 && NE == 4) {
      const float pair = lam[0] + dpp_all<kQuadSwap1>(lam[0]);
      lam_sum += quad_bcast<0>(pair);
      lam_sum += quad_bcast<2>(pair);
    } else if constexpr (TS == 2 || NE == 2) {
#pragma unroll
      for (int p = 0; p < E; ++p)
        lam_sum += lam[p] + dpp_all<kQuadSwap1>(lam[p]);
    } else {
      lam_sum += over_ends_sum<TS, NE, E>(lam);
    }

    if (step == 0) LPLB_STAMP(5);
    double S[KC];
    const double dst = (double)st, dkv = (double)kappa * (double)v;
    if constexpr (!kTile) {
      const float v_col = bpermute(v, sub * TS);
      float t = diagonal ? lam_sum : 0.0f;
      if constexpr (DM == 2) {
        t = __builtin_fmaf(sel[0], quad_bcast<0>(lam[0]), t);
        t = __builtin_fmaf(sel[2], quad_bcast<2>(lam[0]), t);
        t = __builtin_fmaf(sel[1], quad_bcast<1>(lam[0]), t);
        t = __builtin_fmaf(sel[3], quad_bcast<3>(lam[0]), t);
      } else {
        t = __builtin_fmaf(sel[0], quad_bcast<0>(lam[0]), t);
        t = __builtin_fmaf(sel[1], quad_bcast<1>(lam[0]), t);
      }
      const double base = (EXACT || (rank < G && sub < G)) ? dst : 0.0;
      S[0] = __builtin_fma(dkv, (double)v_col, base) + (double)t;
    } else {
      // (LDS float adds without a return value, to my own rank's row; the row was cleared when it was
      // last read)
#pragma unroll
      for (int p = 0; p < E; ++p)
        __hip_atomic_fetch_add(row_in_tile + other_at[p], (NE < TS && sub >= NE) ? 0.0f : -lam[p], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WAVEFRONT);
      __hip_atomic_fetch_add(row_in_tile + own_at, sub == 0 ? lam_sum : 0.0f, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WAVEFRONT);
      v_copy[own_at] = (double)v;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      if constexpr (KC == 1) {
        const double base = (EXACT || (rank < G && sub < G)) ? dst : 0.0;
        S[0] = __builtin_fma(dkv, *my_v, base) + (double)*my_tile;
      } else {
        static_for<(KC + 3) / 4>([&](auto k4c) {
          constexpr int k4 = decltype(k4c)::value;
          const f32x4 t4 = reinterpret_cast<const f32x4 *>(my_tile)[k4];
          const double2 v01 = reinterpret_cast<const double2 *>(my_v)[2 * k4], v23 = reinterpret_cast<const double2 *>(my_v)[2 * k4 + 1];
          const float t[4] = {t4.x, t4.y, t4.z, t4.w};
          const double vc[4] = {v01.x, v01.y, v23.x, v23.y};
          static_for<4>([&](auto uu) {
            constexpr int u4 = decltype(uu)::value, k = 4 * k4 + u4;
            const double base = (EXACT || (rank < G && k * TS + sub < G)) ? dst : 0.0;
            S[k] = __builtin_fma(dkv, vc[u4], base) + (double)t[u4];
          });
        });
      }
      __builtin_amdgcn_wave_barrier();
      clear_my_tile();
    }
    double rhs = (EXACT || rank < G) ? 1000.0 * dkv - dst : 0.0;

    if (step == 0) LPLB_STAMP(6);
    // Gauss-Jordan elimination of [S | rhs] by columns, as in solve_kernel.h: the pivot's entry is
    // cleared as soon as it has been read as the pivot (so the multiple of the pivot row itself is zero),
    // column c + 1 goes through LDS right after its first update, and the next reciprocal is worked out
    // while that is on its way.  The right-hand side is kept by every lane of a rank.
    float y;
    if constexpr (KC == 1) {
      // One entry per lane: both the multiple f of the lane's row (entry (rank, c)) and the pivot row's
      // entry above the lane's column (entry (sub, c), by symmetry) come from column c in LDS, from
      // rows 9 doubles apart.  The chain from pivot to pivot is update -> LDS -> multiply -> update; the
      // next reciprocal is worked out meanwhile, and is set to zero in the pivot's own row.
      double *put = pivot_rows + rank * spread_row_doubles + sub;
      const double *get_row = pivot_rows + rank * spread_row_doubles, *get_col = pivot_rows + sub * spread_row_doubles;
      constexpr int kBuffer = 8 * spread_row_doubles;
      double rinv_of_row = 1.0, rinv = 0.0;
      static_for<GM>([&](auto cc) {
        constexpr int c = decltype(cc)::value;
        constexpr int at = (c % 2) * kBuffer + c;
        put[(c % 2) * kBuffer] = S[0];
        __builtin_amdgcn_wave_barrier();
        const double in_row = get_row[at], in_col = get_col[at];
        __builtin_amdgcn_sched_barrier(0);   // the reads stay here, ahead of their use
        rinv = rcp_f64(readlane(S[0], c * TS + c));
        rinv_of_row = set_rank<TS, c>(rinv_of_row, rinv);
        const double f = in_row * set_rank<TS, c>(rinv, 0.0);
        S[0] = __builtin_fma(-f, in_col, S[0]);
        rhs = __builtin_fma(-f, readlane(rhs, c * TS), rhs);
      });
      y = (float)(rhs * rinv_of_row);
    } else {
      // Several entries per lane.  The TS lanes of row i all need f_i = S[i][c] / pivot: the lane that
      // holds column c hands its entry round with one quad-permute DPP move per half.  That value is also
      // what the row adds to the pivot row in LDS (S[c][i] = S[i][c]), stored part by part, so a lane
      // reads the entries above its own columns, two per 16-byte read, from one of TS addresses.  A lane
      // also updates columns left of the pivot that share a register index with live ones; nothing reads
      // those again.
      constexpr int kStride = KC + 2;                 // doubles between the parts of a pivot row (distinct banks)
      constexpr int kPart = KC < 8 ? KC : 8;          // columns per batch of LDS reads
      constexpr int kParts = KC / kPart;
      static_assert(kParts <= 2 && TS * kStride <= kWave, "pivot rows are fetched in at most two batches");
      const int publish_at = (rank % TS) * kStride + rank / TS;
      const double *my_part = pivot_rows + sub * kStride;
      auto share = [](auto jc, double val) {     // val of lane j of every group of TS lanes
        constexpr int j = decltype(jc)::value;
        constexpr int ctrl = TS == 4 ? j * 0x55 : (j == 0 ? 0xA0 : 0xF5);
        int2 q = __builtin_bit_cast(int2, val);
        q.x = __builtin_amdgcn_mov_dpp(q.x, ctrl, 0xF, 0xF, false);   // (every lane has a source: no old value)
        q.y = __builtin_amdgcn_mov_dpp(q.y, ctrl, 0xF, 0xF, false);
        return __builtin_bit_cast(double, q);
      };
      // columns [q * kPart, (q + 1) * kPart) of the pivot row in buffer `parity`, those from k_from on
      auto load_part = [&](int parity, int q, int k_from, double (&buf)[kPart]) {
        const double2 *src = reinterpret_cast<const double2 *>(my_part + parity * kWave + q * kPart);
#pragma unroll
        for (int j = 0; j < kPart / 2; ++j)
          if (q * kPart + 2 * j + 1 >= k_from) {
            const double2 both = src[j];
            buf[2 * j] = both.x;
            buf[2 * j + 1] = both.y;
          }
        __builtin_amdgcn_sched_barrier(0);   // the reads stay here, ahead of their use
      };
      double head[2][kPart];
      double rinv_even = 1.0, rinv_odd = 1.0;   // (four lanes per rank: one of them serves all ranks)
      double rinv = rcp_f64(readlane(S[0], 0));
      S[0] = lp_clear_lane<1, 0>(S[0], 0);
      double col = share(std::integral_constant<int, 0>{}, S[0]);
      pivot_rows[publish_at] = col;
      __builtin_amdgcn_wave_barrier();
      load_part(0, 0, 0, head[0]);
      static_for<GM>([&](auto cc) {
        constexpr int c = decltype(cc)::value;
        constexpr int k1 = (c + 1) / TS;              // register of column c + 1, the first one still live
        constexpr int q0 = k1 / kPart;
        double body[kPart];
        auto clear = [&](auto kc, double f) {
          constexpr int k = decltype(kc)::value;
          if constexpr (k < KC) {
            if constexpr (k / kPart == q0)
              S[k] = __builtin_fma(-f, head[c % 2][k % kPart], S[k]);
            else
              S[k] = __builtin_fma(-f, body[k % kPart], S[k]);
          }
        };
        if constexpr (TS == 2 && c % 2)
          rinv_odd = set_rank<TS, c>(rinv_odd, rinv);
        else
          rinv_even = set_rank<TS, c>(rinv_even, rinv);
        const double f = col * rinv;   // multiple of row c to subtract from my row (0 in row c)
        double next_pivot = 1.0, estimate = 1.0, error = 0.0, next_col = 0.0;
        if constexpr (q0 + 1 < kParts)
          load_part(c % 2, q0 + 1, 0, body);
        clear(std::integral_constant<int, k1>{}, f);
        if constexpr (c + 1 < GM) {
          constexpr int holder = (c + 1) * TS + (c + 1) % TS;   // lane with entry (c + 1, c + 1)
          next_pivot = readlane(S[k1], holder);
          estimate = __builtin_amdgcn_rcp(next_pivot);
          S[k1] = lp_clear_lane<1, holder>(S[k1], 0);
          next_col = share(std::integral_constant<int, (c + 1) % TS>{}, S[k1]);
          pivot_rows[((c + 1) % 2) * kWave + publish_at] = next_col;
          __builtin_amdgcn_wave_barrier();
          constexpr int k1_next = (c + 2) / TS;
          if constexpr (k1_next < KC)
            load_part((c + 1) % 2, k1_next / kPart, k1_next, head[(c + 1) % 2]);
        }
        rhs = __builtin_fma(-f, readlane(rhs, c * TS), rhs);
        clear(std::integral_constant<int, k1 + 1>{}, f);
        if constexpr (c + 1 < GM)
          error = __builtin_fma(-next_pivot, estimate, 1.0);
        clear(std::integral_constant<int, k1 + 2>{}, f);
        clear(std::integral_constant<int, k1 + 3>{}, f);
        if constexpr (c + 1 < GM) {
          rinv = __builtin_fma(error, estimate, estimate);   // = rcp_f64(next_pivot)
        }
        static_for<(KC > k1 + 4 ? KC - k1 - 4 : 0)>([&](auto kk) {
          clear(std::integral_constant<int, k1 + 4 + decltype(kk)::value>{}, f);
        });
        col = next_col;
      });
      y = (float)(rhs * (TS == 2 && rank % 2 ? rinv_odd : rinv_even));
    }
    y = is_rank ? y : 0.0f;
    if (step == 0) LPLB_STAMP(7);

    // r = A^T w and the direction d = x (c - r); the edge part of w is
    // z = u (h + kappa (m.y - u.h - 1000)), h = -B^T y.
    float yk[E], yrep[E], hp[E], uhp[E];
#pragma unroll
    for (int p = 0; p < E; ++p) {
      const float y_other = bpermute(y, other[p] * TS);
      yk[p] = is_copy ? y_other : y;
      yrep[p] = is_copy ? y : y_other;
      hp[p] = -w[p] * (so[p] * yk[p] + sr[p] * yrep[p]);
      uhp[p] = u_own[p] * hp[p];
    }
    const float sumy = over_ranks_sum<TS>(y);
    const float my_uh = over_ranks_sum<TS>(m * y - over_ends_sum<TS, NE, E>(uhp));   // m.y - u.h
    const float from_M = my_uh - 1000.0f;
    const float shift = kappa * from_M;
    const float d_s = -xs * y;
    const float d_t = xt * (1.0f + sumy);
    const float d_M = xM * (shift * sigma - from_M);    // 1000 - m.y + the sum of z over the edges
    // Step length, minilp.cu:354-362.  NaN marks "not in the window".
    const float none = __builtin_nanf("");
    float d_o[E], d_r[E];
    float cand = win_s ? d_s : none;
#pragma unroll
    for (int p = 0; p < E; ++p) {
      const float z = u[p] * (hp[p] + shift);
      d_o[p] = -xo[p] * (w[p] * yk[p] + z);
      d_r[p] = -xr[p] * (w[p] * yrep[p] + z);
      cand = fmaxf(cand, win_o[p] ? d_o[p] : none);
      cand = fmaxf(cand, win_r[p] ? d_r[p] : none);
    }
    d_max = over_all_max<TS, NE>(fmaxf(cand, fmaxf(d_t, d_M)));
    if (with_zero)
      d_max = fmaxf(d_max, 0.0f);
    const float alpha = (float)step_length((double)d_max);
#pragma unroll
    for (int p = 0; p < E; ++p) {
      xo[p] *= 1.0f - alpha * d_o[p];
      xr[p] *= 1.0f - alpha * d_r[p];
    }
    xs *= 1.0f - alpha * d_s;
    xt *= 1.0f - alpha * d_t;
    xM *= 1.0f - alpha * d_M;
    if (step == 0) LPLB_STAMP(10);
  }

  LPLB_STAMP(11);
  // Feasibility, minilp.cu:369-385.
  float load[E], res = 0.0f;
#pragma unroll
  for (int p = 0; p < E; ++p) {
    load[p] = w[p] * (is_copy ? xr[p] : xo[p]);
    if (on[p])
      res = fmaxf(res, fabsf(xo[p] + xr[p] - xM - 1.0f));
  }
  const float row = xs - xt + m * xM - b + over_ends_sum<TS, NE, E>(load);
  if (is_rank)
    res = fmaxf(res, fabsf(row));
  res = over_all_max<TS, NE>(res);
  const bool ok = (double)d_max < 0.1 && 0.0 <= (double)xM && (double)xM < 1e-4 && (double)res < 0.05;
#pragma unroll
  for (int p = 0; p < E; ++p)
    if (on[p] && !is_copy && (NE >= TS || sub < NE))
      store_share(a, (int64_t)unit * n + edge[p], ok ? xo[p] : 0.5f);
  // Normalised counts of this group, for the caller.
  if (a.gw_out) {
    float *gw = a.gw_out + (int64_t)inst * a.n_experts + grp * G * L;
#pragma unroll
    for (int u = 0; u < KG; ++u)
      if (lane + u * kWave < G * L)
        gw[lane + u * kWave] = out_cnt[u] / wmax;
    for (int i = lane + KG * kWave; i < G * L; i += kWave)
      gw[i] = count_of(grp * G * L + i) / wmax;
  }
  LPLB_STAMP(12);
  return ok ? 1 : 0;
}

// The form of the solver for ROWS LPs per wave with EPL edges per lane, and the LDS it needs per wave.
template <int GM, int DM, int ROWS, int EPL> constexpr bool takes_spread_form() {
  return ROWS == 1 && EPL == 1 && spread_shape(GM, DM);
}
template <int GM, int DM, int ROWS = 1, int EPL = 1> constexpr int lp_pivot_doubles() {
  return takes_spread_form<GM, DM, ROWS, EPL>() ? spread_pivot_doubles(GM) : 2 * kWave;
}
template <int GM, int DM, int ROWS = 1, int EPL = 1> constexpr int lp_tile_floats() {
  return takes_spread_form<GM, DM, ROWS, EPL>() ? spread_tile_floats(GM, DM) : assembly_tile_floats(GM, ROWS);
}
template <int GM, int DM, bool EXACT, int ROWS, int EPL, typename Counts>
__device__ inline int solve_lps(const SolveArgs &a, int first_unit, float *staged_counts, int *rep_of_edge,
                                double *pivot_rows, float *tile, Counts counts_have_come) {
  if constexpr (takes_spread_form<GM, DM, ROWS, EPL>())
    return solve_lp_spread<GM, DM, EXACT>(a, first_unit, staged_counts, rep_of_edge, pivot_rows, tile, counts_have_come);
  else
    return solve_lp<GM, DM, EXACT, ROWS, EPL>(a, first_unit, staged_counts, rep_of_edge, pivot_rows, tile);
}

} // namespace lplb
