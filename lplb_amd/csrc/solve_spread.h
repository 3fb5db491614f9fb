// LP solver, one LP per wave, groups of up to 32 ranks: the group's G x G system spread over all 64
// lanes.  Same problem, method and arithmetic as solve_kernel.h (read that first); what differs is who
// holds what.
//
// A lone wave issues one instruction every 2.3 ns (4.4 ns if it is an fp64 one that needs the one before), whatever the
// instruction does for how many lanes, a reciprocal takes 9 ns, what goes through LDS 30 ns and 3 more for every further
// read: the time of an LP is the number of instructions on its path and the round trips through LDS in it.
// With one lane per rank and one lane per edge (solve_kernel.h) 48 or 56 of the 64 lanes idle, every
// lane carries a whole row of S through assembly and elimination, and what goes from edges to ranks and
// back goes through ten ds_bpermute per step.  Here
//   * wave lane l belongs to rank l / TS (TS = 64 / GM lanes per rank) and holds the columns
//     k * TS + l % TS, k < KC = GM / TS, of that rank's row of S: 1 column at 8 ranks, 4 at 16, 16 at 32;
//   * a rank's lanes also hold the rank's replica edges, both those it is the original of and those whose
//     copy it hosts ("edge ends": end e = 2 d is the rank's own edge in slot d, e = 2 d + 1 the edge
//     copied into slot d; lane l holds ends l % TS + TS * p).  Every edge lives twice, at its two ends,
//     with the same values computed twice; a rank's sums over its edges are DPP adds inside its lanes,
//     and the only value that has to travel is the solution y of the other end's rank;
//   * pivots are taken two at a time, so that there is one round trip through LDS for two.
// Measured per affine-scaling step, one wave on the GPU, pivots one by one -> two at a time (and sums without
// wait states, moves folded into them, no sum over the edges between solution and step length):
// (8, 2) 0.66 -> 0.55 us, half of it elimination; (16, 2) 1.21 -> 1.13; (32, 2) 2.87 -> 2.54, bound by the number of
// instructions.  With one lane per rank and edge (8, 2) took 1.15 us.
// (A form in which rank i is lane i of every 16-lane row and holds its whole row, the elimination made of
// fp64 multiply-adds with a row_newbcast operand, has pivots of 40 instead of 60 ns and no LDS in them; but
// getting the rows into that shape costs 0.25 us a step more than it gains at 8 ranks.  At 16 and 32 ranks, where the
// tile can be read in that shape for nothing, pivots in pairs, a lane with one or two rows and every fourth column: a step takes 0.13 and 0.42 us
// longer, since a row's multiples are worked out by four lanes, not two, in the chain, and the next pair's columns take two stores.)
#pragma once
#include "solve_kernel.h"

namespace lplb {

// Which instantiations take this form (one LP per wave, one edge per lane in the other form).
constexpr bool spread_shape(int gm, int dm) { return gm <= 32 && gm * dm <= 128 && dm <= 8; }

// LDS per wave: what the elimination passes between lanes (8 ranks: the rows of S and the right-hand side, and the
// constants of the pivot rows; else an area per pair of pivots, with the pairs of entries of all rows, zeros and, with four
// lanes per rank, a place for those lanes that hold none, then the right-hand sides) and, except at 8 ranks with at most
// two slots, the tile in which the rows of S are put together, followed by a copy of v.
constexpr int kRow8 = 10;   // 8 ranks: doubles from row to row (pairs on 16-byte boundaries, a column's in distinct banks)
constexpr int spread_part_doubles(int gm) { return 2 * (gm * gm / kWave) + 2; }   // the rows of equal number modulo TS (parts in distinct banks)
constexpr int spread_pair_area(int gm) { return kWave / gm * spread_part_doubles(gm) + 4; }
constexpr int spread_pivot_doubles(int gm) { return gm <= 8 ? 9 * kRow8 + 16 : gm / 2 * spread_pair_area(gm) + gm; }
constexpr bool spread_uses_tile(int gm, int dm) { return gm > 8 || dm > 2; }
constexpr int spread_tile_floats(int gm, int dm) { return spread_uses_tile(gm, dm) ? gm * (gm + 4) + 2 * gm : 4; }

// v of the lane that CTRL names, for controls in which every lane has a source.
template <int CTRL> __device__ inline float dpp_all(float v) {
  // (zeros for lanes without a source, of which there are none, let the compiler fold the move into its user)
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
constexpr int kRowRor8 = 0x128;
template <int LANE> __device__ inline float quad_bcast(float v) { return dpp_all<LANE * 0x55>(v); }

// Sums and maxima across the four 16-lane rows (complete in the last row) and, for maxima, inside them.
// Written out because the compiler splits a DPP operand with a row mask, or one of a maximum, into two to
// four instructions, and does not fill the two wait states that a DPP operand needs with another sum's instructions.
#define LPLB_DPP(OP, REG, CTRL, ROWS) OP "_dpp " REG ", " REG ", " REG " " CTRL " row_mask:" ROWS " bank_mask:0xf\n\t"
#define LPLB_WAIT_DPP(OP, CTRL, ROWS) "s_nop 1\n\t" LPLB_DPP(OP, "%0", CTRL, ROWS)
#define LPLB_ROWS(OP) LPLB_WAIT_DPP(OP, "row_bcast:15", "0xa") LPLB_WAIT_DPP(OP, "row_bcast:31", "0xc")
#define LPLB_MAX(CTRL) LPLB_WAIT_DPP("v_max_f32", CTRL, "0xf")
#define LPLB_MAX_ROWS LPLB_MAX("row_ror:8") LPLB_ROWS("v_max_f32")
__device__ inline float rows_sum(float v) {
  asm(LPLB_ROWS("v_add_f32") : "+v"(v));
  return readlane(v, kWave - 1);
}
__device__ inline void rows_sums(float &v, float &w) {
  asm("s_nop 1\n\t" LPLB_DPP("v_add_f32", "%0", "row_bcast:15", "0xa") LPLB_DPP("v_add_f32", "%1", "row_bcast:15", "0xa")
      "s_nop 0\n\t" LPLB_DPP("v_add_f32", "%0", "row_bcast:31", "0xc") LPLB_DPP("v_add_f32", "%1", "row_bcast:31", "0xc")
      : "+v"(v), "+v"(w));
  v = readlane(v, kWave - 1);
  w = readlane(w, kWave - 1);
}
template <bool Q2, bool H> __device__ inline float wave_max_of_groups(float v) {
  if constexpr (Q2 && H)
    asm(LPLB_MAX("quad_perm:[1,0,3,2]") LPLB_MAX("quad_perm:[2,3,0,1]") LPLB_MAX("row_half_mirror") LPLB_MAX_ROWS : "+v"(v));
  else if constexpr (Q2)
    asm(LPLB_MAX("quad_perm:[1,0,3,2]") LPLB_MAX("quad_perm:[2,3,0,1]") LPLB_MAX_ROWS : "+v"(v));
  else if constexpr (H)
    asm(LPLB_MAX("quad_perm:[1,0,3,2]") LPLB_MAX("row_half_mirror") LPLB_MAX_ROWS : "+v"(v));
  else
    asm(LPLB_MAX("quad_perm:[1,0,3,2]") LPLB_MAX_ROWS : "+v"(v));
  return readlane(v, kWave - 1);
}
#undef LPLB_MAX_ROWS
#undef LPLB_MAX
#undef LPLB_ROWS
#undef LPLB_WAIT_DPP
#undef LPLB_DPP

// %0 += SEL times %1 of lane N of every four
#define LPLB_FMAC(SEL, N) "v_fmac_f32_dpp %0, %1, " SEL " quad_perm:[" #N "," #N "," #N "," #N "] row_mask:0xf bank_mask:0xf\n\t"
// The value is formed here: a product is not contracted with an addition whose operand comes by DPP (two instructions then).
__device__ inline float formed_here(float v) {
  asm("" : "+v"(v));
  return v;
}

// Over the ranks: v is the same in the TS lanes of each rank; the result is wave-uniform.
template <int TS> __device__ inline float over_ranks_in_row(float v) {
  if (TS <= 2) v += dpp_all<kQuadSwap2>(v);
  if (TS <= 4) v += dpp_all<kHalfMirror>(v);
  return v + dpp_all<kRowRor8>(v);
}
template <int TS> __device__ inline float over_ranks_sum(float v) { return rows_sum(over_ranks_in_row<TS>(v)); }
template <int TS> __device__ inline void over_ranks_sums(float &v, float &w) {
  v = over_ranks_in_row<TS>(v);
  w = over_ranks_in_row<TS>(w);
  rows_sums(v, w);
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
  return wave_max_of_groups<(TS <= 2 || NE > 2), (TS <= 4 || NE > 4)>(v);
}

// LDS by its own addresses (32 bits), so that an address can be chosen lane by lane with one move.
typedef __attribute__((address_space(3))) double lds_double;
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) f64x2 lds_f64x2;
typedef int i32x4_in_lds __attribute__((ext_vector_type(4)));
__device__ inline double2 lds_pair(const lds_double *base, int at) {
  const f64x2 v = *reinterpret_cast<const lds_f64x2 *>(base + at);
  return double2{v.x, v.y};
}
// v of the last of every eight lanes.
__device__ inline float last_of_eight(float v) {
  const int q = __builtin_bit_cast(int, quad_bcast<3>(v));
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(q, q, 0x104 /* row_shl:4 */, 0xF, 0x5, false));
}
constexpr int kIdentityPerm = 0xE4;   // quad_perm [0,1,2,3]
// v with the 16-lane row ROW made zero, through its high word only (what is left of a number is a denormal below 2^-1022).
template <int ROW> __device__ inline double clear_dpp_row(double v) {
  int2 q = __builtin_bit_cast(int2, v);
  q.y = __builtin_amdgcn_update_dpp(q.y, 0, kIdentityPerm, 1 << ROW, 0xF, false);
  return __builtin_bit_cast(double, q);
}
// v of the other rank of the pair (2 p, 2 p + 1); v is the same in the TS lanes of each rank.
template <int TS> __device__ inline double rank_partner(double v) {
  constexpr int ctrl = TS == 2 ? kQuadSwap2 : kHalfMirror;
  int2 q = __builtin_bit_cast(int2, v);
  q.x = __builtin_amdgcn_mov_dpp(q.x, ctrl, 0xF, 0xF, false);
  q.y = __builtin_amdgcn_mov_dpp(q.y, ctrl, 0xF, 0xF, false);
  return __builtin_bit_cast(double, q);
}

// Arguments, LDS contracts and the returned value as for solve_lp; pivot_rows has spread_pivot_doubles(GM)
// doubles, tile spread_tile_floats(GM, DM) floats, both 16-byte aligned; rep_of_edge kWave ints, or twice
// that if GM * DM > kWave.
// counts_have_come: called once what does not depend on the counts is done if a.counts_by_caller; returns when the
// counts are in staged_counts (as int32, 16-byte aligned, with a zero behind the last and up to a multiple of four: true), or when they will not come: then -1 is returned, nothing solved or stored.
// STAGED: the counts fit in LDS (a.staged_stride > 0, or they are the caller's).  Known here, a count is an LDS read; else it is
// a load that finds out where its address is and waits for both kinds of memory, one after the other: 0.55 us from the counts' arrival
// until the LP has its weights, 0.25 this way (8 ranks, 256 experts), and as much again at the end for the normalised counts.
template <int GM, int DM, bool EXACT, bool STAGED, typename Counts>
__device__ inline int solve_lp_spread(const SolveArgs &a, int unit, float *staged_counts, int *rep_of_edge,
                                      double *pivot_rows, float *tile, Counts counts_have_come) {
  static_assert(spread_shape(GM, DM) && (GM == 8 || GM == 16 || GM == 32), "a lane holds GM * GM / 64 entries of S");
  constexpr int TS = kWave / GM, KC = GM / TS;
  constexpr int NE = 2 * DM, E = NE > TS ? NE / TS : 1;
  constexpr bool kTile = spread_uses_tile(GM, DM);
  constexpr int KB = 4;   // counts of experts that cannot move a lane prefetches
  const int lane = threadIdx.x % kWave;
  const int rank = lane / TS, sub = lane % TS;
  const int G = EXACT ? GM : a.G, D = EXACT ? DM : a.D;
  const int C = a.C, n = G * D, n_fixed = a.n_fixed;
  const int L = D * C + n_fixed, P = L + D * C;
  const int grp = unit % a.n_group, inst = unit / a.n_group;
  const int32_t *__restrict__ wl = a.workload + (int64_t)inst * a.n_experts;
  const int32_t *__restrict__ p2l = a.phy2log + (int64_t)grp * G * P;
  const bool is_rank = EXACT || rank < G;
  // The counts, as int32: in LDS if they fit there (entry n_experts is a zero), else in global memory.
  const bool staged = STAGED || a.staged_stride > 0 || a.counts_by_caller;
  int32_t *const counts_in_lds = reinterpret_cast<int32_t *>(staged_counts);
  auto index_of = [&](int e) { return e < 0 || e > a.n_experts ? a.n_experts : e; };   // of an expert; no expert: of a zero
  auto count_at = [&](int i) -> float {
    return staged ? (float)counts_in_lds[i] : i < a.n_experts ? (float)wl[i] : 0.0f;
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
  int first_at[E], orig_rank[E];   // (indexes of counts)
#pragma unroll
  for (int p = 0; p < E; ++p) {
    first_at[p] = (on[p] && C > 0) ? p2l[rank * P + slot[p]] : -1;
    orig_rank[p] = on[p] ? a.r2o[rank * D + slot[p]] : 0;
  }
  int fixed_at[KB];
#pragma unroll
  for (int u = 0; u < KB; ++u) {
    const int j = sub + u * TS;
    fixed_at[u] = (is_rank && j < n_fixed) ? p2l[rank * P + D * C + j] : -1;
  }
  int own_max = 0;   // the largest count this lane has seen
  constexpr int KG = 4;   // counts a lane has under way
  if (!a.counts_by_caller) {
#pragma unroll KG
    for (int i = lane; i < a.n_experts; i += kWave) {
      const int32_t cnt = wl[i];
      own_max = max(own_max, cnt);
      if (staged)
        counts_in_lds[i] = cnt;
    }
    if (staged && lane == 0)
      counts_in_lds[a.n_experts] = 0;
  }

  // ---- what the topology alone decides (while the caller's counts are on their way): the other ends of my edge ends
  //      (minilp.cu:203-221) ----
  int edge[E], other[E];
#pragma unroll
  for (int p = 0; p < E; ++p) {
    orig_rank[p] = orig_rank[p] < 0 ? 0 : (orig_rank[p] >= G ? G - 1 : orig_rank[p]);
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
#pragma unroll
  for (int p = 0; p < E; ++p) {
    const int rep = on[p] && !is_copy ? rep_of_edge[edge[p]] : rank;
    other[p] = on[p] ? (is_copy ? orig_rank[p] : rep) : rank;
  }
  // Where my part of S comes from.
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
  // Where the elimination's entries are in LDS.
  lds_double *const pivot_at = (lds_double *)pivot_rows;
  constexpr int kPartDoubles = spread_part_doubles(GM), kPairArea = spread_pair_area(GM);
  lds_double *my_rhs, *my_entry = nullptr, *put_pair[2] = {};
  const lds_double *row_of_pair[GM / 2] = {};   // where a lane finds its row's entries in the pivot columns
  const lds_double *my_column = nullptr;                         // 8 ranks
  const lds_double *my_part = nullptr, *all_rhs = nullptr;   // 16 and 32
  const lds_double *my_diagonal = nullptr, *partners_diagonal = nullptr, *my_off_diagonal = nullptr;
  if constexpr (KC == 1) {
    my_entry = pivot_at + rank * kRow8 + sub;
    my_rhs = pivot_at + 8 * kRow8 + rank;
    my_column = pivot_at + (sub == 7 ? 8 : sub) * kRow8;
    lds_double *constants = pivot_at + 9 * kRow8;   // (-1, 0) four times, (0, -1) four times
    if (lane < 16)
      constants[lane] = lane % 2 == lane / 8 ? -1.0 : 0.0;
#pragma unroll
    for (int p = 0; p < 4; ++p)
      row_of_pair[p] = rank / 2 == p ? constants + rank % 2 * 8 : pivot_at + rank * kRow8;
  } else {
    const int at = (rank % TS) * kPartDoubles + rank / TS * 2;
    constexpr int zeros = TS * kPartDoubles, nowhere = zeros + 2;
    put_pair[0] = pivot_at + (sub < 2 ? at + sub : nowhere);
    put_pair[1] = pivot_at + (sub < 2 ? nowhere : at + sub - 2);
#pragma unroll
    for (int p = 0; p < GM / 2; ++p)
      row_of_pair[p] = pivot_at + (rank / 2 == p ? zeros : at);
    my_part = pivot_at + sub * kPartDoubles;
    all_rhs = pivot_at + GM / 2 * kPairArea;
    my_rhs = pivot_at + GM / 2 * kPairArea + rank;
    if (lane < GM)
      pivot_at[lane / 2 * kPairArea + zeros + lane % 2] = 0.0;
    const lds_double *area = pivot_at + rank / 2 * kPairArea;
    const int partner = rank ^ 1;
    my_diagonal = area + at + rank % 2;
    my_off_diagonal = area + at + 1 - rank % 2;
    partners_diagonal = area + (partner % TS) * kPartDoubles + partner / TS * 2 + partner % 2;
  }
#pragma unroll
  for (int p = 0; p < E; ++p)
    first_at[p] = index_of(first_at[p]);
#pragma unroll
  for (int u = 0; u < KB; ++u)
    fixed_at[u] = index_of(fixed_at[u]);

  // ---- the counts ----
  if (a.counts_by_caller) {
    if (!counts_have_come())
      return -1;
    for (int i = 4 * lane; i < a.n_experts; i += 4 * kWave) {
      const i32x4_in_lds c = *reinterpret_cast<const i32x4_in_lds *>(counts_in_lds + i);
      own_max = max(max(own_max, max(c.x, c.y)), max(c.z, c.w));
    }
  }
  __builtin_amdgcn_wave_barrier();   // staged counts are visible to the whole wave
  float first_cnt[E], fixed_cnt = 0.0f;
#pragma unroll
  for (int p = 0; p < E; ++p)
    first_cnt[p] = count_at(first_at[p]);
#pragma unroll
  for (int u = 0; u < KB; ++u)
    fixed_cnt += count_at(fixed_at[u]);
  const float wmax = wave_max_of_groups<true, true>((float)own_max);

  LPLB_STAMP(1);
  // ---- weights: tokens of the edge's expert set over the largest count (added up first: whole numbers, and one division) ----
  float w[E], w_lap[E];   // w_lap: zero where the edge is no edge of the Laplacian (inactive, or a loop)
#pragma unroll
  for (int p = 0; p < E; ++p) {
    float own = first_cnt[p];
    if (on[p])
      for (int c = 1; c < C; ++c)
        own += count_at(index_of(p2l[rank * P + c * D + slot[p]]));
    own = on[p] && C > 0 ? own / wmax : 0.0f;
    // a copied edge's weight is its original's, found at the even lane of that rank
    const float copied = bpermute(own, orig_rank[p] * TS + (sub & ~1));
    w[p] = on[p] ? (is_copy ? copied : own) : 0.0f;
    w_lap[p] = other[p] == rank ? 0.0f : w[p];
  }
  LPLB_STAMP(2);
  // ---- per-rank constants, the same in all lanes of a rank ----
  // b = -(load of the experts that cannot move), minilp.cu:223-234
  if (is_rank)
    for (int j0 = sub + KB * TS; j0 < n_fixed; j0 += KB * TS) {
      int more_e[KB];
#pragma unroll
      for (int u = 0; u < KB; ++u)
        more_e[u] = j0 + u * TS < n_fixed ? p2l[rank * P + D * C + j0 + u * TS] : -1;
#pragma unroll
      for (int u = 0; u < KB; ++u)
        fixed_cnt += count_at(index_of(more_e[u]));
    }
  fixed_cnt += dpp_all<kQuadSwap1>(fixed_cnt);
  if (TS >= 4) fixed_cnt += dpp_all<kQuadSwap2>(fixed_cnt);
  if (TS >= 8) fixed_cnt += dpp_all<kHalfMirror>(fixed_cnt);
  const float b = is_rank && n_fixed > 0 ? -fixed_cnt / wmax : 0.0f;
  // Big-M column, minilp.cu:275-281: b minus the weights of the rank's ends
  const float m = is_rank ? ((b - over_ends_sum<TS, NE, E>(w)) - 1.0f) + 1.0f : 0.0f;

  LPLB_STAMP(4);
  // ---- affine scaling ----
  float xo[E], xr[E], xs = 1.0f, xt = 1.0f, xM = 1.0f;
  float d_max = 0.0f;
  const int NV = 2 * n + G + 2;
  const int win_lo = a.step_rule == LPLB_STEP_REFERENCE_WINDOW ? (NV > 32 ? NV - 32 : 0) : 0;
  float at_least = a.step_rule != LPLB_STEP_REFERENCE_WINDOW || NV < 32 ? 0.0f : __builtin_nanf("");
  asm("" : "+v"(at_least));   // (one operand of a maximum; known to be one of the two, it becomes a select behind one)
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
      lam[p] = formed_here(w_lap[p] * ao * sr[p]);   // w^2 so sr / (so + sr)
      mine[p] = is_copy ? ar : ao;               // what the edge adds to q of this end's rank
      u_own[p] = is_copy ? 0.0f : u[p];          // every edge once
    }
    const float sum_mine = over_ends_sum<TS, NE, E>(mine), sum_u = over_ends_sum<TS, NE, E>(u_own);
    const float v = is_rank ? m + sum_mine : 0.0f;
    float v_col = 0.0f;
    if constexpr (!kTile) {
      v_col = bpermute(v, sub * TS);
      __builtin_amdgcn_sched_barrier(0);   // (on its way while the sum over the edges is formed)
    }
    const float sigma = over_ranks_sum<TS>(sum_u);
    const float kappa = sM * __builtin_amdgcn_rcpf(1.0f + sM * sigma);
    // the Laplacian's diagonal
    const float lam_sum = ss + over_ends_sum<TS, NE, E>(lam);

    if (step == 0) LPLB_STAMP(5);
    double S[KC];
    const double dst = (double)st, dk = (double)kappa, dv = (double)v, dkv = dk * dv;
    if constexpr (!kTile) {
      float t = diagonal ? lam_sum : 0.0f;
      if constexpr (DM == 2)
        asm("s_nop 1\n\t" LPLB_FMAC("%2", 0) LPLB_FMAC("%4", 2) LPLB_FMAC("%3", 1) LPLB_FMAC("%5", 3)
            : "+v"(t) : "v"(lam[0]), "v"(sel[0]), "v"(sel[1]), "v"(sel[2]), "v"(sel[3]));
      else
        asm("s_nop 1\n\t" LPLB_FMAC("%2", 0) LPLB_FMAC("%3", 1) : "+v"(t) : "v"(lam[0]), "v"(sel[0]), "v"(sel[1]));
      const double base = (EXACT || (rank < G && sub < G)) ? dst : 0.0;
      S[0] = __builtin_fma(dk, dv * (double)v_col, base + (double)t);
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
    double rhs = (EXACT || rank < G) ? __builtin_fma(dk, 1000.0 * dv, -dst) : 0.0;

    if (step == 0) LPLB_STAMP(6);
    // Gauss-Jordan elimination of [S | rhs], two pivots at a time.  Columns c and c + 1 of the rows that are left go
    // through LDS once; from there every lane has its row's entries in them, the two pivot rows' entries above its own
    // columns (by symmetry those columns' entries of the row of that number), the pivot block [a b; b d] and the pivot rows'
    // right-hand sides.  With l = b / a the second pivot is d - b l, and the second pivot row and the entries in its
    // column are what is left after l times the first: the steps of single pivots, so that what the pivots cancel is lost once
    // and the same for all rows.  (The inverse of the block applied to a row loses it anew in every row: one reciprocal less and
    // 0.04 us less a step at 8 ranks, but 67 instead of 29 of 8000 LPs of 56 tokens then miss the feasibility test.  The second
    // reciprocal as a times that of the determinant, to start both at once: 0.56 instead of 0.54 us a step.)  The chain from
    // pair to pair is update -> LDS -> two reciprocals -> update, one round trip through LDS for two pivots.  Lanes also update
    // columns left of the pivots that share a register index with live ones; nothing reads those again.  The right-hand side is
    // kept by every lane of a rank.
    float y;
    struct Pivots {
      double inv_first, inv_second, l;
    };
    auto pivots_of = [](const double2 &ab, double d) {
      Pivots v;
      v.inv_first = rcp_f64(ab.x);
      v.l = ab.y * v.inv_first;
      v.inv_second = rcp_f64(__builtin_fma(-ab.y, v.l, d));
      return v;
    };
    if constexpr (KC == 1) {
      // One entry per lane.  The pivot rows themselves are replaced by the rows divided by the block: as if they were
      // zero and had the entries (-1, 0) and (0, -1), which their lanes read from constants instead.  The last pair comes first:
      // column 7 is not used any more once it has been published, and its lanes go on with the right-hand side (row 8 in LDS),
      // which so ends up in the lanes that sums over the ranks are taken from.
      static_for<GM / 2>([&](auto pc) {
        constexpr int p = GM / 2 - 1 - decltype(pc)::value, c = 2 * p;
        *(p == GM / 2 - 1 || sub < 7 ? my_entry : my_rhs) = S[0];
        if constexpr (p == GM / 2 - 1) {
          *my_rhs = rhs;
          S[0] = sub == 7 ? rhs : S[0];
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const double2 ab = lds_pair(pivot_at, c * kRow8 + c);
        const double d = pivot_at[(c + 1) * kRow8 + c + 1];
        __builtin_amdgcn_sched_barrier(0);   // the reads stay here, ahead of their use, those of the longest chain first
        const double2 in_row = lds_pair(row_of_pair[p], c);
        __builtin_amdgcn_sched_barrier(0);
        const double2 above = lds_pair(my_column, c);
        __builtin_amdgcn_sched_barrier(0);
        S[0] = clear_dpp_row<p>(S[0]);
        const Pivots v = pivots_of(ab, d);
        S[0] = __builtin_fma(-(in_row.x * above.x), v.inv_first, S[0]);
        const double second = __builtin_fma(-in_row.x, v.l, in_row.y) * __builtin_fma(-above.x, v.l, above.y);
        S[0] = __builtin_fma(-second, v.inv_second, S[0]);
      });
      y = (float)S[0];   // (in the last lane of every rank)
    } else {
      // Several entries per lane.  Every pair has an area of its own in LDS: the pairs of entries of all rows, part by
      // part (rows of equal number modulo TS), so that a lane reads those above its own columns from one of TS addresses.
      // The lanes of the pivot rows read zeros for their own row, which leaves it alone; what it takes to divide the
      // right-hand side by the block at the end is still there then.  The next pair's columns are updated first and
      // published, and the rest of the update runs while they are on their way.
      double2 in_row[2], ab[2], r[2], above[2][KC];
      double d[2];
      auto publish = [&](auto pc) {
        constexpr int p = decltype(pc)::value;
        put_pair[TS == 2 ? 0 : p % 2][p * kPairArea] = S[2 * p / TS];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_sched_barrier(0);
      };
      auto fetch = [&](auto pc) {
        constexpr int p = decltype(pc)::value, c = 2 * p, first_live = (c + 2) / TS;
        auto area_of = [](int row) { return (row % TS) * kPartDoubles + row / TS * 2; };
        ab[p % 2] = lds_pair(pivot_at, p * kPairArea + area_of(c));
        d[p % 2] = pivot_at[p * kPairArea + area_of(c + 1) + 1];
        __builtin_amdgcn_sched_barrier(0);   // the reads stay here, ahead of their use, those of the longest chain first
        in_row[p % 2] = lds_pair(row_of_pair[p], p * kPairArea);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = first_live; k < KC; ++k)
          above[p % 2][k] = lds_pair(my_part, p * kPairArea + 2 * k);
        __builtin_amdgcn_sched_barrier(0);
      };
      auto exchange_rhs = [&](auto pc) {
        constexpr int p = decltype(pc)::value;
        *my_rhs = rhs;
        __builtin_amdgcn_wave_barrier();
        r[p % 2] = lds_pair(all_rhs, 2 * p);
        __builtin_amdgcn_sched_barrier(0);
      };
      publish(std::integral_constant<int, 0>{});
      fetch(std::integral_constant<int, 0>{});
      exchange_rhs(std::integral_constant<int, 0>{});
      static_for<GM / 2>([&](auto pc) {
        constexpr int p = decltype(pc)::value, first_live = (2 * p + 2) / TS;
        const Pivots v = pivots_of(ab[p % 2], d[p % 2]);
        // (f1 / f0: what of the second / first row, as it is, to subtract)
        const double f1 = __builtin_fma(-in_row[p % 2].x, v.l, in_row[p % 2].y) * v.inv_second;
        const double f0 = __builtin_fma(-v.l, f1, in_row[p % 2].x * v.inv_first);
        auto update = [&](int k) {
          S[k] = __builtin_fma(-f0, above[p % 2][k].x, __builtin_fma(-f1, above[p % 2][k].y, S[k]));
        };
        auto update_rhs = [&]() { rhs = __builtin_fma(-f1, r[p % 2].y, __builtin_fma(-f0, r[p % 2].x, rhs)); };
        if constexpr (p + 1 < GM / 2) {
          update(first_live);
          publish(std::integral_constant<int, p + 1>{});
          fetch(std::integral_constant<int, p + 1>{});
          update_rhs();
          exchange_rhs(std::integral_constant<int, p + 1>{});
#pragma unroll
          for (int k = first_live + 1; k < KC; ++k)
            update(k);
        } else {
          update_rhs();
        }
      });
      const double own = *my_diagonal, b = *my_off_diagonal, partner = *partners_diagonal, partners_rhs = rank_partner<TS>(rhs);
      const bool is_second = rank % 2;
      const Pivots v = pivots_of(double2{is_second ? partner : own, b}, is_second ? own : partner);
      const double first_rhs = is_second ? partners_rhs : rhs, second_rhs = is_second ? rhs : partners_rhs;
      const double y_second = __builtin_fma(-v.l, first_rhs, second_rhs) * v.inv_second;
      const double y_first = __builtin_fma(-v.l, y_second, first_rhs * v.inv_first);
      y = (float)(is_second ? y_second : y_first);
    }
    y = is_rank ? y : 0.0f;
    if (step == 0) LPLB_STAMP(7);

    // r = A^T w and the direction d = x (c - r); the edge part of w is
    // z = u (h + kappa (m.y - u.h - 1000)), h = -B^T y; m.y - u.h = v.y, because q = B u.
    float y_other[E];
#pragma unroll
    for (int p = 0; p < E; ++p)
      y_other[p] = bpermute(y, other[p] * TS + (KC == 1 ? TS - 1 : 0));
    float sumy = y, vy = formed_here(v * y);
    over_ranks_sums<TS>(vy, sumy);
    if constexpr (KC == 1)
      y = is_rank ? last_of_eight(y) : 0.0f;
    float yk[E], yrep[E], hp[E];
#pragma unroll
    for (int p = 0; p < E; ++p) {
      yk[p] = is_copy ? y_other[p] : y;
      yrep[p] = is_copy ? y : y_other[p];
      hp[p] = -w[p] * (so[p] * yk[p] + sr[p] * yrep[p]);
    }
    const float from_M = vy - 1000.0f;
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
    d_max = over_all_max<TS, NE>(fmaxf(cand, fmaxf(fmaxf(d_t, d_M), at_least)));
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
  // (no float lies between the reference's limits 0.1, 1e-4 and 0.05, which are doubles, and these)
  static_assert(0.1f > 0.1 && 1e-4f < 1e-4 && 0.05f > 0.05, "how the limits round");
  const bool ok = d_max < 0.1f && 0.0f <= xM && xM <= 1e-4f && res < 0.05f;
#pragma unroll
  for (int p = 0; p < E; ++p)
    if (on[p] && !is_copy && (NE >= TS || sub < NE))
      store_share(a, (int64_t)unit * n + edge[p], ok ? xo[p] : 0.5f);
  // Normalised counts of this group, for the caller.
  if (a.gw_out) {
    float *gw = a.gw_out + (int64_t)inst * a.n_experts + grp * G * L;
#pragma unroll KG
    for (int i = lane; i < G * L; i += kWave)
      gw[i] = count_at(grp * G * L + i) / wmax;
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
template <int GM, int DM, bool EXACT, int ROWS, int EPL, bool STAGED, typename Counts>
__device__ inline int solve_lps(const SolveArgs &a, int first_unit, float *staged_counts, int *rep_of_edge,
                                double *pivot_rows, float *tile, Counts counts_have_come) {
  if constexpr (takes_spread_form<GM, DM, ROWS, EPL>())
    return solve_lp_spread<GM, DM, EXACT, STAGED>(a, first_unit, staged_counts, rep_of_edge, pivot_rows, tile, counts_have_come);
  else
    return solve_lp<GM, DM, EXACT, ROWS, EPL, STAGED>(a, first_unit, staged_counts, rep_of_edge, pivot_rows, tile);
}

#undef LPLB_FMAC
} // namespace lplb
