// LP solver, device side: one wave64 per EP group (or four small LPs per wave), no
// workgroup barriers.  Included by the kernels that run it (solve.hip, plan.hip).
//
// Problem (reference: minilp.cu:199-293).  For a group of G ranks with D replica
// slots each, n = G*D replica edges.  Edge j = (k, d) carries the normalised
// token count w_j of rank k's d-th replicated expert set; a copy lives on the
// rank i with r2o[i][d] == k.  Variables: x_o[j] (share kept on k), x_r[j] (share
// sent to the copy), slack s_i per rank, the maximum load t and a Big-M
// artificial x_M.  Constraints: per rank i,
//     sum_{j on i} w_j x_o[j] + sum_{j copied to i} w_j x_r[j] + s_i - t + m_i x_M = b_i,
// per edge x_o[j] + x_r[j] - x_M = 1; minimise t + 1000 x_M.  m makes x = 1 feasible.
//
// Method (reference: minilp.cu:331-400): a fixed number of primal affine-scaling
// steps x <- x (1 - alpha d), d = x (c - A^T w), (A X^2 A^T) w = A X^2 c,
// alpha = 0.999 / d_max, then a feasibility test; same iteration count, step
// rule, thresholds and fallback as the reference.
//
// What is different is how (A X^2 A^T) w = A X^2 c is solved.  The reference
// forms the dense (G+n) x (G+n) matrix and calls a block Cholesky.  A has two
// structural non-zeros per edge column, so eliminating the n edge rows by hand
// (they are diagonal plus a rank-one term) leaves a G x G system
//     S = sum_j lambda_j (e_k - e_i)(e_k - e_i)^T + diag(s^2) + t^2 11^T + kappa v v^T
// -- a weighted graph Laplacian of the replica topology plus a diagonal and two
// rank-one terms -- with right-hand side -t^2 1 + 1000 kappa v, where
//     E_j = x_o^2 + x_r^2, u_j = 1/E_j, lambda_j = w_j^2 x_o^2 x_r^2 u_j,
//     kappa = x_M^2 / (1 + x_M^2 sum u), q = B u, v = m + q.
// Lane i of the wave owns rank i, lane j owns edge j (two edges per lane beyond 64).  S is
// assembled and [S | rhs] reduced by Gauss-Jordan elimination in fp64: the system is tiny,
// and fp64 here removes the 1e-4..1e-3 rounding scatter a 32-bit factorisation shows on
// nearly balanced loads.  Everything else is fp32.  For the elimination, lane i holds row i
// of S; pivots are broadcast with v_readlane, the pivot row's entries with v_readlane or
// through LDS, and every lane updates what it holds.
//
// This form serves four LPs per wave, groups of 33 to 64 ranks and groups with more than 64
// edges or 8 slots per rank; one LP per wave with up to 32 ranks takes the form of
// solve_spread.h, in which a rank's row and edges are spread over its 8, 4 or 2 lanes.
#pragma once
#include "common.h"
#include "reciprocal.h"

namespace lplb {

typedef float f32x4 __attribute__((ext_vector_type(4)));
struct SolveArgs {
  const int32_t *workload;   // [n_inst][n_experts]
  float *gw_out;             // [n_inst][n_experts] or null
  const int32_t *r2o;        // [G][D]
  const int32_t *phy2log;    // [n_group][G][P]
  int32_t *avail;
  float *result;             // [n_inst][n_group][G][D]
  int n_group, G, D, C, n_fixed, n_experts, step_rule, n_steps, n_units;
  int staged_stride;   // floats of LDS per LP for its counts, 0 = read them from global memory
  bool counts_by_caller;   // a.workload is not read: the caller puts the counts into staged_counts (as int32) before its
                           // `counts_have_come` returns
  unsigned long long *tagged_result;  // or null: a copy of a.result for other workgroups of the same launch,
  uint32_t launch;                    // each value written through to memory as (share_tag(launch) << 32) | its bits
  int tagged_copies, tagged_stride;   // ... tagged_copies times, tagged_stride words apart (the pollers spread over the copies)
                                      // (the caller writes share_tag(launch) + 1 for "no result: use the neutral fallback")
  float *shares_in_lds;      // or null: another copy of a.result, for the caller's workgroup
  long long *clocks;         // debug builds: wall-clock stamps of wave 0, lane 0 (else null)
};

// Stamps of the first wave (debug builds only).
#define LPLB_STAMP(k) LPLB_STAMP_AT(blockIdx.x == 0 ? a.clocks : nullptr, k)

template <int CTRL> __device__ inline float dpp(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
constexpr int kQuadSwap1 = 0xB1;    // quad_perm [1,0,3,2]
constexpr int kQuadSwap2 = 0x4E;    // quad_perm [2,3,0,1]
constexpr int kHalfMirror = 0x141;  // reverse within 8 lanes
constexpr int kRowMirror = 0x140;   // reverse within 16 lanes

// Sum of lanes [0, W) (W = 8, 16, 32 or 64; lanes beyond W may hold anything for
// W < 64 as long as whole 16-lane rows are either inside or outside).  The result
// is wave-uniform.
template <int W> __device__ inline float reduce_sum(float v) {
  v += dpp<kQuadSwap1>(v);
  v += dpp<kQuadSwap2>(v);
  v += dpp<kHalfMirror>(v);
  if (W <= 8)
    return readlane(v, 0);
  v += dpp<kRowMirror>(v);
  if (W <= 16)
    return readlane(v, 0);
  if (W <= 32)
    return readlane(v, 0) + readlane(v, 16);
  return (readlane(v, 0) + readlane(v, 16)) + (readlane(v, 32) + readlane(v, 48));
}
// Max with fmaxf semantics (NaN ignored unless everything is NaN).
template <int W> __device__ inline float reduce_max(float v) {
  v = fmaxf(v, dpp<kQuadSwap1>(v));
  v = fmaxf(v, dpp<kQuadSwap2>(v));
  v = fmaxf(v, dpp<kHalfMirror>(v));
  if (W <= 8)
    return readlane(v, 0);
  v = fmaxf(v, dpp<kRowMirror>(v));
  if (W <= 16)
    return readlane(v, 0);
  if (W <= 32)
    return fmaxf(readlane(v, 0), readlane(v, 16));
  return fmaxf(fmaxf(readlane(v, 0), readlane(v, 16)), fmaxf(readlane(v, 32), readlane(v, 48)));
}

// ---- one LP per wave (ROWS == 1) or one LP per 16-lane DPP row (ROWS == 4) ----
// With ROWS == 4 a lane's position inside its row plays the part of the lane id,
// broadcasts are row-local DPP moves (row_newbcast) and reductions stop at the
// row, so four independent LPs share the wave's instruction stream.
constexpr int kRowLanes = 16;
template <int ROWS> struct Layout {
  static constexpr int kWidth = ROWS == 1 ? kWave : kRowLanes;   // lanes that serve one LP
};

template <int LANE> __device__ inline float row_bcast(float v) { return dpp<0x150 + LANE>(v); }
template <int LANE> __device__ inline double row_bcast(double v) {
  int2 p = __builtin_bit_cast(int2, v);
  p.x = __builtin_amdgcn_update_dpp(0, p.x, 0x150 + LANE, 0xF, 0xF, false);
  p.y = __builtin_amdgcn_update_dpp(0, p.y, 0x150 + LANE, 0xF, 0xF, false);
  return __builtin_bit_cast(double, p);
}
// Value of `v` in lane LANE of this LP's lanes.
template <int ROWS, int LANE, typename T> __device__ inline T lp_bcast(T v) {
  if constexpr (ROWS == 1)
    return readlane(v, LANE);
  else
    return row_bcast<LANE>(v);
}
// `old` with lane LANE of this LP's lanes replaced by `v`, a value that is the same in
// all of them.  One LP per wave: v sits in scalar registers and v_writelane puts it into
// the lane (a select would first have to copy it into a vector register).
template <int ROWS, int LANE> __device__ inline double lp_set_lane(double old, double v, int lane) {
  if constexpr (ROWS == 1) {
    int2 o = __builtin_bit_cast(int2, old);
    const int2 n = __builtin_bit_cast(int2, v);
    const int lo = __builtin_amdgcn_readfirstlane(n.x), hi = __builtin_amdgcn_readfirstlane(n.y);
    asm("v_writelane_b32 %0, %1, %2" : "+v"(o.x) : "s"(lo), "n"(LANE));
    asm("v_writelane_b32 %0, %1, %2" : "+v"(o.y) : "s"(hi), "n"(LANE));
    return __builtin_bit_cast(double, o);
  } else {
    return lane == LANE ? v : old;
  }
}
// `old` with lane LANE of this LP's lanes made zero.  One LP per wave: only the high word is
// cleared (one v_writelane instead of two, and it sits in the chain from one pivot to the next).
// What is left is a denormal below 2^-1022 (or zero where denormals are flushed): as a multiplier
// in S[k] -= f * x it changes no entry that is not itself that small.
template <int ROWS, int LANE> __device__ inline double lp_clear_lane(double old, int lane) {
  if constexpr (ROWS == 1) {
    int2 o = __builtin_bit_cast(int2, old);
    asm("v_writelane_b32 %0, 0, %1" : "+v"(o.y) : "n"(LANE));
    return __builtin_bit_cast(double, o);
  } else {
    return lane == LANE ? 0.0 : old;
  }
}
// Reductions over the first W lanes of this LP (W <= 16 when ROWS == 4).
template <int ROWS, int W> __device__ inline float lp_sum(float v) {
  if constexpr (ROWS == 1) {
    return reduce_sum<W>(v);
  } else {
    v += dpp<kQuadSwap1>(v);
    v += dpp<kQuadSwap2>(v);
    v += dpp<kHalfMirror>(v);
    if (W > 8)
      v += dpp<kRowMirror>(v);
    return row_bcast<0>(v);
  }
}
template <int ROWS, int W> __device__ inline float lp_max(float v) {
  if constexpr (ROWS == 1) {
    return reduce_max<W>(v);
  } else {
    v = fmaxf(v, dpp<kQuadSwap1>(v));
    v = fmaxf(v, dpp<kQuadSwap2>(v));
    v = fmaxf(v, dpp<kHalfMirror>(v));
    if (W > 8)
      v = fmaxf(v, dpp<kRowMirror>(v));
    return row_bcast<0>(v);
  }
}


// What says that a share is there, from the launch that found `launch` in its block's counter (formed where it is stored: that
// counter may still be on its way when the LP begins).
__host__ __device__ inline uint32_t share_tag(uint32_t launch) { return ((launch + 1u) << 2) | 1u; }
// Stores a share, and if asked also the copies other workgroups of the running kernel poll (the high word says
// "valid, from this launch", so value and flag arrive in one 8-byte store) and the one in the caller's LDS.
__device__ inline void store_share(const SolveArgs &a, int64_t i, float v) {
  if (a.tagged_result)
    for (int k = 0; k < a.tagged_copies; ++k)
      __hip_atomic_store(a.tagged_result + (int64_t)k * a.tagged_stride + i,
                         ((unsigned long long)share_tag(a.launch) << 32) | __builtin_bit_cast(uint32_t, v), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  if (a.shares_in_lds)
    a.shares_in_lds[i] = v;
  a.result[i] = v;
}

// With one LP per wave a lane's row of S is put together in LDS instead of registers: floats the
// caller provides per wave (row i at i * (GM + 4), so that 16-byte reads of different lanes'
// rows fall into different banks; then GM floats for a broadcast copy of v).
constexpr int assembly_tile_floats(int gm, int rows) { return rows == 1 ? gm * (gm + 4) + gm : 4; }

// GM, DM: register-array sizes (group size and replica slots rounded up).
// EXACT: the group is exactly GM x DM, so every loop bound is a compile-time
// constant; otherwise rows and columns G..GM-1 of the normal-equation system are
// padded with the identity, which keeps the factorisation free of branches.
// ROWS: LPs per wave (1, or 4 when GM <= 16 and GM * DM <= 16).
// EPL: replica edges per lane, 1 or 2 (ROWS == 1 only).  Edge j lives in lane j % 64, place j / 64;
// groups with 65..128 edges take two places.  Everything per rank (the G x G system included) is
// the same either way; what is per edge is done once per place, and a value of edge j is fetched
// from place j / 64 of lane j % 64.
//
// Called by all 64 lanes of a wave; waves share nothing and never synchronise.
//   first_unit     LP (instance * n_group + group) of the wave's first row
//   staged_counts  LDS, ROWS * a.staged_stride floats (unused if the stride is 0; STAGED: it is not)
//   rep_of_edge    LDS, EPL * kWave ints
//   pivot_rows     LDS, 2 * kWave doubles of this wave, 16-byte aligned
//   tile           LDS, assembly_tile_floats(GM, ROWS) floats of this wave, 16-byte aligned
// Returns how many of the wave's LPs passed the feasibility test (same value in
// every lane); the caller adds it to a.avail.
template <int GM, int DM, bool EXACT, int ROWS, int EPL, bool STAGED>
__device__ inline int solve_lp(const SolveArgs &a, int first_unit, float *staged_counts_of_wave,
                               int *rep_of_edge, double *pivot_rows, float *tile) {
  constexpr int WL = Layout<ROWS>::kWidth;   // lanes of one LP
  static_assert(ROWS == 1 || (ROWS == 4 && GM <= kRowLanes && GM * DM <= kRowLanes), "an LP must fit its lanes");
  static_assert(EPL == 1 || (EPL == 2 && ROWS == 1), "two edges per lane only with one LP per wave");
  static_assert(GM % 8 == 0, "pivot rows are read from LDS eight columns at a time");
  constexpr int T = WL / GM;         // lanes that share the work of one rank's b_i
  constexpr int NE = 2 * DM;         // replica edges that touch one rank
  constexpr int KB = ROWS == 1 ? 4 : 16;   // fixed-expert counts a lane prefetches for b_i
  constexpr int WR = GM;             // lanes that can hold a rank
  constexpr int WE = (GM * DM < WL && EPL == 1) ? (GM * DM < 8 ? 8 : GM * DM) : WL;  // ... an edge
  constexpr int KG = ROWS == 1 ? 4 : 16;   // normalised counts a lane prefetches for the output (and loop unrolling)
  const int wave_lane = threadIdx.x % kWave;

  // `lane` is the position inside this LP's lanes, `lane0` the wave lane where they start.
  const int lane = wave_lane % WL, lane0 = wave_lane - lane;
  const int G = EXACT ? GM : a.G, D = EXACT ? DM : a.D;
  const int C = a.C, n = G * D, n_fixed = a.n_fixed;
  const int L = D * C + n_fixed, P = L + D * C;
  // A wave whose last rows have no LP left repeats the last one and discards the result.
  const int n_units = a.n_units;
  const int unit_raw = first_unit + wave_lane / WL;
  const bool unit_on = unit_raw < n_units;
  const int unit = unit_on ? unit_raw : n_units - 1;
  const int grp = unit % a.n_group, inst = unit / a.n_group;
  float *staged_counts = staged_counts_of_wave + wave_lane / WL * a.staged_stride;
  auto gather = [&](auto v, int src) { return bpermute(v, lane0 + src); };
  // value of edge `e` (v[place] of the lane that holds it)
  auto gather_edge = [&](const auto (&v)[EPL], int e) {
    if constexpr (EPL == 1) {
      return bpermute(v[0], lane0 + e);
    } else {
      const auto lo = bpermute(v[0], e & (kWave - 1)), hi = bpermute(v[1], e & (kWave - 1));
      return e < kWave ? lo : hi;
    }
  };
  const int32_t *__restrict__ wl = a.workload + (int64_t)inst * a.n_experts;
  const int32_t *__restrict__ p2l = a.phy2log + (int64_t)grp * G * P;
  const bool is_rank = lane < G;
  bool is_edge[EPL];
  int ek[EPL], ed[EPL];   // original rank of my edge, its replica slot
#pragma unroll
  for (int p = 0; p < EPL; ++p) {
    const int j = lane + p * kWave;
    is_edge[p] = j < n;
    ek[p] = is_edge[p] ? j / D : 0;
    ed[p] = is_edge[p] ? j % D : 0;
  }
  // When they fit, the counts are staged in LDS as floats, so that the gathers
  // through phy2log do not need a second round trip to global memory.
  const bool staged = STAGED || a.staged_stride > 0;
  auto count_of = [&](int e) -> float {
    if (e < 0 || e >= a.n_experts)
      return 0.0f;
    return staged ? staged_counts[e] : (float)wl[e];
  };

  LPLB_STAMP(0);
  // ---- all global reads up front, as independent loads ----
  // (a) my edge's experts: raw count of the first, the rest in the loop below
  int e_first[EPL];
#pragma unroll
  for (int p = 0; p < EPL; ++p)
    e_first[p] = (is_edge[p] && C > 0) ? p2l[ek[p] * P + ed[p]] : -1;
  // (b) the experts of "my" rank that cannot move (T lanes share a rank)
  const int br = lane / T, bsub = lane % T;
  int fixed_e[KB];
#pragma unroll
  for (int u = 0; u < KB; ++u) {
    const int j = bsub + u * T;
    fixed_e[u] = (br < G && j < n_fixed) ? p2l[br * P + D * C + j] : -1;
  }
  // (c) topology row of my rank
  int r2o_row[DM];
#pragma unroll
  for (int d = 0; d < DM; ++d) {
    int k = (is_rank && d < D) ? a.r2o[lane * D + d] : 0;
    r2o_row[d] = k < 0 ? 0 : (k >= G ? G - 1 : k);
  }
  // (d) the counts: the maximum over all experts of all groups, minilp.cu:181-189, and
  // (e) this group's counts, for the normalised-count output at the end
  float wmax = 0.0f;
  float out_cnt[KG];
#pragma unroll KG
  for (int i = lane; i < a.n_experts; i += WL) {
    const float cnt = (float)wl[i];
    wmax = fmaxf(wmax, cnt);
    if (staged)
      staged_counts[i] = cnt;
  }
#pragma unroll
  for (int u = 0; u < KG; ++u) {
    const int i = lane + u * WL;
    out_cnt[u] = (a.gw_out && i < G * L) ? (float)wl[grp * G * L + i] : 0.0f;
  }
  __builtin_amdgcn_wave_barrier();   // staged counts are visible to the whole wave
  float w_first[EPL];
#pragma unroll
  for (int p = 0; p < EPL; ++p)
    w_first[p] = count_of(e_first[p]);
  float fixed_cnt[KB];
#pragma unroll
  for (int u = 0; u < KB; ++u)
    fixed_cnt[u] = count_of(fixed_e[u]);
  wmax = lp_max<ROWS, WL>(wmax);

  LPLB_STAMP(1);
  // ---- per-edge constants (lane j < n): w_j, minilp.cu:203-221 ----
  float w[EPL];
  int erep[EPL];
#pragma unroll
  for (int p = 0; p < EPL; ++p) {
    w[p] = is_edge[p] && C > 0 ? w_first[p] / wmax : 0.0f;
    if (is_edge[p])
      for (int c = 1; c < C; ++c)
        w[p] += count_of(p2l[ek[p] * P + c * D + ed[p]]) / wmax;
    // rank that holds the copy of each edge: invert r2o through LDS
    rep_of_edge[lane0 + lane + p * kWave] = ek[p];
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int d = 0; d < DM; ++d)
    if (is_rank && d < D)
      rep_of_edge[lane0 + r2o_row[d] * D + d] = lane;
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int p = 0; p < EPL; ++p)
    erep[p] = rep_of_edge[lane0 + lane + p * kWave];

  LPLB_STAMP(2);
  // ---- per-rank constants (lane i < G) ----
  // Edge e < DM: my own edge (i, e), other end = where its copy lives.
  // Edge DM + d: the edge copied into my slot d, other end = its original rank.
  // An inactive edge points at myself, which makes all its terms vanish.
  int src[NE], oth[NE];
  float w_e[NE];
  bool slot_on[DM];
#pragma unroll
  for (int d = 0; d < DM; ++d) {
    const bool on = is_rank && d < D;
    slot_on[d] = on;
    src[d] = on ? lane * D + d : 0;
    src[DM + d] = on ? r2o_row[d] * D + d : 0;
    // cross-lane reads stay outside lane-dependent conditions
    const int other = gather_edge(erep, src[d]);
    const float w_own = gather_edge(w, src[d]), w_copy = gather_edge(w, src[DM + d]);
    oth[d] = on ? other : lane;
    oth[DM + d] = on ? r2o_row[d] : lane;
    w_e[d] = on ? w_own : 0.0f;
    w_e[DM + d] = on ? w_copy : 0.0f;
  }
  // Selectors for assembling my row of S: 1 on my own column, -1 on the column
  // of each edge's other end.
  // (One LP per wave: the selectors alone would be hundreds of registers; there the row is put
  // together in LDS instead, see below.)
  constexpr bool kTileAssembly = ROWS == 1;
  constexpr int GS = kTileAssembly ? 1 : GM;
  float mask[NE][GS], diag_mask[GS];
#pragma unroll
  for (int c = 0; c < GS; ++c) {
    diag_mask[c] = (lane == c) ? 1.0f : 0.0f;
#pragma unroll
    for (int e = 0; e < NE; ++e)
      mask[e][c] = (oth[e] == c) ? -1.0f : 0.0f;
  }
  const int own = lane < GM ? lane : GM - 1;
  float *my_tile_row = tile + own * (GM + 4);
  float *v_copy = tile + GM * (GM + 4);

  LPLB_STAMP(3);
  // b_i = -(load of the experts that cannot move), minilp.cu:223-234
  float part = 0.0f;
#pragma unroll
  for (int u = 0; u < KB; ++u)
    part += fixed_cnt[u] / wmax;
  // ranks with more fixed experts than were prefetched: the rest in batches of
  // independent loads (added in the same order as one by one)
  if (br < G)
    for (int j0 = bsub + KB * T; j0 < n_fixed; j0 += KB * T) {
      int more_e[KB];
#pragma unroll
      for (int u = 0; u < KB; ++u)
        more_e[u] = j0 + u * T < n_fixed ? p2l[br * P + D * C + j0 + u * T] : -1;
#pragma unroll
      for (int u = 0; u < KB; ++u)
        if (j0 + u * T < n_fixed)
          part += count_of(more_e[u]) / wmax;
    }
  if (T >= 2) part += dpp<kQuadSwap1>(part);
  if (T >= 4) part += dpp<kQuadSwap2>(part);
  if (T >= 8) part += dpp<kHalfMirror>(part);
  const float part_of_rank = gather(part, (lane * T) & (WL - 1));
  const float b = is_rank ? -part_of_rank : 0.0f;
  // Big-M column, minilp.cu:275-281: b_i minus the other entries of row i.
  float m = b;
#pragma unroll
  for (int e = 0; e < NE; ++e)
    m -= w_e[e];
  m = (m - 1.0f) + 1.0f;
  if (!is_rank)
    m = 0.0f;

  LPLB_STAMP(4);
  // ---- affine scaling ----
  float xo[EPL], xr[EPL], xs = 1.0f, xt = 1.0f, xM = 1.0f;
#pragma unroll
  for (int p = 0; p < EPL; ++p)
    xo[p] = xr[p] = 1.0f;
  float d_max = 0.0f;
  const int NV = 2 * n + G + 2;
  const int win_lo = a.step_rule == LPLB_STEP_REFERENCE_WINDOW ? (NV > 32 ? NV - 32 : 0) : 0;
  const bool with_zero = a.step_rule != LPLB_STEP_REFERENCE_WINDOW || NV < 32;
  bool win_o[EPL], win_r[EPL];
#pragma unroll
  for (int p = 0; p < EPL; ++p) {
    win_o[p] = is_edge[p] && lane + p * kWave >= win_lo;
    win_r[p] = is_edge[p] && n + lane + p * kWave >= win_lo;
  }
  const bool win_s = is_rank && 2 * n + lane >= win_lo;
  const double row_on = is_rank ? 1.0 : 0.0;

  for (int step = 0; step < a.n_steps; ++step) {
    const float ss = xs * xs, st = xt * xt, sM = xM * xM;
    float so[EPL], sr[EPL], u[EPL], ao[EPL], ar[EPL], lam[EPL];
    float u_all = 0.0f;
#pragma unroll
    for (int p = 0; p < EPL; ++p) {
      so[p] = xo[p] * xo[p];
      sr[p] = xr[p] * xr[p];
      u[p] = is_edge[p] ? __builtin_amdgcn_rcpf(so[p] + sr[p]) : 0.0f;
      const float wu = w[p] * u[p];
      ao[p] = wu * so[p];
      ar[p] = wu * sr[p];
      lam[p] = w[p] * ao[p] * sr[p];             // w^2 so sr / (so + sr)
      u_all = p == 0 ? u[p] : u_all + u[p];
    }
    const float sigma = lp_sum<ROWS, WE>(u_all);
    const float kappa = sM * __builtin_amdgcn_rcpf(1.0f + sM * sigma);

    float q = 0.0f, lam_e[NE], lam_sum = ss;
#pragma unroll
    for (int d = 0; d < DM; ++d) {
      const float q_own = gather_edge(ao, src[d]), q_copy = gather_edge(ar, src[DM + d]);
      const float l_own = gather_edge(lam, src[d]), l_copy = gather_edge(lam, src[DM + d]);
      // an inactive slot or a self-loop (oth == lane) contributes nothing to S;
      // an inactive slot contributes nothing to q either
      q += slot_on[d] ? q_own + q_copy : 0.0f;
      lam_e[d] = (oth[d] == lane) ? 0.0f : l_own;
      lam_e[DM + d] = (oth[DM + d] == lane) ? 0.0f : l_copy;
      lam_sum += lam_e[d] + lam_e[DM + d];
    }
    const float v = is_rank ? m + q : 0.0f;

    if (step == 0) LPLB_STAMP(5);
    // Row `lane` of S and its right-hand side, fp64.
    double S[GM];
    const double dst = (double)st, dkv = (double)kappa * (double)v;
    const float st_col = is_rank ? st : 0.0f;
    if constexpr (kTileAssembly) {
      // The Laplacian part of my row: zero it, subtract every edge's weight at the column of
      // its other end, add the diagonal (LDS float adds, no return value: they queue up in
      // program order, so each entry is the same sum, in the same order, as with selectors),
      // read it back.  A lane touches only its own row.  v of every rank comes back from a
      // copy in LDS, four ranks per read from a wave-uniform address.
      const f32x4 zero{0.0f, 0.0f, 0.0f, 0.0f};
      if (lane < GM) {
#pragma unroll
        for (int c4 = 0; c4 < GM / 4; ++c4)
          reinterpret_cast<f32x4 *>(my_tile_row)[c4] = zero;
        v_copy[own] = v;
#pragma unroll
        for (int e = 0; e < NE; ++e)
          __hip_atomic_fetch_add(my_tile_row + oth[e], -lam_e[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        __hip_atomic_fetch_add(my_tile_row + own, lam_sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      static_for<GM / 4>([&](auto c4c) {
        constexpr int c4 = decltype(c4c)::value;
        const f32x4 t4 = reinterpret_cast<const f32x4 *>(my_tile_row)[c4];
        const f32x4 v4 = reinterpret_cast<const f32x4 *>(v_copy)[c4];
        const float t[4] = {t4.x, t4.y, t4.z, t4.w}, vc[4] = {v4.x, v4.y, v4.z, v4.w};
        static_for<4>([&](auto uu) {
          constexpr int u = decltype(uu)::value, c = 4 * c4 + u;
          const double base = EXACT ? dst : (double)lp_bcast<ROWS, c>(st_col) * row_on;
          S[c] = __builtin_fma(dkv, (double)vc[u], base) + (double)t[u];
        });
      });
    } else {
      static_for<GM>([&](auto cc) {
        constexpr int c = decltype(cc)::value;
        float t = diag_mask[c] * lam_sum;
#pragma unroll
        for (int e = 0; e < NE; ++e)
          t = __builtin_fmaf(mask[e][c], lam_e[e], t);
        const double base = EXACT ? dst : (double)lp_bcast<ROWS, c>(st_col) * row_on;
        S[c] = __builtin_fma(dkv, (double)lp_bcast<ROWS, c>(v), base) + (double)t;
      });
    }
    double rhs = (1000.0 * dkv - dst) * (EXACT ? 1.0 : row_on);

    if (step == 0) LPLB_STAMP(6);
    // Gauss-Jordan elimination of [S | rhs] by columns: lane i owns row i, column c
    // is cleared in every other row at once, so no triangular solves (and no
    // transposed factor) are needed afterwards.  Row c's entries are read from lane
    // c, whose own multiple f is zero.  S is symmetric positive definite: no pivoting.
    // The only serial chain is pivot -> reciprocal -> f -> entry (c+1, c+1) -> next
    // pivot; it is written out in that order, with the rest of column step c (which
    // nothing waits for) placed between the links of the next reciprocal, because
    // the compiler keeps the order it is given here.  (Computing the next pivot one step
    // ahead from three more broadcasts, in uniform arithmetic, gives bit-identical results
    // and takes the vector update out of the chain, but costs 9 instructions per pivot and
    // was slower at 8 ranks.)
    // A lane's own multiple must be zero.  Rather than selecting on the chain (f is the
    // link between reciprocal and update), the lane's diagonal entry is cleared as soon
    // as it has been read as the pivot, one step ahead.
    float y;
    double my_pivot = 1.0;
    double pivot = lp_bcast<ROWS, 0>(S[0]);
    double rinv = rcp_f64(pivot);
    // One LP per wave: the entries of pivot row c that the other rows need, S[c][c2] for
    // c2 > c, are not fetched from lane c one by one (two v_readlane each).  The part of S
    // that is still being eliminated stays symmetric (up to rounding), so they are also
    // column c as it is spread over the lanes, S[c2][c] in lane c2: one LDS write of that
    // register puts the whole row into LDS, and reads from a wave-uniform address hand two
    // entries at a time to every lane.  LDS instructions do not take the vector ALU's issue
    // slots, which are what bounds a lone wave.  Column c + 1 is final right after the first
    // update of step c; it is written then, so the round trip through LDS overlaps the rest
    // of step c and the reciprocal of the next pivot and is not part of the serial chain.
    // Two buffers take turns, so a step's reads need not all be issued before the next write.
    // (Four LPs per wave, each 16-lane row reading its own LP's column: 16384 LPs 30.9 -> 27.6 us.)
    constexpr bool kRowFromLds = ROWS == 4 || GM >= 16;
    constexpr int kChunk = 8;                       // columns per batch of LDS reads (GM is a multiple)
    constexpr int kChunks = GM / kChunk;
    constexpr int kBodySets = kChunks > 2 ? 2 : 1;  // chunks after a step's first are fetched one chunk ahead
    // chunk q of the row in buffer `parity`: columns 8 q .. 8 q + 7, four 16-byte reads
    auto load_chunk = [&](int parity, int q, double (&buf)[kChunk]) {
      const double2 *src = reinterpret_cast<const double2 *>(pivot_rows + parity * kWave + lane0 + q * kChunk);
#pragma unroll
      for (int j = 0; j < kChunk / 2; ++j) {
        const double2 both = src[j];
        buf[2 * j] = both.x;
        buf[2 * j + 1] = both.y;
      }
      // The reads stay where they are written, ahead of their use: left alone, the compiler
      // moves each one down to the instruction that needs it (fewer live registers) and the
      // wave then waits out every LDS round trip.
      __builtin_amdgcn_sched_barrier(0);
    };
    // The first chunk a step needs is fetched during the step before, right after the column
    // has been written (two sets of registers take turns).
    double head[2][kChunk];
    auto publish_column = [&](auto cc) {
      constexpr int c = decltype(cc)::value;
      if constexpr (kRowFromLds && c < GM) {
        pivot_rows[(c % 2) * kWave + lane0 + lane] = S[c];   // (every lane writes: no branch; lanes >= GM are never read)
        __builtin_amdgcn_wave_barrier();
        if constexpr (c + 1 < GM)
          load_chunk(c % 2, (c + 1) / kChunk, head[c % 2]);
      }
    };
    publish_column(std::integral_constant<int, 0>{});
    S[0] = lp_clear_lane<ROWS, 0>(S[0], lane);
    static_for<GM>([&](auto cc) {
      constexpr int c = decltype(cc)::value;
      constexpr int q0 = (c + 1) / kChunk;          // chunk of column c + 1
      double body[kBodySets][kChunk];
      // S[c2] -= f * (row c)[c2]
      auto clear = [&](auto c2c, double f) {
        constexpr int c2 = decltype(c2c)::value;
        if constexpr (c2 < GM) {
          if constexpr (!kRowFromLds) {
            S[c2] = __builtin_fma(-f, lp_bcast<ROWS, c>(S[c2]), S[c2]);
          } else if constexpr (c2 / kChunk == q0) {
            S[c2] = __builtin_fma(-f, head[c % 2][c2 % kChunk], S[c2]);
          } else {
            // entering a new chunk: fetch the one after it, and keep the compiler from pulling
            // every later fetch up here (the rows would not fit the registers)
            if constexpr (c2 % kChunk == 0 && kBodySets == 2) {
              __builtin_amdgcn_sched_barrier(0);
              if constexpr (c2 / kChunk + 1 < kChunks)
                load_chunk(c % 2, c2 / kChunk + 1, body[(c2 / kChunk + 1) % kBodySets]);
            }
            S[c2] = __builtin_fma(-f, body[(c2 / kChunk) % kBodySets][c2 % kChunk], S[c2]);
          }
        }
      };
      my_pivot = lp_set_lane<ROWS, c>(my_pivot, pivot, lane);
      const double f = S[c] * rinv;   // multiple of row c to subtract from my row (0 in lane c)
      double next_pivot = 1.0, estimate = 1.0, error = 0.0;
      if constexpr (kRowFromLds && q0 + 1 < kChunks)
        load_chunk(c % 2, q0 + 1, body[(q0 + 1) % kBodySets]);
      clear(std::integral_constant<int, c + 1>{}, f);
      publish_column(std::integral_constant<int, c + 1>{});
      if constexpr (c + 1 < GM) {
        next_pivot = lp_bcast<ROWS, c + 1>(S[c + 1]);
        estimate = __builtin_amdgcn_rcp(next_pivot);
        S[c + 1] = lp_clear_lane<ROWS, c + 1>(S[c + 1], lane);
      }
      rhs = __builtin_fma(-f, lp_bcast<ROWS, c>(rhs), rhs);
      clear(std::integral_constant<int, c + 2>{}, f);
      if constexpr (c + 1 < GM)
        error = __builtin_fma(-next_pivot, estimate, 1.0);
      clear(std::integral_constant<int, c + 3>{}, f);
      clear(std::integral_constant<int, c + 4>{}, f);
      if constexpr (c + 1 < GM) {
        rinv = __builtin_fma(error, estimate, estimate);   // = rcp_f64(next_pivot)
        pivot = next_pivot;
      }
      static_for<(GM > c + 5 ? GM - c - 5 : 0)>([&](auto kk) {
        constexpr int k = decltype(kk)::value;
        // From 32 ranks on a row's broadcasts would fill the scalar registers if the
        // compiler hoisted them all; fence them off in groups of eight columns.
        if constexpr (!kRowFromLds && GM >= 32 && k % 8 == 0)
          __builtin_amdgcn_sched_barrier(0);
        clear(std::integral_constant<int, c + 5 + k>{}, f);
      });
    });
    if (step == 0) LPLB_STAMP(7);
    y = is_rank ? (float)(rhs * rcp_f64(my_pivot)) : 0.0f;

    if (step == 0) LPLB_STAMP(8);
    // r = A^T w and the direction d = x (c - r); the edge part of w is
    // z = u (h - kappa u.h + kappa (m.y - 1000)), h = -B^T y.
    float yk[EPL], yrep[EPL], hp[EPL];
    float uhp_all = 0.0f;
#pragma unroll
    for (int p = 0; p < EPL; ++p) {
      yk[p] = gather(y, ek[p]);
      yrep[p] = gather(y, erep[p]);
      hp[p] = -w[p] * (so[p] * yk[p] + sr[p] * yrep[p]);
      uhp_all = p == 0 ? u[p] * hp[p] : uhp_all + u[p] * hp[p];
    }
    const float my = lp_sum<ROWS, WR>(m * y);
    const float sumy = lp_sum<ROWS, WR>(y);
    const float uh = lp_sum<ROWS, WE>(uhp_all);
    const float shift = kappa * (my - 1000.0f) - kappa * uh;
    const float sumz = uh + shift * sigma;       // = sum of z over the edges
    float d_o[EPL], d_r[EPL];
#pragma unroll
    for (int p = 0; p < EPL; ++p) {
      const float z = u[p] * (hp[p] + shift);
      d_o[p] = -xo[p] * (w[p] * yk[p] + z);
      d_r[p] = -xr[p] * (w[p] * yrep[p] + z);
    }
    const float d_s = -xs * y;
    const float d_t = xt * (1.0f + sumy);
    const float d_M = xM * (1000.0f - (my - sumz));

    if (step == 0) LPLB_STAMP(9);
    // Step length, minilp.cu:354-362.  NaN marks "not in the window".
    float cand = __builtin_nanf("");
#pragma unroll
    for (int p = 0; p < EPL; ++p) {
      cand = win_o[p] ? fmaxf(cand, d_o[p]) : cand;
      cand = win_r[p] ? fmaxf(cand, d_r[p]) : cand;
    }
    cand = win_s ? fmaxf(cand, d_s) : cand;
    cand = lane == 0 ? fmaxf(fmaxf(cand, d_t), d_M) : cand;
    d_max = lp_max<ROWS, WE>(cand);
    if (with_zero)
      d_max = fmaxf(d_max, 0.0f);
    const float alpha = (float)(0.999 / (double)d_max);
#pragma unroll
    for (int p = 0; p < EPL; ++p) {
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
  float res = 0.0f;
  {
    float row = xs - xt + m * xM - b;
#pragma unroll
    for (int d = 0; d < DM; ++d) {
      const float a_o = gather_edge(xo, src[d]), a_r = gather_edge(xr, src[DM + d]);
      row += w_e[d] * a_o + w_e[DM + d] * a_r;
    }
    if (is_rank)
      res = fmaxf(res, fabsf(row));
#pragma unroll
    for (int p = 0; p < EPL; ++p)
      if (is_edge[p])
        res = fmaxf(res, fabsf(xo[p] + xr[p] - xM - 1.0f));
    res = lp_max<ROWS, WE>(res);
  }
  const bool ok = (double)d_max < 0.1 && 0.0 <= (double)xM && (double)xM < 1e-4 &&
                  (double)res < 0.05;
  const int n_ok = __popcll(__ballot(lane == 0 && ok && unit_on));
#pragma unroll
  for (int p = 0; p < EPL; ++p)
    if (is_edge[p] && unit_on)
      a.result[(int64_t)unit * n + lane + p * kWave] = ok ? xo[p] : 0.5f;
  // Normalised counts of this group, for the caller.
  if (a.gw_out && unit_on) {
    float *gw = a.gw_out + (int64_t)inst * a.n_experts + grp * G * L;
#pragma unroll
    for (int u = 0; u < KG; ++u)
      if (lane + u * WL < G * L)
        gw[lane + u * WL] = out_cnt[u] / wmax;
    for (int i = lane + KG * WL; i < G * L; i += WL)
      gw[i] = count_of(grp * G * L + i) / wmax;
  }
  LPLB_STAMP(12);
  return n_ok;
}

} // namespace lplb
