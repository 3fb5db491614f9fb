// The whole plan of a batch as one kernel launch: device code and the launch of one variant.
// plan.hip holds the entry points, the admission of launches and the chain of kernels that serves
// everything else; plan_8.hip, plan_16.hip and plan_32.hip instantiate this file by group size.
//
// Every kernel boundary of the chain (histogram, scan, LP, redirect) costs 3-5 us on this GPU although the
// kernels have 1-8 us of work.  Here the LP workgroups (one per four LPs, first in the grid) and one
// workgroup per slice of the indices run side by side in a single grid:
//   slice workgroup: load the indices once (they stay in registers as 16-bit expert ids) -> histogram of the
//     slice in LDS -> publish it and the replicated sets' part of it -> bitmaps of the replicated sets, the other slices' counts
//     of those -> ordinals and hashes -> wait for the LP's shares -> choose original or replica, store;
//   LP workgroup: (own-histogram mode: collect the slices' histograms ->) solve -> publish the shares.
// A batch of up to 3584 indices that feeds the LP itself is one workgroup that does both (plan_in_one_workgroup):
// nothing is exchanged and nothing has to be resident beside it.
//
// What crosses workgroups are 8-byte words that say themselves whether they are complete, so that there is no
// counter of arrivals between a slice's counts and their readers and no acknowledgement to wait for:
// every word carries the launch's tag in its high half, and a launch overwrites the words of the launch before it
// (which has ended; so nothing has to be cleared either).
//   * A slice publishes its counts, two of 16 bits per word, as soon as its tokens are in the histogram (one barrier): those of
//     the replicated sets for every other slice, the whole histogram for the slices that add up the batch's totals.
//   * The totals are added up by up to 64 of the slices, each for eight words of every slice's histogram, and
//     published once more; the LP workgroups and the first slice collect those.  (Whole rows of 64 slices would be 64 KiB for an
//     LP workgroup, 1 us at the 68 bytes per ns that one CU reads past the caches with 16-byte loads.  As atomic
//     adds to shared totals they run into the rate of the atomic units, about 5 per ns over the whole GPU: 1.6 us
//     for 64 slices, 6.6 us for 256.)
// A word takes 0.3-0.5 us from one CU to another; what the hops cost beyond that is the waves' own instructions, so whatever
// the counts do not wait for (ordinals inside a slice, the LP's topology) is done while they are on their way.
// Per call, own histogram, before / after the counts went out ahead of the ordinals, units of 16-byte loads instead of sums by
// the whole workgroup, and one batch of arguments: [8192 x 8] 10.9 -> 10.2 us, [262144 x 8] 19.3 -> 17.7, counts supplied
// [8192 x 8] 8.1 -> 7.7; ahead of everything that looks at the mapping as well (clear_plan_tables): 9.3, 15.2 and 6.8.  What bounds
// it at [8192 x 8], from the first workgroup's start: 1.4 us until a slice's counts are out, 2.2 until the LP has the totals (0.4 the
// adding wave's addresses, 0.5 its loads, 0.5 its sums and stores, 0.8 until the LP has seen them), 3.7 of LP, 0.3-0.5 until its
// shares are seen, 0.5 until the last index is stored.
// Words are written and read with agent-scope atomics (plan_sync.h).
// The workgroups wait for each other, so the whole grid has to be resident: its size is bounded by what fits
// the GPU, and the host admits a launch only while the plans still executing leave room for it.
// Every wait is bounded all the same.  A wait that runs out is counted, the workgroup sends every token of its
// slice to the expert's original slot (which needs nothing from other workgroups), physical_counts is filled
// with -1 by the workgroup that writes them if it is among those, and the block of words is marked as unusable:
// plans that use it later send every token to the original slot and count one more failure each, until
// lplb_plan_sync_timeouts has reported the failures and cleared the block.
#pragma once
#include "map_kernel.h"
#include "plan_sync.h"
#include "scan.h"
#include "solve_spread.h"

namespace lplb {

constexpr int kPlanWaves = 8, kPlanThreads = kPlanWaves * kWave;
constexpr int kPlanLdsLimit = 160 * 1024 - 7680;   // dynamic LDS; the kernels have up to 4.1 KiB of static LDS besides
constexpr int kDefaultMaxPolls = 1 << 22;   // a few seconds of polling before a wait gives up
// LPs per LP workgroup: waves 0..3 of a workgroup sit on the CU's four SIMDs, and an LP
// wave is bound by instruction issue, so a fifth LP on the same CU would slow two of them
// down (8 LPs in one workgroup: 17.0 us per plan against 13.5 us).  Batches with more
// groups get more LP workgroups.
constexpr int kLpsPerWorkgroup = 4, kMaxLpWorkgroups = 8;
// Ahead of its use, an LP workgroup's dynamic LDS holds per LP wave the pivot rows and the assembly tile, then
// the counts.
template <int GM, int DM> constexpr size_t plan_lp_area_bytes() {
  return lp_pivot_doubles<GM, DM>() * sizeof(double) + lp_tile_floats<GM, DM>() * sizeof(float);
}

// The counts an LP works on, in LDS, with the zeros behind them and at least one word more, the last.
constexpr size_t counts_bytes(int n_logical) { return (size_t)(n_logical / 4 * 4 + 8) * sizeof(int32_t); }

// One block of these per stream that plans (kSyncSlots of them per device), offsets in ints:
//   [kGenAt] launches that have used the block; (value + 1) tags what a launch publishes;
//   [kPoisonAt] non-zero: a wait ran out in this block (see above); [kTimeoutsAt] waits that
//   ran out since the library was loaded (never cleared);
//   [kAvailAt + 2 p] (8 bytes) who has touched the caller's counter of feasible LPs in the launch with tag
//   parity p: bit k = LP k was feasible and has been (or is being) added, bit 32 = a wait ran out, so the
//   batch is not balanced as a whole and whoever set the bit took the LPs added so far back out; an LP
//   that finds bit 32 set does not add itself.  The reference's callers read "counter == number of
//   groups" as "this batch was balanced" (tests/test_solve.py:58, scripts/run_ep16_cube8p2e.py:61).
//   every launch clears the word of the other parity;
//   from kLpHereAt: one word per LP workgroup, with the launch's tag once it is resident;
//   from kSharesAt: the LP's shares as words (tag << 32) | float bits with tag = (launch tag << 2) | 1 (valid)
//   or 2 (there will be none); up to kShareCopies copies, kMaxShares words apart: polls of one line queue up in
//   memory, so slice s polls copy s % copies;
//   from kSetRowsAt: per slice set_words words with its tokens of the replicated sets, two sets per word;
//   from kHistRowsAt: per slice hist_words words with its histogram, two experts per word;
//   from kTotalsAt: one word per expert with the batch's tokens;
//   from kDoneAt: per slice and, behind them, per LP the number (PlanArgs::seq) of the last launch with a number in
//   which it has read all it reads of this block (the first slice's number is in the high half of [kAdvancedAt], with what
//   the last launch has set [kGenAt] to in the low half): before the block passes to another stream, whose launches the
//   device does not order behind this one, wait_for_last_user waits for these.
constexpr int kGenAt = 0, kPoisonAt = 1, kTimeoutsAt = 4, kAdvancedAt = 6, kAvailAt = 10;
constexpr unsigned long long kGaveUp = 1ull << 32;
constexpr int kMaxSlices = 256, kMaxPlanExperts = 1024, kMaxShares = 1024, kShareCopies = 8;
constexpr int kLpHereAt = 16, kSharesAt = kLpHereAt + 2 * kMaxLpWorkgroups, kMaxSetWords = kMaxPlanExperts / 2, kMaxHistWords = kMaxPlanExperts / 2;
constexpr int kSetRowsAt = kSharesAt + 2 * kMaxShares * kShareCopies;
constexpr int kHistRowsAt = kSetRowsAt + 2 * kMaxSlices * kMaxSetWords;
constexpr int kTotalsAt = kHistRowsAt + 2 * kMaxSlices * kMaxHistWords;
constexpr int kMaxLps = kLpsPerWorkgroup * kMaxLpWorkgroups;
constexpr int kDoneAt = kTotalsAt + 2 * kMaxPlanExperts;
constexpr int kDoneStride = 16;   // ints from word to word: stores to one 64-byte line queue up (16 in a line: plan [8192 x 8] 8.35 -> 8.6 us)
constexpr int kSlotInts = kDoneAt + (kMaxSlices + kMaxLps) * kDoneStride, kSyncSlots = 8;
constexpr int kLooseTimeoutsAt = kSyncSlots * kSlotInts, kSyncInts = kLooseTimeoutsAt + 16;   // behind the blocks: waits that ran out in a launch that uses none (scan_and_solve)
static_assert(kSharesAt % 16 == 0 && kSetRowsAt % 16 == 0 && kHistRowsAt % 16 == 0 && kTotalsAt % 16 == 0 && kSlotInts % 16 == 0, "rows start on 64-byte lines");

struct PlanArgs {
  const int64_t *idx;
  int64_t n, per;
  int n_slices, n_lp_workgroups;
  int n_share_copies;    // copies of the LP's shares: a power of two, at most kShareCopies
  int set_words;         // words per slice for its counts of the replicated sets: a power of two >= 8
  int unit_lanes_log2, unit_blocks, unit_block_bits;   // how what slices add up is cut into units: lanes of a slice, blocks of slices, bits that number those
  int hist_words;        // ... for its histogram: a multiple of 8 that holds n_logical counts
  int adders, adder_words;     // slices that add up the totals, for adder_words words (a power of two >= 8) of every histogram each
  int expected_slices;   // = n_slices unless a fault is injected
  int max_polls;
  const int32_t *o2r, *phy2log;
  int32_t *totals;   // [n_logical] this GPU's tokens per expert, out
  int64_t *out;
  int32_t *physical_counts;   // [n_ranks * P] tokens per physical expert, or null
  int32_t *avail;
  RedirectShape sh;
  int n_rep;
  uint32_t magic_L, magic_cd, magic_D, magic_G;   // fast_div_magic of L, C * D, D, G
  SolveArgs solve;   // result = the shares (o_weight); workload is replaced by the batch's own counts if local_counts
  int local_counts;
  int *sync;
  int *arrived_word;   // pinned host memory, or null: receives seq once every workgroup of the launch has arrived
  int seq;             // number of the launch among those of its block, or -1: captured, it has none
};

// plan.hip: admission and launch of one kernel (see there).  lds: dynamic LDS of the launch.
struct KernelFootprint {   // one per kernel variant
  std::atomic<int> regs{-1}, static_lds{0};
  std::atomic<uint64_t> much_lds_allowed{0};   // bit per device: the kernel may use more than 64 KiB of dynamic LDS
};
typedef void (*PlanKernel)(PlanArgs);
int launch_plan(PlanKernel kernel, KernelFootprint &footprint, bool waits_for_others, PlanArgs &a, size_t lds, hipStream_t s,
                bool *done);
// plan_8.hip, plan_16.hip, plan_32.hip: the variants for group sizes up to 8, 16, 32.
struct ScanSolveArgs;
int scan_and_solve_up_to_8(const ScanSolveArgs &a, hipStream_t s);
int scan_and_solve_up_to_16(const ScanSolveArgs &a, hipStream_t s);
int scan_and_solve_up_to_32(const ScanSolveArgs &a, hipStream_t s);
int launch_plan_up_to_8(PlanArgs &a, hipStream_t s, bool *done);
int launch_plan_up_to_16(PlanArgs &a, hipStream_t s, bool *done);
int launch_plan_up_to_32(PlanArgs &a, hipStream_t s, bool *done);

// A wait ran out: count it, switch the block of words off, and make sure the caller's counter of
// feasible LPs does not vouch for this batch (the first to give up takes back what the LPs have added).
__device__ inline void give_up(const PlanArgs &a, unsigned long long *avail_state) {
  agent_add(a.sync + kTimeoutsAt, 1);
  agent_store(a.sync + kPoisonAt, 1);
  const unsigned long long before = __hip_atomic_fetch_or(avail_state, kGaveUp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int added = __popcll(before & 0xffffffffull);
  if (!(before & kGaveUp) && added > 0)
    atomicAdd(a.avail, -added);
}

// Debug builds: stamps of the first and the last slice workgroup and of the first LP workgroup.
#define LPLB_PLAN_STAMP(k)                                                                     \
  LPLB_STAMP_AT(a.solve.clocks == nullptr ? nullptr                                            \
                : blockIdx.x == a.n_lp_workgroups ? a.solve.clocks + 64                        \
                : blockIdx.x == gridDim.x - 1 ? a.solve.clocks + 80                            \
                : blockIdx.x == 0 ? a.solve.clocks + 96 : nullptr, k)

// Debug builds: stamps of every slice workgroup (the buffer must hold 128 + 8 * slices).
#ifdef LPLB_PHASE_CLOCKS
#define LPLB_SLICE_STAMP(k)                                                                    \
  do {                                                                                         \
    if (a.solve.clocks && threadIdx.x == 0)                                                    \
      a.solve.clocks[128 + 8 * (blockIdx.x - a.n_lp_workgroups) + (k)] = wall_clock64();       \
  } while (0)
#else
#define LPLB_SLICE_STAMP(k) do { } while (0)
#endif

// ---- a slice's tables in LDS ----
// Per logical expert; all zeros: no slot and no set, as for masked and out-of-range tokens (entry n_logical).
// Sets are numbered from 1 in the order of minilp.cu:478-495, 0 is no set, so that what is empty is zero throughout.
struct __attribute__((aligned(8))) PlanRoute {
  int32_t not_original;   // complement of the original's physical slot
  int32_t set;
  __device__ int32_t original() const { return ~not_original; }
};
// One ranking slot per (wave, replicated set, chunk of 64 indices), K chunks per wave.
constexpr int64_t kLongestSlice = 16 * kPlanThreads;   // 16 chunks per wave
constexpr int kLongChunks = 8, kLongPasses = 8;        // of a long slice: chunks per wave and pass, passes
constexpr int kFewestLongSlices = 64;   // past 8192 indices
// Up to 8192 indices.  At 8 ranks, slices of 8192, us a plan in the other form / in passes, in 32, 64, 128 and 200 slices: counts supplied, 16 sets
// 12.3 / 11.7, 12.3 / 11.7, 12.9 / 12.2, 13.6 / 12.9, 32 sets 12.5 / 11.9, 12.7 / 11.9, 13.3 / 12.6, 14.6 / 14.2, 64 sets 13.7 / 12.4, 14.0 / 12.5, 15.1 / 13.9, 16.3 / 15.5;
// own counts, 64 sets 14.6 / 14.3, 14.9 / 14.5, 15.7 / 15.2, 16.5 / 15.6; 128 sets, as the chain in 31 slices and in passes in 32, 21.3 / 15.1.  Fewer slices
// would gain as much, down to 8 (counts supplied, 16 sets 12.1 / 11.5; own counts, 128 sets 20.9 / 14.9), less or nothing with two (32 ranks on their
// own counts 23.1 / 23.5); tests/test_gpu_parity.py names 31 slices with 80 sets as the chain's.
constexpr int kFewestSlicesInPasses = 32;
constexpr int64_t kLongestOfLongSlices = kLongPasses * kLongChunks * kPlanThreads;
// (K = 0: a long slice, without its records, which lie behind the rest)
constexpr int slice_record_bytes(int k) { return k > 0 ? rank_record_bytes_single(k) : 0; }
// (what a slice's workgroup keeps beside its tables: missing, block_sums)
constexpr int kBlockSums = 17, kSliceFlags = 2 + kBlockSums;
template <int K> static size_t plan_slice_lds_bytes(int n_logical, int n_rep) {
  return (size_t)(n_rep + 1) * sizeof(RepEntry) + (size_t)kPlanWaves * (n_rep + 1) * slice_record_bytes(K) +
         (size_t)(n_logical + 2) * sizeof(PlanRoute) + (size_t)(n_logical + 16 + kSliceFlags) * sizeof(int32_t) +
         (size_t)(3 + kPlanWaves) * n_rep * sizeof(int32_t);
}
// A long slice's row per (wave, replicated set), and one for tokens without a set: the bitmaps of the chunks that are ranked at once
// and the wave's tokens of the set so far (with 8 more bytes a row for the LDS banks).
constexpr int kRankChunks = 4, kRankRowBytes = kRankChunks * 8 + 8;
constexpr int kFewSets = 32;        // up to which slices of 16 chunks per wave that feed the LP have bitmaps of all chunks
constexpr int kLongMaxSets = 255;   // sets of a long slice are bytes
__host__ __device__ constexpr size_t long_slice_records_at(int n_logical, int n_rep) {
  return ((size_t)(n_rep + 1) * sizeof(RepEntry) + (size_t)(n_logical + 2) * sizeof(PlanRoute) + (size_t)(n_logical + 16 + kSliceFlags) * sizeof(int32_t) +
          (size_t)(3 + kPlanWaves) * n_rep * sizeof(int32_t) + 15) / 16 * 16;
}
inline size_t long_slice_lds_bytes(int n_logical, int n_rep, int hist_words) {
  return long_slice_records_at(n_logical, n_rep) + (size_t)kPlanWaves * ((n_rep + 1) * kRankRowBytes + 2 * hist_words * sizeof(int32_t)) +
         (size_t)(n_logical + 16) / 16 * 16;
}
// Slices past kLongestSlice of more than 8 ranks, or with more than kFewSets sets, ask for more than they use: 220 bytes a row, the sets padded to
// the next multiple of sixteen past their number, which is what their tables once took.  It is a rule of dispatch in the guise of a size: by it such
// batches are the chain where these would not fit a CU, or not on enough CUs at once, and those that are cut so hold that LDS for nothing.
// tests/test_gpu_parity.py names as the chain's, of these, 16 ranks with 32 sets in 256 slices, 32 ranks with 64 sets and 256 experts, and 8 ranks with
// 64 sets on their own counts (256 slices).  For 8 ranks with counts supplied or more than four groups no test does, and there the chain
// is the slower: [1048576 x 8] in 256 slices, 64 sets 41.5 against 34.3 us, 128 sets 45.7 against 36.5.  (Up to kFewSets sets, 32 of 8 ranks,
// [1048576 x 8] as the chain and so: 44.6 and 32.8 us, [524288 x 8] 27.0 and 20.4.)
inline size_t longest_slices_lds_bytes(int n_logical, int n_rep, int hist_words) {
  return long_slice_lds_bytes(n_logical, n_rep, hist_words) +
         (size_t)kPlanWaves * ((n_rep / 16 * 16 + 16) * 220 - (n_rep + 1) * kRankRowBytes);
}
struct SliceTables {
  RepEntry *reps;           // [R + 1] by set; of set 0: a test that never sends a token away
  PlanRoute *route;         // [n_logical + 1]
  unsigned char *records;   // [waves][R + 1][record bytes]
  int32_t *hist;            // [more than n_logical, a multiple of 16] the slice's histogram, then zeros; in the first slice at last the batch's
  int32_t *missing;         // [2] [0] some counts did not come, [1] some share will not come
  int32_t *block_sums;      // [kBlockSums] what the workgroup's units have added up of the totals, the last: how many of them have
  // By set, the first at [1]; [0], of no set, is an entry of what lies before:
  int32_t *before, *total;  // tokens of the set before this slice, in the whole batch
  int32_t *set_expert;      // the expert whose tokens the set has; n_logical (which has none): it has none
  int32_t *of_wave;         // [waves][R] ... in each wave; later, with those before this slice, before each wave
};
template <int K> __device__ inline SliceTables carve_tables(unsigned char *lds, int nl, int R) {
  SliceTables t;
  t.reps = reinterpret_cast<RepEntry *>(lds);
  t.route = reinterpret_cast<PlanRoute *>(t.reps + R + 1);
  t.records = reinterpret_cast<unsigned char *>(t.route + ((nl + 2) & ~1));   // (16-byte aligned, as what lies before it is)
  t.hist = reinterpret_cast<int32_t *>(t.records + (size_t)kPlanWaves * (R + 1) * slice_record_bytes(K));
  t.missing = t.hist + nl / 16 * 16 + 16;
  t.block_sums = t.missing + 2;
  t.before = t.missing + kSliceFlags - 1;
  t.total = t.before + R;
  t.set_expert = t.total + R;
  t.of_wave = t.set_expert + R;
  if (K == 0)
    t.records = lds + long_slice_records_at(nl, R);
  return t;
}

// What the table build reads of global memory, as unconditional loads from clamped addresses ahead of the index
// loads; and where a set belongs.
struct SetOfPlan {
  int ep_rank, place, d, group_rank;
};
__device__ inline SetOfPlan set_of_plan(const PlanArgs &a, int i) {
  const int cd = a.sh.C * a.sh.D;
  SetOfPlan s;
  s.ep_rank = (int)fast_div((uint32_t)i, a.magic_cd);
  s.place = i - s.ep_rank * cd;
  s.d = s.place - (int)fast_div((uint32_t)s.place, a.magic_D) * a.sh.D;
  s.group_rank = s.ep_rank - (int)fast_div((uint32_t)s.ep_rank, a.magic_G) * a.sh.G;
  return s;
}
__device__ inline int slot_of_plan(const PlanArgs &a, int e) {
  return e + (int)fast_div((uint32_t)e, a.magic_L) * (a.sh.P - a.sh.L);
}
// Half of the waves look after the experts, the others after the sets: the fewer instructions a wave has in front of its counts,
// the better (below).  With that, empty entries that are all zeros (one loop clears everything) and places of 32 bits, counts are out
// 1.4 instead of 1.6 us after the start: plan [8192 x 8] 7.0 -> 6.85 us, run [262144 x 8] 15.45 -> 15.25, [1048576 x 8] 34.7 -> 33.4.
constexpr int kPlanHalf = kPlanThreads / 2;
struct PlanTableLoads {
  int slot, expert, second;   // an original's slot and its expert, that of the next kPlanHalf; or a set's replica and its expert
  int physical_le0;           // phy2log of physical slot tid, where it is asked for
};
__device__ inline PlanTableLoads issue_plan_table_loads(const PlanArgs &a, int tid, int wave_s, bool with_physical) {
  PlanTableLoads t{};
  if (wave_s < kPlanWaves / 2) {
    const int nl = a.sh.n_logical;
    t.slot = slot_of_plan(a, min(tid, nl - 1));
    t.expert = a.phy2log[t.slot];
    if (nl > kPlanHalf)
      t.second = a.phy2log[slot_of_plan(a, min(tid + kPlanHalf, nl - 1))];
  } else {
    const int i = min(tid - kPlanHalf, a.n_rep - 1);
    const SetOfPlan s = set_of_plan(a, i);
    t.expert = a.phy2log[s.ep_rank * a.sh.P + s.place];
    t.second = a.o2r[s.group_rank * a.sh.D + s.d];
    t.slot = (s.ep_rank - s.group_rank + 1) * a.sh.P - a.sh.C * a.sh.D + s.place;   // (on the group's first rank)
  }
  if (with_physical)
    t.physical_le0 = a.phy2log[min(tid, a.sh.n_ranks * a.sh.P - 1)];
  return t;
}
// What a slice does before its counts are out is what the LP waits for, and it is bound by instructions: the loads
// have come 0.9 us after the workgroup started, when the LDS has just been cleared (a launch begins with an empty instruction cache:
// an instruction that runs once costs three times what it does in a loop).  So tokens are counted without a look at the mapping, the
// mapping is entered in the same interval between two barriers, and the bitmaps are marked behind the publishing.  Per call,
// against tables first and a route looked up for every token that is counted: run [8192 x 8] 9.55 -> 9.3 us, [32768 x 8] 10.45 -> 9.9,
// [100000 x 8] 12.6 -> 11.7, [262144 x 8] 16.85 -> 15.4, [16384 x 8] at 32 ranks 20.85 -> 20.25; in one workgroup [128 x 8] 7.2 -> 7.05.
// (Beyond that, the sets' totals and the waves' bases worked out ahead of the barrier instead of behind it: no faster; the places of
// the first totals to add up worked out while the loads are on their way: 0.3 us slower.)

// Everything empty: zeros from the routes to the totals (which lie side by side, so that this is one loop, of one turn for most).  A
// workgroup barrier has to follow.
template <int K> __device__ inline void clear_plan_tables(const SliceTables &t, int tid) {
  auto clear = [&](void *from, void *to) {   // (the end may reach into what is written behind the barrier)
    const int n16 = (int)(reinterpret_cast<unsigned char *>(to) - reinterpret_cast<unsigned char *>(from) + 15) / 16;
    const i32x4 zero{0, 0, 0, 0};
    for (int i = tid; i < n16; i += kPlanThreads)
      reinterpret_cast<i32x4 *>(from)[i] = zero;
  };
  clear(t.route, t.set_expert + 1);   // (in a long slice the records, which lie elsewhere, are the waves' own)
}
// Where an expert's tokens go when nothing is redirected and which replicated set (if any) it belongs to
// (minilp.cu:466-496).  A workgroup barrier has to follow.
__device__ inline void enter_plan_tables(const PlanArgs &a, const SliceTables &t, const PlanTableLoads &l, int tid, int wave_s) {
  const int nl = a.sh.n_logical, R = a.n_rep;
  if (wave_s < kPlanWaves / 2) {
    auto enter_expert = [&](int slot, int le) {
      if ((uint32_t)le < (uint32_t)nl)
        t.route[le].not_original = ~slot;
    };
    if (tid < nl)
      enter_expert(l.slot, l.expert);
    if (nl > kPlanHalf) {
      if (tid + kPlanHalf < nl)
        enter_expert(slot_of_plan(a, tid + kPlanHalf), l.second);
      for (int e = tid + 2 * kPlanHalf; e < nl; e += kPlanHalf) {
        const int s = slot_of_plan(a, e);
        enter_expert(s, a.phy2log[s]);
      }
    }
  } else {
    // (of two sets that name the same expert the later one wins, as a sequential pass over the sets would have it)
    auto enter_set = [&](int i, int slot, int le, int host) {
      const bool ok = (uint32_t)le < (uint32_t)nl;
      if (ok)
        atomicMax(&t.route[le].set, i + 1);
      t.reps[i + 1] = RepEntry{0, 0u, 0, slot + host * a.sh.P};
      t.set_expert[i + 1] = ok ? le : nl;
    };
    const int i0 = tid - kPlanHalf;
    if (i0 < R)
      enter_set(i0, l.slot, l.expert, l.second);
    if (i0 == kPlanHalf - 1)
      t.reps[0] = RepEntry{1, 0xffffffffu, INT32_MAX, -1};   // "no replica": every token stays
    if (R > kPlanHalf)
      for (int i = i0 + kPlanHalf; i < R; i += kPlanHalf) {
        const SetOfPlan s = set_of_plan(a, i);
        enter_set(i, (s.ep_rank - s.group_rank + 1) * a.sh.P - a.sh.C * a.sh.D + s.place, a.phy2log[s.ep_rank * a.sh.P + s.place],
                  a.o2r[s.group_rank * a.sh.D + s.d]);
      }
  }
}
// The expert whose tokens a set has, once the routes are there; n_logical: none (of two sets that name the same expert only one
// has the tokens).
__device__ inline int expert_of_set(const PlanArgs &a, const SliceTables &t, int set) {
  const int e = t.set_expert[set];
  return t.route[e].set == set ? e : a.sh.n_logical;
}

// K chunks of 64 indices from w0 on (uniform); places past the last before `end` (not 0) repeat that, until mask_chunks is called
// once something else has been done.  (Loads that some lanes leave out, or a look at what was loaded, wait for all loads before.)
// Places are below 2^32: a batch has fewer than 2^31 indices.
template <int K> __device__ inline void load_chunks(int64_t (&raw)[K], const int64_t *idx, uint32_t w0, uint32_t end, int lane) {
  const int64_t *src = idx + w0;
  if (w0 + K * kWave <= end) {
#pragma unroll
    for (int c = 0; c < K; ++c)
      raw[c] = __builtin_nontemporal_load(src + lane + c * kWave);
  } else {
    const int last = (int)(end - 1 - w0);
#pragma unroll
    for (int c = 0; c < K; ++c)
      raw[c] = __builtin_nontemporal_load(src + min(c * kWave + lane, last));
  }
}
template <int K> __device__ inline void mask_chunks(int64_t (&raw)[K], uint32_t w0, uint32_t end, int lane) {
  if (w0 + K * kWave > end) {
    const int last = (int)(end - 1 - w0);
#pragma unroll
    for (int c = 0; c < K; ++c)
      raw[c] = c * kWave + lane <= last ? raw[c] : -1;
  }
}
template <int K> __device__ inline void store_chunks(const int32_t (&o)[K], int64_t *out, uint32_t w0, uint32_t end, int lane) {
  int64_t *dst = out + w0 + lane;
  if (w0 + K * kWave <= end) {
#pragma unroll
    for (int c = 0; c < K; ++c)
      __builtin_nontemporal_store((int64_t)o[c], dst + c * kWave);
  } else {
    const int last = (int)(end - 1 - w0);
#pragma unroll
    for (int c = 0; c < K; ++c)
      if (c * kWave + lane <= last)
        __builtin_nontemporal_store((int64_t)o[c], dst + c * kWave);
  }
}
// The value is computed at this point and not moved down to where it is first used.
template <typename T> __device__ inline void worked_out_here(T &v) { asm volatile("" : "+v"(v)); }
// Between the phases a token is kept as its expert id only, two ids per register (the route is looked up
// again where it is needed): the waits are long and registers bound how many workgroups are resident.
template <int N> __device__ inline int packed_expert(const uint32_t (&packed)[N], int c) {
  return (int)((packed[c / 2] >> (16 * (c % 2))) & 0xffffu);
}
template <int N> __device__ inline void pack_expert(uint32_t (&packed)[N], int c, int e) {
  packed[c / 2] = (c % 2) ? packed[c / 2] | ((uint32_t)e << 16) : (uint32_t)e;
}

// ---- a slice's tokens: histogram and bitmaps, the tokens of the earlier chunks and waves ----
template <int K> struct SliceTokens {
  static constexpr int kRec = rank_record_bytes_single(K);
  __device__ static ChunkSlot *slot(unsigned char *my_records, int set, int c) {
    return reinterpret_cast<ChunkSlot *>(my_records + __umul24((uint32_t)set, (uint32_t)kRec)) + c;
  }
  // Counts the wave's tokens in t.hist; needs nothing of the mapping.
  __device__ static void count(const PlanArgs &a, const SliceTables &t, const int64_t (&raw)[K], uint32_t (&packed)[(K + 1) / 2]) {
    const int nl = a.sh.n_logical;
#pragma unroll
    for (int c = 0; c < K; ++c) {
      const bool valid = (uint64_t)raw[c] < (uint64_t)nl;   // -1, other negatives and too large ids fail
      pack_expert(packed, c, valid ? (int)raw[c] : nl);
      if (valid)
        atomicAdd(&t.hist[(int)raw[c]], 1);
    }
  }
  // A slot's bits become the chunk's tokens of its set.  The wave's own slots: no barrier.
  __device__ static void mark(const PlanArgs &a, const SliceTables &t, unsigned char *my_records, const uint32_t (&packed)[(K + 1) / 2], int lane) {
    constexpr int N = K < 8 ? K : 8;   // (reads ahead of the first update: the compiler keeps their order, and each would be waited for)
    const unsigned long long my_bit = 1ull << lane;
#pragma unroll
    for (int c0 = 0; c0 < K; c0 += N) {
      int set[N];
#pragma unroll
      for (int c = 0; c < N; ++c)
        set[c] = t.route[packed_expert(packed, c0 + c)].set;
#pragma unroll
      for (int c = 0; c < N; ++c)
        if (set[c] != 0)
          atomicOr(reinterpret_cast<unsigned long long *>(slot(my_records, set[c], c0 + c)), my_bit);
    }
    own_slots_are_written();
  }
  // The tokens of each set in the wave's earlier chunks into the slots, those in the whole wave into t.of_wave.  lane = set:
  // the chunks' pop-counts add up as they are read.  (lane = (set, chunk) with a scan over the lanes of a set takes as many instructions
  // at 16 sets and eight times as many at 128.  Counts supplied, [100000 x 8]: 64 sets 15.2 -> 12.8 us, 32 sets 12.1 -> 11.3; [16384 x 8]
  // with 128 sets 11.0 -> 10.2; [262144 x 8] with 16 sets 18.0 -> 17.9.)
  __device__ static void starts_in_wave(const PlanArgs &a, const SliceTables &t, unsigned char *my_records, int lane, int wave_s) {
    const int R = a.n_rep;
    for (int q = lane + 1; q <= R; q += kWave) {
      unsigned long long bits[K];
#pragma unroll
      for (int c = 0; c < K; ++c)
        bits[c] = *reinterpret_cast<const unsigned long long *>(slot(my_records, q, c));
      int before = 0;
#pragma unroll
      for (int c = 0; c < K; ++c) {
        slot(my_records, q, c)->start = before;
        before += __popcll(bits[c]);
      }
      t.of_wave[wave_s * R + q] = before;
    }
  }
  // What t.of_wave has becomes the tokens of each set before each wave's first, by the second half of the waves, a lane a set.  A
  // workgroup barrier on either side.  (A table of its own for these takes 32 bytes a set: two slices of 16 chunks with 32 sets and 512
  // experts did not fit a CU any more, and [262144 x 8] at 16 ranks ran as the chain.)
  __device__ static void bases(const PlanArgs &a, const SliceTables &t, int tid) {
    const int R = a.n_rep;
    for (int q = tid - kPlanHalf + 1; q <= R; q += kPlanHalf) {
      int32_t in_wave[kPlanWaves - 1];
#pragma unroll
      for (int w = 0; w < kPlanWaves - 1; ++w)
        in_wave[w] = t.of_wave[w * R + q];
      int32_t base = t.before[q];
#pragma unroll
      for (int w = 0; w < kPlanWaves; ++w) {
        t.of_wave[w * R + q] = base;
        if (w < kPlanWaves - 1)
          base += in_wave[w];
      }
    }
  }
  // The same where the workgroup holds the whole batch: from the bitmaps of the `turn` waves before this one, records_of(w)
  // their records.
  template <typename Records>
  __device__ static void starts_of_batch(const PlanArgs &a, unsigned char *my_records, int lane, int turn, Records records_of) {
    const int R = a.n_rep, c = lane % K;
    for (int p0 = 0; p0 < R * K; p0 += kWave) {
      const bool live = p0 + lane < R * K;
      const int q = live ? (p0 + lane) / K + 1 : 0;
      int earlier = 0;
      for (int w = 0; w < turn; ++w)
        earlier += __popcll(*reinterpret_cast<const unsigned long long *>(slot(records_of(w), q, c)));
      ChunkSlot *mine = slot(my_records, q, c);
      const int own = __popcll(*reinterpret_cast<const unsigned long long *>(mine));
      const int start = group_sum<K>(earlier) + group_exclusive_scan<K>(own, c);
      if (live)
        mine->start = start;
    }
    own_slots_are_written();
  }
  __device__ static void own_slots_are_written() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // base: of the wave's sets, or null: part of the starts.
  __device__ static int32_t hash(const SliceTables &t, unsigned char *my_records, const int32_t *base, int e, int c) {
    const int set = t.route[e].set;
    const int32_t before = base ? base[set] : 0;   // (of no set: whatever is there)
    const i32x4 s = *reinterpret_cast<const i32x4 *>(slot(my_records, set, c));   // bits_lo, bits_hi, start
    const i32x4 x = *reinterpret_cast<const i32x4 *>(&t.reps[set]);               // total, magic, -, -
    const int32_t k =
        __builtin_amdgcn_mbcnt_hi((uint32_t)s.y, __builtin_amdgcn_mbcnt_lo((uint32_t)s.x, (uint32_t)(s.z + before)));
    return ordinal_hash<false>(k, x.x, (uint32_t)x.y);
  }
};

// Tokens per physical expert (= bincount of the output) from a slice's tables; hist: of the batch.
// le0: phy2log of slot tid (or of any slot if there is none), read ahead of time.
__device__ inline void plan_physical_counts(const PlanArgs &a, const SliceTables &t, int le0, bool ok, int tid) {
  const int nl = a.sh.n_logical;
  for (int i = tid; i < a.sh.n_ranks * a.sh.P; i += kPlanThreads) {
    const int le = !ok ? -1 : i == tid ? le0 : a.phy2log[i];
    int32_t v = ok ? 0 : -1;
    if (le >= 0 && le < nl) {
      const PlanRoute rt = t.route[le];
      if (rt.set == 0) {
        v = rt.original() == i ? t.hist[le] : 0;
      } else {
        const RepEntry x = t.reps[rt.set];
        const int32_t kept = kept_on_original(x.total, x.expected);
        v = rt.original() == i ? kept : (x.replica == i ? x.total - kept : 0);
      }
    }
    a.physical_counts[i] = v;
  }
}
__device__ inline void set_total(RepEntry &x, int32_t total) {
  x.total = total;
  x.magic = total >= 1 ? 0xffffffffu / (uint32_t)total : 0u;
}

// ---- collecting words ----
__device__ inline unsigned long long tagged_word(uint32_t tag, uint32_t v) { return ((unsigned long long)tag << 32) | v; }
// Up to N words per lane (its first `mine`), all with the launch's tag: polls those that are not in yet until they are or
// max_polls polls have passed; words past `mine` are 0.  Whole waves; false: the wait ran out.
template <int N, typename Address>
__device__ inline bool collect_words(uint32_t (&words)[N], uint32_t tag, int mine, int max_polls, Address address) {
  unsigned long long v[N];
#pragma unroll
  for (int k = 0; k < N; ++k)
    v[k] = k < mine ? ~(unsigned long long)tag << 32 : (unsigned long long)tag << 32;
  for (int polls = 0; polls < max_polls; ++polls) {
#pragma unroll
    for (int k = 0; k < N; ++k)
      if ((uint32_t)(v[k] >> 32) != tag)
        v[k] = agent_load(address(k));
    bool all_in = true;
#pragma unroll
    for (int k = 0; k < N; ++k)
      all_in = all_in && (uint32_t)(v[k] >> 32) == tag;
    if (__all(all_in)) {
#pragma unroll
      for (int k = 0; k < N; ++k)
        words[k] = (uint32_t)v[k];
      return true;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  return false;
}
// What slices add up of each other's rows is cut into units, one wave's work each: kUnitSlices slices' words at eight adjacent
// places (more if there are fewer slices).  lane = (slice, pair of words); a lane loads the pairs of four slices at once.
// No barrier, and nothing to clear first.  (One CU reads such words at 25 bytes per ns with 8-byte loads, one a lane, and at 68
// with four and more 16-byte loads a lane on their way.)
constexpr int kUnitSlices = 64, kUnitLoads = 4;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// The sum over the slices of a unit, for N values of every lane; lanes_log2: of a slice.
template <int N> __device__ inline void over_slices_of_unit(uint32_t (&v)[N], int lanes_log2) {
  if (lanes_log2 == 2)
#pragma unroll
    for (int j = 0; j < N; ++j)
      v[j] += (uint32_t)dpp_int<0x124>((int)v[j]);   // row_ror:4
  if (lanes_log2 <= 3)
#pragma unroll
    for (int j = 0; j < N; ++j)
      v[j] += (uint32_t)dpp_int<0x128>((int)v[j]);   // row_ror:8
  if (lanes_log2 <= 4)
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const u32x2 s = __builtin_amdgcn_permlane16_swap(v[j], v[j], false, false);
      v[j] = s.x + s.y;
    }
  if (lanes_log2 <= 5)
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const u32x2 s = __builtin_amdgcn_permlane32_swap(v[j], v[j], false, false);
      v[j] = s.x + s.y;
    }
}
// Where a lane finds its pairs of words of a unit: words 2 (lane % lanes of a slice) and the next of the rows from `rows` on (16-byte
// aligned; lanes past the last of `words` words, an even number, repeat that), of the slices of block `block` (past the last
// slice: that one again).
struct UnitAt {
  const unsigned long long *at[kUnitLoads];
};
__device__ inline UnitAt unit_at(const PlanArgs &a, const unsigned long long *rows, int stride, int words, int block, int lane) {
  const int per_round = kWave >> a.unit_lanes_log2, p0 = block * kUnitSlices + (lane >> a.unit_lanes_log2);
  const unsigned long long *mine = rows + min(2 * (lane & ((1 << a.unit_lanes_log2) - 1)), words - 2);
  UnitAt u;
#pragma unroll
  for (int k = 0; k < kUnitLoads; ++k)
    u.at[k] = mine + min(p0 + k * per_round, a.n_slices - 1) * stride;
  return u;
}
// Adds a unit up: the four counts of a lane's words over the slices into sums[0..3] and, if BEFORE, over the slices before `slice`
// into sums[4..7].  Whole waves; false: some never came.
// LONG: slices of up to kLongestOfLongSlices indices.
template <bool BEFORE, bool LONG>
__device__ inline bool add_up_unit(const PlanArgs &a, const UnitAt &u, int block, uint32_t tag, int slice, int lane,
                                   uint32_t (&sums)[BEFORE ? 8 : 4]) {
  if (a.expected_slices != a.n_slices)   // (an injected fault: one slice never comes)
    return false;
  const int per_round = kWave >> a.unit_lanes_log2, p0 = block * kUnitSlices + (lane >> a.unit_lanes_log2);
  u32x4 v[kUnitLoads];
  bool all_in = false;
  for (int polls = 0; polls < a.max_polls; ++polls) {
    if (!all_in) {
      agent_load_pairs(v, u.at);
      uint32_t off = 0;
#pragma unroll
      for (int k = 0; k < kUnitLoads; ++k)
        off |= (v[k].y ^ tag) | (v[k].w ^ tag);
      all_in = off == 0;
    }
    if (__all(all_in))
      break;
    __builtin_amdgcn_s_sleep(1);
  }
  if constexpr (LONG) {
    static_assert(kLongestOfLongSlices < 65536, "two counts to a word");
#pragma unroll
    for (int j = 0; j < (BEFORE ? 8 : 4); ++j)
      sums[j] = 0;
#pragma unroll
    for (int k = 0; k < kUnitLoads; ++k) {
      const int p = p0 + k * per_round;
      const uint32_t counts[4] = {v[k].x & 0xffffu, v[k].x >> 16, v[k].z & 0xffffu, v[k].z >> 16};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sums[j] += p < a.n_slices ? counts[j] : 0u;
        if constexpr (BEFORE)
          sums[4 + j] += p < slice ? counts[j] : 0u;
      }
    }
  } else {
    // (two counts to a word: of four slices they stay below 2^16)
    static_assert(kUnitLoads * kLongestSlice < 65536, "sums of two 16-bit counts side by side");
    u32x2 total{0, 0}, before{0, 0};
#pragma unroll
    for (int k = 0; k < kUnitLoads; ++k) {
      const int p = p0 + k * per_round;
      const u32x2 counts{v[k].x, v[k].z};
      total += p < a.n_slices ? counts : u32x2{0, 0};
      before += BEFORE && p < slice ? counts : u32x2{0, 0};
    }
    sums[0] = total.x & 0xffffu, sums[1] = total.x >> 16, sums[2] = total.y & 0xffffu, sums[3] = total.y >> 16;
    if constexpr (BEFORE)
      sums[4] = before.x & 0xffffu, sums[5] = before.x >> 16, sums[6] = before.y & 0xffffu, sums[7] = before.y >> 16;
  }
  over_slices_of_unit(sums, a.unit_lanes_log2);
  return __all(all_in);
}
// The batch's totals into `counts` (LDS), by every wave of the workgroup.  Returns whether this wave's have come.
__device__ inline bool collect_totals(const PlanArgs &a, int32_t *counts, uint32_t tag, int tid, int wave_s) {
  const unsigned long long *totals = reinterpret_cast<const unsigned long long *>(a.sync + kTotalsAt);
  const int nl = a.sh.n_logical;
  if (a.expected_slices != a.n_slices)   // (an injected fault: one slice never comes)
    return false;
  for (int e0 = wave_s * kWave; e0 < nl; e0 += kPlanThreads) {
    const int e = e0 + tid % kWave;
    uint32_t count[1];
    if (!collect_words<1>(count, tag, e < nl, a.max_polls, [&](int) { return totals + e; }))
      return false;
    if (e < nl)
      counts[e] = (int32_t)count[0];
  }
  return true;
}

// Waves of a workgroup that wait for some of the others without a barrier for all: what one has done to the LDS before it arrives
// is there for those that have waited.  (Whoever is waited for arrives before it waits itself, so every wait ends.)
__device__ inline void wave_arrives(int *arrived, int lane) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  if (lane == 0)
    __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline void wait_for_waves(const int *arrived, int waves) {
  while (__hip_atomic_load(arrived, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < waves)
    __builtin_amdgcn_s_sleep(1);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// By whole waves of a workgroup that have added to words in LDS: true for the wave that comes last, which sees what all `waves`
// of them have added.  (On either side of the count a wait for the LDS and no more; only with more than 64 slices.)
__device__ inline bool last_wave_to_arrive(int *arrived, int waves, int lane) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  int before = 0;
  if (lane == 0)
    before = __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  const bool last = __builtin_amdgcn_readfirstlane(before) == waves - 1;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  return last;
}
// What others have published, unit by unit: the batch's totals of this slice's share of the experts, if it is one of
// those that add them up; the tokens of each replicated set before this slice and in the whole batch.
enum class Units { kTotals, kSets };
template <bool LONG, Units WHICH>
__device__ __forceinline__ void add_up_published(const PlanArgs &a, const SliceTables &t, int slice, uint32_t tag, int lane, int wave_s,
                                                 int *missing, int *block_sums) {
  const int R = a.n_rep, set_lanes = a.set_words;
  unsigned long long *set_rows = reinterpret_cast<unsigned long long *>(a.sync + kSetRowsAt);
  unsigned long long *hist_rows = reinterpret_cast<unsigned long long *>(a.sync + kHistRowsAt);
  const int unit_lanes = 1 << a.unit_lanes_log2, unit_words_log2 = a.unit_lanes_log2 + 1, block_bits = a.unit_block_bits;
  const int first_word = slice * a.adder_words, my_words = slice < a.adders ? min(a.adder_words, a.hist_words - first_word) : 0;
  const int adder_units = ((my_words + (1 << unit_words_log2) - 1) >> unit_words_log2) << block_bits;
  const int units = adder_units + (((set_lanes + (1 << unit_words_log2) - 1) >> unit_words_log2) << block_bits);
  unsigned long long *totals = reinterpret_cast<unsigned long long *>(a.sync + kTotalsAt);
  for (int unit = kPlanWaves - 1 - wave_s; unit < units; unit += kPlanWaves) {   // the last waves first: the others have published
    const int block = unit & ((1 << block_bits) - 1);
    if (block >= a.unit_blocks || (WHICH == Units::kSets && unit < adder_units))
      continue;
    if (unit >= adder_units) {
      if (WHICH == Units::kTotals)
        break;
      const int word0 = (unit - adder_units) >> block_bits << unit_words_log2;
      uint32_t sums[8];
      if (add_up_unit<true, LONG>(a, unit_at(a, set_rows + word0, a.set_words, set_lanes - word0, block, lane), block, tag, slice, lane, sums)) {
        const int first_set = 2 * word0 + 4 * lane;
        if (lane < unit_lanes)   // (words past set_lanes have no sets)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (first_set + j < R) {
              atomicAdd(&t.total[first_set + j + 1], (int32_t)sums[j]);
              atomicAdd(&t.before[first_set + j + 1], (int32_t)sums[4 + j]);
            }
      } else {
        missing[0] = 1;
      }
    } else {
      const int at = unit >> block_bits << unit_words_log2, word0 = first_word + at;
      uint32_t sums[4];
      if (add_up_unit<false, LONG>(a, unit_at(a, hist_rows + word0, a.hist_words, my_words - at, block, lane), block, tag,
                                   slice, lane, sums)) {
        bool all_in = true;
        if (a.unit_blocks > 1) {   // (eight words then, in one unit per block: the wave that comes last publishes)
          if (lane < 4)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              atomicAdd(&block_sums[4 * lane + j], (int32_t)sums[j]);
          all_in = last_wave_to_arrive(&block_sums[16], a.unit_blocks, lane);
          if (all_in && lane < 4)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              sums[j] = (uint32_t)block_sums[4 * lane + j];
        }
        if (all_in && lane < unit_lanes && 2 * lane < my_words - at) {   // (words behind the last expert's have zeros and are not read)
          unsigned long long *to = totals + 2 * word0 + 4 * lane;
          agent_store_pairs(to, u32x4{sums[0], tag, sums[1], tag}, u32x4{sums[2], tag, sums[3], tag});
        }
      } else {
        missing[0] = 1;
      }
    }
  }
}

// By one wave of a slice that has every slice's counts.
__device__ __forceinline__ void say_that_all_arrived(const PlanArgs &a, uint32_t tag, int lane) {
  // Every slice has published its counts; once the LP workgroups have shown up too, no workgroup waits for one that is
  // not resident yet.  Tell the host, which then stops counting this launch against what the GPU can hold at
  // once (a posted write to host memory).  Told at the end, behind the LP, plans on several streams found the GPU
  // full more often and ran as the chain: [16384 x 8] at 32 ranks in turn on 4 streams 11.0 us a plan, 0.34 of them
  // as one launch; told here 9.9 us, 0.50.
  uint32_t here[1];
  if (collect_words<1>(here, tag, lane < a.n_lp_workgroups, a.max_polls,
                       [&](int) { return reinterpret_cast<const unsigned long long *>(a.sync + kLpHereAt) + lane; }))
    __hip_atomic_store(a.arrived_word, a.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// The LP's shares: every set's thread polls its own; value and tag arrive in the same word.  missing[1]: some will not come.
__device__ __forceinline__ void collect_shares(const PlanArgs &a, const SliceTables &t, int slice, int gen, unsigned long long *avail_state,
                                               int tid) {
  const int R = a.n_rep;
  const unsigned long long *shares = reinterpret_cast<const unsigned long long *>(a.sync + kSharesAt);
  const uint32_t tag_valid = share_tag((uint32_t)gen), tag_none = tag_valid + 1u;
  for (int i = tid; i < R; i += kPlanThreads) {
    const SetOfPlan s = set_of_plan(a, i);
    const unsigned long long *word_at = shares + (slice & (a.n_share_copies - 1)) * kMaxShares + s.ep_rank * a.sh.D + s.d;
    unsigned long long word = 0;
    int polls = 0;
    uint32_t got = 0;
    // (no sleep between polls, each of which takes a trip to memory: a share is seen up to 64 clocks sooner, run [1024 x 8] 9.25 -> 9.1 us,
    // [262144 x 8] 15.35 -> 15.25.  Other streams' work does not notice it, with the sleep / without: beside plans of 32 ranks, whose lanes
    // poll for 15 us, a 256 MiB copy takes 252-263 / 256 us and a bf16 product of 4096 267-277 / 265-267)
    while ((got = (uint32_t)((word = agent_load(word_at)) >> 32)) != tag_valid && got != tag_none && ++polls < a.max_polls) {
    }
    if (got == tag_valid) {
      t.reps[i + 1].expected = expected_on_original(__builtin_bit_cast(float, (uint32_t)word), t.total[i + 1]);
    } else {
      if (got != tag_none)
        give_up(a, avail_state);
      t.missing[1] = 1;
    }
  }
}
// The slice has read all it reads of this block of words.  (By a whole wave: the same word from every lane is one store.)
__device__ __forceinline__ void slice_has_read_all(const PlanArgs &a, int slice, int gen, int wave_s) {
  if (slice == 0 && wave_s == 0) {
    // Every slice's counts and every LP's shares carry this launch's tag, so every workgroup has read it: the
    // next launch takes the next one.
    agent_store(a.sync + kGenAt, (gen + 1) & 0x3fffffff);
    agent_store(reinterpret_cast<unsigned long long *>(a.sync + kAvailAt) + (1 - (gen & 1)), 0ull);
    unsigned long long *advanced = reinterpret_cast<unsigned long long *>(a.sync + kAdvancedAt);
    agent_store(advanced, tagged_word(a.seq >= 0 ? (uint32_t)a.seq : (uint32_t)(agent_load(advanced) >> 32), (gen + 1) & 0x3fffffff));
  } else if (wave_s == 0 && a.seq >= 0) {
    agent_store(a.sync + kDoneAt + slice * kDoneStride, a.seq);
  }
}

// Normalised counts of the experts from `first` on, `n` of them, for the caller, by nt threads (whole waves): each count over the
// largest of all.
__device__ inline void write_normalised_counts(const PlanArgs &a, const int32_t *counts, int first, int n, int thread, int nt, int lane) {
  int32_t most = 0;
  for (int e = lane; e < a.sh.n_logical; e += kWave)
    most = max(most, counts[e]);
  const float wmax = wave_max_of_groups<true, true>((float)most);
  for (int i = thread; i < n; i += nt)
    a.solve.gw_out[first + i] = (float)counts[first + i] / wmax;
}
// An LP workgroup of a plan: one wave per LP, the others help to collect the counts and write the normalised ones (by the LP waves
// themselves, at their end, those took 0.8 us, and what is counted for the caller behind them came as much later).
template <int GM, int DM, bool EXACT>
__device__ __forceinline__ void lp_workgroup(const PlanArgs &a, unsigned char *smem_raw, int *rep_of_edge_all, unsigned long long gen_and_poison,
                                             int tid, int lane, int wave_s) {
  const int nl = a.sh.n_logical, pid = blockIdx.x;
  unsigned long long *shares = reinterpret_cast<unsigned long long *>(a.sync + kSharesAt);
  SolveArgs sa = a.solve;
  const int first_lp = pid * kLpsPerWorkgroup;          // of this workgroup
  const int n_lps = min(kLpsPerWorkgroup, sa.n_units - first_lp);
  LPLB_PLAN_STAMP(0);
  if (tid == kPlanThreads - kWave)   // (a wave without an LP)
    agent_store(reinterpret_cast<unsigned long long *>(a.sync + kLpHereAt) + pid, tagged_word((uint32_t)gen_and_poison + 1u, 0));
  // dynamic LDS of an LP workgroup: [LP wave][pivot rows | assembly tile], then the counts
  constexpr size_t kLpArea = plan_lp_area_bytes<GM, DM>();
  static_assert(kLpArea % 16 == 0, "the LP waves' areas keep 16-byte alignment");
  unsigned char *my_area = smem_raw + (size_t)min(wave_s, kLpsPerWorkgroup - 1) * kLpArea;
  float *staged = reinterpret_cast<float *>(smem_raw + kLpsPerWorkgroup * kLpArea);
  int *const missing = reinterpret_cast<int *>(staged) + sa.staged_stride - 1;   // some counts did not come (own-histogram mode)
  sa.launch = (uint32_t)gen_and_poison;
  sa.gw_out = nullptr;   // (written by the waves without an LP)
  auto switched_off = [&]() { return (gen_and_poison >> 32) != 0; };
  // Own-histogram mode: the LP waves' table loads are on their way when they and the other waves turn to the
  // batch's histogram.  (Switched off: no slice will publish.)
  auto counts_have_come = [&]() -> bool {
    if (tid >= kPlanThreads - 4)   // the zeros behind the counts
      reinterpret_cast<int32_t *>(staged)[nl + tid - (kPlanThreads - 4)] = 0;
    worked_out_here(gen_and_poison);
    const bool mine = !switched_off() && collect_totals(a, reinterpret_cast<int32_t *>(staged), (uint32_t)gen_and_poison + 1u, tid, wave_s);
    if (!mine && lane == 0)
      missing[0] = 1;
    __syncthreads();
    return missing[0] == 0;
  };
  if (a.local_counts) {
    if (tid == 0)
      missing[0] = 0;
    __syncthreads();
  }
  LPLB_PLAN_STAMP(1);
  if (wave_s < n_lps) {
    __builtin_amdgcn_s_setprio(1);
    // (own-histogram mode: every LP of the batch reads the one staged copy)
    float *mine = a.local_counts ? staged : staged + (size_t)wave_s * sa.staged_stride;
    const int n_ok = solve_lps<GM, DM, EXACT, 1, 1, true>(
        sa, first_lp + wave_s, mine, rep_of_edge_all + wave_s * kWave, reinterpret_cast<double *>(my_area),
        reinterpret_cast<float *>(my_area + lp_pivot_doubles<GM, DM>() * sizeof(double)), counts_have_come);
    worked_out_here(gen_and_poison);
    unsigned long long *avail_state = reinterpret_cast<unsigned long long *>(a.sync + kAvailAt) + (gen_and_poison & 1);
    if (n_ok < 0) {
      // no counts, no solution: tell the slices not to wait for this LP's shares
      if (wave_s == 0 && lane == 0 && !switched_off())
        give_up(a, avail_state);
      const int n_edges = sa.G * sa.D;
      for (int j = lane; j < n_edges; j += kWave)
        for (int k = 0; k < a.n_share_copies; ++k)
          agent_store(shares + (int64_t)k * kMaxShares + (int64_t)(first_lp + wave_s) * n_edges + j,
                      (unsigned long long)(share_tag(sa.launch) + 1u) << 32);
    } else if (lane == 0 && n_ok > 0 && !switched_off()) {
      // feasible: count it for the caller unless some workgroup has already given up on this batch
      const unsigned long long before = __hip_atomic_fetch_or(avail_state, 1ull << (first_lp + wave_s), __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_AGENT);
      if (!(before & kGaveUp))
        atomicAdd(a.avail, n_ok);
    }
    if (lane == 0 && a.seq >= 0)
      agent_store(a.sync + kDoneAt + (kMaxSlices + first_lp + wave_s) * kDoneStride, a.seq);
  } else if (!a.local_counts || counts_have_come()) {
    const int helper = kLpsPerWorkgroup * kWave, per_lp = sa.G * (sa.D * sa.C + sa.n_fixed);
    if (tid >= helper)
      write_normalised_counts(a, a.local_counts ? reinterpret_cast<const int32_t *>(staged) : sa.workload, first_lp * per_lp, n_lps * per_lp,
                              tid - helper, kPlanThreads - helper, lane);
  }
}

// K: 64-index chunks per wave.
// Registers: up to 16 ranks the kernel as a whole is held to 128 VGPRs (two workgroups per CU), which is what
// lets 256 slices and the LPs be resident together; the LP of 32 ranks takes more.
constexpr int plan_workgroups_per_cu(int group_size) { return group_size <= 16 ? 2 : 1; }
template <int GM, int DM, bool EXACT, int K>
__global__ __launch_bounds__(kPlanThreads, 2 * plan_workgroups_per_cu(GM)) void plan_in_one_launch(PlanArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  __shared__ int rep_of_edge_all[kLpsPerWorkgroup * kWave];
  const int nl = a.sh.n_logical, R = a.n_rep;
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave_s = __builtin_amdgcn_readfirstlane(tid / kWave);   // wave-uniform
  const int pid = blockIdx.x;
  // (one argument of every 64 bytes of them: the others then come out of the scalar cache)
  fetch_arguments_now(a.idx, a.unit_blocks, a.sh.G, a.solve.workload, a.solve.n_group, a.solve.tagged_result, a.sync);
  // Which launch of this block of words this is (the same value in every workgroup: it is advanced only once
  // all of them have read it), and whether the block is switched off.  Both are looked at once the loads behind this one
  // are on their way.
  static_assert(kGenAt == 0 && kPoisonAt == 1, "one word");
  unsigned long long gen_and_poison = agent_load(reinterpret_cast<const unsigned long long *>(a.sync));

  if (pid < a.n_lp_workgroups) {
    // ------------------------------------------------------------ the LPs
    lp_workgroup<GM, DM, EXACT>(a, smem_raw, rep_of_edge_all, gen_and_poison, tid, lane, wave_s);
    LPLB_PLAN_STAMP(2);
    return;
  }

  // --------------------------------------------------------------- a slice
  const int slice = pid - a.n_lp_workgroups;
  const SliceTables t = carve_tables<K>(smem_raw, nl, R);
  unsigned char *my_records = t.records + (size_t)wave_s * ((R + 1) * rank_record_bytes_single(K));
  int *const missing = t.missing;
  const uint32_t end = (uint32_t)min(a.n, a.per * (slice + 1)), w0 = (uint32_t)a.per * (uint32_t)slice + wave_s * (K * kWave);   // this wave's first index (uniform)
  LPLB_PLAN_STAMP(0);
  LPLB_SLICE_STAMP(0);
  // Where a slice shares a CU with an LP workgroup (grids with more workgroups than CUs), its waves go first until the counts are in:
  // the LP wave issues an instruction nearly every cycle it may, also where counts are supplied and it has begun, and a slice wave on
  // the same SIMD would be starved for as long as the LP runs, with every other slice waiting for it.
  __builtin_amdgcn_s_setprio(2);

  // ---- small table reads, the index loads right behind them, the tables while they are on their way ----
  const PlanTableLoads tl = issue_plan_table_loads(a, tid, wave_s, slice == 0 && a.physical_counts);
  int64_t raw[K];
  load_chunks<K>(raw, a.idx, w0, end, lane);
  clear_plan_tables<K>(t, tid);
  __syncthreads();
  LPLB_PLAN_STAMP(10);
  enter_plan_tables(a, t, tl, tid, wave_s);
  // ---- the tokens ----
  uint32_t packed[(K + 1) / 2];
  mask_chunks<K>(raw, w0, end, lane);
  SliceTokens<K>::count(a, t, raw, packed);
  __syncthreads();
  LPLB_PLAN_STAMP(8);
  LPLB_SLICE_STAMP(1);
  // ---- this slice's counts, for every workgroup: the histogram by the first half of the waves, the sets by the others ----
  worked_out_here(gen_and_poison);
  const int gen = (int)(uint32_t)gen_and_poison;
  const bool poisoned = (gen_and_poison >> 32) != 0;
  const uint32_t tag = (uint32_t)gen + 1u;
  unsigned long long *avail_state = reinterpret_cast<unsigned long long *>(a.sync + kAvailAt) + (gen & 1);
  unsigned long long *set_rows = reinterpret_cast<unsigned long long *>(a.sync + kSetRowsAt);
  unsigned long long *hist_rows = reinterpret_cast<unsigned long long *>(a.sync + kHistRowsAt);
  const int set_lanes = a.set_words;
  if (!poisoned) {
    constexpr int kHalf = kPlanThreads / 2;
    if (tid < kHalf) {
      for (int e2 = tid; e2 < a.hist_words; e2 += kHalf) {
        const int2 both = reinterpret_cast<const int2 *>(t.hist)[e2];
        agent_store(hist_rows + slice * a.hist_words + e2, tagged_word(tag, (uint32_t)both.x | (uint32_t)both.y << 16));
      }
    } else {
      for (int i = tid - kHalf; i < 2 * set_lanes; i += kHalf) {   // lane = set, the word from the second of its two
        const int e = t.set_expert[min(i, R - 1) + 1];
        const int tokens = i < R && t.route[e].set == i + 1 ? t.hist[e] : 0;
        const uint32_t both = (uint32_t)dpp_int<kQuadSwap1>(tokens) | (uint32_t)tokens << 16;
        if (i & 1)
          agent_store(set_rows + slice * a.set_words + i / 2, tagged_word(tag, both));
      }
    }
  } else if (slice == 0 && tid == 0) {
    agent_add(a.sync + kTimeoutsAt, 1);   // one more plan that this block of words could not serve
  }
  LPLB_PLAN_STAMP(1);
  LPLB_SLICE_STAMP(2);
  // ---- what others have published, unit by unit: the batch's totals of this slice's share of the experts, if it is one of
  //      those that add them up and the LP waits for them; the tokens of each replicated set before this slice and in the whole batch.
  //      In between, while words are on their way, the tokens of each set in this slice's earlier chunks ----
  // (the waves that add up totals go first on their SIMDs meanwhile: run [32768 x 8] 10.0 -> 9.9 us, [100000 x 8] 11.8 -> 11.6)
  if (!poisoned) {
    if (slice < a.adders && wave_s >= kPlanWaves / 2)
      __builtin_amdgcn_s_setprio(3);
    add_up_published<false, Units::kTotals>(a, t, slice, tag, lane, wave_s, missing, t.block_sums);
    __builtin_amdgcn_s_setprio(2);
  }
  SliceTokens<K>::mark(a, t, my_records, packed, lane);
  SliceTokens<K>::starts_in_wave(a, t, my_records, lane, wave_s);
  if (!poisoned)
    add_up_published<false, Units::kSets>(a, t, slice, tag, lane, wave_s, missing, t.block_sums);
  LPLB_PLAN_STAMP(11);
  if (poisoned)
    missing[0] = 1;
  __syncthreads();
  LPLB_PLAN_STAMP(2);
  LPLB_SLICE_STAMP(4);
  bool ok = missing[0] == 0;   // (the same in every thread)
  if (!ok && !poisoned && tid == 0)
    give_up(a, avail_state);
  // From here on it is the slice that has time.  (At 2 for its whole length, the one that shares a CU with the LP slowed its first step
  // from 0.6 to 1.7 us while it hashed: [262144 x 8] 17.5 -> 16.7 us.)
  __builtin_amdgcn_s_setprio(0);
  int32_t h[K];   // hashes of this thread's tokens: worked out while the LP is still running
  if (ok) {
    if (wave_s < kPlanWaves / 2)
      for (int q = tid + 1; q <= R; q += kPlanHalf)
        set_total(t.reps[q], t.total[q]);
    else
      SliceTokens<K>::bases(a, t, tid);
    if (slice == 0 && wave_s == kPlanWaves - 1 && a.arrived_word)
      say_that_all_arrived(a, tag, lane);
    if (slice == 0 && !collect_totals(a, t.hist, tag, tid, wave_s)) {   // for the caller (and for the counts below)
      if (lane == 0)
        give_up(a, avail_state);
      missing[1] = 1;
    }
    __syncthreads();
    LPLB_PLAN_STAMP(3);
    if (slice == 0)
      for (int e = tid; e < nl; e += kPlanThreads)
        a.totals[e] = t.hist[e];
    // With 16 chunks the table reads go eight at a time (all at once would not fit the registers), and the hashes are
    // finished before the wait: the compiler otherwise carries what they read (six registers a token) through the wait
    // and hashes behind it, which at 128 registers makes it split live ranges, and it has put the copy of such a split
    // (chunk 8's ids, in a variant of this kernel) behind the loop above ahead of the instruction that switches the
    // lanes on again: copied in no lane, lost in all.  97 registers this way at 8 ranks.  tests/test_host.py looks for such copies in the built library.
#pragma unroll
    for (int c = 0; c < K; ++c) {
      h[c] = SliceTokens<K>::hash(t, my_records, t.of_wave + wave_s * R, packed_expert(packed, c), c);
      if (K > 8 && c % 8 == 7) {
#pragma unroll
        for (int j = c - 7; j <= c; ++j)
          worked_out_here(h[j]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    LPLB_PLAN_STAMP(4);
    // ---- the LP's shares: every set's thread polls its own; value and tag arrive in the same word ----
    collect_shares(a, t, slice, gen, avail_state, tid);
    __syncthreads();
    LPLB_PLAN_STAMP(5);
    ok = missing[1] == 0;
    slice_has_read_all(a, slice, gen, wave_s);
  }
  LPLB_PLAN_STAMP(6);
  // ---- choose and store; if a wait ran out, every token goes to its original slot ----
  int32_t o[K];
#pragma unroll
  for (int c = 0; c < K; ++c) {
    const int e = packed_expert(packed, c);
    const PlanRoute rt = t.route[e];
    o[c] = rt.original();
    if (ok) {
      const RepEntry x = t.reps[rt.set];
      o[c] = h[c] >= x.expected ? x.replica : rt.original();
    }
    if (K > 8 && c % 8 == 7)
      __builtin_amdgcn_sched_barrier(0);
  }
  if (slice == 0 && a.physical_counts)
    plan_physical_counts(a, t, tl.physical_le0, ok, tid);
  store_chunks<K>(o, a.out, w0, end, lane);
  LPLB_PLAN_STAMP(7);
  LPLB_SLICE_STAMP(3);
}

// Slices of more than kLongestSlice indices (batches of more than 256 x 8192 on 256 CUs), and shorter ones with many replicated sets:
// the same exchange, with the tokens of a wave in passes of eight chunks.  The chain reads the indices twice and leaves the memory
// idle while its LP runs; here they are read once and stay in registers (11 bits of expert, 12 of ordinal among the wave's tokens of
// the set), and the ordinals are worked out while the LP is running.  At 8 ranks, as the chain and so: [1048576 x 8] 42 and 33.5-35.1 us;
// 2097153 indices in 256 slices 22.7 and 17.3, 4200000 30.5 and 23.3; 524289 in 64 slices 21.8 and 16.6, 1280000 27.9 and 22.4.
// Read 9.3 and written 11.2 us by kernels that do nothing else.  What bounds it: 10.5 us until the last index is
// counted, 4 until the LP has the totals, 5 until its shares are seen, then the choice and the stores (9) with the second half
// of the ordinals between them: a pass of those is about 1 us a wave, waits for the LDS and instructions in
// turn.  With every pass unrolled, for the registers' sake, the code is 58 KiB, nearly the instruction cache of two CUs.
// The histogram is per wave: what is in the waves before then costs nothing more than the sums, and
// a lookup of the set beside the histogram's update made the counting twice as long (the LDS serves them in turn).
// Ordinals: a bitmap of a chunk says who is ahead of a token in the chunk, a running count per (wave, set) what is ahead of the chunk,
// and a chunk's first token of a set adds to that.  The instructions do not go with the number of sets, and a row has 40 bytes where
// bitmaps of 16 chunks with their starting ordinals have 272, of which 64 sets take a CU.
// So, against the chain, 8 ranks in four and eight groups (64 and 128 sets): [131072 x 8] 18.2 -> 13.9 and 22.1 -> 15.9 us, [262144 x 8] 23.8 -> 16.5 and
// 29.3 -> 18.5, [196608 x 8] 15.8 -> 14.9 and 25.1 -> 17.9; 16 sets at [1048576 x 8] 32.3 -> 32.1.
// Against bitmaps of all 16 chunks (slices of 4097 to 8192): counts supplied, at 16, 32 and 64 sets [262144 x 8] 13.4 -> 12.7, 14.4 -> 13.7, 15.0 -> 15.0,
// [196608 x 8] 12.9 -> 12.6, 14.1 -> 13.7, 16.0 -> 15.0; own counts, which leave later here (loads and table of sets ahead of them), 15.1 -> 15.2, 15.7 -> 15.5
// and 14.35 -> 14.5, 14.7 -> 14.7, but 64 sets 16.0 -> 15.2.  Eight chunks (up to 4096) are the faster with bitmaps of all of them while
// those fit: [131072 x 8] 11.9 and 12.7, counts supplied 9.9 and 10.1.
template <int GM, int DM, bool EXACT>
__global__ __launch_bounds__(kPlanThreads, 2 * plan_workgroups_per_cu(GM)) void plan_of_long_slices(PlanArgs a) {
  constexpr int K = kLongChunks;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  __shared__ int rep_of_edge_all[kLpsPerWorkgroup * kWave];
  const int nl = a.sh.n_logical, R = a.n_rep;
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave_s = __builtin_amdgcn_readfirstlane(tid / kWave);   // wave-uniform
  const int pid = blockIdx.x;
  fetch_arguments_now(a.idx, a.unit_blocks, a.sh.G, a.solve.workload, a.solve.n_group, a.solve.tagged_result, a.sync);
  unsigned long long gen_and_poison = agent_load(reinterpret_cast<const unsigned long long *>(a.sync));
  if (pid < a.n_lp_workgroups) {
    lp_workgroup<GM, DM, EXACT>(a, smem_raw, rep_of_edge_all, gen_and_poison, tid, lane, wave_s);
    return;
  }
  const int slice = pid - a.n_lp_workgroups;
  const SliceTables t = carve_tables<0>(smem_raw, nl, R);
  int *const missing = t.missing;
  const int hist_len = 2 * a.hist_words, rows_bytes = (R + 1) * kRankRowBytes;
  // [waves][R + 1][kRankRowBytes], [waves][hist_len], [n_logical + 1]
  unsigned char *my_rows = t.records + wave_s * rows_bytes;
  int32_t *wave_hists = reinterpret_cast<int32_t *>(t.records + kPlanWaves * rows_bytes);
  int32_t *my_hist = wave_hists + wave_s * hist_len;
  unsigned char *set_of_expert = reinterpret_cast<unsigned char *>(wave_hists + kPlanWaves * hist_len);   // four to a word: lanes rarely meet in a bank
  const int64_t begin = slice_begin(a.n, a.per, slice);
  const int64_t end = slice_begin(a.n, a.per, slice + 1);
  const int wave_len = (int)(a.per + kPlanThreads - 1) / kPlanThreads * kWave;   // this wave's indices, whole chunks
  const int64_t w0 = begin + (int64_t)wave_s * wave_len;
  const int last = (int)(min(end, w0 + wave_len) - 1 - w0);   // place of its last index; -1 and less: it has none
  const int passes = (wave_len + K * kWave - 1) / (K * kWave);
  LPLB_PLAN_STAMP(0);
  LPLB_SLICE_STAMP(0);
  __builtin_amdgcn_s_setprio(2);   // (to the end: its ordinals take longer than the LP beside them; [1048576 x 8] 33.3 us with and without a step back)

  const PlanTableLoads tl = issue_plan_table_loads(a, tid, wave_s, slice == 0 && a.physical_counts);
  // (places past the last repeat it: without a branch the loads of the next pass stay on their way while one is counted)
  const int64_t *mine = a.idx + w0;
  auto load_pass = [&](int64_t (&v)[K], int p) {
#pragma unroll
    for (int c = 0; c < K; ++c)
      v[c] = __builtin_nontemporal_load(mine + min((p * K + c) * kWave + lane, last));
  };
  int64_t raw[2][K];
  load_pass(raw[0], 0);
  for (int e = lane; e < hist_len; e += kWave)
    my_hist[e] = 0;
  for (int i = lane; i < rows_bytes / 8; i += kWave)
    reinterpret_cast<unsigned long long *>(my_rows)[i] = 0ull;
  clear_plan_tables<0>(t, tid);
  __syncthreads();
  enter_plan_tables(a, t, tl, tid, wave_s);
  __syncthreads();
  for (int e = tid; e <= nl; e += kPlanThreads)   // (read behind the next barrier)
    set_of_expert[e] = (unsigned char)(t.route[e].set ? t.route[e].set - 1 : R);   // (from 0 on here; of no set: R)
  LPLB_PLAN_STAMP(10);

  // ---- the tokens: every wave counts its own ----
  uint32_t token[kLongPasses * K];   // expert; later with the token's ordinal among the wave's tokens of its set in the high half
#pragma unroll
  for (int p = 0; p < kLongPasses; ++p) {
    load_pass(raw[(p + 1) & 1], min(p + 1, passes - 1));
#pragma unroll
    for (int c = 0; c < K; ++c) {
      const int64_t v = raw[p & 1][c];
      const bool valid = (uint64_t)v < (uint64_t)nl && (p * K + c) * kWave + lane <= last;   // -1, other negatives and too large ids fail
      token[p * K + c] = valid ? (uint32_t)v : (uint32_t)nl;
      if (valid)
        atomicAdd(&my_hist[token[p * K + c]], 1);
    }
    if (p + 1 >= passes)
      break;
  }
  __syncthreads();
  LPLB_PLAN_STAMP(8);
  LPLB_SLICE_STAMP(1);
  worked_out_here(gen_and_poison);
  const int gen = (int)(uint32_t)gen_and_poison;
  const bool poisoned = (gen_and_poison >> 32) != 0;
  const uint32_t tag = (uint32_t)gen + 1u;
  unsigned long long *avail_state = reinterpret_cast<unsigned long long *>(a.sync + kAvailAt) + (gen & 1);
  if (wave_s >= kPlanWaves / 2)   // (they publish sets and add up totals while the others are at their ordinals already)
    __builtin_amdgcn_s_setprio(3);
  if (!poisoned) {
    unsigned long long *set_rows = reinterpret_cast<unsigned long long *>(a.sync + kSetRowsAt);
    unsigned long long *hist_rows = reinterpret_cast<unsigned long long *>(a.sync + kHistRowsAt);
    constexpr int kHalf = kPlanThreads / 2;
    if (tid < kHalf) {
      for (int e2 = tid; e2 < a.hist_words; e2 += kHalf) {
        int2 both{0, 0};
#pragma unroll
        for (int w = 0; w < kPlanWaves; ++w) {
          const int2 of_wave = reinterpret_cast<const int2 *>(wave_hists + w * hist_len)[e2];
          both.x += of_wave.x;
          both.y += of_wave.y;
        }
        agent_store(hist_rows + slice * a.hist_words + e2, tagged_word(tag, (uint32_t)both.x | (uint32_t)both.y << 16));
      }
    } else {
      // lane = (word, set of its two, wave): what is in the waves before, and the word from the lane that has the last wave's
      for (int i = tid - kHalf; i < 16 * a.set_words; i += kHalf) {
        const int w = i % kPlanWaves, q = i / kPlanWaves, x = q < R ? expert_of_set(a, t, q + 1) : nl;
        const int own = x < nl ? wave_hists[w * hist_len + x] : 0;
        const int before = group_exclusive_scan<kPlanWaves>(own, w);
        if (q < R)
          t.of_wave[w * R + q + 1] = before;   // (in a long slice: in the waves before)
        const int first = row_shr<8>(before + own);
        if (i % 16 == 15)
          agent_store(set_rows + slice * a.set_words + i / 16, tagged_word(tag, (uint32_t)first | (uint32_t)(before + own) << 16));
      }
    }
  } else if (slice == 0 && tid == 0) {
    agent_add(a.sync + kTimeoutsAt, 1);   // one more plan that this block of words could not serve
  }
  LPLB_PLAN_STAMP(1);
  LPLB_SLICE_STAMP(2);
  if (!poisoned)
    add_up_published<true, Units::kTotals>(a, t, slice, tag, lane, wave_s, missing, t.block_sums);
  // ---- while the others' words are on their way: ordinals among the wave's tokens, pass by pass (the wave's own records: no barrier) ----
  __builtin_amdgcn_s_setprio(2);
  const uint32_t my_bit = 1u << lane % 32;
  const int my_half = lane / 32 * 4;
  auto rank_chunks = [&](uint32_t *mine) {
    uint32_t set[kRankChunks];
    unsigned char *row[kRankChunks];
    bool in_set[kRankChunks];
    // (all reads ahead of the first update: the compiler keeps their order, and each would be waited for)
#pragma unroll
    for (int c = 0; c < kRankChunks; ++c)
      set[c] = set_of_expert[mine[c]];
#pragma unroll
    for (int c = 0; c < kRankChunks; ++c) {
      row[c] = my_rows + __umul24(set[c], (uint32_t)kRankRowBytes);
      in_set[c] = set[c] < (uint32_t)R;
      if (in_set[c])
        atomicOr(reinterpret_cast<uint32_t *>(row[c] + c * 8 + my_half), my_bit);
    }
    SliceTokens<K>::own_slots_are_written();
    uint2 bits[kRankChunks];
#pragma unroll
    for (int c = 0; c < kRankChunks; ++c)
      bits[c] = *reinterpret_cast<const uint2 *>(row[c] + c * 8);
    uint32_t before[kRankChunks], so_far[kRankChunks];
#pragma unroll
    for (int c = 0; c < kRankChunks; ++c)
      before[c] = __builtin_amdgcn_mbcnt_hi(bits[c].y, __builtin_amdgcn_mbcnt_lo(bits[c].x, 0));
    // The LDS serves a wave's instructions in the order they were issued: a chunk's tokens read what the chunks before it have added.
#pragma unroll
    for (int c = 0; c < kRankChunks; ++c) {
      uint32_t *of_set = reinterpret_cast<uint32_t *>(row[c] + kRankChunks * 8);
      so_far[c] = *of_set;
      if (in_set[c] && before[c] == 0) {   // the chunk's first token of its set; its bitmap is empty again behind it
        __hip_atomic_fetch_add(of_set, (uint32_t)(__popc(bits[c].x) + __popc(bits[c].y)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        *reinterpret_cast<uint2 *>(row[c] + c * 8) = uint2{0, 0};
      }
    }
#pragma unroll
    for (int c = 0; c < kRankChunks; ++c) {
      mine[c] |= (so_far[c] + before[c]) << 16;   // (without a set: whatever is there)
      worked_out_here(mine[c]);
    }
  };
  auto rank_pass = [&](int p) {
#pragma unroll
    for (int c = 0; c < K; c += kRankChunks)
      rank_chunks(token + p * K + c);
  };
#pragma unroll
  for (int p = 0; p < kLongPasses / 2; ++p)
    if (p < passes)
      rank_pass(p);
  if (!poisoned)
    add_up_published<true, Units::kSets>(a, t, slice, tag, lane, wave_s, missing, t.block_sums);
  LPLB_PLAN_STAMP(11);
  if (poisoned)
    missing[0] = 1;
  __syncthreads();
  LPLB_PLAN_STAMP(2);
  LPLB_SLICE_STAMP(4);
  bool ok = missing[0] == 0;   // (the same in every thread)
  if (!ok && !poisoned && tid == 0)
    give_up(a, avail_state);
  int32_t *my_bases = t.of_wave + wave_s * R;
  if (ok) {
    for (int q = tid + 1; q <= R; q += kPlanThreads)
      set_total(t.reps[q], t.total[q]);
    for (int q = lane + 1; q <= R; q += kWave)
      my_bases[q] += t.before[q];
    if (slice == 0 && wave_s == kPlanWaves - 1 && a.arrived_word)
      say_that_all_arrived(a, tag, lane);
    if (slice == 0) {   // for the caller (and for the counts below)
      if (!collect_totals(a, t.hist, tag, tid, wave_s)) {
        if (lane == 0)
          give_up(a, avail_state);
        missing[1] = 1;
      }
      __syncthreads();
      for (int e = tid; e < nl; e += kPlanThreads)
        a.totals[e] = t.hist[e];
    }
    LPLB_PLAN_STAMP(3);
    LPLB_PLAN_STAMP(4);
    collect_shares(a, t, slice, gen, avail_state, tid);
    __syncthreads();
    LPLB_PLAN_STAMP(5);
    ok = missing[1] == 0;
    slice_has_read_all(a, slice, gen, wave_s);
  }
  LPLB_PLAN_STAMP(6);
  // ---- choose and store; if a wait ran out, every token goes to its original slot ----
  if (slice == 0 && a.physical_counts)
    plan_physical_counts(a, t, tl.physical_le0, ok, tid);
  int64_t *out = a.out + w0;
  auto store_pass = [&](int p) {
    int32_t o[K];
#pragma unroll
    for (int c = 0; c < K; ++c) {
      const uint32_t e = token[p * K + c] & 0xffffu, k = token[p * K + c] >> 16;
      const PlanRoute rt = t.route[e];
      o[c] = rt.original();
      if (ok) {
        const RepEntry x = t.reps[rt.set];   // (without a replica: stays whatever the hash)
        const int32_t h = ordinal_hash<true>(my_bases[rt.set] + (int32_t)k, x.total, x.magic);
        o[c] = h >= x.expected ? x.replica : rt.original();
      }
    }
    if ((p + 1) * K * kWave - 1 <= last) {
#pragma unroll
      for (int c = 0; c < K; ++c)
        __builtin_nontemporal_store((int64_t)o[c], out + (p * K + c) * kWave + lane);
    } else {
#pragma unroll
      for (int c = 0; c < K; ++c)
        if ((p * K + c) * kWave + lane <= last)
          __builtin_nontemporal_store((int64_t)o[c], out + (p * K + c) * kWave + lane);
    }
  };
  // (the second half's ordinals between the first half's stores, which take longer)
#pragma unroll
  for (int p = 0; p < kLongPasses; ++p) {
    if (p < passes)
      store_pass(p);
    if (p < kLongPasses / 2 && p + kLongPasses / 2 < passes)
      rank_pass(p + kLongPasses / 2);
  }
  LPLB_PLAN_STAMP(7);
  LPLB_SLICE_STAMP(3);
}

// A short batch that feeds the LP itself, as one workgroup: the LPs are solved by its first waves between the
// histogram and the choice.  Bound by the chain indices -> histogram (1.1 us) -> LP -> choice, of which the slices' form above adds
// two round trips through memory between slices and LP.  The LP reads the histogram where the tokens were counted; bitmaps, ordinals
// and where each set's share will be are worked out by the other waves while it runs, and those wait for each other by a count in
// LDS, since a barrier would wait for the LP.  (With the bitmaps marked by all waves ahead of the LP: [7 x 8] 6.75 instead of 6.4 us,
// [128 x 8] 7.0 and 6.7.)
// Up to as many indices as leave the LP waves, which come last in the order of the indices, without any at eight chunks a wave.
// One LP, in one workgroup / as slices: 3584 indices 7.6 / 8.9 us, 4096 9.7 / 8.9; two LPs, 3072 7.8 / 9.1, 3584 10.3 / 9.2; four, 2048
// 8.4 / 9.25, 2560 11.0 / 9.25; (16, 2) 3584 10.9 / 12.1, 4096 13.9 / 12.1; (32, 2) 3584 18.3 / 19.4, 4096 22.7 / 19.4.  With eight LPs
// every wave has one: 128 indices (two chunks in one wave) 8.5 / 9.2, 192 9.45 / 9.25.  Where the slices are refused, up to eight
// chunks in every wave.
constexpr int kSingleMaxLps = kPlanWaves;
constexpr int64_t kSingleMaxIndices = 8 * kPlanThreads;
constexpr int64_t single_max_indices(int n_lps) { return (n_lps < kPlanWaves ? 8 * (kPlanWaves - n_lps) : 2) * kWave; }
template <int GM, int DM, bool EXACT, int K>
__global__ __launch_bounds__(kPlanThreads, 2) void plan_in_one_workgroup(PlanArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  __shared__ int rep_of_edge_all[kSingleMaxLps * kWave];
  __shared__ float share_of[kSingleMaxLps * kWave];
  __shared__ int marked;   // waves whose tokens are in their bitmaps
  const int nl = a.sh.n_logical, R = a.n_rep;
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave_s = __builtin_amdgcn_readfirstlane(tid / kWave);
  fetch_arguments_now(a.idx, a.unit_blocks, a.sh.G, a.solve.workload, a.solve.n_group, a.solve.tagged_result, a.sync);
  // LDS: the LP waves' areas, the slice's tables
  constexpr size_t kLpArea = plan_lp_area_bytes<GM, DM>();
  const int n_lps = a.solve.n_units;
  const SliceTables t = carve_tables<K>(smem_raw + n_lps * kLpArea, nl, R);
  const int turn = (wave_s - n_lps) & (kPlanWaves - 1);   // this wave's place in the order of the indices
  auto records_of = [&](int place) { return t.records + (size_t)place * ((R + 1) * rank_record_bytes_single(K)); };
  unsigned char *my_records = records_of(turn);
  const uint32_t n = (uint32_t)a.n, w0 = turn * (K * kWave);
  const bool has_tokens = w0 < n;
  const int waves_with_tokens = (int)((n + K * kWave - 1) / (K * kWave));
  int64_t raw[K];
  load_chunks<K>(raw, a.idx, w0, n, lane);
  const PlanTableLoads tl = issue_plan_table_loads(a, tid, wave_s, a.physical_counts);
  LPLB_PLAN_STAMP(0);
  uint32_t packed[(K + 1) / 2];
  // (called by the LP waves once their own table loads are on their way)
  auto count_the_tokens = [&]() -> bool {
    clear_plan_tables<K>(t, tid);
    if (tid == 0)
      marked = 0;
    __syncthreads();
    enter_plan_tables(a, t, tl, tid, wave_s);
    mask_chunks<K>(raw, w0, n, lane);
    SliceTokens<K>::count(a, t, raw, packed);
    __syncthreads();
    if (has_tokens) {
      SliceTokens<K>::mark(a, t, my_records, packed, lane);
      for (int q = lane + 1; q <= R; q += kWave) {   // (every wave enters the same values)
        const SetOfPlan s = set_of_plan(a, q - 1);
        set_total(t.reps[q], t.hist[expert_of_set(a, t, q)]);
        t.reps[q].expected = s.ep_rank * a.sh.D + s.d;   // until the shares are there: where its share will be
      }
      wave_arrives(&marked, lane);
    }
    LPLB_PLAN_STAMP(8);
    return true;
  };
  if (wave_s < n_lps) {
    unsigned char *area = smem_raw + wave_s * kLpArea;
    SolveArgs sa = a.solve;
    sa.shares_in_lds = share_of;
    sa.gw_out = nullptr;   // (written below, by waves that do not solve)
    const int n_ok = solve_lps<GM, DM, EXACT, 1, 1, true>(sa, wave_s, reinterpret_cast<float *>(t.hist), rep_of_edge_all + wave_s * kWave,
                                                    reinterpret_cast<double *>(area),
                                                    reinterpret_cast<float *>(area + lp_pivot_doubles<GM, DM>() * sizeof(double)),
                                                    count_the_tokens);
    if (lane == 0 && n_ok > 0)
      atomicAdd(a.avail, n_ok);
  } else {
    count_the_tokens();
  }
  // The totals and the normalised counts go out while the LPs are solved.
  if (wave_s >= n_lps || n_lps == kPlanWaves) {
    const int first = n_lps == kPlanWaves ? 0 : n_lps * kWave;
    int32_t most = 0;
    for (int i = 4 * lane; i < nl; i += 4 * kWave) {
      const i32x4 c = *reinterpret_cast<const i32x4 *>(t.hist + i);
      most = max(max(most, max(c.x, c.y)), max(c.z, c.w));
    }
    const float wmax = wave_max_of_groups<true, true>((float)most);
    for (int e = tid - first; e < nl; e += kPlanThreads - first) {
      const int32_t count = t.hist[e];
      a.totals[e] = count;
      a.solve.gw_out[e] = (float)count / wmax;
    }
  }
  int32_t h[K];
  if (has_tokens) {
    wait_for_waves(&marked, waves_with_tokens);
    SliceTokens<K>::starts_of_batch(a, my_records, lane, turn, records_of);
#pragma unroll
    for (int c = 0; c < K; ++c)
      h[c] = SliceTokens<K>::hash(t, my_records, nullptr, packed_expert(packed, c), c);
  }
  if (wave_s < n_lps) {
    wait_for_waves(&marked, waves_with_tokens);   // (and its own shares have been stored)
    const int per_group = a.sh.G * a.sh.C * a.sh.D;
    for (int i = lane; i < per_group; i += kWave) {
      RepEntry &x = t.reps[wave_s * per_group + i + 1];
      x.expected = expected_on_original(share_of[x.expected], x.total);
    }
  }
  __syncthreads();
  LPLB_PLAN_STAMP(2);
  if (has_tokens) {
    int32_t o[K];
#pragma unroll
    for (int c = 0; c < K; ++c) {
      const PlanRoute rt = t.route[packed_expert(packed, c)];
      const RepEntry x = t.reps[rt.set];
      o[c] = h[c] >= x.expected ? x.replica : rt.original();
    }
    store_chunks<K>(o, a.out, w0, n, lane);
  }
  if (a.physical_counts)
    plan_physical_counts(a, t, tl.physical_le0, true, tid);
  LPLB_PLAN_STAMP(7);
}

// ---- long batches that feed the LPs themselves: scan over the slices and LPs as one launch behind the histogram ----
// The first workgroup solves up to four LPs; the others turn the histogram's rows into running sums, as
// prefix_over_slices does, and hand every expert's total over in the vector that will hold the normalised counts
// (kNoTotal until then: set by the histogram's launch, so nothing outlives the plan).  Against two launches the LP's
// table loads and the second launch's start are off the path: [1048576 x 8] 44.2 -> 42.3 us for the whole
// plan.  The waiting workgroup is one in a grid of a few, and those it waits for wait for nobody; its wait is bounded
// all the same (other kernels may keep the rest of the grid off the GPU).  If it runs out it is counted, the LPs are not
// solved, nothing is added to avail_num, every share is 0.5 and global_workload is NaN: a total that comes later replaces
// kNoTotal only.
struct ScanSolveArgs {
  SolveArgs solve;
  int32_t *counts;   // [n_blocks][n_experts]
  int32_t *totals;   // the words of solve.gw_out
  int n_blocks, max_polls;
  int expected_blocks;   // = n_blocks unless a fault is injected
  int *timeouts;
};
constexpr int kScanSolveLps = kScanThreads / kWave;
template <int GM, int DM, bool EXACT> __global__ __launch_bounds__(kScanThreads) void scan_and_solve(ScanSolveArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  __shared__ int rep_of_edge_all[kScanSolveLps * kWave];
  __shared__ int missing;
  __shared__ ScanLds scan_lds;
  const int nl = a.solve.n_experts;
  if (blockIdx.x > 0) {
    scan_columns(a.counts, a.n_blocks, nl, blockIdx.x - 1, scan_lds, [&](int e, int32_t sum) { agent_replace(a.totals + e, kNoTotal, sum); });
    return;
  }
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave_s = __builtin_amdgcn_readfirstlane(tid / kWave);
  constexpr size_t kLpArea = plan_lp_area_bytes<GM, DM>();
  float *staged = reinterpret_cast<float *>(smem_raw + a.solve.n_units * kLpArea);
  if (tid == 0)
    missing = 0;
  __syncthreads();
  const bool can_come = a.expected_blocks == a.n_blocks;   // (an injected fault: one slice never comes)
  auto counts_have_come = [&]() -> bool {
    if (tid < 4)   // the zeros behind the counts
      reinterpret_cast<int32_t *>(staged)[nl + tid] = 0;
    for (int e = tid; e < nl; e += kScanThreads) {
      int32_t sum = kNoTotal;
      for (int polls = 0; polls < a.max_polls && (sum = agent_load(a.totals + e)) == kNoTotal; ++polls)
        __builtin_amdgcn_s_sleep(1);
      if (sum == kNoTotal || !can_come)
        missing = 1;
      reinterpret_cast<int32_t *>(staged)[e] = sum;
    }
    __syncthreads();   // (from here on the totals may be overwritten by the normalised counts)
    return missing == 0;
  };
  if (wave_s >= a.solve.n_units) {
    counts_have_come();
    return;
  }
  unsigned char *area = smem_raw + wave_s * kLpArea;
  const int n_ok = solve_lps<GM, DM, EXACT, 1, 1, true>(a.solve, wave_s, staged, rep_of_edge_all + wave_s * kWave,
                                                  reinterpret_cast<double *>(area),
                                                  reinterpret_cast<float *>(area + lp_pivot_doubles<GM, DM>() * sizeof(double)),
                                                  counts_have_come);
  if (n_ok > 0 && lane == 0)
    atomicAdd(a.solve.avail, n_ok);
  if (n_ok < 0) {   // the wait ran out
    for (int j = lane; j < a.solve.G * a.solve.D; j += kWave)
      a.solve.result[wave_s * a.solve.G * a.solve.D + j] = 0.5f;
    if (wave_s == 0) {
      for (int e = lane; e < nl; e += kWave)
        agent_store(a.totals + e, 0x7fc00000);   // NaN
      if (lane == 0)
        agent_add(a.timeouts, 1);
    }
  }
}

// ---- host side: which variant ----
template <int GM, int DM> static int launch_scan_and_solve(const ScanSolveArgs &a, hipStream_t s) {
  const size_t lds = a.solve.n_units * plan_lp_area_bytes<GM, DM>() + counts_bytes(a.solve.n_experts);
  static_assert(kScanSolveLps * plan_lp_area_bytes<GM, DM>() + counts_bytes(kMaxPlanExperts) <= 62 * 1024, "LDS of a kernel without asking for more");
  const dim3 grid(1 + (a.solve.n_experts + kScanCols - 1) / kScanCols), block(kScanThreads);
  if (a.solve.G == GM && a.solve.D == DM)
    launch(scan_and_solve<GM, DM, true>, grid, block, lds, s, a);
  else
    launch(scan_and_solve<GM, DM, false>, grid, block, lds, s, a);
  LPLB_HIP_TRY(hipGetLastError());
  return LPLB_OK;
}
// K: as in plan_in_one_launch; 0: long slices.
template <int GM, int DM, bool EXACT, int K>
static int launch_plan_slices(PlanArgs &a, hipStream_t s, bool *done) {
  const size_t lds_slice = K > 0 ? plan_slice_lds_bytes<K>(a.sh.n_logical, a.n_rep)
                           : a.per <= kLongestSlice || (GM <= 8 && a.n_rep <= kFewSets)
                               ? long_slice_lds_bytes(a.sh.n_logical, a.n_rep, a.hist_words)
                               : longest_slices_lds_bytes(a.sh.n_logical, a.n_rep, a.hist_words);
  // LP workgroups: their waves' working areas, then the counts (one copy per LP, or one for all of the batch's own)
  const size_t lp_areas = kLpsPerWorkgroup * plan_lp_area_bytes<GM, DM>();
  const size_t one_copy = counts_bytes(a.sh.n_logical);
  const size_t all_copies = (size_t)min(a.solve.n_units, kLpsPerWorkgroup) * one_copy;
  const size_t lds = max(lds_slice, lp_areas + (a.local_counts ? one_copy : all_copies));
  a.solve.staged_stride = (int)(one_copy / sizeof(int32_t));
  if (lds > (size_t)kPlanLdsLimit || (K == 0 && a.n_rep > kLongMaxSets))
    return LPLB_OK;
  static KernelFootprint footprint;
  if constexpr (K > 0)
    return launch_plan(plan_in_one_launch<GM, DM, EXACT, K>, footprint, true, a, lds, s, done);
  else
    return launch_plan(plan_of_long_slices<GM, DM, EXACT>, footprint, true, a, lds, s, done);
}
template <int GM, int DM, bool EXACT, int K> static int launch_plan_single(PlanArgs &a, hipStream_t s, bool *done) {
  const size_t lds = a.solve.n_units * plan_lp_area_bytes<GM, DM>() + plan_slice_lds_bytes<K>(a.sh.n_logical, a.n_rep);
  if (lds > (size_t)kPlanLdsLimit)
    return LPLB_OK;
  a.solve.staged_stride = a.sh.n_logical;
  static KernelFootprint footprint;
  return launch_plan(plan_in_one_workgroup<GM, DM, EXACT, K>, footprint, false, a, lds, s, done);
}
template <int GM, int DM, bool EXACT> static int launch_plan_shape(PlanArgs &a, hipStream_t s, bool *done) {
  if (a.n_lp_workgroups == 0) {   // as few chunks per wave as leave the LP waves without tokens
    const int64_t per_chunk = (kPlanWaves - min(a.solve.n_units, kPlanWaves - 1)) * kWave;
    return a.n <= 2 * per_chunk ? launch_plan_single<GM, DM, EXACT, 2>(a, s, done)
           : a.n <= 4 * per_chunk ? launch_plan_single<GM, DM, EXACT, 4>(a, s, done)
                                  : launch_plan_single<GM, DM, EXACT, 8>(a, s, done);
  }
  // Slices of up to 8192 indices in passes too, where there are many: whose tables fit no other way, or not twice on a CU; with 16
  // chunks per wave also those that are the faster for it (plan_of_long_slices).
  const bool many = a.n_slices >= kFewestSlicesInPasses;
  const auto in_passes = [&]() { return launch_plan_slices<GM, DM, EXACT, 0>(a, s, done); };
  if (a.per > kLongestSlice)
    return in_passes();
  int rc = LPLB_OK;
  if (a.per > 8 * kPlanThreads && many && (!a.local_counts || a.n_rep > kFewSets)) {
    rc = in_passes();
    if (rc != LPLB_OK || *done)
      return rc;
  }
  rc = a.per <= kPlanThreads       ? launch_plan_slices<GM, DM, EXACT, 1>(a, s, done)
       : a.per <= 2 * kPlanThreads ? launch_plan_slices<GM, DM, EXACT, 2>(a, s, done)
       : a.per <= 4 * kPlanThreads ? launch_plan_slices<GM, DM, EXACT, 4>(a, s, done)
       : a.per <= 8 * kPlanThreads ? launch_plan_slices<GM, DM, EXACT, 8>(a, s, done)
                                   : launch_plan_slices<GM, DM, EXACT, 16>(a, s, done);
  return rc == LPLB_OK && !*done && many ? in_passes() : rc;
}
template <int GM, int DM> static int launch_plan_padded_or_not(PlanArgs &a, hipStream_t s, bool *done) {
  return a.sh.G == GM && a.sh.D == DM ? launch_plan_shape<GM, DM, true>(a, s, done) : launch_plan_shape<GM, DM, false>(a, s, done);
}

} // namespace lplb
