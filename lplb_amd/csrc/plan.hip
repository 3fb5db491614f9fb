// Whole plan in one call: histogram -> LP solve -> redirect on one stream, as one kernel launch
// (plan_kernel.h) where that applies, else as the three entry points' kernels one after the other (histogram,
// scan, LP, redirect).  With the global counts supplied the chain's LP does not depend on this GPU's histogram:
// it is enqueued first and the histogram launch does not wait for it (it still starts after everything the LP
// launch waited for).
#include "plan_admit.h"
#include "plan_kernel.h"
#include <mutex>
#include <stdio.h>

namespace lplb {

static __device__ __attribute__((aligned(4096))) int g_plan_sync[kSyncInts];
// Slices of the one-launch plan, in indices (the longest: kLongestSlice).  While a wave adds up the counts of all slices (64) and the GPU
// has no other plan, as short as 512 (run [2048 x 8] 9.2 -> 9.0 us, [4096 x 8] 9.3 -> 9.15, counts supplied [1024 x 8] 6.9 -> 6.75, at 32 ranks
// [2048 x 8] 17.2 -> 16.75; [8192 x 8] in 128 slices 9.4 as in 64).  They take twice the workgroups, which a captured plan would keep for good
// and other streams' plans would be refused for, ten times what is gained: of 16 ranks and [4096 x 8] six captured plans instead of eight
// ran as one launch, of 32 ranks, where a CU holds one workgroup, three instead of six.
constexpr int64_t kShortestSlice = 1024, kShortestSliceAlone = 512;
static std::atomic<bool> g_cooperative{true};   // any thread may flip it while others plan
static std::atomic<long long> g_one_launch_plans{0};
// Test hook (lplb_plan_inject_fault): the next launch with a wait in it (one-launch plan, or scan and LP of a long
// batch) expects this many slices more than its grid has and gives up after this many polls.
static std::atomic<int> g_fault_extra_slices{0}, g_fault_max_polls{0};

// ---- host side: which launches may run as one kernel (the rules: plan_admit.h) ----
struct PlanDevice {
  int *sync = nullptr;
  int *arrived = nullptr;       // pinned host memory, one word per slot, written by the kernels (see PlanArgs); null until a
                                // plan is launched outside a capture, inside which it cannot be allocated
  int n_cus = 0;
  PlanAdmission<kSyncSlots> admission;
};
static std::mutex g_plan_guard;
static PlanDevice g_plan_devices[64];

// The current device and the address of its words (nothing is allocated: a captured call may be the first one).
static int plan_words(int **out, int *ordinal) {
  static std::atomic<int *> known[64];
  int dev = -1;
  LPLB_HIP_TRY(hipGetDevice(&dev));
  LPLB_REQUIRE(dev >= 0 && dev < 64, LPLB_EUNSUPPORTED, "plan: device ordinal %d", dev);
  int *words = known[dev].load(std::memory_order_acquire);
  if (!words) {
    LPLB_HIP_TRY(hipGetSymbolAddress(reinterpret_cast<void **>(&words), HIP_SYMBOL(g_plan_sync)));
    known[dev].store(words, std::memory_order_release);
  }
  *out = words;
  *ordinal = dev;
  return LPLB_OK;
}

// Looks the per-device state up.
static int plan_device(PlanDevice **out, int *ordinal = nullptr) {
  int *words = nullptr;
  int dev = -1;
  const int rc = plan_words(&words, &dev);
  if (rc != LPLB_OK)
    return rc;
  PlanDevice &d = g_plan_devices[dev];
  if (ordinal)
    *ordinal = dev;
  static std::mutex first_use;
  std::lock_guard<std::mutex> lock(first_use);
  if (!d.sync) {
    d.n_cus = current_device_cu_count();
    LPLB_REQUIRE(d.n_cus > 0, LPLB_EHIP, "plan: cannot read the CU count of device %d", dev);
    d.sync = words;
  }
  *out = &d;
  return LPLB_OK;
}

// The first thing that a stream runs in a block it has taken over: the launch of the stream before has arrived, but
// some of its slices may still have to read their shares.  Its workgroups are resident and wait for nothing else, so
// this ends; should it not, the block is switched off as after any wait that ran out.  (A replay of a captured
// takeover finds the words at this number or a later one.)
__global__ void wait_for_last_user(int *sync, int slices, int lps, int seq, int max_polls) {
  const int i = threadIdx.x;
  bool done = i >= slices + lps;
  const auto reached = [seq](int number) { return ((number - seq) & kSeqMask) <= kSeqMask / 2; };
  for (int polls = 0; polls < max_polls && !done; ++polls) {
    if (i == 0) {   // its last stores have landed, too
      const unsigned long long advanced = agent_load(reinterpret_cast<const unsigned long long *>(sync + kAdvancedAt));
      const int gen = (int)(uint32_t)advanced;
      done = reached((int)(advanced >> 32)) && agent_load(sync + kGenAt) == gen &&
             agent_load(reinterpret_cast<const unsigned long long *>(sync + kAvailAt) + (gen & 1)) == 0;
    } else {
      done = reached(agent_load(sync + kDoneAt + (i < slices ? i : kMaxSlices + i - slices) * kDoneStride));
    }
    done = done || agent_load(sync + kPoisonAt) != 0;   // (a block that is off, or is switched off now, is not read)
    __builtin_amdgcn_s_sleep(1);
  }
  if (!done) {
    agent_add(sync + kTimeoutsAt, 1);
    agent_store(sync + kPoisonAt, 1);
  }
}

// Workgroups of one kernel variant that fit a CU: bounded by the vector registers (512 per
// SIMD lane, allocated in blocks of 8, at most 8 waves per SIMD) and by the LDS (160 KiB per
// CU).  Worked out from the kernel's own attributes; the runtime's occupancy query changes
// its answer once a kernel has been allowed more than 64 KiB of dynamic LDS.
static int workgroups_per_cu(const void *kernel, KernelFootprint &known, int waves, size_t lds) {
  int regs = known.regs.load(std::memory_order_acquire);
  if (regs < 0) {
    hipFuncAttributes attr;
    if (hipFuncGetAttributes(&attr, kernel) != hipSuccess || attr.numRegs <= 0)
      return 0;
    known.static_lds.store((int)attr.sharedSizeBytes, std::memory_order_relaxed);
    regs = attr.numRegs;
    known.regs.store(regs, std::memory_order_release);
  }
  const int per_wave = (regs + 7) / 8 * 8;
  const int waves_per_simd = min(8, 512 / per_wave);
  const int by_registers = waves_per_simd * 4 / waves;
  const int by_lds = (int)((size_t)(160 * 1024) / (lds + (size_t)known.static_lds.load(std::memory_order_relaxed) + 256));
  return min(by_registers, by_lds);
}

static bool cut_for_a_plan_alone(const PlanArgs &a) { return a.per <= kShortestSliceAlone && a.n > kShortestSliceAlone; }

// Launches one variant, if the whole grid fits the GPU beside the plans that are still executing (a kernel whose
// workgroups do not wait for others always does).  *done = false: it does not; nothing was enqueued.
int launch_plan(PlanKernel kernel, KernelFootprint &footprint, bool waits_for_others, PlanArgs &a, size_t lds, hipStream_t s,
                bool *done) {
  PlanDevice *d = nullptr;
  int dev = -1;
  int rc = plan_device(&d, &dev);
  if (rc != LPLB_OK)
    return rc;
  if (lds > 64 * 1024 && !(footprint.much_lds_allowed.load(std::memory_order_acquire) >> dev & 1)) {
    LPLB_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kPlanLdsLimit));
    footprint.much_lds_allowed.fetch_or(1ull << dev, std::memory_order_release);
  }
  const int n_workgroups = max(a.n_slices + a.n_lp_workgroups, 1);
  std::unique_lock<std::mutex> lock(g_plan_guard, std::defer_lock);
  PlanAdmission<kSyncSlots>::Admitted admitted;
  bool capturing = false;
  if (waits_for_others) {
    const int fit = workgroups_per_cu(reinterpret_cast<const void *>(kernel), footprint, kPlanWaves, lds);
    if (fit <= 0 || n_workgroups > (int)(kResidencyBudget * fit * d->n_cus))
      return LPLB_OK;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &capture) != hipSuccess)
      capture = hipStreamCaptureStatusNone;
    capturing = capture == hipStreamCaptureStatusActive;
    const float cost = (float)n_workgroups / (float)(fit * d->n_cus);
    lock.lock();   // held over the launch: admission and launch order agree
    if (!capturing && !d->arrived) {
      LPLB_HIP_TRY(hipHostMalloc(reinterpret_cast<void **>(&d->arrived), kSyncSlots * sizeof(int), hipHostMallocDefault));
      for (int i = 0; i < kSyncSlots; ++i)
        d->arrived[i] = 0;
    }
    admitted = d->admission.admit(s, cost, capturing, d->arrived, cut_for_a_plan_alone(a));
    if (admitted.slot < 0)
      return LPLB_OK;
    a.sync = d->sync + (size_t)admitted.slot * kSlotInts;
    if (admitted.wait_slices > 0) {
      hipLaunchKernelGGL(wait_for_last_user, dim3(1), dim3(kMaxSlices + kMaxLps), 0, s, a.sync, admitted.wait_slices,
                         admitted.wait_lps, admitted.wait_seq, kDefaultMaxPolls);
      LPLB_HIP_TRY(hipGetLastError());
    }
    a.solve.tagged_result = reinterpret_cast<unsigned long long *>(a.sync + kSharesAt);
    a.solve.tagged_copies = a.n_share_copies;
    a.solve.tagged_stride = kMaxShares;
    a.expected_slices = a.n_slices + g_fault_extra_slices.exchange(0);
    const int fault_polls = g_fault_max_polls.exchange(0);
    a.max_polls = fault_polls > 0 ? fault_polls : kDefaultMaxPolls;
    // (a captured launch keeps its share of the GPU until it is forgotten, and reports nothing)
    a.seq = admitted.seq;
    a.arrived_word = capturing ? nullptr : d->arrived + admitted.slot;
  }
  launch(kernel, dim3(n_workgroups), dim3(kPlanThreads), lds, s, a);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess)
    return fail(LPLB_EHIP, "plan: launch failed: %s", hipGetErrorString(err));
  if (waits_for_others)
    d->admission.launched(admitted, capturing, a.n_slices, a.solve.n_units);
  g_one_launch_plans.fetch_add(1, std::memory_order_relaxed);
  *done = true;
  return LPLB_OK;
}

// LP shapes that are built here: (8, 1) (8, 2) (8, 4) (16, 1) (16, 2) (32, 1) (32, 2) and what pads into them
static bool lp_shape_is_built(int G, int D) { return G <= 8 ? D <= 4 : G <= 32 && D <= 2; }

// The shortest of 1024, 2048, 4096, 8192 indices per slice (or of 512 and those) with which at most `most` slices, which is no more than
// kMaxSlices, than the caller allows and than the GPU holds at once, cover the batch.  false: they cannot.
static bool cut_into_slices(PlanArgs &a, int64_t shortest, int most) {
  int64_t len = shortest;
  while (len < kLongestSlice && (a.n + len - 1) / len > (len < kShortestSlice ? min(most, kUnitSlices) : most))
    len *= 2;
  a.per = slice_len(a.n, (int)min((a.n + len - 1) / len, (int64_t)most));
  // Past that as many long slices as there may be, unless these are few: a caller that allows few workgroups keeps the chain.
  // (So many may turn out not to be resident at once: up to 16 ranks `most` is for two per CU, and the tables of 32 sets and more
  // leave room for one.  launch_plan refuses those.)
  if (a.per > kLongestSlice && (a.per > kLongestOfLongSlices || most < kFewestLongSlices))
    return false;
  const int n = a.n_slices = (int)((a.n + a.per - 1) / a.per);   // (rounding the length up may have emptied the last ones)
  a.adder_words = 8;
  while (a.adder_words * n < a.hist_words)
    a.adder_words *= 2;
  a.adders = (a.hist_words + a.adder_words - 1) / a.adder_words;
  a.n_share_copies = 1;
  while (a.n_share_copies < kShareCopies && a.n_share_copies * 8 < n)
    a.n_share_copies *= 2;
  a.unit_lanes_log2 = n > 32 ? 2 : n > 16 ? 3 : n > 8 ? 4 : n > 4 ? 5 : 6;
  a.unit_blocks = (n + kUnitSlices - 1) / kUnitSlices;
  a.unit_block_bits = a.unit_blocks > 2 ? 2 : a.unit_blocks - 1;
  return true;
}

// Tries the one-launch plan.  *done = false: shape or size outside what it covers, or no
// room on the GPU right now; nothing was enqueued.
static int try_one_launch(const int64_t *idx, int64_t n_elements, const int32_t *counts, const int32_t *r2o,
                          const int32_t *o2r, const int32_t *phy2log, int n_group, int G, int D, int C, int P,
                          int n_blocks, int32_t *counts_by_block, float *global_workload, float *o_weight,
                          int32_t *avail_num, int64_t *out, int32_t *physical_counts, int step_rule, int n_steps,
                          hipStream_t s, bool *done) {
  *done = false;
  const int L = P - D * C, n_fixed = L - D * C;
  const int n_logical = n_group * G * L, n_rep = n_group * G * C * D;
  if (!g_cooperative || n_elements <= 0 || n_rep == 0)
    return LPLB_OK;
  if (!lp_shape_is_built(G, D) || n_group > kLpsPerWorkgroup * kMaxLpWorkgroups || n_group * G * D > kMaxShares || global_workload == nullptr ||
      n_logical > kMaxPlanExperts || n_group * G * P >= 65536)
    return LPLB_OK;
  PlanArgs a{};   // every field the host does not set below is zero
  a.idx = idx; a.n = n_elements;
  a.set_words = 8;
  while (2 * a.set_words < n_rep)
    a.set_words *= 2;
  a.hist_words = ((n_logical + 1) / 2 + 7) / 8 * 8;
  a.o2r = o2r; a.phy2log = phy2log;
  a.totals = counts_by_block + (int64_t)(n_blocks - 1) * n_logical; a.out = out;
  a.physical_counts = physical_counts; a.avail = avail_num;
  a.sh = RedirectShape{n_logical, n_group * G, G, D, C, L, P};
  a.n_rep = n_rep;
  a.magic_L = fast_div_magic((uint32_t)L); a.magic_cd = fast_div_magic((uint32_t)(C * D));
  a.magic_D = fast_div_magic((uint32_t)D); a.magic_G = fast_div_magic((uint32_t)G);
  a.local_counts = counts == nullptr;
  SolveArgs &sa = a.solve;
  sa.workload = counts; sa.gw_out = global_workload; sa.r2o = r2o; sa.phy2log = phy2log;
  sa.avail = avail_num; sa.result = o_weight; sa.n_group = n_group; sa.G = G; sa.D = D; sa.C = C;
  sa.n_fixed = n_fixed; sa.n_experts = n_logical; sa.step_rule = step_rule; sa.n_steps = n_steps;
  sa.n_units = n_group; sa.counts_by_caller = counts == nullptr;
  sa.clocks = debug_clocks();
  const auto launch_variant = G <= 8 ? launch_plan_up_to_8 : G <= 16 ? launch_plan_up_to_16 : launch_plan_up_to_32;
  // A short batch that feeds the LPs itself is one workgroup, unless its tables do not fit a CU (or a fault is to be
  // injected, which needs workgroups that wait): up to single_max_indices, where that is the faster form, ahead of the slices, and up to
  // kSingleMaxIndices where those are refused: it needs no room and no block of words, and is no slower than the chain (4096 indices, one
  // LP 9.7 / 12.3 us, four 12.7 / 13.0, of 16 ranks 13.9 / 15.4, of 32 22.7 / 23.4).
  const bool single = counts == nullptr && n_group <= kSingleMaxLps && n_elements <= kSingleMaxIndices && g_fault_extra_slices == 0;
  const bool single_first = single && n_elements <= single_max_indices(n_group);
  const auto try_single = [&]() -> int {
    a.n_lp_workgroups = 0;
    a.n_slices = 1;
    a.per = slice_len(n_elements, 1);
    return launch_variant(a, s, done);
  };
  int rc = single_first ? try_single() : LPLB_OK;
  if (rc != LPLB_OK || *done)
    return rc;
  a.n_lp_workgroups = (n_group + kLpsPerWorkgroup - 1) / kLpsPerWorkgroup;
  const int resident = (int)(kResidencyBudget * plan_workgroups_per_cu(G) * current_device_cu_count());
  const int most = min(min(n_blocks, kMaxSlices), resident - a.n_lp_workgroups);
  if (most >= 1 && cut_into_slices(a, kShortestSliceAlone, most) && cut_for_a_plan_alone(a))
    rc = launch_variant(a, s, done);
  if (rc == LPLB_OK && !*done && most >= 1 && cut_into_slices(a, kShortestSlice, most))
    rc = launch_variant(a, s, done);
  return rc == LPLB_OK && !*done && single && !single_first ? try_single() : rc;
}

} // namespace lplb

extern "C" int lplb_plan_set_cooperative(int enabled) {
  lplb::g_cooperative = enabled != 0;
  return LPLB_OK;
}

extern "C" int lplb_plan_forget_captured(lplb_stream_t stream) {
  using namespace lplb;
  PlanDevice *d = nullptr;
  const int rc = plan_device(&d);
  if (rc != LPLB_OK)
    return rc;
  std::lock_guard<std::mutex> lock(g_plan_guard);
  d->admission.forget_captured(stream);
  return LPLB_OK;
}

extern "C" int lplb_plan_sync_timeouts(int *count) {
  using namespace lplb;
  LPLB_REQUIRE(count != nullptr, LPLB_EINVAL, "plan_sync_timeouts: null pointer");
  PlanDevice *d = nullptr;
  const int rc = plan_device(&d);
  if (rc != LPLB_OK)
    return rc;
  // Everything enqueued so far has ended after this, so a block that is switched off can be
  // cleared without a launch looking at it (the caller must not enqueue plans from other
  // threads meanwhile, as the header says).
  LPLB_HIP_TRY(hipDeviceSynchronize());
  LPLB_HIP_TRY(hipMemcpy(count, d->sync + kLooseTimeoutsAt, sizeof(int), hipMemcpyDeviceToHost));
  for (int slot = 0; slot < kSyncSlots; ++slot) {
    int *block = d->sync + (size_t)slot * kSlotInts;
    int head[kTimeoutsAt + 1] = {};
    LPLB_HIP_TRY(hipMemcpy(head, block, sizeof(head), hipMemcpyDeviceToHost));
    *count += head[kTimeoutsAt];
    if (head[kPoisonAt] != 0) {
      // back to the state of a block that has never been used; the failures stay counted, and the numbers of launches say
      // that all so far have ended (a captured wait_for_last_user asks for them whenever its graph is replayed)
      const int number = d->admission.number_of(slot);
      const int advanced[2] = {0, number};
      LPLB_HIP_TRY(hipMemset(block, 0, kTimeoutsAt * sizeof(int)));
      LPLB_HIP_TRY(hipMemset(block + kTimeoutsAt + 1, 0, (size_t)(kDoneAt - kTimeoutsAt - 1) * sizeof(int)));
      LPLB_HIP_TRY(hipMemcpy(block + kAdvancedAt, advanced, sizeof(advanced), hipMemcpyHostToDevice));
      LPLB_HIP_TRY(hipMemsetD32(reinterpret_cast<hipDeviceptr_t>(block + kDoneAt), number, kSlotInts - kDoneAt));
    }
  }
  LPLB_HIP_TRY(hipDeviceSynchronize());
  {
    std::lock_guard<std::mutex> lock(g_plan_guard);
    d->admission.device_is_idle();
  }
  return LPLB_OK;
}

namespace lplb {
// dst[0] = waits that ran out on this device so far, dst[1] = blocks of counters switched off right now
__global__ void report_plan_health(const int *sync, int32_t *dst) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    int timeouts = agent_load(sync + kLooseTimeoutsAt), off = 0;
    for (int slot = 0; slot < kSyncSlots; ++slot) {
      timeouts += agent_load(sync + (size_t)slot * kSlotInts + kTimeoutsAt);
      off += agent_load(sync + (size_t)slot * kSlotInts + kPoisonAt) != 0;
    }
    dst[0] = timeouts;
    dst[1] = off;
  }
}
} // namespace lplb

extern "C" int lplb_plan_poll_timeouts(int32_t *dst, lplb_stream_t stream) {
  using namespace lplb;
  LPLB_REQUIRE(dst != nullptr, LPLB_EINVAL, "plan_poll_timeouts: null pointer");
  PlanDevice *d = nullptr;
  const int rc = plan_device(&d);
  if (rc != LPLB_OK)
    return rc;
  launch(report_plan_health, dim3(1), dim3(kWave), 0, static_cast<hipStream_t>(stream), d->sync, dst);
  LPLB_HIP_TRY(hipGetLastError());
  return LPLB_OK;
}

extern "C" int lplb_plan_one_launch_count(long long *count) {
  LPLB_REQUIRE(count != nullptr, LPLB_EINVAL, "plan_one_launch_count: null pointer");
  *count = lplb::g_one_launch_plans.load(std::memory_order_relaxed);
  return LPLB_OK;
}

extern "C" int lplb_plan_inject_fault(int extra_slices_expected, int max_polls) {
  LPLB_REQUIRE(extra_slices_expected >= 0 && max_polls >= 0, LPLB_EINVAL, "plan_inject_fault: negative argument");
  lplb::g_fault_extra_slices = extra_slices_expected;
  lplb::g_fault_max_polls = max_polls;
  return LPLB_OK;
}

namespace lplb {

// The body of lplb_plan: argument checks, then the one-launch form or the chain.
static int plan_checked(const int64_t *idx, int64_t n_elements, const int32_t *global_counts, const int32_t *r2o,
                        const int32_t *o2r, const int32_t *phy2log, int n_group, int group_size, int dup_per_rank,
                        int n_combined_experts, int n_local_experts, int n_blocks, int32_t *counts_by_block,
                        float *global_workload, float *o_weight, int32_t *avail_num, int64_t *out,
                        int32_t *physical_counts, int step_rule, int n_steps, lplb_stream_t stream) {
  LPLB_REQUIRE(n_group > 0 && group_size > 0 && dup_per_rank > 0 && n_blocks > 0, LPLB_EINVAL,
               "plan: n_group=%d group_size=%d dup_per_rank=%d n_blocks=%d must be positive",
               n_group, group_size, dup_per_rank, n_blocks);
  const int L = n_local_experts - dup_per_rank * n_combined_experts;
  const int n_fixed = L - dup_per_rank * n_combined_experts;
  LPLB_REQUIRE(L > 0 && n_fixed >= 0 && n_combined_experts >= 0, LPLB_EINVAL,
               "plan: n_local_experts=%d does not fit %d x %d replicas", n_local_experts,
               dup_per_rank, n_combined_experts);
  LPLB_REQUIRE(counts_by_block != nullptr, LPLB_EINVAL, "plan: null counts_by_block");
  LPLB_REQUIRE(n_elements >= 0 && n_elements <= INT32_MAX && (idx || n_elements == 0), LPLB_EINVAL,
               "plan: bad idx / n_elements=%lld", (long long)n_elements);
  LPLB_REQUIRE((reinterpret_cast<uintptr_t>(idx) & 7) == 0, LPLB_EINVAL, "plan: idx must be 8-byte aligned");
  LPLB_REQUIRE(r2o && o2r && phy2log && o_weight && avail_num && (out || n_elements == 0), LPLB_EINVAL,
               "plan: null pointer");
  LPLB_REQUIRE(step_rule == LPLB_STEP_REFERENCE_WINDOW || step_rule == LPLB_STEP_FULL_MAX, LPLB_EINVAL,
               "plan: unknown step_rule %d", step_rule);
  LPLB_REQUIRE(n_steps >= 0, LPLB_EINVAL, "plan: n_steps=%d", n_steps);
  // refused before anything is enqueued, not by the last of the chain's kernels
  LPLB_REQUIRE(!(physical_counts && n_elements > (INT32_MAX - 41) / 499), LPLB_EUNSUPPORTED,
               "plan: physical_counts needs n_elements <= %d", (INT32_MAX - 41) / 499);
  const int n_logical = n_group * group_size * L;
  hipStream_t s = static_cast<hipStream_t>(stream);
  bool done = false;
  int rc = try_one_launch(idx, n_elements, global_counts, r2o, o2r, phy2log, n_group, group_size, dup_per_rank,
                          n_combined_experts, n_local_experts, n_blocks, counts_by_block, global_workload,
                          o_weight, avail_num, out, physical_counts, step_rule, n_steps, s, &done);
  if (rc != LPLB_OK || done)
    return rc;
  if (global_counts) {
    rc = lplb_solve(global_counts, global_workload, r2o, phy2log, n_group, group_size, dup_per_rank,
                    n_combined_experts, n_fixed, avail_num, o_weight, step_rule, n_steps, stream);
    if (rc != LPLB_OK)
      return rc;
    rc = enqueue_count(idx, n_elements, n_logical, n_blocks, counts_by_block, s, /*any_order=*/true);
    if (rc != LPLB_OK)
      return rc;
  } else if (g_cooperative && lp_shape_is_built(group_size, dup_per_rank) && n_group <= kScanSolveLps &&
             n_logical <= kMaxPlanExperts && n_elements > 0 && global_workload != nullptr) {
    ScanSolveArgs a{};
    int *words = nullptr;
    int dev = -1;
    rc = plan_words(&words, &dev);
    if (rc != LPLB_OK)
      return rc;
    a.timeouts = words + kLooseTimeoutsAt;
    a.counts = counts_by_block;
    a.totals = reinterpret_cast<int32_t *>(global_workload);
    a.n_blocks = n_blocks;
    a.expected_blocks = n_blocks + g_fault_extra_slices.exchange(0);
    const int fault_polls = g_fault_max_polls.exchange(0);
    a.max_polls = fault_polls > 0 ? fault_polls : kDefaultMaxPolls;
    SolveArgs &sa = a.solve;
    sa.gw_out = global_workload; sa.r2o = r2o; sa.phy2log = phy2log; sa.avail = avail_num; sa.result = o_weight;
    sa.n_group = sa.n_units = n_group; sa.G = group_size; sa.D = dup_per_rank; sa.C = n_combined_experts;
    sa.n_fixed = n_fixed; sa.n_experts = n_logical; sa.step_rule = step_rule; sa.n_steps = n_steps;
    sa.counts_by_caller = true;
    rc = enqueue_histogram(idx, n_elements, n_logical, n_blocks, counts_by_block, a.totals, s);
    if (rc != LPLB_OK)
      return rc;
    rc = group_size <= 8 ? scan_and_solve_up_to_8(a, s) : group_size <= 16 ? scan_and_solve_up_to_16(a, s) : scan_and_solve_up_to_32(a, s);
    if (rc != LPLB_OK)
      return rc;
  } else {
    rc = lplb_count_idx(idx, n_elements, n_logical, n_blocks, counts_by_block, stream);
    if (rc != LPLB_OK)
      return rc;
    rc = lplb_solve(counts_by_block + (int64_t)(n_blocks - 1) * n_logical, global_workload, r2o, phy2log,
                    n_group, group_size, dup_per_rank, n_combined_experts, n_fixed, avail_num, o_weight,
                    step_rule, n_steps, stream);
    if (rc != LPLB_OK)
      return rc;
  }
  return lplb_map_idx(idx, o_weight, counts_by_block, o2r, phy2log, n_elements, n_group,
                      group_size, dup_per_rank, n_combined_experts, n_local_experts, n_blocks, out,
                      physical_counts, stream);
}

// ---- the plan for callers that cannot allocate ----
// The slice table of a plan (counts_by_block of lplb_plan: n_blocks rows of n_logical
// counters that the workgroups exchange) lives in this array instead of a buffer of the
// caller's.  Every GPU the library runs on holds its own copy until the process ends.
constexpr int64_t kScratchInts = 1 << 18;   // 1 MiB: e.g. 256 slices x 1024 logical experts
static __device__ __align__(256) int32_t scratch[kScratchInts];

// Per device: the table's address (the array's name is only a host-side handle: looked up once, at the
// first call on the device) and who used the table last.  One table serves every stream, so a call from
// another stream is refused while the last user's kernels may still be running; `done` is recorded
// behind each call and is made, like the address, at that first call, which therefore has to happen
// outside a stream capture.  A call captured into a graph keeps the table for its stream for good.
struct ScratchUse {
  int32_t *table = nullptr;
  int *finished = nullptr;   // pinned host memory: the number of the last call whose kernels have all ended
  int seq = 0;               // number of the last call
  hipStream_t stream = nullptr;
  bool used = false, captured = false;
};
static ScratchUse g_scratch_use[64];
static std::mutex g_scratch_guard;

static int scratch_of_current_device(ScratchUse **use) {
  int dev = -1;
  LPLB_HIP_TRY(hipGetDevice(&dev));
  LPLB_REQUIRE(dev >= 0 && dev < 64, LPLB_EUNSUPPORTED, "plan_noalloc: device ordinal %d", dev);
  ScratchUse &u = g_scratch_use[dev];
  if (!u.table) {
    int32_t *p = nullptr;
    LPLB_HIP_TRY(hipGetSymbolAddress(reinterpret_cast<void **>(&p), HIP_SYMBOL(scratch)));
    LPLB_REQUIRE(p != nullptr, LPLB_EHIP, "plan_noalloc: no device address for the slice table");
    LPLB_HIP_TRY(hipHostMalloc(reinterpret_cast<void **>(&u.finished), sizeof(int), hipHostMallocDefault));
    *u.finished = 0;
    u.table = p;
  }
  *use = &u;
  return LPLB_OK;
}

// The last kernel of a call: copies the batch's totals out (n may be 0) and says, in pinned host memory, that
// every kernel of call number `seq` has ended (kernels of one stream end in the order they were enqueued).
__global__ void copy_ints_and_report(const int32_t *__restrict__ src, int32_t *__restrict__ dst, int n, int *finished,
                                     int seq) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    dst[i] = src[i];
  if (i == 0 && finished)
    __hip_atomic_store(finished, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

} // namespace lplb

extern "C" int lplb_plan(const int64_t *idx, int64_t n_elements,
                         const int32_t *global_counts, const int32_t *r2o,
                         const int32_t *o2r, const int32_t *phy2log, int n_group,
                         int group_size, int dup_per_rank, int n_combined_experts,
                         int n_local_experts, int n_blocks, int32_t *counts_by_block,
                         float *global_workload, float *o_weight, int32_t *avail_num,
                         int64_t *out, int32_t *physical_counts, int step_rule, int n_steps,
                         lplb_stream_t stream) {
  return lplb::plan_checked(idx, n_elements, global_counts, r2o, o2r, phy2log, n_group, group_size, dup_per_rank,
                            n_combined_experts, n_local_experts, n_blocks, counts_by_block, global_workload,
                            o_weight, avail_num, out, physical_counts, step_rule, n_steps, stream);
}

extern "C" int lplb_plan_noalloc(const int64_t *idx, int64_t n_elements,
                                 const int32_t *global_counts, const int32_t *r2o,
                                 const int32_t *o2r, const int32_t *phy2log, int n_group,
                                 int group_size, int dup_per_rank, int n_combined_experts,
                                 int n_local_experts, int n_blocks, int32_t *local_counts,
                                 float *global_workload, float *o_weight, int32_t *avail_num,
                                 int64_t *out, int32_t *physical_counts, int step_rule, int n_steps,
                                 lplb_stream_t stream) {
  using namespace lplb;
  LPLB_REQUIRE(n_group > 0 && group_size > 0 && dup_per_rank > 0 && n_blocks > 0 && n_combined_experts >= 0,
               LPLB_EINVAL, "plan_noalloc: n_group=%d group_size=%d dup_per_rank=%d n_blocks=%d must be positive",
               n_group, group_size, dup_per_rank, n_blocks);
  const int64_t L = (int64_t)n_local_experts - (int64_t)dup_per_rank * n_combined_experts;
  LPLB_REQUIRE(L > 0, LPLB_EINVAL, "plan_noalloc: n_local_experts=%d does not fit %d x %d replicas", n_local_experts,
               dup_per_rank, n_combined_experts);
  const int64_t n_logical = (int64_t)n_group * group_size * L;
  LPLB_REQUIRE((int64_t)n_blocks * n_logical <= kScratchInts, LPLB_EUNSUPPORTED,
               "plan_noalloc: n_blocks=%d x %lld logical experts = %lld counters exceed the built-in slice table of "
               "%lld; use fewer slices or lplb_plan with a workspace of your own",
               n_blocks, (long long)n_logical, (long long)((int64_t)n_blocks * n_logical), (long long)kScratchInts);
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &capture) != hipSuccess)
    capture = hipStreamCaptureStatusNone;
  const bool capturing = capture == hipStreamCaptureStatusActive;
  std::lock_guard<std::mutex> lock(g_scratch_guard);   // held over the call: check, enqueue and record agree
  ScratchUse *use = nullptr;
  int rc = scratch_of_current_device(&use);
  if (rc != LPLB_OK)
    return rc;
  if (use->used && use->stream != s) {
    const bool busy = use->captured || __atomic_load_n(use->finished, __ATOMIC_ACQUIRE) != use->seq;
    LPLB_REQUIRE(!busy, LPLB_EBUSY,
                 "plan_noalloc: the built-in slice table is in use by a plan on another stream%s; wait for it, keep "
                 "such plans on one stream, or use lplb_plan with a workspace of your own",
                 use->captured ? " (captured into a graph, which keeps it)" : "");
  }
  int32_t *table = use->table;
  // Nothing in the table has to start at zero: every row is written (by the slice that
  // owns it) before anything reads it, and rows beyond n_blocks are never read.
  rc = plan_checked(idx, n_elements, global_counts, r2o, o2r, phy2log, n_group, group_size, dup_per_rank,
                    n_combined_experts, n_local_experts, n_blocks, table, global_workload, o_weight, avail_num, out,
                    physical_counts, step_rule, n_steps, stream);
  // Whatever was enqueued may touch the table, also when a later step of the chain failed: the call is
  // numbered and its last kernel reports the number (a captured call reports nothing: it keeps the table).
  use->used = true;
  use->stream = s;
  use->captured = use->captured || capturing;
  if (!capturing)
    use->seq = (use->seq + 1) & 0x3fffffff;
  const int n_copy = rc == LPLB_OK && local_counts != nullptr ? (int)n_logical : 0;
  launch(copy_ints_and_report, dim3((unsigned)((n_copy + 255) / 256 > 0 ? (n_copy + 255) / 256 : 1)), dim3(256), 0, s,
         table + (int64_t)(n_blocks - 1) * n_logical, local_counts, n_copy, capturing ? nullptr : use->finished, use->seq);
  if (hipGetLastError() != hipSuccess && rc == LPLB_OK)
    rc = fail(LPLB_EHIP, "plan_noalloc: launch failed");
  return rc;
}
