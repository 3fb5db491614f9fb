// Which plans run as one launch side by side, and which block of words each of them uses: the host's bookkeeping.
// No call of the runtime here, so that the rules can be driven on a CPU (tests/test_host.py).
//
// A block belongs to one stream at a time (launches that share one must not overlap, which stream order guarantees).
// One whose last launch has arrived as a whole -- none of its workgroups waits for one that is not resident -- may pass
// to another stream; what runs there first has to wait until that launch has read its last word (Admitted::wait_*).
// A block with a launch captured into a graph stays with its stream and counts as executing: a replay may
// come at any time and the host does not see it.
#pragma once

namespace lplb {

// Up to this share of the GPU's resident workgroups may belong to plans that wait for
// their own workgroups; the rest stays free for their stragglers and for other kernels.
constexpr float kResidencyBudget = 0.80f;
constexpr int kSeqMask = 0x3fffffff;   // launches are numbered modulo this + 1

template <int SLOTS> class PlanAdmission {
public:
  struct Admitted {
    int slot = -1;                                     // -1: run the chain
    int seq = 0;                                       // number the launch carries, -1: none (captured)
    int wait_slices = 0, wait_lps = 0, wait_seq = 0;   // the launch of another stream to wait for (no slices: none)
  };

  // One launch that takes `cost` of the GPU's resident workgroups, on `stream`.  arrived[i]: number of the last launch of
  // slot i that has said that all of its workgroups have arrived (may be null until a launch outside a capture is admitted).
  // if_alone: only while no other stream's plan may be executing, and if no graph keeps the share for good.
  Admitted admit(const void *stream, float cost, bool capturing, const int *arrived, bool if_alone = false) {
    Admitted got;
    int slot = -1;
    for (int i = 0; i < SLOTS && slot < 0; ++i)
      if (slots_[i].used && slots_[i].stream == stream)
        slot = i;
    for (int i = 0; i < SLOTS && slot < 0; ++i)
      if (!slots_[i].used)
        slot = i;
    if (slot < 0)
      slot = left_by_its_stream(arrived);
    if (slot < 0)
      return got;
    float executing = 0.0f;
    for (int i = 0; i < SLOTS; ++i)
      if (i != slot && is_executing(i, arrived))
        executing += slots_[i].cost;
    if (executing + cost > kResidencyBudget)
      return got;
    Slot &s = slots_[slot];
    if (if_alone && (executing > 0.0f || capturing || s.captured))
      return got;
    if (!s.used || s.stream != stream) {
      s.stream = stream;
      s.cost = 0.0f;
      s.used = true;
      s.captured = s.maybe_executing = false;
    }
    // (a launch in front of this one on the stream may be the one that is executing)
    s.cost = is_executing(slot, arrived) && s.cost > cost ? s.cost : cost;
    s.captured = s.captured || capturing;
    s.used_at = ++admitted_;
    got.slot = slot;
    // (a replay would leave its number over that of a later launch)
    got.seq = capturing ? -1 : (s.seq + 1) & kSeqMask;
    // Until this stream has run a launch of its own here, every one of its launches waits, not the first only: one that is
    // being captured does not run now, and its graph may be replayed after the next or never.
    if (s.slices > 0 && s.last_stream != stream) {
      got.wait_slices = s.slices;
      got.wait_lps = s.lps;
      got.wait_seq = s.seq;
    }
    return got;
  }

  // It has been enqueued (or captured).
  void launched(const Admitted &a, bool capturing, int slices, int lps) {
    if (capturing)
      return;
    Slot &s = slots_[a.slot];
    s.maybe_executing = true;
    s.last_stream = s.stream;
    s.seq = a.seq;
    s.slices = slices;
    s.lps = lps;
  }

  // The graphs that hold launches captured on `stream` are gone and their replays have ended.  (What the stream has enqueued
  // outside a capture may be executing, and counts on until it has arrived.)
  void forget_captured(const void *stream) {
    for (Slot &s : slots_)
      if (s.used && s.stream == stream)
        s.captured = false;
  }

  int number_of(int slot) const { return slots_[slot].seq; }

  // Nothing enqueued so far is still running.
  void device_is_idle() {
    for (Slot &s : slots_) {
      s.maybe_executing = false;
      s.slices = s.lps = 0;
    }
  }

private:
  struct Slot {
    const void *stream = nullptr;        // who may use it
    const void *last_stream = nullptr;   // where the latest launch outside a capture ran
    int seq = 0;                         // that launch's number
    int slices = 0, lps = 0;             // ... and whose done words a launch of another stream has to see (0: nothing to wait for)
    float cost = 0.0f;                   // share of the GPU's resident workgroups its launches take
    bool used = false, captured = false;
    bool maybe_executing = false;        // a launch was enqueued and has not been seen to have arrived since
    unsigned long long used_at = 0;      // the last launch admitted to it, among all
  };
  // May a launch of this slot still need room on the GPU?  Looking at the word asks nothing of the runtime, the stream
  // (which other threads may be capturing on, or may have destroyed) is not touched, and nothing waits.
  bool is_executing(int i, const int *arrived) {
    Slot &s = slots_[i];
    if (!s.used)
      return false;
    if (s.captured)
      return true;
    if (s.maybe_executing && __atomic_load_n(arrived + i, __ATOMIC_ACQUIRE) == s.seq)
      s.maybe_executing = false;
    return s.maybe_executing;
  }
  // The slot that passes on to another stream, -1: all are executing.  Taking one that its stream is about to use again makes
  // that stream take another, and so on, with a wait in front of every plan.  So: the one that has not been used for
  // longest, if that is long; else the streams in use are more than the slots, and as many of them as possible keep
  // theirs if the one used last goes round among the rest.  Plans of [8192 x 8] in turn on 6, 8, 12 streams, against the
  // first slot that is not executing: 7.1 -> 4.8, 7.4 -> 4.8, 6.9 -> 6.2 us a plan.
  int left_by_its_stream(const int *arrived) {
    int oldest = -1, newest = -1;
    for (int i = 0; i < SLOTS; ++i)
      if (!is_executing(i, arrived)) {
        oldest = oldest < 0 || slots_[i].used_at < slots_[oldest].used_at ? i : oldest;
        newest = newest < 0 || slots_[i].used_at > slots_[newest].used_at ? i : newest;
      }
    return oldest >= 0 && admitted_ - slots_[oldest].used_at >= 4 * SLOTS ? oldest : newest;
  }
  Slot slots_[SLOTS];
  unsigned long long admitted_ = 0;
};

} // namespace lplb
