"""Host logic that needs no GPU: topologies, the redundancy mapping, the EPLB
reorder (against vectors written by the reference's own eplb.py), the Planner's
derived state, the synthetic workloads, and the C-ABI surface of the HIP library."""
import ctypes
import hashlib
import json
import re
from pathlib import Path

import numpy as np
import pytest
import torch

from lplb_amd import Planner, _native, eplb, synth, topology
from lplb_amd.mapping import build_redundancy_mapping
from tests.helpers import BATCHED_LPS, PLACEMENTS, REFERENCE_SOLVE_CASES

ROOT = Path(__file__).resolve().parent.parent
GOLDEN = ROOT / "tests" / "golden"


# --------------------------------------------------------------- topologies
def test_topologies_are_column_permutations():
    for r2o in (topology.CUBE_8P2E, topology.RING_8P, topology.HYPERCUBE_16P2E, topology.torus_2d(8, 4),
                topology.torus_2d(4, 4)):
        assert topology.is_valid_r2o(r2o)
        assert not np.any(r2o == np.arange(r2o.shape[0])[:, None])        # no replica on its own rank
    assert not topology.is_valid_r2o(np.array([[0, 1], [0, 0]]))
    t = topology.torus_2d(8, 4)
    assert t.shape == (32, 2) and t[0].tolist() == [4, 1] and t[31].tolist() == [3, 28]


# ------------------------------------------------------------- EPLB reorder
def test_eplb_matches_reference_vectors():
    """Vectors written by tests/golden/make_eplb_vectors.py from the reference's eplb.py
    (tie-free weights)."""
    for c in json.loads((GOLDEN / "eplb_vectors.json").read_text()):
        w = np.array(c["weight"])
        phy2log, log2phy, logcnt = eplb.rebalance_experts(w, c["num_replicas"], c["num_groups"], c["num_nodes"],
                                                          c["num_gpus"])
        np.testing.assert_array_equal(phy2log, c["phy2log"])
        np.testing.assert_array_equal(logcnt, c["logcnt"])
        want = np.array(c["log2phy"])
        if c["num_replicas"] == c["n_logical"]:
            np.testing.assert_array_equal(log2phy, want)
        else:
            # replicas of one expert carry equal loads, so which of them is "replica 0" is a tie
            np.testing.assert_array_equal(np.sort(log2phy, axis=-1), np.sort(want, axis=-1))


def test_balanced_packing_properties():
    rng = np.random.default_rng(0)
    w = rng.random((3, 24)).astype(np.float32)
    pack, rank = eplb.balanced_packing(w, 6)
    for layer in range(3):
        assert sorted(np.bincount(pack[layer], minlength=6)) == [4] * 6
        for p in range(6):
            assert sorted(rank[layer][pack[layer] == p]) == [0, 1, 2, 3]
    # heaviest-first greedy never does worse than putting the 4 heaviest together
    loads = np.array([[w[l][pack[l] == p].sum() for p in range(6)] for l in range(3)])
    assert np.all(loads.max(1) <= np.sort(w, axis=1)[:, -4:].sum(1))
    pack1, rank1 = eplb.balanced_packing(w[:, :6], 6)
    assert np.array_equal(pack1, np.broadcast_to(np.arange(6), (3, 6))) and not rank1.any()


@pytest.mark.parametrize("n_log,n_phy,groups,nodes,gpus", [
    (1, 1, 1, 1, 1), (7, 8, 1, 1, 8), (24, 24, 8, 8, 8), (63, 64, 3, 1, 4), (256, 256, 4, 2, 32), (258, 264, 2, 2, 8),
    (1290, 1296, 10, 2, 16)])                               # groups of 1, 3, 8, 21, 64, 129 experts: every way of adding them up
@pytest.mark.parametrize("weights", ["distinct", "ties", "spread", "nan"])
def test_native_placement_equals_the_numpy_restatement(n_log, n_phy, groups, nodes, gpus, weights):
    from oracle import eplb_numpy
    rng = np.random.default_rng(n_log)
    w = {"distinct": rng.random((2, n_log)) * 1e6, "ties": rng.integers(0, 4, (2, n_log)),
         "spread": rng.lognormal(0, 3, (2, n_log)), "nan": np.where(rng.random((2, n_log)) < 0.1, np.nan, 1.0)}[weights]
    for got, want in zip(eplb.rebalance_experts(w, n_phy, groups, nodes, gpus),
                         eplb_numpy.rebalance_experts(w, n_phy, groups, nodes, gpus)):
        np.testing.assert_array_equal(got, want)
    if n_log % 8 == 0 and n_log >= 16:
        args = (topology.CUBE_8P2E, 8, n_log, n_log + 16, w[0], nodes)
        for got, want in zip(build_redundancy_mapping(*args), eplb_numpy.build_redundancy_mapping(*args)):
            np.testing.assert_array_equal(got, want)
            assert got.dtype == want.dtype and got.shape == want.shape


@pytest.mark.parametrize("infinite", [1, 5, 40, 64])
def test_packing_never_fills_a_pack_twice(infinite):
    """Loads of infinity are all alike: the lightest of them may be a pack that has no room left."""
    rng = np.random.default_rng(infinite)
    weight = rng.random((3, 64)).astype(np.float32)
    for row in weight:
        row[rng.permutation(64)[:infinite]] = np.inf
    weight[2, 0] = np.nan
    pack, place = eplb.balanced_packing(weight, 8)
    for p, r in zip(pack, place):
        assert sorted(zip(p.tolist(), r.tolist())) == [(k, m) for k in range(8) for m in range(8)]
    phy2log, log2phy, logcnt = eplb.rebalance_experts(weight, 64, 4, 2, 8)
    assert np.array_equal(np.sort(phy2log, axis=1), np.tile(np.arange(64), (3, 1))) and logcnt.max() == 1


# ------------------------------------------------------ redundancy mapping
@pytest.mark.parametrize("case", REFERENCE_SOLVE_CASES, ids=[c[0] for c in REFERENCE_SOLVE_CASES])
@pytest.mark.parametrize("with_history", [False, True])
def test_redundancy_mapping_layout(case, with_history):
    _, r2o, nl, ep, red, _, _ = case
    r2o = np.asarray(r2o)
    G, D = r2o.shape
    n_phys = nl + red * ep
    L, P = nl // ep, n_phys // ep
    C = (P - L) // D
    rng = np.random.default_rng(1)
    hist = rng.integers(1, 1 << 20, size=nl) if with_history else None
    phy2log, log2phy, logcnt = build_redundancy_mapping(r2o, ep, nl, n_phys, hist, n_nodes=max(1, ep // 8))
    assert phy2log.shape == (n_phys,) and phy2log.dtype == np.int32
    per_rank = phy2log.reshape(ep // G, G, P)
    # the first L slots of all ranks are a permutation of the logical experts
    assert sorted(per_rank[:, :, :L].reshape(-1)) == list(range(nl))
    # replica (c, d) of group-rank i copies slot (c, d) of group-rank r2o[i, d]
    for g in range(ep // G):
        for i in range(G):
            for c in range(C):
                for d in range(D):
                    assert per_rank[g, i, L + c * D + d] == per_rank[g, r2o[i, d], c * D + d]
    if with_history:
        # every rank keeps its experts heaviest first, so its replicated ones are its heaviest
        h = hist[per_rank[:, :, :L]]
        assert np.all(np.diff(h, axis=-1) <= 0)
    else:
        assert np.array_equal(per_rank[:, :, :L].reshape(-1), np.arange(nl))
    # log2phy: original first, then the replica; at most one replica each (lplb/planner.py:165-178)
    assert logcnt.max() == 2 and logcnt.sum() == n_phys
    for e in range(nl):
        slots = [s for s in log2phy[e] if s >= 0]
        assert len(slots) == logcnt[e] and all(phy2log[s] == e for s in slots)
        assert slots[0] % P < L and all(s % P >= L for s in slots[1:])


def test_redundancy_mapping_rejects_doubly_replicated_experts():
    bad = np.array([[1, 1], [0, 0]]).T            # both ranks copy rank 1's slot-0 expert
    with pytest.raises(AssertionError):
        build_redundancy_mapping(np.array([[1], [1]]), 2, 4, 6)
    del bad


# ------------------------------------------------------------------ Planner
def test_planner_derived_state_on_cpu():
    p = Planner(torch.from_numpy(topology.CUBE_8P2E), 256 + 2 * 32, 256, 32, device="cpu")
    assert (p.group_size, p.num_redundants, p.n_group, p.ep_size) == (8, 2, 4, 32)
    assert (p.n_local_routed_experts, p.n_local_logical_routed_experts, p.combined_redundant_experts) == (10, 8, 1)
    assert p.r2o.dtype == torch.int32 and p.o2r.dtype == torch.int32 and p.o2r.is_contiguous()
    r2o, o2r = p.r2o.numpy(), p.o2r.numpy()
    for d in range(2):
        assert np.array_equal(r2o[o2r[:, d], d], np.arange(8))             # o2r inverts r2o column-wise
    assert p.phy2log.shape == (320,) and p.phy2log.dtype == torch.int32
    phy2log, log2phy, logcnt = p.update_redundancy_mapping(torch.arange(256, 0, -1) * 1000)
    assert phy2log is p.phy2log and log2phy.shape == (256, 2) and int(logcnt.max()) == 2
    assert all(t.dtype == torch.int32 for t in (phy2log, log2phy, logcnt))
    # ep_size defaults to the group size (needs a group), combined replicas
    with pytest.raises(AssertionError):
        Planner(torch.from_numpy(topology.CUBE_8P2E), 320, 256, device="cpu")
    p4 = Planner(torch.from_numpy(topology.CUBE_8P2E), 256 + 4 * 32, 256, 32, device="cpu")
    assert p4.combined_redundant_experts == 2 and p4.phy2log.numel() == 384


def test_planner_needs_a_gpu_for_the_kernels():
    p = Planner(torch.from_numpy(topology.RING_8P), 64 + 8, 64, 8, device="cpu")
    idx = torch.zeros(16, dtype=torch.int64)
    with pytest.raises(RuntimeError):
        p.run(idx, torch.zeros(1, dtype=torch.int32), 4)
    with pytest.raises(NotImplementedError):
        p.init_from_deep_ep(None)


def test_planner_surfaces_waits_that_ran_out(monkeypatch):
    """Planner.run looks at the one-launch plan's health report every few calls; a non-zero count must reach the
    user (a warning, the attribute) and switch the one-launch form on again.  The report itself needs a GPU;
    what is done with it does not."""
    from lplb_amd import _native as native
    p = Planner(torch.from_numpy(topology.RING_8P), 64 + 8, 64, 8, device="cpu")
    rearmed = []
    monkeypatch.setattr(native, "plan_sync_timeouts", lambda: rearmed.append(1) or 5)
    import warnings as w
    with w.catch_warnings():
        w.simplefilter("error")
        p._handle_plan_health(0, 0)                    # healthy: silent
    assert p.plan_timeouts == 0 and not rearmed
    with pytest.warns(RuntimeWarning, match="not balanced"):
        p._handle_plan_health(3, 1)
    assert rearmed == [1] and p.plan_timeouts == 5     # the synchronous call's own count after re-arming
    with pytest.warns(RuntimeWarning):
        p._handle_plan_health(7, 0)                    # counted since, but no block is off: nothing to re-arm
    assert rearmed == [1] and p.plan_timeouts == 7
    with w.catch_warnings():
        w.simplefilter("error")
        p._handle_plan_health(7, 0)                    # nothing new
    # the look itself is spaced out and never happens on a CPU planner before the kernels are needed
    calls = []
    monkeypatch.setattr(native, "plan_poll_timeouts", lambda dst, stream=None: calls.append(dst))
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda self: self)
    monkeypatch.setattr("lplb_amd.planner._stream", lambda t: 0)
    p.health_check_every = 4
    for _ in range(9):
        p._look_at_plan_health(torch.zeros(1))
    assert len(calls) == 2 and calls[0] is calls[1] and calls[0].dtype == torch.int32


def test_compiled_solver_argument_checks():
    """Same refusals as the reference's extension (csrc/plugin.cpp:494-530, 582-584, 605-628)."""
    s = _native.CompiledSolver(1, 8, 2, 34, 1)
    assert s.n_experts == 256
    idx = torch.zeros(16, dtype=torch.int64)
    with pytest.raises(RuntimeError):
        s.count_idx(idx, 4)                       # not on a GPU
    with pytest.raises(RuntimeError):
        s.count_idx(idx.int(), 4)                 # wrong dtype
    with pytest.raises(RuntimeError):
        s.solve(torch.zeros(1, 8, 32, dtype=torch.int32), torch.zeros(8, 2, dtype=torch.int32),
                torch.zeros(272, dtype=torch.int32), torch.zeros(1, dtype=torch.int32))
    with pytest.raises(RuntimeError):
        s.map_idx(idx, torch.zeros(1, 8, 2), torch.zeros(4, 256, dtype=torch.int32), torch.zeros(8, 2, dtype=torch.int32),
                  torch.zeros(272, dtype=torch.int32), 4)


# ---------------------------------------------------------------- workloads
def test_synthetic_inputs_are_deterministic_and_well_formed():
    digests = {}
    for name in ("cpu_ref_ep8", "v3_ep8_cube", "ep16_hypercube", "ep32_torus"):
        a, b = synth.make_inputs(name, tokens=512), synth.make_inputs(name, tokens=512)
        for x, y in ((a.indices, b.indices), (a.global_counts, b.global_counts), (a.phy2log, b.phy2log)):
            assert np.array_equal(x, y)
        c = a.cfg
        assert a.indices.shape == (512, c.topk) and a.indices.dtype == np.int64
        assert a.indices.min() >= 0 and a.indices.max() < c.n_logical
        assert all(len(set(row)) == c.topk for row in a.indices[:64])      # distinct experts per token
        assert a.global_counts.dtype == np.int32 and a.global_counts.sum() == c.ep_size * c.tokens * c.topk
        assert abs(a.popularity.sum() - 1) < 1e-12
        digests[name] = hashlib.sha256(a.indices.tobytes() + a.global_counts.tobytes()).hexdigest()
    assert len(set(digests.values())) == 4
    m = synth.make_inputs("cpu_ref_ep8", mask_fraction=0.25)
    assert 0.15 < (m.indices == -1).mean() < 0.35
    sc = synth.sweep_counts(4)
    assert sc.shape == (4, 256) and not np.array_equal(sc[0], sc[1])
    hot = synth.make_inputs("ep32_torus", tokens=8).popularity
    assert (hot > 5.0 / 256).sum() >= 3


# ------------------------------------------------------------------- C ABI
def _declared_symbols():
    text = (ROOT / "include" / "lplb_hip.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(lplb_[a-z_0-9]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = _native.load()
    declared = _declared_symbols()
    assert "lplb_count_idx" in declared and "lplb_solve" in declared and "lplb_map_idx" in declared
    for name in declared:
        assert getattr(lib, name) is not None
    assert sorted(_native.exported_symbols()) == declared
    assert lib.lplb_abi_version() == _native.ABI_VERSION == 7
    header = (ROOT / "include" / "lplb_hip.h").read_text()
    assert f"#define LPLB_ABI_VERSION {_native.ABI_VERSION}" in header
    assert f"#define LPLB_COUNT_TOTALS_MAX_INDICES {_native.COUNT_TOTALS_MAX_INDICES}\n" in header
    assert f"#define LPLB_COUNT_TOTALS_MAX_EXPERTS {_native.COUNT_TOTALS_MAX_EXPERTS}\n" in header


def test_entry_points_reject_bad_arguments_before_touching_the_gpu():
    lib = _native.load()
    buf = (ctypes.c_int64 * 4)()
    p = ctypes.cast(buf, ctypes.c_void_p)
    assert lib.lplb_count_idx(p, 4, 0, 4, p, None) == 1
    assert b"n_experts" in lib.lplb_last_error()
    assert lib.lplb_count_idx(p, -1, 8, 4, p, None) == 1
    assert lib.lplb_count_idx(p, 4, 8, 4, None, None) == 1
    assert lib.lplb_count_idx(p, 4, 1 << 20, 4, p, None) == 2           # histogram does not fit LDS
    assert lib.lplb_count_totals(p, 4, 0, p, None) == 1
    assert lib.lplb_count_totals(p, 4, 8, None, None) == 1
    assert lib.lplb_count_totals(p, 1 << 20, 8, p, None) == 2          # a long batch: histogram and scan serve it
    assert lib.lplb_count_totals_add(p, 4, 0, p, None, None) == 1
    assert lib.lplb_count_totals_add(p, 4, 8, None, None, None) == 1
    assert lib.lplb_count_totals_add(p, 4, 8, p, p, None) == 1            # totals and clear are one vector
    assert b"same vector" in lib.lplb_last_error()
    assert lib.lplb_count_totals_add(p, 4, 1 << 20, p, None, None) == 2   # histogram does not fit LDS
    assert lib.lplb_count_totals_add(p, 1 << 20, 8, p, None, None) == 2   # a long batch
    assert lib.lplb_solve(p, p, p, p, 1, 16, 9, 1, 2, p, p, 0, 5, None) == 2   # 144 edges > two per lane of a wave
    assert b"128 replica edges" in lib.lplb_last_error()
    assert lib.lplb_solve(p, p, p, p, 1, 4, 17, 1, 2, p, p, 0, 5, None) == 2   # more than 16 slots per rank
    assert lib.lplb_solve(p, p, p, p, 1, 65, 1, 1, 2, p, p, 0, 5, None) == 2   # more ranks than lanes
    assert lib.lplb_solve(p, p, p, p, 1, 8, 2, 1, 2, p, p, 7, 5, None) == 1    # unknown step rule
    assert lib.lplb_solve(p, None, p, p, 1, 8, 2, 1, 2, p, p, 0, 5, None) == 1
    assert lib.lplb_solve_batched(p, None, p, p, 0, 1, 8, 2, 1, 2, p, p, 0, 5, None) == 1
    assert lib.lplb_map_idx(p, p, p, p, p, 4, 1, 8, 2, 1, 2, 4, p, None, None) == 1  # 2 slots per rank cannot hold 2 replicas
    assert lib.lplb_map_idx(p, p, p, p, None, 4, 1, 8, 2, 1, 34, 4, p, None, None) == 1
    assert lib.lplb_plan(p, 4, None, p, p, p, 1, 8, 2, 1, 34, 0, p, p, p, p, p, None, 0, 5, None) == 1
    assert lib.lplb_copy_calibration(p, p, 3, None) == 1
    # an index array needs its natural alignment only; 4 bytes off is refused
    odd = ctypes.c_void_p(p.value + 4)
    assert lib.lplb_count_idx(odd, 4, 8, 4, p, None) == 1 and b"8-byte" in lib.lplb_last_error()
    assert lib.lplb_plan(odd, 4, None, p, p, p, 1, 8, 2, 1, 34, 4, p, p, p, p, p, None, 0, 5, None) == 1
    # tokens per physical expert come from a closed form that assumes 499 k + 41 does not wrap
    assert lib.lplb_plan(p, 5_000_000, None, p, p, p, 1, 8, 2, 1, 34, 256, p, p, p, p, p, p, 0, 5, None) == 2
    assert b"physical_counts" in lib.lplb_last_error()
    assert lib.lplb_map_idx(p, p, p, p, p, 5_000_000, 1, 8, 2, 1, 34, 256, p, p, None) == 2


def test_cross_workgroup_helpers_compile_to_the_forms_the_plan_relies_on(tmp_path):
    """The workgroups of the one-launch plan exchange 8-byte words, tag above value, that say themselves whether they are
    there (lplb_amd/csrc/plan_sync.h).  That works across the GPU's eight L2 caches because such a word is written by one
    store past the caches (dwordx2, sc1), read by one load past them (dwordx2, sc1) and loaded anew by every poll, and
    because nothing invalidates or writes back a cache (the L2 holds the batch's indices while the workgroups talk).  Compile the
    helpers on their own and look at what the compiler makes of them, so that a toolchain that lowers them
    differently fails here and not silently on the GPU; and look for cache maintenance in the built kernels."""
    import shutil
    import subprocess
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("no hipcc")
    probe = tmp_path / "probe.hip"
    probe.write_text('''
#include "plan_kernel.h"
using namespace lplb;
extern "C" __global__ void store_word(unsigned long long *word, unsigned tag, unsigned v) { agent_store(word + threadIdx.x, tagged_word(tag, v)); }
extern "C" __global__ void load_word(const unsigned long long *word, unsigned long long *out) { out[threadIdx.x] = agent_load(word + threadIdx.x); }
extern "C" __global__ void store_pairs(unsigned long long *words, u32x4 v, u32x4 w) { agent_store_pairs(words + 4 * threadIdx.x, v, w); }
extern "C" __global__ void store_int(int *p, int v) { agent_store(p + threadIdx.x, v); }
extern "C" __global__ void load_int(const int *p, int *out) { out[threadIdx.x] = agent_load(p + threadIdx.x); }
extern "C" __global__ void add_int(int *p) { agent_add(p + threadIdx.x, 3); }
extern "C" __global__ void replace_int(int *p, int v) { agent_replace(p + threadIdx.x, -1, v); }
extern "C" __global__ void collect(const unsigned long long *words, unsigned tag, unsigned *out, int *came) {
  unsigned got[4];
  const bool all = collect_words<4>(got, tag, 4, 1000, [&](int k) { return words + 4 * threadIdx.x + k; });
  for (int k = 0; k < 4; ++k)
    out[4 * threadIdx.x + k] = got[k];
  came[threadIdx.x] = all;
}
''')
    asm = tmp_path / "probe.s"
    subprocess.run([hipcc, "-O3", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-S",
                    f"-I{ROOT / 'lplb_amd' / 'csrc'}", str(probe), "-o", str(asm)], check=True, capture_output=True)
    text = asm.read_text()
    body = {name: text.split(f"\n{name}:")[1].split("s_endpgm")[0]
            for name in ("store_word", "load_word", "store_pairs", "store_int", "load_int", "add_int", "replace_int", "collect")}
    memory = {name: re.findall(r"(?:global|flat|buffer)_\w+ .*", code) for name, code in body.items()}
    for name, form in (("store_word", r"global_store_dwordx2 .* sc1$"), ("store_int", r"global_store_dword .* sc1$")):
        assert len(memory[name]) == 1 and re.match(form, memory[name][0]), (name, memory[name])      # one store, past the caches
    # two words by one store; its data registers may not be written by the next two instructions, which the compiler does not see
    # to behind a store that it did not choose itself
    pairs_then_wait = r"(\tglobal_store_dwordx4 .* sc1\n){2}\ts_nop [1-9]"
    assert len(memory["store_pairs"]) == 2 and re.search(pairs_then_wait, body["store_pairs"]), body["store_pairs"]
    for name, form in (("load_word", r"global_load_dwordx2 .* sc1$"), ("load_int", r"global_load_dword .* sc1$")):
        assert re.match(form, memory[name][0]), (name, memory[name])
        assert sum("_load_" in m for m in memory[name]) == 1
    # read-modify-writes are carried out by the atomic unit behind the caches (no cached copy to go stale)
    assert re.match(r"global_atomic_add v", memory["add_int"][0]) and re.match(r"global_atomic_cmpswap v", memory["replace_int"][0])
    # a poll: sleep and four loads past the caches inside the loop
    before, loop = body["collect"].split("=>This", 1)
    polled = re.findall(r"global_load_dwordx2 .*", loop)
    assert "s_sleep" in loop and "global_load" not in before.rpartition("\n.LBB")[0], "a poll does not load anew"
    assert len(polled) >= 4 and all(p.endswith("sc1") for p in polled), polled
    assert "buffer_inv" not in text and "buffer_wbl2" not in text, "a cache is invalidated or written back"
    kernels = pairs = 0
    for name, code in _device_code(_native.LIB_PATH):
        if "plan_in_one_launch" in name or "plan_of_long_slices" in name or "scan_and_solve" in name or "wait_for_last_user" in name:
            kernels += 1
            assert not any(op.startswith(("buffer_inv", "buffer_wbl2")) for _, op, _ in code), name
            for (_, op, _), (_, behind, _) in zip(code, code[1:]):
                if re.match(pair := r"global_store_dwordx4 .* sc1$", op):
                    pairs += 1
                    assert re.match(rf"s_nop [1-9]|{pair}", behind), (name, op, behind)
    assert kernels >= 14 * 6 + 14 + 1 and pairs >= 14 * 6 * 2, (kernels, pairs)


def test_a_debug_build_without_a_buffer_stamps_nothing(tmp_path):
    """Builds with phase clocks write them to a buffer that the caller sets; until one is set no kernel may take a place in it
    for an address.  The kernels' stamp macros on the host, with and without a buffer, in the first, a middle and the last workgroup."""
    import subprocess
    csrc = ROOT / "lplb_amd" / "csrc"
    macros = [re.search(rf"#define {name}\(k\)(?:.*\\\n)*.*\n", (csrc / source).read_text()).group()
              for name, source in (("LPLB_STAMP", "solve_kernel.h"), ("LPLB_PLAN_STAMP", "plan_kernel.h"), ("LPLB_MAP_STAMP", "map.hip"))]
    (tmp_path / "stamps.cpp").write_text('''
#include <cstdint>
struct { unsigned x; } blockIdx, gridDim;
struct Solve { long long *clocks; };
struct Args { long long *clocks; int n_lp_workgroups; Solve solve; };
static long long *seen;
#define LPLB_STAMP_AT(ptr, k) seen = (ptr)
''' + "".join(macros) + '''
extern "C" long stamped(int which, unsigned block, unsigned blocks, int lps, long long *clocks) {
  blockIdx.x = block; gridDim.x = blocks;
  Args a{clocks, lps, {clocks}};
  if (which == 0) LPLB_STAMP(3); else if (which == 1) LPLB_PLAN_STAMP(3); else LPLB_MAP_STAMP(3);
  return reinterpret_cast<intptr_t>(seen);
}
''')
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", str(tmp_path / "stamps.cpp"), "-o", str(tmp_path / "stamps.so")],
                   check=True, capture_output=True)
    stamped = ctypes.CDLL(str(tmp_path / "stamps.so")).stamped
    stamped.restype, stamped.argtypes = ctypes.c_long, [ctypes.c_int, ctypes.c_uint, ctypes.c_uint, ctypes.c_int, ctypes.c_void_p]
    for which in range(3):
        for blocks in (1, 2, 7):
            places = [stamped(which, block, blocks, 1, 4096) for block in range(blocks)]
            assert all(p == 0 or p >= 4096 for p in places) and any(places)
            assert [stamped(which, block, blocks, 1, None) for block in range(blocks)] == [0] * blocks, which


def test_lps_are_packed_where_that_was_measured_to_pay(tmp_path):
    """Four LPs to a wave or one: the rule (lplb_amd/csrc/solve_pack.h) against the measurements that stand above it.  Nowhere may it choose
    the form that was slower by more than 3 % (two runs of one form differ by up to that)."""
    import subprocess
    (tmp_path / "pack.cpp").write_text('''
#include "solve_pack.h"
extern "C" int pays(int G, int D, int per_rank, int n_experts, int per_simd) { return lplb::packing_pays(G, D, per_rank, n_experts, per_simd); }
''')
    header = ROOT / "lplb_amd" / "csrc" / "solve_pack.h"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{header.parent}",
                    str(tmp_path / "pack.cpp"), "-o", str(tmp_path / "pack.so")], check=True, capture_output=True)
    pays = ctypes.CDLL(str(tmp_path / "pack.so")).pays
    text = header.read_text()
    counts = [int(n) for n in re.search(r"of a rank, in all((?: +\d+)+) LPs", text).group(1).split()]
    rows = re.findall(r"^//   \((\d+), (\d+)\) +(\d+) +(\d+) +((?:[\d.]+ / *[\d.]+ *)+)", text, flags=re.M)
    assert len(rows) >= 17 and counts[0] == 2048 and {(G, D) for G, D, *_ in rows} >= {("8", "1"), ("8", "2"), ("16", "1")}
    chosen = set()
    for G, D, per_rank, n_experts, times in rows:
        both = [(float(lone), float(packed)) for lone, packed in re.findall(r"([\d.]+) / *([\d.]+)", times)]
        assert len(both) == len(counts)
        for n, (lone, packed) in zip(counts, both):
            packs = pays(int(G), int(D), int(per_rank), int(n_experts), -(-n // 1024))
            chosen.add(packs)
            slower, faster = (packed, lone) if packs else (lone, packed)
            assert slower <= 1.03 * faster, (G, D, per_rank, n_experts, n, lone, packed)
    assert chosen == {0, 1}
    assert not any(pays(G, D, per_rank, per_rank * G, 1) for G in range(1, 17) for D in (1, 2, 4) for per_rank in (1, 32, 1024))   # alone on its SIMD
    # the batches that the GPU's test takes for packed ones and for lone ones are
    for name, r2o, ep, n_logical, n_inst, packed in BATCHED_LPS:
        n_lps = n_inst * (ep // len(r2o))
        assert pays(len(r2o), np.asarray(r2o).shape[1], n_logical // ep, n_logical, -(-n_lps // 1024)) == packed, name


def test_redirect_takes_as_many_chunks_per_pass_as_was_measured_to_pay(tmp_path):
    """Four or eight chunks: the rule (lplb_amd/csrc/redirect_chunks.h) against the measurements that stand above it.  Nowhere may it choose
    the form that was slower by more than 3 % (two runs of one form differ by up to that)."""
    import subprocess
    (tmp_path / "chunks.cpp").write_text('''
#include "redirect_chunks.h"
extern "C" int chunks(long long per_wave, int n_sets, int n_slices, int n_cus) { return lplb::redirect_chunks(per_wave, n_sets, n_slices, n_cus); }
''')
    header = ROOT / "lplb_amd" / "csrc" / "redirect_chunks.h"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{header.parent}",
                    str(tmp_path / "chunks.cpp"), "-o", str(tmp_path / "chunks.so")], check=True, capture_output=True)
    chunks = ctypes.CDLL(str(tmp_path / "chunks.so")).chunks
    chunks.argtypes = [ctypes.c_longlong, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    text = header.read_text()
    per_wave = [int(n) for n in re.search(r"chunks of a wave in all: ([\d, ]+)", text).group(1).split(", ")]
    rows = re.findall(r"^//  +(\d+) of +(\d+), +(\d+) +((?:[\d.]+ / *[\d.]+ *)+)", text, flags=re.M)
    assert len(rows) == 15 and per_wave[0] == 16
    chosen = set()
    for sets, _experts, slices, times in rows:
        both = [(float(four), float(eight)) for four, eight in re.findall(r"([\d.]+) / *([\d.]+)", times)]
        assert len(both) == len(per_wave)
        for n, (four, eight) in zip(per_wave, both):
            k = chunks(n, int(sets), int(slices), 256)
            chosen.add(k)
            slower, faster = (eight, four) if k == 8 else (four, eight)
            assert slower <= 1.03 * faster, (sets, slices, n, four, eight)
    assert chosen == {4, 8}
    assert [chunks(n, 16, 1, 256) for n in (1, 2, 3, 7, 8, 15)] == [1, 1, 2, 2, 4, 4]
    assert not any(chunks(n, sets, 129, 256) == 8 or chunks(n, sets, 1, 0) == 8 for n in range(1, 600) for sets in (0, 16, 128))


def test_the_last_wave_to_add_up_totals_sees_what_the_others_have_added(tmp_path):
    """With more than 64 slices several waves of a workgroup add to the same sums in LDS, count themselves, and the one that comes
    last reads the sums.  Nothing but fences keeps the compiler from moving the count ahead of a wave's own additions, or the
    reads ahead of the count: look for both, and for the waits that they become, where the waves do this."""
    import shutil
    import subprocess
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("no hipcc")
    probe = tmp_path / "probe.hip"
    probe.write_text('''
#include "plan_kernel.h"
using namespace lplb;
extern "C" __global__ void add_up(PlanArgs a, SliceTables t, uint32_t tag) {
  __shared__ int missing[2], block_sums[17];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  add_up_published<LONG_SLICES, Units::kTotals>(a, t, blockIdx.x, tag, lane, wave, missing, block_sums);
}
''')

    def compiled(form, *flags):
        out = tmp_path / "probe.out"
        subprocess.run([hipcc, "-O3", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-S", *flags,
                        f"-I{ROOT / 'lplb_amd' / 'csrc'}", f"-DLONG_SLICES={form}", str(probe), "-o", str(out)], check=True, capture_output=True)
        return out.read_text()

    for form in ("false", "true"):
        steps = ""
        for line in compiled(form, "-emit-llvm").split("define ")[1].splitlines():
            if "fence" in line:
                steps += "R" if "release" in line else "A"
            elif re.search(r"atomicrmw .*addrspace\(3\)", line):
                steps += "c" if "block_sums, i32 64)" in line else "+"
            elif re.search(r"= load .*addrspace\(3\)", line):
                steps += "l"
        assert re.fullmatch(r"\++RcAl+", steps), steps
        order = [m.group(1) for m in re.finditer(r"^\s+(ds_add_u32|ds_add_rtn_u32|ds_read\w+|s_waitcnt .*lgkmcnt\(0\))",
                                                 compiled(form), flags=re.M)]
        steps = "".join({"ds_add_u32": "+", "ds_add_rtn_u32": "c"}.get(o, "l" if o.startswith("ds_read") else "w") for o in order)
        assert re.search(r"\++w+cw+l", steps), steps


def test_the_lp_s_reciprocals_have_all_of_fp64(tmp_path):
    """An LP's step length is rounded to fp32 only at its end (minilp.cu:361 divides in fp64): with the hardware's estimate off by
    up to 2^-23 either way (v_rcp_f64's bound), the reciprocal keeps an error of that squared and the last roundings,
    and the quotient, corrected once more, one rounding only.  lplb_amd/csrc/reciprocal.h on the host, against long double."""
    import subprocess
    (tmp_path / "reciprocal.cpp").write_text('''
#define __device__
static double relative_error;
static double __builtin_amdgcn_rcp(double a) { return 1.0 / a * (1.0 + relative_error); }
#include "reciprocal.h"
extern "C" double step_length_error(double d, double estimate_error) {
  relative_error = estimate_error;
  const long double exact = (long double)0.999 / (long double)d;
  return (double)(((long double)lplb::step_length(d) - exact) / exact);
}
extern "C" double reciprocal_error(double d, double estimate_error) {
  relative_error = estimate_error;
  return (double)((long double)lplb::rcp_f64(d) * (long double)d - 1.0L);
}
''')
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", f"-I{ROOT / 'lplb_amd' / 'csrc'}",
                    str(tmp_path / "reciprocal.cpp"), "-o", str(tmp_path / "reciprocal.so")], check=True, capture_output=True)
    lib = ctypes.CDLL(str(tmp_path / "reciprocal.so"))
    for fn in (lib.step_length_error, lib.reciprocal_error):
        fn.restype, fn.argtypes = ctypes.c_double, [ctypes.c_double, ctypes.c_double]
    rng = np.random.default_rng(0)
    for d in np.exp(rng.uniform(np.log(1e-30), np.log(1e30), 5000)):
        off = float(rng.choice([-1, 1, rng.uniform(-1, 1)])) * 2.0 ** -23
        assert abs(lib.step_length_error(d, off)) <= 1.001 * 2.0 ** -53, (d, off)
        # the estimate's error squared; one rounding each of the residual (at most 2^-23 of the result) and of the sum
        assert abs(lib.reciprocal_error(d, off)) <= 1.01 * 2.0 ** -46 + 1.001 * 2.0 ** -53, (d, off)


@pytest.fixture(scope="module")
def admission(tmp_path_factory):
    """lplb_amd/csrc/plan_admit.h with eight blocks, driven from the host: (admit, launched, forget, idle, arrived)."""
    import subprocess
    d = tmp_path_factory.mktemp("admit")
    (d / "admit.cpp").write_text('''
#include "plan_admit.h"
using A = lplb::PlanAdmission<8>;
static A a;
static A::Admitted last;
extern "C" void reset() { a = A(); }
extern "C" void admit(long stream, float cost, int capturing, const int *arrived, int if_alone, int *out) {
  last = a.admit(reinterpret_cast<const void *>(stream), cost, capturing, arrived, if_alone);
  const int got[] = {last.slot, last.seq, last.wait_slices, last.wait_lps, last.wait_seq};
  for (int i = 0; i < 5; ++i) out[i] = got[i];
}
extern "C" void launched(int capturing, int slices, int lps) { a.launched(last, capturing, slices, lps); }
extern "C" void forget(long stream) { a.forget_captured(reinterpret_cast<const void *>(stream)); }
extern "C" void idle() { a.device_is_idle(); }
''')
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{ROOT / 'lplb_amd' / 'csrc'}",
                    str(d / "admit.cpp"), "-o", str(d / "admit.so")], check=True, capture_output=True)
    lib = ctypes.CDLL(str(d / "admit.so"))

    class Admission:
        """Streams are numbers; plan() admits and launches, and returns (slot, number, what it waits for or None)."""
        def __init__(self):
            self.arrived = (ctypes.c_int * 8)()
            lib.reset()

        def plan(self, stream, cost=0.1, capturing=False, slices=64, lps=1, if_alone=False):
            out = (ctypes.c_int * 5)()
            lib.admit(ctypes.c_long(stream), ctypes.c_float(cost), int(capturing), self.arrived, int(if_alone), out)
            if out[0] >= 0:
                lib.launched(int(capturing), slices, lps)
            return out[0], out[1], tuple(out[2:]) if out[2] else None

        def has_arrived(self, got):
            self.arrived[got[0]] = got[1]

        forget = staticmethod(lambda stream: lib.forget(ctypes.c_long(stream)))
        idle = staticmethod(lib.idle)
    return Admission


def _eight_streams_have_planned(admission):
    adm = admission()
    for stream in range(1, 9):
        got = adm.plan(stream)
        assert got[0] == stream - 1 and got[2] is None
        adm.has_arrived(got)
    return adm


def test_a_block_taken_over_inside_a_capture_is_waited_for_outside_it_too(admission):
    """A ninth stream takes a block over whose last launch has arrived but may still be reading.  If that happens in a
    capture, the wait that is recorded has not run when the stream's next plan is enqueued, or another graph is
    replayed: every launch of the stream waits until one outside a capture has."""
    adm = _eight_streams_have_planned(admission)
    first = adm.plan(9, capturing=True)
    assert first[0] >= 0 and first[2] == (64, 1, 1)
    assert adm.plan(9, capturing=True)[::2] == first[::2]     # a second graph may be replayed before the first
    assert adm.plan(9, slices=32)[::2] == first[::2]
    assert adm.plan(9)[::2] == (first[0], None) and adm.plan(9, capturing=True)[::2] == (first[0], None)
    # a takeover outside a capture: once
    adm = _eight_streams_have_planned(admission)
    assert adm.plan(9)[2] == (64, 1, 1) and adm.plan(9)[2] is None


def test_a_short_plan_queued_behind_a_long_one_does_not_hide_its_share_of_the_gpu(admission):
    adm = admission()
    adm.plan(1, cost=0.6)
    short = adm.plan(1, cost=0.1)
    assert adm.plan(2, cost=0.3)[0] == -1     # 0.6 may still be executing
    adm.has_arrived(short)
    assert adm.plan(2, cost=0.3)[0] == 1
    adm.plan(1, cost=0.1)
    assert adm.plan(2, cost=0.6)[0] == 1      # the long one is over


def test_forgetting_captured_plans_does_not_forget_a_plan_that_still_executes(admission):
    """The graphs captured on a stream may be gone while a plan enqueued outside a capture is still executing there: its
    block does not pass on before that launch has arrived, its share of the GPU stays taken, and the next stream waits
    for its readers.  Captured launches have no number, so that a replay leaves none over a later launch's."""
    adm = _eight_streams_have_planned(admission)
    running = adm.plan(1, cost=0.5, slices=200, lps=3)
    captured = adm.plan(1, capturing=True)
    assert captured == (0, -1, None)
    adm.forget(1)
    assert adm.plan(9, cost=0.4)[0] == -1                # 0.5 of the GPU is still taken
    for stream in range(2, 9):
        adm.plan(stream, cost=0.01)
    assert adm.plan(9, cost=0.01)[0] == -1               # and so is block 0, like the others
    adm.has_arrived(running)
    got = adm.plan(9, cost=0.4)
    assert got[0] == 0 and got[2] == (200, 3, running[1])


def test_a_plan_takes_more_of_the_gpu_only_while_it_is_alone(admission):
    """Short slices take twice the workgroups: only while no other stream's plan may be executing, and not where a captured graph
    keeps the share, its own or that of one captured on the stream before."""
    adm = admission()
    other = adm.plan(1)
    assert adm.plan(2, if_alone=True)[0] == -1 and adm.plan(2)[0] == 1
    adm.idle()
    assert adm.plan(3, if_alone=True)[0] == 2 and adm.plan(3, if_alone=True)[0] == 2   # (its own last one is ahead of it on the stream)
    assert adm.plan(4, if_alone=True)[0] == -1
    adm.idle()
    assert adm.plan(3, if_alone=True, capturing=True)[0] == -1 and other[0] == 0
    assert adm.plan(3, capturing=True)[0] == 2
    assert adm.plan(3, if_alone=True)[0] == -1 and adm.plan(3)[0] == 2
    adm.forget(3)
    adm.idle()
    assert adm.plan(3, if_alone=True)[0] == 2


def test_as_many_streams_as_there_are_blocks_keep_one_each(admission):
    """Streams that plan in turn settle on a block each, whoever used the blocks before: their plans then wait for
    no other stream.  Of more streams than there are blocks, all but one block's worth keep theirs."""
    for streams, most_waits in ((8, 0), (9, 2), (12, 5)):   # a round, once they have settled
        adm = _eight_streams_have_planned(admission)
        for rep in range(12):
            waits = 0
            for stream in range(11, 11 + streams):
                got = adm.plan(stream)
                adm.has_arrived(got)
                waits += got[2] is not None
        assert waits <= most_waits, (streams, waits)


def test_no_kernel_spills_vector_registers():
    """The build leaves the compiler's per-kernel resource report next to each object
    (lplb_amd/csrc/*.resources.txt).  No kernel may spill vector registers: besides being slow,
    a spill placed where only part of a wave is active (seen with this compiler in a variant of the
    one-launch plan, between a divergent loop and the instruction that restores the execution mask) loses
    the value in the inactive lanes.  The variants are sized so that none spills; this keeps it so."""
    reports = sorted((Path(__file__).parent.parent / "lplb_amd" / "csrc").glob("*.resources.txt"))
    if not reports:
        pytest.skip("no resource reports: the library was not built here")
    n_kernels, spilling = 0, []
    for report in reports:
        name = None
        for line in report.read_text().splitlines():
            m = re.search(r"Function Name: (\S+)", line)
            if m:
                name, n_kernels = m.group(1), n_kernels + 1
            m = re.search(r"VGPRs Spill: (\d+)", line)
            if m and int(m.group(1)) > 0:
                spilling.append((report.name, name, int(m.group(1))))
    assert n_kernels > 100, n_kernels
    assert not spilling, spilling


def _device_code(library):
    """(kernel, its instructions as (address, text, branch target or None)) of the gfx950 code in a library built here."""
    import shutil
    import subprocess
    import tempfile
    objdump = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
    if not Path(objdump).exists():
        pytest.skip("no llvm-objdump")
    with tempfile.TemporaryDirectory() as d:
        shutil.copy(library, d)
        subprocess.run([objdump, "--offloading", Path(library).name], cwd=d, check=True, capture_output=True)
        for part in sorted(Path(d).glob("*gfx950")):
            text = subprocess.run([objdump, "-d", str(part)], check=True, capture_output=True, text=True).stdout
            for kernel in re.split(r"^[0-9a-f]+ <", text, flags=re.M)[1:]:
                yield kernel.split(">")[0], _instructions(kernel)


def _instructions(text):
    found = re.findall(r"^\s+(\S.*?)\s*// ([0-9A-F]+): [0-9A-F ]+(?:<\S+\+0x([0-9a-f]+)>)?", text, flags=re.M)
    first = int(found[0][1], 16) if found else 0
    return [(int(at, 16), op, first + int(target, 16) if target else None) for op, at, target in found]


def _registers(text):
    single = {int(r) for r in re.findall(r"\bv(\d+)\b", text)}
    return single.union(*(range(int(a), int(b) + 1) for a, b in re.findall(r"\bv\[(\d+):(\d+)\]", text)))


def _copies_in_switched_off_lanes(code):
    """Vector copies and spills that stand where control has come together again but the lanes are still off (between the
    target of a skip, or the end of a loop, and the instruction that restores the execution mask), or between the
    instruction that narrows the mask and its branch, and whose result nothing reads before the mask changes: only a live
    range that the register allocator has split looks like that, and the lanes that are off lose its value."""
    copy = re.compile(r"v_mov_b(?:32|64)\w* v\S+ v|v_accvgpr|scratch_")
    index = {at: i for i, (at, _, _) in enumerate(code)}
    restores, narrows = r"s_(?:or|andn2)_saveexec|s_or_b64 exec,", r"s_(?:and|andn2)_saveexec|s_(?:mov|and|andn2)_b64 exec,"
    starts = [(index[target], restores) for _, op, target in code if op.startswith("s_cbranch_execz") and target in index]
    starts += [(i + 1, restores) for i, (_, op, _) in enumerate(code) if op.startswith("s_cbranch_execnz")]
    starts += [(i + 1, "s_cbranch_exec") for i, (_, op, _) in enumerate(code) if re.match(narrows, op)]
    hits = []
    for start, until in sorted(set(starts)):
        copies = []
        for at, op, _ in code[start:start + 200]:
            if re.match(until, op):
                hits += [(hex(where), text) for where, text, _ in copies]
                break
            if re.match(r"s_\w+saveexec|s_\w+ exec,|s_c?branch|s_endpgm", op):
                break
            operands = op.split(None, 1)[1] if " " in op else ""
            read = _registers(operands if op.startswith(("ds_", "global_", "buffer_", "flat_")) else operands.partition(",")[2])
            copies = [c for c in copies if not c[2] & read]
            if copy.match(op):
                copies.append((at, op, _registers(operands.partition(",")[0])))
    return hits


def test_no_kernel_copies_a_register_while_its_lanes_are_off():
    """This compiler, short of registers, splits live ranges and may place the copy where the lanes are still switched off
    (it lost the ids of one chunk of 64 tokens in every wave of a variant of the one-launch plan).  The kernels are built so that it does
    not have to; this looks through all of them in the built library."""
    planted = """
	s_cbranch_execz 3      // 000000000100: BF880003 <kernel+0x10>
	global_store_dword v[2:3], v6, off // 000000000104: DC708000 007F0602
	s_cbranch_execnz 65533 // 00000000010C: BF89FFFD <kernel+0x4>
	v_mov_b32_e32 v26, v57 // 000000000110: 7E340339
	s_or_b64 exec, exec, s[4:5] // 000000000114: 87FE047E
	v_and_b32_e32 v108, 0xffff, v38 // 000000000118: 26D84CFF 0000FFFF
"""
    assert _copies_in_switched_off_lanes(_instructions(planted)) != []
    assert _copies_in_switched_off_lanes(_instructions(planted.replace("v26, v57 //", "v26, 0 //"))) == []
    n_kernels, lost = 0, []
    for name, code in _device_code(_native.LIB_PATH):
        n_kernels += 1
        lost += [(name, hit) for hit in _copies_in_switched_off_lanes(code)]
    assert n_kernels > 100, n_kernels
    assert not lost, lost[:20]


def test_prepared_mapping_follows_the_mapping_and_not_its_address(monkeypatch):
    """A new mapping may come to lie where an old one was, with the same version: the tables prepared for the redirect
    are built anew for it, and for one changed in place, but not for the same one again."""
    planner = Planner(torch.from_numpy(topology.CUBE_8P2E), 272, 256, 8, device="cpu", gpus_per_node=8)

    class Solver:
        def prepare_mapping(self, o2r, phy2log):
            return phy2log.clone()
    monkeypatch.setattr("lplb_amd.planner._device_index", lambda t: 0)
    monkeypatch.setattr("lplb_amd.planner._stream_on", lambda i: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    planner._solver = Solver()
    planner.__class__ = type("OnCpu", (Planner,), {"solver": property(lambda self: self._solver)})
    memory = planner.phy2log.numpy().copy()
    planner.phy2log = torch.from_numpy(memory)
    first = planner._prepared_mapping()
    assert planner._prepared_mapping() is first
    address = planner.phy2log.data_ptr()
    memory[:] = memory[::-1].copy()
    planner.phy2log = torch.from_numpy(memory)
    assert planner.phy2log.data_ptr() == address and planner.phy2log._version == 0
    assert torch.equal(planner._prepared_mapping(), planner.phy2log)
    planner.phy2log[0] += 1
    assert torch.equal(planner._prepared_mapping(), planner.phy2log)
    planner.update_redundancy_mapping(torch.arange(256) ** 2)
    assert torch.equal(planner._prepared_mapping(), planner.phy2log)


def test_prepared_mapping_is_used_on_the_stream_that_built_it_only(monkeypatch):
    """Nothing orders another stream behind the launch that fills the tables, and a captured launch fills them at its
    replays only."""
    planner = Planner(torch.from_numpy(topology.CUBE_8P2E), 272, 256, 8, device="cpu", gpus_per_node=8)
    built, now = [], {"stream": 1, "capturing": False}

    class Solver:
        def prepare_mapping(self, o2r, phy2log):
            assert not now["capturing"]
            built.append(now["stream"])
            return phy2log.clone()
    planner._solver = Solver()
    planner.__class__ = type("OnCpu", (Planner,), {"solver": property(lambda self: self._solver)})
    monkeypatch.setattr("lplb_amd.planner._device_index", lambda t: 0)
    monkeypatch.setattr("lplb_amd.planner._stream_on", lambda i: now["stream"])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: now["capturing"])
    tables = {}
    for now["stream"], now["capturing"], has_one in [(1, True, False), (1, False, True), (2, True, False), (2, False, True),
                                                     (1, True, True), (1, False, True), (2, True, True)]:
        table = planner._prepared_mapping()
        assert (table is not None) == has_one
        assert not has_one or tables.setdefault(now["stream"], table) is table
    assert built == [1, 2]
    now["capturing"] = False
    for now["stream"] in range(3, 40):
        planner._prepared_mapping()
    assert len(planner._prepared[5]) == 16


def test_binding_is_that_of_this_python_and_torch(monkeypatch):
    """Another interpreter does not find the module, one with another torch is told to build it again."""
    import sysconfig
    _native.load()
    assert Path(_native._binding.__file__).name == "_binding" + sysconfig.get_config_var("EXT_SUFFIX")
    monkeypatch.setattr(_native, "_lib", None)
    monkeypatch.setattr(torch, "__version__", "0.1.2+other")
    with pytest.raises(RuntimeError, match="built for torch"):
        _native.load()


def test_build_is_for_the_running_interpreter(monkeypatch):
    import subprocess
    import sys
    commands = []

    def run(command, **kw):
        commands.append(command)
        return subprocess.CompletedProcess(command, 0, "", "")
    monkeypatch.setattr(_native.subprocess, "run", run)
    _native.build()
    assert f"PYTHON={sys.executable}" in commands[0]


def test_placement_needs_no_gpu_library(tmp_path):
    """Expert placement runs on the host, also where neither the GPU library nor the binding has been built."""
    import shutil
    import subprocess
    import sys
    shutil.copytree(ROOT / "lplb_amd", tmp_path / "lplb_amd", ignore=shutil.ignore_patterns("_binding*", "liblplb_hip.so", "csrc"))
    program = """
import numpy as np, torch
from lplb_amd import Planner, _native, eplb, topology
assert not _native.LIB_PATH.exists()
planner = Planner(torch.from_numpy(topology.CUBE_8P2E), 272, 256, 8, device="cpu", gpus_per_node=8)
planner.update_redundancy_mapping(torch.arange(256) ** 2)
eplb.rebalance_experts(np.arange(64, dtype=np.float32)[None], 72, 4, 2, 8)
try:
    eplb.rebalance_experts(np.zeros((1, 64), np.float32), 71, 4, 2, 8)
except AssertionError as e:
    assert "71" in str(e), e
else:
    raise SystemExit("71 physical experts on 8 GPUs")
print("placed")
"""
    got = subprocess.run([sys.executable, "-c", program], cwd=tmp_path, capture_output=True, text=True)
    assert got.returncode == 0 and got.stdout.strip() == "placed", got.stderr[-2000:]


def test_a_deployment_that_the_gpu_does_not_place_allocates_nothing_there(monkeypatch):
    """Whether the placement kernel covers a deployment is asked before its tables are allocated, once per deployment; and the
    question refuses what is no deployment at all."""
    lib = _native.load()
    for name, (r2o, ep, n_logical, replicas, covered) in PLACEMENTS.items():
        assert lib.lplb_place_experts_covers(*r2o.shape, ep, n_logical, n_logical + replicas * ep, ep // 8) == covered, name
    assert lib.lplb_place_experts_covers(8, 2, 8, 128, 144, 1) == 1
    for wrong in ((0, 2, 8, 128, 144, 1), (8, 0, 8, 128, 144, 1), (8, 2, 12, 128, 144, 1), (8, 2, 8, 129, 144, 1), (8, 2, 8, 128, 128, 1),
                  (8, 2, 8, 128, 145, 1), (8, 2, 8, 128, 144, 0), (8, 2, 8, -128, 144, 1), (8, 2, 8, 128, 136, 1), (8, 2, 8, 8, 24, 1)):
        assert lib.lplb_place_experts_covers(*wrong) == 0, wrong

    class History:
        dtype, device = torch.int64, torch.device("cuda", 0)
        is_contiguous, numel, data_ptr = staticmethod(lambda: True), staticmethod(lambda: 136), staticmethod(lambda: 0)
    asked = []

    class Library:
        lplb_place_experts_covers = staticmethod(lambda *shape: asked.append(shape) or lib.lplb_place_experts_covers(*shape))

    def no_tables(*args, **kwargs):
        raise AssertionError("a table was allocated")
    monkeypatch.setattr(_native, "load", lambda: Library)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch, "empty", no_tables)
    _native.placement_covers.cache_clear()
    for _ in range(3):
        assert _native.place_experts(History, torch.from_numpy(topology.CUBE_8P2E), 8, 152, 1) is None
    assert asked == [(8, 2, 8, 136, 152, 1)]


def test_which_large_nodes_the_gpu_places():
    """Up to 384 experts packed at once, and everything that the call for smaller nodes covers."""
    covers = _native.load().lplb_place_on_large_nodes_covers
    for name, (r2o, ep, n_logical, replicas, covered) in PLACEMENTS.items():
        assert covers(*r2o.shape, ep, n_logical, n_logical + replicas * ep, ep // 8) == 1, name
    for per_node, covered in ((136, 1), (256, 1), (384, 1), (392, 0)):
        assert covers(8, 2, 8, per_node, per_node + 16, 1) == covered, per_node
    assert covers(8, 2, 16, 512, 512 + 32, 2) == 1 and covers(8, 2, 16, 512, 512 + 32, 1) == 0   # a node each; both groups on one
    assert covers(8, 2, 8, 129, 144, 1) == 0 and covers(0, 2, 8, 128, 144, 1) == 0               # no deployments


def test_placement_reports_memory_that_runs_out():
    """No C++ exception leaves the library: a call whose working memory cannot be had fails like any other."""
    import subprocess
    import sys
    program = """
import resource
import numpy as np
from lplb_amd import _native, eplb
_native.load_host()
n = 1 << 24
weight, pack, rank = np.zeros((1, n), np.float32), np.empty((1, n), np.int64), np.empty((1, n), np.int64)
r2o, out = np.zeros((1, 1), np.int32), np.zeros(8 * n, np.int32)
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + (1 << 20), resource.RLIM_INFINITY))
lib = _native.load_host()
p = lambda a: a.ctypes.data
codes = [lib.lplb_balanced_packing(p(weight), 1, n, 2, p(pack), p(rank)),
         lib.lplb_rebalance_experts(p(weight), 1, n, n, 1, 1, 1, p(pack), p(rank), p(pack)),
         lib.lplb_build_mapping(None, None, p(r2o), 1, 1, 1, n, n, 1, p(out), p(out), p(out))]
resource.setrlimit(resource.RLIMIT_AS, (resource.RLIM_INFINITY, resource.RLIM_INFINITY))
print(codes, lib.lplb_last_error())
"""
    got = subprocess.run([sys.executable, "-c", program], cwd=ROOT, capture_output=True, text=True)
    assert got.returncode == 0 and got.stdout.startswith("[1, 1, 1] b'expert placement"), (got.returncode, got.stdout, got.stderr[-500:])


def test_compiled_solver_takes_the_reference_argument_list():
    """csrc/plugin.cpp:665-667 / lplb/planner.py:26-35: (resource_path, n_group, group_size, dup_per_rank,
    block_dim, n_local_experts, n_combined_experts, pg)."""
    from lplb_amd import _native
    short = _native.CompiledSolver(2, 8, 2, 34, 1)
    ref = _native.CompiledSolver("/somewhere/resources", 2, 8, 2, 256, 34, 1, None)
    kw = _native.CompiledSolver(resource_path="x", n_group=2, group_size=8, dup_per_rank=2, block_dim=256,
                                n_local_experts=34, n_combined_experts=1, pg="a group")
    for s_ in (ref, kw):
        assert (s_.n_group, s_.group_size, s_.dup_per_rank, s_.n_local_experts, s_.n_combined_experts, s_.n_experts) == \
               (short.n_group, short.group_size, short.dup_per_rank, short.n_local_experts, short.n_combined_experts,
                short.n_experts)
    assert kw.pg == "a group" and ref.pg is None
    with pytest.raises(TypeError):
        _native.CompiledSolver("/somewhere/resources", 2, 8, 2, 256, 34)
    with pytest.raises(TypeError):
        _native.CompiledSolver(2, 8, 2, 34, 1, None)
