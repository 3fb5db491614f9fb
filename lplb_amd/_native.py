"""Binding of ``liblplb_hip.so`` and the ``CompiledSolver`` facade the planner talks to: ctypes for
setting up and looking into, ``csrc/binding.cpp`` for what runs per batch.  The facade keeps the method names, argument order, return values and
argument checks of the reference's pybind11 class (csrc/plugin.cpp:459-470,
491-660); underneath it only forwards device pointers and the current stream to
the C ABI declared in ``include/lplb_hip.h``.

There is no CPU or pure-PyTorch fallback: if the shared library is missing or a
tensor is not on a GPU, the call raises.
"""
from __future__ import annotations

import ctypes
import functools
import re
import subprocess
import sys
from pathlib import Path

import torch

_PKG = Path(__file__).resolve().parent
LIB_PATH = _PKG / "liblplb_hip.so"
HOST_LIB_PATH = _PKG / "liblplb_host.so"   # expert placement alone, for hosts without a GPU
ABI_VERSION = 7
# limits of lplb_count_totals (LPLB_COUNT_TOTALS_MAX_* of include/lplb_hip.h)
COUNT_TOTALS_MAX_INDICES = 131072
COUNT_TOTALS_MAX_EXPERTS = 1024

STEP_REFERENCE_WINDOW = 0
STEP_FULL_MAX = 1
REFERENCE_STEPS = 5

_lib: ctypes.CDLL | None = None
_host_lib: ctypes.CDLL | None = None
_binding = None   # the extension module of csrc/binding.cpp, once load() has run

_vp = ctypes.c_void_p
_i = ctypes.c_int
_i64 = ctypes.c_int64

_SIGNATURES = {
    "lplb_abi_version": (_i, []),
    "lplb_last_error": (ctypes.c_char_p, []),
    "lplb_time_next_launch": (None, [_vp, _vp]),
    "lplb_copy_calibration": (_i, [_vp, _vp, _i64, _vp]),
    "lplb_copy_calibration_series": (_i, [_vp, _vp, _i64, _i, _vp, _vp, _vp]),
    "lplb_slice_histogram_series": (_i, [_vp, _i64, _i, _i, _vp, _i, _vp, _vp, _vp]),
    "lplb_copy_shape_series": (_i, [_vp, _vp, _i64, _i, _i, _i, _i, _i, _vp, _vp, _vp]),
    "lplb_map_idx_prepared_series": (_i, [_vp, _vp, _vp, _vp, _i64, _i, _i, _i, _i, _i, _i, _vp, _i, _vp, _vp, _vp]),
    "lplb_count_idx": (_i, [_vp, _i64, _i, _i, _vp, _vp]),
    "lplb_count_totals": (_i, [_vp, _i64, _i, _vp, _vp]),
    "lplb_count_totals_add": (_i, [_vp, _i64, _i, _vp, _vp, _vp]),
    "lplb_solve": (_i, [_vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _vp, _vp, _i, _i, _vp]),
    "lplb_solve_batched": (_i, [_vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _vp, _vp, _i, _i, _vp]),
    "lplb_map_idx": (_i, [_vp, _vp, _vp, _vp, _vp, _i64, _i, _i, _i, _i, _i, _i, _vp, _vp, _vp]),
    "lplb_prepared_mapping_bytes": (_i64, [_i, _i, _i, _i, _i]),
    "lplb_prepare_mapping": (_i, [_vp, _vp, _i, _i, _i, _i, _i, _vp, _i64, _vp]),
    "lplb_map_idx_prepared": (_i, [_vp, _vp, _vp, _vp, _i64, _i, _i, _i, _i, _i, _i, _vp, _vp, _vp]),
    "lplb_plan_set_cooperative": (_i, [_i]),
    "lplb_plan_forget_captured": (_i, [_vp]),
    "lplb_plan_sync_timeouts": (_i, [_vp]),
    "lplb_plan_poll_timeouts": (_i, [_vp, _vp]),
    "lplb_plan_one_launch_count": (_i, [_vp]),
    "lplb_plan_inject_fault": (_i, [_i, _i]),
    "lplb_count_one_launch_count": (_i, [_vp]),
    "lplb_count_recounts": (_i, [_vp]),
    "lplb_count_inject_fault": (_i, []),
    "lplb_plan": (_i, [_vp, _i64, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _vp]),
    "lplb_balanced_packing": (_i, [_vp, _i, _i, _i, _vp, _vp]),
    "lplb_replicate_experts": (_i, [_vp, _i, _i, _i, _vp, _vp, _vp]),
    "lplb_rebalance_experts": (_i, [_vp, _i, _i, _i, _i, _i, _i, _vp, _vp, _vp]),
    "lplb_build_mapping": (_i, [_vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _vp, _vp, _vp]),
    "lplb_place_experts_covers": (_i, [_i, _i, _i, _i, _i, _i]),
    "lplb_place_on_large_nodes_covers": (_i, [_i, _i, _i, _i, _i, _i]),
    "lplb_place_on_large_nodes": (_i, [_vp, _i, _vp, _i, _i, _i, _i, _i, _i, _vp, _vp, _vp, _vp]),
    "lplb_place_on_large_nodes_begin": (_i, [_vp, _i, _vp, _i, _i, _i, _i, _i, _i, _vp, _vp, _vp, _vp]),
    "lplb_place_wait": (_i, [_vp]),
    "lplb_place_experts": (_i, [_vp, _i, _vp, _i, _i, _i, _i, _i, _i, _vp, _vp, _vp, _vp]),
    "lplb_plan_noalloc": (_i, [_vp, _i64, _vp, _vp, _vp, _vp, _i, _i, _i, _i, _i, _i, _vp, _vp, _vp, _vp, _vp, _vp, _i, _i, _vp]),
}


_HOST_FUNCTIONS = ("lplb_last_error", "lplb_balanced_packing", "lplb_replicate_experts", "lplb_rebalance_experts",
                   "lplb_build_mapping")


def build(verbose: bool = False) -> Path:
    """Compile the HIP library for gfx950 and the Python binding with the Makefile in ``csrc/``."""
    proc = subprocess.run(["make", "-C", str(_PKG / "csrc"), "-B", "-j4", f"PYTHON={sys.executable}"], capture_output=True,
                          text=True)
    if verbose or proc.returncode != 0:
        print(proc.stdout)
        print(proc.stderr)
    if proc.returncode != 0:
        raise RuntimeError("building liblplb_hip.so failed")
    return LIB_PATH


def load() -> ctypes.CDLL:
    global _lib, _binding
    if _lib is not None:
        return _lib
    if not LIB_PATH.exists():
        raise RuntimeError(
            f"{LIB_PATH} is missing: build it with `make -C {_PKG / 'csrc'}` "
            "(hipcc, --offload-arch=gfx950). There is no fallback path.")
    lib = ctypes.CDLL(str(LIB_PATH))
    for name, (res, args) in _SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    if lib.lplb_abi_version() != ABI_VERSION:
        raise RuntimeError(f"liblplb_hip.so has ABI {lib.lplb_abi_version()}, expected {ABI_VERSION}")
    try:
        from . import _binding as binding
    except ImportError as e:
        raise RuntimeError(f"lplb_amd/_binding for this Python and torch is missing or does not load: build it with "
                           f"`make -C {_PKG / 'csrc'} PYTHON={sys.executable}`") from e
    if binding.torch_version != re.match(r"[\d.]*\d|", torch.__version__).group():   # (without a pre-release's letters)
        raise RuntimeError(f"lplb_amd/_binding was built for torch {binding.torch_version}, this is {torch.__version__}: build it "
                           f"again with `make -B -C {_PKG / 'csrc'} PYTHON={sys.executable}`")
    binding.bind(str(LIB_PATH), UnsupportedShape)
    _lib, _binding = lib, binding
    return lib


def load_host() -> ctypes.CDLL:
    """The functions that run on the host (expert placement), from a library that needs neither a GPU nor ROCm."""
    global _host_lib
    if _host_lib is None:
        if not HOST_LIB_PATH.exists():
            raise RuntimeError(f"{HOST_LIB_PATH} is missing: build it with `make -C {_PKG / 'csrc'} host` (a C++ compiler)")
        lib = ctypes.CDLL(str(HOST_LIB_PATH))
        for name in _HOST_FUNCTIONS:
            fn = getattr(lib, name)
            fn.restype, fn.argtypes = _SIGNATURES[name]
        _host_lib = lib
    return _host_lib


def exported_symbols() -> list[str]:
    return list(_SIGNATURES)


def set_plan_cooperative(enabled: bool) -> None:
    """Let ``plan`` run short batches as one kernel launch (default) or always as the chain of kernels."""
    _check(load().lplb_plan_set_cooperative(1 if enabled else 0))


def plan_forget_captured(stream: "torch.cuda.Stream") -> None:
    """Give back the share of the GPU that one-launch plans captured on ``stream`` keep reserved; for callers
    who have destroyed every graph that holds such a plan."""
    _check(load().lplb_plan_forget_captured(stream.cuda_stream))


def plan_sync_timeouts() -> int:
    """Waits between workgroups of the one-launch plan that ran out on the current device (0 when healthy)."""
    count = ctypes.c_int(-1)
    _check(load().lplb_plan_sync_timeouts(ctypes.byref(count)))
    return count.value


def plan_poll_timeouts(dst: torch.Tensor, stream: int | None = None) -> None:
    """Enqueue the health report: dst (two int32, on the GPU or in pinned host memory) receives the number of
    waits that ran out on the current device and the number of blocks of counters switched off."""
    _require(dst.dtype == torch.int32 and dst.numel() >= 2 and dst.is_contiguous() and (dst.is_cuda or dst.is_pinned()),
             "dst: two int32 on the GPU or in pinned host memory")
    _check(load().lplb_plan_poll_timeouts(dst.data_ptr(), stream))


def plan_one_launch_count() -> int:
    """Plans of this process that ran as one kernel launch (the others ran the chain of kernels)."""
    count = ctypes.c_longlong(-1)
    _check(load().lplb_plan_one_launch_count(ctypes.byref(count)))
    return count.value


def count_one_launch_count() -> int:
    """Histograms with running sums of this process that ran as one kernel launch (the others took two)."""
    count = ctypes.c_longlong(-1)
    _check(load().lplb_count_one_launch_count(ctypes.byref(count)))
    return count.value


def count_recounts() -> int:
    """How often slices of such a histogram have counted for themselves on the current device (waits for it)."""
    count = ctypes.c_int(-1)
    _check(load().lplb_count_recounts(ctypes.byref(count)))
    return count.value


# LPLB_INT32 ... LPLB_FLOAT64 of include/lplb_hip.h
_HISTORY_TYPES = {torch.int32: 0, torch.int64: 1, torch.float32: 2, torch.float64: 3}


@functools.lru_cache(maxsize=256)
def placement_covers(group_size: int, dup_per_rank: int, ep_size: int, n_logical: int, n_physical: int, n_nodes: int,
                     large_nodes: bool = False) -> bool:
    """Whether place_experts has a kernel for this deployment.  (Kept: a call that is refused costs the host path as much as
    the question.)"""
    lib = load()
    covers = lib.lplb_place_on_large_nodes_covers if large_nodes else lib.lplb_place_experts_covers
    return covers(group_size, dup_per_rank, ep_size, n_logical, n_physical, n_nodes) != 0


def place_experts(history: torch.Tensor, r2o: torch.Tensor, ep_size: int, n_physical: int, n_nodes: int,
                  large_nodes: bool = False) -> torch.Tensor | None:
    """build_redundancy_mapping for a history on the current device, by a kernel there: its three arrays as parts of
    one int32 tensor [n_physical + 3 * n_logical] on that device, complete on return; None if the kernel does not cover it.
    large_nodes: also with more than 128 experts on a node."""
    begun = place_experts_begin(history, r2o, ep_size, n_physical, n_nodes, large_nodes)
    if begun is None:
        return None
    place_wait(begun[1])
    return begun[0]


def place_experts_begin(history: torch.Tensor, r2o: torch.Tensor, ep_size: int, n_physical: int, n_nodes: int,
                        large_nodes: bool = True) -> tuple[torch.Tensor, int] | None:
    """place_experts without the wait: the table and what to hand to place_wait before anything but this stream's work reads it."""
    kind = _HISTORY_TYPES.get(history.dtype)
    if kind is None or not history.is_contiguous() or _device_index(history) != torch.cuda.current_device():
        return None
    n_logical = history.numel()
    group_size, dup_per_rank = r2o.shape
    if not placement_covers(group_size, dup_per_rank, ep_size, n_logical, n_physical, n_nodes, large_nodes):
        return None
    table = torch.empty(n_physical + 3 * n_logical, dtype=torch.int32, device=history.device)
    at, stream = table.data_ptr(), _stream(history)
    _check(load().lplb_place_on_large_nodes_begin(history.data_ptr(), kind, r2o.data_ptr(), group_size, dup_per_rank, ep_size, n_logical,
                                                  n_physical, n_nodes, at, at + 4 * n_physical, at + 4 * (n_physical + 2 * n_logical), stream))
    return table, stream


def place_wait(stream: int) -> None:
    _check(load().lplb_place_wait(stream))


class UnsupportedShape(RuntimeError):
    """The library has no kernel for this shape (LPLB_EUNSUPPORTED)."""


def _check(rc: int) -> None:
    if rc != 0:
        kind = UnsupportedShape if rc == 2 else RuntimeError
        raise kind(f"lplb_hip error {rc}: {load().lplb_last_error().decode()}")


def check_host(rc: int) -> None:
    """Result of the host-side placement functions, whose argument checks are assertions like the reference's."""
    if rc != 0:
        raise AssertionError(load_host().lplb_last_error().decode())


def _require(cond: bool, what: str) -> None:
    if not cond:
        raise RuntimeError(f"LPLB assertion failed: {what}")


# Handle of torch's current stream on the device with this index (the raw query is ten times cheaper than
# building a torch.cuda.Stream object, which matters at 10 us per plan).
_stream_on = getattr(torch._C, "_cuda_getCurrentRawStream", None) or (lambda i: torch.cuda.current_stream(i).cuda_stream)


def _device_index(t: torch.Tensor) -> int:
    return t.device.index if t.device.index is not None else torch.cuda.current_device()


def _stream(t: torch.Tensor) -> int:
    """Handle of torch's current stream on t's device."""
    return _stream_on(_device_index(t))


class CompiledSolver:
    """Launches the three planning kernels for one (n_group, G, D, P, C) shape."""

    def __init__(self, *args, **kwargs) -> None:
        """Two ways to construct one.  The reference's own argument list (csrc/plugin.cpp:665-667,
        as lplb/planner.py:26-35 passes it):
            CompiledSolver(resource_path, n_group, group_size, dup_per_rank, block_dim,
                           n_local_experts, n_combined_experts, pg)
        where resource_path (the CUDA templates' folder) and block_dim (every kernel here picks its
        own workgroup size) are accepted and ignored and pg is kept as .pg for the caller; or the
        five numbers that matter:
            CompiledSolver(n_group, group_size, dup_per_rank, n_local_experts, n_combined_experts)"""
        self.pg = None
        if args and isinstance(args[0], (str, bytes)) or "resource_path" in kwargs:
            names = ("resource_path", "n_group", "group_size", "dup_per_rank", "block_dim", "n_local_experts",
                     "n_combined_experts", "pg")
        else:
            names = ("n_group", "group_size", "dup_per_rank", "n_local_experts", "n_combined_experts")
        if len(args) > len(names):
            raise TypeError(f"CompiledSolver takes {len(names)} arguments {names}, got {len(args)}")
        given = dict(zip(names, args))
        for k, v in kwargs.items():
            if k not in names or k in given:
                raise TypeError(f"CompiledSolver: unexpected or repeated argument {k!r}")
            given[k] = v
        missing = [k for k in names if k not in given and k != "pg"]
        if missing:
            raise TypeError(f"CompiledSolver: missing arguments {missing}")
        n_group, group_size, dup_per_rank = int(given["n_group"]), int(given["group_size"]), int(given["dup_per_rank"])
        n_local_experts, n_combined_experts = int(given["n_local_experts"]), int(given["n_combined_experts"])
        self.pg = given.get("pg")
        self.lib = load()
        self.n_group = n_group
        self.group_size = group_size
        self.dup_per_rank = dup_per_rank
        self.n_local_experts = n_local_experts
        self.n_combined_experts = n_combined_experts
        # csrc/plugin.cpp:464-466
        self.n_experts = (n_local_experts - dup_per_rank * n_combined_experts) * group_size * n_group
        self.step_rule = STEP_REFERENCE_WINDOW
        self.n_steps = REFERENCE_STEPS

    # -- csrc/plugin.cpp:491-578 -------------------------------------------------
    def solve(self, local_workload: torch.Tensor, r2o: torch.Tensor, phy2log: torch.Tensor,
              avail_num: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
        return _binding.solve(self.n_group, self.group_size, self.dup_per_rank, self.n_combined_experts,
                              self.n_local_experts, self.step_rule, self.n_steps, local_workload, r2o, phy2log, avail_num)

    def solve_batched(self, workloads: torch.Tensor, r2o: torch.Tensor, phy2log: torch.Tensor,
                      avail_num: torch.Tensor, want_global: bool = False):
        """workloads int32 [n_instances, n_group, G, L] -> result fp32 [n_instances, n_group, G, D]."""
        return _binding.solve_batched(self.n_group, self.group_size, self.dup_per_rank, self.n_combined_experts,
                                      self.n_local_experts, self.step_rule, self.n_steps, workloads, r2o, phy2log,
                                      avail_num, want_global)

    # -- csrc/plugin.cpp:580-600 -------------------------------------------------
    def count_idx(self, idx: torch.Tensor, n_sms: int, block_dim: int = 256, *,
                  out: torch.Tensor | None = None) -> tuple[torch.Tensor, torch.Tensor]:
        """out: optional int32 [n_sms, n_experts] table to fill instead of a new one (no counterpart in the
        reference, which allocates on every call)."""
        _require(block_dim == 256, "slices are aligned to 256 indices")
        return _binding.count_idx(self.n_group, self.group_size, self.dup_per_rank, self.n_combined_experts,
                                  self.n_local_experts, self.step_rule, self.n_steps, idx, n_sms, out)

    def count_totals(self, idx: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
        """This GPU's tokens per logical expert (what count_idx returns first) without the table per slice, in
        one kernel launch; short batches only (UnsupportedShape beyond 131072 indices or 1024 experts).  No
        counterpart in the reference."""
        _require(idx.dtype == torch.int64 and idx.is_cuda and idx.is_contiguous(), "idx is a contiguous int64 GPU tensor")
        if out is None:
            out = torch.empty(self.n_experts, dtype=torch.int32, device=idx.device)
        else:
            _require(out.dtype == torch.int32 and out.is_cuda and out.is_contiguous() and out.numel() == self.n_experts,
                     "out: int32 [n_experts], contiguous, on the GPU")
        _check(self.lib.lplb_count_totals(idx.data_ptr(), idx.numel(), self.n_experts, out.data_ptr(), _stream(idx)))
        return out

    def count_totals_add(self, idx: torch.Tensor, totals: torch.Tensor, clear: torch.Tensor | None = None) -> torch.Tensor:
        """Adds this GPU's tokens per logical expert to ``totals`` (which the caller has zeroed), one kernel launch
        of a few workgroups (short batches only: UnsupportedShape beyond 131072 indices); the same launch sets
        ``clear`` to zero, so a caller that swaps two vectors from call to call never zeroes one itself.  No
        counterpart in the reference."""
        _require(idx.dtype == torch.int64 and idx.is_cuda and idx.is_contiguous(), "idx is a contiguous int64 GPU tensor")
        for name, t in (("totals", totals), ("clear", clear)):
            _require(t is None or (t.dtype == torch.int32 and t.is_cuda and t.is_contiguous() and
                                   t.numel() == self.n_experts and t.device == idx.device),
                     f"{name}: int32 [n_experts], contiguous, on idx's GPU")
        _check(self.lib.lplb_count_totals_add(idx.data_ptr(), idx.numel(), self.n_experts, totals.data_ptr(),
                                              None if clear is None else clear.data_ptr(), _stream(idx)))
        return totals

    # -- csrc/plugin.cpp:602-660 -------------------------------------------------
    def map_idx(self, mapping_idx: torch.Tensor, o_weight: torch.Tensor, local_workload_split_by_sm: torch.Tensor,
                o2r: torch.Tensor, phy2log: torch.Tensor, n_sms: int, block_dim: int = 256,
                physical_counts: torch.Tensor | None = None, prepared: torch.Tensor | None = None) -> torch.Tensor:
        """prepared: optional table from prepare_mapping(o2r, phy2log) (no counterpart in the reference,
        which rebuilds it in every block); the result is the same with and without it."""
        _require(block_dim == 256, "slices are aligned to 256 indices")
        return _binding.map_idx(self.n_group, self.group_size, self.dup_per_rank, self.n_combined_experts,
                                self.n_local_experts, self.step_rule, self.n_steps, mapping_idx, o_weight,
                                local_workload_split_by_sm, o2r, phy2log, n_sms, physical_counts, prepared)

    def prepared_mapping_bytes(self) -> int:
        n = self.lib.lplb_prepared_mapping_bytes(self.n_group, self.group_size, self.dup_per_rank,
                                                 self.n_combined_experts, self.n_local_experts)
        _require(n > 0, "a shape the prepared table can describe")
        return n

    def prepare_mapping(self, o2r: torch.Tensor, phy2log: torch.Tensor) -> torch.Tensor:
        """The mapping-only part of the redirect's tables as an opaque int32 tensor for map_idx(prepared=...);
        valid until phy2log or o2r change."""
        _require(o2r.dtype == torch.int32 and o2r.is_cuda and o2r.is_contiguous()
                 and tuple(o2r.shape) == (self.group_size, self.dup_per_rank), "o2r is a contiguous int32 [G, D] GPU tensor")
        _require(phy2log.dtype == torch.int32 and phy2log.is_cuda and phy2log.is_contiguous() and phy2log.dim() == 1
                 and phy2log.size(0) == self.group_size * self.n_group * self.n_local_experts,
                 "phy2log is a contiguous int32 [n_group * group_size * n_local_experts] GPU tensor")
        n_bytes = self.prepared_mapping_bytes()
        table = torch.empty((n_bytes + 3) // 4, dtype=torch.int32, device=phy2log.device)
        _check(self.lib.lplb_prepare_mapping(o2r.data_ptr(), phy2log.data_ptr(), self.n_group, self.group_size,
                                             self.dup_per_rank, self.n_combined_experts, self.n_local_experts,
                                             table.data_ptr(), n_bytes, _stream(phy2log)))
        return table

    # -- lplb/planner.py:245-266 in one library call -----------------------------
    def plan(self, idx: torch.Tensor, r2o: torch.Tensor, o2r: torch.Tensor, phy2log: torch.Tensor,
             avail_num: torch.Tensor, n_sms: int, global_counts: torch.Tensor | None = None,
             workspace: dict | None = None,
             physical_counts: torch.Tensor | None = None) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
        """Histogram, LP solve and redirect of one batch.  Returns (physical indices, o_weight,
        workspace table whose last row holds this GPU's tokens per logical expert).  ``global_counts`` (int32 [n_logical]) replaces this GPU's own histogram
        as the LP's workload.  ``workspace`` may carry preallocated ``out``, ``by_sm``, ``o_weight``
        and ``global_workload`` tensors to reuse; the last three are stored into it for the next call."""
        return _binding.plan(self.n_group, self.group_size, self.dup_per_rank, self.n_combined_experts,
                             self.n_local_experts, self.step_rule, self.n_steps, idx, r2o, o2r, phy2log, avail_num,
                             n_sms, global_counts, workspace, physical_counts)
