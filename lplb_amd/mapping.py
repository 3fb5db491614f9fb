"""Physical <-> logical expert layout of the planner (host side; the work is done by csrc/mapping.hip).

Per EP rank the physical slots are laid out as

    [ C*D originals that have a replica (slot = c*D + d) | n_fixed other originals | C*D replicas ]

where replica slot ``(c, d)`` of group-rank ``i`` copies original slot ``(c, d)`` of
group-rank ``r2o[i, d]``.  This is the layout the solver and redirect kernels index
(reference: lplb/planner.py:115-182).
"""
from __future__ import annotations

import numpy as np

from . import _native


def build_redundancy_mapping(r2o: np.ndarray, ep_size: int, n_logical: int, n_physical: int,
                             workload: np.ndarray | None = None, n_nodes: int = 1, out: np.ndarray | None = None):
    """Returns (phy2log int32 [n_physical], log2phy int32 [n_logical, 2], logcnt int32 [n_logical]).

    workload: optional per-logical-expert history.  When given, experts are first
    spread over ranks with EPLB (reorder only, no replication) and each rank's
    experts are sorted heaviest first, so the heaviest C*D of every rank get the
    replicas (lplb/planner.py:127-147).  Equal histories keep index order.
    out: optional int32 [n_physical + 3 * n_logical] buffer, contiguous, that the three arrays become parts of.
    Raises AssertionError unless every logical expert ends up with at most one
    replica and at least one expert has one (lplb/planner.py:173).
    """
    r2o = np.ascontiguousarray(r2o, dtype=np.int32)
    G, D = r2o.shape
    weight = history = None
    if workload is not None:
        workload = np.asarray(workload).reshape(-1)
        assert workload.size == n_logical
        weight = np.ascontiguousarray(workload, dtype=np.float32)
        history = np.ascontiguousarray(workload, dtype=np.float64)
    if out is None:
        out = np.empty(n_physical + 3 * n_logical, dtype=np.int32)
    assert out.shape == (n_physical + 3 * n_logical,)
    at = out.ctypes.data
    _native.check_host(_native.load().lplb_build_mapping(
        None if weight is None else weight.ctypes.data, None if history is None else history.ctypes.data, r2o.ctypes.data,
        G, D, ep_size, n_logical, n_physical, n_nodes, at, at + 4 * n_physical, at + 4 * (n_physical + 2 * n_logical)))
    return (out[:n_physical], out[n_physical:n_physical + 2 * n_logical].reshape(n_logical, 2),
            out[n_physical + 2 * n_logical:])
