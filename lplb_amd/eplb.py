"""Static expert placement (EPLB) used by ``Planner.update_redundancy_mapping``.

It runs once per re-shuffle, never per batch; the work is done by the library on the host
(csrc/mapping.hip).  Behaviour follows the reference's embedded EPLB (lplb/eplb.py:6-190):
greedy longest-processing-time packing into equally sized packs, optional replication of
the currently heaviest expert, and the hierarchical groups -> nodes -> GPUs policy.  All
weights are handled in float32 like there.

Tie-breaking: items of equal weight are taken in index order (stable sort) and
a tie between packs goes to the lowest pack index.  The reference leaves the
first to an unstable sort, so results can differ from it only when weights tie.
"""
from __future__ import annotations

import numpy as np

from . import _native


def balanced_packing(weight: np.ndarray, num_packs: int) -> tuple[np.ndarray, np.ndarray]:
    """Pack n weighted items into ``num_packs`` packs of exactly n/num_packs items,
    heaviest first, each into the lightest pack that still has room
    (lplb/eplb.py:6-46).

    weight: [X, n].  Returns (pack_index [X, n], rank_in_pack [X, n]), int64.
    """
    weight = np.ascontiguousarray(weight, dtype=np.float32)
    n_layers, n_items = weight.shape
    assert n_items % num_packs == 0
    pack_index = np.empty(weight.shape, dtype=np.int64)
    rank_in_pack = np.empty(weight.shape, dtype=np.int64)
    _native.check_host(_native.load().lplb_balanced_packing(weight.ctypes.data, n_layers, n_items, num_packs,
                                                            pack_index.ctypes.data, rank_in_pack.ctypes.data))
    return pack_index, rank_in_pack


def replicate_experts(weight: np.ndarray, num_phy: int) -> tuple[np.ndarray, np.ndarray, np.ndarray]:
    """Add ``num_phy - num_log`` replicas, each time to the expert whose
    per-replica load is currently largest (lplb/eplb.py:49-77).

    Returns (phy2log [X, num_phy], replica rank [X, num_phy], logcnt [X, num_log]).
    """
    weight = np.ascontiguousarray(weight, dtype=np.float32)
    n, num_log = weight.shape
    assert num_phy >= num_log
    phy2log = np.empty((n, num_phy), dtype=np.int64)
    rank = np.empty((n, num_phy), dtype=np.int64)
    logcnt = np.empty((n, num_log), dtype=np.int64)
    _native.check_host(_native.load().lplb_replicate_experts(weight.ctypes.data, n, num_log, num_phy, phy2log.ctypes.data,
                                                             rank.ctypes.data, logcnt.ctypes.data))
    return phy2log, rank, logcnt


def rebalance_experts_hierarchical(weight: np.ndarray, num_physical_experts: int, num_groups: int,
                                   num_nodes: int, num_gpus: int):
    """Groups -> nodes, replicate inside nodes, physical experts -> GPUs
    (lplb/eplb.py:80-148).  Returns (phy2log, phyrank, logcnt), each [layers, ...]."""
    weight = np.ascontiguousarray(weight, dtype=np.float32)
    n_layers, n_log = weight.shape
    phy2log = np.empty((n_layers, num_physical_experts), dtype=np.int64)
    phyrank = np.empty((n_layers, num_physical_experts), dtype=np.int64)
    logcnt = np.empty((n_layers, n_log), dtype=np.int64)
    _native.check_host(_native.load().lplb_rebalance_experts(weight.ctypes.data, n_layers, n_log, num_physical_experts,
                                                             num_groups, num_nodes, num_gpus, phy2log.ctypes.data,
                                                             phyrank.ctypes.data, logcnt.ctypes.data))
    return phy2log, phyrank, logcnt


def rebalance_experts(weight: np.ndarray, num_replicas: int, num_groups: int, num_nodes: int,
                      num_gpus: int):
    """Entry point (lplb/eplb.py:151-190).  weight: [layers, num_logical].
    Returns (phy2log [layers, num_replicas], log2phy [layers, num_logical, X],
    logcnt [layers, num_logical]), int64."""
    weight = np.asarray(weight, dtype=np.float32)
    n_layers, n_log = weight.shape
    if num_groups % num_nodes == 0:
        phy2log, phyrank, logcnt = rebalance_experts_hierarchical(
            weight, num_replicas, num_groups, num_nodes, num_gpus)
    else:
        phy2log, phyrank, logcnt = rebalance_experts_hierarchical(
            weight, num_replicas, 1, 1, num_gpus)
    max_cnt = int(logcnt.max())
    log2phy = np.full((n_layers, n_log * max_cnt), -1, dtype=np.int64)
    np.put_along_axis(log2phy, phy2log * max_cnt + phyrank,
                      np.broadcast_to(np.arange(num_replicas, dtype=np.int64), phy2log.shape), axis=-1)
    return phy2log, log2phy.reshape(n_layers, n_log, max_cnt), logcnt
