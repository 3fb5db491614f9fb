"""numpy restatement of the expert placement (packing, replication, hierarchical policy, the planner's layout of
physical experts); test infrastructure only.  The package's own is native (lplb_amd/csrc/mapping.hip)."""
from __future__ import annotations

import numpy as np


def balanced_packing(weight: np.ndarray, num_packs: int) -> tuple[np.ndarray, np.ndarray]:
    """Pack n weighted items into ``num_packs`` packs of exactly n/num_packs items,
    heaviest first, each into the lightest pack that still has room
    (lplb/eplb.py:6-46).

    weight: [X, n].  Returns (pack_index [X, n], rank_in_pack [X, n]), int64.
    """
    weight = np.asarray(weight, dtype=np.float32)
    n_layers, n_items = weight.shape
    assert n_items % num_packs == 0
    cap = n_items // num_packs
    if cap == 1:
        pack_index = np.broadcast_to(np.arange(n_items, dtype=np.int64), weight.shape).copy()
        return pack_index, np.zeros_like(pack_index)

    order = np.argsort(-weight, axis=-1, kind="stable")
    pack_index = np.full(weight.shape, -1, dtype=np.int64)
    rank_in_pack = np.full(weight.shape, -1, dtype=np.int64)
    for layer in range(n_layers):
        load = np.zeros(num_packs, dtype=np.float32)
        fill = np.zeros(num_packs, dtype=np.int64)
        for item in order[layer]:
            masked = np.where(fill < cap, load, np.float32(np.inf))
            pack = int(np.argmin(masked))
            pack_index[layer, item] = pack
            rank_in_pack[layer, item] = fill[pack]
            load[pack] += weight[layer, item]
            fill[pack] += 1
    return pack_index, rank_in_pack


def replicate_experts(weight: np.ndarray, num_phy: int) -> tuple[np.ndarray, np.ndarray, np.ndarray]:
    """Add ``num_phy - num_log`` replicas, each time to the expert whose
    per-replica load is currently largest (lplb/eplb.py:49-77).

    Returns (phy2log [X, num_phy], replica rank [X, num_phy], logcnt [X, num_log]).
    """
    weight = np.asarray(weight, dtype=np.float32)
    n, num_log = weight.shape
    assert num_phy >= num_log
    phy2log = np.tile(np.arange(num_phy, dtype=np.int64), (n, 1))
    rank = np.zeros((n, num_phy), dtype=np.int64)
    logcnt = np.ones((n, num_log), dtype=np.int64)
    rows = np.arange(n)
    for slot in range(num_log, num_phy):
        pick = np.argmax(weight / logcnt.astype(np.float32), axis=-1)
        phy2log[:, slot] = pick
        rank[:, slot] = logcnt[rows, pick]
        logcnt[rows, pick] += 1
    return phy2log, rank, logcnt


def _inverse_perm(perm: np.ndarray) -> np.ndarray:
    inv = np.empty_like(perm)
    np.put_along_axis(inv, perm, np.broadcast_to(np.arange(perm.shape[1]), perm.shape), axis=1)
    return inv


def rebalance_experts_hierarchical(weight: np.ndarray, num_physical_experts: int, num_groups: int,
                                   num_nodes: int, num_gpus: int):
    """Groups -> nodes, replicate inside nodes, physical experts -> GPUs
    (lplb/eplb.py:80-148).  Returns (phy2log, phyrank, logcnt), each [layers, ...]."""
    weight = np.asarray(weight, dtype=np.float32)
    n_layers, n_log = weight.shape
    assert n_log % num_groups == 0
    group_size = n_log // num_groups
    assert num_groups % num_nodes == 0
    groups_per_node = num_groups // num_nodes
    assert num_gpus % num_nodes == 0
    assert num_physical_experts % num_gpus == 0
    phy_per_gpu = num_physical_experts // num_gpus

    # 1. whole expert groups onto nodes
    tokens_per_group = weight.reshape(n_layers, num_groups, group_size).sum(-1, dtype=np.float32)
    g_pack, g_rank = balanced_packing(tokens_per_group, num_nodes)
    log2mlog = (((g_pack * groups_per_node + g_rank) * group_size)[..., None]
                + np.arange(group_size, dtype=np.int64)).reshape(n_layers, -1)
    mlog2log = _inverse_perm(log2mlog)

    # 2. replicas inside each node
    log_per_node = n_log // num_nodes
    tokens_per_mlog = np.take_along_axis(weight, mlog2log, axis=-1).reshape(-1, log_per_node)
    phy2mlog, phyrank, mlogcnt = replicate_experts(tokens_per_mlog, num_physical_experts // num_nodes)

    # 3. physical experts onto the node's GPUs
    tokens_per_phy = np.take_along_axis(tokens_per_mlog / mlogcnt.astype(np.float32), phy2mlog, axis=-1)
    p_pack, p_rank = balanced_packing(tokens_per_phy, num_gpus // num_nodes)
    phy2pphy = p_pack * phy_per_gpu + p_rank
    pphy2phy = _inverse_perm(phy2pphy)

    pphy2mlog = np.take_along_axis(phy2mlog, pphy2phy, axis=-1)
    pphy2mlog = (pphy2mlog.reshape(n_layers, num_nodes, -1)
                 + (np.arange(num_nodes, dtype=np.int64) * log_per_node)[None, :, None]
                 ).reshape(n_layers, -1)
    pphy2log = np.take_along_axis(mlog2log, pphy2mlog, axis=-1)
    pphyrank = np.take_along_axis(phyrank, pphy2phy, axis=-1).reshape(n_layers, -1)
    logcnt = np.take_along_axis(mlogcnt.reshape(n_layers, -1), log2mlog, axis=-1)
    return pphy2log, pphyrank, logcnt


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


def build_redundancy_mapping(r2o: np.ndarray, ep_size: int, n_logical: int, n_physical: int,
                             workload: np.ndarray | None = None, n_nodes: int = 1):
    """Returns (phy2log int32 [n_physical], log2phy int32 [n_logical, 2], logcnt int32 [n_logical]).

    workload: optional per-logical-expert history.  When given, experts are first
    spread over ranks with EPLB (reorder only, no replication) and each rank's
    experts are sorted heaviest first, so the heaviest C*D of every rank get the
    replicas (lplb/planner.py:127-147).  Equal histories keep index order.
    Raises AssertionError unless every logical expert ends up with at most one
    replica and at least one expert has one (lplb/planner.py:173).
    """
    r2o = np.asarray(r2o, dtype=np.int64)
    G, D = r2o.shape
    n_group = ep_size // G
    L = n_logical // ep_size
    P = n_physical // ep_size
    C = (P - L) // D

    if workload is None:
        nored = np.arange(n_logical, dtype=np.int64)
    else:
        workload = np.asarray(workload).reshape(-1)
        assert workload.size == n_logical
        nored = rebalance_experts(workload[None].astype(np.float32), n_logical, n_group,
                                  n_nodes, ep_size)[0][0]
    nored = nored.reshape(n_group, G, L)
    if workload is not None:
        order = np.argsort(-workload[nored].astype(np.float64), axis=-1, kind="stable")
        nored = np.take_along_axis(nored, order, axis=-1)

    tored = nored[:, :, :C * D].reshape(n_group, G, C, D)
    # replica (c, d) on rank i <- original (c, d) of rank r2o[i, d]
    dup = tored[:, r2o, :, np.arange(D)[None, :]]          # [G, D, n_group, C]
    dup = dup.transpose(2, 0, 3, 1)                        # [n_group, G, C, D]
    phy2log = np.concatenate([nored, dup.reshape(n_group, G, C * D)], axis=-1).reshape(-1)
    assert phy2log.shape[0] == n_physical, (phy2log.shape, n_physical)

    # log2phy lists originals before replicas: walk physical ids by (local slot, rank).
    by_slot = np.arange(n_physical).reshape(ep_size, P).T.reshape(-1)
    logs = phy2log[by_slot]
    order = np.argsort(logs, kind="stable")
    logcnt = np.bincount(logs, minlength=n_logical)
    max_cnt = int(logcnt.max())
    assert max_cnt == 2, f"every logical expert may have at most one replica (got {max_cnt} copies)"
    starts = np.cumsum(logcnt) - logcnt
    sorted_logs = logs[order]
    pos = np.arange(order.size) - starts[sorted_logs]
    log2phy = np.full((n_logical, max_cnt), -1, dtype=np.int32)
    log2phy[sorted_logs, pos] = by_slot[order]
    return phy2log.astype(np.int32), log2phy, logcnt.astype(np.int32)
