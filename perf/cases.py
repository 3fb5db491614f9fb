"""The planner's work, as timed cases.

A case is one deployment (replica topology, EP size, experts, replicas per rank), one batch of routing
decisions (tokens x topk, popularity, masked entries) and one of the paths a user of the package takes:

  run        Planner.run: histogram, LP and redirect of this GPU's batch in one call
  plan       CompiledSolver.plan with the counts of all ranks supplied, as behind an all-reduce of the
             caller's own
  steps      count_workload, solve_probs and weighted_select_target one after the other, for callers that
             want the histogram and the shares themselves
  batched    CompiledSolver.solve_batched: many LPs over one mapping (what-if searches, many layers at once)
  reshuffle  Planner.update_redundancy_mapping: which experts get the replicas, from the load history

Deployments and distributions are those of lplb_amd/synth.py and of the solver tests: Zipf popularity in a
random order, a lognormal factor per batch, topk different experts per token.
"""
from __future__ import annotations

import math

import torch

from lplb_amd import Planner, topology

TOPOLOGIES = {
    "cube8": topology.CUBE_8P2E,
    "ring8": topology.RING_8P,
    "hypercube16": topology.HYPERCUBE_16P2E,
    "torus32": topology.torus_2d(8, 4),
}
# (topology, EP ranks, logical experts, replicas per rank)
DEPLOYMENTS = [
    ("cube8", 8, 32, 2),
    ("cube8", 8, 256, 2),
    ("cube8", 8, 256, 4),
    ("cube8", 32, 256, 2),
    ("cube8", 32, 256, 4),
    ("cube8", 64, 256, 2),
    ("ring8", 32, 256, 1),
    ("hypercube16", 16, 256, 2),
    ("torus32", 32, 256, 2),
]
MAX_TOKENS = 1 << 20
MAX_INDICES = 8 * MAX_TOKENS
MAX_COUNTED = 4_000_000  # indices up to which the tokens per physical expert are asked for
MAX_LPS = 16384          # of 8 ranks; larger groups cost about the square of their size
JITTER = 0.3             # sigma of the lognormal factor per batch
POOL_ROWS = 32768        # token rows drawn one by one; longer batches draw their rows from these
GPUS_PER_NODE = 8


def _case(name, path, deployment, tokens=0, topk=8, zipf=1.0, hot=0, masked=0.0, n_sms=256, counts=False, lps=0):
    topo, ep_size, n_logical, redundants = deployment
    case = {"path": path, "topology": topo, "ep_size": ep_size, "n_logical": n_logical, "redundants": redundants,
            "zipf": zipf, "hot": hot}
    if path in ("run", "plan", "steps"):
        case.update(tokens=tokens, topk=topk, masked=masked, n_sms=n_sms)
    if path in ("run", "plan"):
        case.update(counts=counts)
    if path == "batched":
        case.update(lps=lps)
    return dict(case, name=name) if name else case


def listed():
    ep8 = ("cube8", 8, 256, 2)
    return [
        # decoding with a handful of sequences: nothing but latency
        _case("run_decode_7x8", "run", ep8, 7),
        # a decode step of a loaded server, some rows padding
        _case("run_decode_128x8", "run", ep8, 128, masked=0.05),
        # prefill of one rank at the shape the benchmark is quoted on
        _case("run_ep8_8192x8", "run", ep8, 8192),
        # the same with the counts of all ranks at hand, and the tokens per physical expert for the dispatch
        _case("plan_ep8_8192x8", "plan", ep8, 8192, counts=True),
        # ragged: four EP groups, two expert sets per replica slot, fewer workgroups, padding in the batch
        _case("run_ep32_groups_5003x6", "run", ("cube8", 32, 256, 4), 5003, topk=6, masked=0.05, n_sms=64, counts=True),
        # larger groups and their heavier LPs
        _case("plan_ep16_4096x8", "plan", ("hypercube16", 16, 256, 2), 4096, zipf=1.1),
        _case("run_ep32_torus_16384x8", "run", ("torus32", 32, 256, 2), 16384, zipf=1.5, hot=3),
        # the three steps called separately on a long prefill
        _case("steps_ep8_32768x8", "steps", ep8, 32768),
        # the throughput sweep's batch, and one four times as long
        _case("run_sweep_262144x8", "run", ep8, 262144),
        _case("run_longest_1048576x8", "run", ep8, MAX_TOKENS),
        # the throughput sweep's LPs
        _case("batched_2048", "batched", ep8, lps=2048),
        # between batches, every few minutes: new load history, new replicas
        _case("reshuffle_ep32", "reshuffle", ("cube8", 32, 256, 2)),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    path = rng.choices(["run", "plan", "steps", "batched", "reshuffle"], [45, 20, 15, 12, 8])[0]
    deployment = rng.choice(DEPLOYMENTS)
    zipf = round(rng.uniform(0.8, 1.3), 3)
    if path == "reshuffle":
        return _case(None, path, deployment, zipf=zipf)
    if path == "batched":
        group = TOPOLOGIES[deployment[0]].shape[0]
        most = MAX_LPS * 64 // group ** 2 // (deployment[1] // group)
        return _case(None, path, deployment, zipf=zipf, lps=_log_uniform(rng, 1, most))
    tokens, topk = _log_uniform(rng, 1, MAX_TOKENS), rng.choice([1, 2, 4, 6, 8, 8])
    return _case(None, path, deployment, tokens, topk=topk, zipf=zipf, masked=rng.choice([0.0, 0.0, 0.05]),
                 n_sms=rng.choice([256, 256, 256, 64]),
                 counts=rng.random() < 0.3 and tokens * topk <= MAX_COUNTED)


def _popularity(case, generator):
    """Zipf over a random order of the experts, a few of them raised to ten times the mean."""
    n, dev = case["n_logical"], generator.device
    rank = torch.randperm(n, generator=generator, device=dev).double() + 1
    p = rank.pow(-case["zipf"])
    p /= p.sum()
    if case["hot"]:
        p[torch.randperm(n, generator=generator, device=dev)[:case["hot"]]] = 10.0 / n
        p /= p.sum()
    return p


def _batch_popularity(p, generator, lead=()):
    q = p * torch.exp(JITTER * torch.randn(*lead, p.numel(), generator=generator, device=p.device, dtype=p.dtype))
    return q / q.sum(-1, keepdim=True)


def _routing(case, q, generator):
    """int64 [tokens, topk]: topk different experts per token, drawn by popularity (Gumbel top-k)."""
    dev = generator.device
    rows = min(case["tokens"], POOL_ROWS)
    noise = torch.rand(rows, q.numel(), generator=generator, device=dev).clamp_(1e-20, 1 - 1e-7)
    idx = (torch.log(q).float() - torch.log(-torch.log(noise))).topk(case["topk"], dim=1).indices
    if case["tokens"] > rows:
        idx = idx[torch.randint(rows, (case["tokens"],), generator=generator, device=dev)]
    if case["masked"]:
        idx.masked_fill_(torch.rand(idx.shape, generator=generator, device=dev) < case["masked"], -1)
    return idx.contiguous()


def _counts(q, total, generator):
    """int32 counts of `total` tokens spread by q, with the scatter of independent draws."""
    noise = torch.randn(q.shape, generator=generator, device=q.device, dtype=q.dtype)
    return (q * total + (q * (1 - q) * total).sqrt() * noise).round().clamp(min=0).to(torch.int32)


def prepare(case, seed):
    dev = torch.device("cuda")
    generator = torch.Generator(device=dev).manual_seed(seed)
    r2o = torch.from_numpy(TOPOLOGIES[case["topology"]])
    ep_size, n_logical = case["ep_size"], case["n_logical"]
    planner = Planner(r2o, n_logical + case["redundants"] * ep_size, n_logical, ep_size, device=dev,
                      gpus_per_node=GPUS_PER_NODE)
    p = _popularity(case, generator)
    state = {"path": case["path"], "planner": planner}
    history = (p * 2 ** 24).round().to(torch.int64)
    if case["path"] == "reshuffle":
        state["history"] = (_batch_popularity(p, generator) * 2 ** 24).round().to(torch.int64)
        return state
    planner.update_redundancy_mapping(history)
    state["avail"] = torch.zeros(1, dtype=torch.int32, device=dev)
    if case["path"] == "batched":
        q = _batch_popularity(p, generator, (case["lps"],))
        counts = _counts(q, ep_size * 65536, generator)
        state["workloads"] = counts.view(case["lps"], planner.n_group, planner.group_size, -1)
        return state
    q = _batch_popularity(p, generator)
    state["idx"] = _routing(case, q, generator)
    state["n_sms"] = case["n_sms"]
    if case["path"] == "plan":
        state["global_counts"] = _counts(q, ep_size * case["tokens"] * case["topk"], generator)
        state["workspace"] = {}
    if case.get("counts"):
        state["physical_counts"] = torch.empty(planner.n_routed_experts, dtype=torch.int32, device=dev)
    return state


def run(state):
    planner, path = state["planner"], state["path"]
    if path == "reshuffle":
        return planner.update_redundancy_mapping(state["history"])
    avail = state["avail"]
    if path == "batched":
        shares = planner.solver.solve_batched(state["workloads"], planner.r2o, planner.phy2log, avail)
        return {"shares": shares, "feasible": avail}
    idx, n_sms = state["idx"], state["n_sms"]
    if path == "steps":
        counts, by_slice = planner.count_workload(idx, n_sms)
        shares, workload = planner.solve_probs(counts, avail)
        out = planner.weighted_select_target(idx, shares, by_slice, n_sms)
        return {"indices": out, "by_slice": by_slice, "shares": shares, "workload": workload, "feasible": avail}
    physical = state.get("physical_counts")
    if path == "plan":
        out, shares, by_slice = planner.solver.plan(idx, planner.r2o, planner.o2r, planner.phy2log, avail, n_sms,
                                                    global_counts=state["global_counts"], workspace=state["workspace"],
                                                    physical_counts=physical)
        return {"indices": out, "shares": shares, "counts": by_slice[-1], "feasible": avail, "physical": physical}
    out = planner.run(idx, avail, n_sms, physical_counts=physical)
    return {"indices": out, "feasible": avail, "physical": physical}


def work(case):
    """Indices in and out once (int64), the tables and counts of the path once; per LP five steps, each the
    factorisation of the ranks' system, its two triangular solves and a few operations per replica edge."""
    r2o = TOPOLOGIES[case["topology"]]
    group, slots = r2o.shape
    ep_size, n_logical = case["ep_size"], case["n_logical"]
    n_groups, n_physical = ep_size // group, n_logical + case["redundants"] * ep_size
    edges = group * slots
    if case["path"] == "reshuffle":
        return {"bytes": 8 * n_logical + 4 * (n_physical + 3 * n_logical), "flops": 0}
    tables = 4 * (n_physical + 2 * r2o.size)
    lps = n_groups * case.get("lps", 1)
    lp_flops = 5 * (group ** 3 / 3 + 2 * group ** 2 + 40 * edges)
    if case["path"] == "batched":
        return {"bytes": lps * 4 * (n_logical // n_groups + edges) + tables, "flops": lps * lp_flops}
    n = case["tokens"] * case["topk"]
    moved = 16 * n + tables + 4 * n_groups * edges
    if case["path"] == "steps":
        moved += 4 * n_logical * (case["n_sms"] + 1)
    if case["path"] == "plan":
        moved += 8 * n_logical
    if case.get("counts"):
        moved += 4 * n_physical
    return {"bytes": moved, "flops": lps * lp_flops}


def tolerance(case):
    """Counts, slots and mappings are whole numbers.  The shares are the result of five fp32 interior-point steps;
    a share that differs in its last digits can move the one token of its expert that sits on the rounding edge."""
    if case["path"] == "reshuffle":
        return "exact"
    return {"rel": 1e-4, "max": 1e-3, "differ": 1e-3}
