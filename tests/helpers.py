"""Shared builders for the parity tests: reference-test-style workloads
(tests/test_solve.py:40-49 of the reference draws them from the CUDA generator,
which cannot be reproduced, so the same distributions are drawn from numpy)."""
from __future__ import annotations

from dataclasses import dataclass

import numpy as np

from lplb_amd import topology
from lplb_amd.mapping import build_redundancy_mapping

# (name, r2o, n_logical, ep_size, redundants per rank, reorder, balance tolerance):
# the reference's solver test matrix, tests/test_solve.py:16-21.
REFERENCE_SOLVE_CASES = [
    ("cube8_ep32", topology.CUBE_8P2E, 256, 32, 2, True, 1.07),
    ("cube8_ep32_c2", topology.CUBE_8P2E, 256, 32, 4, False, 1.07),
    ("cube8_ep64", topology.CUBE_8P2E, 256, 64, 2, True, 1.1),
    ("ring8_ep32", topology.RING_8P, 256, 32, 1, True, 1.07),
    ("hypercube16", topology.HYPERCUBE_16P2E, 256, 16, 2, True, 1.03),
    ("torus8x4", topology.torus_2d(8, 4), 256, 32, 2, False, 1.01),
]
# The balance tolerances above hold for the reference's CUDA-generator draw.  For a
# numpy draw they hold only when the LP optimum itself admits them (a ring with one
# replica cannot flatten every draw), so each case uses a seed whose HiGHS optimum
# is inside the tolerance.
CASE_SEED = {"cube8_ep32": 42, "cube8_ep32_c2": 42, "cube8_ep64": 42, "ring8_ep32": 3,
             "hypercube16": 42, "torus8x4": 42}


def shifted_ring(g, shifts):
    return np.array([[(i + s) % g for s in shifts] for i in range(g)], np.int32)


# Batches of LPs around the places where the number of LPs to a wave changes (on 1024 SIMDs):
# (name, r2o, ep_size, n_logical, LP instances, four to a wave?)
BATCHED_LPS = [
    ("cube8x2", topology.CUBE_8P2E, 8, 256, 1541, False),
    ("ring8x1", shifted_ring(8, [1]), 8, 128, 1538, False),
    ("ring6x2_padded", shifted_ring(6, [1, 2]), 6, 60, 1537, False),  # rounded up to the 8 x 2 instantiation
    ("ring16x1", shifted_ring(16, [1]), 32, 256, 771, True),         # two groups per instance
    # exact and padded instantiations packed from more than three LPs per SIMD on, last wave part full
    ("cube8x2_packed", topology.CUBE_8P2E, 8, 256, 3077, True),
    ("ring8x1_packed", shifted_ring(8, [1]), 8, 128, 3074, True),
    ("ring6x2_packed", shifted_ring(6, [1, 2]), 6, 60, 3073, True),
    ("ring8x1_last_lone", shifted_ring(8, [1]), 8, 128, 3072, False),
    # beyond 8 ranks from more than one
    ("ring16x1_packed", shifted_ring(16, [1]), 16, 128, 1025, True),
    ("ring13x1_packed", shifted_ring(13, [1]), 13, 104, 1026, True),
    ("ring16x1_last_lone", shifted_ring(16, [1]), 16, 128, 1024, False),
    ("cube8x2_three_per_simd", topology.CUBE_8P2E, 8, 256, 3072, False),
    ("ring6x2_four_per_simd", shifted_ring(6, [1, 2]), 6, 60, 4096, True),
    ("cube8x2_five_per_simd", topology.CUBE_8P2E, 8, 256, 4097, False),
    ("ring8x1_six_per_simd", shifted_ring(8, [1]), 8, 128, 5123, True),
    # as many experts as make the sixth per SIMD, or the fourth, too much for packing; two groups per instance packed
    ("cube8x2_six_per_simd", topology.CUBE_8P2E, 8, 256, 5121, False),
    ("cube8x2_seven_per_simd", topology.CUBE_8P2E, 8, 256, 6147, True),
    ("cube8x2_512_experts_four_per_simd", topology.CUBE_8P2E, 8, 512, 3077, False),
    ("cube8x2_two_groups", topology.CUBE_8P2E, 16, 256, 1539, True),
]


RING_64 = shifted_ring(64, [1])
# Deployments around what is placed on the GPU: (r2o, ep_size, n_logical, replicas per rank, covered?)
PLACEMENTS = {
    "ring8_8": (topology.RING_8P, 8, 8, 1, True), "cube8_128": (topology.CUBE_8P2E, 8, 128, 2, True),
    "cube8_136": (topology.CUBE_8P2E, 8, 136, 2, False), "cube8x2_256": (topology.CUBE_8P2E, 16, 256, 4, True),
    "cube8x8_512": (topology.CUBE_8P2E, 64, 512, 2, True), "ring8x4_256": (topology.RING_8P, 32, 256, 1, True),
    "hyper16_96": (topology.HYPERCUBE_16P2E, 16, 96, 2, True), "torus32_128": (topology.torus_2d(8, 4), 32, 128, 2, True),
    "torus32x2_256": (topology.torus_2d(8, 4), 64, 256, 2, False), "ring64_128": (RING_64, 64, 128, 1, True),
    "ring64_64": (RING_64, 64, 64, 1, True),
}


@dataclass
class Shape:
    r2o: np.ndarray
    ep_size: int
    n_logical: int
    n_physical: int

    @property
    def G(self): return self.r2o.shape[0]
    @property
    def D(self): return self.r2o.shape[1]
    @property
    def n_group(self): return self.ep_size // self.G
    @property
    def L(self): return self.n_logical // self.ep_size
    @property
    def P(self): return self.n_physical // self.ep_size
    @property
    def C(self): return (self.P - self.L) // self.D
    @property
    def n_fixed(self): return self.L - self.C * self.D
    @property
    def o2r(self): return np.argsort(self.r2o, axis=0, kind="stable").astype(np.int32)


def reference_style_case(r2o, n_logical, ep_size, red, reorder, seed=42, gpus_per_node=8):
    """History ~ N(1, 0.15) * 2^20 and batch workload ~ N(1, 0.3) * 2^12, clamped at 0."""
    rng = np.random.default_rng(seed)
    shape = Shape(np.asarray(r2o, np.int32), ep_size, n_logical, n_logical + red * ep_size)
    hist = None
    if reorder:
        hist = (np.clip(rng.standard_normal(n_logical) * 0.15 + 1, 0, None) * 2 ** 20).astype(np.int64)
    phy2log, log2phy, logcnt = build_redundancy_mapping(shape.r2o, ep_size, n_logical, shape.n_physical, hist,
                                                        n_nodes=max(1, ep_size // gpus_per_node))
    workload = (np.clip(rng.standard_normal(n_logical) * 0.3 + 1, 0, None) * 2 ** 12).astype(np.int32)
    return shape, hist, phy2log, log2phy, workload
