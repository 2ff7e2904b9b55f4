"""The dense coarsest level (csrc/amg.hip, coarse_inverse) at the edges of its 32-pivot blocks: on a
mesh of n + 1 nodes kept as one level, the V-cycle is the operator's inverse."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import boundary_tris

pytestmark = pytest.mark.gpu


def tet_chain(n_nodes: int):
    """Consecutive nodes of a helix, every four of them a regular tetrahedron (edge 10 mm)."""
    i = np.arange(n_nodes)
    th = np.arccos(-2.0 / 3.0) * i
    r = 3.0 * np.sqrt(3.0) / 10.0
    nodes = 10.0 * np.stack([r * np.cos(th), r * np.sin(th), i / np.sqrt(10.0)], 1)
    tets = np.stack([i[:-3], i[1:-2], i[2:-1], i[3:]], 1).astype(np.int32)
    p = nodes[tets]
    det = np.einsum("ij,ij->i", np.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]), p[:, 3] - p[:, 0])
    tets[det < 0] = tets[det < 0][:, [0, 2, 1, 3]]
    return nodes, tets


@pytest.mark.parametrize("n", [3, 31, 32, 33, 63, 65, 333])
def test_one_level_vcycle_is_the_inverse(oracle_mod, n):
    from cunibs_amd import fem
    nodes, tets = tet_chain(n + 1)
    tags = np.ones(len(tets), np.int32)
    skin = boundary_tris(tets, nodes)
    a = oracle_mod.build_context(nodes, tets, tags, skin, hierarchy=False).reduced.dense()
    b = np.random.default_rng(n).standard_normal((n, 4)).astype(np.float32)
    ctx = fem.SolverContext(nodes, tets, tags, skin, aggregation=fem.AggregationParams(min_coarse_rows=4096))
    try:
        assert ctx.info.n_levels == 0
        got = ctx.vcycle(b)
    finally:
        ctx.free()
    want = np.linalg.solve(a, b.astype(np.float64))
    # an elimination's FP64 rounding, n eps cond, and the result's FP32 rounding
    assert np.abs(got - want).max() <= (6e-8 + n * 2.3e-16 * np.linalg.cond(a)) * np.abs(want).max()
