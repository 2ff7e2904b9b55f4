"""The V-cycle's row kernels where a mesh's rows end inside an ELL slice (8 rows), a wavefront or a
block, in both layouts of the finest level, against the FP64 V-cycle."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import boundary_tris, kuhn_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(10, 10, 8), (11, 10, 7), (12, 12, 12), (40, 6, 5)])
def test_vcycle_with_ragged_rows(oracle_mod, shape):
    from cunibs_amd import fem
    nodes, tets = kuhn_grid(*shape, jitter=0.2, seed=1)
    tags = np.ones(len(tets), np.int32)
    mesh = (nodes, tets, tags, boundary_tris(tets, nodes))
    oc = oracle_mod.build_context(*mesh)
    b = np.random.default_rng(0).standard_normal((oc.reduced.n, 8)).astype(np.float32)
    want = np.stack([oracle_mod.vcycle_apply(oc.hier, c.astype(np.float64)) for c in b.T], 1)
    ctx = fem.SolverContext(*mesh)
    try:
        assert ctx.info.n_levels >= 1
        for layout in (1, 2):
            ctx.set_tuning(layout=layout)
            for k in (1, 2, 4, 8):
                got = ctx.vcycle(np.ascontiguousarray(b[:, :k]))
                # the bound of the V-cycle's other tests: some hundred FP32 roundings in a row
                assert np.linalg.norm(got - want[:, :k]) < 1e-5 * np.linalg.norm(want[:, :k])
    finally:
        ctx.free()
