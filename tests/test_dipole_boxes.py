"""The block N-body (csrc/dipole.hip) against the dipoles' closed form in FP64, with and without the
box method, at the sizes where its parts change: the widths at which waves share a placement, ragged
widths, the smallest coil the boxes take, coils whose moments are parallel and not, and the two
depths of the boxes."""

from __future__ import annotations

import numpy as np
import pytest

from cunibs_amd import synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[8.0, 3.2, 2.0])  # below the box method, three levels, four
def ctx(request):
    from cunibs_amd import fem
    head = synthetic.shell_head(request.param, perturb_rms_mm=1.0, seed=2)
    c = fem.SolverContext(head.nodes_mm, head.tet_nodes, head.tet_tags, head.skin_tris)
    yield c
    c.free()


def nodal(ctx, pos, mom, sites):
    from cunibs_amd import fem
    ex = {"dadt_nodes": 1}
    res = fem.solve_placements_block(ctx, pos, mom, sites, 1e6, magnitude=False, metrics=False, extra=ex,
                                     tolerance=0.5)  # the solve itself is not looked at
    return ex["dadt_nodes"], [r.transform for r in res]


def closed_form(pos, mom, tf, nodes_mm):
    s = pos @ tf[:3, :3].T + tf[:3, 3] * 1e-3
    m = mom @ tf[:3, :3].T
    out = np.empty((nodes_mm.shape[0], 3))
    for i, x in enumerate(nodes_mm * 1e-3):
        d = x - s
        out[i] = 0.1 * (np.cross(m, d) / (np.linalg.norm(d, axis=1) ** 3)[:, None]).sum(0)
    return out


@pytest.mark.parametrize("k,dipoles,bent", [(1, 2400, False), (1, 256, True), (2, 255, False), (3, 257, True),
                                            (5, 600, False), (8, 1002, True), (17, 300, False)])
def test_block_dadt_matches_the_closed_form(ctx, k, dipoles, bent):
    coil = synthetic.figure8_coil(seed=3, per_layer=-(-dipoles // 6))
    pos, mom = coil.positions_m[:dipoles].copy(), coil.moments[:dipoles].copy()
    if bent:
        mom += 0.1 * np.abs(mom).max() * np.random.default_rng(1).standard_normal(mom.shape)
    sites = synthetic.cap_sites(k, seed=k, distance_range_mm=(3.0, 8.0))
    got, tf = nodal(ctx, pos, mom, sites)
    rng = np.random.default_rng(0)
    pick = np.unique(np.concatenate([rng.integers(0, ctx.n_nodes, 600), [0, ctx.n_nodes - 1],
                                     np.argsort(ctx.nodes_mm[:, 2])[-200:]]))
    for i in range(k):
        want = closed_form(pos, mom, tf[i], ctx.nodes_mm[pick])
        err = np.linalg.norm(got[i][pick] - want, axis=1)
        # 2-norm: the truncation of the boxes (1e-7 of the field) and FP32 pair terms whose r - s is
        # rounded to 2^-24 of 0.1 m: 6e-9 m over the 3 mm of the closest pairs, three times in the cube.
        assert np.linalg.norm(err) <= 6e-6 * np.linalg.norm(want)
        # At a single node the contributions of the two wings cancel; bounded by the field's scale there.
        assert err.max() <= 2e-5 * np.abs(want).max()


def test_a_placement_does_not_depend_on_its_block(ctx):
    coil = synthetic.figure8_coil(seed=4)
    sites = synthetic.cap_sites(9, seed=5)
    whole, _ = nodal(ctx, coil.positions_m, coil.moments, sites)
    for lo, hi in ((0, 1), (1, 3), (3, 8)):  # waves share a placement eight, four and two ways
        part, _ = nodal(ctx, coil.positions_m, coil.moments, sites[lo:hi])
        np.testing.assert_array_equal(part, whole[lo:hi])


@pytest.mark.parametrize("k", [1, 3, 17])
def test_right_hand_sides_sum_to_zero(ctx, k):
    """A field without sources puts no net current into the head: what FP32 rounding leaves of the sum
    is taken back, to one rounding (2^-24) of the largest entry and of the ground node's own."""
    from cunibs_amd import fem
    coil = synthetic.figure8_coil(seed=6)
    ex = {"rhs": 1}
    fem.solve_placements_block(ctx, coil.positions_m, coil.moments, synthetic.cap_sites(k, seed=k), 1e6,
                               magnitude=False, metrics=False, extra=ex, tolerance=0.5)
    b = ex["rhs"].astype(np.float64)
    assert np.all(np.abs(b.sum(1)) <= 2.0 * 2.0**-24 * np.abs(b).max(1))


@pytest.fixture(scope="module")
def fine():
    """A million nodes: deeper leaves, and the node pass that takes a block of workgroups per chunk."""
    from cunibs_amd import fem
    head = synthetic.shell_head(1.5, perturb_rms_mm=1.0, seed=2)
    c = fem.SolverContext(head.nodes_mm, head.tet_nodes, head.tet_tags, head.skin_tris)
    assert c.n_nodes >= 800000  # more than 8,192 chunks of 64 nodes
    yield c
    c.free()


def bent_coil(dipoles, tilt_deg=14.0):
    """Two wings tilted towards the head, whose moments differ in direction."""
    coil = synthetic.figure8_coil(seed=3, per_layer=-(-dipoles // 6))
    pos, mom = coil.positions_m[:dipoles].copy(), coil.moments[:dipoles].copy()
    for side in (-1.0, 1.0):
        t, wing = side * np.radians(tilt_deg), pos[:, 0] * side > 0
        turn = np.array([[np.cos(t), 0.0, -np.sin(t)], [0.0, 1.0, 0.0], [np.sin(t), 0.0, np.cos(t)]])
        pos[wing], mom[wing] = pos[wing] @ turn.T, mom[wing] @ turn.T
    return pos, mom


def rounding_bound(pos, mom, tf, nodes_mm):
    """What FP32 may cost where a coil is summed as W x r - P with |r - s|^2 = |r|^2 + |s|^2 - 2 r.s, r and s
    from the coil's origin: three roundings of |r|^2 + |s|^2 in a distance cubed, eight more of a term, and
    one for each addition, of terms as large as w |m| (|r| + |s|)."""
    s = pos @ tf[:3, :3].T
    m = np.linalg.norm(mom, axis=1)
    out = np.empty(nodes_mm.shape[0])
    for i, x in enumerate(nodes_mm * 1e-3 - tf[:3, 3] * 1e-3):
        d2 = ((x - s) ** 2).sum(1)
        size = (x @ x) + (s * s).sum(1)
        term = m * (np.sqrt(x @ x) + np.sqrt((s * s).sum(1))) / d2**1.5
        out[i] = 0.1 * 2.0**-24 * (term * (3 * 1.5 * size / d2 + 8 + len(m))).sum()
    return out


@pytest.mark.parametrize("k,dipoles,bent", [(9, 2400, False), (17, 300, False), (32, 601, False), (9, 1801, True),
                                            (17, 400, True), (32, 2400, True)])
def test_wide_blocks_on_a_fine_mesh(fine, k, dipoles, bent):
    """Against the closed form, and bit for bit against the same placements in narrow blocks, whose node
    passes are others (and, for a bent coil, sum the near chunks themselves)."""
    coil = synthetic.figure8_coil(seed=3, per_layer=-(-dipoles // 6))
    pos, mom = bent_coil(dipoles) if bent else (coil.positions_m[:dipoles], coil.moments[:dipoles])
    sites = synthetic.cap_sites(k, seed=k, distance_range_mm=(12.0, 14.0) if bent else (3.0, 8.0))
    got, tf = nodal(fine, pos, mom, sites)
    pick = np.random.default_rng(k).choice(fine.n_nodes, 400, replace=False)
    for i in (0, k // 2, k - 1):
        near = np.argsort(np.linalg.norm(fine.nodes_mm - tf[i][:3, 3], axis=1))[:200]
        rows = np.concatenate([pick, near])
        want = closed_form(pos, mom, tf[i], fine.nodes_mm[rows])
        err = np.linalg.norm(got[i][rows] - want, axis=1)
        if bent:
            bound = rounding_bound(pos, mom, tf[i], fine.nodes_mm[rows])
            assert np.all(err <= bound + 2e-5 * np.abs(want).max())
        else:
            assert np.linalg.norm(err) <= 6e-6 * np.linalg.norm(want)  # as above
    for lo, hi in ((0, 1), (3, 5), (k - 8, k)):
        part, _ = nodal(fine, pos, mom, sites[lo:hi])
        np.testing.assert_array_equal(part, got[lo:hi])


@pytest.mark.parametrize("k", [1, 12])
def test_a_bent_coil_that_all_but_touches_nodes(ctx, k):
    """Wings that reach into the scalp, within half a millimetre of nodes: the caller's order, whatever the
    order of the dipoles does to their clusters."""
    pos, mom = bent_coil(1500)
    sites = synthetic.cap_sites(k, seed=7, distance_range_mm=(2.0, 3.0))
    got, tf = nodal(ctx, pos, mom, sites)
    i = k - 1
    near = np.argsort(np.linalg.norm(ctx.nodes_mm - tf[i][:3, 3], axis=1))[:600]
    want = closed_form(pos, mom, tf[i], ctx.nodes_mm[near])
    err = np.linalg.norm(got[i][near] - want, axis=1)
    print(f"k={k} n={ctx.n_nodes}: {np.linalg.norm(err) / np.linalg.norm(want):.2e} of the 2-norm")
    assert np.all(err <= rounding_bound(pos, mom, tf[i], ctx.nodes_mm[near]))


def test_a_general_coils_sweep_equals_its_blocks(ctx):
    """The N-body beside a solve, on a capped grid, for a coil whose moments differ."""
    from cunibs_amd import fem
    pos, mom = bent_coil(900)
    sites = synthetic.cap_sites(11, seed=9, distance_range_mm=(12.0, 14.0))
    blocks = [r.metrics for i in range(0, 11, 4)
              for r in fem.solve_placements_block(ctx, pos, mom, sites[i:i + 4], 1e6, magnitude=False)]
    try:
        for cap in (0, 1, 7, 100):
            ctx.set_tuning(coil_blocks=cap)
            sweep = fem.solve_sweep(ctx, pos, mom, sites, 1e6, block_k=4, recycle=0)
            np.testing.assert_array_equal(sweep["metrics"], np.stack(blocks))
    finally:
        ctx.set_tuning(coil_blocks=0)


@pytest.mark.parametrize("bent,pairs,pairs_deep", [(False, 80000000, 200000000), (True, 240000000, 320000000)])
def test_both_sides_of_the_box_rule(ctx, bent, pairs, pairs_deep):
    """The last coil without boxes and the first with them, against the closed form."""
    first = max(256, -(-(pairs_deep if ctx.n_nodes >= 400000 else pairs) // ctx.n_nodes))
    for dipoles in (first - 1, first) if first < 4000 else (2000,):
        coil = synthetic.figure8_coil(seed=3, per_layer=-(-dipoles // 6))
        pos, mom = coil.positions_m[:dipoles].copy(), coil.moments[:dipoles].copy()
        if bent:
            mom += 0.1 * np.abs(mom).max() * np.random.default_rng(1).standard_normal(mom.shape)
        got, tf = nodal(ctx, pos, mom, synthetic.cap_sites(2, seed=3))
        pick = np.random.default_rng(2).choice(ctx.n_nodes, 400, replace=False)
        want = closed_form(pos, mom, tf[1], ctx.nodes_mm[pick])
        err = np.linalg.norm(got[1][pick] - want, axis=1)
        assert np.linalg.norm(err) <= 6e-6 * np.linalg.norm(want)  # as above
        assert err.max() <= 2e-5 * np.abs(want).max()


def test_a_coil_of_more_than_two_to_the_25_dipoles():
    """Nearly all of them without a moment."""
    from cunibs_amd import fem
    head = synthetic.shell_head(10.0, seed=2)
    n = 2**25 + 1
    rng = np.random.default_rng(0)
    live = np.append(rng.choice(n - 1, 63, replace=False), n - 1)
    pos, mom = np.zeros((n, 3)), np.zeros((n, 3))
    pos[live], mom[live, 2] = rng.uniform(-0.03, 0.03, (64, 3)) * [1.0, 1.0, 0.1], 1e-3
    ctx = fem.SolverContext(head.nodes_mm, head.tet_nodes, head.tet_tags, head.skin_tris)
    try:
        got, tf = nodal(ctx, pos, mom, synthetic.cap_sites(1, seed=1, distance_mm=8.0))
        want = closed_form(pos[live], mom[live], tf[0], ctx.nodes_mm)
    finally:
        ctx.free()
    err = np.linalg.norm(got[0] - want, axis=1)
    assert np.linalg.norm(err) <= 6e-6 * np.linalg.norm(want)  # as above: a zero term adds no rounding


def box_mesh(cells):
    """A box of 1 mm cells, six positively oriented tetrahedra each, and two triangles of its top."""
    side = cells + 1
    axis = np.arange(side, dtype=np.float64)
    nodes = np.stack(np.meshgrid(axis, axis, axis, indexing="ij"), -1).reshape(-1, 3)
    i = np.arange(cells, dtype=np.int32)
    base = ((i[:, None, None] * side + i[None, :, None]) * side + i).reshape(-1)
    step = np.array([side * side, side, 1], np.int32)
    tets = np.empty((6, base.size, 4), np.int32)
    for q, (a, b, odd) in enumerate(((0, 1, 0), (0, 2, 1), (1, 0, 1), (1, 2, 0), (2, 0, 0), (2, 1, 1))):
        path = [base, base + step[a], base + step[a] + step[b], base + step.sum()]
        if odd:
            path[1], path[2] = path[2], path[1]
        tets[q] = np.stack(path, 1)
    top = cells
    corner = [(x * side + y) * side + top for x, y in ((0, 0), (cells, 0), (cells, cells), (0, cells))]
    return nodes, tets.reshape(-1, 4), np.array([[corner[0], corner[1], corner[2]], [corner[0], corner[2], corner[3]]],
                                               np.int32)


def test_the_deepest_boxes():
    from cunibs_amd import fem
    nodes, tets, skin = box_mesh(147)
    assert nodes.shape[0] >= 3200000
    c = fem.SolverContext(nodes, tets, np.full(tets.shape[0], 2, np.int32), skin)
    try:
        coil = synthetic.figure8_coil(seed=3, per_layer=400)
        at = np.array([73.0, 73.0, 147.0])
        sites = [(at + [10.0 * i, 0.0, 0.0], at + [10.0 * i, 50.0, 0.0], 4.0) for i in range(9)]
        for k in (1, 9):
            got, tf = nodal(c, coil.positions_m, coil.moments, sites[:k])
            pick = np.random.default_rng(k).choice(c.n_nodes, 400, replace=False)
            want = closed_form(coil.positions_m, coil.moments, tf[k - 1], c.nodes_mm[pick])
            err = np.linalg.norm(got[k - 1][pick] - want, axis=1)
            assert np.linalg.norm(err) <= 6e-6 * np.linalg.norm(want)  # as above
            assert err.max() <= 2e-5 * np.abs(want).max()
    finally:
        c.free()
