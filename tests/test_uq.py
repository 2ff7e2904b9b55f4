"""Conductivity uncertainty: the sampling law (the reference's tests/test_uq_sampling.py tier, CPU)
and the multi-matrix block solve against per-sample FP64 oracle solves (GPU)."""

from __future__ import annotations

import numpy as np
import pytest


def test_sampling_is_seeded_lognormal_with_the_table_mean():
    from cunibs_amd.uq import draw_lognormal
    tags = [1, 2, 3, 4, 5]
    a = draw_lognormal(tags, 20000, 0.2, seed=3)
    b = draw_lognormal(tags, 20000, 0.2, seed=3)
    np.testing.assert_array_equal(a, b)
    s0 = np.array([0.126, 0.275, 1.654, 0.010, 0.465])
    np.testing.assert_allclose(a.mean(axis=0), s0, rtol=0.01)  # mean-preserving form
    np.testing.assert_allclose(np.log(a).std(axis=0), 0.2, rtol=0.03)
    med = draw_lognormal(tags, 20000, 0.2, seed=4, mean_preserving=False)
    np.testing.assert_allclose(np.median(med, axis=0), s0, rtol=0.02)
    assert not np.array_equal(a, draw_lognormal(tags, 20000, 0.2, seed=5))


@pytest.mark.gpu
def test_uq_samples_match_per_sample_fp64_solves(head4, coil, oracle_mod):
    from cunibs_amd import fem, synthetic, uq
    ctx = fem.SolverContext(head4.nodes_mm, head4.tet_nodes, head4.tet_tags, head4.skin_tris)
    try:
        site = synthetic.SPHERE_SITE
        tags = ctx.uq_prepare(coil.positions_m, coil.moments, site, 1e6)
        assert tags == [1, 2, 3, 4, 5]
        sigma = uq.draw_lognormal(tags, 5, 0.2, seed=11)
        sigma[0] = [fem.TISSUE_CONDUCTIVITY[t] for t in tags]  # the nominal table
        res = ctx.uq_solve(sigma)
        nominal = fem.solve_placements_block(ctx, coil.positions_m, coil.moments, [site], 1e6)[0]
        assert np.linalg.norm(res[0].magnE - nominal.magnE) <= 1e-5 * np.linalg.norm(nominal.magnE)
        gm = ctx.tet_tags == 2
        for i in (1, 3, 4):
            table = dict(fem.TISSUE_CONDUCTIVITY)
            table.update({t: float(s) for t, s in zip(tags, sigma[i])})
            octx = oracle_mod.build_context(head4.nodes_mm, head4.tet_nodes, head4.tet_tags, head4.skin_tris,
                                            conductivity=table)
            ref = oracle_mod.solve_site(octx, coil.positions_m, coil.moments, site, 1e6, tol=1e-12)
            assert res[i].relative_residual <= 1e-6
            err = np.linalg.norm(res[i].magnE[gm] - ref["magnE"][gm]) / np.linalg.norm(ref["magnE"][gm])
            assert err < 1e-4
            assert float(res[i].metrics[0]) == pytest.approx(float(ref["magnE"][gm].max()), rel=1e-3)
        mean, var, count = ctx.uq_moments()
        assert count == 5
        stack = np.stack([r.magnE.astype(np.float64) for r in res])
        np.testing.assert_allclose(mean, stack.mean(axis=0), rtol=1e-12, atol=1e-12)
        np.testing.assert_allclose(var, stack.var(axis=0, ddof=1), rtol=1e-6, atol=1e-9 * stack.max() ** 2)
        # The initial guess (run.py:154-200) changes where a draw starts, not where it lands: from
        # zero the same draws reach the same field, in more iterations.
        info = ctx.uq_guess_info()
        assert info["rank"] == len(tags) and info["nominal_iterations"] > 0
        cold = ctx.uq_solve(sigma, initial_guess=False)
        for a, b in zip(res, cold):
            assert np.linalg.norm(a.magnE - b.magnE) <= 2e-5 * np.linalg.norm(b.magnE)
        assert sum(r.iterations for r in res) < sum(r.iterations for r in cold)
        assert res[0].iterations <= 2  # the nominal draw starts at x_nom
    finally:
        ctx.free()



@pytest.mark.gpu
def test_placements_prepared_anew_keep_the_captured_iterations(head8, coil):
    """A second placement's draws replay the iterations captured for the first's, whatever was allocated
    in between, and give what a context of their own gives."""
    from cunibs_amd import fem, synthetic, uq
    mesh = (head8.nodes_mm, head8.tet_nodes, head8.tet_tags, head8.skin_tris)
    sites = synthetic.cap_sites(3, seed=29)

    def draws(ctx, site):
        tags = ctx.uq_prepare(coil.positions_m, coil.moments, site, 1e6)
        sigma = uq.draw_lognormal(tags, 11, 0.2, seed=2)
        fields = [r.magnE for part in (sigma[:8], sigma[8:]) for r in ctx.uq_solve(part)]
        return np.stack(fields), ctx.uq_moments()

    ctx, others = fem.SolverContext(*mesh), []
    try:
        draws(ctx, sites[0])  # every width's buffers and captures, the single-column solve's second ones
        draws(ctx, sites[0])
        count = ctx.graph_execs()
        for site in sites:
            fields, (mean, var, n) = draws(ctx, site)
            assert ctx.graph_execs() == count
            assert n == 11
            others.append(fem.SolverContext(*mesh))  # takes the memory that the placement gave back
            want, (want_mean, want_var, _) = draws(others[-1], site)
            np.testing.assert_array_equal(fields, want)
            np.testing.assert_array_equal(mean, want_mean)
            np.testing.assert_array_equal(var, want_var)
    finally:
        for c in (ctx, *others):
            c.free()


@pytest.mark.gpu
def test_asking_for_the_potential_changes_nothing_else(head8, coil):
    from cunibs_amd import fem, synthetic, uq
    ctx = fem.SolverContext(head8.nodes_mm, head8.tet_nodes, head8.tet_tags, head8.skin_tris)
    try:
        tags = ctx.uq_prepare(coil.positions_m, coil.moments, synthetic.SPHERE_SITE, 1e6)
        sigma = uq.draw_lognormal(tags, 5, 0.2, seed=7)
        plain = ctx.uq_solve(sigma, vectors=True)
        asked = ctx.uq_solve(sigma, vectors=True, potential=True)
    finally:
        ctx.free()
    for a, b in zip(plain, asked):
        np.testing.assert_array_equal(a.E, b.E)
        np.testing.assert_array_equal(a.magnE, b.magnE)
        np.testing.assert_array_equal(a.metrics, b.metrics)
        assert a.relative_residual == b.relative_residual


@pytest.mark.gpu
def test_the_spread_of_few_draws_matches_fp64_solves(head8, coil, oracle_mod):
    """Ten draws' standard deviation, element by element. A solve to 1e-6 leaves 2e-5 of a draw's field at
    most, and a standard deviation moves by no more than that of the draws' errors, which is sqrt(n / (n - 1))
    of their root mean square."""
    from cunibs_amd import fem, synthetic, uq
    mesh = (head8.nodes_mm, head8.tet_nodes, head8.tet_tags, head8.skin_tris)
    site = synthetic.SPHERE_SITE
    ctx = fem.SolverContext(*mesh)
    try:
        tags = ctx.uq_prepare(coil.positions_m, coil.moments, site, 1e6)
        sigma = uq.draw_lognormal(tags, 10, 0.2, seed=13)
        ctx.uq_solve(sigma, magnitude=False)
        mean, var, _ = ctx.uq_moments()
    finally:
        ctx.free()
    want = np.stack([oracle_mod.solve_site(
        oracle_mod.build_context(*mesh, conductivity={**fem.TISSUE_CONDUCTIVITY, **dict(zip(tags, map(float, row)))}),
        coil.positions_m, coil.moments, site, 1e6, tol=1e-12)["magnE"] for row in sigma])
    spread = want.std(axis=0, ddof=1)
    assert np.linalg.norm(mean - want.mean(axis=0)) <= 2e-5 * np.linalg.norm(want.mean(axis=0))
    assert np.linalg.norm(np.sqrt(var) - spread) <= 2e-5 * np.sqrt(10.0 / 9.0) * np.linalg.norm(mean)


@pytest.mark.gpu
def test_draws_carry_no_net_current(head8, coil):
    """A draw's right-hand side is brought to a zero sum after its tissues' vectors are combined, so its
    potential is off by no more of a constant than a block's of the same conductivities (1e-6 of its norm
    each; up to 7e-6 if the tissues' vectors are balanced instead, whose combination rounds anew)."""
    from cunibs_amd import fem, synthetic, uq
    ctx = fem.SolverContext(head8.nodes_mm, head8.tet_nodes, head8.tet_tags, head8.skin_tris)
    try:
        for site in synthetic.cap_sites(4, seed=31):
            tags = ctx.uq_prepare(coil.positions_m, coil.moments, site, 1e6)
            sigma = uq.draw_lognormal(tags, 3, 0.2, seed=2)
            got = ctx.uq_solve(sigma, potential=True)
            rows = fem.conductivity_rows([dict(zip(tags, map(float, r))) for r in sigma])
            want = fem.solve_placements_block(ctx, coil.positions_m, coil.moments, [site] * 3, 1e6, potential=True,
                                              sigma=rows)
            for a, b in zip(got, want):
                assert abs((a.v - b.v).mean()) * np.sqrt(a.v.size) <= 2e-6 * np.linalg.norm(b.v)
    finally:
        ctx.free()


@pytest.mark.gpu
def test_per_placement_conductivities_match_fp64_solves(head4, coil, oracle_mod):
    """solve_placements_block(sigma=...): every placement of a block with its own conductivities,
    against the FP64 oracle built with that placement's table; the nominal row reproduces the
    plain solve."""
    from cunibs_amd import fem, synthetic
    ctx = fem.SolverContext(head4.nodes_mm, head4.tet_nodes, head4.tet_tags, head4.skin_tris)
    try:
        sites = synthetic.cap_sites(3, seed=9)
        overrides = [None, {1: 0.2, 2: 0.4, 4: 0.006}, {3: 1.2, 5: 0.3}]
        rows = fem.conductivity_rows(overrides)
        res = fem.solve_placements_block(ctx, coil.positions_m, coil.moments, sites, 1e6, sigma=rows)
        plain = fem.solve_placements_block(ctx, coil.positions_m, coil.moments, sites[:1], 1e6)[0]
        assert np.linalg.norm(res[0].magnE - plain.magnE) <= 2e-5 * np.linalg.norm(plain.magnE)
        gm = ctx.tet_tags == 2
        for i in (1, 2):
            table = dict(fem.TISSUE_CONDUCTIVITY)
            table.update(overrides[i])
            octx = oracle_mod.build_context(head4.nodes_mm, head4.tet_nodes, head4.tet_tags, head4.skin_tris,
                                            conductivity=table)
            ref = oracle_mod.solve_site(octx, coil.positions_m, coil.moments, sites[i], 1e6, tol=1e-12)
            assert res[i].relative_residual <= 1e-6
            err = np.linalg.norm(res[i].magnE[gm] - ref["magnE"][gm]) / np.linalg.norm(ref["magnE"][gm])
            assert err < 1e-4
        with pytest.raises(ValueError):
            bad = rows.copy()
            bad[1, 3] = -1.0
            fem.solve_placements_block(ctx, coil.positions_m, coil.moments, sites, 1e6, sigma=bad)
    finally:
        ctx.free()


def test_reference_sampling_law_per_tissue_cov():
    """config.py:56-72: log-normal with E[sigma] = sigma_0 and the tissue's coefficient of
    variation; the normal law clamps at 1e-6 sigma_0; overrides replace the default table."""
    from cunibs_amd import fem
    from cunibs_amd.uq import DEFAULT_TISSUE_COV, ConductivityUQConfig, sample_conductivities
    tags = (1, 2, 3, 5)
    cfg = ConductivityUQConfig(n_samples=40000, seed=2)
    a = sample_conductivities(cfg, tags)
    assert a.shape == (40000, 4) and (a > 0).all()
    np.testing.assert_array_equal(a, sample_conductivities(cfg, tags))
    s0 = np.array([fem.TISSUE_CONDUCTIVITY[t] for t in tags])
    cov = np.array([DEFAULT_TISSUE_COV[t] for t in tags])
    np.testing.assert_allclose(a.mean(axis=0), s0, rtol=0.01)
    np.testing.assert_allclose(a.std(axis=0) / a.mean(axis=0), cov, rtol=0.05)
    # log sigma is normal with variance log(1 + cov^2)
    np.testing.assert_allclose(np.log(a).var(axis=0), np.log1p(cov ** 2), rtol=0.05)
    fixed = sample_conductivities(ConductivityUQConfig(n_samples=8, tissue_cov={t: 0.0 for t in tags}), tags)
    np.testing.assert_array_equal(fixed, np.tile(s0, (8, 1)))
    wide = sample_conductivities(ConductivityUQConfig(n_samples=20000, seed=1, distribution="normal",
                                                      tissue_cov={1: 3.0, 2: 0.1, 3: 0.1, 5: 0.1}), tags)
    assert wide[:, 0].min() == pytest.approx(1e-6 * s0[0])  # the clamp floor is reached
    with pytest.raises(KeyError):
        ConductivityUQConfig().cov_for(42)


def test_tissue_sensitivity_recovers_a_log_linear_response():
    """result.py:31-61: for y = c prod sigma_j^b_j the regression recovers b exactly, so the shares
    are b_j^2 Var(log sigma_j) / Var(log y) (summing to one up to the draws' sample correlation);
    an output that ignores a tissue gets zero share."""
    from cunibs_amd.uq import ConductivityUQConfig, ConductivityUQResult, sample_conductivities
    tags = (1, 2, 3)
    sig = sample_conductivities(ConductivityUQConfig(n_samples=400, seed=5), tags)
    b = np.array([2.0, 0.0, -1.0])
    y = 0.7 * np.exp(np.log(sig) @ b)
    r = ConductivityUQResult(None, None, None, 400, tags, sig, None, None, None, None, "c", 1e6, y, y * 2.0,
                             np.zeros((400, 3)), {"roi": y ** 0.5})
    share = r.tissue_sensitivity("peak")
    lx = np.log(sig)
    expect = b ** 2 * lx.var(axis=0) / np.log(y).var()
    np.testing.assert_allclose([share[t] for t in tags], expect, rtol=1e-9, atol=1e-12)
    assert sum(share.values()) == pytest.approx(1.0, abs=0.1)
    assert share[2] == pytest.approx(0.0, abs=1e-12)
    assert r.tissue_sensitivity("roi") == pytest.approx(share)  # a power of y has the same shares
    with pytest.raises(ValueError, match="Unknown output"):
        r.tissue_sensitivity("nope")


def test_tissue_sensitivity_on_an_orthogonal_design():
    """Closed form: on a two-level full factorial design the centred log-conductivity columns are
    exactly orthogonal, so a log-linear response with slopes b has shares b_j^2 s_j^2 /
    sum_k b_k^2 s_k^2 (half-ranges s_j), summing to one; a tissue held fixed gets share 0 and a
    constant output gives all zeros."""
    import itertools
    from cunibs_amd.uq import ConductivityUQResult
    tags = (1, 2, 3, 5)
    half = np.array([0.1, 0.3, 0.2, 0.0])  # tag 5 never varies
    levels = np.array(list(itertools.product((-1.0, 1.0), repeat=3)))
    logs = np.concatenate([levels * half[:3], np.zeros((8, 1))], axis=1) + np.log([0.1, 0.3, 1.6, 0.5])
    b = np.array([1.5, -0.5, 2.0, 7.0])
    y = np.exp(0.3 + (logs - logs.mean(0)) @ b)

    def make(out):
        return ConductivityUQResult(None, None, None, 8, tags, np.exp(logs), None, None, None, None, "c", 1e6,
                                    out, np.ones(8), np.zeros((8, 3)), {})

    share = make(y).tissue_sensitivity("peak")
    w = b[:3] ** 2 * half[:3] ** 2
    np.testing.assert_allclose([share[t] for t in tags[:3]], w / w.sum(), rtol=1e-12)
    assert share[5] == 0.0
    assert sum(share.values()) == pytest.approx(1.0, rel=1e-12)
    assert make(y).tissue_sensitivity("focality") == dict.fromkeys(tags, 0.0)


@pytest.mark.gpu
@pytest.mark.parametrize("recovery", ["raw", "harmonic"])
def test_subject_uq_with_fixed_conductivities_reproduces_simulate(head4, coil, recovery):
    """With every coefficient of variation zero each draw is the nominal model, so the Monte Carlo
    mean is the deterministic field of Subject.simulate under the same recovery, its spread is
    zero, and every draw's peak is the deterministic peak."""
    from cunibs_amd import synthetic
    from cunibs_amd.simulation import Placement, Subject
    from cunibs_amd.uq import ConductivityUQConfig
    subj = Subject(head4)
    try:
        place = Placement(*synthetic.SPHERE_SITE)
        det = subj.simulate(coil, place, 1e6, magnitude=True, recovery=recovery)
        cfg = ConductivityUQConfig(n_samples=6, tissue_cov={t: 0.0 for t in range(1, 11)})
        r = subj.simulate_conductivity_uq(coil, place, cfg, 1e6, moments=True, recovery=recovery)
        assert r.recovery == recovery and r.n_samples == 6 and r.perturbed_tags == (1, 2, 3, 4, 5)
        assert r.sigma_samples.shape == (6, 5)
        ref = det.magnE.astype(np.float64)
        assert np.linalg.norm(r.mean_magnE - ref) <= 2e-5 * np.linalg.norm(ref)
        assert float(np.max(r.std_magnE)) <= 1e-5 * float(ref.max())
        np.testing.assert_allclose(r.peak_samples, det.peak_magnE(), rtol=2e-5)
        assert r.peak_mean_magnE() == pytest.approx(det.peak_magnE(), rel=2e-5)
        assert r.max_local_cov() <= 1e-4
        lean = subj.simulate_conductivity_uq(coil, place, cfg, 1e6, recovery=recovery)
        assert lean.mean_magnE is None and lean.summary is not None
    finally:
        subj.free()


@pytest.mark.gpu
def test_subject_uq_draws_spread_and_attribute_to_tissues(head4, coil):
    """Perturbing gray matter alone: the draws spread the peak, the ROI records each draw's mean
    |E| over the region it names, and the whole log-variance of the peak goes to that tissue."""
    from cunibs_amd import synthetic
    from cunibs_amd.simulation import Placement, Subject
    from cunibs_amd.uq import ConductivityUQConfig
    subj = Subject(head4)
    try:
        place = Placement(*synthetic.SPHERE_SITE)
        gm = np.nonzero(subj.mesh.tet_tags == 2)[0]
        w = np.full(gm.size, 1.0 / gm.size)
        cfg = ConductivityUQConfig(n_samples=24, seed=3, perturbed_tags=(2,), tissue_cov={2: 0.3})
        r = subj.simulate_conductivity_uq(coil, place, cfg, 1e6, moments=True, recovery="raw",
                                          record_rois={"gm_mean": (gm, w)})
        assert r.sigma_samples.shape == (24, 1) and r.perturbed_tags == (2,)
        assert np.std(r.peak_samples) > 1e-3 * np.mean(r.peak_samples)
        assert r.roi_samples["gm_mean"].shape == (24,) and (r.roi_samples["gm_mean"] > 0).all()
        share = r.tissue_sensitivity("peak")
        assert set(share) == {2} and 0.5 < share[2] <= 1.0 + 1e-9
        assert r.iterations is not None and (r.iterations > 0).all()
    finally:
        subj.free()


@pytest.mark.parametrize("moments", [True, False])
def test_uq_result_save_load_round_trip(tmp_path, moments):
    """result.py:182-256 there: the draws, per-draw scalars, ROI records and summary come back;
    moment arrays the run did not keep load as None."""
    from cunibs_amd.simulation import Placement
    from cunibs_amd.uq import ConductivityUQResult, ConductivityUQSummary
    rng = np.random.default_rng(1)
    m, n = 30, 7
    summary = ConductivityUQSummary(
        {"region": "gray_matter", "peak_magnE": 0.4, "peak_location_mm": np.array([1.0, 2.0, 3.0]),
         "center_of_gravity_mm": np.array([0.0, 1.0, 2.0]), "region_volume_m3": 2e-6,
         "focality_m3": {"0.5": 1e-7, "0.75": 5e-8},
         "distribution": {"mean": 0.1, "std": 0.02, "p50": 0.1, "p95": 0.2, "p99": 0.3, "p99.9": 0.35}}, 0.12)
    mom = (lambda a: a) if moments else (lambda a: None)
    r = ConductivityUQResult(
        mom(rng.random(m).astype(np.float32)), mom(rng.random(m).astype(np.float32)),
        mom(rng.random(m).astype(np.float32)), n, (1, 2), rng.random((n, 2)), mom(rng.random(m).astype(np.float32)),
        mom(rng.integers(1, 4, m).astype(np.int32)), mom(rng.random((m, 3))),
        Placement([0.0, 0.0, 90.0], [0.0, 50.0, 90.0], 4.0), "D70", 1e6, rng.random(n), rng.random(n),
        rng.random((n, 3)), {} if moments else {"m1": rng.random(n)}, summary, "harmonic")
    r.save(tmp_path / "uq.h5")
    b = ConductivityUQResult.load(tmp_path / "uq.h5")
    for name in ("mean_magnE", "std_magnE", "cov_magnE", "vols", "tet_tags", "barycenters_mm"):
        if getattr(r, name) is None:
            assert getattr(b, name) is None
        else:
            np.testing.assert_array_equal(getattr(b, name), getattr(r, name))
    for name in ("sigma_samples", "peak_samples", "focality_samples", "peak_location_samples"):
        np.testing.assert_array_equal(getattr(b, name), getattr(r, name))
    assert set(b.roi_samples) == set(r.roi_samples)
    for k in r.roi_samples:
        np.testing.assert_array_equal(b.roi_samples[k], r.roi_samples[k])
    assert (b.n_samples, b.perturbed_tags, b.coil_name, b.didt, b.recovery) == (n, (1, 2), "D70", 1e6, "harmonic")
    assert b.summary.max_local_cov == 0.12 and b.summary.mean_field["peak_magnE"] == 0.4
    assert b.tissue_sensitivity("peak") == pytest.approx(r.tissue_sensitivity("peak"))
