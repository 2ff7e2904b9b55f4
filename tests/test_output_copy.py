"""Fields copied through the ring of pinned chunks (csrc/output_copy.hpp) against those below its
smallest size: the norm of E, element by element, is the |E| of the same block. The hand-over itself, with
every byte looked at, on the CPU."""

from __future__ import annotations

import subprocess
from pathlib import Path

import numpy as np
import pytest

from cunibs_amd import synthetic

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def host_program(tmp_path_factory):
    out = tmp_path_factory.mktemp("copy") / "output_copy_host"
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{ROOT / 'cunibs_amd' / 'csrc'}", str(ROOT / "tests" / "output_copy_host.cpp"), "-o", str(out)],
                   check=True, capture_output=True, text=True)
    return out


@pytest.mark.parametrize("failing,no_pinned", [(-1, 0), (-1, 1), (2, 0), (3, 0), (5, 0), (7, 0)])
def test_ring_hands_over_every_byte(host_program, failing, no_pinned):
    """Whole, without pinned memory, and when an allocation of one of the threads fails (the first two are
    the copy's own tables)."""
    done = subprocess.run([str(host_program), str(failing), str(no_pinned)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout + done.stderr


@pytest.fixture(scope="module")
def ctx():
    from cunibs_amd import fem
    head = synthetic.shell_head(4.0, perturb_rms_mm=1.0, seed=2)
    c = fem.SolverContext(head.nodes_mm, head.tet_nodes, head.tet_tags, head.skin_tris)
    yield c
    c.free()


@pytest.mark.gpu
@pytest.mark.parametrize("k", [1, 2, 4, 5])  # E of 3.7, 7.4, 14.9 and 18.6 MB: below the ring, within it, past it
def test_fields_through_the_ring(ctx, k):
    from cunibs_amd import fem
    coil = synthetic.figure8_coil(seed=3, per_layer=40)
    sites = synthetic.cap_sites(k, seed=k)
    res = fem.solve_placements_block(ctx, coil.positions_m, coil.moments, sites, 1e6, vectors=True, potential=True,
                                     tolerance=0.5)
    for r in res:
        norm = np.linalg.norm(r.E.astype(np.float64), axis=1)
        # three FP32 products and sums and a square root: 4 eps
        assert np.all(np.abs(norm - r.magnE) <= 4 * 2.0 ** -24 * norm + 1e-30)
        assert np.all(np.isfinite(r.v))
