"""The performance cases: what a user of this package has it do, over the range of sizes it is used at.

A head is five shells (white matter, gray matter, CSF, bone, scalp) on a lattice of ``spacing`` mm cut
into tetrahedra, as the package's own synthetic heads are, with the shells' surfaces bumped by a few
millimetres, every node moved a little off the lattice and, with ``refine`` > 0, that share of the
tetrahedra cut into four around a new node, so that rows are as irregular as an unstructured head's.
Spacings run from 10 mm (a quick look) over 3-2 mm (ordinary) to 1.5 mm (a million nodes). Coils are
figure-8 windings, flat (all dipole moments along one direction) or bent around the head (they are
not), of a few hundred to a few thousand dipoles. Placements are spread over the upper part of the
head. The seed makes the inputs: the head's shape (its lattice and shells are the case's), the sites,
the coil's windings, the conductivities.

Paths, each through the entry points that a program calls:

``simulate``  one placement through ``Subject.simulate``, with its fields
``fields``    a few placements through ``Subject.iter_simulate``, with every field they can return
``sweep``     many placements through ``Subject.iter_simulate``, summaries only
``sigma``     a block in which every placement has its own conductivities
``uq``        a conductivity Monte Carlo of one placement
``warm``      a sweep that starts from a reduced basis of earlier solutions
``setup``     a head's solver context and its recovery operator, from the mesh, and one cycle of its hierarchy
``network``   the learned warm start: gradients of one batch, and predictions
"""

from __future__ import annotations

import math

import numpy as np
import torch

from cunibs_amd import fem, learned, uq
from cunibs_amd.mesh import HeadMesh
from cunibs_amd.simulation import Coil, Placement, Subject

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
RADII_MM = (70.0, 75.0, 78.0, 86.0, 92.0)
SIGMA = {1: 0.126, 2: 0.275, 3: 1.654, 4: 0.010, 5: 0.465}
GRAY = 2
DIDT = 1e6
FIELDS = ("magnE", "E", "v", "E_slots")


def listed():
    return [
        # A quick look at one placement on a coarse head: latency and launches.
        {"name": "simulate_small", "path": "simulate", "spacing": 8.0, "refine": 0.0, "coil": "flat",
         "dipoles": 964, "recovery": "raw"},
        # One placement on an unstructured head of a region-of-interest study, with the default recovery.
        {"name": "simulate_irregular", "path": "simulate", "spacing": 4.0, "refine": 0.12, "coil": "bent",
         "dipoles": 1500, "recovery": "harmonic"},
        # One placement on a fine head, with its fields: what an interactive planner calls.
        {"name": "simulate_fine", "path": "simulate", "spacing": 2.0, "refine": 0.0, "coil": "flat",
         "dipoles": 2400, "recovery": "harmonic"},
        # A handful of placements whose fields are all kept, recovered per tissue.
        {"name": "fields_five", "path": "fields", "spacing": 3.0, "refine": 0.0, "coil": "flat", "dipoles": 2400,
         "placements": 5, "recovery": "spr_tissue"},
        # The headline: a sweep over a million-node head in the default blocks, default recovery.
        {"name": "sweep_fine", "path": "sweep", "spacing": 1.5, "refine": 0.0, "coil": "flat", "dipoles": 2400,
         "placements": 64, "block_k": 16, "recovery": "harmonic"},
        # A sweep on an unstructured head with a bent coil; the last block is ragged.
        {"name": "sweep_bent_ragged", "path": "sweep", "spacing": 2.5, "refine": 0.1, "coil": "bent",
         "dipoles": 1800, "placements": 41, "block_k": 16, "recovery": "raw"},
        # The widest blocks, raw field.
        {"name": "sweep_wide", "path": "sweep", "spacing": 2.5, "refine": 0.0, "coil": "flat", "dipoles": 964,
         "placements": 96, "block_k": 32, "recovery": "raw"},
        # Every placement of a block with its own tissue conductivities (training sets, sensitivity).
        {"name": "sigma_block", "path": "sigma", "spacing": 3.0, "refine": 0.0, "coil": "flat", "dipoles": 2400,
         "placements": 12, "recovery": "raw"},
        # Conductivity uncertainty of one placement.
        {"name": "uq_draws", "path": "uq", "spacing": 2.5, "refine": 0.0, "coil": "flat", "dipoles": 2400,
         "draws": 64, "recovery": "harmonic"},
        # A sweep warm-started from the solutions of earlier placements.
        {"name": "warm_sweep", "path": "warm", "spacing": 3.0, "refine": 0.0, "coil": "flat", "dipoles": 2400,
         "placements": 40, "block_k": 8, "snapshots": 64, "recovery": "raw"},
        # What a new head costs before its first placement.
        {"name": "setup_head", "path": "setup", "spacing": 2.0, "refine": 0.05, "recovery": "harmonic"},
        # One batch of the warm-start network's training, and its predictions.
        {"name": "network_batch", "path": "network", "rows": 2048, "hidden": 512, "outputs": 256},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    path = rng.choice(["simulate", "simulate", "fields", "sweep", "sweep", "sweep", "sigma", "uq", "warm", "setup",
                       "network"])
    if path == "network":
        return {"path": path, "rows": int(_log(rng, 17, 4096)), "hidden": 16 * rng.randint(4, 32),
                "outputs": 16 * rng.randint(1, 16)}
    fine = {"simulate": 1.7, "fields": 2.6, "sweep": 1.8, "sigma": 2.4, "uq": 2.4, "warm": 2.8, "setup": 1.8}[path]
    case = {"path": path, "spacing": round(_log(rng, fine, 10.0), 3),
            "refine": rng.choice([0.0, 0.0, round(rng.uniform(0.02, 0.15), 3)])}
    if case["refine"] > 0.0 and path not in ("setup",):
        case["spacing"] = max(case["spacing"], round(1.35 * fine, 3))
    case["recovery"] = rng.choice(["raw", "harmonic", "harmonic", "spr_tissue"])
    if path == "setup":
        return case
    case["coil"] = rng.choice(["flat", "flat", "bent"])
    case["dipoles"] = int(_log(rng, 300, 4000))
    if path == "fields":
        case["placements"] = rng.randint(2, 9)
        case["recovery"] = rng.choice(["harmonic", "spr_tissue"])
    elif path == "sweep":
        case["block_k"] = rng.choice([2, 4, 5, 8, 11, 16, 16, 16, 32])
        case["placements"] = case["block_k"] + rng.randint(1, 48)
    elif path == "sigma":
        case["placements"] = rng.randint(2, 16)
    elif path == "uq":
        case["draws"] = rng.randint(7, 72)
    elif path == "warm":
        case["block_k"] = rng.choice([4, 8, 16])
        case["placements"] = case["block_k"] + rng.randint(1, 24)
        case["snapshots"] = rng.choice([32, 48, 64])
    return case


# --------------------------------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------------------------------

# Corner x + 2 y + 4 z of a cell; the six tetrahedra around its 0-7 diagonal.
_CORNERS = torch.tensor([[c & 1, (c >> 1) & 1, c >> 2] for c in range(8)])
_TETS = torch.tensor([[0, 1, 3, 7], [0, 3, 2, 7], [0, 2, 6, 7], [0, 6, 4, 7], [0, 4, 5, 7], [0, 5, 1, 7]])


def head(spacing: float, refine: float, seed: int):
    """(nodes_mm, tet_nodes, tet_tags, skin_tris) as NumPy arrays. The elements are the case's own, so
    that results of two seeds have the same sizes; where the nodes lie is the seed's."""
    rng = np.random.default_rng(1)
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    cut_gen = torch.Generator(device=DEVICE).manual_seed(1)
    h = float(spacing)
    cells = int(math.ceil(2.0 * (RADII_MM[-1] + 7.0 + h) / h))
    side = cells + 1
    lo = -0.5 * cells * h
    axis = torch.arange(cells, device=DEVICE)
    cell = torch.stack(torch.meshgrid(axis, axis, axis, indexing="ij"), -1).reshape(-1, 3)
    corners, tets = _CORNERS.to(DEVICE), _TETS.to(DEVICE)
    centre = corners[tets].double().mean(1)  # (6, 3)
    x = lo + h * (cell[:, None, :] + centre[None])
    r = x.norm(dim=-1)
    u = x / r.clamp_min(1e-9)[..., None]
    bump = torch.zeros_like(r)
    for _ in range(6):
        w = torch.tensor(rng.normal(0.0, 1.6, 3), device=DEVICE)
        bump += 1.1 * torch.cos(u @ w + rng.uniform(0.0, 2.0 * math.pi))
    shell = torch.searchsorted(torch.tensor(RADII_MM, device=DEVICE, dtype=torch.float64), r - bump)
    ci, ti = torch.nonzero(shell < len(RADII_MM), as_tuple=True)
    tags = shell[ci, ti] + 1
    at = (cell[ci][:, None, :] + corners[tets][ti])  # (m, 4, 3)
    lin = at[..., 0] + side * (at[..., 1] + side * at[..., 2])
    used, tet = torch.unique(lin, return_inverse=True)
    nodes = lo + h * torch.stack([used % side, (used // side) % side, used // (side * side)], -1).double()
    nodes += 0.08 * h * (2.0 * torch.rand(nodes.shape, generator=gen, device=DEVICE, dtype=torch.float64) - 1.0)
    stretch = np.random.default_rng([seed, 1]).normal(0.0, 0.02, (3, 3))
    nodes = nodes @ (torch.eye(3, dtype=torch.float64) + torch.from_numpy(stretch + stretch.T)).to(DEVICE)
    if refine > 0.0:
        cut = torch.rand(tet.shape[0], generator=cut_gen, device=DEVICE) < refine
        old, mid = tet[cut], nodes.shape[0] + torch.arange(int(cut.sum()), device=DEVICE)
        nodes = torch.cat([nodes, nodes[old].mean(1)])
        new = old[:, None, :].repeat(1, 4, 1)
        for i in range(4):
            new[:, i, i] = mid
        tet = torch.cat([tet[~cut], new.reshape(-1, 4)])
        tags = torch.cat([tags[~cut], tags[cut].repeat_interleave(4)])
    n = nodes.shape[0]
    faces = tet[:, [[1, 2, 3], [0, 3, 2], [0, 1, 3], [0, 2, 1]]].reshape(-1, 3)
    s = faces.sort(dim=1).values
    key, order = ((s[:, 0] * n + s[:, 1]) * n + s[:, 2]).sort()
    same = key[1:] == key[:-1]
    edge = torch.zeros(1, dtype=torch.bool, device=DEVICE)
    outer = order[~(torch.cat([edge, same]) | torch.cat([same, edge]))].sort().values
    f = faces[outer]
    normal = torch.linalg.cross(nodes[f[:, 1]] - nodes[f[:, 0]], nodes[f[:, 2]] - nodes[f[:, 0]])
    inward = (normal * (nodes[tet.reshape(-1)[outer]] - nodes[f[:, 0]])).sum(-1) > 0
    f[inward] = f[inward][:, [0, 2, 1]]
    return (nodes.cpu().numpy(), tet.int().cpu().numpy(), tags.int().cpu().numpy(), f.int().cpu().numpy())


def coil(kind: str, dipoles: int, seed: int) -> Coil:
    """Two wings of three layers of dipoles on a spiral; "bent" tilts each wing towards the head."""
    rng = np.random.default_rng([seed, 2])
    per = max(1, dipoles // 6)
    i = np.arange(per)
    rad, ang = 35.0 * np.sqrt((i + 0.5) / per), i * math.pi * (3.0 - math.sqrt(5.0))
    pos, mom = [], []
    for sign in (-1.0, 1.0):
        tilt = sign * math.radians(14.0) if kind == "bent" else 0.0
        for z in (0.0, -1.5, -3.0):
            x = rad * np.cos(ang) + sign * 38.0
            p = np.stack([x, rad * np.sin(ang), np.full(per, z)], 1) + rng.normal(0.0, 0.1, (per, 3))
            rot = np.array([[math.cos(tilt), 0.0, -math.sin(tilt)], [0.0, 1.0, 0.0],
                            [math.sin(tilt), 0.0, math.cos(tilt)]])
            pos.append(p @ rot.T)
            mom.append(np.tile(rot @ [0.0, 0.0, -sign * 10.0 * math.pi * 0.035**2 / per], (per, 1)))
    return Coil(np.concatenate(pos) * 1e-3, np.concatenate(mom), name=f"{kind}_{dipoles}")


def sites(count: int, seed: int):
    """Placements on the upper part of the head, any handle angle, 2 to 8 mm off the scalp."""
    rng = np.random.default_rng([seed, 3])
    out = []
    for _ in range(count):
        ct, ph, a = rng.uniform(0.5, 1.0), rng.uniform(0.0, 2.0 * math.pi), rng.uniform(0.0, 2.0 * math.pi)
        st = math.sqrt(1.0 - ct * ct)
        d = np.array([st * math.cos(ph), st * math.sin(ph), ct])
        e1 = np.array([ct * math.cos(ph), ct * math.sin(ph), -st])
        e2 = np.array([-math.sin(ph), math.cos(ph), 0.0])
        out.append(Placement(92.0 * d, 92.0 * d + 50.0 * (math.cos(a) * e1 + math.sin(a) * e2), rng.uniform(2.0, 8.0)))
    return out


def conductivities(count: int, seed: int) -> np.ndarray:
    """One log-normal draw of the five tissues' conductivities per placement."""
    z = np.random.default_rng([seed, 4]).standard_normal((count, len(SIGMA)))
    return np.array(list(SIGMA.values())) * np.exp(0.2 * z)


def _triples(placements):
    return [(p.center_mm, p.handle_mm, p.distance_mm) for p in placements]


def prepare(case, seed):
    if case["path"] == "network":
        rng = np.random.default_rng([seed, 5])
        x = rng.normal(size=(case["rows"], learned.N_INPUTS)).astype(np.float32)
        decay = 1.0 / (1.0 + np.arange(case["outputs"]))
        t = (np.sin(x @ rng.normal(size=(learned.N_INPUTS, case["outputs"]))) * decay).astype(np.float32)
        net = learned.WarmStartNetwork(n_out=case["outputs"], hidden=case["hidden"], seed=seed % 65536)
        return {"case": case, "net": net, "x": x, "t": t}
    nodes, tets, tags, skin = head(case["spacing"], case["refine"], seed)
    state = {"case": case, "seed": seed, "mesh": (nodes, tets, tags, skin)}
    if case["path"] == "setup":
        rhs = np.random.default_rng([seed, 6]).standard_normal((nodes.shape[0] - 1, 1))
        state["rhs"] = rhs.astype(np.float32)
        return state
    state["subject"] = subject = Subject(HeadMesh(nodes, tets, tags, skin))
    subject.context  # a head's context is built once and kept
    state["coil"] = c = coil(case["coil"], case["dipoles"], seed)
    state["sites"] = sites(case.get("placements", 1), seed)
    if case["path"] == "sigma":
        table = conductivities(case["placements"], seed)
        state["rows"] = fem.conductivity_rows([dict(zip(SIGMA, map(float, row))) for row in table])
    if case["path"] == "uq":
        state["config"] = uq.ConductivityUQConfig(n_samples=case["draws"], seed=seed)
    if case["path"] == "warm":
        ctx, earlier = subject.context, _triples(sites(case["snapshots"], seed + 7919))
        ctx.warm_reset(case["snapshots"])
        for i in range(0, len(earlier), 16):
            fem.solve_placements_block(ctx, c.positions_m, c.moments, earlier[i:i + 16], DIDT, metrics=False,
                                       magnitude=False, collect=True)
        ctx.warm_finalize()
    return state


# --------------------------------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------------------------------


def _summaries(rows):
    """The gray-matter summaries of several placements, one array per quantity. The peak's place is
    left out: it is the position of a maximum, and two elements may tie for it."""
    return {
        "peak": np.array([r["peak_magnE"] for r in rows]),
        "center_mm": np.array([r["center_of_gravity_mm"] for r in rows]),
        "volume": np.array([r["region_volume_m3"] for r in rows]),
        "focality": np.array([list(r["focality_m3"].values()) for r in rows]),
        "distribution": np.array([list(r["distribution"].values()) for r in rows]),
    }


def _results(results):
    out = {"transform": np.array([r.transform for r in results]), "summary": _summaries([r.summary for r in results])}
    for name in FIELDS:
        if getattr(results[0], name) is not None:
            out[name] = [getattr(r, name) for r in results]
    return out


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "network":
        net = state["net"]
        loss, gradients = net.gradients(state["x"], state["t"])
        return {"loss": loss, "gradients": gradients, "prediction": net.predict(state["x"])}
    recovery = case["recovery"]
    if path == "setup":
        ctx = fem.SolverContext(*state["mesh"])
        slots, averaged = ctx.recovery_build(recovery) if recovery != "raw" else (0, 0)
        # The operator, and one cycle of the preconditioner, which goes through the whole hierarchy.
        out = {"normals": ctx.skin_normals(), "operator": ctx.reduced()[2], "cycle": ctx.vcycle(state["rhs"]),
               "slots": slots, "averaged": averaged}
        ctx.free()
        return out
    subject, c = state["subject"], state["coil"]
    if path == "simulate":
        return _results([subject.simulate(c, state["sites"][0], DIDT, magnitude=True, vectors=True, potential=True,
                                          recovery=recovery)])
    if path == "fields":
        return _results(list(subject.iter_simulate(c, state["sites"], DIDT, magnitude=True, vectors=True,
                                                   potential=True, nodal=True, recovery=recovery)))
    if path == "sweep":
        return _results(list(subject.iter_simulate(c, state["sites"], DIDT, recovery=recovery,
                                                   block_k=case["block_k"])))
    if path == "uq":
        r = subject.simulate_conductivity_uq(c, state["sites"][0], state["config"], DIDT, moments=True,
                                             recovery=recovery)
        return {"mean": r.mean_magnE, "std": r.std_magnE, "peak": r.peak_samples, "focality": r.focality_samples,
                "sigma": r.sigma_samples}
    ctx = subject.context
    if path == "sigma":
        out = fem.solve_placements_block(ctx, c.positions_m, c.moments, _triples(state["sites"]), DIDT,
                                         potential=True, recovery=recovery, sigma=state["rows"])
        return {"transform": np.array([r.transform for r in out]), "v": [r.v for r in out],
                "magnE": [r.magnE for r in out], "summary": _summaries([fem.metrics_dict(r.metrics) for r in out])}
    out = fem.solve_sweep(ctx, c.positions_m, c.moments, _triples(state["sites"]), DIDT, case["block_k"],
                          recovery=recovery, warm_start=True)
    return {"transform": out["transforms"], "summary": _summaries([fem.metrics_dict(m) for m in out["metrics"]])}


# --------------------------------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------------------------------


def _sizes(case):
    """Nodes, tetrahedra and operator entries of the case's head (within a few per cent)."""
    n = 3.4e6 / case["spacing"] ** 3
    m = 5.75 * n
    cut = case["refine"] * m
    return n + cut, m + 3 * cut, 15 * n + 9 * cut


def work(case):
    if case["path"] == "network":
        rows, hid, out = case["rows"], case["hidden"], case["outputs"]
        weights = 16 * hid + hid * hid + hid * out
        return {"bytes": 4.0 * (2 * weights + rows * (16 + 2 * out)), "flops": 8.0 * rows * weights}
    n, m, nnz = _sizes(case)
    mesh = 24.0 * n + 20.0 * m
    if case["path"] == "setup":  # the mesh in; gradients, operator (FP64) and a hierarchy of about its size out
        slots = 0.0 if case["recovery"] == "raw" else 16.0 * m + 16.0 * 65 * n * (case["recovery"] == "harmonic")
        return {"bytes": mesh + 52.0 * m + 24.0 * nnz + slots, "flops": 200.0 * m}
    k = {"simulate": 1, "uq": case.get("draws", 1)}.get(case["path"], case.get("placements", 1))
    # Per placement the dipole sum; per column about 15 iterations of a product and a cycle (about seven products).
    dipole = 20.0 * n * case["dipoles"] * (1 if case["path"] == "uq" else k)
    solve = 15.0 * 8.0 * 2.0 * nnz * k
    out = {"simulate": 16.0 * m + 8.0 * n, "fields": 16.0 * m + 20.0 * n, "sigma": 4.0 * m + 8.0 * n}.get(case["path"], 0.0)
    return {"bytes": mesh + 52.0 * m + 12.0 * nnz + out * k + 8.0 * n * k, "flops": dipole + solve}


def tolerance(case):
    if case["path"] == "network":
        return {"rel": 1e-2}  # the predictions run in bf16
    if case["path"] == "setup":
        return {"rel": 1e-5}
    return {"rel": 5e-4}  # solved to a residual of 1e-6, from dipole sums of 32-bit terms


# --------------------------------------------------------------------------------------------------
# The same in 64 bits
# --------------------------------------------------------------------------------------------------


def _spread(v):
    out = np.zeros_like(v)
    for b in range(21):
        out |= ((v >> np.uint64(b)) & np.uint64(1)) << np.uint64(3 * b)
    return out


def _laid_out(mesh):
    """The mesh in the order results are indexed by: nodes along a Morton curve, tetrahedra by lowest node."""
    nodes, tets, tags, skin = mesh
    low = nodes.min(0)
    q = ((nodes - low) / (nodes.max(0) - low) * 2097151.0).astype(np.uint64)
    order = np.argsort(_spread(q[:, 0]) | _spread(q[:, 1]) << np.uint64(1) | _spread(q[:, 2]) << np.uint64(2),
                       kind="stable")
    rank = np.empty(order.shape[0], np.int64)
    rank[order] = np.arange(order.shape[0])
    t = rank[tets]
    first = np.argsort(t.min(1), kind="stable")
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEVICE)  # noqa: E731
    return d(nodes[order]), d(t[first]), d(tags[first].astype(np.int64)), d(rank[skin])


def _unit(v):
    return v / v.norm(dim=-1, keepdim=True).clamp_min(1e-300)


def _normals(x, tri):
    """Area-weighted face normals, spread to the nodes and gathered back twice."""
    face = torch.linalg.cross(x[tri[:, 1]] - x[tri[:, 0]], x[tri[:, 2]] - x[tri[:, 0]])
    for i in range(2):
        node = torch.zeros_like(x).index_add_(0, tri.reshape(-1), face.repeat_interleave(3, 0))
        face = _unit((node if i == 0 else _unit(node))[tri].sum(1))
    return face


def _closest(p, a, b, c):
    """Closest points of triangles (a, b, c) to p: the plane's if inside, else the nearest on an edge."""
    ab, ac, ap = b - a, c - a, p - a
    dot = lambda u, v: (u * v).sum(-1, keepdim=True)  # noqa: E731
    aa, bb, cc, d1, d2 = dot(ab, ab), dot(ab, ac), dot(ac, ac), dot(ab, ap), dot(ac, ap)
    det = aa * cc - bb * bb
    v, w = (cc * d1 - bb * d2) / det, (aa * d2 - bb * d1) / det
    best = a + v * ab + w * ac
    far = torch.where((v >= 0) & (w >= 0) & (v + w <= 1), (best - p).norm(dim=-1, keepdim=True), torch.inf)
    for s, e in ((a, b), (a, c), (b, c)):
        q = s + ((dot(p - s, e - s) / dot(e - s, e - s)).clamp(0, 1)) * (e - s)
        d = (q - p).norm(dim=-1, keepdim=True)
        best, far = torch.where(d < far, q, best), torch.minimum(d, far)
    return best, far[:, 0]


def _frames(x, tri, placements):
    nrm = _normals(x, tri)
    out = []
    for s in placements:
        q, far = _closest(torch.from_numpy(s.center_mm).to(DEVICE), x[tri[:, 0]], x[tri[:, 1]], x[tri[:, 2]])
        i = int(far.argmin())
        proj, z = q[i], -nrm[i]
        y = _unit(torch.from_numpy(s.handle_mm).to(DEVICE) - proj)
        y = _unit(y - z * (y @ z))
        t = torch.eye(4, device=DEVICE, dtype=torch.float64)
        t[:3, 0], t[:3, 1], t[:3, 2], t[:3, 3] = torch.linalg.cross(y, z), y, z, proj + s.distance_mm * nrm[i]
        out.append(t)
    return torch.stack(out)


def _dadt(x, frames, c):
    """d/dt of the vector potential at the nodes, (n, 3, k), by the dipoles' closed form."""
    out = torch.empty(x.shape[0], 3, frames.shape[0], device=DEVICE, dtype=torch.float64)
    for j, t in enumerate(frames):
        s = torch.from_numpy(c.positions_m).to(DEVICE) @ t[:3, :3].T + t[:3, 3] * 1e-3
        mom = torch.from_numpy(c.moments).to(DEVICE) @ t[:3, :3].T
        mxs = torch.linalg.cross(mom, s)
        for lo in range(0, x.shape[0], 32768):
            r = x[lo:lo + 32768] * 1e-3
            w = ((r[:, None, :] - s[None]) ** 2).sum(-1) ** -1.5
            out[lo:lo + 32768, :, j] = DIDT * 1e-7 * (torch.linalg.cross(w @ mom, r) - w @ mxs)
    return out


def _solve(apply, diag, b):
    """Jacobi-preconditioned CG on every column, to 1e-11."""
    x, r = torch.zeros_like(b), b.clone()
    z = r / diag
    p, rz, goal = z.clone(), (r * z).sum(0), 1e-11 * b.norm(dim=0)
    for i in range(6000):
        ap = apply(p)
        a = torch.where(rz > 0, rz / (p * ap).sum(0), 0.0)
        x += a * p
        r -= a * ap
        if i % 25 == 24 and bool((r.norm(dim=0) <= goal).all()):
            break
        z = r / diag
        new = (r * z).sum(0)
        p = z + torch.where(rz > 0, new / rz, 0.0) * p
        rz = new
    return x


def _quantiles(v, w, qs):
    order = np.argsort(v, kind="stable")
    v, w = v[order], w[order]
    cw = np.cumsum(w)
    return np.interp(qs, (cw - 0.5 * w) / cw[-1], v)


def _summary(mag, vol, bary):
    p = _quantiles(mag, vol, [float(np.float32(q)) for q in (0.5, 0.95, 0.99, 0.999)])
    mean = (vol * mag).sum() / vol.sum()
    std = math.sqrt((vol * (mag - mean) ** 2).sum() / vol.sum())
    return {"peak_magnE": mag.max(), "center_of_gravity_mm": ((vol * mag)[:, None] * bary).sum(0) / (vol * mag).sum(),
            "region_volume_m3": vol.sum(),
            "focality_m3": {"0.5": vol[mag >= 0.5 * p[3]].sum(), "0.75": vol[mag >= 0.75 * p[3]].sum()},
            "distribution": dict(zip(("mean", "std", "p50", "p95", "p99", "p99.9"), (mean, std, *p)))}


def _network(case, seed):
    s = prepare(case, seed)
    x = torch.from_numpy(((s["x"] - s["net"].mean) / s["net"].scale)).double()
    p = torch.from_numpy(s["net"].params()).double().requires_grad_()
    hid, out, n_in = case["hidden"], case["outputs"], learned.N_INPUTS
    at, y = 0, x
    for i, (a, b) in enumerate(((n_in, hid), (hid, hid), (hid, out))):
        y = y @ p[at:at + a * b].view(a, b) + p[at + a * b:at + a * b + b]
        at += a * b + b
        y = torch.nn.functional.gelu(y) if i < 2 else y
    loss = ((y - torch.from_numpy(s["t"]).double()) ** 2).mean()
    loss.backward()
    return {"loss": float(loss), "gradients": p.grad, "prediction": (y * torch.from_numpy(s["net"].out_scale)).detach()}


def exact(case, seed):
    """Frames, potential and, for the raw field, E, |E| and the summaries. A recovered field has none
    here (which polynomial a patch takes is decided by thresholds on its rounding), nor has a case
    that would take too long."""
    path = case["path"]
    if path == "network":
        return _network(case, seed)
    if path == "uq":
        return None
    x, tet, tags, tri = _laid_out(head(case["spacing"], case["refine"], seed))
    n, m, k = x.shape[0], tet.shape[0], case.get("placements", 1)
    raw = case["recovery"] == "raw"
    if path in ("sweep", "warm") and not raw or n * k * case.get("dipoles", 0) > 4e10 or n * k > 2.5e7:
        return None
    e = (x[tet[:, 1:]] - x[tet[:, :1]]) * 1e-3
    vol = torch.linalg.det(e) / 6.0
    g = torch.linalg.inv(e).transpose(1, 2)
    g = torch.cat([-g.sum(1, keepdim=True), g], 1)  # (m, 4, 3)
    vol = vol.abs()
    table = torch.zeros(k, 6, device=DEVICE, dtype=torch.float64)
    table[:, 1:] = torch.tensor(list(SIGMA.values()), device=DEVICE)
    if path == "sigma":
        table[:, 1:] = torch.from_numpy(conductivities(k, seed)).to(DEVICE)
    vs = vol[:, None] * table.T[tags]  # (m, k)
    ground = int(x[:, 2].argmin())
    gg = torch.einsum("mid,mjd->mij", g, g)
    if path != "sigma":
        at = torch.stack([tet[:, :, None].expand(-1, 4, 4).reshape(-1), tet[:, None, :].expand(-1, 4, 4).reshape(-1)])
        a = torch.sparse_coo_tensor(at, (gg * vs[:, :1, None]).reshape(-1), (n, n)).coalesce()
    if path == "setup":
        keep = (a.indices() != ground).all(0)
        return {"normals": _normals(x, tri), "operator": a.values()[keep], "cycle": None}
    c, placements = coil(case["coil"], case["dipoles"], seed), sites(k, seed)
    frames = _frames(x, tri, placements)
    da = _dadt(x, frames, c)
    de = da[tet].mean(1)  # (m, 3, k)
    rhs = -torch.einsum("mid,mdk->mik", g, de) * vs[:, None, :]
    b = torch.zeros(n, k, device=DEVICE, dtype=torch.float64).index_add_(0, tet.reshape(-1), rhs.reshape(-1, k))
    if path == "sigma":

        def product(p):
            q = torch.einsum("mij,mjk->mik", gg, p[tet]) * vs[:, None, :]
            return torch.zeros_like(p).index_add_(0, tet.reshape(-1), q.reshape(-1, k))
    else:
        a = a.to_sparse_csr()

        def product(p):
            return a @ p

    def grounded(p):
        q = product(p)
        q[ground] = 0.0
        return q

    diag = torch.zeros_like(b).index_add_(0, tet.reshape(-1), (gg.diagonal(dim1=1, dim2=2)[..., None] * vs[:, None, :]).reshape(-1, k))
    b[ground] = 0.0
    v = _solve(grounded, diag, b)
    out = {"transform": frames, "summary": None}
    if path in ("simulate", "fields", "sigma"):
        out["v"] = list(v.T)
    if not raw:
        return out
    rows, field, size = [], [], []
    gray = (tags == GRAY).nonzero()[:, 0]
    bary = x[tet].mean(1)[gray].cpu().numpy()
    for j in range(k):
        ej = -torch.einsum("mid,mi->md", g, v[tet, j]) - de[:, :, j]
        mag = ej.norm(dim=1)
        rows.append(_summary(mag[gray].cpu().numpy(), vol[gray].cpu().numpy(), bary))
        field.append(ej)
        size.append(mag)
    out["summary"] = _summaries(rows)
    if path in ("simulate", "sigma"):
        out["magnE"] = size
    if path == "simulate":
        out["E"] = field
    return out
