"""Workloads of the geometry-query path, as a user's program runs them.

Each case is a dict of plain values; `prepare` builds what such a program
holds before the call (context, trees, device inputs made from a seed), `run`
is one pass through the public calls of `xdg_amd.capi.Context`, `exact` the
same answers from plain float64 torch where a direct formula exists.

Geometry is the repository's own: icospheres, three nested spheres in a cube,
a lattice of spheres in a box, a perturbed sphere, and the unit cube split
into jittered Kuhn tetrahedra.
"""
import functools
import math

import numpy as np
import torch

from xdg_amd import capi
from xdg_amd import geometry as G

INFTY = float(np.finfo(np.float64).max)
RADII = (5.0, 10.0, 15.0)  # nested spheres
HALF = 20.0                # half edge of the cube around them
PITCH = 2.0                # sphere lattice
PLUCKER_TOL = 20.0 * 2.220446049250313e-16  # containment tolerance of a tetrahedron


def listed():
    return [
        # a Monte Carlo code that traces its particles in small banks: launch latency counts
        {"name": "ray_fire_1k", "kind": "ray_fire", "geom": "sphere", "subdiv": 5, "n": 1000, "prec": "mixed",
         "orient": "exiting", "excl": 2, "tmax": False},
        # one volume, default precision: rays of a track-length scan from inside a sphere
        {"name": "ray_fire_sphere_1m_fp64", "kind": "ray_fire", "geom": "sphere", "subdiv": 5, "n": 1_000_000,
         "prec": "plain", "orient": "exiting", "excl": 0, "tmax": False},
        # the headline: every ray in the volume that holds its origin
        {"name": "ray_fire_nested_10m_mixed", "kind": "ray_fire", "geom": "nested", "subdiv": 6, "n": 10_000_000,
         "prec": "mixed", "orient": "exiting", "excl": 0, "tmax": False},
        # locating source particles before a transport run
        {"name": "find_volume_4m_mixed", "kind": "find_volume", "subdiv": 6, "n": 4_000_000, "prec": "mixed"},
        # checking sites of a sampled source against one cell (rejection sampling), default precision
        {"name": "point_in_volume_1m_fp64", "kind": "piv", "subdiv": 6, "n": 1_000_003, "prec": "plain"},
        # distance to the nearest boundary: safety distances of a particle bank
        {"name": "closest_100k", "kind": "closest", "subdiv": 5, "n": 100_003},
        # mesh tally start: the element of each collision site
        {"name": "find_element_1m", "kind": "find_element", "mesh": 64, "n": 1_000_000},
        # track-length tally of a large batch on a large mesh
        {"name": "segments_4m_mesh64", "kind": "segments", "mesh": 64, "n": 4_000_000, "tally": True,
         "short": False},
        # track-length tally of an ordinary batch: flights of about a tenth of the mesh, on a smaller mesh
        {"name": "segments_200k_mesh32_short", "kind": "segments", "mesh": 32, "n": 200_001, "tally": True,
         "short": True},
        # particles walking the mesh element by element with collisions
        {"name": "mesh_walk_1m_mesh64", "kind": "mesh_walk", "mesh": 64, "n": 1_048_576, "mfp": 0.1},
        # whole particle histories in a lattice of 512 spheres
        {"name": "transport_1m_lattice8", "kind": "transport", "lattice": 8, "subdiv": 4, "n": 1_048_576,
         "mfp": 2.0, "p_absorb": 0.3, "prec": "mixed"},
        # gradients of 4 M ray distances for a surface fit
        {"name": "adjoint_4m", "kind": "adjoint", "subdiv": 6, "n": 4_000_000, "miss": 0.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ray_fire", "ray_fire", "find_volume", "piv", "closest", "find_element", "segments",
                       "segments", "mesh_walk", "transport", "adjoint"])
    if kind == "ray_fire":
        geom = rng.choice(["sphere", "nested"])
        return {"kind": kind, "geom": geom, "subdiv": rng.randint(3, 6), "n": _log(rng, 64, 10_000_000),
                "prec": rng.choice(["mixed", "plain"]), "orient": rng.choice(["exiting", "exiting", "any"]),
                "excl": rng.choice([0, 0, 1, 4]), "tmax": rng.choice([False, False, True])}
    if kind in ("find_volume", "piv"):
        return {"kind": kind, "subdiv": rng.randint(4, 6), "n": _log(rng, 1000, 4_000_000),
                "prec": rng.choice(["mixed", "plain"])}
    if kind == "closest":
        return {"kind": kind, "subdiv": rng.randint(3, 6), "n": _log(rng, 1000, 400_000)}
    if kind == "find_element":
        return {"kind": kind, "mesh": rng.choice([9, 16, 23, 32, 47, 64]), "n": _log(rng, 1000, 4_000_000)}
    if kind == "segments":
        return {"kind": kind, "mesh": rng.choice([9, 16, 23, 32, 47, 64]), "n": _log(rng, 1000, 3_900_000),
                "tally": rng.choice([True, True, True, False]), "short": rng.choice([True, False])}
    if kind == "mesh_walk":
        return {"kind": kind, "mesh": rng.choice([9, 16, 23, 32, 47, 64]), "n": _log(rng, 10_000, 1_000_000),
                "mfp": rng.choice([0.1, 0.3, 1.0])}
    if kind == "transport":
        return {"kind": kind, "lattice": rng.randint(2, 7), "subdiv": rng.randint(3, 4),
                "n": _log(rng, 10_000, 1_000_000), "mfp": rng.choice([1.0, 2.0, 4.0]),
                "p_absorb": rng.choice([0.2, 0.3, 0.5]), "prec": rng.choice(["mixed", "plain"])}
    return {"kind": "adjoint", "subdiv": rng.randint(4, 6), "n": _log(rng, 1000, 3_900_000),
            "miss": rng.choice([0.0, 0.05])}


# ---- geometry, built once per process (it does not depend on the seed) -----

@functools.lru_cache(maxsize=None)
def _model(geom, size, subdiv):
    """Surface model and the tree arrays of each of its volumes."""
    if geom == "sphere":
        m = G.single_sphere(subdiv, 10.0)
    elif geom == "nested":
        m = G.nested_spheres(subdiv, RADII, HALF)
    elif geom == "lattice":
        m = G.sphere_lattice(size, subdiv, 0.8, PITCH)
    else:
        m = G.perturbed_sphere(subdiv, 10.0, 0.05)
    return m, {v: m.tree_arrays(v) + (m.bump(v),) for v in m.volumes}


@functools.lru_cache(maxsize=None)
def _mesh(n):
    mesh = G.kuhn_cube(n, 0.2, seed=4)
    bm = mesh.boundary_model()
    return mesh, bm.tree_arrays(bm.ipc) + (bm.bump(bm.ipc),)


def _surface(ctx, arrays):
    v9, faces, surfs, flips, bump = arrays
    return ctx.build_surface_tree(v9.reshape(-1, 3), np.arange(3 * v9.shape[0], dtype=np.int32).reshape(-1, 3),
                                  faces, surfs, flips, bump)


def _mesh_trees(ctx, n):
    """The mesh's element tree with its implicit-complement boundary attached."""
    mesh, arrays = _mesh(n)
    et = ctx.build_element_tree(mesh.verts, mesh.tets, mesh.adj, mesh.face_order)
    ctx.attach_boundary(et, _surface(ctx, arrays), mesh.bface_elem)
    return et, mesh


# ---- inputs -----------------------------------------------------------------

def _dev():
    return torch.device("cuda", 0) if torch.cuda.is_available() else torch.device("cpu")


def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(1_000_003 * (seed % 1_000_003) + 17)
    return g


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device=_dev(), dtype=torch.float64)


def _iso(g, n):
    d = torch.randn(n, 3, generator=g, device=_dev(), dtype=torch.float64)
    return (d / d.norm(dim=1, keepdim=True)).contiguous()


def _ball(g, n, radius):
    return (_iso(g, n) * (radius * _uniform(g, n, 1) ** (1.0 / 3.0))).contiguous()


def _inputs(case, seed):
    """The device inputs of a case: a dict of tensors made from the seed alone."""
    g, n, kind = _gen(seed), case["n"], case["kind"]
    if kind == "ray_fire":
        x = {"org": _ball(g, n, 9.0) if case["geom"] == "sphere" else (32.0 * _uniform(g, n, 3) - 16.0).contiguous(),
             "dirs": _iso(g, n)}
        if case["excl"]:  # the last faces hit, a few of them still near the ray
            nf = _model(case["geom"], 0, case["subdiv"])[0].tris.shape[0]
            x["excl"] = torch.randint(0, nf, (n, case["excl"]), generator=g, device=_dev(),
                                      dtype=torch.int64).to(torch.int32)
        if case["tmax"]:  # flight lengths
            x["tmax"] = -6.0 * torch.log(1.0 - _uniform(g, n))
        return x
    if kind in ("find_volume", "piv"):
        return {"pts": (32.0 * _uniform(g, n, 3) - 16.0).contiguous(), "dirs": _iso(g, n)}
    if kind == "closest":
        return {"pts": _ball(g, n, 14.0)}
    if kind == "find_element":
        return {"pts": _uniform(g, n, 3)}
    if kind == "segments":
        p0 = _uniform(g, n, 3)
        if not case["short"]:
            return {"p0": p0, "p1": _uniform(g, n, 3)}
        length = -0.1 * torch.log(1.0 - _uniform(g, n, 1))
        return {"p0": p0, "p1": (p0 + length * _iso(g, n)).clamp(0.0, 1.0).contiguous()}
    if kind == "adjoint":
        m = _model("perturbed", 0, case["subdiv"])[0]
        verts = torch.from_numpy(m.verts).to(_dev())
        tris = torch.from_numpy(m.tris).to(_dev())
        # hits spread over the surface, seen from origins inside it
        face = torch.randint(0, tris.shape[0], (n,), generator=g, device=_dev(), dtype=torch.int64)
        b = _uniform(g, n, 2)
        b = torch.where((b.sum(1) > 1.0).unsqueeze(1), 1.0 - b, b)
        v = verts[tris[face].long()]
        hit = v[:, 0] + b[:, :1] * (v[:, 1] - v[:, 0]) + b[:, 1:] * (v[:, 2] - v[:, 0])
        org = _ball(g, n, 9.0)
        ray = hit - org
        t = ray.norm(dim=1)
        dirs = (ray / t.unsqueeze(1)).contiguous()
        w = torch.randn(n, generator=g, device=_dev(), dtype=torch.float64)
        lost = _uniform(g, n) < case["miss"]
        t = torch.where(lost, torch.full_like(t, INFTY), t)
        face = torch.where(lost, torch.full_like(face, -1), face).to(torch.int32)
        return {"org": org, "dirs": dirs, "t": t, "face": face, "w": w, "verts": verts, "tris": tris}
    return {}


def _prec(case):
    return capi.MIXED if case["prec"] == "mixed" else capi.PLAIN


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    dev = _dev()
    ctx = capi.Context(0)
    s = {"case": case, "ctx": ctx}
    s.update(_inputs(case, seed))
    if kind == "ray_fire":
        m, arrays = _model(case["geom"], 0, case["subdiv"])
        s["tree"] = _surface(ctx, arrays[m.volumes[0]])
        if case["geom"] == "nested":
            vols = list(m.volumes)
            trees = [s["tree"]] + [_surface(ctx, arrays[v]) for v in vols[1:]]
            vol = ctx.find_volume(trees, vols, m.ipc, s["org"], s["dirs"], precision=capi.MIXED)
            lut = torch.zeros(max(vols) + 1, dtype=torch.int32, device=dev)
            for v, t in zip(vols, trees):
                lut[v] = t
            s["tree_per_ray"] = lut[vol.long()].contiguous()
        s["out"] = (torch.empty(n, dtype=torch.float64, device=dev), torch.empty(n, dtype=torch.int32, device=dev),
                    torch.empty(n, dtype=torch.int32, device=dev))
    elif kind in ("find_volume", "piv"):
        m, arrays = _model("nested", 0, case["subdiv"])
        if kind == "piv":
            s["tree"] = _surface(ctx, arrays[3])
        else:
            s["vols"] = list(m.volumes)
            s["trees"] = [_surface(ctx, arrays[v]) for v in s["vols"]]
            s["ipc"] = m.ipc
            s["out"] = torch.empty(n, dtype=torch.int32, device=dev)
    elif kind == "closest":
        m, arrays = _model("sphere", 0, case["subdiv"])
        s["tree"] = _surface(ctx, arrays[1])
    elif kind in ("find_element", "segments", "mesh_walk"):
        s["tree"], mesh = _mesh_trees(ctx, case["mesh"])
        s["seed"] = seed % (1 << 31)
        if kind == "mesh_walk" or (kind == "segments" and case["tally"]):
            s["tally"] = torch.zeros(mesh.tets.shape[0], dtype=torch.int64, device=dev)
        if kind == "segments":
            s["out"] = (torch.empty(n, dtype=torch.int32, device=dev), torch.empty(n, dtype=torch.int64, device=dev))
    elif kind == "transport":
        m, arrays = _model("lattice", case["lattice"], case["subdiv"])
        vols = [v for v in m.volumes if v != m.ipc]
        trees = [_surface(ctx, arrays[v]) for v in vols]
        length = PITCH * case["lattice"]
        s["handle"] = ctx.transport_create(vols, trees, m.ipc, m.senses, seed % (1 << 31), 3, [0.0] * 3, [length] * 3,
                                           case["mfp"], case["p_absorb"])
        # the shape the autotuner settles on for this problem
        ctx.transport_set_config(s["handle"], block=256, lds_stack=16, chunk=1, refill=32)
        s["nvol"] = len(vols)
        s["out"] = ctx.transport_outputs(len(vols), n)
    elif kind == "adjoint":
        s["gv"] = torch.empty_like(s["verts"])
        s["go"] = torch.empty_like(s["org"])
        s["gd"] = torch.empty_like(s["dirs"])
    torch.cuda.synchronize()
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "ray_fire":
        return ctx.ray_fire(s["tree"], s["org"], s["dirs"], tmax=s.get("tmax"),
                            orientation=capi.EXITING if case["orient"] == "exiting" else capi.ANY,
                            excl=s.get("excl"), precision=_prec(case), tree_per_ray=s.get("tree_per_ray"),
                            out=s["out"])
    if kind == "find_volume":
        return ctx.find_volume(s["trees"], s["vols"], s["ipc"], s["pts"], s["dirs"], precision=_prec(case),
                               out=s["out"])
    if kind == "piv":
        return ctx.point_in_volume(s["tree"], s["pts"], s["dirs"], precision=_prec(case))
    if kind == "closest":
        return ctx.closest(s["tree"], s["pts"])
    if kind == "find_element":
        return ctx.find_element(s["tree"], s["pts"])
    if kind == "segments":
        if not case["tally"]:
            return ctx.tally_segments(s["tree"], s["p0"], s["p1"], out=s["out"])
        s["tally"].zero_()
        count, sequence = ctx.tally_segments(s["tree"], s["p0"], s["p1"], tally=s["tally"], out=s["out"])
        return count, sequence, s["tally"]
    if kind == "mesh_walk":
        s["tally"].zero_()
        out = ctx.mesh_walk(s["tree"], 0, case["n"], s["seed"], 3, [0.0] * 3, [1.0] * 3, case["mfp"],
                            tally=s["tally"])
        return out + (s["tally"],)
    if kind == "transport":
        return ctx.transport_run(s["handle"], 0, case["n"], s["nvol"], precision=_prec(case), out=s["out"])
    s["gv"].zero_()
    ctx.ray_distance_adjoint(s["org"], s["dirs"], s["t"], s["face"], s["w"], s["verts"], s["tris"], s["gv"],
                             s["go"], s["gd"])
    return {"verts": s["gv"], "org": s["go"], "dirs": s["gd"]}


# ---- what a pass cannot do without ------------------------------------------

def _tri_bytes(tris):
    return 12 * tris + 24 * (tris // 2 + 2)  # connectivity and a closed surface's vertices


def work(case):
    kind, n = case["kind"], case["n"]
    if kind in ("ray_fire", "find_volume", "piv", "closest"):
        tris = 20 * 4 ** case["subdiv"]
        shells = 3 if kind == "find_volume" or case.get("geom") == "nested" else (2 if kind == "piv" else 1)
        mesh = _tri_bytes(shells * tris)
        per = {"ray_fire": 48 + 16, "find_volume": 48 + 4, "piv": 48 + 1, "closest": 24 + 12}[kind]
        per += 4 * case.get("excl", 0) + (8 if case.get("tmax") else 0) + (4 if case.get("geom") == "nested" else 0)
        # a descent of the hierarchy (one box of about 20 operations per
        # level) and one triangle of about 100
        flops = n * (20.0 * math.log2(tris) + 100.0) * (2.0 if kind == "find_volume" else 1.0)
        return {"bytes": float(n * per + mesh), "flops": flops}
    if kind in ("find_element", "segments", "mesh_walk"):
        tets = 6 * case["mesh"] ** 3
        mesh = 32 * tets + 24 * (case["mesh"] + 1) ** 3
        if kind == "find_element":
            return {"bytes": float(28 * n + mesh), "flops": n * (6.0 * math.log2(tets) + 60.0)}
        tally = 8 * tets if case.get("tally", True) else 0
        # elements a flight crosses: 3.73 per cell width of its length; about
        # 200 operations each (six edge values and the exit distance)
        if kind == "segments":
            steps = n * (1.0 + 3.73 * case["mesh"] * (0.095 if case["short"] else 0.6617))
            return {"bytes": float(n * (48 + 12) + mesh + tally), "flops": 200.0 * steps}
        track = {0.1: 1.05, 0.3: 0.66, 1.0: 0.50}[case["mfp"]]
        steps = n * (1.0 + 3.73 * case["mesh"] * track)
        return {"bytes": float(n * 21 + mesh + tally), "flops": 250.0 * steps}
    if kind == "transport":
        tris = case["lattice"] ** 3 * 20 * 4 ** case["subdiv"]
        events = 1.0 / case["p_absorb"] + 1.0
        return {"bytes": float(n * 13 + _tri_bytes(tris)),
                "flops": n * events * (20.0 * math.log2(tris) + 300.0)}
    tris = 20 * 4 ** case["subdiv"]
    return {"bytes": float(n * (48 + 8 + 4 + 8 + 48) + _tri_bytes(tris) + 24 * (tris // 2 + 2)),
            "flops": 90.0 * n}


def tolerance(case):
    # Every query returns the bits of one fixed sequence of float64 operations
    # (distances, identifiers, hashes, fixed-point tallies); only the
    # vertex gradients are float64 sums in no fixed order (two orders differ
    # by 1e-16 to 9e-16 of the result).
    if case["kind"] == "adjoint":
        return {"rel": 4e-15}
    return "exact"


# ---- the same answers in plain float64 ---------------------------------------

def _planes(verts, tris):
    """Outward unit normals and offsets of a convex polyhedron's faces."""
    v = torch.from_numpy(verts).to(_dev())[torch.from_numpy(tris).to(_dev()).long()]
    nrm = torch.linalg.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    nrm = nrm / nrm.norm(dim=1, keepdim=True)
    return nrm, (nrm * v[:, 0]).sum(1)


def _inside_sphere(pts, subdiv, radius):
    """Is each point inside the icosphere (the convex hull of its vertices)?
    Only points between its inscribed and circumscribed spheres need faces."""
    v, f = G.icosphere(subdiv, radius)
    nrm, off = _planes(v, f)
    r = pts.norm(dim=1)
    inside = r < off.min()
    near = torch.nonzero((r >= off.min()) & (r <= radius)).squeeze(1)
    for c in near.split(max(1, (1 << 27) // nrm.shape[0])):
        inside[c] = (pts[c] @ nrm.t() <= off).all(dim=1)
    return inside


def _closest_distance(p, v):
    """Distance from points p (n, 3) to triangles v (m, 3, 3): (n, m), by the
    regions of the triangle's plane (vertices, edges, face)."""
    a, e0, e1 = v[:, 0], v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    e2 = e1 - e0
    best = None
    for q0, e in ((a, e0), (a, e1), (v[:, 1], e2)):
        # |p - q0|^2 - 2 s (p - q0).e + s^2 |e|^2, differences formed first
        d = [p[:, k:k + 1] - q0[:, k] for k in range(3)]
        s = ((d[0] * e[:, 0] + d[1] * e[:, 1] + d[2] * e[:, 2]) / (e * e).sum(1)).clamp(0.0, 1.0)
        r2 = sum((d[k] - s * e[:, k]) ** 2 for k in range(3))
        best = r2 if best is None else torch.minimum(best, r2)
    nrm = torch.linalg.cross(e0, e1)
    nn = (nrm * nrm).sum(1)
    d = [p[:, k:k + 1] - a[:, k] for k in range(3)]
    u1, u0 = torch.linalg.cross(e1, nrm) / nn.unsqueeze(1), torch.linalg.cross(nrm, e0) / nn.unsqueeze(1)
    bu = d[0] * u1[:, 0] + d[1] * u1[:, 1] + d[2] * u1[:, 2]
    bv = d[0] * u0[:, 0] + d[1] * u0[:, 1] + d[2] * u0[:, 2]
    h2 = (d[0] * nrm[:, 0] + d[1] * nrm[:, 1] + d[2] * nrm[:, 2]) ** 2 / nn
    return torch.where((bu >= 0) & (bv >= 0) & (bu + bv <= 1), h2, best).sqrt()


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "ray_fire" and case["geom"] == "sphere" and not case["tmax"]:
        m = _model("sphere", 0, case["subdiv"])[0]
        if n * m.tris.shape[0] > 1 << 35:
            return None
        x = _inputs(case, seed)
        nrm, off = _planes(m.verts, m.tris)
        t = torch.empty(n, dtype=torch.float64, device=_dev())
        for c in torch.arange(n, device=_dev()).split(max(1, (1 << 27) // nrm.shape[0])):
            den = x["dirs"][c] @ nrm.t()
            tc = torch.where(den > 0, (off - x["org"][c] @ nrm.t()) / den, float("inf"))
            t[c], first = tc.min(dim=1)
            if case["excl"]:  # an excluded first face lets the ray out of the convex body
                t[c] = torch.where((x["excl"][c].long() == first.unsqueeze(1)).any(dim=1), INFTY, t[c])
        return t, None, None
    if kind in ("find_volume", "piv"):
        x = _inputs(case, seed)
        inside = [_inside_sphere(x["pts"], case["subdiv"], r) for r in RADII]
        if kind == "piv":
            return (inside[2] & ~inside[1]).to(torch.uint8)
        return (4 - inside[0].int() - inside[1].int() - inside[2].int()).to(torch.int32)
    if kind == "closest":
        m = _model("sphere", 0, case["subdiv"])[0]
        if n * m.tris.shape[0] > 1 << 32:
            return None
        p = _inputs(case, seed)["pts"]
        v = torch.from_numpy(m.verts[m.tris]).to(_dev())
        step = max(1, (1 << 25) // v.shape[0])
        return torch.cat([_closest_distance(c, v).min(dim=1).values for c in p.split(step)]), None
    if kind == "find_element":
        mesh = _mesh(case["mesh"])[0]
        k = case["mesh"]
        tets = torch.from_numpy(mesh.verts[mesh.tets]).to(_dev())
        lam = torch.linalg.inv((tets[:, 1:] - tets[:, :1]).transpose(1, 2).contiguous())
        out = []
        for p in _inputs(case, seed)["pts"].split(1 << 18):
            best = torch.full((p.shape[0],), tets.shape[0], dtype=torch.int64, device=_dev())
            cell = (p * k).long().clamp(0, k - 1)
            for dx in (-1, 0, 1):  # a jittered cell reaches into its neighbours only
                for dy in (-1, 0, 1):
                    for dz in (-1, 0, 1):
                        c = cell + torch.tensor([dx, dy, dz], device=_dev())
                        ok = ((c >= 0) & (c < k)).all(dim=1)
                        c = c.clamp(0, k - 1)
                        first = 6 * (c[:, 0] + k * (c[:, 1] + k * c[:, 2]))
                        for j in range(6):
                            l3 = ((p - tets[first + j, 0]).unsqueeze(1) * lam[first + j]).sum(2)
                            l0 = 1.0 - l3.sum(1)
                            tol = PLUCKER_TOL
                            hit = ok & (l3 >= -tol).all(dim=1) & (l0 >= -tol) & (l0 <= 1 + tol) & (l3 <= 1 + tol).all(1)
                            best = torch.where(hit, torch.minimum(best, first + j), best)
            out.append(torch.where(best < tets.shape[0], best, -1).to(torch.int32))
        return torch.cat(out)
    if kind == "adjoint":
        x = _inputs(case, seed)
        ok = x["face"] >= 0
        f = x["face"].clamp(min=0).long()
        i = x["tris"][f].long()
        v0, v1, v2 = x["verts"][i[:, 0]], x["verts"][i[:, 1]], x["verts"][i[:, 2]]
        e1, e2 = v1 - v0, v2 - v0
        nn = torch.linalg.cross(e1, e2)
        t = torch.where(ok, x["t"], 0.0).unsqueeze(1)
        w = torch.where(ok, x["w"] / (nn * x["dirs"]).sum(1), 0.0).unsqueeze(1)
        q = v0 - (x["org"] + t * x["dirs"])
        a1, a2 = torch.linalg.cross(e2, q), torch.linalg.cross(q, e1)
        gv = torch.zeros_like(x["verts"])
        for idx, term in ((i[:, 0], nn - a1 - a2), (i[:, 1], a1), (i[:, 2], a2)):
            gv.index_add_(0, idx, w * term)
        return {"verts": gv, "org": -w * nn, "dirs": -w * t * nn}
    return None
