"""Performance cases: the work a program that uses this package has it do.

A case is a dict of plain values. Kinds, each through its public entry points:

  sdf     quest.SignedDistance.computeDistances on new query points
  grad    the same with the adjoint to queries and vertices
  fit     one iteration of a shape fit: updateVertices (BVH rebuild), forward,
          adjoint to the vertices, vertex step
  quads   computeDistances over quad cells
  find    spin.BVH searches (points, boxes or rays; 2-D or 3-D; double or
          float), with the BVH built in the same pass or held by the program
  hex     quest.findCandidatesBVH between two hexahedral meshes
  isect   quest.findTriMeshIntersectionsBVH

Meshes are closed surfaces: icospheres (level L has 20 * 4^L triangles), tori
and cube spheres, with a radius that varies smoothly and, where `noise` is
set, from vertex to vertex. Queries fill a box around the mesh ("box"), lie
near the surface ("near"), or are half of each ("mixed"). All inputs are made
on the GPU from the seed.
"""
import functools
import math

import torch

from axom_amd import autograd, quest, spin, synth

DEV = "cuda"
F64, F32, I32 = torch.float64, torch.float32, torch.int32


def listed():
    return [
        # the smallest call: a physics code asks for the distance and normal of
        # a thousand points against a small mesh (launches and latency count)
        {"name": "sdf_1k_l4", "kind": "sdf", "mesh": "ico", "size": 4, "noise": 1e-3,
         "wave": 0.0, "queries": "box", "nq": 1000, "fp": "fp64", "normals": True, "soa": False},
        # an ordinary batch of an odd size on separate coordinate arrays
        {"name": "sdf_30k_l5_soa", "kind": "sdf", "mesh": "ico", "size": 5, "noise": 1e-3,
         "wave": 0.05, "queries": "mixed", "nq": 30011, "fp": "fp64", "normals": True,
         "soa": True},
        # the benchmark's step: a grid's worth of points around an 81,920-triangle
        # surface, distance, closest point and element, then the adjoint
        {"name": "grad_4m_l6", "kind": "grad", "mesh": "ico", "size": 6, "noise": 1e-3,
         "wave": 0.0, "queries": "box", "nq": 4_000_000, "fp": "fp64", "autograd": False},
        # training through the autograd function: near-surface samples of a
        # wavy 327,680-triangle surface
        {"name": "grad_1m_l7_near", "kind": "grad", "mesh": "ico", "size": 7, "noise": 0.0,
         "wave": 0.1, "queries": "near", "nq": 1_000_000, "fp": "fp64", "autograd": True},
        # a large mesh with the FP32-traversal form: 2,097,152 triangles, half the
        # points near the surface, a ragged count
        {"name": "sdf_4m_torus2m_fp32", "kind": "sdf", "mesh": "torus", "size": 1024,
         "noise": 0.0, "wave": 0.02, "queries": "mixed", "nq": 4_000_037, "fp": "fp32",
         "normals": False, "soa": False},
        # one iteration of the shape-fitting loop on 1,310,720 triangles: the
        # largest work of a single step
        {"name": "fit_8m_l8_fp32", "kind": "fit", "size": 8, "wave": 2e-3, "nq": 8_000_000,
         "fp": "fp32"},
        # a hexahedral code's boundary surface: quad cells
        {"name": "quads_1m_98k", "kind": "quads", "size": 128, "wave": 0.02,
         "nq": 1_000_003, "normals": True},
        # rebuild over moving boxes, then points: a contact or particle step
        {"name": "build_points_100k_1m", "kind": "find", "what": "points", "dims": 3,
         "float": "f64", "fp": "fp64", "nbox": 100_000, "nq": 1_000_000, "build": True},
        # 2-D points into held overlapping boxes (tens of candidates a point)
        {"name": "points2d_100k_1m", "kind": "find", "what": "points", "dims": 2,
         "float": "f64", "fp": "fp64", "nbox": 100_000, "nq": 1_000_000, "build": False},
        # rays against held boxes: a long tail of long rays
        {"name": "rays_100k_100k", "kind": "find", "what": "rays", "dims": 3, "float": "f64",
         "fp": "fp64", "nbox": 100_000, "nq": 100_000, "build": False},
        # candidate pairs between two overlapping hexahedral meshes (remap)
        {"name": "hex_64_60", "kind": "hex", "n": 64, "m": 60},
        # mesh checking: self-intersections of two crossing noisy surfaces
        {"name": "isect_2m6", "kind": "isect", "size": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    kind = rng.choice(["sdf", "sdf", "grad", "grad", "fit", "quads", "find", "find", "find",
                       "hex", "isect"])
    fp = rng.choice(["fp64", "fp32"])
    if kind in ("sdf", "grad"):
        mesh = rng.choice(["ico", "ico", "torus"])
        size = rng.randint(3, 7) if mesh == "ico" else _log_int(rng, 24, 1024)
        c = {"kind": kind, "mesh": mesh, "size": size,
             "noise": rng.choice([0.0, 1e-3]) if mesh == "ico" and size <= 6 else 0.0,
             "wave": rng.choice([0.0, 0.02, 0.1]) if mesh == "ico" else 0.02,
             "queries": rng.choice(["box", "near", "mixed"]), "nq": _log_int(rng, 500, 4_000_000),
             "fp": fp}
        if kind == "sdf":
            return {**c, "normals": rng.random() < 0.5, "soa": rng.random() < 0.5}
        return {**c, "autograd": rng.random() < 0.5}
    if kind == "fit":
        return {"kind": kind, "size": rng.randint(4, 7), "wave": rng.choice([2e-3, 0.05]),
                "nq": _log_int(rng, 20_000, 4_000_000), "fp": fp}
    if kind == "quads":
        return {"kind": kind, "size": _log_int(rng, 8, 160), "wave": rng.choice([0.0, 0.02]),
                "nq": _log_int(rng, 1000, 2_000_000), "normals": rng.random() < 0.5}
    if kind == "find":
        what, dims = rng.choice(["points", "boxes", "rays"]), rng.choice([2, 3, 3])
        most = (20_000 if dims == 2 else 100_000) if what == "rays" else \
            (100_000 if dims == 2 else 500_000)
        return {"kind": kind, "what": what, "dims": dims,
                "float": rng.choice(["f64", "f64", "f32"]), "fp": fp,
                "nbox": _log_int(rng, 1000, most),
                "nq": _log_int(rng, 1000, 100_000 if what == "rays" else 1_000_000),
                "build": rng.random() < 0.5}
    if kind == "hex":
        return {"kind": kind, "n": rng.randint(8, 72), "m": rng.randint(8, 72)}
    return {"kind": kind, "size": rng.randint(4, 8)}


# ------------------------------------------------------------------ inputs ----
def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1_000_003 + stream) % (1 << 62))
    return g


def _uniform(g, shape, lo, hi, dtype=F64):
    return (torch.rand(shape, generator=g, device=DEV, dtype=F64) * (hi - lo) + lo).to(dtype)


@functools.lru_cache(maxsize=1)
def _icosphere(level):
    v, t = synth.icosphere(level)
    return torch.as_tensor(v, device=DEV), torch.as_tensor(t, device=DEV)


def _torus_unit(n):
    """Angles (u, w) of an n x n vertex grid and its 2 n^2 outward triangles."""
    a = 2.0 * math.pi * torch.arange(n, device=DEV, dtype=F64) / n
    u, w = torch.meshgrid(a, a, indexing="ij")
    i = torch.arange(n, device=DEV)[:, None]
    j = torch.arange(n, device=DEV)[None, :]
    i1, j1 = (i + 1) % n, (j + 1) % n
    p, q, r, s = i * n + j, i1 * n + j, i1 * n + j1, i * n + j1
    tri = torch.cat([torch.stack([p, q, r], -1).reshape(-1, 3),
                     torch.stack([p, r, s], -1).reshape(-1, 3)])
    return u.reshape(-1), w.reshape(-1), tri.to(I32)


def _wave(unit, amp, g):
    """1 + amp * a smooth function of the direction, its phase from the seed."""
    ph = _uniform(g, (2,), 0.0, 2.0 * math.pi)
    theta = torch.atan2(unit[:, 1], unit[:, 0])
    phi = torch.acos(unit[:, 2].clamp(-1.0, 1.0))
    return 1.0 + amp * torch.sin(4.0 * theta + ph[0]) * torch.cos(3.0 * phi + ph[1]) * \
        torch.sin(phi) ** 2


def _mesh(case, seed):
    g = _gen(seed, 1)
    if case.get("mesh", "ico") == "torus":
        u, w, tri = _torus_unit(case["size"])
        ph = _uniform(g, (2,), 0.0, 2.0 * math.pi)
        r = 0.3 + case["wave"] * torch.sin(7.0 * u + ph[0]) * torch.cos(5.0 * w + ph[1])
        c = 1.0 + r * torch.cos(w)
        return torch.stack([c * torch.cos(u), c * torch.sin(u), r * torch.sin(w)], 1), tri
    unit, tri = _icosphere(case["size"])
    rad = _wave(unit, case["wave"], g)
    if case.get("noise", 0.0) > 0.0:
        rad = rad * (1.0 + _uniform(g, (unit.shape[0],), -case["noise"], case["noise"]))
    return (unit * rad[:, None]).contiguous(), tri


def _near(v, tri, nq, g, off):
    t = torch.randint(tri.shape[0], (nq,), generator=g, device=DEV)
    b = _uniform(g, (nq, 2), 0.0, 1.0)
    b = torch.where((b.sum(1) > 1.0)[:, None], 1.0 - b, b)
    A, B, C = (v[tri[t, k].long()] for k in range(3))
    n = torch.linalg.cross(B - A, C - A)
    n = n / torch.linalg.vector_norm(n, dim=1, keepdim=True)
    return A + b[:, :1] * (B - A) + b[:, 1:] * (C - A) + _uniform(g, (nq, 1), -off, off) * n


def _queries(case, v, tri, seed):
    g = _gen(seed, 2)
    nq, how = case["nq"], case.get("queries", "box")
    lo, hi = v.min(0).values, v.max(0).values
    n_near = 0 if how == "box" else nq if how == "near" else nq - nq // 2
    pad = 0.5 * float((hi - lo).max()) * (0.2 if how == "mixed" else 0.5)
    box = torch.rand((nq - n_near, 3), generator=g, device=DEV, dtype=F64) * \
        (hi - lo + 2 * pad) + (lo - pad)
    near = _near(v, tri, n_near, g, 0.1 if how == "near" else 0.01)
    return torch.cat([box, near]).contiguous()


def _quad_sphere(n, wave, seed):
    """6 n x n grids of quads on the cube's sides, projected to a wavy sphere."""
    a = torch.linspace(-1.0, 1.0, n + 1, device=DEV, dtype=F64)
    p, q = (x.reshape(-1) for x in torch.meshgrid(a, a, indexing="ij"))
    m = n + 1
    i, j = torch.meshgrid(torch.arange(n, device=DEV), torch.arange(n, device=DEV), indexing="ij")
    quad = torch.stack([i * m + j, (i + 1) * m + j, (i + 1) * m + j + 1, i * m + j + 1],
                       -1).reshape(-1, 4)
    vs, qs = [], []
    for axis in range(3):
        for side in (-1.0, 1.0):
            cols = [None] * 3
            cols[axis] = torch.full_like(p, side)
            cols[(axis + 1) % 3], cols[(axis + 2) % 3] = p, q
            vs.append(torch.stack(cols, 1))
            qs.append((quad if side > 0 else quad.flip(1)) + len(qs) * m * m)
    v = torch.cat(vs)
    v = v / torch.linalg.vector_norm(v, dim=1, keepdim=True)
    return (v * _wave(v, wave, _gen(seed, 1))[:, None]).contiguous(), torch.cat(qs).to(I32)


def _hex_grid(n, h, origin, jitter, angle, g):
    m = n + 1
    a = torch.arange(m, device=DEV)
    v = torch.stack(torch.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3).to(F64) * h
    v = v + _uniform(g, v.shape, -jitter, jitter)
    c, ca, sa = 0.5 * n * h, math.cos(angle), math.sin(angle)
    x, y = v[:, 0] - c, v[:, 1] - c
    v = torch.stack([c + ca * x - sa * y, c + sa * x + ca * y, v[:, 2]], 1) + origin
    b = torch.arange(n, device=DEV)
    i, j, k = torch.meshgrid(b, b, b, indexing="ij")
    p = ((i * m + j) * m + k).reshape(-1)
    di, dj, dk = m * m, m, 1
    corner = [0, di, di + dj, dj, dk, di + dk, di + dj + dk, dj + dk]
    return v.contiguous(), torch.stack([p + o for o in corner], 1).to(I32)


def _rounded_box(p):
    """Signed distance to the rounded box the shape fit aims at."""
    q = p.abs() - torch.tensor([0.8, 0.6, 0.5], device=DEV, dtype=F64) + 0.1
    return torch.linalg.vector_norm(q.clamp(min=0.0), dim=1) + \
        q.max(1).values.clamp(max=0.0) - 0.1


def _find_inputs(case, seed):
    g = _gen(seed, 3)
    d, dt = case["dims"], F32 if case["float"] == "f32" else F64
    nb, nq = case["nbox"], case["nq"]
    c, h = _uniform(g, (nb, d), 0.0, 1.0), _uniform(g, (nb, d), 0.001, 0.01)
    boxes = torch.cat([c - h, c + h], 1).to(dt).contiguous()
    p = _uniform(g, (nq, d), 0.0, 1.0)
    if case["what"] == "points":
        return boxes, p.to(dt).contiguous()
    if case["what"] == "boxes":
        e = _uniform(g, (nq, d), 0.001, 0.01)
        return boxes, torch.cat([p - e, p + e], 1).to(dt).contiguous()
    r = torch.randn((nq, d), generator=g, device=DEV, dtype=F64)
    make = spin.make_rays2d if d == 2 else spin.make_rays
    return boxes, make(p.to(dt).contiguous(), r.to(dt).contiguous(), dtype=dt)


# -------------------------------------------------------------- preparation ----
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("sdf", "grad"):
        v, tri = _mesh(case, seed)
        q = _queries(case, v, tri, seed)
        nq = q.shape[0]
        s = {"case": case, "v": v, "nq": nq, "q": q,
             "sdf": quest.SignedDistance(v, tri, fp_mode=case["fp"]),
             "cp": torch.empty((nq, 3), device=DEV, dtype=F64),
             "elem": torch.empty(nq, device=DEV, dtype=I32)}
        if kind == "sdf":
            s["normal"] = torch.empty((nq, 3), device=DEV, dtype=F64) if case["normals"] else None
            if case["soa"]:
                s["q"] = tuple(q[:, k].contiguous() for k in range(3))
        else:
            s["g"] = torch.randn(nq, generator=_gen(seed, 4), device=DEV, dtype=F32)
            if case["autograd"]:
                s["g"] = s["g"].to(F64)
        return s
    if kind == "fit":
        v, tri = _mesh(case, seed)
        q = _uniform(_gen(seed, 2), (case["nq"], 3), -1.2, 1.2)
        return {"case": case, "v": v, "q": q, "target": _rounded_box(q),
                "sdf": quest.SignedDistance(v, tri, fp_mode=case["fp"]),
                "elem": torch.empty(case["nq"], device=DEV, dtype=I32)}
    if kind == "quads":
        v, quads = _quad_sphere(case["size"], case["wave"], seed)
        off = torch.arange(0, 4 * quads.shape[0] + 1, 4, device=DEV, dtype=I32)
        q = _uniform(_gen(seed, 2), (case["nq"], 3), -1.5, 1.5)
        nq = case["nq"]
        return {"case": case, "q": q, "nq": nq,
                "sdf": quest.SignedDistance(v, quads.reshape(-1), cell_offsets=off),
                "cp": torch.empty((nq, 3), device=DEV, dtype=F64),
                "normal": torch.empty((nq, 3), device=DEV, dtype=F64) if case["normals"] else None,
                "elem": torch.empty(nq, device=DEV, dtype=I32)}
    if kind == "find":
        boxes, q = _find_inputs(case, seed)
        dt = F32 if case["float"] == "f32" else F64
        bvh = spin.BVH(boxes, fp_mode=case["fp"], NDIMS=case["dims"], FloatType=dt)
        nq = case["nq"]
        return {"case": case, "bvh": bvh, "boxes": boxes, "q": q,
                "offsets": torch.empty(nq, device=DEV, dtype=I32),
                "counts": torch.empty(nq, device=DEV, dtype=I32),
                "ids": torch.zeros(_room(case), device=DEV, dtype=I32)}
    g = _gen(seed, 5)
    if kind == "hex":
        n, m = case["n"], case["m"]
        iv, ic = _hex_grid(n, 1.0 / n, 0.0, 0.2 / n, 0.0, g)
        qv, qc = _hex_grid(m, 1.0 / m, 0.003, 0.2 / m, 0.3, g)
        return {"case": case, "args": (iv, ic, qv, qc),
                "pairs": torch.zeros((32 * max(n, m) ** 3, 2), device=DEV, dtype=I32)}
    unit, tri = _icosphere(case["size"])
    edge = float(torch.linalg.vector_norm(unit[tri[0, 0].long()] - unit[tri[0, 1].long()]))
    v = unit + 0.25 * edge * torch.randn(unit.shape, generator=g, device=DEV, dtype=F64)
    shift = torch.tensor([0.5, 0.1, 0.0], device=DEV, dtype=F64)
    return {"case": case, "args": (torch.cat([v, v + shift]).contiguous(),
                                   torch.cat([tri, tri + unit.shape[0]]).contiguous()),
            "pairs": torch.zeros((4096 + tri.shape[0] // 8, 2), device=DEV, dtype=I32)}


# --------------------------------------------------------------------- pass ----
def _room(case):
    """Ids a search's program has room for: about twice the expected number."""
    d, nb = case["dims"], case["nbox"]
    per = {"points": 0.011 ** d, "boxes": 0.022 ** d,
           "rays": 2.0e-4 if d == 3 else 0.012}[case["what"]]
    return int(2.0 * per * nb * case["nq"]) + 8192


def _keep(room, found):
    """A search's list (its length varies) in the program's own array."""
    n = min(found.shape[0], room.shape[0])
    room[:n].copy_(found[:n])
    return room


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("sdf", "quads"):
        d = state["sdf"].computeDistances(state["nq"], state["q"], outClosestPts=state["cp"],
                                          outNormals=state["normal"], outElem=state["elem"])
        return {"dist": d, "cp": state["cp"], "normal": state["normal"], "elem": state["elem"]}
    if kind == "grad":
        if case["autograd"]:
            q = state["q"].detach().requires_grad_(True)
            v = state["v"].detach().requires_grad_(True)
            d = autograd.signed_distance(q, v, state["sdf"], fp_mode=case["fp"])
            gq, gv = torch.autograd.grad(d, (q, v), state["g"])
            return {"dist": d.detach(), "gq": gq, "gv": gv}
        d = state["sdf"].computeDistances(state["nq"], state["q"], outClosestPts=state["cp"],
                                          outElem=state["elem"])
        gq, gv = state["sdf"].backward(state["q"], d, state["elem"], state["g"])
        return {"dist": d, "cp": state["cp"], "elem": state["elem"], "gq": gq, "gv": gv}
    if kind == "fit":
        sdf, q, nq = state["sdf"], state["q"], case["nq"]
        sdf.updateVertices(state["v"])
        d = sdf.computeDistances(nq, q, outElem=state["elem"])
        g = ((d - state["target"]) * (2.0 / nq)).to(F32)
        _, gv = sdf.backward(q, d, state["elem"], g, want_query=False)
        return {"dist": d, "elem": state["elem"], "gv": gv, "v": state["v"] - 1e-3 * gv}
    if kind == "find":
        bvh, nq = state["bvh"], case["nq"]
        if case["build"]:
            bvh.initialize(state["boxes"])
        find = {"points": bvh.findPoints, "boxes": bvh.findBoundingBoxes,
                "rays": bvh.findRays}[case["what"]]
        ids = find(state["offsets"], state["counts"], nq, state["q"])
        return {"offsets": state["offsets"], "counts": state["counts"],
                "ids": _keep(state["ids"], ids)}
    if kind == "hex":
        return {"pairs": _keep(state["pairs"], quest.findCandidatesBVH(*state["args"]))}
    pairs, degenerate = quest.findTriMeshIntersectionsBVH(*state["args"])
    return {"pairs": _keep(state["pairs"], pairs), "degenerate": degenerate}


# --------------------------------------------------------------------- work ----
def _ntris(case):
    if case["kind"] == "quads":
        return 6 * case["size"] ** 2
    return 2 * case["size"] ** 2 if case.get("mesh") == "torus" else 20 * 4 ** case["size"]


def work(case):
    """Bytes: every input and output once (a mesh: 84 bytes a cell, its corners
    and connectivity; a tree built or held: 156 bytes a box). Operations: one
    descent of the tree (two box tests of 20 operations a level) per query,
    and for a distance one triangle (100)."""
    kind = case["kind"]
    if kind in ("sdf", "grad", "fit", "quads"):
        nt, nq = _ntris(case), case["nq"]
        per = {"sdf": 60 + (24 if case.get("normals") else 0), "grad": 88, "fit": 44,
               "quads": 60 + (24 if case.get("normals") else 0)}[kind]
        if kind == "grad" and not case["autograd"]:
            per += 24
        extra = 24 * nt // 2 if kind in ("grad", "fit") else 0
        if kind == "fit":
            extra += 156 * nt
        flops = nq * (40.0 * math.log2(nt) + 100.0) + (50.0 * nq if kind != "sdf" else 0.0)
        return {"bytes": float(nq * per + nt * 84 + extra), "flops": flops}
    if kind == "find":
        w = 4 if case["float"] == "f32" else 8
        d = case["dims"] * (1 if case["what"] == "points" else 2)
        nb, nq = case["nbox"], case["nq"]
        return {"bytes": float(nq * (d * w + 8) + nb * (156 if case["build"] else 108)),
                "flops": nq * 40.0 * math.log2(nb) + (200.0 * nb if case["build"] else 0.0)}
    if kind == "hex":
        n, m = case["n"] ** 3, case["m"] ** 3
        return {"bytes": float((n + m) * 56 + n * 156 + m * 8 * 12),
                "flops": m * 40.0 * math.log2(n) + 200.0 * (n + m)}
    nt = 40 * 4 ** case["size"]
    return {"bytes": float(nt * (84 + 156)), "flops": nt * (40.0 * math.log2(nt) + 200.0)}


# -------------------------------------------------------------------- exact ----
_PAIRS = 2.0e9  # triangle-query pairs that take a few seconds


def _tri_closest(q, T):
    """(squared distance, point, weights) of each query's closest point on each
    of its triangles, q (n, 1, 3), T (1, t, 3, 3), by the nearest of the plane
    projection (where inside) and the three edges."""
    A, B, C = T[..., 0, :], T[..., 1, :], T[..., 2, :]

    def edge(P, Q, i, j):
        e = Q - P
        s = (((q - P) * e).sum(-1) / (e * e).sum(-1)).clamp(0.0, 1.0)
        w = [torch.zeros_like(s)] * 3
        w[i], w[j] = 1.0 - s, s
        x = P + s[..., None] * e
        return ((q - x) ** 2).sum(-1), torch.stack(w, -1)

    best, w = edge(A, B, 0, 1)
    for P, Q, i, j in ((B, C, 1, 2), (A, C, 0, 2)):
        d, we = edge(P, Q, i, j)
        less = d < best
        best, w = torch.where(less, d, best), torch.where(less[..., None], we, w)
    n = torch.linalg.cross(B - A, C - A)
    nn = (n * n).sum(-1)
    wb = (torch.linalg.cross((q - A).expand(-1, A.shape[1], -1),
                             (C - A).expand(q.shape[0], -1, -1)) * n).sum(-1) / nn
    wc = (torch.linalg.cross((B - A).expand(q.shape[0], -1, -1),
                             (q - A).expand(-1, A.shape[1], -1)) * n).sum(-1) / nn
    inside = (wb > 0.0) & (wc > 0.0) & (wb + wc < 1.0)
    d = (((q - A) * n).sum(-1)) ** 2 / nn
    wf = torch.stack([1.0 - wb - wc, wb, wc], -1)
    best = torch.where(inside & (d < best), d, best)
    return best, torch.where(inside[..., None], wf, w)


def _brute(v, tri, q):
    """Signed distance, closest point, triangle and weights by trying every
    triangle; the sign from the solid angle the surface covers."""
    T = v[tri.long()]
    nq, nt = q.shape[0], T.shape[0]
    tc = 4096
    qc = max(1, 4_000_000 // tc)
    sd, cp, el, wt = [], [], [], []
    for a in range(0, nq, qc):
        p = q[a:a + qc]
        best = torch.full((p.shape[0],), math.inf, device=DEV, dtype=F64)
        elem = torch.zeros(p.shape[0], device=DEV, dtype=torch.long)
        w = torch.zeros((p.shape[0], 3), device=DEV, dtype=F64)
        angle = torch.zeros(p.shape[0], device=DEV, dtype=F64)
        for b in range(0, nt, tc):
            Tb = T[None, b:b + tc]
            d, ww = _tri_closest(p[:, None, :], Tb)
            m, k = d.min(1)
            less = m < best
            best = torch.where(less, m, best)
            elem = torch.where(less, k + b, elem)
            w = torch.where(less[:, None], ww[torch.arange(p.shape[0], device=DEV), k], w)
            X, Y, Z = (Tb[..., k, :] - p[:, None, :] for k in range(3))
            x, y, z = (torch.linalg.vector_norm(c, dim=-1) for c in (X, Y, Z))
            num = (X * torch.linalg.cross(Y, Z)).sum(-1)
            den = x * y * z + (X * Y).sum(-1) * z + (Y * Z).sum(-1) * x + (Z * X).sum(-1) * y
            angle += 2.0 * torch.atan2(num, den).sum(1)
        inside = angle > 2.0 * math.pi
        sd.append(torch.where(inside, -1.0, 1.0) * best.sqrt())
        cp.append((w[..., None] * T[elem]).sum(1))
        el.append(elem)
        wt.append(w)
    return torch.cat(sd), torch.cat(cp), torch.cat(el), torch.cat(wt)


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("sdf", "grad", "fit", "quads"):
        return None
    if float(case["nq"]) * _ntris(case) * (2 if kind == "quads" else 1) > _PAIRS:
        return None
    if kind == "quads":
        v, c = _quad_sphere(case["size"], case["wave"], seed)
        tri = torch.stack([c[:, [0, 1, 2]], c[:, [0, 2, 3]]], 1).reshape(-1, 3)
        q = _uniform(_gen(seed, 2), (case["nq"], 3), -1.5, 1.5)
    else:
        v, tri = _mesh(case, seed)
        q = _uniform(_gen(seed, 2), (case["nq"], 3), -1.2, 1.2) if kind == "fit" else \
            _queries(case, v, tri, seed)
    d, cp, elem, w = _brute(v, tri, q)
    if kind in ("sdf", "quads"):
        return {"dist": d, "cp": cp, "normal": None, "elem": None}
    if kind == "fit":
        up = ((d - _rounded_box(q)) * (2.0 / case["nq"])).to(F32).to(F64)
    else:
        up = torch.randn(case["nq"], generator=_gen(seed, 4), device=DEV, dtype=F32).to(F64)
    gq = (up / d)[:, None] * (q - cp)
    gv = torch.zeros_like(v)
    for k in range(3):
        gv.index_add_(0, tri[elem, k].long(), -w[:, k:k + 1] * gq)
    if kind == "fit":
        return {"dist": d, "elem": None, "gv": gv, "v": v - 1e-3 * gv}
    if case["autograd"]:
        return {"dist": d, "gq": gq, "gv": gv}
    return {"dist": d, "cp": cp, "elem": None, "gq": gq, "gv": gv}
