"""The point, box and ray searches on the compact nodes (halves, scaled per node)
give the oracle's lists, order included, over the forms a search takes: 2-D and
3-D, double and float trees, two-array and interleaved points, both calls
(one-call and count-then-fill), and the inputs where a rounded box could decide
differently: queries on the faces of the scaled boxes and one step either side,
scenes far from the origin, boxes of very different sizes, flat and invalid
boxes, rays along axes, through corners, from far away and of extreme lengths,
and coordinates that are not finite. Results are integers: no tolerance.
"""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from axom_amd import _lib as L  # noqa: E402
from axom_amd import quest, spin  # noqa: E402
from oracle import oracle as orc  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=DEV)


def _scene(name, n, nd, rng):
    """(n, 2 nd) boxes: min, max."""
    c = rng.random((n, nd))
    h = rng.uniform(0.0005, 0.03, (n, nd))
    if name == "far":  # boxes of 2^-20 of their distance to the origin
        c = 1.0e6 + c
    elif name == "scales":  # sizes and distances over twelve decades
        s = 10.0 ** rng.uniform(-12, 0, (n, 1))
        c, h = 0.5 + (c - 0.5) * s, h * s
    elif name == "tiny":
        c, h = c * 1e-90, h * 1e-90
    elif name == "huge":  # past the range of the compact nodes
        c, h = c * 1e120, h * 1e120
    elif name == "flat":
        h[rng.random(n) < 0.5, rng.integers(nd)] = 0.0
        h[rng.random(n) < 0.2] = 0.0
    elif name == "same":
        c[:], h[:] = 0.5, 0.01
    b = np.concatenate([c - h, c + h], 1)
    if name == "invalid":
        b[::7, 0], b[::7, nd] = b[::7, nd].copy(), b[::7, 0].copy()
        b[::11] = [np.finfo(np.float64).max / 8] * nd + [-np.finfo(np.float64).max / 8] * nd
        b[n - 1] = b[max(1, n - 2)]
    elif name == "nan":
        b[n // 2, 0] = np.nan
    return b


def _queries(kind, nq, nd, boxes, leaf_boxes, dtype, rng):
    ok = np.isfinite(boxes).all(1) & (boxes[:, :nd] <= boxes[:, nd:]).all(1)
    b = boxes[ok] if ok.any() else boxes
    lo, hi = b[:, :nd].min(0), b[:, nd:].max(0)
    p = lo + (hi - lo) * rng.uniform(-0.05, 1.05, (nq, nd))
    # on the faces of the leaves' scaled boxes, and one step either side
    k = nq // 2
    f = leaf_boxes[rng.integers(leaf_boxes.shape[0], size=k)].reshape(k, 2, nd)
    u = rng.random((k, nd))
    q = f[:, 0] + (f[:, 1] - f[:, 0]) * u
    ax, side = rng.integers(nd, size=k), rng.integers(2, size=k)
    face = f[np.arange(k), side, ax].astype(dtype)
    step = rng.integers(-1, 2, size=k)
    face = np.where(step < 0, np.nextafter(face, dtype(-np.inf)),
                    np.where(step > 0, np.nextafter(face, dtype(np.inf)), face))
    q[np.arange(k), ax] = face
    p[:k] = q
    p[k] = np.inf
    p[k + 1, 0] = -np.inf
    p[k + 2, 0] = np.nan
    p[k + 3] = np.nan
    if kind == "points":
        return p.astype(dtype)
    h = (hi - lo) * rng.uniform(0.0, 0.02, (nq, nd)) * (rng.random((nq, 1)) < 0.7)
    q = np.concatenate([p - h, p + h], 1)
    q[k + 4, 0], q[k + 4, nd] = hi[0], lo[0]  # an inverted query
    q[k + 5, nd] = np.nan
    q[k + 6, :nd], q[k + 6, nd:] = -np.inf, np.inf
    return q.astype(dtype)


def _rays(nq, nd, boxes, leaf_boxes, dtype, rng):
    ok = np.isfinite(boxes).all(1) & (boxes[:, :nd] <= boxes[:, nd:]).all(1)
    b = boxes[ok] if ok.any() else boxes
    lo, hi = b[:, :nd].min(0), b[:, nd:].max(0)
    ext = (hi - lo).max()
    o = lo + (hi - lo) * rng.uniform(-0.2, 1.2, (nq, nd))
    d = rng.normal(size=(nq, nd))
    f = leaf_boxes[rng.integers(leaf_boxes.shape[0], size=nq)].reshape(nq, 2, nd)
    corner = f[np.arange(nq)[:, None], rng.integers(2, size=(nq, nd)), np.arange(nd)[None]]
    k = np.arange(nq) % 12
    m = k == 1  # along an axis, in a face's plane or a step from it
    ax = rng.integers(nd, size=nq)
    d[m] = 0.0
    d[m, ax[m]] = np.where(rng.random(m.sum()) < 0.5, 1.0, -1.0)
    o[m] = np.where(np.arange(nd)[None] == ax[m, None], o[m], corner[m])
    m = k == 2  # one axis taken as zero, the others not
    d[m, ax[m]] = rng.choice([0.0, 1e-17, -1e-17, 1e-9, -3e-8], m.sum())
    o[m, ax[m]] = corner[m, ax[m]]
    m = (k == 3) | (k == 4)  # at a corner
    d[m] = corner[m] - o[m]
    m = k == 5  # from far away, at a corner
    o[m] = o[m] + 10.0 ** rng.uniform(0, 9, (m.sum(), 1)) * ext * d[m]
    d[m] = corner[m] - o[m]
    m = k == 6  # from a corner
    o[m] = corner[m]
    d /= np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-300)
    m = k == 7  # not unit
    d[m] *= 10.0 ** rng.uniform(-25, 25, (m.sum(), 1))
    m = k == 8
    bad = rng.choice([np.nan, np.inf, -np.inf, 0.0, 1e-310], (m.sum(), 2 * nd))
    q = np.concatenate([o, d], 1)
    q[m] = np.where(rng.random(bad.shape) < 0.4, bad, q[m])
    q[8] = np.nan
    q[20, nd:] = 0.0
    with np.errstate(over="ignore"):
        return q.astype(dtype)


def _find(g, kind, prims, nq):
    off = torch.empty(nq, dtype=torch.int32, device=DEV)
    cnt = torch.empty_like(off)
    f = {"points": g.findPoints, "boxes": g.findBoundingBoxes, "rays": g.findRays}[kind]
    cand = f(off, cnt, nq, prims)
    return off.cpu().numpy(), cnt.cpu().numpy(), cand.cpu().numpy()


@pytest.mark.parametrize("scene", ["plain", "far", "scales", "tiny", "huge", "flat", "same",
                                   "invalid", "nan"])
@pytest.mark.parametrize("nd,dtype", [(3, np.float64), (2, np.float64), (3, np.float32),
                                      (2, np.float32)])
@pytest.mark.parametrize("n", [2, 3, 65, 4097])
def test_find_on_compact_nodes(scene, nd, dtype, n):
    rng = np.random.default_rng([n, nd, sorted(["plain", "far", "scales", "tiny", "huge", "flat",
                                                "same", "invalid", "nan"]).index(scene)])
    if dtype is np.float32 and scene in ("tiny", "huge"):
        pytest.skip("outside the float range")
    with np.errstate(over="ignore"):
        boxes = _scene(scene, n, nd, rng).astype(dtype)
    kw = dict(FloatType=torch.float32) if dtype is np.float32 else {}
    g = spin.BVH(NDIMS=nd, scaleFactor=1.000123, **kw)
    g.initialize(_t(boxes))
    o = orc.OracleBVH(boxes, 1.000123, ndims=nd, dtype=dtype)
    oe = o.export()
    leaf = oe["nodes"][oe["children"] < 0]
    if leaf.shape[1] == 6 and nd == 2:
        leaf = leaf[:, [0, 1, 3, 4]]
    good = np.isfinite(leaf).all(1)
    nq = 331
    for kind in ("points", "boxes"):
        q = _queries(kind, nq, nd, boxes.astype(np.float64), leaf[good], dtype, rng)
        ooff, ocnt, ocand = o.find(kind, q)
        off, cnt, cand = _find(g, kind, _t(q), nq)
        assert np.array_equal(cnt, ocnt), (kind, np.flatnonzero(cnt != ocnt)[:5])
        assert np.array_equal(off, ooff) and np.array_equal(cand, ocand), kind
        if kind == "points":  # separate coordinate arrays
            off, cnt, cand = _find(g, kind, tuple(_t(q[:, d]) for d in range(nd)), nq)
            assert np.array_equal(cnt, ocnt) and np.array_equal(cand, ocand)
    for nq in (31, 5000):
        q = _rays(nq, nd, boxes.astype(np.float64), leaf[good], dtype, rng)
        ooff, ocnt, ocand = o.find("rays", q)
        off, cnt, cand = _find(g, "rays", _t(q), nq)
        assert np.array_equal(cnt, ocnt), ("rays", nq, np.flatnonzero(cnt != ocnt)[:5])
        assert np.array_equal(off, ooff) and np.array_equal(cand, ocand), ("rays", nq)


@pytest.mark.parametrize("kind", ["boxes", "rays"])
def test_count_then_fill_on_compact_nodes(kind):
    """The two-call search: the fill walks again and writes the counted lists."""
    rng = np.random.default_rng(5)
    boxes = _scene("plain", 20_011, 3, rng)
    g, o = spin.BVH(_t(boxes)), orc.OracleBVH(boxes, 1.000123)
    q = boxes[:777]
    if kind == "rays":
        e = o.export()
        q = _rays(777, 3, boxes, e["nodes"][e["children"] < 0], np.float64, rng)
    code = {"boxes": L.QUERY_BOXES, "rays": L.QUERY_RAYS}[kind]
    ooff, ocnt, ocand = o.find(kind, q)
    t = _t(q)
    n = q.shape[0]
    off = torch.empty(n, dtype=torch.int32, device=DEV)
    cnt = torch.empty_like(off)
    tot = ctypes.c_int64()
    args = (ctypes.c_void_p(t.data_ptr()), None, None, 6, n, g._tol)
    L.check(L.lib().axsq_bvh_find_count(g._h, code, *args[:5], g._tol, spin._ptr(off),
                                        spin._ptr(cnt), ctypes.byref(tot), None))
    assert tot.value == ocand.size and np.array_equal(cnt.cpu().numpy(), ocnt)
    cand = torch.empty(tot.value, dtype=torch.int32, device=DEV)
    L.check(L.lib().axsq_bvh_find_fill(g._h, code, *args[:5], g._tol, spin._ptr(off),
                                       spin._ptr(cnt), spin._ptr(cand), None))
    assert np.array_equal(cand.cpu().numpy(), ocand)


@pytest.mark.parametrize("scene", ["plain", "far", "flat", "sizes", "huge"])
@pytest.mark.parametrize("n", [3, 63, 64, 65, 513, 6000])
def test_self_intersections_on_compact_nodes(scene, n):
    """Pairs met once, from their lower leaf, are the reference's pairs: soups
    whose triangles hit more others than are kept, lie in a plane (boxes without
    extent), are far from the origin (boxes thin by units in the last place) or
    differ in size by six decades; a huge one takes the general walk."""
    rng = np.random.default_rng(n)
    size = (0.4 / n) ** (1 / 3)
    s = 10.0 ** rng.uniform(-6, 0, (n, 1, 1)) if scene == "sizes" else 1.0
    v = rng.uniform(-1, 1, (n, 1, 3)) + s * rng.normal(0, size, (n, 3, 3))
    if scene == "flat":
        v[: n // 2, :, 2] = 0.25
        v[n // 2 :, :, 0] = np.round(v[n // 2 :, :, 0], 1)
    elif scene == "far":
        v = v + 2.0**24
        v[:, :, 0] = 2.0**24 + rng.integers(0, 3, (n, 3)) * 2.0**-28
    elif scene == "huge":
        v = v * 1e120
    t = np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    v = np.ascontiguousarray(v.reshape(-1, 3))
    pairs, degen = quest.findTriMeshIntersectionsBVH(_t(v), _t(t))
    want, want_degen = orc.mesh_self_intersections(v, t)
    assert np.array_equal(pairs.cpu().numpy().reshape(-1, 2), want.reshape(-1, 2))
    assert np.array_equal(degen.cpu().numpy(), want_degen)


def test_pair_lists_in_arrays_of_their_own_and_in_the_callers_memory():
    """Both forms of the two pair searches give the same lists; an allocator
    that gives nothing ends the call with an error and no result."""
    rng = np.random.default_rng(9)
    n = 700
    v = rng.uniform(-1, 1, (n, 1, 3)) + rng.normal(0, 0.08, (n, 3, 3))
    x, y, z = (_t(v.reshape(-1, 3)[:, d]) for d in range(3))
    t = _t(np.arange(3 * n, dtype=np.int32).reshape(n, 3))
    vp = ctypes.c_void_p

    def take(ptr, count):
        out = torch.empty(count, dtype=torch.int32, device=DEV)
        hip = ctypes.CDLL("libamdhip64.so")
        assert hip.hipMemcpy(vp(out.data_ptr()), ptr, ctypes.c_size_t(4 * count), 3) == 0
        L.check(L.lib().axsq_free(ptr))
        return out.cpu().numpy()

    pairs, degen = quest.findTriMeshIntersectionsBVH((x, y, z), t)
    a, b, d, np_, nd = vp(), vp(), vp(), ctypes.c_int64(), ctypes.c_int64()
    mesh = (spin._ptr(x), spin._ptr(y), spin._ptr(z), 3 * n, spin._ptr(t), n)
    L.check(L.lib().axsq_mesh_self_intersections(
        *mesh, 1e-8, ctypes.byref(a), ctypes.byref(b), ctypes.byref(np_), ctypes.byref(d),
        ctypes.byref(nd), None))
    assert np_.value == pairs.shape[0] > 0 and nd.value == degen.numel()
    assert np.array_equal(np.stack([take(a, np_.value), take(b, np_.value)], 1),
                          pairs.cpu().numpy())
    L.check(L.lib().axsq_free(d))

    pairs = quest.findCandidatesBVH((x, y, z), t, (x, y, z), t)
    L.check(L.lib().axsq_mesh_candidates(*mesh, *mesh, 3, ctypes.byref(a), ctypes.byref(b),
                                         ctypes.byref(np_), None))
    assert np_.value == pairs.shape[0] > n
    assert np.array_equal(np.stack([take(a, np_.value), take(b, np_.value)], 1),
                          pairs.cpu().numpy())

    none = L.ALLOC_FN(lambda ctx, nbytes: None)
    rc = L.lib().axsq_mesh_candidates_alloc(*mesh, *mesh, 3, none, None, ctypes.byref(a),
                                            ctypes.byref(np_), None)
    assert rc == L.ERRORS_BY_NAME["AXSQ_ERR_NOMEM"] and not a.value and np_.value == 0


@pytest.mark.parametrize("nverts", [131071, 131072, 131073])
def test_self_intersections_either_side_of_packed_vertices(nverts):
    """From 131,072 vertices on the triangles are read through packed records."""
    rng = np.random.default_rng(nverts)
    n = 4001
    v = rng.random((nverts, 3))
    ids = rng.choice(nverts - 1, size=3 * n, replace=False).astype(np.int32)
    ids[-1] = nverts - 1
    t = ids.reshape(n, 3)
    v[t[:, 1:]] = v[t[:, :1]] + rng.normal(0.0, 0.03, (n, 2, 3))
    t[7, 1] = t[7, 0]  # no area
    pairs, degen = quest.findTriMeshIntersectionsBVH(_t(v), _t(t))
    opairs, odegen = orc.mesh_self_intersections(v, t, nthreads=8)
    assert opairs.shape[0] > 100 and odegen.tolist() == [7]
    assert np.array_equal(pairs.cpu().numpy(), opairs)
    assert np.array_equal(degen.cpu().numpy(), odegen)
