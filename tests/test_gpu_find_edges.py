"""The candidate searches and pair tests at the edges of the compact nodes' number
range and of their index range: results are integers, equal to the oracle's, order
included.
"""
import time

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


def _check(boxes, scale, dtype, queries):
    """Searches of the tree over `boxes` against the oracle; queries: kind -> prims."""
    nd = boxes.shape[1] // 2
    kw = dict(FloatType=torch.float32) if dtype is np.float32 else {}
    g = spin.BVH(_t(boxes), scaleFactor=scale, NDIMS=nd, **kw)
    o = orc.OracleBVH(boxes, scale, ndims=nd, dtype=dtype)
    for kind, q in queries.items():
        ooff, ocnt, ocand = o.find(kind, q)
        n = q.shape[0]
        off = torch.empty(n, dtype=torch.int32, device=DEV)
        cnt = torch.empty_like(off)
        f = {"points": g.findPoints, "boxes": g.findBoundingBoxes, "rays": g.findRays}[kind]
        cand = f(off, cnt, n, _t(q))
        assert np.array_equal(cnt.cpu().numpy(), ocnt), kind
        assert np.array_equal(off.cpu().numpy(), ooff), kind
        assert np.array_equal(cand.cpu().numpy(), ocand), kind


def _beyond_faces(lo, hi, nd, dtype, size, rng):
    """Points and small boxes from one step to 2^-13 of `size` beyond a face of
    [lo, hi], or as far inside it, the other coordinates well inside."""
    n = 400
    p = lo + (hi - lo) * rng.uniform(0.1, 0.9, (n, nd))
    ax, side = rng.integers(nd, size=n), rng.integers(2, size=n)
    face = np.where(side == 0, lo, hi).astype(dtype)
    by = size * 2.0 ** rng.uniform(-30, -13, n) * rng.choice([-1, 1, 1], n)
    out = np.where(side == 0, face - by, face + by).astype(dtype)
    step = np.nextafter(face, np.where(side == 0, -np.inf, np.inf).astype(dtype))
    out = np.where(rng.random(n) < 0.2, step, out)
    p = p.astype(dtype)
    p[np.arange(n), ax] = out
    b = np.concatenate([p, p], 1)
    far = np.where(side == 0, out - dtype(0.1 * size), out + dtype(0.1 * size)).astype(dtype)
    b[np.arange(n), ax + nd * (side == 0)] = out
    b[np.arange(n), ax + nd * (side == 1)] = far
    b = np.concatenate([np.minimum(b[:, :nd], b[:, nd:]), np.maximum(b[:, :nd], b[:, nd:])], 1)
    return p, b.astype(dtype)


@pytest.mark.parametrize("eps", [2.0**-24, 2.0**-22, 2.0**-21, 2.0**-19, 2.0**-15])
@pytest.mark.parametrize("nd,dtype,depth", [
    (3, np.float64, 0), (2, np.float64, 0), (3, np.float32, 0), (2, np.float32, 0),
    (3, np.float64, 12), (2, np.float64, 12), (3, np.float64, 27), (2, np.float64, 27)])
def test_extents_just_below_a_power_of_two(eps, nd, dtype, depth):
    """A node's extents, with their margins, round out past the range they are
    scaled to; a query just outside such a face is in no box."""
    rng = np.random.default_rng([depth, nd])
    w = (1.0 - eps) * 2.0**-depth  # half width of a cluster around the origin
    lo = np.full(nd, -w)
    b = [np.concatenate([lo * 0.9, -lo]), np.concatenate([lo, -lo * 0.9])]
    if depth:  # two far boxes around it, so that the cluster is small in the tree
        b.append(np.concatenate([np.full(nd, 0.9), np.full(nd, 1.0)]))
        b.append(np.concatenate([np.full(nd, -1.0), np.full(nd, -0.9)]))
    boxes = np.array(b).astype(dtype)
    p, q = _beyond_faces(-w, w, nd, dtype, w, rng)
    _check(boxes, 1.0, dtype, {"points": p, "boxes": q})


@pytest.mark.parametrize("nd,dtype", [(3, np.float64), (2, np.float64), (3, np.float32)])
@pytest.mark.parametrize("n", [4, 64, 600, 4097, 262_145, 300_001])
def test_boxes_with_nan_coordinates(n, nd, dtype):
    """A box's NaN bound gives way to any other in a union, so which boxes an inner
    node holds depends on how its union is put together: as the reference's."""
    rng = np.random.default_rng([n, nd])
    h = 0.5 / n ** (1.0 / nd)
    c = rng.random((n, nd))
    e = rng.uniform(0.2 * h, h, (n, nd))
    boxes = np.concatenate([c - e, c + e], 1)
    k = np.flatnonzero(rng.random(n) < 0.2)
    k = k if k.size else np.array([n // 2])
    boxes[k, rng.integers(2 * nd, size=k.size)] = np.nan
    boxes[k[::3]] = np.nan
    # the root's bounds, from minima whose order is open, hold whatever it is
    boxes[[0, -1]] = [-0.2] * nd + [1.2] * nd
    p = rng.random((2000, nd))
    q = np.concatenate([p - h, p + h], 1)
    d = rng.normal(size=(200, nd))
    r = np.concatenate([p[:200], d / np.linalg.norm(d, axis=1, keepdims=True)], 1)
    _check(boxes.astype(dtype), 1.000123, dtype,
           {"points": p.astype(dtype), "boxes": q.astype(dtype), "rays": r.astype(dtype)})


def _search(g, p):
    off = torch.empty(p.shape[0], dtype=torch.int32, device=DEV)
    cnt = torch.empty_like(off)
    return off, cnt, g.findPoints(off, cnt, p.shape[0], p)


@pytest.mark.parametrize("nq", [1, 63, 64, 65, 1000])
def test_kept_ids_beside_queries_with_more(nq):
    """Waves whose queries have none, few, all that are kept and more than are kept."""
    rng = np.random.default_rng(nq)
    sizes = [500, 64, 65, 63, 10, 3, 1]
    boxes = np.concatenate([np.tile([[2.0 * k] * 3 + [2.0 * k + 1] * 3], (m, 1))
                            for k, m in enumerate(sizes)])
    rng.shuffle(boxes)
    p = rng.integers(0, len(sizes) + 2, nq)[:, None] * 2.0 + rng.uniform(0.1, 0.9, (nq, 3))
    g, o = spin.BVH(_t(boxes)), orc.OracleBVH(boxes, 1.000123)
    ooff, ocnt, ocand = o.find("points", p)
    for _ in range(2):  # the first search of a tree fills by a second walk
        off, cnt, cand = _search(g, _t(p))
        assert np.array_equal(cnt.cpu().numpy(), ocnt)
        assert np.array_equal(off.cpu().numpy(), ooff)
        assert np.array_equal(cand.cpu().numpy(), ocand)


def test_candidate_total_next_to_the_int32_limit():
    """The kept ids of the last queries end 5 below 2^31 - 1."""
    many, few = 65536, 10
    boxes = torch.tensor([[0.0] * 3 + [1.0] * 3], dtype=torch.float64, device=DEV)
    boxes = torch.cat([boxes.repeat(many, 1), boxes.repeat(few, 1) + 2.0])
    na, nb = 32767, 6553
    p = torch.full((na + nb, 3), 0.5, dtype=torch.float64, device=DEV)
    p[na:] = 2.5
    total = na * many + nb * few
    assert total == 2**31 - 6
    g = spin.BVH(boxes)
    for _ in range(2):
        off, cnt, cand = _search(g, p)
        assert cand.numel() == total
        assert bool((cnt[:na] == many).all()) and bool((cnt[na:] == few).all())
        ids = torch.arange(many + few, dtype=torch.int32, device=DEV)
        assert bool((cand[na * many:].view(nb, few) == ids[many:]).all())
        a = cand[:na * many].view(na, many)
        assert all(bool((a[r:r + 2048] == ids[:many]).all()) for r in range(0, na, 2048))
        del cand, a


@pytest.mark.parametrize("nd,dtype", [(3, np.float64), (2, np.float64), (3, np.float32),
                                      (2, np.float32)])
@pytest.mark.parametrize("n", [1, 2, 3, 65, 4097])
@pytest.mark.parametrize("others", [False, True])
def test_equal_boxes_without_extent(n, others, nd, dtype):
    """Boxes that are all one point, and the same among others: queries at the
    point, one step from it and elsewhere."""
    rng = np.random.default_rng([n, nd])
    at = np.full((1, nd), 0.7)
    boxes = np.repeat(np.concatenate([at, at], 1), n, 0)
    if others:
        c = rng.random((n, nd))
        boxes = np.concatenate([boxes, np.concatenate([c - 0.01, c + 0.01], 1)])
        rng.shuffle(boxes)
    boxes = boxes.astype(dtype)
    p = np.repeat(at, 60, 0).astype(dtype)
    p[20:40] = np.nextafter(p[20:40], rng.choice([0.0, 1.0], (20, nd)).astype(dtype))
    p[40:] = rng.random((20, nd))
    q = np.concatenate([p, p], 1)
    q[::3, nd:] += dtype(0.01)
    d = rng.normal(size=(60, nd)).astype(dtype)
    r = np.concatenate([p - d * (np.arange(60)[:, None] % 2).astype(dtype), d], 1)
    _check(boxes, 1.000123, dtype, {"points": p, "boxes": q, "rays": r})


def test_equal_boxes_without_extent_are_passed_over():
    """A search that misses such a tree ends at its root: 20,000 points and 200,000
    boxes took 149 ms where every node was visited, 0.1 at the root."""
    rng = np.random.default_rng(3)
    n = 200_000
    c = rng.random((n, 3))
    p = _t(rng.random((20_000, 3)) + 2.0)

    def best(boxes):
        g, t = spin.BVH(_t(boxes)), []
        for _ in range(4):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            _, cnt, _ = _search(g, p)
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b))
        assert int(cnt.sum()) == 0
        return min(t)

    spread = best(np.concatenate([c, c], 1))
    assert best(np.full((n, 6), 0.5)) < 10.0 + 20.0 * spread


@pytest.mark.parametrize("nd,dtype", [(3, np.float64), (2, np.float64), (3, np.float32)])
@pytest.mark.parametrize("depth", [5, 28, 29, 30, 31, 50])
def test_boundless_queries_beside_an_invalid_box(depth, nd, dtype):
    """A query that holds everything, at a small node one of whose children is
    invalid."""
    w = 1.5 * 2.0**-depth
    far = np.finfo(dtype).max / 8
    boxes = np.array([[-1.0] * nd + [-0.9] * nd, [-w] * nd + [w] * nd, [far] * nd + [-far] * nd,
                      [0.9] * nd + [1.0] * nd]).astype(dtype)
    big = np.array([1.0, 1e15, 1e20, 1e25, 1e30, 1e36, far, np.inf])
    q = np.repeat(big[:, None], 2 * nd, 1)
    q[:, :nd] *= -1.0
    p = np.concatenate([q[:, nd:], q[:, :nd], q[:, :nd] * (-1.0) ** np.arange(nd)])
    _check(boxes, 1.0, dtype, {"points": p.astype(dtype), "boxes": q.astype(dtype)})


@pytest.mark.parametrize("ntris", [1, 7, 2_000_000])
@pytest.mark.parametrize("some", [False, True])
def test_vertex_ids_out_of_range_cost_no_pairs(ntris, some):
    """Refused as before, in the time of a tree build: no pair is tested for
    triangles without vertices, however many they are."""
    rng = np.random.default_rng(ntris)
    v = rng.random((99, 3))
    t = np.full((ntris, 3), 99, np.int32)
    t[ntris // 2:] = -1
    if some:
        t[: min(ntris - 1, 33)] = np.arange(99).reshape(33, 3)[: min(ntris - 1, 33)]
    v, t = _t(v), _t(t)
    quest.findTriMeshIntersectionsBVH(v, t[:1] * 0)  # the library and its memory are there
    torch.cuda.synchronize()
    a = time.perf_counter()
    with pytest.raises(L.AxsqError, match="outside"):
        quest.findTriMeshIntersectionsBVH(v, t)
    assert time.perf_counter() - a < 5.0


def _cells(n, nd):
    """n^nd cells of the unit cube in order, a little apart."""
    c = np.stack(np.meshgrid(*[np.arange(n)] * nd, indexing="ij"), -1).reshape(-1, nd)
    return np.concatenate([c + 0.1, c + 0.9], 1) / n


@pytest.mark.parametrize("nd,dtype", [(3, np.float64), (2, np.float64), (3, np.float32)])
@pytest.mark.parametrize("far", [1e4, 1e9, 1e11, 1e12, 1e15, 1e30])
def test_small_boxes_in_large_bounds(far, nd, dtype):
    """A box of 10^4 to 10^30 times the others' extent among them."""
    rng = np.random.default_rng(nd)
    boxes = np.concatenate([_cells(11, nd), [[-far] * nd + [far] * nd]]).astype(dtype)
    p = rng.uniform(-0.1, 1.1, (500, nd))
    p[::50] *= far
    h = rng.uniform(0.0, 0.1, (500, 1))
    d = rng.normal(size=(100, nd))
    _check(boxes, 1.000123, dtype,
           {"points": p.astype(dtype), "boxes": np.concatenate([p - h, p + h], 1).astype(dtype),
            "rays": np.concatenate([p[:100], d], 1).astype(dtype)})


def test_small_boxes_in_large_bounds_are_told_apart():
    """100,000 points among 64,000 cells and a box for everything: 52 ms where each
    point visited every node, 0.2 with the nodes that tell the cells apart."""
    cells = _cells(40, 3)
    p = _t(np.random.default_rng(1).random((100_000, 3)))

    def best(boxes):
        g, t = spin.BVH(_t(boxes)), []
        for _ in range(4):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            _search(g, p)
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b))
        return min(t)

    alone = best(cells)
    assert best(np.concatenate([cells, [[-1e15] * 3 + [1e15] * 3]])) < 2.0 + 20.0 * alone


@pytest.mark.parametrize("nverts", [524_287, 524_288, 524_289])
def test_self_intersections_either_side_of_the_vertex_records(nverts):
    """From 524,288 vertices on the triangles are read through packed records."""
    rng = np.random.default_rng(nverts)
    n = 3000
    v = rng.random((nverts, 3))
    ids = rng.choice(nverts - 1, size=3 * n, replace=False).astype(np.int32)
    ids[-1] = nverts - 1
    t = ids.reshape(n, 3)
    v[t[:, 1:]] = v[t[:, :1]] + rng.normal(0.0, 0.03, (n, 2, 3))
    t[7, 1] = t[7, 0]  # no area
    pairs, degen = quest.findTriMeshIntersectionsBVH(_t(v), _t(t))
    opairs, odegen = orc.mesh_self_intersections(v, t, nthreads=8)
    assert opairs.shape[0] > 50 and odegen.tolist() == [7]
    assert np.array_equal(pairs.cpu().numpy(), opairs)
    assert np.array_equal(degen.cpu().numpy(), odegen)
