"""Meshes on which oriented boxes gain little: flat and noisy height fields along the
axes, flat boxes, slender triangles, triangles that do not meet. The walk a call
takes depends on what they gain, on the tree's size and on the batch; the outputs
are those of the reference walk, bit for bit, and no call is much slower."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from axom_amd import quest, synth  # noqa: E402
from oracle import oracle as orc  # noqa: E402
from tests.test_gpu_sdf import _compare, _eval, _t  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _grid(n, z):
    g = np.linspace(-1.0, 1.0, n + 1)
    x, y = np.meshgrid(g, g, indexing="ij")
    v = np.stack([x, y, z(x, y)], -1).reshape(-1, 3)
    i = np.arange(n)[:, None] * (n + 1) + np.arange(n)[None]
    t = [np.stack([i, i + n + 1, i + n + 2], -1), np.stack([i, i + n + 2, i + 1], -1)]
    return v, np.concatenate([a.reshape(-1, 3) for a in t]).astype(np.int32)


def _mesh(name):
    rng = np.random.default_rng(7)
    if name == "flat":  # 131,328 triangles
        return _grid(257, lambda x, y: 0.0 * x)
    if name == "noise":  # 132,098, noise of a cell's size
        return _grid(257, lambda x, y: rng.normal(0.0, 0.008, x.shape))
    if name == "small noise":  # 20,000
        return _grid(100, lambda x, y: rng.normal(0.0, 0.02, x.shape))
    if name == "cube":  # 135,000
        v, q = synth.cube_sphere(107, project=False)
        return v, np.concatenate([q[:, [0, 1, 2]], q[:, [0, 2, 3]]]).astype(np.int32)
    if name == "soup":
        n = 20_000
        v = rng.uniform(-1, 1, (n, 1, 3)) + rng.normal(0.0, 0.05, (n, 3, 3))
        return v.reshape(-1, 3), np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    n = 20_000  # a cylinder of 40,000 triangles, height 2 and 3e-4 wide
    a = 2.0 * np.pi * np.arange(n) / n
    v = np.concatenate([np.stack([np.cos(a), np.sin(a), 0 * a + s], 1) for s in (-1.0, 1.0)])
    k, k1 = np.arange(n), (np.arange(n) + 1) % n
    return v, np.concatenate([np.stack([k, k1, k1 + n], 1),
                              np.stack([k, k1 + n, k + n], 1)]).astype(np.int32)


def _handles(monkeypatch, v, t, **kw):
    """A handle as a program creates it, and one that keeps the reference walk."""
    a = quest.SignedDistance(_t(v), _t(t), **kw)
    monkeypatch.setenv("AXSQ_SDF_MIXED_PASS2", "fp64")  # as by default
    return a, quest.SignedDistance(_t(v), _t(t), **kw)


@pytest.mark.parametrize("mesh,sizes", [
    ("flat", (16_385, 65_536, 65_537)), ("noise", (32_769, 65_536, 65_537)),
    ("cube", (65_537,)), ("small noise", (32_769, 131_073, 786_433)),
    ("soup", (32_769, 786_433)), ("slender", (131_072, 131_073))])
def test_outputs_are_the_reference_walks(monkeypatch, mesh, sizes):
    v, t = _mesh(mesh)
    rng = np.random.default_rng(2)
    q = rng.uniform(-1.5, 1.5, (sizes[-1], 3))
    q[::5] = v[t[rng.integers(0, t.shape[0], q[::5].shape[0]), 0]] + rng.normal(
        0.0, 1e-3, q[::5].shape)
    a, b = _handles(monkeypatch, v, t)
    o = orc.OracleSDF(v, t).eval(q[:4000], nthreads=8)
    # a large batch first, then smaller ones on the same mesh, and after a move
    for n in (*sizes[::-1], 4000):
        g, r = _eval(a, q[:n]), _eval(b, q[:n])
        for k in ("dist", "cp", "elem", "normal"):
            assert np.array_equal(g[k], r[k]), (n, k)
        _compare({k: x[:4000] for k, x in g.items()}, o)
    moved = v + np.array([0.2, 0.0, 0.1]) * np.sin(3.0 * v[:, [1]])
    a.updateVertices(_t(moved))
    b.updateVertices(_t(moved))
    for n in (sizes[0], sizes[-1]):
        g, r = _eval(a, q[:n]), _eval(b, q[:n])
        for k in ("dist", "cp", "elem", "normal"):
            assert np.array_equal(g[k], r[k]), (n, k)


@pytest.mark.parametrize("size", [1, 400])
def test_flat_quad_cells(monkeypatch, size):
    n = size
    i = np.arange(n)[:, None] * (n + 1) + np.arange(n)[None]
    quads = np.stack([i, i + n + 1, i + n + 2, i + 1], -1).reshape(-1).astype(np.int32)
    v, _ = _grid(n, lambda x, y: 0.0 * x)
    off = np.arange(0, quads.size + 1, 4, dtype=np.int32)
    a = quest.SignedDistance(_t(v), _t(quads), cell_offsets=_t(off))
    monkeypatch.setenv("AXSQ_SDF_MIXED_PASS2", "fp64")
    b = quest.SignedDistance(_t(v), _t(quads), cell_offsets=_t(off))
    q = np.random.default_rng(3).uniform(-1.5, 1.5, (70_000, 3))
    g, r = _eval(a, q), _eval(b, q)
    for k in ("dist", "cp", "elem", "normal"):
        assert np.array_equal(g[k], r[k]), k


def test_a_curved_surface_that_becomes_flat(monkeypatch):
    """What the boxes gained before the vertices moved does not decide afterwards."""
    flat, t = _mesh("flat")
    hill = flat + np.array([0.0, 0.0, 0.3]) * np.sin(3.0 * flat[:, [0]]) * np.cos(2.0 * flat[:, [1]])
    q = np.random.default_rng(4).uniform(-1.5, 1.5, (70_000, 3))
    a, b = _handles(monkeypatch, hill, t)
    for v in (hill, *[flat] * 9, hill):  # asked again by the eighth move
        a.updateVertices(_t(v))
        b.updateVertices(_t(v))
        for n in (70_000, 17_000):
            g, r = _eval(a, q[:n]), _eval(b, q[:n])
            for k in ("dist", "cp", "elem", "normal"):
                assert np.array_equal(g[k], r[k]), (n, k)


def _best(sdf, q):
    t = []
    for _ in range(6):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        sdf.computeDistances(q.shape[0], q)
        b.record()
        torch.cuda.synchronize()
        t.append(a.elapsed_time(b))
    return min(t)


@pytest.mark.parametrize("z", [0.0, 0.002])
def test_no_slower_than_the_reference_walk(monkeypatch, z):
    """1M queries about a flat and a noisy height field of 1.28M triangles: 1.0 and
    8.3 ms with the culled walk, 0.6 and 2.4 with the reference walk."""
    rng = np.random.default_rng(5)
    v, t = _grid(800, lambda x, y: rng.normal(0.0, 1.0, x.shape) * z)
    q = _t(rng.uniform(-1.5, 1.5, (1_000_000, 3)))
    a, b = _handles(monkeypatch, v, t)
    assert _best(a, q) < 1.4 * _best(b, q)
