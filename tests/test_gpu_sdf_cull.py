"""The culled signed-distance walk (oriented child boxes, one lane or one wave
per query) against the oracle: distances, closest points, signs and elements
bit for bit, unit normals within 1e-12 (device acos may differ from glibc by
an ulp; the walk itself adds the same terms in the same order).

The sizes are those where the dispatch or a kernel changes: a wave and one
more or less, the small-batch limit and one more, meshes at the node-size
classes of the box build (8 and 1,024 leaves), one triangle; and the inputs
those the walk hands on to the reference walk or to the whole-wave walk:
queries near the centre of a closed surface, far away, not finite, on the
surface and at shared vertices, triangles without a useful tolerance."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from axom_amd import quest, synth  # noqa: E402
from oracle import oracle as orc  # noqa: E402
from tests import refmeshes  # noqa: E402
from tests.test_gpu_sdf import _compare, _eval, _t  # noqa: E402
from tests.test_oracle_quads import mixed_cells, quad_cells  # noqa: E402

pytestmark = pytest.mark.gpu


def _check(v, t, q, watertight=True, sign=True, fp_modes=("fp64", "fp32"), sdf=None):
    o = orc.OracleSDF(v, t, watertight=watertight, compute_sign=sign).eval(q, nthreads=8)
    for fp in fp_modes:
        g = _eval(quest.SignedDistance(_t(v), _t(t), watertight, sign, fp_mode=fp), q, fp)
        if fp == "fp64":
            _compare(g, o)
        else:  # its own order among tied triangles: the distance and side are the same
            assert np.array_equal(g["dist"], o["dist"])


@pytest.mark.parametrize("nq", [1, 2, 63, 64, 65, 1000, 4096, 4097, 16_383, 16_384, 16_385,
                                16_449, 65_536, 65_537])
def test_batch_sizes(nq):
    v, t, q = synth.workload2(nq=nq, level=2)
    _check(v, t, q)


@pytest.mark.parametrize("nu,nv", [(3, 3), (4, 8), (5, 8), (16, 32), (17, 31), (96, 64)])
def test_mesh_sizes_around_the_node_classes(nu, nv):
    v, t = synth.torus(nu, nv)
    q = np.concatenate([synth.surface_samples(v, t, 5, 0, 5000, -0.01, 0.01),
                        synth.uniform(5, 1, 45_000, -1.5, 1.5).reshape(-1, 3)])
    _check(v, t, q)
    _check(v, t, q[:1500], watertight=False)
    _check(v, t, q[-1500:], sign=False)


@pytest.mark.parametrize("ntri", [1, 2, 7, 8, 9])
@pytest.mark.parametrize("nq", [100, 17_000])
def test_few_triangles(ntri, nq):
    rng = np.random.default_rng(ntri)
    v = rng.uniform(-1, 1, (3 * ntri, 3))
    t = np.arange(3 * ntri, dtype=np.int32).reshape(-1, 3)
    q = np.concatenate([rng.uniform(-2, 2, (nq - 10, 3)), v[rng.integers(0, 3 * ntri, 10)]])
    _check(v, t, q, watertight=False)


@pytest.mark.parametrize("nq", [3000, 30_000, 70_000])
def test_long_walks_and_centre(nq):
    """A round sphere from inside: most of the surface at one distance."""
    v, t = synth.icosphere(5)
    q = np.concatenate([synth.uniform(21, 0, 3 * (nq - 1200), -0.02, 0.02).reshape(-1, 3),
                        synth.uniform(21, 1, 3 * 1000, -1e-4, 1e-4).reshape(-1, 3),
                        np.zeros((100, 3)), 1e-7 * synth.uniform(21, 2, 300, -1, 1).reshape(-1, 3)])
    _check(v, t, q)


@pytest.mark.parametrize("nq", [2000, 20_000])
def test_vertices_edges_and_surface_points(nq):
    v, t, _ = synth.workload2(nq=1, level=3)
    rng = np.random.default_rng(8)
    f = t[rng.integers(0, t.shape[0], nq // 4)]
    mid = 0.5 * (v[f[:, 0]] + v[f[:, 1]])
    face = (v[f[:, 0]] + v[f[:, 1]] + v[f[:, 2]]) / 3.0
    out = v[f[:, 0]] * rng.uniform(1.0, 2.0, (nq // 4, 1))
    _check(v, t, np.concatenate([v[f[:, 2]], mid, face, out, out + 1e-7]))


def test_planar_cube_of_quads_and_triangles():
    """Axis-aligned faces: boxes of no thickness, many equal distances."""
    v, quads = synth.cube_sphere(5, project=False)
    g = np.linspace(-2.0, 2.0, 26)
    q = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    t = np.concatenate([quads[:, [0, 1, 2]], quads[:, [0, 2, 3]]])
    _check(v, t, q)
    for cells in (quad_cells(quads), mixed_cells(quads)[:2]):
        for n in (q.shape[0], 500):  # 17,576: a lane each
            s = quest.SignedDistance(_t(v), _t(cells[0]), cell_offsets=_t(cells[1]))
            o = orc.OracleSDF(v, cells[0], cell_offsets=cells[1]).eval(q[:n], nthreads=8)
            _compare(_eval(s, q[:n]), o)


@pytest.mark.parametrize("nq", [2000, 20_000])
def test_far_and_non_finite_queries(nq):
    v, t, q = synth.workload2(nq=nq, level=4)
    q = q.copy()
    q[::7] *= 20.0
    q[3::70] *= 1e6
    q[5::210] = np.nan
    q[6::210, 1] = np.inf
    _check(v, t, q)


@pytest.mark.parametrize("scale,shift", [(1e-3, 0.0), (1e4, 0.0), (1.0, 1e6), (1e-6, 0.0),
                                         (2e-2, 3.0)])
def test_scaled_and_shifted_meshes(scale, shift):
    v, t, q = synth.workload2(nq=18_000, level=4)
    for n in (18_000, 1000):
        _check(v * scale + shift, t, q[:n] * scale + shift)


@pytest.mark.parametrize("nq", [12_000, 20_000])
@pytest.mark.parametrize("level,scale,shift", [(2, 1.0, 0.0), (5, 1.0, 0.0), (5, 1.0, 50.0),
                                               (5, 30.0, 1e5), (6, 0.01, 0.0)])
def test_fp32_order_is_the_reference_walks(monkeypatch, level, scale, shift, nq):
    """With FP32 traversal the first of several tied triangles wins, in the order
    of float comparisons: the reference walk's own outputs, bit for bit, where
    queries tie (vertices, edges, points over them) near, far and in between."""
    v, t, _ = synth.workload2(nq=1, level=level)
    rng = np.random.default_rng(nq + level)
    n = nq // 4
    f = t[rng.integers(0, t.shape[0], n)]
    mid = 0.5 * (v[f[:, 0]] + v[f[:, 1]])
    off = 1.0 + 10.0 ** rng.uniform(-6, 0.3, (n, 1))
    q = np.concatenate([v[f[:, 0]], mid, v[f[:, 1]] * off, mid * off])
    v, q = v * scale + shift, q * scale + shift
    g = _eval(quest.SignedDistance(_t(v), _t(t), fp_mode="fp32"), q, "fp32")
    monkeypatch.setenv("AXSQ_SDF_BUDGET", "65536")  # the reference walk, on FP32 nodes alone
    sdf = quest.SignedDistance(_t(v), _t(t), fp_mode="fp32")
    r = _eval(sdf, q, "fp32")
    assert sdf.lastSuspended() == 0
    for k in ("dist", "cp", "elem", "normal"):
        assert np.array_equal(g[k], r[k]), k


@pytest.mark.parametrize("dy", [5e-4, 1e-5, 1e-8, 0.0])
def test_children_split_along_the_normal(dy):
    """Two triangles stacked along their mean normal, their centroids a little
    apart sideways, too: queries beside them, at one distance from both, see the
    nearer centroid by that sideways part alone."""
    v = np.array([[0, 1, 0], [1, 1, 0], [0.5, 0, 0],
                  [0, 1, 1], [1, 1, 1], [0.5, -2 * dy, 1 + 0.25 * dy]])
    t = np.array([[0, 1, 2], [3, 4, 5]], np.int32)
    rng = np.random.default_rng(3)
    q = np.stack([rng.uniform(0.1, 0.9, 20_000), rng.uniform(1.1, 3.0, 20_000),
                  np.full(20_000, 0.5)], 1)
    for n in (20_000, 500):
        _check(v, t, q[:n], watertight=False)


def test_sliver_and_repeated_corners():
    """Triangles with equal corners keep the boxes; a sliver without a useful
    closest-point tolerance sends the mesh to the reference walk."""
    v, t, q = synth.workload2(nq=18_000, level=4)
    rep = np.stack([t[:50, 0], t[:50, 0], t[:50, 1]], 1)
    _check(v, np.concatenate([t, rep]).astype(np.int32), q)
    nv = v.shape[0]
    v2 = np.concatenate([v, 0.5 * (v[t[:5, 0]] + v[t[:5, 1]])])
    sl = np.stack([t[:5, 0], t[:5, 1], nv + np.arange(5)], 1)
    _check(v2, np.concatenate([t, sl]).astype(np.int32), q)


def test_many_terms_at_a_pole():
    v, t = refmeshes.sphere_uv_mesh([0.0, 0.0, 0.0], 1.0, 25, 20)
    z = np.linspace(1.05, 2.0, 3000)
    q = np.concatenate([np.stack([0 * z, 0 * z, z], 1), np.stack([0 * z, 0 * z, -z], 1),
                        synth.uniform(4, 1, 45_000, -1.0, 1.0).reshape(-1, 3)])
    _check(v, t, q)
    _check(v, t, q[:300])


def test_moved_vertices_rebuild_the_boxes():
    v, t, q = synth.workload2(nq=20_000, level=4)
    sdf = quest.SignedDistance(_t(v), _t(t))
    _compare(_eval(sdf, q), orc.OracleSDF(v, t).eval(q, nthreads=8))
    v2 = v * np.array([1.3, 0.7, 1.0])
    sdf.updateVertices(_t(v2))
    _compare(_eval(sdf, q), orc.OracleSDF(v2, t).eval(q, nthreads=8))
    _compare(_eval(sdf, q[:5]), orc.OracleSDF(v2, t).eval(q[:5]))


def test_strides_and_streams():
    v, t, q = synth.workload2(nq=18_000, level=4)
    o = orc.OracleSDF(v, t).eval(q, nthreads=8)
    sdf = quest.SignedDistance(_t(v), _t(t))
    soa = tuple(_t(q[:, k]) for k in range(3))
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for s in streams:
        with torch.cuda.stream(s):
            d = sdf.computeDistances(q.shape[0], soa)
        s.synchronize()
        assert np.array_equal(d.cpu().numpy(), o["dist"])
