"""The stable radix sort at the sizes where its tiles and paths change, through
the two results it decides: the tree arrays of a large build (Morton keys sorted,
equal keys in input order) and the adjoint's sums over queries of a triangle in
query order. Integers and bits: no tolerance."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from axom_amd import quest, spin, synth  # noqa: E402
from oracle import oracle as orc  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=DEV)


# past the build's small sort: tiles of 4,096 keys, their rows scanned 1,024
# tiles at a time (4,194,304 keys are 1,024 tiles)
@pytest.mark.parametrize("n", [262_145, 266_240, 266_241, 1_000_003])
def test_large_build_order(n):
    rng = np.random.default_rng(n)
    c = np.round(rng.random((n, 3)) * 40) / 40  # few cells: long runs of equal keys
    boxes = np.concatenate([c, c + 0.01], 1)
    g, o = spin.BVH(_t(boxes)), orc.OracleBVH(boxes, 1.000123)
    ex, oe = g.export(), o.export()
    assert np.array_equal(ex["mcodes"].cpu().numpy().view(np.uint32), oe["mcodes"])
    assert np.array_equal(ex["leafs"].cpu().numpy(), oe["leafs"])


@pytest.mark.parametrize("nq", [255, 1025, 65_537, 262_144, 262_145, 270_001, 4_198_401])
def test_queries_of_a_triangle_in_order(nq):
    """A triangle's vertex gradient is the sum over its queries in ascending
    order: given the same queries in the sequential order of one lane."""
    v, t = synth.icosphere(1)  # 80 triangles: thousands of queries each
    rng = np.random.default_rng(nq)
    p = rng.uniform(-1.5, 1.5, (nq, 3))
    s = quest.SignedDistance(_t(v), _t(t))
    q = _t(p)
    elem = torch.empty(nq, dtype=torch.int32, device=DEV)
    d = s.computeDistances(nq, q, outElem=elem)
    gout = torch.ones(nq, dtype=torch.float32, device=DEV)
    gq, gv = s.backward(q, d, elem, gout)
    # two runs agree bit for bit, and so does the sum over the same queries
    # given one triangle at a time
    gq2, gv2 = s.backward(q, d, elem, gout)
    assert torch.equal(gq, gq2) and torch.equal(gv, gv2)
    e = elem.cpu().numpy()
    order = np.argsort(e, kind="stable")
    i = torch.as_tensor(order, device=DEV)
    gq3, gv3 = s.backward(q[i].contiguous(), d[i].contiguous(), elem[i].contiguous(), gout)
    assert torch.equal(gq3, gq[i]) and torch.equal(gv3, gv)


@pytest.mark.parametrize("few", [True, False])
def test_adjoint_sums_of_short_and_long_segments(few):
    """Vertex gradients are the sequential sums over each triangle's queries,
    with no query, a few, and a wave's batch of 64 more or less, over triangles
    that share a wave or not; without the vertices' part the
    query gradients are the same, and an id out of range is refused either way."""
    v, t = synth.icosphere(2)
    nt = t.shape[0]
    # 320 triangles: below and above 16 queries a triangle on average
    counts = [0, 0, 1, 8, 9, 63, 64, 65, 95, 97, 128, 129, 1000] + [3 if few else 20] * (nt - 15)
    counts += [0, 0]
    rng = np.random.default_rng(3)
    elem = rng.permutation(np.repeat(np.arange(nt), counts)).astype(np.int32)
    nq = elem.size
    tri = v[t[elem]]
    w = rng.dirichlet(np.ones(3), nq)
    p = np.einsum("ij,ijk->ik", w, tri) * rng.uniform(1.05, 1.5, (nq, 1))
    s = quest.SignedDistance(_t(v), _t(t))
    q, e = _t(p), _t(elem)
    d = torch.ones(nq, dtype=torch.float64, device=DEV)
    gout = _t(rng.normal(size=nq).astype(np.float32))
    gq, gv = s.backward(q, d, e, gout)
    only_q, none = s.backward(q, d, e, gout, want_vertices=False)
    assert none is None and torch.equal(only_q, gq)
    ogq, ogv = orc.OracleSDF(v, t).backward(p, d.cpu().numpy(), elem, gout.cpu().numpy())
    assert np.array_equal(gq.cpu().numpy(), ogq) and np.array_equal(gv.cpu().numpy(), ogv)
    e[5] = nt
    for wv in (True, False):
        with pytest.raises(RuntimeError):
            s.backward(q, d, e, gout, want_vertices=wv)
