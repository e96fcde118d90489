"""Saved walks that reach leaves before any subtree of theirs: a triangle with one
corner far away is a leaf beside all others, so that it waits on the stack when the
step budget runs out. Against the oracle, bit for bit."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from axom_amd import quest  # noqa: E402
from oracle import oracle as orc  # noqa: E402
from tests.test_gpu_sdf import _compare, _eval, _t  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp,cells", [("fp64", False), ("fp32", False), ("fp64", True)])
@pytest.mark.parametrize("far", [100.0, 1e4, 1e9])
@pytest.mark.parametrize("budget", [5, 20, 50, 100, 300])
def test_leaves_on_the_saved_stack(monkeypatch, fp, cells, budget, far):
    rng = np.random.default_rng(6)
    n = 2000
    v = rng.uniform(-1, 1, (n, 1, 3)) + rng.normal(0.0, 0.05, (n, 3, 3))
    v[7, 2] = far * np.array([1.0, 0.9, -1.1])
    q = v[7, 2] * rng.uniform(-0.1, 1.1, (4000, 1)) + far * 10.0 ** rng.uniform(-3, 0, (4000, 1)) \
        * rng.normal(size=(4000, 3))
    v, t = v.reshape(-1, 3), np.arange(3 * n, dtype=np.int32).reshape(n, 3)
    kw = {}
    if cells:  # one quad among triangles
        conn = np.concatenate([[0, 1, 2, 5], t[2:].reshape(-1)]).astype(np.int32)
        off = np.concatenate([[0], np.arange(4, conn.size + 1, 3)]).astype(np.int32)
        o = orc.OracleSDF(v, conn, cell_offsets=off)
        t, kw = conn, dict(cell_offsets=_t(off))
    else:
        o = orc.OracleSDF(v, t)
    o = o.eval(q, nthreads=8)
    monkeypatch.setenv("AXSQ_SDF_BUDGET", str(budget))
    sdf = quest.SignedDistance(_t(v), _t(t), fp_mode=fp, **kw)
    g = _eval(sdf, q, fp)
    if fp == "fp64":
        _compare(g, o)
    else:  # its own order among tied triangles
        assert np.array_equal(np.abs(g["dist"]), np.abs(o["dist"]))
    assert sdf.lastSuspended() > 0 or (budget >= 100 and far == 100.0)  # else short walks
