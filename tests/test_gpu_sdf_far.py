"""Signed distances of meshes far from the origin, against the oracle, bit for bit:
the coordinates' own rounding is then larger than the margins that follow the
mesh's size."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from axom_amd import synth  # noqa: E402
from tests.test_gpu_sdf_cull import _check  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq", [2000, 40_000])
@pytest.mark.parametrize("shift", [1e10, 1e11, 4e11, 1e12])
@pytest.mark.parametrize("level", [2, 3])
def test_ties_far_from_the_origin(level, shift, nq):
    """Points over vertices and edges: which of the tied triangles wins is decided
    by the order in which a node's children are visited."""
    v, t, _ = synth.workload2(nq=1, level=level)
    rng = np.random.default_rng([level, nq])
    n = nq // 4
    f = t[rng.integers(0, t.shape[0], n)]
    mid = 0.5 * (v[f[:, 0]] + v[f[:, 1]])
    off = 1.0 + 10.0 ** rng.uniform(-3, 0.3, (n, 1))
    q = np.concatenate([v[f[:, 0]], mid, v[f[:, 1]] * off, mid * off])
    at = shift * np.array([1.0, -0.7, 0.9])
    _check(v + at, t, q + at, fp_modes=("fp64",))
