"""The two pair kernels of the tangent-point metric (matrix cores where every
distance and weight is a normal number, vector ALU elsewhere) at the edges of
their tiles and of the rule, against the FP64 oracle."""
import numpy as np
import pytest

import oracle
from baemm_amd import Helmholtz_HIP
from baemm_amd.meshes import torus

pytestmark = pytest.mark.gpu

# the bound of the metric's other tests: weights to a few 2^-24 times the exponent,
# FP32 sums
NEAR = 5e-6


# triangles 2 a b around a wave (64), a work-group (256), the four sources of a load
# (66, 258, 510) and the segments
@pytest.mark.parametrize("a,b", [(8, 4), (11, 3), (16, 8), (43, 3), (17, 15), (40, 16)])
@pytest.mark.parametrize("q,p", [(6.0, 12.0), (2.5, 4.75)])
# 1: ordinary; 1e-9 and 1e9: squared distances outside the rule's range
@pytest.mark.parametrize("size", [1.0, 1e-9, 1e9])
def test_metric_at_tile_edges_and_sizes(a, b, q, p, size):
    V, T = torus(1.0, 0.4, a, b)
    rng = np.random.default_rng(a + b)
    V = size * (V + 0.01 * rng.standard_normal(V.shape) * (a < 20))
    m = oracle.Mesh(V, T)
    x = rng.standard_normal((m.nv, 3))
    ref = (oracle.tp_metric(m, q, p) @ x.ravel()).reshape(-1, 3)
    with Helmholtz_HIP(V, T) as H:
        y = H.TangentPointMetric(x, q, p)
    assert np.linalg.norm(y - ref) < NEAR * np.linalg.norm(ref)


def test_metric_keeps_components_apart():
    """A NaN in one component leaves the other two as they are."""
    V, T = torus(1.0, 0.4, 20, 9)
    rng = np.random.default_rng(5)
    x = rng.standard_normal((V.shape[0], 3))
    bad = x.copy()
    bad[11, 1] = np.nan
    with Helmholtz_HIP(V, T) as H:
        y, z = H.TangentPointMetric(x, 6.0, 12.0), H.TangentPointMetric(bad, 6.0, 12.0)
    assert np.array_equal(y[:, [0, 2]], z[:, [0, 2]])
    assert not np.any(np.isfinite(z[:, 1]))
