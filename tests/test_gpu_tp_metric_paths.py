"""The two pair kernels of the tangent-point metric (matrix cores where the least
distance of two centroids is not too small next to the mesh, vector ALU
elsewhere) at the edges of their tiles and of the rule, against the FP64 oracle."""
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
# 1: ordinary; 1e-9 and 1e9: weights whose FP32 products need scaled lengths
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


# meshes of the size of a light wave in metres up to that of a planet's orbit: second
# weights of 1e45 and 1e-38 without the scaled lengths
@pytest.mark.parametrize("q,p", [(6.0, 12.0), (2.5, 4.75), (3.0, 1.5)])
@pytest.mark.parametrize("size", [1e-11, 1e-8, 3e-8, 1e-7, 1e-6, 1e7, 1e8, 5e8, 1e12])
def test_metric_at_any_size(q, p, size):
    V, T = torus(1.0, 0.4, 17, 15)
    x = np.random.default_rng(2).standard_normal((V.shape[0], 3))
    ref = (oracle.tp_metric(oracle.Mesh(size * V, T), q, p) @ x.ravel()).reshape(-1, 3)
    with Helmholtz_HIP(size * V, T) as H:
        y = H.TangentPointMetric(x, q, p)
    assert np.linalg.norm(y - ref) < NEAR * np.linalg.norm(ref)


# two facing sheets around the least distance of the rule (5.7e-7 here).  Every
# facing pair has the same distance, so the roundings of log2 r2 and of its product
# with the exponent do not average: an ulp of each on top of the bound
@pytest.mark.parametrize("gap", [1e-2, 1e-4, 1e-6, 2e-7, 1e-7])
def test_metric_of_two_facing_sheets(gap):
    n = 9
    u = np.linspace(-0.5, 0.5, n)
    X, Y = np.meshgrid(u, u, indexing="ij")
    k = np.arange(n * n).reshape(n, n)
    a, b, c, d = (v.ravel() for v in (k[:-1, :-1], k[1:, :-1], k[1:, 1:], k[:-1, 1:]))
    T = np.vstack([np.stack([a, b, c], 1), np.stack([a, c, d], 1)])
    sheet = np.stack([X.ravel(), Y.ravel(), 0.0 * X.ravel()], 1)
    V = np.vstack([sheet, sheet + [0.0, 0.0, gap]])
    T = np.vstack([T, T[:, ::-1] + n * n])
    x = np.random.default_rng(4).standard_normal((V.shape[0], 3))
    ref = (oracle.tp_metric(oracle.Mesh(V, T), 6.0, 12.0) @ x.ravel()).reshape(-1, 3)
    with Helmholtz_HIP(V, T) as H:
        y = H.TangentPointMetric(x, 6.0, 12.0)
    expo, lg = 5 / 3, abs(2 * np.log2(gap))
    ulps = expo * np.spacing(np.float32(lg)) + np.spacing(np.float32(expo * lg))
    assert np.linalg.norm(y - ref) < (NEAR + np.log(2) * ulps) * np.linalg.norm(ref)
