"""The one-launch PCG of the mass inverse at the edges of its variants (rows per
thread, groups of entries per row, the largest mesh it takes) and the
multi-block PCG beyond them."""
import numpy as np
import pytest
import scipy.sparse as sp

from baemm_amd import Helmholtz_HIP
from baemm_amd.meshes import torus

pytestmark = pytest.mark.gpu

# The lumped mass matrix preconditions element by element to a condition number
# of at most 4 (eigenvalues in [1/4, 1]), so 20 steps reduce the error in the
# energy norm by 2 * 3^-20 = 5.7e-10; the residual norm differs from it by the
# square roots of the condition and of the areas' ratio, below 10 together.
BOUND = 6e-9


def _residuals(V, T, X):
    with Helmholtz_HIP(V, T) as H:
        ptr, idx, val = H.MassMatrix()
        Y = np.zeros_like(X)
        H.ApplyMassInverse(X, Y, 1e-10)
    M = sp.csr_matrix((val, idx, ptr), shape=(V.shape[0],) * 2)
    return np.linalg.norm(M @ Y - X, axis=0), np.linalg.norm(X, axis=0)


@pytest.mark.parametrize("a,b", [(5, 5), (16, 16), (37, 7), (32, 16), (27, 19), (32, 32), (41, 25), (64, 32), (683, 3),
                                 (64, 48), (75, 41), (64, 64), (241, 17), (96, 64), (125, 50), (128, 64), (149, 55),
                                 (128, 96), (160, 77), (128, 128), (164, 100), (204, 100), (202, 101)])
def test_vertex_counts(a, b):
    V, T = torus(1.0, 0.4, a, b)
    rng = np.random.default_rng(a)
    for ncols in (1, 11):
        res, norm = _residuals(V, T, rng.standard_normal((a * b, ncols)))
        assert np.all(res <= BOUND * norm), (a * b, ncols, (res / norm).max())


@pytest.mark.parametrize("k", [3, 7, 8, 12, 40, 600, 1018, 1019, 1500])
def test_long_rows(k):
    """A double cone over a ring of k vertices: two rows of k + 1 entries, the
    others of five."""
    phi = 2 * np.pi * np.arange(k) / k
    V = np.vstack([np.stack([np.cos(phi), np.sin(phi), 0 * phi], 1), [[0, 0, 1.0], [0, 0, -1.0]]])
    i, j = np.arange(k), (np.arange(k) + 1) % k
    T = np.vstack([np.stack([i, j, 0 * i + k], 1), np.stack([j, i, 0 * i + k + 1], 1)])
    rng = np.random.default_rng(k)
    X = rng.standard_normal((k + 2, 3)) + 1j * rng.standard_normal((k + 2, 3))
    X[:, 1] = 0.0   # a zero column stays zero
    res, norm = _residuals(V, T, X)
    assert np.all(res <= 10 * BOUND * norm)


def test_columns_do_not_share_faults_and_strides_hold():
    V, T = torus(1.0, 0.4, 60, 40)
    n = V.shape[0]
    rng = np.random.default_rng(1)
    X = rng.standard_normal((n, 9))
    with Helmholtz_HIP(V, T) as H:
        clean = np.zeros((n, 9))
        H.ApplyMassInverse(X, clean, 1e-10)
        bad = X.copy()
        bad[3, 4] = np.nan
        bad[5, 6] = np.inf
        out = np.full((n, 13), 7.0)
        H.ApplyMassInverse(bad, out[:, :9], 1e-10)
    good = [0, 1, 2, 3, 5, 7, 8]
    assert np.array_equal(out[:, good], clean[:, good])
    assert np.all(out[:, 9:] == 7.0)
