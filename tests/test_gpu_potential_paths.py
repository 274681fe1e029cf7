"""The potential on the split-FP16 matrix-core kernels: the bounds of the
distances that set their scale (from the bounding sphere for points outside it, from
a pass over all pairs otherwise), the general form of chunks without a double
layer, and the sizes where the FP32 matrix instructions take over, against the
FP64 oracle."""
import numpy as np
import pytest

import oracle
from baemm_amd import Helmholtz_HIP
from baemm_amd.meshes import fibonacci_sphere, icosphere, torus

pytestmark = pytest.mark.gpu

# FP32 arithmetic, as the other apply tests
NEAR = 3e-6

SLDL = [0.0, 1.0 - 0.5j, -0.75 + 1j, 0.0]
SL = [0.0, 1.0 - 0.5j, 0.0, 0.0]


def _meshes():
    V, T = icosphere(3)
    W, S = torus(1.0, 0.4, 30, 12)
    return {"sphere": (V, T), "cigar": (V * [5.0, 1.0, 0.5], T), "off the origin": (V + [8.0, -4.0, 2.0], T),
            "torus": (W, S)}


# points on a sphere around the mesh's bounding sphere of radius R: 1.02, 1.09 and 1.11
# (about the least gap of 0.1 R for the bound from the sphere), 1.5 R and 40 R
@pytest.mark.parametrize("mesh", list(_meshes()))
@pytest.mark.parametrize("far", [1.02, 1.09, 1.11, 1.5, 40.0])
@pytest.mark.parametrize("rows", [[SLDL, SLDL], [SLDL, SL], [SL, SL]])
def test_split_potential_outside(mesh, far, rows):
    V, T = _meshes()[mesh]
    centre = 0.5 * (V.min(0) + V.max(0))
    R = np.linalg.norm(V - centre, axis=1).max()
    pts = centre + fibonacci_sphere(150) * far * R
    K, wcs, kappa, coeff = 2, 5, [1.5, 3.0], np.array(rows).ravel()
    rng = np.random.default_rng(5)
    B = rng.standard_normal((V.shape[0], K * wcs)) + 1j * rng.standard_normal((V.shape[0], K * wcs))
    ref = oracle.apply_near_field(oracle.Mesh(V, T), 1.0, B, 0.0, np.zeros((150, K * wcs)), kappa, coeff, K * wcs, wcs,
                                  pts)
    # the coordinates are rounded to FP32: a shift of up to 2^-24 of their size, next
    # to the distance, and for the wave next to 1 / kappa
    gap = min((far - 1.0) * R, 1.0 / max(kappa))
    tol = NEAR + 2.0 ** -22 * np.abs(pts).max() / gap
    with Helmholtz_HIP(V, T) as H:
        for mode, kernel in (("mixed", 0), ("mixed", 1), ("mixed", 2), ("fp32", 2), ("fp32_mfma", 2)):
            H.SetPrecision(mode)
            H.SetMixedKernel(kernel)
            U = np.zeros((150, K * wcs), np.complex128)
            H.ApplyNearFieldOperators_PL(1.0, B, 0.0, U, kappa, coeff, K * wcs, wcs, evaluation_points=pts)
            assert np.linalg.norm(U - ref) < tol * np.linalg.norm(ref), (mode, kernel)


def test_split_potential_where_coordinates_round():
    """At 2.5e6 from the origin FP32 coordinates are 0.25 apart: a point 0.13 off the
    bounding sphere lands 0.007 from a centroid.  All kernels see the same rounded
    coordinates; the scale has to hold for these distances."""
    V, T = icosphere(3)
    off = np.array([2.5e6, 0.3, 0.1])
    pts = off + 1.13 * fibonacci_sphere(800)
    W, kappa, coeff = 4, [0.05], np.array(SLDL)
    rng = np.random.default_rng(6)
    B = rng.standard_normal((V.shape[0], W)) + 1j * rng.standard_normal((V.shape[0], W))
    out = []
    with Helmholtz_HIP(V + off, T) as H:
        for mode, kernel in (("fp32", 2), ("mixed", 0), ("mixed", 1)):
            H.SetPrecision(mode)
            H.SetMixedKernel(kernel)
            U = np.zeros((800, W), np.complex128)
            H.ApplyNearFieldOperators_PL(1.0, B, 0.0, U, kappa, coeff, W, W, evaluation_points=pts)
            out.append(U)
    assert np.all(np.isfinite(out[0]))
    for U in out[1:]:
        assert np.linalg.norm(U - out[0]) < NEAR * np.linalg.norm(out[0])


def test_split_potential_keeps_points_apart():
    """A point that is not finite spoils its own row alone."""
    V, T = torus(1.0, 0.4, 40, 16)
    pts = 2.0 * fibonacci_sphere(200)
    W, kappa, coeff = 4, [2.0], np.array(SLDL)
    rng = np.random.default_rng(7)
    B = rng.standard_normal((V.shape[0], W)) + 1j * rng.standard_normal((V.shape[0], W))
    ref = oracle.apply_near_field(oracle.Mesh(V, T), 1.0, B, 0.0, np.zeros((200, W)), kappa, coeff, W, W, pts)
    bad = pts.copy()
    bad[17] = np.nan
    bad[90, 1] = np.inf
    good = np.setdiff1d(np.arange(200), [17, 90])
    with Helmholtz_HIP(V, T) as H:
        for mode, kernel in (("fp32", 2), ("mixed", 0), ("mixed", 1), ("fp32_mfma", 2)):
            H.SetPrecision(mode)
            H.SetMixedKernel(kernel)
            U = np.zeros((200, W), np.complex128)
            H.ApplyNearFieldOperators_PL(1.0, B, 0.0, U, kappa, coeff, W, W, evaluation_points=bad)
            assert np.linalg.norm(U[good] - ref[good]) < NEAR * np.linalg.norm(ref[good]), (mode, kernel)


# 5,400 triangles: just below and above the pairs where FP32_MFMA goes over to the
# split products, and K = 2 on either side of half as many points
@pytest.mark.parametrize("K,P", [(1, 7407), (1, 7408), (2, 3703), (2, 3704)])
def test_fp32_mfma_potential_at_its_rule(K, P):
    V, T = torus(1.0, 0.4, 90, 30)
    W, kappa, coeff = 6 * K, [2.0, 3.5][:K], np.array([SLDL] * K).ravel()
    rng = np.random.default_rng(P)
    B = rng.standard_normal((V.shape[0], W)) + 1j * rng.standard_normal((V.shape[0], W))
    pts = fibonacci_sphere(P) * rng.uniform(1.7, 2.5, (P, 1))
    some = np.append(rng.choice(P - 1, 200, replace=False), P - 1)
    ref = oracle.apply_near_field(oracle.Mesh(V, T), 1.0, B, 0.0, np.zeros((201, W)), kappa, coeff, W, 6, pts[some])
    with Helmholtz_HIP(V, T) as H:
        H.SetPrecision("fp32_mfma")
        U = np.zeros((P, W), np.complex128)
        H.ApplyNearFieldOperators_PL(1.0, B, 0.0, U, kappa, coeff, W, 6, evaluation_points=pts)
    assert np.linalg.norm(U[some] - ref) < NEAR * np.linalg.norm(ref)
