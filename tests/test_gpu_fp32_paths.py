"""The kernels the FP32 precision chooses from (vector ALU, split FP16 on the
matrix cores, FP32 on the matrix cores) at the edges of the rule and of the
kernels' tiles, against the FP64 oracle."""
import numpy as np
import pytest

import oracle
from baemm_amd import Helmholtz_HIP
from baemm_amd.meshes import fibonacci_sphere, torus

pytestmark = pytest.mark.gpu

# FP32 arithmetic: geometry and kernel values to a few 2^-24, sums of up to
# 2,048 sources in FP32; the bound the apply tests use for every precision
NEAR = 3e-6


def _apply(H, B, kappa, coeff, W, wcs):
    C = np.zeros_like(B)
    H.ApplyBoundaryOperators_PL(1.0, B, 0.0, C, kappa, coeff, W, wcs)
    return C


# triangles 2 a b around the multiples of the 128- and 256-target tiles and the
# mesh sizes where the rule changes kernels (256 triangles from 9 columns on,
# 4,096 with 5 to 8, 8,192 below); three chunks (a launch of two and one of one)
@pytest.mark.parametrize("a,b", [(11, 11), (16, 8), (43, 3), (64, 32), (205, 10), (64, 64), (273, 15)])
@pytest.mark.parametrize("K,wcs", [(1, 1), (1, 4), (2, 5), (1, 8), (1, 9), (3, 16), (1, 17), (1, 64)])
@pytest.mark.parametrize("row", [(0.5, 0, 1, 0), (0.25, 1 - 0.5j, -0.75 + 1j, 0.3)])
def test_fp32_apply_at_tile_and_rule_edges(a, b, K, wcs, row):
    V, T = torus(1.0, 0.4, a, b)
    W, kappa = K * wcs, [1.5 + 0.25 * q for q in range(K)]
    coeff = np.array(row * K, np.complex128)
    rng = np.random.default_rng(a + 7 * W)
    B = rng.standard_normal((V.shape[0], W)) + 1j * rng.standard_normal((V.shape[0], W))
    m = oracle.Mesh(V, T)
    rows = rng.choice(V.shape[0], 24, replace=False)
    ref = oracle.apply_boundary_rows(m, 1.0, B, 0.0, np.zeros((24, W), np.complex128), kappa, coeff, W, wcs, rows)
    with Helmholtz_HIP(V, T) as H:
        for mode in ("fp32", "fp32_mfma"):
            H.SetPrecision(mode)
            C = _apply(H, B, kappa, coeff, W, wcs)
            assert np.linalg.norm(C[rows] - ref) < NEAR * np.linalg.norm(ref), mode


@pytest.mark.parametrize("wcs", [4, 16])
@pytest.mark.parametrize("gap", [1e-5, 0.0])
def test_fp32_apply_where_two_centroids_nearly_or_fully_coincide(wcs, gap):
    """Two parallel copies of a triangle at distance gap (0: coincident
    centroids, whose own rows are not finite): the least distance no longer fits
    the FP16 range, and every other row keeps FP32 accuracy."""
    V, T = torus(1.0, 0.4, 40, 16)
    t = V[T[5]]
    n = np.cross(t[1] - t[0], t[2] - t[0])
    n /= np.linalg.norm(n)
    V = np.vstack([V, t + gap * n])
    T = np.vstack([T, [[len(V) - 3, len(V) - 2, len(V) - 1]]])
    kappa, coeff = [2.0], np.array([0.5, -2j, 1.0, 0.0])
    rng = np.random.default_rng(wcs)
    B = rng.standard_normal((V.shape[0], wcs)) + 1j * rng.standard_normal((V.shape[0], wcs))
    m = oracle.Mesh(V, T)
    touched = set(T[5]) | set(T[-1])
    rows = np.array([v for v in range(0, V.shape[0], 9) if v not in touched])
    ref = oracle.apply_boundary_rows(m, 1.0, B, 0.0, np.zeros((len(rows), wcs), np.complex128), kappa, coeff, wcs,
                                     wcs, rows)
    with Helmholtz_HIP(V, T) as H:
        for mode in ("fp32", "fp32_mfma"):
            H.SetPrecision(mode)
            C = _apply(H, B, kappa, coeff, wcs, wcs)
            assert np.linalg.norm(C[rows] - ref) < NEAR * np.linalg.norm(ref), mode


def test_fp32_columns_do_not_share_range_or_faults():
    """Columns of very different size, an all-zero column and one with a NaN and
    an Inf: each column depends on itself alone."""
    V, T = torus(1.0, 0.4, 48, 24)
    W = 16
    rng = np.random.default_rng(3)
    B = rng.standard_normal((V.shape[0], W)) + 1j * rng.standard_normal((V.shape[0], W))
    B[:, 1] *= 1e-30
    B[:, 2] *= 1e30
    B[:, 3] = 0.0
    bad = B.copy()
    bad[7, 4] = np.nan
    bad[9, 5] = np.inf
    kappa, coeff = [3.0], np.array([0.5, -3j, 1.0, 0.0])
    ref = oracle.apply_boundary(oracle.Mesh(V, T), 1.0, B, 0.0, np.zeros_like(B), kappa, coeff, W, W)
    with Helmholtz_HIP(V, T) as H:
        C = _apply(H, B, kappa, coeff, W, W)
        D = _apply(H, bad, kappa, coeff, W, W)
    for k in range(W):
        if k == 3:
            assert np.all(C[:, k] == 0.0)
            continue
        assert np.linalg.norm(C[:, k] - ref[:, k]) < NEAR * np.linalg.norm(ref[:, k]), k
    good = [k for k in range(W) if k not in (4, 5)]
    assert np.array_equal(D[:, good], C[:, good])
    assert not np.any(np.isfinite(D[:, 4])) and not np.any(np.isfinite(D[:, 5]))


# the mixed precision on small meshes takes the vector-ALU kernel with segments
# of 16 sources, and the matrix cores once a kernel or segments are set: 64, 66,
# 264, 896, 900 and 2,750 triangles around one source block and the rule's sizes,
# from one wave to sixteen of the segment sums
DBL, ADJ, ALL = (0.5, -1j, 1, 0), (0.5, -1j, 0, 1), (0.25, 1 - 0.5j, -0.75 + 1j, 0.3)


# several wave numbers: at and above the sizes from which MIXED is on the matrix
# cores; all operators: the wave-specialised kernel only in more than 16 columns, on up
# to 40 tiles
@pytest.mark.parametrize("a,b,K,wcs,row,kernel", [
    (6, 5, 4, 16, DBL, 0), (6, 5, 7, 9, DBL, 0), (16, 8, 8, 8, DBL, 0), (32, 16, 4, 8, DBL, 0), (37, 23, 5, 5, DBL, 0),
    (64, 32, 4, 4, DBL, 0), (64, 32, 6, 1, DBL, 0), (64, 20, 2, 8, DBL, 0), (64, 20, 3, 5, ADJ, 0), (64, 16, 4, 3, ADJ, 0),
    (64, 40, 3, 4, ADJ, 0), (16, 8, 4, 16, ALL, 0), (64, 48, 4, 3, ALL, 0), (64, 64, 3, 8, ALL, 0),
    (68, 51, 2, 16, ALL, 0), (16, 8, 2, 17, ALL, 1), (64, 40, 1, 24, ALL, 1), (64, 40, 1, 33, ALL, 1),
    (64, 41, 1, 33, ALL, 0), (64, 41, 2, 24, ALL, 0)])
def test_mixed_automatic_kernel(a, b, K, wcs, row, kernel):
    """The automatic kernel is the one named, bit for bit, and not the FP32 one."""
    V, T = torus(1.0, 0.4, a, b)
    W, kappa = K * wcs, [0.5 + 0.125 * q for q in range(K)]
    coeff = np.array(row * K, np.complex128)
    rng = np.random.default_rng(a + W)
    B = rng.standard_normal((V.shape[0], W)) + 1j * rng.standard_normal((V.shape[0], W))
    rows = rng.choice(V.shape[0], 24, replace=False)
    ref = oracle.apply_boundary_rows(oracle.Mesh(V, T), 1.0, B, 0.0, np.zeros((24, W), np.complex128), kappa, coeff, W,
                                     wcs, rows)
    with Helmholtz_HIP(V, T) as H:
        H.SetPrecision("mixed")
        C = _apply(H, B, kappa, coeff, W, wcs)
        H.SetMixedKernel(kernel)
        assert np.array_equal(C, _apply(H, B, kappa, coeff, W, wcs))
    assert np.linalg.norm(C[rows] - ref) < NEAR * np.linalg.norm(ref)


def test_fp32_all_operators_in_few_columns_are_on_the_vector_alu():
    """On a mesh above 32,768 triangles: which MFMA kernel is selected changes nothing
    (their automatic segments differ, and the rounding with them)."""
    V, T = torus(1.0, 0.4, 184, 90)
    rng = np.random.default_rng(5)
    B = rng.standard_normal((V.shape[0], 3)) + 1j * rng.standard_normal((V.shape[0], 3))
    with Helmholtz_HIP(V, T) as H:
        C = []
        for kernel in (0, 1):
            H.SetMixedKernel(kernel)
            C.append(_apply(H, B, [1.5, 2.0, 2.5], np.array(ALL * 3, np.complex128), 3, 1))
    assert np.array_equal(*C)


@pytest.mark.parametrize("a,b", [(8, 4), (11, 3), (12, 11), (28, 16), (30, 15), (55, 25)])
@pytest.mark.parametrize("K,wcs", [(1, 1), (2, 3), (1, 8), (1, 16), (2, 17)])
def test_mixed_small_apply_and_far_field(a, b, K, wcs):
    V, T = torus(1.0, 0.4, a, b)
    W, kappa = K * wcs, [1.25 + 0.5 * q for q in range(K)]
    coeff = np.array([0.5, 0.5 - 1j, 1 + 0.25j, 0.0] * K, np.complex128)
    rng = np.random.default_rng(a * b + W)
    B = rng.standard_normal((V.shape[0], W)) + 1j * rng.standard_normal((V.shape[0], W))
    m = oracle.Mesh(V, T)
    ref = oracle.apply_boundary(m, 1.0, B, 0.0, np.zeros_like(B), kappa, coeff, W, wcs)
    with Helmholtz_HIP(V, T) as H:
        H.SetPrecision("mixed")
        for kernel, segments in ((2, 0), (0, 0), (2, 3), (2, 0)):
            H.SetMixedKernel(kernel)
            H.SetSegments(segments)
            C = _apply(H, B, kappa, coeff, W, wcs)
            assert np.linalg.norm(C - ref) < NEAR * np.linalg.norm(ref), (kernel, segments)
    for n in (1, 65, 1100):
        d = rng.standard_normal((n, 3))
        d /= np.linalg.norm(d, axis=1)[:, None]
        F = rng.standard_normal((n, W)) + 1j * rng.standard_normal((n, W))
        far = oracle.apply_far_field(oracle.Mesh(V, T, d), 2.0, B, 0.5, F, kappa, coeff, W, wcs)
        with Helmholtz_HIP(V, T, d) as H:
            H.SetPrecision("mixed")
            G = F.copy()
            H.ApplyFarFieldOperators_PL(2.0, B, 0.5, G, kappa, coeff, W, wcs)
        assert np.linalg.norm(G - far) < NEAR * np.linalg.norm(far), n


# segments of 16 to 64 sources as far as their work-groups are resident together: 64
# columns and more, about 176, 256, 436 and 512 work-groups of 64 sources
@pytest.mark.parametrize("a,b,n", [(63, 22, 1000), (64, 32, 2000), (68, 51, 1000), (64, 32, 4000)])
@pytest.mark.parametrize("K,wcs", [(1, 64), (3, 21), (6, 32)])
def test_far_field_of_many_columns(a, b, n, K, wcs):
    V, T = torus(1.0, 0.4, a, b)
    W, kappa = K * wcs, [1.25 + 0.25 * q for q in range(K)]
    coeff = np.array([0.5, 0.5 - 1j, 1 + 0.25j, 0.0] * K, np.complex128)
    rng = np.random.default_rng(n + W)
    B = rng.standard_normal((V.shape[0], W)) + 1j * rng.standard_normal((V.shape[0], W))
    d = fibonacci_sphere(n)
    some = np.append(rng.choice(n - 1, 40, replace=False), n - 1)
    far = oracle.apply_far_field(oracle.Mesh(V, T, d[some]), 2.0, B, 0.0, np.zeros((41, W), np.complex128), kappa, coeff,
                                 W, wcs)
    G = np.zeros((n, W), np.complex128)
    with Helmholtz_HIP(V, T, d) as H:
        H.ApplyFarFieldOperators_PL(2.0, B, 0.0, G, kappa, coeff, W, wcs)
    assert np.linalg.norm(G[some] - far) < NEAR * np.linalg.norm(far)


# The rounding of an accumulation on the matrix cores grows with its length, so the
# automatic segments are at least those at which the error against 64 bits is no
# larger than the vector ALU's: 32 of them on 9,920 triangles (100 steps of 8 sources
# each instead of 39: 1.03 of the error).  1 %: rounding of the same rows
def test_automatic_accumulations_on_a_mesh_of_ordinary_size():
    V, T = torus(1.0, 0.4, 80, 62)
    W, kappa, coeff = 8, [4.0], np.array([0.5, -4j, 1.0, 0.0])
    rng = np.random.default_rng(8)
    B = rng.standard_normal((V.shape[0], W)) + 1j * rng.standard_normal((V.shape[0], W))
    rows = rng.choice(V.shape[0], 600, replace=False)
    ref = oracle.apply_boundary_rows(oracle.Mesh(V, T), 1.0, B, 0.0, np.zeros((600, W), np.complex128), kappa, coeff, W,
                                     W, rows)
    with Helmholtz_HIP(V, T) as H:
        for mode in ("fp32", "fp32_mfma"):
            H.SetPrecision(mode)
            err = []
            for segments in (0, 32):
                H.SetSegments(segments)
                err.append(np.linalg.norm(_apply(H, B, kappa, coeff, W, W)[rows] - ref))
            assert err[0] <= 1.01 * err[1], (mode, err)


# the potential: as many accumulations as the vector ALU makes (FP32, 128 sources
# each here), and for MIXED no route whose error is larger than the matrix cores'
@pytest.mark.parametrize("mode,a,b,P,K,wcs", [("fp32", 176, 58, 2500, 2, 32), ("mixed", 90, 30, 10001, 1, 4)])
def test_automatic_accumulations_of_the_potential(mode, a, b, P, K, wcs):
    V, T = torus(1.0, 0.4, a, b)
    W, kappa = K * wcs, [4.0 + q for q in range(K)]
    coeff = np.array([c for k in kappa for c in (0.0, -1j * k, 1.0, 0.0)])
    rng = np.random.default_rng(P)
    B = rng.standard_normal((V.shape[0], W)) + 1j * rng.standard_normal((V.shape[0], W))
    pts = fibonacci_sphere(P) * rng.uniform(1.7, 2.5, (P, 1))
    some = rng.choice(P, 200, replace=False)
    ref = oracle.apply_near_field(oracle.Mesh(V, T), 1.0, B, 0.0, np.zeros((200, W), np.complex128), kappa, coeff, W,
                                  wcs, pts[some])
    with Helmholtz_HIP(V, T) as H:
        H.SetPrecision(mode)
        err = []
        for kernel, segments in ((2, 0), (0, 160 if mode == "fp32" else 0)):
            H.SetMixedKernel(kernel)
            H.SetSegments(segments)
            U = np.zeros((P, W), np.complex128)
            H.ApplyNearFieldOperators_PL(1.0, B, 0.0, U, kappa, coeff, W, wcs, evaluation_points=pts)
            err.append(np.linalg.norm(U[some] - ref))
    assert err[0] <= 1.01 * err[1], err


# Columns near the ends of the FP32 range, on meshes small and large: the products of
# kernel values and sources stay normal numbers, the split's scales (of the column
# and of the kernel values, 2^110 and 2^24 on the mesh of size 100) leave the FP32
# range by themselves or together
@pytest.mark.parametrize("size,scale", [(1.0, 1e-33), (1.0, 1e-34), (100.0, 1e-31), (1e-3, 1e30), (1.0, 1e33)])
@pytest.mark.parametrize("row", [(0.5, -2j, 1.0, 0.0), (0.5, -2j, 0.0, 1.0), (0.25, 1 - 0.5j, -0.75 + 1j, 0.3)])
def test_fp32_columns_at_the_ends_of_the_range(size, scale, row):
    V, T = torus(size, 0.4 * size, 48, 24)
    W, kappa, coeff = 16, [2.0 / size], np.array(row) * [size, 1.0, size, size]
    rng = np.random.default_rng(12)
    B = rng.standard_normal((V.shape[0], W)) + 1j * rng.standard_normal((V.shape[0], W))
    m = oracle.Mesh(V, T)
    ref = oracle.apply_boundary(m, 1.0, B, 0.0, np.zeros_like(B), kappa, coeff, W, W)
    pts = 2.0 * size * fibonacci_sphere(64)
    refn = oracle.apply_near_field(m, 1.0, B, 0.0, np.zeros((64, W)), kappa, coeff, W, W, pts)
    with Helmholtz_HIP(V, T) as H:
        for mode, kernel in (("fp32", 2), ("mixed", 0), ("fp32_mfma", 2)):
            H.SetPrecision(mode)
            H.SetMixedKernel(kernel)
            C = _apply(H, scale * B, kappa, coeff, W, W) / scale
            assert np.linalg.norm(C - ref) < NEAR * np.linalg.norm(ref), mode
            U = np.zeros((64, W), np.complex128)
            if row[1] or row[2]:
                H.ApplyNearFieldOperators_PL(1.0, scale * B, 0.0, U, kappa, coeff, W, W, evaluation_points=pts)
                assert np.linalg.norm(U / scale - refn) < NEAR * np.linalg.norm(refn), mode


@pytest.mark.parametrize("j", [2, 3])
def test_fp32_wave_numbers_of_very_different_coefficients(j):
    """A double layer (or its adjoint) of 1e-41 beside one of 1: the quotient with the
    single layer, 1e41, is no FP32 number, and the second wave number's kernel values
    are far below the first's scale."""
    V, T = torus(1.0, 0.4, 48, 24)
    K, wcs, kappa = 2, 16, [2.0, 3.0]
    coeff = np.zeros((2, 4), np.complex128)
    coeff[:, 0], coeff[:, 1], coeff[:, j] = 0.5, 1.0 - 1j, [1e-41, 1.0]
    rng = np.random.default_rng(2)
    B = rng.standard_normal((V.shape[0], K * wcs)) + 1j * rng.standard_normal((V.shape[0], K * wcs))
    ref = oracle.apply_boundary(oracle.Mesh(V, T), 1.0, B, 0.0, np.zeros_like(B), kappa, coeff.ravel(), K * wcs, wcs)
    with Helmholtz_HIP(V, T) as H:
        C = _apply(H, B, kappa, coeff.ravel(), K * wcs, wcs)
    assert np.linalg.norm(C - ref) < NEAR * np.linalg.norm(ref)
