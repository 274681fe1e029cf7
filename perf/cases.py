"""Timing cases: what a program that uses this package has it do.

Boundary-operator applies on device arrays, from the smallest meshes to the headline size and in each
arithmetic mode; the far field and the potential; the forward solve and the adjoint derivative with their
GMRES iterations; the batched apply of many meshes; the tangent-point metric of the Gauss-Newton solve.
Meshes are perturbed icospheres (320 ... 81,920 triangles) and torus grids of any size; wave numbers keep at
least ten points per wavelength.  `exact` restates each path in 64 bits with torch, from the formulas.
"""
import ctypes
import math

import numpy as np
import torch

from baemm_amd import Helmholtz_HIP, _lib
from baemm_amd.meshes import fibonacci_sphere, perturbed_sphere, random_directions, torus

FOUR_PI = 4.0 * math.pi
SL_DL_FLOPS = 43   # real operations per pair and wave number: single and double layer values
ALL_FLOPS = 57     # with the adjoint double layer
PLANE_FLOPS = 14   # plane-wave kernels (far field)


def listed():
    return [
        # the smallest call: a tiny mesh and few columns, as in a smoke test or a parameter scan; all launches
        dict(name="apply_320_w4_fp32", kind="apply", mesh="sphere", level=2, K=1, wcs=4, kappa=2.0, ops="potential",
             precision="fp32", elem="c64"),
        # a small scatterer with the example's 16 incident waves; one Arnoldi step of a small mixed solve
        dict(name="apply_1280_w16_mixed", kind="apply", mesh="sphere", level=3, K=1, wcs=16, kappa=4.0,
             ops="potential", precision="mixed", elem="c64"),
        # odd sizes: a torus grid that fills no tile, two wave numbers of five columns, all four operators
        dict(name="apply_torus2806_all_fp32", kind="apply", mesh="torus", a=61, b=23, K=2, wcs=5, kappa=5.5,
             ops="all", precision="fp32", elem="c64"),
        # an ordinary mesh with a ragged column count, the FP32 matrix-core mode
        dict(name="apply_20480_w24_mfma32", kind="apply", mesh="sphere", level=5, K=1, wcs=24, kappa=12.0,
             ops="potential", precision="fp32_mfma", elem="c64"),
        # the headline operator (two wave numbers of 32 columns) in mixed precision
        dict(name="apply_81920_w64_mixed", kind="apply", mesh="sphere", level=6, K=2, wcs=32, kappa=16.0, ops="sldl",
             precision="mixed", elem="c128"),
        # the same in the default precision
        dict(name="apply_81920_w64_fp32", kind="apply", mesh="sphere", level=6, K=2, wcs=32, kappa=16.0, ops="sldl",
             precision="fp32", elem="c128"),
        # the scattered field at a cloud of points, host arrays in and out (what a plotting program calls)
        dict(name="potential_20480_p20001_fp32", kind="potential", mesh="sphere", level=5, K=1, wcs=16, kappa=10.0,
             ops="potential", precision="fp32", points=20001),
        # the far field at the example's 256 directions, device arrays
        dict(name="far_38400_m256_w32", kind="far", mesh="torus", a=240, b=80, K=1, wcs=32, kappa=10.0,
             ops="potential", precision="fp32", meas=256, elem="c64"),
        # the forward solve in the default precision: incident waves, GMRES to 1e-6, far field (host arrays)
        dict(name="solve_far_20480_w32_fp32", kind="solve_far", mesh="sphere", level=5, K=1, wcs=32, kappa=6.0,
             precision="fp32", meas=256),
        # the backward direction: Neumann data, Herglotz wave and two Dirichlet-to-Neumann solves, mixed precision
        dict(name="solve_adj_5120_w16_mixed", kind="solve_adj", mesh="sphere", level=4, K=1, wcs=16, kappa=6.0,
             precision="mixed", meas=256),
        # many meshes of uneven size applied in one call, mixed precision
        dict(name="batch_24_mixed", kind="batch", n=24, mix=4, lo=3, hi=5, precision="mixed", elem="c64"),
        # one apply of the Gauss-Newton solve's tangent-point metric (host arrays)
        dict(name="tp_metric_20480", kind="tp_metric", mesh="sphere", level=5, q=6.0, p=12.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _edge(case):
    """Mean edge length of the case's mesh, about."""
    if case["mesh"] == "sphere":
        return 1.2 / 2 ** case["level"]
    return max(2.0 * math.pi * 1.2 / case["a"], 2.0 * math.pi * 0.4 / case["b"])


def _draw_mesh(rng, case, lo, hi):
    """A mesh of lo to hi triangles: an icosphere level or a torus grid of any size."""
    if rng.random() < 0.35:
        levels = [l for l in range(2, 7) if lo <= 20 * 4 ** l <= hi]
        if levels:
            case.update(mesh="sphere", level=rng.choice(levels))
            return
    n = _log_int(rng, lo, hi)
    b = max(5, int(round(math.sqrt(n / 6.0))))
    case.update(mesh="torus", a=max(8, n // (2 * b)), b=b)


def _draw_kappa(rng, case, most=32.0):
    top = max(1.0, min(most, 2.0 * math.pi / (10.0 * _edge(case))))
    case["kappa"] = round(rng.uniform(1.0, top) * 64) / 64   # a value that 32 bits hold


def draw(rng):
    kind = rng.choices(["apply", "potential", "far", "solve_far", "solve_adj", "batch", "tp_metric"],
                       [6, 2, 1, 2, 2, 1, 1])[0]
    case = dict(kind=kind)
    if kind == "batch":
        case.update(n=rng.randint(4, 40), mix=rng.randrange(1 << 20), lo=2, hi=rng.choice([3, 4, 5]),
                    precision=rng.choice(["fp32", "mixed"]), elem=rng.choice(["c64", "c128"]))
        return case
    if kind == "tp_metric":
        _draw_mesh(rng, case, 320, 30000)
        case.update(q=6.0, p=12.0)
        return case
    if kind in ("solve_far", "solve_adj"):
        _draw_mesh(rng, case, 320, 12000)
        case.update(K=1, wcs=_log_int(rng, 1, 32), precision=rng.choice(["fp32", "mixed", "fp32_mfma"]),
                    meas=_log_int(rng, 60, 400))
        _draw_kappa(rng, case, 10.0)
        return case
    _draw_mesh(rng, case, 320, 60000)
    K = rng.choice([1, 1, 1, 2, 2, 3])
    case.update(K=K, wcs=_log_int(rng, 1, 64 // K), precision=rng.choice(["fp32", "fp32", "mixed", "mixed", "fp32_mfma"]))
    _draw_kappa(rng, case)
    if kind == "apply":
        case.update(ops=rng.choice(["potential", "sldl", "dtn", "all"]), elem=rng.choice(["c64", "c128"]))
    elif kind == "potential":
        case.update(ops="potential", points=_log_int(rng, 200, 20000))
    else:
        case.update(ops="potential", meas=_log_int(rng, 60, 1000), elem=rng.choice(["c64", "c128"]))
    return case


# ------------------------------------------------------------------ inputs

def _mesh(case, seed):
    if case["mesh"] == "sphere":
        return perturbed_sphere(case["level"], seed=seed)
    return torus(1.0, 0.36 + 0.08 * np.random.default_rng(seed).random(), case["a"], case["b"])


def _kappas(case):
    K = case["K"]
    return [case["kappa"] * (q + 1) / K for q in range(K)]


def _rows(case):
    """Coefficient rows (mass, single, double, adjoint double layer) of each wave number."""
    rows = []
    for q, k in enumerate(_kappas(case)):
        if case["ops"] == "potential":
            rows.append([0.5, -1j * k, 1.0, 0.0])
        elif case["ops"] == "dtn":
            rows.append([0.5, -1j * k, 0.0, 1.0])
        elif case["ops"] == "sldl":
            rows.append([0.0, 1.0, 1.0, 0.0] if q % 2 == 0 else [0.5, -1j * k, 1.0, 0.0])
        else:
            rows.append([0.5 + 0.25j, 1.0 - 0.5j, -0.75 + 1j, 0.3 - 0.9j])
    return np.array(rows, np.complex128)


def _normal(rng, rows, cols):
    return rng.standard_normal((rows, cols)) + 1j * rng.standard_normal((rows, cols))


def _torch_type(case):
    return torch.complex64 if case["elem"] == "c64" else torch.complex128


def _batch_items(case):
    """(level, wave number, columns, coefficient kind) of each mesh of a batch."""
    rng = np.random.default_rng(case["mix"])
    items = []
    for _ in range(case["n"]):
        level = int(rng.integers(case["lo"], case["hi"] + 1))
        top = min(16.0, 2.0 * math.pi / (12.0 / 2 ** level))
        items.append((level, round(float(rng.uniform(1.0, max(1.0, top))) * 64) / 64, 2 ** int(rng.integers(0, 7))))
    return items


def _inputs(case, seed):
    """Meshes and host arrays of the case, from the seed alone."""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "batch":
        out = []
        for i, (level, kappa, W) in enumerate(_batch_items(case)):
            V, T = perturbed_sphere(level, seed=seed + 1000 * i)
            out.append((V, T, kappa, W, _normal(rng, V.shape[0], W)))
        return out
    V, T = _mesh(case, seed)
    if kind == "tp_metric":
        return V, T, rng.standard_normal((V.shape[0], 3))
    W = case["K"] * case["wcs"]
    if kind == "solve_far":
        return V, T, random_directions(W, seed=seed), None
    if kind == "solve_adj":
        return V, T, random_directions(W, seed=seed), 0.05 * _normal(rng, case["meas"], W)
    B = _normal(rng, V.shape[0], W)
    if kind == "potential":
        pts = fibonacci_sphere(case["points"]) * rng.uniform(1.7, 2.5, (case["points"], 1))
        return V, T, B, pts
    return V, T, B, None


_STREAM = []


def _stream():
    """The stream the device-array calls run on (a program's own, at default priority)."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


_ONE = (ctypes.c_double * 2)(1.0, 0.0)
_ZERO = (ctypes.c_double * 2)(0.0, 0.0)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, case=case)
    if kind == "batch":
        Hs, Bs, Cs = [], [], []
        for V, T, kappa, W, B in _inputs(case, seed):
            H = Helmholtz_HIP(V, T)
            H.SetPrecision(case["precision"])
            H.LoadBoundaryOperators_PL([kappa], np.array([0.5, -1j * kappa, 1.0, 0.0]), W, W)
            Hs.append(H)
            Bs.append(torch.from_numpy(B).to("cuda", _torch_type(case)))
            Cs.append(torch.zeros_like(Bs[-1]))
        n = len(Hs)
        s.update(H=Hs, B=Bs, C=Cs, n=n, hs=(ctypes.c_void_p * n)(*[H._h.value for H in Hs]),
                 pB=(ctypes.c_void_p * n)(*[t.data_ptr() for t in Bs]),
                 pC=(ctypes.c_void_p * n)(*[t.data_ptr() for t in Cs]),
                 ld=(ctypes.c_int64 * n)(*[t.shape[1] for t in Bs]),
                 elem=_lib.C64 if case["elem"] == "c64" else _lib.C128, L=_lib.load(), stream=_stream().cuda_stream)
        torch.cuda.synchronize()
        return s
    if kind == "tp_metric":
        V, T, x = _inputs(case, seed)
        s.update(H=Helmholtz_HIP(V, T), x=x, q=case["q"], p=case["p"])
        return s
    V, T, first, second = _inputs(case, seed)
    meas = fibonacci_sphere(case["meas"]) if "meas" in case else None
    H = Helmholtz_HIP(V, T, meas)
    H.SetPrecision(case["precision"])
    s.update(H=H, kappa=_kappas(case))
    if kind in ("solve_far", "solve_adj"):
        s.update(K=case["K"], wcs=case["wcs"], dirs=first, g=second)
        return s
    W = case["K"] * case["wcs"]
    H.LoadParameters(s["kappa"], _rows(case), W, case["wcs"])
    if kind == "potential":
        s.update(B=first, pts=second, U=np.zeros((second.shape[0], W), np.complex128))
        return s
    B = torch.from_numpy(first).to("cuda", _torch_type(case))
    C = torch.zeros((B.shape[0] if kind == "apply" else case["meas"], W), dtype=B.dtype, device="cuda")
    L = _lib.load()
    s.update(B=B, C=C, W=W, elem=_lib.C64 if case["elem"] == "c64" else _lib.C128, stream=_stream().cuda_stream,
             call=L.baemm_apply_boundary_dev if kind == "apply" else L.baemm_apply_far_field_dev)
    torch.cuda.synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind in ("apply", "far"):
        _lib.check(s["call"](s["H"]._h, _ONE, s["B"].data_ptr(), s["W"], s["elem"], _ZERO, s["C"].data_ptr(), s["W"],
                             s["elem"], s["stream"]), s["H"]._h)
        return s["C"]
    if kind == "batch":
        _lib.check(s["L"].baemm_apply_boundary_batch(s["n"], s["hs"], None, s["pB"], s["ld"], s["elem"], None, s["pC"],
                                                     s["ld"], s["elem"], s["stream"]))
        return s["C"]
    if kind == "potential":
        return s["H"].ApplyNearFieldOperators_PL(1.0, s["B"], 0.0, s["U"], evaluation_points=s["pts"])
    if kind == "solve_far":
        return s["H"].FarField(s["kappa"], s["K"], s["dirs"], s["wcs"], cg_tol=1e-10, gmres_tol=1e-6)
    if kind == "solve_adj":
        return s["H"].AdjointDerivative_FF(s["kappa"], s["K"], s["dirs"], s["wcs"], s["g"], cg_tol=1e-10, gmres_tol=1e-6)
    return s["H"].TangentPointMetric(s["x"], s["q"], s["p"])


# -------------------------------------------------------------------- work

def _sizes(case):
    if case["mesh"] == "sphere":
        return 10 * 4 ** case["level"] + 2, 20 * 4 ** case["level"]
    return case["a"] * case["b"], 2 * case["a"] * case["b"]


def work(case):
    """Operations of the pair sums (kernel values and the complex contraction) and the bytes of the inputs and
    outputs.  The solves count nine operator applies a solve, about what GMRES needs here."""
    kind = case["kind"]
    if kind == "batch":
        flops = nbytes = 0.0
        for level, _, W in _batch_items(case):
            nv, nt = 10 * 4 ** level + 2, 20 * 4 ** level
            flops += float(nt) * nt * (8 * W + SL_DL_FLOPS)
            nbytes += 32.0 * nt + 2.0 * nv * W * (8 if case["elem"] == "c64" else 16)
        return dict(bytes=nbytes, flops=flops)
    nv, nt = _sizes(case)
    if kind == "tp_metric":
        return dict(bytes=32.0 * nt + 48.0 * nv, flops=45.0 * nt * nt)
    K, W = case["K"], case["K"] * case["wcs"]
    if kind in ("apply", "far"):
        per = ALL_FLOPS if case["ops"] == "all" else SL_DL_FLOPS
        m = nt if kind == "apply" else case["meas"]
        size = 8.0 if case["elem"] == "c64" else 16.0
        return dict(bytes=32.0 * nt + size * W * (nv + (nv if kind == "apply" else m)),
                    flops=float(m) * nt * (8 * W + (per if kind == "apply" else PLANE_FLOPS) * K))
    if kind == "potential":
        P = case["points"]
        return dict(bytes=32.0 * nt + 24.0 * P + 16.0 * W * (nv + P), flops=float(P) * nt * (8 * W + SL_DL_FLOPS * K))
    applies = 9 if kind == "solve_far" else 18
    flops = applies * float(nt) * nt * (8 * W + SL_DL_FLOPS * K) + float(case["meas"]) * nt * (8 * W + PLANE_FLOPS * K)
    return dict(bytes=applies * (32.0 * nt + 32.0 * W * nv) + 16.0 * case["meas"] * W, flops=flops)


# ------------------------------------------------- the same values in 64 bits

class _Geometry:
    """Centroids, unit normals, areas, incidence and the single-layer self term of a triangle mesh."""

    def __init__(self, V, T):
        self.V = torch.from_numpy(np.ascontiguousarray(V, np.float64)).to("cuda")
        self.T = torch.from_numpy(np.ascontiguousarray(T, np.int64)).to("cuda")
        X = self.V[self.T]
        self.nv, self.nt = self.V.shape[0], self.T.shape[0]
        self.mid = X.mean(1)
        N = 0.5 * torch.linalg.cross(X[:, 1] - X[:, 0], X[:, 2] - X[:, 0])
        self.area = N.norm(dim=1)
        self.nrm = N / self.area[:, None]
        # integral of 1/|x - centroid| over the triangle, edge by edge, divided by the area
        u = X - self.mid[:, None, :]
        length = u.norm(dim=2)
        total = torch.zeros_like(self.area)
        for e in range(3):
            a, b = (e + 1) % 3, (e + 2) % 3
            ab = (u[:, a] * u[:, b]).sum(1)
            p, q = length[:, a] ** 2 - ab, length[:, b] ** 2 - ab
            edge = (p + q).abs().sqrt()
            sa, sb = p / (length[:, a] * edge), q / (length[:, b] * edge)
            total += length[:, a] * (1.0 - sa * sa).sqrt() * (torch.atanh(sa) + torch.atanh(sb))
        self.self_term = total / self.area

    def faces(self, X):
        """Area-weighted triangle values of vertex values: a/3 (X0 + X1 + X2)."""
        return X[self.T].sum(1) * (self.area / 3.0)[:, None]

    def vertices(self, F):
        """The transpose of faces."""
        G = F * (self.area / 3.0)[:, None]
        out = torch.zeros((self.nv,) + tuple(F.shape[1:]), dtype=F.dtype, device=F.device)
        for k in range(3):
            out.index_add_(0, self.T[:, k], G)
        return out

    def mass(self, X):
        """P1 mass matrix times X: a/6 on the diagonal and a/12 off it, triangle by triangle."""
        s = X[self.T]
        total = s.sum(1)
        out = torch.zeros_like(X)
        for k in range(3):
            out.index_add_(0, self.T[:, k], (total + s[:, k]) * (self.area / 12.0)[:, None])
        return out

    def mass_solve(self, X):
        if not hasattr(self, "_mass"):
            self._mass = torch.linalg.lu_factor(self.mass(torch.eye(self.nv, dtype=torch.float64, device="cuda")))
        if X.is_complex():
            return torch.complex(self.mass_solve(X.real.contiguous()), self.mass_solve(X.imag.contiguous()))
        return torch.linalg.lu_solve(*self._mass, X)


def _pair_values(g, x, n, first, kappa, c, self_pairs):
    """Kernel values of targets x (normals n, index of the first of them) against all triangles of g, for one
    wave number: real and imaginary parts of c1 E/r + (c2 z.n_j - c3 z.n_i)(i kappa r - 1) E/r^3."""
    d = [g.mid[:, k][None, :] - x[:, k][:, None] for k in range(3)]
    r2 = d[0] ** 2 + d[1] ** 2 + d[2] ** 2
    if self_pairs:
        rows = torch.arange(x.shape[0], device="cuda")
        r2[rows, first + rows] = 1.0
    r = r2.sqrt()
    w = torch.zeros_like(r, dtype=torch.complex128)
    if c[2] != 0:
        w += complex(c[2]) * (d[0] * g.nrm[:, 0] + d[1] * g.nrm[:, 1] + d[2] * g.nrm[:, 2])
    if c[3] != 0:
        w -= complex(c[3]) * (d[0] * n[:, 0:1] + d[1] * n[:, 1:2] + d[2] * n[:, 2:3])
    del d
    w *= torch.complex(-torch.ones_like(r), kappa * r)
    w /= r2
    w += complex(c[1])
    w *= torch.polar(1.0 / r, kappa * r)
    if self_pairs:
        w[rows, first + rows] = complex(c[1]) * (g.self_term[first:first + x.shape[0]] + 1j * kappa)
    return w


def _pair_sums(g, x, n, kappas, rows, b, wcs, self_pairs):
    out = torch.empty((x.shape[0], b.shape[1]), dtype=torch.complex128, device="cuda")
    step = max(1, (1 << 26) // g.nt)
    for q, kappa in enumerate(kappas):
        c = rows[q] / FOUR_PI
        bq = b[:, q * wcs:(q + 1) * wcs].contiguous()
        for i in range(0, x.shape[0], step):
            A = _pair_values(g, x[i:i + step], None if n is None else n[i:i + step], i, kappa, c, self_pairs)
            out[i:i + step, q * wcs:(q + 1) * wcs] = A @ bq
    return out


def _boundary(g, kappas, rows, B, wcs):
    out = g.vertices(_pair_sums(g, g.mid, g.nrm, kappas, rows, g.faces(B), wcs, True))
    MB = g.mass(B)
    for q in range(len(kappas)):
        out[:, q * wcs:(q + 1) * wcs] += complex(rows[q][0]) * MB[:, q * wcs:(q + 1) * wcs]
    return out


def _operator(g, kappa, row):
    """The dense boundary operator c0 M + AvT (K + D) Av of one wave number."""
    c = row / FOUR_PI
    P = torch.zeros((g.nt, g.nv), dtype=torch.complex128, device="cuda")
    step = max(1, (1 << 26) // g.nt)
    for i in range(0, g.nt, step):
        A = _pair_values(g, g.mid[i:i + step], g.nrm[i:i + step], i, kappa, c, True) * (g.area / 3.0)
        for k in range(3):
            P[i:i + step].index_add_(1, g.T[:, k], A)
    out = g.vertices(P)
    del P
    return out + complex(row[0]) * g.mass(torch.eye(g.nv, dtype=torch.float64, device="cuda"))


def _plane(g, u, kappas, c1, c2, wcs, b=None, sign=-1.0):
    """Plane-wave values (c1 + sign i kappa (u.n) c2) exp(sign i kappa u.y), c1 and c2 per wave number: triangles x
    directions, or with b the sums over the triangles."""
    un, uy = g.nrm @ u.T, g.mid @ u.T
    out = []
    for q, k in enumerate(kappas):
        F = (complex(c1[q]) + sign * 1j * k * complex(c2[q]) * un) * torch.polar(torch.ones_like(uy), sign * k * uy)
        out.append(F if b is None else F.T @ b[:, q * wcs:(q + 1) * wcs])
    return out


def _far(g, meas, kappas, rows, B, wcs):
    u = torch.from_numpy(meas).to("cuda")
    return torch.cat(_plane(g, u, kappas, rows[:, 1] / FOUR_PI, rows[:, 2] / FOUR_PI, wcs, g.faces(B)), 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        out = []
        for V, T, kappa, W, B in _inputs(case, seed):
            Bt = torch.from_numpy(B).to("cuda").to(_torch_type(case)).to(torch.complex128)
            out.append(_boundary(_Geometry(V, T), [kappa], np.array([[0.5, -1j * kappa, 1.0, 0.0]]), Bt, W))
        return out
    if kind == "tp_metric":
        return _exact_metric(case, seed)
    V, T, first, second = _inputs(case, seed)
    g = _Geometry(V, T)
    kappas, wcs = _kappas(case), case["wcs"]
    if kind in ("apply", "far", "potential"):
        B = torch.from_numpy(first).to("cuda")
        if kind == "potential":
            x = torch.from_numpy(second).to("cuda")
            return _pair_sums(g, x, None, kappas, _rows(case), g.faces(B), wcs, False).cpu().numpy()
        B = B.to(_torch_type(case)).to(torch.complex128)
        if kind == "far":
            return _far(g, fibonacci_sphere(case["meas"]), kappas, _rows(case), B, wcs)
        return _boundary(g, kappas, _rows(case), B, wcs)
    meas = fibonacci_sphere(case["meas"])
    d = torch.from_numpy(first[:wcs]).to("cuda")
    if kind == "solve_far":
        # incident waves -e^{i kappa d.x}; (1/2 M - i kappa S + K) phi = incident; far field of phi
        waves = _plane(g, d, kappas, [-1.0] * len(kappas), [0.0] * len(kappas), wcs, sign=1.0)
        rows = np.array([[0.5, -1j * k, 1.0, 0.0] for k in kappas])
        phi = [torch.linalg.solve(_operator(g, k, rows[q]), g.vertices(waves[q])) for q, k in enumerate(kappas)]
        return _far(g, meas, kappas, rows, torch.cat(phi, 1), wcs).cpu().numpy()
    # Neumann data and the Herglotz wave's, both by (1/2 M - i kappa S + K'); their product along the normals
    u = torch.from_numpy(meas).to("cuda")
    gg = torch.from_numpy(second).to("cuda").conj().resolve_conj()
    waves = _plane(g, d, kappas, [-1j * k for k in kappas], [1.0] * len(kappas), wcs, sign=1.0)
    her = _plane(g, u, kappas, [-1j * k / len(meas) for k in kappas], [1.0 / len(meas)] * len(kappas), wcs)
    du, dv = [], []
    for q, k in enumerate(kappas):
        lu = torch.linalg.lu_factor(_operator(g, k, np.array([0.5, -1j * k, 0.0, 1.0])))
        du.append(torch.linalg.lu_solve(*lu, g.vertices(waves[q])))
        dv.append(torch.linalg.lu_solve(*lu, g.vertices(her[q] @ gg[:, q * wcs:(q + 1) * wcs])))
    du, dv = torch.cat(du, 1), torch.cat(dv, 1)
    x = (du * dv).sum(1, keepdim=True).real.contiguous()
    Y = g.mass_solve(g.vertices(g.faces(x) / g.area[:, None] * g.nrm) * (-1.0 / du.shape[1]))
    return Y.cpu().numpy(), du.cpu().numpy()


def _exact_metric(case, seed):
    """The tangent-point metric: pairs of triangles with weights w = a_S a_T |d|^(-2 sigma - 2) on the differences of
    the face gradients, and w k, k = (n_S.d)^2 / |d|^4, on those of the face averages."""
    V, T, x = _inputs(case, seed)
    g = _Geometry(V, T)
    x = torch.from_numpy(x).to("cuda")
    sigma = (case["p"] - 2.0) / case["q"] - 1.0
    X = g.V[g.T]
    # hat-function gradients: n x (opposite edge) / (2 a)
    grad = torch.stack([torch.linalg.cross(g.nrm, X[:, (k + 2) % 3] - X[:, (k + 1) % 3]) for k in range(3)], 1)
    grad = grad / (2.0 * g.area)[:, None, None]
    xf = x[g.T]
    du = torch.einsum("tki,tkj->tij", grad, xf).reshape(g.nt, 9)
    ub = xf.mean(1)
    Ru, Rb = torch.empty_like(du), torch.empty_like(ub)
    step = max(1, (1 << 26) // g.nt)
    for i in range(0, g.nt, step):
        d = g.mid[i:i + step, None, :] - g.mid[None, :, :]
        r2 = (d * d).sum(2)
        rows = torch.arange(r2.shape[0], device="cuda")
        r2[rows, i + rows] = 1.0
        w = g.area[i:i + step, None] * g.area[None, :] * r2 ** (-sigma - 1.0)
        w[rows, i + rows] = 0.0
        k = ((d * g.nrm[i:i + step, None, :]).sum(2) ** 2 + (d * g.nrm[None, :, :]).sum(2) ** 2) / r2 ** 2
        Ru[i:i + step] = 2.0 * (w.sum(1, keepdim=True) * du[i:i + step] - w @ du)
        wk = w * k
        Rb[i:i + step] = wk.sum(1, keepdim=True) * ub[i:i + step] - wk @ ub
    out = torch.zeros_like(x)
    for k in range(3):
        out.index_add_(0, g.T[:, k], torch.einsum("ti,tij->tj", grad[:, k], Ru.reshape(g.nt, 3, 3)) + Rb / 3.0)
    return out.cpu().numpy()
