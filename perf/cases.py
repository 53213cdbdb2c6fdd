"""The calls whose speed matters, with the inputs a simulation has in hand for them.

Six kinds of calls, each through the entry points a program binds to:

* ``step``:     one global time step of a layer, the proxy kernel ``all``
                (predictor, volume and local flux, neighbour flux);
* ``calls``:    the same step as a time cluster issues it, one batched call per
                kernel, on the reference GPU build's storage (128-byte blocks,
                compact star matrices), with the derivatives kept and the
                solution evaluated in between as receivers and faults do;
* ``lts``:      one macro step of rate-2 local time stepping in four clusters
                (60/25/10/5 % of the cells), eagerly or from the captured graph;
* ``fault``:    the two element kernels around a friction solve: space-time
                interpolation to the fault points and the nodal flux back;
* ``friction``: one friction-law-103 solve of a fault in mid-rupture;
* ``train``:    one training step of the friction solver's warm-start network.

Every input comes from torch generators on the GPU, physical operators
included (random affine tetrahedra with random links, or a conforming periodic
box of jittered tetrahedra), and ``exact`` evaluates the same step in 64 bits
with dense matrix products of matrices integrated here.
"""
from __future__ import annotations

import functools
import math
from types import SimpleNamespace

import numpy as np
import torch

from seissol_amd import _capi
from seissol_amd._capi import FaultLayer, Layer, ptr
from seissol_amd.dr import DeviceDrFaces, DrFaces
from seissol_amd.friction import FrictionParameters, FrictionSolver, WarmStartTrainer, mlp_param_count
from seissol_amd.kernels import Engine, Local, Neighbor, Spacetime, Time
from seissol_amd.lts import LocalTimeStepping
from seissol_amd.proxy import run_proxy

F64 = torch.float64
MATRIX_CORE = ("bf16x3", "bf16x6", "f16x3")
FACE_NODES = ((0, 2, 1), (0, 1, 3), (0, 3, 2), (1, 2, 3))
# column-major positions of the non-zeros of an elastic star matrix
STAR_NONZEROS = (6, 7, 8, 15, 16, 17, 24, 25, 26, 33, 34, 43, 44, 51, 53, 54, 57, 59, 64, 66, 67, 74, 76, 77)
FRACTIONS = (0.6, 0.25, 0.1, 0.05)
RHO, VP, VS, EDGE, CFL = (2000.0, 3000.0), 6000.0, 3464.0, 100.0, 0.5


def listed():
    return [
        # one rank's layer at production size, the fast form on the proxy's random links
        dict(name="step_f16x3_o6_1m", kind="step", arithmetic="f16x3", order=6, cells=1_000_000, mesh="proxy",
             star="compact", align=0),
        # the double-precision drop-in on the proxy's layer
        dict(name="step_fp64_o6_400k", kind="step", arithmetic="fp64", order=6, cells=400_000, mesh="proxy",
             star="dense", align=0),
        # a single-precision run of an ordinary partition
        dict(name="step_fp32_o6_100k", kind="step", arithmetic="fp32", order=6, cells=100_000, mesh="proxy",
             star="compact", align=128),
        # a strong-scaled partition with a ragged tail and ghost cells
        dict(name="step_f16x3_o4_29k", kind="step", arithmetic="f16x3", order=4, cells=29_987, mesh="periodic",
             star="compact", align=0),
        # the smallest layers: latency of one step
        dict(name="step_fp64_o4_500", kind="step", arithmetic="fp64", order=4, cells=500, mesh="periodic",
             star="dense", align=0),
        # a time cluster's own sequence of batched calls, drop-in precision and storage
        dict(name="calls_fp64_o6_50k", kind="calls", arithmetic="fp64", order=6, cells=50_001, mesh="periodic",
             star="compact", align=128),
        # four clusters, 600k cells, the fast form
        dict(name="lts_f16x3_o5_600k", kind="lts", arithmetic="f16x3", order=5, nx=60, ny=50, nz=40, graph=False),
        # four clusters of a small double-precision partition, replayed from its graph
        dict(name="lts_fp64_o4_9k", kind="lts", arithmetic="fp64", order=4, nx=32, ny=8, nz=8, graph=True),
        # a fault through a double-precision partition
        dict(name="fault_fp64_o6_10k", kind="fault", arithmetic="fp64", order=6, faces=10_000, cells=50_000),
        # a smaller fault under the fast form (its dynamic-rupture kernels run in single precision)
        dict(name="fault_f16x3_o5_3k", kind="fault", arithmetic="f16x3", order=5, faces=3_001, cells=20_000),
        # the friction solve of the planar fault of 20,000 faces and 25 points
        dict(name="friction_o4_20k", kind="friction", order=4, faces=20_000, start="plain"),
        # one step of the warm-start training loop
        dict(name="train_1024", kind="train", batch=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "calls", "lts", "lts", "fault", "friction"])
    if kind == "step":
        arithmetic = rng.choice(["f16x3", "f16x3", "fp64", "fp64", "fp32", "bf16x3", "bf16x6"])
        order = rng.randint(3, 7) if arithmetic in MATRIX_CORE else rng.randint(2, 8)
        # work per cell grows like order^5: no drawn layer costs more than the largest listed one
        top = 200_000 if arithmetic in MATRIX_CORE else 60_000
        return dict(kind=kind, arithmetic=arithmetic, order=order,
                    cells=_log(rng, 300, top * min(1.0, (6 / order) ** 3)), mesh=rng.choice(["proxy", "periodic"]),
                    star=rng.choice(["dense", "compact"]), align=rng.choice([0, 128]))
    if kind == "calls":
        return dict(kind=kind, arithmetic=rng.choice(["fp64", "fp64", "fp32"]), order=rng.randint(3, 7),
                    cells=_log(rng, 500, 30_000), mesh=rng.choice(["proxy", "periodic"]),
                    star=rng.choice(["dense", "compact"]), align=rng.choice([0, 128]))
    if kind == "lts":
        arithmetic = rng.choice(["f16x3", "f16x3", "fp64", "fp32"])
        return dict(kind=kind, arithmetic=arithmetic, order=rng.randint(3, 6), nx=2 * rng.randint(16, 30),
                    ny=2 * rng.randint(2, 8), nz=2 * rng.randint(2, 8), graph=rng.random() < 0.5)
    if kind == "fault":
        faces = _log(rng, 100, 10_000)
        return dict(kind=kind, arithmetic=rng.choice(["fp64", "fp32", "f16x3"]), order=rng.randint(3, 7), faces=faces,
                    cells=4 * faces + rng.randint(0, 4 * faces))
    return dict(kind=kind, order=rng.randint(3, 6), faces=_log(rng, 200, 20_000),
                start=rng.choice(["plain", "closed_form"]))


# --------------------------------------------------------------------------
# reference element: basis, global matrices (64 bits, integrated here)
# --------------------------------------------------------------------------

def num_basis(order):
    return order * (order + 1) * (order + 2) // 6


def _jacobi(n, a, b, x, y):
    """y^n P_n^(a,b)(x / y)."""
    if n == 0:
        return 1.0 + 0.0 * x
    p0, p1 = 1.0 + 0.0 * x, 0.5 * (a - b) * y + (1.0 + 0.5 * (a + b)) * x
    for m in range(2, n + 1):
        s = 2.0 * m + a + b
        p0, p1 = p1, ((s - 1) * ((a * a - b * b) * y + s * (s - 2) * x) * p1
                      - 2 * (m + a - 1) * (m + b - 1) * s * y * y * p0) / (2 * m * (m + a + b) * (s - 2))
    return p1


def _tet(order, xi, eta, zeta):
    """[B][points] values of the orthogonal basis of the reference tetrahedron."""
    out = []
    for deg in range(order):
        for k in range(deg + 1):
            for j in range(deg - k + 1):
                i = deg - j - k
                out.append(_jacobi(i, 0, 0, 2 * xi - 1 + eta + zeta, 1 - eta - zeta)
                           * _jacobi(j, 2 * i + 1, 0, 2 * eta - 1 + zeta, 1 - zeta)
                           * _jacobi(k, 2 * i + 2 * j + 2, 0, 2 * zeta - 1, 1.0 + 0.0 * zeta))
    return np.array(out)


def _tri(order, chi, tau):
    return np.array([_jacobi(deg - j, 0, 0, 2 * chi - 1 + tau, 1 - tau)
                     * _jacobi(j, 2 * (deg - j) + 1, 0, 2 * tau - 1, 1.0 + 0.0 * tau)
                     for deg in range(order) for j in range(deg + 1)])


def _turn(h, chi, tau):
    return ((tau, chi), (1 - chi - tau, tau), (chi, 1 - chi - tau), (chi, tau))[h]


def _on_face(f, a, b):
    return ((b, a, 0 * a), (a, 0 * a, b), (0 * a, b, a), (1 - a - b, a, b))[f]


@functools.lru_cache(maxsize=None)
def matrices(order):
    """K^T_j, K_j [3][B][B], R_f = rDivM_f [4][B][B2], T_f = fMrT_f [4][B2][B] and the
    neighbour products N[f][j][h] = rDivM_f fP_h rT_j [4][4][3][B][B]."""
    g, w = np.polynomial.legendre.leggauss(order + 2)
    g, w = 0.5 * (g + 1), 0.5 * w
    a, b, c = (m.ravel() for m in np.meshgrid(g, g, g, indexing="ij"))
    wa, wb, wc = (m.ravel() for m in np.meshgrid(w, w, w, indexing="ij"))
    pts = [a * (1 - b) * (1 - c), b * (1 - c), c]
    w3 = wa * wb * wc * (1 - b) * (1 - c) ** 2
    phi = _tet(order, *pts)
    mass = (phi * phi * w3).sum(1)
    kt, k = [], []
    for d in range(3):  # derivatives by the complex step (exact to rounding)
        z = [p.astype(complex) for p in pts]
        z[d] = z[d] + 1e-100j
        dphi = _tet(order, *z).imag / 1e-100
        kt.append((phi * w3) @ dphi.T / mass[:, None])
        k.append((dphi * w3) @ phi.T / mass[:, None])
    a, b = (m.ravel() for m in np.meshgrid(g, g, indexing="ij"))
    wa, wb = (m.ravel() for m in np.meshgrid(w, w, indexing="ij"))
    chi, tau, w2 = a * (1 - b), b, wa * wb * (1 - b)
    psi = _tri(order, chi, tau)
    mass2 = (psi * psi * w2).sum(1)
    fmrt = np.array([(psi * w2) @ _tet(order, *_on_face(f, chi, tau)).T for f in range(4)])
    rdivm = np.array([m.T / mass[:, None] / mass2[None, :] for m in fmrt])
    fp = [(psi * w2) @ _tri(order, *_turn(h, chi, tau)).T for h in range(3)]
    rt = fmrt / mass2[None, :, None]
    nb = np.array([[[rdivm[f] @ fp[h] @ rt[j] for h in range(3)] for j in range(4)] for f in range(4)])
    return np.array(kt), np.array(k), rdivm, fmrt, nb, rt, np.array(fp)


@functools.lru_cache(maxsize=None)
def stroud(order):
    """(points [n][2], weights [n], V [4][4][n][B], VTW [4][4][B][n], resample [n][n])."""
    m = order + 1
    i = np.arange(m)
    # Gauss-Jacobi (1, 0) by the eigenvalues of its recurrence
    diag = -1.0 / ((2 * i + 1) * (2 * i + 3))
    off = np.sqrt(i[1:] * (i[1:] + 1) / (2.0 * i[1:] + 1) ** 2)
    x, v = np.linalg.eigh(np.diag(diag) + np.diag(off, 1) + np.diag(off, -1))
    wx = 0.5 * v[0] ** 2  # the weight 1 - chi integrates to 1/2 on [0, 1]
    s, ws = np.polynomial.legendre.leggauss(m)
    chi, s, ws = 0.5 * (x + 1), 0.5 * (s + 1), 0.5 * ws
    pts = np.array([(chi[a], (1 - chi[a]) * s[b]) for a in range(m)[::-1] for b in range(m)[::-1]])
    w = np.array([wx[a] * ws[b] for a in range(m)[::-1] for b in range(m)[::-1]])
    g, gw = np.polynomial.legendre.leggauss(order + 2)
    g, gw = 0.5 * (g + 1), 0.5 * gw
    a, b, c = (q.ravel() for q in np.meshgrid(g, g, g, indexing="ij"))
    wa, wb, wc = (q.ravel() for q in np.meshgrid(gw, gw, gw, indexing="ij"))
    phi = _tet(order, a * (1 - b) * (1 - c), b * (1 - c), c)
    mass = (phi * phi * wa * wb * wc * (1 - b) * (1 - c) ** 2).sum(1)
    V = np.array([[_tet(order, *_on_face(f, *_turn((h - 1) % 4, pts[:, 0], pts[:, 1]))).T for h in range(4)]
                  for f in range(4)])
    VTW = V.transpose(0, 1, 3, 2) * w / mass[:, None]
    psi = _tri(order, pts[:, 0], pts[:, 1])
    resample = (psi.T / (psi * psi * w).sum(1)) @ (psi * w)
    return pts, w, V, VTW, resample


def time_integral(order, t0, t1):
    return [(t1 ** (i + 1) - t0 ** (i + 1)) / math.factorial(i + 1) for i in range(order)]


def gauss_times(order, dt):
    g, w = np.polynomial.legendre.leggauss(order)
    return 0.5 * (g + 1) * dt, 0.5 * w * dt


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _uniform(gen, shape, lo, hi):
    return torch.rand(shape, generator=gen, dtype=F64, device="cuda") * (hi - lo) + lo


def _randint(gen, hi, shape, dtype):
    return torch.randint(0, hi, shape, generator=gen, device="cuda").to(dtype)


def _affine_tets(gen, n):
    """Well-shaped random affine images of the reference tetrahedron, det in [0.5, 2]."""
    J = torch.eye(3, dtype=F64, device="cuda") + _uniform(gen, (n, 3, 3), -0.35, 0.35)
    J = torch.where((torch.linalg.det(J) < 0.2)[:, None, None], torch.eye(3, dtype=F64, device="cuda"), J)
    J = J * (_uniform(gen, (n,), 0.5, 2.0) / torch.linalg.det(J)).pow(1 / 3)[:, None, None]
    x0 = _uniform(gen, (n, 1, 3), -10.0, 10.0)
    return torch.cat([x0, x0 + J.transpose(1, 2)], 1)


@functools.lru_cache(maxsize=None)
def _box_tables():
    """Corners [2][5][4][3] of the five tetrahedra of even and odd cubes and, per face, the
    neighbour (cube offset, tetrahedron, side, orientation) [2][5][4][6]."""
    tets = (((0, 3, 5, 6), (1, 0, 3, 5), (2, 0, 3, 6), (4, 0, 5, 6), (7, 3, 5, 6)),
            ((1, 2, 4, 7), (0, 1, 2, 4), (3, 1, 2, 7), (5, 1, 4, 7), (6, 2, 4, 7)))
    corner = np.zeros((2, 5, 4, 3), np.int64)
    for par in range(2):
        for t in range(5):
            p = np.array([[c & 1, c >> 1 & 1, c >> 2 & 1] for c in tets[par][t]])
            if np.linalg.det(p[1:] - p[0]) < 0:
                p[[2, 3]] = p[[3, 2]]
            corner[par, t] = p
    faces = {}
    for i in range(-1, 3):
        for j in range(-1, 3):
            for k in range(-1, 3):
                for t in range(5):
                    p = corner[(i + j + k) % 2, t] + (i, j, k)
                    for f in range(4):
                        key = frozenset(map(tuple, p[list(FACE_NODES[f])]))
                        faces.setdefault(key, []).append(((i, j, k), t, f))
    link = np.zeros((2, 5, 4, 6), np.int64)
    for par in range(2):
        c = np.array((par, 0, 0))
        for t in range(5):
            p = corner[par, t] + c
            for f in range(4):
                own = list(map(tuple, p[list(FACE_NODES[f])]))
                (cube, t2, f2), = [x for x in faces[frozenset(own)] if x[:2] != (tuple(c), t)]
                q = corner[sum(cube) % 2, t2] + cube
                turn = [tuple(v) for v in q[list(FACE_NODES[f2])]].index(own[0])
                link[par, t, f] = (*(np.array(cube) - c), t2, f2, turn)
    return corner, link


def _periodic_box(gen, nx, ny, nz):
    """vertices [n][4][3], neighbours, relations and the cube column x of each cell
    (cells ordered by x, then y, z) of a jittered periodic box."""
    corner, link = (torch.from_numpy(a).cuda() for a in _box_tables())
    dims = torch.tensor((nx, ny, nz), device="cuda")
    i, j, k = torch.meshgrid(*(torch.arange(m, device="cuda") for m in (nx, ny, nz)), indexing="ij")
    cube = torch.stack([i, j, k], -1).reshape(-1, 1, 1, 3)
    par = cube.sum(-1).reshape(-1) % 2
    grid = cube + corner[par]
    wrap = grid % dims
    jitter = _uniform(gen, (nx, ny, nz, 3), -0.1 * EDGE, 0.1 * EDGE)
    vertices = grid.to(F64) * EDGE + jitter[wrap[..., 0], wrap[..., 1], wrap[..., 2]]
    rel = link[par]
    nb = (cube + rel[..., :3]) % dims
    neighbors = ((nb[..., 0] * ny + nb[..., 1]) * nz + nb[..., 2]) * 5 + rel[..., 3]
    column = cube[:, 0, 0, 0].repeat_interleave(5)
    return (vertices.reshape(-1, 4, 3), neighbors.reshape(-1, 4).to(torch.int32),
            rel[..., 4:].reshape(-1, 4, 2).to(torch.uint8), column)


def _box_dims(cells):
    m = max(4, 2 * math.ceil((cells / 5) ** (1 / 3) / 2))
    best = None
    for ny in range(max(4, m - 4), m + 3, 2):
        for nz in range(max(4, m - 4), m + 3, 2):
            nx = max(4, 2 * math.ceil(cells / (10 * ny * nz)))
            if best is None or nx * ny * nz < best[0]:
                best = (nx * ny * nz, (nx, ny, nz))
    return best[1]


def _coefficients(mat):
    """Transposed coefficient matrices M_d(q, p) [n][3][9][9] of (rho, lambda, mu)."""
    rho, lam, mu = mat.unbind(-1)
    M = torch.zeros((*rho.shape, 3, 9, 9), dtype=F64, device="cuda")
    normal = ((0, 1, 2), (1, 0, 2), (2, 0, 1))
    shear = (((3, 7), (5, 8)), ((3, 6), (4, 8)), ((4, 7), (5, 6)))
    for d in range(3):
        M[..., d, 6 + d, normal[d][0]] = -(lam + 2 * mu)
        M[..., d, 6 + d, normal[d][1]] = -lam
        M[..., d, 6 + d, normal[d][2]] = -lam
        M[..., d, d, 6 + d] = -1 / rho
        for s, v in shear[d]:
            M[..., d, v, s] = -mu
            M[..., d, s, v] = -1 / rho
    return M


def _face_frame(v, f):
    """Unit normal and tangents and twice the area of face f."""
    p = v[:, list(FACE_NODES[f])]
    s = p[:, 1] - p[:, 0]
    n = torch.linalg.cross(s, p[:, 2] - p[:, 0])
    t = torch.linalg.cross(n, s)
    area2 = n.norm(dim=-1)
    return n / area2[:, None], s / s.norm(dim=-1, keepdim=True), t / t.norm(dim=-1, keepdim=True), area2


def _rotations(n, s, t):
    """T (face frame to global) and its inverse for the 6 stresses and 3 velocities."""
    T = torch.zeros((len(n), 9, 9), dtype=F64, device="cuda")
    Ti = torch.zeros_like(T)
    base = (n, s, t)
    pairs = ((0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2))
    for r, (x, y) in enumerate(pairs):
        for c, (a, b) in enumerate(pairs):
            u, w = base[a], base[b]
            T[:, r, c] = u[:, x] * w[:, y] + (u[:, y] * w[:, x] if c > 2 else 0)
            u, w = base[x], base[y]
            Ti[:, r, c] = u[:, a] * w[:, b] + (u[:, b] * w[:, a] if c > 2 else 0)
    for i in range(3):
        for k in range(3):
            T[:, 6 + i, 6 + k] = base[k][:, i]
            Ti[:, 6 + k, 6 + i] = base[k][:, i]
    return T, Ti


def _operators(vertices, mat, neighbors):
    """star [n][3][9][9], aplus, aminus [n][4][9][9] as (q, p), chunk by chunk."""
    n = len(vertices)
    star = torch.empty((n, 3, 9, 9), dtype=F64, device="cuda")
    ap, am = torch.empty((2, n, 4, 9, 9), dtype=F64, device="cuda")
    for a in range(0, n, 1 << 17):
        sl = slice(a, min(n, a + (1 << 17)))
        v, m = vertices[sl], mat[sl]
        J = (v[:, 1:] - v[:, :1]).transpose(1, 2)
        M = _coefficients(m)
        star[sl] = torch.einsum("nrd,ndqp->nrqp", torch.linalg.inv(J), M)
        det = torch.linalg.det(J).abs()
        for f in range(4):
            nrm, s, t, area2 = _face_frame(v, f)
            T, Ti = _rotations(nrm, s, t)
            other = mat[neighbors[sl, f].long()]
            # state at the interface from the impedances of the P and the two S waves
            qL = torch.zeros((len(v), 9, 9), dtype=F64, device="cuda")
            qN = torch.zeros_like(qL)
            for stress, vel, mod in ((0, 6, 1), (3, 7, 0), (5, 8, 0)):
                zl = (m[:, 0] * (mod * m[:, 1] + (1 + mod) * m[:, 2])).sqrt()
                zn = (other[:, 0] * (mod * other[:, 1] + (1 + mod) * other[:, 2])).sqrt()
                z = zl + zn
                qL[:, vel, vel], qN[:, vel, vel] = zl / z, zn / z
                qL[:, stress, vel], qN[:, stress, vel] = -1 / z, 1 / z
                qL[:, stress, stress], qN[:, stress, stress] = zn / z, zl / z
                qL[:, vel, stress], qN[:, vel, stress] = -zl * zn / z, zl * zn / z
            scale = (-area2 / det)[:, None, None]
            for q, out in ((qL, ap), (qN, am)):
                out[sl, f] = scale * (Ti.transpose(1, 2) @ (q @ M[:, 0]) @ T.transpose(1, 2))
    return star, ap, am


def _cfl_step(vertices, mat, order):
    J = vertices[:, 1:] - vertices[:, :1]
    area = sum(0.5 * _face_frame(vertices, f)[3] for f in range(4))
    vp = ((mat[:, 1] + 2 * mat[:, 2]) / mat[:, 0]).sqrt()
    return CFL * 2 * 3 * torch.linalg.det(J).abs() / 6 / area / (vp * (2 * order - 1))


def _materials(gen, n):
    rho = _uniform(gen, (n,), *RHO)
    mu = rho * VS ** 2
    return torch.stack([rho, rho * VP ** 2 - 2 * mu, mu], 1)


def _real(case):
    return F64 if case["arithmetic"] == "fp64" else torch.float32


def _rows(m, case):
    """Rows of a block of m basis functions in the layer's layout."""
    a = max(1, case.get("align", 0) // (8 if case["arithmetic"] == "fp64" else 4))
    return (m + a - 1) // a * a


def _column_major(x):
    return x.transpose(-1, -2).contiguous()


def _cell_inputs(case, seed):
    """The layer's arrays in the real type of the case (cells beyond `cells` are ghosts)."""
    gen = _gen(seed)
    order, kind = case["order"], case["kind"]
    B, rt = num_basis(order), _real(case)
    x = SimpleNamespace(order=order, B=B, cluster=None)
    scale = 1.0
    if kind == "lts":
        x.vertices, x.neighbors, x.relations, column = _periodic_box(gen, case["nx"], case["ny"], case["nz"])
        x.n = len(x.vertices)
        # bands of cube columns: cluster 0, then 1, 2, 3, 2, 1, each at least one column wide
        nx = case["nx"]
        half = [max(1, round(f * nx / 2)) for f in FRACTIONS[1:3]]
        last = max(1, round(FRACTIONS[3] * nx))
        widths = [nx - 2 * sum(half) - last, half[0], half[1], last, half[1], half[0]]
        ids = torch.tensor(np.repeat((0, 1, 2, 3, 2, 1), widths), device="cuda")
        cl = ids[column]
        perm = torch.argsort(cl, stable=True)
        inv = torch.empty_like(perm)
        inv[perm] = torch.arange(x.n, device="cuda")
        x.vertices, x.relations = x.vertices[perm], x.relations[perm].contiguous()
        x.neighbors = inv[x.neighbors[perm].long()].to(torch.int32)
        x.cluster = cl[perm]
        x.start = np.concatenate([[0], np.cumsum(torch.bincount(x.cluster, minlength=4).cpu().numpy())])
    elif case["mesh"] == "proxy":
        x.n = case["cells"]
        x.vertices = _affine_tets(gen, x.n)
        x.neighbors = _randint(gen, x.n, (x.n, 4), torch.int32)
        x.relations = torch.stack([_randint(gen, 4, (x.n, 4), torch.uint8), _randint(gen, 3, (x.n, 4), torch.uint8)],
                                  -1).contiguous()
        scale = 2.0 ** -32  # random links make the solution grow from step to step
    else:
        x.vertices, x.neighbors, x.relations, _ = _periodic_box(gen, *_box_dims(case["cells"]))
        x.n = case["cells"]
    total = len(x.vertices)
    mat = _materials(gen, total)
    if x.cluster is not None:  # slower waves where the steps are larger
        mat[:, 1:] *= (0.25 ** x.cluster.to(F64))[:, None]
    x.dt = float(_cfl_step(x.vertices, mat, order).min()) if x.cluster is None else float(
        (_cfl_step(x.vertices, mat, order) / 2.0 ** x.cluster).min())
    star, ap, am = _operators(x.vertices, mat, x.neighbors)
    star = _column_major(star).reshape(total, 3, 81)
    if case.get("star", "dense") == "compact":
        star = star[:, :, list(STAR_NONZEROS)]
    x.star = star.to(rt).contiguous()
    x.aplus = _column_major(ap).reshape(total, 4, 81).to(rt)
    x.aminus = _column_major(am).reshape(total, 4, 81).to(rt)
    ld = _rows(B, case)
    x.dofs = torch.zeros((total, 9, ld), dtype=rt, device="cuda")
    x.dofs[:, :, :B] = (_uniform(gen, (total, 9, B), -1.0, 1.0) * scale).to(rt)
    x.total, x.ld = total, ld
    if x.cluster is not None:
        x.setup = _lts_bits(x.cluster, x.neighbors)
    return x


def _lts_bits(cl, nb):
    """LTS bits of every cell (neighbours at most one cluster apart)."""
    other = cl[nb.long()]
    own = cl[:, None]
    face = 2 ** torch.arange(4, device="cuda")
    bits = ((own < other) * face).sum(1) + ((own == other) * face * 16).sum(1)
    bits |= (own < other).any(1) * _capi.SDG_LTS_ACCUMULATE_BUFFERS
    bits |= (own > other).any(1) * _capi.SDG_LTS_HAS_DERIVATIVES
    bits |= (own <= other).any(1) * _capi.SDG_LTS_HAS_BUFFERS
    acc = (bits & _capi.SDG_LTS_ACCUMULATE_BUFFERS) > 0
    bits |= (acc & ((bits & 0xF0) > 0)) * _capi.SDG_LTS_HAS_DERIVATIVES
    bits |= ((own == other) * acc[nb.long()] * face).sum(1)
    return bits


def _derivative_reals(case):
    return sum(9 * _rows(num_basis(case["order"] - i), case) for i in range(case["order"]))


def _engine(case):
    eng = Engine(case["order"], case["arithmetic"])
    eng.set_layout(case.get("align", 0), case.get("star", "dense"))
    return eng


def _layer(case, x, derivatives):
    """The sdg_layer view of the inputs, its work arrays included."""
    rt = x.dofs.dtype
    x.integrated = torch.zeros_like(x.dofs)
    x.derivatives = (torch.zeros((x.total, _derivative_reals(case)), dtype=rt, device="cuda") if derivatives else None)
    x.traces = None
    if case["kind"] == "step" and (case["arithmetic"] in MATRIX_CORE or
                                   (case["arithmetic"] == "fp64" and 3 <= case["order"] <= 7)):
        B2 = case["order"] * (case["order"] + 1) // 2
        x.traces = torch.zeros((x.total, 4, 9, (B2 + 3) // 4 * 4), dtype=rt, device="cuda")
    bits = None
    if x.cluster is not None:
        x.bits16 = x.setup.to(torch.int16)
        bits = ptr(x.bits16)
    x.view = Layer(x.n, ptr(x.dofs), ptr(x.integrated), ptr(x.derivatives), ptr(x.star), ptr(x.aplus),
                   ptr(x.aminus), ptr(x.neighbors), ptr(x.relations), None, ptr(x.traces), bits, 0, 0, 0)
    return x


def _fault_inputs(case, seed):
    gen = _gen(seed)
    order, nf, n, rt = case["order"], case["faces"], case["cells"], _real(case)
    B, P = num_basis(order), (order + 1) ** 2
    x = SimpleNamespace(n=n, nf=nf)
    vertices, mat = _affine_tets(gen, n), _materials(gen, n)
    # every fault face joins two cells of its own
    cells = torch.randperm(n, generator=gen, device="cuda")[:2 * nf]
    x.plus, x.minus = cells[:nf].to(torch.int32), cells[nf:].to(torch.int32)
    sides = _randint(gen, 4, (2, nf), torch.int64)
    turn = _randint(gen, 3, (nf,), torch.int64) + 1
    x.info = torch.stack([sides[0], sides[1], turn], 1).to(torch.uint8)
    x.mapping = torch.full((n, 4), -1, dtype=torch.int32, device="cuda")
    ids = torch.arange(nf, dtype=torch.int32, device="cuda")
    x.mapping[x.plus.long(), sides[0]] = ids
    x.mapping[x.minus.long(), sides[1]] = ids
    v = vertices[x.plus.long()]
    frames = [_face_frame(v, f) for f in range(4)]
    pick = lambda i: torch.stack([f[i] for f in frames])[sides[0], torch.arange(nf, device="cuda")]
    area2 = pick(3)
    T, Ti = _rotations(pick(0), pick(1), pick(2))
    x.tinv = Ti.reshape(nf, 81).contiguous()  # TinvT column by column
    flux = []
    for cell, sign in ((x.plus, -1.0), (x.minus, 1.0)):
        w = vertices[cell.long()]
        det = torch.linalg.det(w[:, 1:] - w[:, :1]).abs()
        F = (sign * area2 / det)[:, None, None] * (_coefficients(mat[cell.long()])[:, 0] @ T.transpose(1, 2))
        flux.append(_column_major(F).reshape(nf, 81))
    x.flux_plus, x.flux_minus = flux
    x.dt = float(_cfl_step(vertices, mat, order).min())
    tp, _ = gauss_times(order, x.dt)
    x.coeffs = np.array([[t ** d / math.factorial(d) for d in range(order)] for t in tp])
    # derivatives of a smooth solution: each order larger by 1 / dt
    parts = []
    for d in range(order):
        parts.append(_uniform(gen, (n, 9 * num_basis(order - d)), -1.0, 1.0) / x.dt ** d)
    x.derivatives = torch.cat(parts, 1).to(rt)
    x.imposed_plus = _uniform(gen, (nf, 9, P), -1.0, 1.0)
    x.imposed_minus = _uniform(gen, (nf, 9, P), -1.0, 1.0)
    x.dofs = _uniform(gen, (n, 9, B), -1.0, 1.0).to(rt)
    return x


FAULT_TIME = 0.4  # well after the nucleation


def _friction_inputs(case, seed):
    """A fault in mid-rupture: 30 % of the points slide (1e-3 to 3 m/s), the others creep; every
    point starts in the quasi-steady balance of its slip rate and the waves perturb the tractions."""
    gen = _gen(seed)
    order, nf = case["order"], case["faces"]
    P = (order + 1) ** 2
    shape = (nf, P)
    prm = FrictionParameters()
    a, sl0 = _uniform(gen, shape, 0.008, 0.02), _uniform(gen, shape, 0.2, 0.5)
    f0, muw, b, srw = 0.6, 0.2, 0.014, 0.1
    zp, zs = 2670.0 * 6000.0, 2670.0 * 3464.0
    sliding = torch.rand((nf, 1), generator=gen, device="cuda") < 0.3
    logv = torch.where(sliding, _uniform(gen, shape, -3.0, 0.5), _uniform(gen, shape, -16.0, -9.0))
    v = 10.0 ** logv
    shear = torch.where(sliding, _uniform(gen, shape, 25e6, 45e6), _uniform(gen, shape, 60e6, 80e6))
    normal = 120e6
    mu = (shear - 0.5 * zs * v) / normal
    psi = a * torch.log(2 * prm.rs_sr0 / v * torch.sinh(mu / a))
    stress = torch.zeros((nf, 6, P), dtype=F64, device="cuda")
    stress[:, 0], stress[:, 3] = -normal, shear
    full = lambda c: torch.full(shape, c, dtype=F64, device="cuda")
    A = dict(rs_a=a, rs_sl0=sl0, rs_f0=full(f0), rs_muw=full(muw), rs_b=full(b), rs_srw=full(srw),
             state_variable=psi, mu=mu, slip_rate1=v.clone(), slip_rate2=full(0.0), slip_rate_magnitude=v.clone(),
             initial_stress=stress, initial_pressure=full(0.0),
             nucleation_stress=torch.zeros_like(stress), nucleation_pressure=full(0.0),
             imp_and_eta=torch.tensor([zp, zs, zp, zs, zp / 2, zs / 2, 2 / zs, 1 / zp, 1 / zs, 1 / zp, 1 / zs],
                                      dtype=F64, device="cuda").repeat(nf, 1))
    for k in ("traction1", "traction2", "slip1", "slip2", "accumulated_slip", "rupture_time", "peak_slip_rate",
              "dyn_stress_time"):
        A[k] = full(0.0)
    for k in ("rupture_time_pending", "dyn_stress_time_pending", "convergence_inner", "convergence_outer"):
        A[k] = torch.ones(shape, dtype=torch.uint8, device="cuda")
    for k in ("q_interpolated_plus", "q_interpolated_minus"):
        q = _uniform(gen, (nf, order, 9, P), -1e6, 1e6)
        q[:, :, 6:] = _uniform(gen, (nf, order, 3, P), -0.02, 0.02)
        # the slip of the point is in the velocities of its two sides
        q[:, :, 7] += (v * (0.5 if k.endswith("minus") else -0.5))[:, None]
        q[:, :, 3] -= 0.5 * zs * v[:, None]
        A[k] = q
    for k in ("imposed_state_plus", "imposed_state_minus"):
        A[k] = torch.zeros((nf, 9, P), dtype=F64, device="cuda")
    return A, prm


def _train_inputs(case, seed):
    gen = _gen(seed)
    n = case["batch"]
    x = torch.empty((n, 7), dtype=F64, device="cuda")
    for j, (lo, hi) in enumerate(((-16, 2), (0, 2), (-1.5, 0.5), (25, 60), (-16, 1), (0.8, 2.0))):
        x[:, j] = _uniform(gen, (n,), lo, hi)
    x[:, 6] = -0.5 * torch.tanh(0.3 * (x[:, 0] - x[:, 1])) + 0.01 * _uniform(gen, (n,), -1.0, 1.0)
    params = torch.zeros(mlp_param_count(), dtype=F64, device="cuda")
    params[:6], params[6:12] = x[:, :6].mean(0), x[:, :6].std(0)
    params[12], params[13] = x[:, 6].mean(), x[:, 6].std()
    params[14:206] = _uniform(gen, (192,), -0.7, 0.7)
    params[238:1262] = _uniform(gen, (1024,), -0.3, 0.3)
    params[1294:1326] = _uniform(gen, (32,), -0.3, 0.3)
    return x.float(), params.float()


# --------------------------------------------------------------------------
# a user's program
# --------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    s = SimpleNamespace(case=case, kind=kind)
    if kind in ("step", "calls", "lts"):
        s.engine = _engine(case)
        s.x = _layer(case, _cell_inputs(case, seed), derivatives=kind != "step")
        s.coeffs = time_integral(case["order"], 0.0, s.x.dt)
        if kind == "calls":
            s.spacetime, s.time, s.local, s.neighbor = (c(s.engine) for c in (Spacetime, Time, Local, Neighbor))
            s.half = [(0.5 * s.x.dt) ** i / math.factorial(i) for i in range(case["order"])]
            s.evaluated = torch.zeros_like(s.x.dofs)
        if kind == "lts":
            s.x.lts = SimpleNamespace(num_clusters=4, cluster_start=s.x.start, dt0=s.x.dt)
            s.clusters = LocalTimeStepping(s.engine, s.x)
    elif kind == "fault":
        s.engine = _engine(case)
        s.x = x = _fault_inputs(case, seed)
        P = (case["order"] + 1) ** 2
        host = (t.cpu().numpy() for t in (x.plus, x.minus, x.info, x.mapping, x.tinv, x.flux_plus, x.flux_minus))
        x.faces = DeviceDrFaces(DrFaces(*host, imp_and_eta=None, points=P))
        x.view = Layer(x.n, ptr(x.dofs), None, ptr(x.derivatives), None, None, None, None, None, None, None, None,
                       0, 0, 0)
        x.q_plus, x.q_minus = torch.zeros((2, x.nf, case["order"], 9, P), dtype=F64, device="cuda")
    elif kind == "friction":
        s.arrays, prm = _friction_inputs(case, seed)
        P = (case["order"] + 1) ** 2
        s.view = FaultLayer(case["faces"], P, P, case["order"], 0,
                            *[ptr(s.arrays.get(k)) for k in _capi.FAULT_FIELDS])
        s.solver = FrictionSolver(prm, case["order"])
        s.solver.closed_form_start = case["start"] == "closed_form"
        s.solver.setupLayer(s)
        tp, s.weights = gauss_times(case["order"], 1e-3)
        s.delta = FrictionSolver.computeDeltaT(tp)
    else:
        s.samples, params = _train_inputs(case, seed)
        s.trainer = WarmStartTrainer()
        s.trainer.params.copy_(params)
    return s


def run(s):
    if s.kind == "step":
        run_proxy(s.engine, s.x, "all", 1, s.x.dt)
        # the matrix-core forms hand only face traces between their passes
        return [s.x.dofs] if s.case["arithmetic"] in MATRIX_CORE else [s.x.dofs, s.x.integrated]
    if s.kind == "calls":
        s.spacetime.computeBatchedAder(s.coeffs, s.x.dt, s.x.view)
        s.time.evaluateBatched(s.half, s.x.derivatives, s.evaluated, s.x.n)
        s.local.computeBatchedIntegral(s.x.view)
        s.neighbor.computeBatchedNeighborsIntegral(s.x.view)
        return [s.x.dofs, s.x.integrated, s.x.derivatives, s.evaluated]
    if s.kind == "lts":
        s.clusters.advance(1, graph=s.case["graph"])
        return [s.x.dofs, s.x.integrated, s.x.derivatives]
    if s.kind == "fault":
        x = s.x
        x.faces.interpolate(s.engine, x.coeffs, x.derivatives, x.q_plus, x.q_minus)
        x.faces.nodal_flux(s.engine, x.view, x.imposed_plus, x.imposed_minus)
        return [x.q_plus, x.q_minus, x.dofs]
    if s.kind == "friction":
        s.solver.evaluate(FAULT_TIME, s.delta, s.weights)
        return {k: s.arrays[k] for k in FRICTION_OUTPUTS}
    t = s.trainer
    t.loss_grad(s.samples)
    t.adam(3e-3)
    return [t.loss, t.grads, t.params, t.m, t.v]


FRICTION_OUTPUTS = ("state_variable", "slip_rate1", "slip_rate2", "slip_rate_magnitude", "mu", "traction1", "traction2",
                    "slip1", "slip2", "accumulated_slip", "rupture_time", "peak_slip_rate", "dyn_stress_time",
                    "rupture_time_pending", "dyn_stress_time_pending", "convergence_inner", "convergence_outer",
                    "imposed_state_plus", "imposed_state_minus")


# --------------------------------------------------------------------------
# work
# --------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _nonzeros(order):
    kt, k, rdivm, fmrt, _, rt, fp = matrices(order)
    count = lambda m: int((np.abs(m) > 1e-12 * np.abs(m).max()).sum())
    ck = 0
    for d in range(1, order):
        rows, cols = num_basis(order - d), num_basis(order - d + 1)
        ck += count(kt[:, :rows, :cols]) * 9 + 3 * 24 * rows
    B, B2 = num_basis(order), order * (order + 1) // 2
    local = count(k) * 9 + 3 * 24 * B + (count(fmrt) + count(rdivm)) * 9 + 4 * 81 * B2
    neigh = (count(rt) + 4 * count(fp) / 3 + count(rdivm)) * 9 + 4 * 81 * B2
    return 2.0 * ck, 2.0 * local, 2.0 * neigh


def work(case):
    kind = case["kind"]
    if kind == "friction":
        points = case["faces"] * (case["order"] + 1) ** 2
        # both sides' interpolated states (7 of 9 components), 25 fields in, 19 + 18 values out; about
        # three slip-rate solves of two residuals per time point, some 200 operations each
        return {"bytes": points * 8.0 * (14 * case["order"] + 25 + 33), "flops": points * case["order"] * 6 * 200.0}
    if kind == "train":
        P = 1327
        return {"bytes": case["batch"] * 28.0 + P * 4.0 * 8, "flops": case["batch"] * P * 6.0}
    order, rs = case["order"], 8 if case["arithmetic"] == "fp64" else 4
    B = num_basis(order)
    D = sum(9 * num_basis(order - i) for i in range(order))
    if kind == "fault":
        nf, P = case["faces"], (order + 1) ** 2
        flops = nf * 2 * (2.0 * P * D + 2 * 81 * (D // 9) + 2.0 * order * 9 * P * order / 2)
        flops += nf * 2 * (2 * 81 * P + 2.0 * 9 * P * B)
        return {"bytes": nf * 2.0 * (D * rs + 81 * 8 + order * 9 * P * 8 + 2 * 9 * B * rs + (9 * P + 81) * 8),
                "flops": flops}
    ck, local, neigh = _nonzeros(order)
    star = 72 if case.get("star") == "compact" else 243
    cell = (2 * 9 * B + star + 648) * rs + 24.0
    if kind == "step":
        if case["arithmetic"] not in MATRIX_CORE:
            cell += 9 * B * rs  # the time integral is an output
        return {"bytes": case["cells"] * cell, "flops": case["cells"] * (ck + local + neigh)}
    if kind == "calls":
        return {"bytes": case["cells"] * (cell + (2 * 9 * B + D) * rs), "flops": case["cells"] * (ck + local + neigh)}
    cells = 5 * case["nx"] * case["ny"] * case["nz"]
    updates = cells * sum(f * 2 ** (3 - c) for c, f in enumerate(FRACTIONS))
    return {"bytes": updates * (cell + 9 * B * rs), "flops": updates * (ck + local + neigh)}


# --------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------

def _device(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _dense_star(x):
    star = x.star.to(F64)
    if star.shape[-1] == 24:
        out = torch.zeros((len(star), 3, 81), dtype=F64, device="cuda")
        out[:, :, list(STAR_NONZEROS)] = star
        star = out
    return star.reshape(-1, 3, 9, 9)  # [cell][direction][p][q]


def _by_quantity(A, X):
    """Y[e, p, :] = sum_q X[e, q, :] A[e][p][q]."""
    return torch.bmm(A, X)


def _predict(order, dofs, star):
    """Time derivatives dQ_d [e][9][B(O - d)]."""
    kt = _device(matrices(order)[0])
    out = [dofs]
    for d in range(1, order):
        rows, cols = num_basis(order - d), num_basis(order - d + 1)
        out.append(-sum(_by_quantity(star[:, j], out[-1] @ kt[j, :rows, :cols].T) for j in range(3)))
    return out


def _taylor(order, c, ders):
    out = torch.zeros_like(ders[0])
    for d in range(order):
        out[:, :, :ders[d].shape[2]] += c[d] * ders[d]
    return out


def _local_flux(order, I, star, aplus):
    _, k, rdivm, fmrt, _, _, _ = (_device(m) for m in matrices(order))
    out = sum(_by_quantity(star[:, j], I @ k[j].T) for j in range(3))
    for f in range(4):
        out = out + _by_quantity(aplus[:, f].reshape(-1, 9, 9), I @ fmrt[f].T) @ rdivm[f].T
    return out


def _neighbor_flux(order, I_of, nb, rel, aminus):
    """sum_f N[f][side][turn] I_nb A-_f; I_of(f, rows) gives the neighbours' integrals."""
    N = _device(matrices(order)[4])
    n = len(nb)
    out = torch.zeros((n, 9, num_basis(order)), dtype=F64, device="cuda")
    for f in range(4):
        variant = rel[:, f, 0].long() * 3 + rel[:, f, 1].long()
        for v in range(12):
            rows = (variant == v).nonzero()[:, 0]
            if len(rows):
                Y = I_of(f, rows) @ N[f, v // 3, v % 3].T
                out[rows] += _by_quantity(aminus[rows, f].reshape(-1, 9, 9).to(F64), Y)
    return out


CHUNK = 1 << 16


def _exact_step(case, seed):
    x = _cell_inputs(case, seed)
    order, B = x.order, x.B
    c = time_integral(order, 0.0, x.dt)
    half = [(0.5 * x.dt) ** i / math.factorial(i) for i in range(order)]
    star = _dense_star(x)
    dofs = x.dofs.to(F64)
    I = torch.zeros((x.total, 9, B), dtype=F64, device="cuda")
    evaluated = torch.zeros_like(dofs)
    ders = torch.zeros((x.total, _derivative_reals(case)) if case["kind"] == "calls" else (0,), dtype=F64, device="cuda")
    for a in range(0, x.n, CHUNK):
        sl = slice(a, min(x.n, a + CHUNK))
        D = _predict(order, dofs[sl, :, :B].clone(), star[sl])
        I[sl] = _taylor(order, c, D)
        if case["kind"] == "calls":
            evaluated[sl, :, :B] = _taylor(order, half, D)
            _store_derivatives(case, ders, sl, D)
        dofs[sl, :, :B] += _local_flux(order, I[sl], star[sl], x.aplus[sl].to(F64))
    for a in range(0, x.n, CHUNK):
        sl = slice(a, min(x.n, a + CHUNK))
        nb = x.neighbors[sl]
        dofs[sl, :, :B] += _neighbor_flux(order, lambda f, r: I[nb[r, f].long()], nb, x.relations[sl], x.aminus[sl])
    integrated = torch.zeros_like(dofs)
    integrated[:, :, :B] = I
    if case["kind"] == "calls":
        return [dofs, integrated, ders, evaluated]
    return [dofs] if case["arithmetic"] in MATRIX_CORE else [dofs, integrated]


def _store_derivatives(case, out, cells, D, keep=None):
    off = 0
    for d in D:
        ld = _rows(d.shape[2], case)
        block = out[cells, off:off + 9 * ld].reshape(-1, 9, ld)
        block[:, :, :d.shape[2]] = d if keep is None else torch.where(keep[:, None, None], d, block[:, :, :d.shape[2]])
        out[cells, off:off + 9 * ld] = block.reshape(-1, 9 * ld)
        off += 9 * ld


def _exact_lts(case, seed):
    x = _cell_inputs(case, seed)
    order, B, dt0 = x.order, x.B, x.dt
    star, dofs = _dense_star(x), x.dofs.to(F64)
    cl, nbs = x.cluster, x.neighbors.long()
    # each cluster's derivatives, the time they are expanded at and the integral of its last step and
    # over the two steps that a slower neighbour sees
    D = [None] * 4
    begin = [0] * 4
    single = torch.zeros((x.n, 9, B), dtype=F64, device="cuda")
    pair = torch.zeros_like(single)

    def step(c, k):
        sl = slice(int(x.start[c]), int(x.start[c + 1]))
        w = time_integral(order, 0.0, dt0 * 2 ** c)
        D[c] = _predict(order, dofs[sl].clone(), star[sl])
        begin[c] = k
        single[sl] = _taylor(order, w, D[c])
        pair[sl] = single[sl] + (pair[sl] if (k >> c) & 1 else 0)
        dofs[sl] += _local_flux(order, single[sl], star[sl], x.aplus[sl].to(F64))
        if c > 0:
            step(c - 1, k)
            step(c - 1, k + (1 << (c - 1)))
        nb = nbs[sl]

        def integral(f, rows):
            at = nb[rows, f]
            other = cl[at]
            out = torch.where((other < c)[:, None, None], pair[at], single[at])
            slow = (other > c).nonzero()[:, 0]
            if len(slow):
                t = dt0 * (k - begin[c + 1])
                sub = time_integral(order, t, t + dt0 * 2 ** c)
                first = int(x.start[c + 1])
                out[slow] = _taylor(order, sub, [d[at[slow] - first] for d in D[c + 1]])
            return out

        dofs[sl] += _neighbor_flux(order, integral, nb, x.relations[sl], x.aminus[sl])

    step(3, 0)
    has = lambda bit: (x.setup & bit) > 0
    buffers = torch.where(has(_capi.SDG_LTS_ACCUMULATE_BUFFERS)[:, None, None], pair, single)
    buffers = torch.where(has(_capi.SDG_LTS_HAS_BUFFERS)[:, None, None], buffers, torch.zeros_like(buffers))
    ders = torch.zeros((x.n, _derivative_reals(case)), dtype=F64, device="cuda")
    keep = has(_capi.SDG_LTS_HAS_DERIVATIVES)
    for c in range(4):
        sl = slice(int(x.start[c]), int(x.start[c + 1]))
        _store_derivatives(case, ders, sl, D[c], keep[sl])
    return [dofs, buffers, ders]


def _exact_fault(case, seed):
    x = _fault_inputs(case, seed)
    order, nf = case["order"], x.nf
    B, P = num_basis(order), (order + 1) ** 2
    V, VTW = (_device(m) for m in stroud(order)[2:4])
    coeffs = _device(x.coeffs)
    TinvT = x.tinv.reshape(nf, 9, 9)  # [p][q]
    q = torch.zeros((2, nf, order, 9, P), dtype=F64, device="cuda")
    dofs = x.dofs.to(F64)
    for side, (cells, flux, imposed) in enumerate(((x.plus, x.flux_plus, x.imposed_plus),
                                                   (x.minus, x.flux_minus, x.imposed_minus))):
        face = x.info[:, side].long()
        turn = x.info[:, 2].long() if side else torch.zeros_like(face)
        for v in range(16):
            rows = (face * 4 + turn == v).nonzero()[:, 0]
            if not len(rows):
                continue
            e = cells[rows].long()
            D, off = [], 0
            for d in range(order):
                m = num_basis(order - d)
                D.append(x.derivatives[e, off:off + 9 * m].reshape(-1, 9, m).to(F64) @ V[v // 4, v % 4, :, :m].T)
                off += 9 * m
            for o in range(order):
                at = sum(coeffs[o, d] * D[d] for d in range(order))
                q[side, rows, o] = torch.bmm(TinvT[rows], at)
            GF = torch.bmm(flux[rows].reshape(-1, 9, 9), imposed[rows])  # [p][point]
            dofs[e] += GF @ VTW[v // 4, v % 4].T
    return [q[0], q[1], dofs]


def _exact_friction(case, seed):
    A, prm = _friction_inputs(case, seed)
    order = case["order"]
    tp, weights = gauss_times(order, 1e-3)
    delta = np.diff(tp, prepend=0.0)
    delta[-1] += tp[0]
    a, sl0, f0, muw, b, srw = (A[k] for k in ("rs_a", "rs_sl0", "rs_f0", "rs_muw", "rs_b", "rs_srw"))
    ie = A["imp_and_eta"][:, :, None]
    sr0, tol = prm.rs_sr0, prm.rs_slip_rate_tolerance
    qp, qm, stress = A["q_interpolated_plus"], A["q_interpolated_minus"], A["initial_stress"]
    tiny = 1e-45

    def state(ref, dt, v):
        low = (f0 - (b - a) * torch.log(v / sr0)).clamp_min(0.0)
        mu_ss = muw + (low - muw) / (1 + (v / srw) ** 8) ** 0.125
        c = mu_ss / a
        ss = a * (c.abs() + torch.log(sr0 / v * -torch.sign(c) * torch.expm1(-2 * c.abs())))
        pre = -v * (dt / sl0)
        return ss * -torch.expm1(pre) + torch.exp(pre) * ref

    def mu_of(v, psi):
        # a asinh(z exp(c)) = a (c + log(z + sqrt(z^2 + exp(-2 c)))), both written without overflow
        z, c = 0.5 / sr0 * v, psi / a
        big = c + torch.log(z + torch.sqrt(z * z + torch.exp(-2 * c.clamp_min(0.0))))
        w = z * torch.exp(c.clamp_max(10.0))
        large = c + torch.log2(z).clamp_min(0.0) * math.log(2.0) > 10.0
        return a * torch.where(large, big, torch.asinh(w))

    def dmu_of(v, psi):
        z, c = 0.5 / sr0 * v, psi / a
        return a * (0.5 / sr0) / torch.sqrt(z * z + torch.exp(-2 * c))

    psi, mu = A["state_variable"].clone(), A["mu"].clone()
    s1, s2 = A["slip_rate1"].clone(), A["slip_rate2"].clone()
    out = {k: A[k].clone() for k in FRICTION_OUTPUTS}
    m, pl = torch.zeros_like(out["imposed_state_plus"]), torch.zeros_like(out["imposed_state_plus"])
    time = FAULT_TIME
    for o in range(order):
        dt, start = float(delta[o]), time
        time += dt
        n = ie[:, 4] * (qm[:, o, 6] - qp[:, o, 6] + qp[:, o, 0] * ie[:, 7] + qm[:, o, 0] * ie[:, 9])
        t1 = ie[:, 5] * (qm[:, o, 7] - qp[:, o, 7] + qp[:, o, 3] * ie[:, 8] + qm[:, o, 3] * ie[:, 10])
        t2 = ie[:, 5] * (qm[:, o, 8] - qp[:, o, 8] + qp[:, o, 5] * ie[:, 8] + qm[:, o, 5] * ie[:, 10])
        normal = (n + stress[:, 0] + A["initial_pressure"]).clamp_max(0.0)
        shear = torch.hypot(stress[:, 3] + t1, stress[:, 5] + t2)
        inv = ie[:, 6]
        srm = torch.hypot(s1, s2).clamp_min(tiny)
        ref, mid = psi, srm.clone()
        outer = torch.ones((len(srm), 1), dtype=torch.bool, device="cuda")  # faces still iterating
        last = torch.ones_like(srm, dtype=torch.bool)
        for j in range(prm.rs_state_variable_updates):
            psi = torch.where(outer, state(ref, dt, mid), psi)
            test = srm.clone()
            if case["start"] == "closed_form" and j == 0:
                S, N = inv * shear, inv * normal.abs() * a
                c = S / N
                lv = math.log(2 * sr0) - psi / a + c + torch.log(-0.5 * torch.expm1(-2 * c))
                creep = (S > 0) & (N > 0) & (lv < math.log(0.5 * tol))
                test = torch.where(creep, torch.exp(lv).clamp_min(tiny), test)
            busy = outer.clone()
            for _ in range(prm.rs_max_slip_rate_updates):
                mf = mu_of(test, psi)
                g = -inv * (normal.abs() * mf - shear) - test
                done = busy & (g.abs() < tol).all(1, keepdim=True)
                mu = torch.where(done, mf, mu)
                busy = busy & ~done
                if not bool(busy.any()):
                    break
                dg = -inv * (normal.abs() * dmu_of(test, psi)) - 1.0
                test = torch.where(busy, (test - g / dg).clamp_min(tiny), test)
            out["convergence_inner"] &= (~busy | (g.abs() < tol)).to(torch.uint8)
            near = (test - srm).abs() < prm.rs_state_tolerance
            last = torch.where(outer, near, last)
            mid = torch.where(outer, 0.5 * (srm + test), mid)
            srm = torch.where(outer, test, srm)
            outer = outer & ~near.all(1, keepdim=True)
            if not bool(outer.any()):
                break
        out["convergence_outer"] &= last.to(torch.uint8)
        psi = state(ref, dt, mid)
        mu = mu_of(srm, psi)
        f1, f2 = stress[:, 3] + t1, stress[:, 5] + t2
        div = -mu * normal + ie[:, 5] * srm
        s1, s2 = srm * f1 / div, srm * f2 / div
        r1, r2 = t1 - ie[:, 5] * s1, t2 - ie[:, 5] * s2
        out["traction1"], out["traction2"] = r1, r2
        out["accumulated_slip"] += srm * dt
        out["slip1"] += s1 * dt
        out["slip2"] += s2 * dt
        began = (out["rupture_time_pending"] > 0) & (srm > 0.001)
        out["rupture_time"] = torch.where(began, torch.full_like(srm, start), out["rupture_time"])
        out["rupture_time_pending"][began] = 0
        weak = ((out["rupture_time"] > 0) & (out["rupture_time"] <= start) & (out["dyn_stress_time_pending"] > 0)
                & (mu <= muw + 0.05 * (f0 - muw)))
        out["dyn_stress_time"] = torch.where(weak, torch.full_like(srm, start), out["dyn_stress_time"])
        out["dyn_stress_time_pending"][weak] = 0
        out["peak_slip_rate"] = torch.maximum(out["peak_slip_rate"], srm)
        w = float(weights[o])
        for acc, q, sign, zp, zs in ((m, qm, -1.0, ie[:, 9], ie[:, 10]), (pl, qp, 1.0, ie[:, 7], ie[:, 8])):
            acc[:, 0] += w * n
            acc[:, 3] += w * r1
            acc[:, 5] += w * r2
            acc[:, 6] += w * (q[:, o, 6] + sign * zp * (n - q[:, o, 0]))
            acc[:, 7] += w * (q[:, o, 7] + sign * zs * (r1 - q[:, o, 3]))
            acc[:, 8] += w * (q[:, o, 8] + sign * zs * (r2 - q[:, o, 5]))
    out["state_variable"] = A["state_variable"] + (psi - A["state_variable"]) @ _device(stroud(order)[4]).T
    out.update(slip_rate1=s1, slip_rate2=s2, slip_rate_magnitude=srm, mu=mu, imposed_state_plus=pl,
               imposed_state_minus=m)
    return out


def _exact_train(case, seed):
    samples, params = _train_inputs(case, seed)
    x, p = samples.double(), params.double().requires_grad_(True)
    z = (x[:, :6] - p[:6].detach()) / p[6:12].detach()
    h = torch.tanh(z @ p[14:206].reshape(32, 6).T + p[206:238])
    h = torch.tanh(h @ p[238:1262].reshape(32, 32).T + p[1262:1294])
    y = h @ p[1294:1326] + p[1326]
    loss = (y - (x[:, 6] - p[12].detach()) / p[13].detach()).square().mean()
    g, = torch.autograd.grad(loss, p)
    m, v = 0.1 * g, 0.001 * g * g
    new = p.detach() - 3e-3 * (m / 0.1) / ((v / 0.001).sqrt() + 1e-8)
    new[:14] = p.detach()[:14]
    return [loss.detach().reshape(1), g, new, m, v]


def exact(case, seed):
    return {"step": _exact_step, "calls": _exact_step, "lts": _exact_lts, "fault": _exact_fault,
            "friction": _exact_friction, "train": _exact_train}[case["kind"]](case, seed)
