"""Meshes whose cells differ in their number of faces: triangles beside quads in 2-D; prisms,
pyramids, tetrahedra and hexahedra in 3-D; cells without internal faces."""
import itertools
import math

import numpy as np

from dugksfoam_amd import cases
from dugksfoam_amd.foam import cell_geometry, face_geometry

R, T0 = 208.0, 273.0


def _hull(points, cell):
    """The cell's faces as vertex lists, outward."""
    c = points[list(set(itertools.chain.from_iterable(cell)))].mean(axis=0)
    out = []
    for f in cell:
        Cf, Sf = face_geometry(points, [np.array(f)])
        out.append(tuple(f) if Sf[0] @ (Cf[0] - c) > 0 else tuple(reversed(f)))
    return out


def _prism(bottom, top):
    """Faces of the prism over a polygon: bottom, top, sides."""
    n = len(bottom)
    return [list(bottom), list(top)] + [[bottom[i], bottom[(i + 1) % n], top[(i + 1) % n], top[i]] for i in range(n)]


def build(name, points, cells, patch_of, patches, dim, nv, K=0, xi_sigma=4.0, kn=0.1):
    """A case of the given cells (lists of faces, each a list of points).  patch_of(centre, normal) names
    a boundary face's patch (None: an empty direction); patches: dict name -> maker(sides) in face order."""
    points = np.asarray(points, float)
    table = {}
    for c, cell in enumerate(cells):
        for f in _hull(points, cell):
            table.setdefault(tuple(sorted(f)), []).append((c, f))
    internal = sorted((v[0][0], v[1][0], v[0][1]) for v in table.values() if len(v) == 2)
    boundary = [v[0] for v in table.values() if len(v) == 1]
    own = np.array([i[0] for i in internal], dtype=np.int64)
    nei = np.array([i[1] for i in internal], dtype=np.int64)
    faces = [np.array(i[2]) for i in internal] + [np.array(b[1]) for b in boundary]
    Cf, Sf = face_geometry(points, faces)
    owner = np.concatenate([own, [b[0] for b in boundary]]).astype(np.int64)
    C, V = cell_geometry(Cf, Sf, owner, nei, len(cells))
    nfi = own.size
    sides = {k: [] for k in patches}
    for f in range(nfi, len(faces)):
        k = patch_of(Cf[f], Sf[f] / np.linalg.norm(Sf[f]))
        if k is not None:
            sides[k].append(f)
    pl = []
    for k, make in patches.items():
        s = sorted(sides[k], key=lambda f: tuple(np.round(Cf[f], 9)))
        pl.append(make(k, dict(owner=owner[s], Sf=Sf[s], Cf=Cf[s])))
    geo = cases._assemble(name, dim, C, V, own, nei, Sf[:nfi], Cf[:nfi], pl)
    xi_max = xi_sigma * math.sqrt(R * T0)
    xi, w = cases.dv_newton_cotes(xi_max, nv)
    dt = cases.fv_courant_dt(geo["V"], geo["owner"], geo["neighbour"], geo["Sf"], nfi, math.sqrt(dim) * xi_max, 0.5)
    mu = cases.mu_from_kn(kn, R, T0, 1.0)
    c = cases._finish(geo, xi, w, xi_max, R, 0.5, T0, mu, 2.0 / 3.0, K, 1.0, T0, dt)
    s = np.sin(2 * np.pi * c.C + np.arange(3))
    a = math.sqrt(R * T0)
    c.rho0 = 1.0 + 0.03 * s[:, 0] * s[:, 1]
    c.T0 = T0 * (1.0 + 0.02 * s[:, 1] * s[:, 2])
    c.U0 = np.where(np.arange(3) < dim, 0.05 * a * s[:, [1, 2, 0]], 0.0)
    return c


def wall(u=0.0, T=T0):
    return lambda name, sd: cases._wall(name, sd, (u, 0.0, 0.0), T)


def cyclic(other):
    """other: index of the coupled patch."""
    return lambda name, sd: cases.Patch(name, cases.PATCH_CYCLIC, sd["owner"], sd["Sf"], sd["Cf"], neighbour_patch=other)


def far_field(name, sd):
    n = sd["owner"].size
    return cases.Patch(name, cases.PATCH_FARFIELD, sd["owner"], sd["Sf"], sd["Cf"], T=np.full(n, T0), rho=np.full(n, 1.02))


def pressure_in(name, sd):
    return cases.Patch(name, cases.PATCH_PRESSURE_IN, sd["owner"], sd["Sf"], sd["Cf"], T=np.full(sd["owner"].size, T0),
                       pressure=1.05 * R * T0)


def zero_gradient(name, sd):
    return cases.Patch(name, cases.PATCH_ZEROGRADIENT, sd["owner"], sd["Sf"], sd["Cf"])


def mirror(kind):
    t = {"symmetryMod": cases.PATCH_SYMMETRY, "symmetryPlane": cases.PATCH_SYMMETRY_PLANE}[kind]
    return lambda name, sd: cases.Patch(name, t, sd["owner"], sd["Sf"], sd["Cf"])


def box_side(dim, lo=0.0, hi=1.0):
    """Names the side of a box that a boundary face lies on; None across the empty directions."""
    def side(x, n):
        a = int(np.argmax(np.abs(n)))
        if a >= dim:
            return None
        if abs(x[a] - lo) < 1e-9 and n[a] < -0.999:
            return "xyz"[a] + "0"
        if abs(x[a] - hi) < 1e-9 and n[a] > 0.999:
            return "xyz"[a] + "1"
        raise ValueError("not on the box")
    return side


def grid_points(nx, ny, nz, dz=0.1):
    """Points of a grid on the unit square or cube (nz = 1: one cell of thickness dz)."""
    z = np.array([0.0, dz]) if nz == 1 else np.linspace(0, 1, nz + 1)
    X = np.stack(np.meshgrid(np.linspace(0, 1, nx + 1), np.linspace(0, 1, ny + 1), z, indexing="ij"), -1)
    return X.reshape(-1, 3), lambda i, j, k: (i * (ny + 1) + j) * (z.size) + k


def split_columns(nx, ny, nz, split):
    """Hexahedra; the columns that split(i, j) picks are cut into two prisms along a diagonal, which
    alternates."""
    pts, v = grid_points(nx, ny, nz)
    cells = []
    for i, j, k in itertools.product(range(nx), range(ny), range(nz)):
        q = [(i, j), (i + 1, j), (i + 1, j + 1), (i, j + 1)]
        parts = [q]
        if split(i, j):
            parts = [[q[0], q[1], q[2]], [q[0], q[2], q[3]]] if (i + j) % 2 else [[q[0], q[1], q[3]], [q[1], q[2], q[3]]]
        cells += [_prism([v(a, b, k) for a, b in p], [v(a, b, k + 1) for a, b in p]) for p in parts]
    return pts, cells


def split_pyramids(n, split):
    """Hexahedra; those that split(i, j, k) picks are cut into six pyramids about their centre."""
    pts, v = grid_points(n, n, n, dz=1.0)
    pts, cells = list(pts), []
    for i, j, k in itertools.product(range(n), repeat=3):
        q = [v(i, j, k), v(i + 1, j, k), v(i + 1, j + 1, k), v(i, j + 1, k)]
        t = [v(i, j, k + 1), v(i + 1, j, k + 1), v(i + 1, j + 1, k + 1), v(i, j + 1, k + 1)]
        hexa = _prism(q, t)
        if not split(i, j, k):
            cells.append(hexa)
            continue
        m = len(pts)
        pts.append((np.array([i, j, k]) + 0.5) / n)
        cells += [[f] + [[f[a], f[(a + 1) % 4], m] for a in range(4)] for f in hexa]
    return np.array(pts), cells


def tetrahedra(n):
    """n^3 cubes of five tetrahedra each, mirrored from cube to cube so that they meet face to face."""
    pts, v = grid_points(n, n, n, dz=1.0)
    cells = []
    for i, j, k in itertools.product(range(n), repeat=3):
        at = lambda b: v(i + (b & 1), j + (b >> 1 & 1), k + (b >> 2 & 1))
        flip = 7 if (i + j + k) % 2 else 0
        for t in ((0, 1, 2, 4), (3, 1, 2, 7), (5, 1, 4, 7), (6, 2, 4, 7), (1, 2, 4, 7)):
            p = [at(b ^ flip) for b in t]
            cells.append([list(f) for f in itertools.combinations(p, 3)])
    return pts, cells


def merge(cells, pairs):
    """Joins cells a, b of each pair over the faces they share."""
    out = list(cells)
    for a, b in pairs:
        fa = {tuple(sorted(f)): f for f in cells[a]}
        fb = {tuple(sorted(f)): f for f in cells[b]}
        out[a] = [f for k, f in fa.items() if k not in fb] + [f for k, f in fb.items() if k not in fa]
        out[b] = None
    return [c for c in out if c is not None]


def pairs(n):
    """n^3 hexahedra (n even), every other one joined to its neighbour along x: 10 faces."""
    pts, cells = split_columns(n, n, n, lambda i, j: False)
    at = lambda i, j, k: (i * n + j) * n + k
    return pts, merge(cells, [(at(i, j, k), at(i + 1, j, k)) for i in range(0, n, 2) for j in range(n) for k in range(n)
                              if (i // 2 + j + k) % 2 == 0])


def pentagons(n):
    """The columns of n^3 hexahedra (n even) by twos along x: the first with half of the second, a prism over a
    pentagon (7 faces), and the other half, a prism over a triangle."""
    pts, v = grid_points(n, n, n, dz=1.0)
    cells = []
    for i, j, k in itertools.product(range(0, n, 2), range(n), range(n)):
        p, q = (i, j), (i, j + 1)
        a, b, c, d = (i + 1, j), (i + 2, j), (i + 2, j + 1), (i + 1, j + 1)
        parts = [[p, a, b, d, q], [b, c, d]] if j % 2 else [[p, a, c, d, q], [a, b, c]]
        cells += [_prism([v(x, y, k) for x, y in r], [v(x, y, k + 1) for x, y in r]) for r in parts]
    return pts, cells
