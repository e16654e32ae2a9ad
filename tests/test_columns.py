"""The step kernels over velocity columns (lines.h) at the edges of their tiles: 3 points an axis,
odd grids (velocities along the faces), 63 and 64 columns, tiles that end in a partial one, axes that do
not ascend; every stencil size they take; cells of internal and of every kind of boundary face.

Tolerance: a macroscopic field is a velocity sum of terms of the size rho, rho sqrt(R T), T and
rho (R T)^1.5, here of at most 2e4 terms, over 3 steps.  FP64 sums in two orders differ by a few
1e-16 sqrt(terms) a step, under 1e-13 of that size; the bar is 1e-12 of it.  FP32 storage rounds each
stored value to 6e-8 of itself: 1e-6 of that size."""
import ctypes
import dataclasses

import numpy as np
import pytest

import mixed_meshes as mm
from dugksfoam_amd import cases
from dugksfoam_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _descending(c):
    return dataclasses.replace(c, xi=c.xi[::-1].copy(), xi_weights=c.xi_weights[::-1].copy())


def _shuffled(c):
    p = np.random.default_rng(3).permutation(c.xi.size)
    return dataclasses.replace(c, xi=c.xi[p].copy(), xi_weights=c.xi_weights[p].copy())


CASES = {
    "1d_3": lambda: cases.fourier_flow(9, nv=3),
    "1d_64": lambda: cases.fourier_flow(9, nv=64),
    "1d_63": lambda: cases.fourier_flow(9, nv=63, K=2),
    "1d_open": lambda: cases.shock_tube(10, nv=9),
    "2d_3": lambda: cases.cavity(4, 3, xi_sigma=1.7),
    "2d_31": lambda: cases.cavity(5, 31),
    "2d_64": lambda: cases.cavity(3, 64, K=1),
    "2d_61": lambda: cases.cavity(3, 61),
    "2d_descending": lambda: _descending(cases.cavity(4, 12)),
    "2d_shuffled": lambda: _shuffled(cases.cavity(4, 9)),
    "triangles_25": lambda: cases.delaunay_cavity(30, 5, nv=25),
    "triangles_64": lambda: cases.delaunay_cavity(30, 5, nv=64),
    "cyclic": lambda: cases.channel(8, 4, 2.0, 1.0, nv=11),
    "symmetry": lambda: cases.symmetry_cavity(4, 8, nv=11),
    "plane": lambda: cases.symmetry_cavity(4, 8, nv=28, kind="symmetryPlane"),
    "pressure": lambda: cases.pressure_channel(8, 4, nv=27),
    "zero_gradient": lambda: cases.open_channel(8, 4, nv=13, outlet="zeroGradient"),
    "batch": lambda: cases.batch(n_cases=3, nmin=3, nmax=5, nv=10, seed=2),
    "3d_3": lambda: cases.cavity(3, 3, dim=3, xi_sigma=1.7),
    "3d_8_K2": lambda: cases.cavity(3, 8, dim=3, K=2),
    "3d_9": lambda: cases.cavity(4, 9, dim=3),
    "3d_21": lambda: cases.cavity(3, 21, dim=3),
    "3d_shuffled": lambda: _shuffled(cases.cavity(3, 6, dim=3, K=1)),
}


def _off(c, a, b):
    """Largest difference of two sets of fields over the size of the terms they sum."""
    rt = c.R * np.max(b["T"])
    size = dict(rho=np.max(b["rho"]), U=np.sqrt(rt), T=np.max(b["T"]), q=np.max(b["rho"]) * rt ** 1.5)
    return max(float(np.max(np.abs(a[k] - b[k])) / size[k]) for k in size)


@pytest.mark.parametrize("which", list(CASES))
def test_columns_match_the_oracle(which, oracle_lib, monkeypatch):
    c = CASES[which]()
    o = oracle_lib.Oracle(c)
    o.init_equilibrium()
    o.step(nsteps=3)
    for storage, tol in (("fp64", 1e-12), ("fp32", 1e-6)):
        print(which, storage, flush=True)
        e = Engine(c, storage=storage)
        assert e.face_values() and e.face_mfma() and e.blocks()[0] == 64
        e.init_equilibrium()
        e.step(nsteps=3)
        assert _off(c, e.macro(), o.macro()) <= tol
        assert _off(c, e.face_macro(), o.face_macro()) <= tol
        # the state image holds the velocities in the order of the other layout, both ways
        monkeypatch.setenv("DUGKS_FACE_MFMA", "0")
        r = Engine(c, storage=storage)
        monkeypatch.delenv("DUGKS_FACE_MFMA")
        img = e.save_state()
        r.init_equilibrium()
        r.load_state(img)
        assert r.save_state() == img
        cells = np.arange(c.n_cells, dtype=np.int32)
        for x, y in zip(e.df(cells), r.df(cells)):
            assert np.array_equal(x, y)
        r.step(nsteps=2)
        e.load_state(img)
        e.step(nsteps=2)
        assert _off(c, e.macro(), r.macro()) <= tol
        e.close()
        r.close()
    o.close()


def _on_columns(e):
    """True when the engine runs the column kernels: they have one shape, and nothing is tuned."""
    e.autotune(True)
    left = e.autotune_steps_left()
    e.autotune(False)
    return left == 0


def _box(dim, cells, name, nv, K=0, **sides):
    """The unit square or cube of the given cells; walls, the y1 one moving, but for `sides`."""
    p = {a + s: mm.wall(20.0 if a + s == "y1" else 0.0) for a in "xyz"[:dim] for s in "01"}
    p.update(sides)
    return mm.build(name, *cells, mm.box_side(dim), p, dim, nv, K=K)


def _islands_2d(K, first):
    """Four triangles and two quads, each cell on its own.  The first two triangles couple their vertical edges
    (a cyclic pair); the first face of the third is a far field; the fourth has walls only."""
    pts, cells = [], []
    shapes = [[(0, 0), (1, 0), (0, 1)], [(5, 0), (5, 1), (4, 1)], [(6, 0), (7, 0), (6, 1)], [(8, 0), (9, 0), (9, 1)],
              [(10, 0), (11, 0), (11, 1), (10, 1)], [(11, 0), (12, 0), (12, 1), (11, 1)]]
    for s in shapes:
        n = len(pts)
        pts += [(x, y, z) for z in (0.0, 0.1) for x, y in s]
        k = len(s)
        cells.append(mm._prism(list(range(n, n + k)), list(range(n + k, n + 2 * k))))

    def patch(x, n):
        if abs(n[2]) > 0.9:
            return None
        if abs(n[0]) > 0.999 and x[0] in (0.0, 5.0):
            return "c0" if x[0] == 0.0 else "c1"
        return "far" if abs(x[0] - 6.0) < 1e-9 else "walls"

    kinds = {"c0": mm.cyclic(1), "c1": mm.cyclic(0), "far": first, "walls": mm.wall(15.0)}
    return mm.build("islands", pts, cells, patch, kinds, 2, 13, K=K)


def _islands_3d(K):
    """Single prisms and tetrahedra: two prisms coupled by a cyclic pair, a tetrahedron with a far field first,
    one with walls only."""
    pts, cells = [], []
    for s in ([(0, 0), (1, 0), (0, 1)], [(5, 0), (5, 1), (4, 1)]):
        n = len(pts)
        pts += [(x, y, z) for z in (0.0, 1.0) for x, y in s]
        cells.append(mm._prism([n, n + 1, n + 2], [n + 3, n + 4, n + 5]))
    for x in (6.0, 8.0):
        n = len(pts)
        pts += [(x, 0, 0), (x + 1, 0, 0), (x, 1, 0), (x, 0, 1)]
        cells.append([[n + i for i in range(4) if i != j] for j in range(4)])

    def patch(x, n):
        if abs(n[0]) > 0.999 and x[0] in (0.0, 5.0):
            return "c0" if x[0] == 0.0 else "c1"
        return "far" if abs(x[0] - 6.0) < 1e-9 else "walls"

    kinds = {"c0": mm.cyclic(1), "c1": mm.cyclic(0), "far": mm.far_field, "walls": mm.wall(15.0)}
    return mm.build("islands3d", pts, cells, patch, kinds, 3, 7, K=K)


def _strip(nz=1):
    """Quads (hexahedra) in one row between walls, every third column cut into two triangles (prisms): each
    cell has a wall."""
    return mm.split_columns(7, 1, nz, lambda i, j: i % 3 != 1)


# Cells with fewer faces than the kernels have slots, each with a wall or an open face
PADDED = {
    "strip": lambda: _box(2, _strip(), "strip", 12),
    "strip_odd_K2": lambda: _box(2, _strip(), "strip", 9, K=2),
    "strip_cyclic": lambda: _box(2, _strip(), "strip", 13, x0=mm.cyclic(1), x1=mm.cyclic(0)),
    "strip_pressure": lambda: _box(2, _strip(), "strip", 11, K=2, x0=mm.pressure_in, x1=mm.far_field),
    "strip_zero_gradient": lambda: _box(2, _strip(), "strip", 10, x0=mm.far_field, x1=mm.zero_gradient),
    "strip_mirror": lambda: _box(2, _strip(), "strip", 11, y0=mm.mirror("symmetryMod")),
    "strip_plane": lambda: _box(2, _strip(), "strip", 8, y0=mm.mirror("symmetryPlane")),
    "islands": lambda: _islands_2d(0, mm.far_field),
    "islands_K2": lambda: _islands_2d(2, mm.pressure_in),
    "prisms": lambda: _box(3, _strip(3), "prisms", 7),
    "prisms_K2": lambda: _box(3, _strip(2), "prisms", 6, K=2, x0=mm.cyclic(1), x1=mm.cyclic(0)),
    "pyramids": lambda: _box(3, mm.split_pyramids(1, lambda i, j, k: True), "pyramids", 9, z1=mm.far_field),
    "pyramids_K2": lambda: _box(3, mm.split_pyramids(1, lambda i, j, k: True), "pyramids", 6, K=2),
    "islands_3d": lambda: _islands_3d(0),
    "islands_3d_K2": lambda: _islands_3d(2),
}


@pytest.mark.parametrize("which", list(PADDED))
def test_cells_with_fewer_faces_than_slots(which, oracle_lib):
    c = PADDED[which]()
    o = oracle_lib.Oracle(c)
    o.init_equilibrium()
    o.step(nsteps=4)
    for storage, tol in (("fp64", 1e-12), ("fp32", 1e-6)):
        print(which, storage, flush=True)
        e = Engine(c, storage=storage)
        assert _on_columns(e)
        e.init_equilibrium()
        e.step(nsteps=4)
        assert _off(c, e.macro(), o.macro()) <= tol
        assert _off(c, e.face_macro(), o.face_macro()) <= tol
        e.close()
    o.close()


def _used_memory(value=0xff):
    """Leaves freed device memory that holds NaNs, in blocks of the sizes that small engines allocate."""
    hip = ctypes.CDLL("libamdhip64.so")
    blocks = []
    for size in (1 << 12, 1 << 14, 1 << 16, 1 << 18, 1 << 20):
        for _ in range(40):
            q = ctypes.c_void_p()
            assert hip.hipMalloc(ctypes.byref(q), ctypes.c_size_t(size)) == 0
            assert hip.hipMemset(q, value, ctypes.c_size_t(size)) == 0
            blocks.append(q)
    assert hip.hipDeviceSynchronize() == 0
    for q in blocks:
        assert hip.hipFree(q) == 0


def _tri(split):
    return mm.split_columns(5, 4, 1, split)


# The same with internal and cyclic faces only
PADDED_PLAIN = {
    "triangles_and_quads": lambda: _box(2, _tri(lambda i, j: (i + 2 * j) % 3 == 0), "mixed", 13),
    "triangles_and_quads_K2": lambda: _box(2, _tri(lambda i, j: (i + 2 * j) % 3 != 0), "mixed", 10, K=2),
    "periodic": lambda: _box(2, _tri(lambda i, j: (i + j) % 2 == 0), "mixed", 12, x0=mm.cyclic(1), x1=mm.cyclic(0),
                             y0=mm.cyclic(3), y1=mm.cyclic(2)),
    "prisms": lambda: _box(3, mm.split_columns(4, 4, 3, lambda i, j: (i + j) % 2 == 0), "prisms", 7),
    "pyramids": lambda: _box(3, mm.split_pyramids(3, lambda i, j, k: (i + j + k) % 2 == 1), "pyramids", 6, K=2),
    "tetrahedra": lambda: _box(3, mm.tetrahedra(2), "tets", 9),
    "tetrahedra_K2": lambda: _box(3, mm.tetrahedra(2), "tets", 6, K=2, x0=mm.cyclic(1), x1=mm.cyclic(0), z0=mm.far_field),
}


@pytest.mark.parametrize("which", list(PADDED_PLAIN))
def test_inner_cells_with_fewer_faces_than_slots(which, oracle_lib):
    """Also in memory that held NaNs before: slots without a face hold no values of their own."""
    c = PADDED_PLAIN[which]()
    o = oracle_lib.Oracle(c)
    o.init_equilibrium()
    o.step(nsteps=4)
    for storage, tol in (("fp64", 1e-12), ("fp32", 1e-6)):
        print(which, storage, flush=True)
        _used_memory()
        e = Engine(c, storage=storage)
        assert _on_columns(e)
        e.init_equilibrium()
        e.step(nsteps=4)
        assert _off(c, e.macro(), o.macro()) <= tol
        assert _off(c, e.face_macro(), o.face_macro()) <= tol
        e.close()
    o.close()


@pytest.mark.parametrize("dt_over_tau", [3.88, 4.05])
def test_mass_where_one_minus_r_is_small(dt_over_tau):
    """S8 takes g~ from gbar through 1 / (1 - r), here 98 and -242.  The cell's mass must not see its rounding:
    gas at rest between plates of its own temperature, with a velocity grid whose sums are exact to 1e-17,
    keeps its mass to the nine roundings of one part in 2^53 from one gbar to the next, 1e-15 a step if all
    fell the same way."""
    c = cases.fourier_flow(20, 64, T_left=273.0, T_right=273.0, xi_sigma=9.0)
    tau = c.mu_ref / (c.R * 273.0)
    c = dataclasses.replace(c, mu_ref=c.mu_ref * (c.dt / dt_over_tau) / tau)
    e = Engine(c)
    assert _on_columns(e)
    e.init_equilibrium()
    e.step(nsteps=1)
    m = float(np.sum(c.V * e.macro()["rho"]))
    n = 2000
    e.step(nsteps=n)
    drift = (float(np.sum(c.V * e.macro()["rho"])) / m - 1.0) / n
    print("drift a step", drift, flush=True)
    assert abs(drift) <= 1e-15
    e.close()


def test_tuning_waits_for_kernels_that_have_shapes(oracle_lib):
    """Switched on while the column kernels run, the tuner starts with the first step of other kernels, as
    dugks_set_face_values(h, 0) brings them."""
    c = cases.cavity(6, 12)
    e = Engine(c)
    e.autotune(True)
    assert e.autotune_steps_left() == 0
    e.init_equilibrium()
    e.step(nsteps=2)
    e.set_face_values(False)
    left = e.autotune_steps_left()
    assert left > 0
    e.step(nsteps=left)
    assert e.autotune_steps_left() == 0
    o = oracle_lib.Oracle(c)
    o.init_equilibrium()
    o.step(nsteps=2 + left)
    assert _off(c, e.macro(), o.macro()) <= 1e-12
    e.close()
    o.close()


@pytest.mark.parametrize("which,storage", [("2d", "fp64"), ("2d", "fp32"), ("cyclic_K2", "fp64"), ("1d", "fp64"),
                                           ("3d_K2", "fp32"), ("prisms", "fp64")])
def test_rows_follow_the_kernels(which, storage, oracle_lib, monkeypatch):
    """Without face values the engine is the one that never had columns: the same shapes and bits.  Switched to
    and fro between steps it keeps its state: as far from the oracle as without (3 + 2 + 2 steps)."""
    c = {"2d": lambda: cases.cavity(5, 41), "cyclic_K2": lambda: cases.channel(8, 4, 2.0, 1.0, nv=11, K=2),
         "1d": lambda: cases.fourier_flow(9, nv=63), "3d_K2": lambda: cases.cavity(3, 9, dim=3, K=2),
         "prisms": lambda: _box(3, _strip(3), "prisms", 7)}[which]()
    tol = 1e-12 if storage == "fp64" else 1e-6
    e = Engine(c, storage=storage)
    columns = e.blocks()
    e.set_face_values(False)
    monkeypatch.setenv("DUGKS_FACE_MFMA", "0")
    r = Engine(c, storage=storage)
    monkeypatch.delenv("DUGKS_FACE_MFMA")
    r.set_face_values(False)
    assert e.blocks() == r.blocks() and e.cell_blocks() == r.cell_blocks()
    for x in (e, r):
        x.init_equilibrium()
        x.step(nsteps=3)
    cells = np.arange(c.n_cells, dtype=np.int32)
    for a, b in ((e.macro(), r.macro()), (e.face_macro(), r.face_macro())):
        assert all(np.array_equal(a[k], b[k]) for k in a)
    assert all(np.array_equal(a, b) for a, b in zip(e.df(cells), r.df(cells)))
    e.set_face_values(True)
    assert _on_columns(e) and e.blocks() == columns
    assert all(np.array_equal(a, b) for a, b in zip(e.df(cells), r.df(cells)))
    img = r.save_state()
    e.load_state(img)
    assert all(np.array_equal(a, b) for a, b in zip(e.df(cells), r.df(cells)))
    e.step(nsteps=2)
    e.set_face_values(False)
    e.step(nsteps=2)
    o = oracle_lib.Oracle(c)
    o.init_equilibrium()
    o.step(nsteps=7)
    assert _off(c, e.macro(), o.macro()) <= tol
    assert _off(c, e.face_macro(), o.face_macro()) <= tol
    e.load_state(img)
    assert all(np.array_equal(a, b) for a, b in zip(e.df(cells), r.df(cells)))
    for x in (e, r):
        x.step(nsteps=2)
    a, b = e.macro(), r.macro()
    assert all(np.array_equal(a[k], b[k]) for k in a)
    for x in (e, r):
        x.close()
    o.close()
