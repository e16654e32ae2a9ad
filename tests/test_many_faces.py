"""Cells of more faces than the column kernels take (4 in 2-D, 6 in 3-D), which keep k_face_values,
k_face_moments_mx and k_cell: the steps, the matrix-core face moments against the vector sums, the fused
tail of k_cell against kernels of its own, and the online tuner, which has shapes to choose from there only.

Tolerances: those of the column kernels' test (sums of up to 2e4 terms in two orders: 1e-12 of the terms'
size, 1e-6 with FP32 storage, over 4 steps; roundings add up at most in proportion to the steps); the two forms of the tail are the same arithmetic and bit-identical."""
import numpy as np
import pytest

import mixed_meshes as mm
from dugksfoam_amd import cases
from dugksfoam_amd.engine import Engine
from test_columns import _box, _off

pytestmark = pytest.mark.gpu

CASES = {
    "polygons": lambda: cases.agglomerated_cavity(9, nv=12, block=3),
    "polygons_K1": lambda: cases.agglomerated_cavity(12, nv=9, block=4, K=1),
    "polyhedra_7": lambda: _box(3, mm.pentagons(4), "pentagons", 8),
    "polyhedra_7_K2": lambda: _box(3, mm.pentagons(4), "pentagons", 7, K=2, z0=mm.cyclic(5), z1=mm.cyclic(4)),
    "polyhedra_10": lambda: _box(3, mm.pairs(4), "pairs", 9),
    "polyhedra_10_K2": lambda: _box(3, mm.pairs(4), "pairs", 6, K=2, z1=mm.far_field),
}


def _run(c, storage, n):
    e = Engine(c, storage=storage)
    e.init_equilibrium()
    e.step(nsteps=n)
    return e


@pytest.mark.parametrize("storage,tol", [("fp64", 1e-12), ("fp32", 1e-6)])
@pytest.mark.parametrize("which", list(CASES))
def test_steps_and_variants(which, storage, tol, oracle_lib, monkeypatch):
    c = CASES[which]()
    o = oracle_lib.Oracle(c)
    o.init_equilibrium()
    o.step(nsteps=4)
    e = _run(c, storage, 4)
    assert e.face_mfma() and e.fused_cell()
    assert _off(c, e.macro(), o.macro()) <= tol and _off(c, e.face_macro(), o.face_macro()) <= tol
    monkeypatch.setenv("DUGKS_FACE_MFMA", "0")
    v = _run(c, storage, 4)
    monkeypatch.delenv("DUGKS_FACE_MFMA")
    assert not v.face_mfma()
    assert _off(c, v.macro(), e.macro()) <= tol and _off(c, v.face_macro(), e.face_macro()) <= tol
    monkeypatch.setenv("DUGKS_FUSE_S1", "0")
    u = _run(c, storage, 4)
    monkeypatch.delenv("DUGKS_FUSE_S1")
    assert not u.fused_cell()
    for a, b in ((u.macro(), e.macro()), (u.face_macro(), e.face_macro())):
        assert all(np.array_equal(a[k], b[k]) for k in a)
    # the tuner's candidates are real steps
    e.autotune(True)
    left = e.autotune_steps_left()
    assert left > 0
    e.step(nsteps=left)
    assert e.autotune_steps_left() == 0
    o.step(nsteps=left)
    assert _off(c, e.macro(), o.macro()) <= tol * (4 + left) / 4
    for x in (e, v, u):
        x.close()
    o.close()
