"""The adjoint's workgroup shapes (64, 128 and 256 lanes a point, rows in LDS or in memory) against the
host build of the same code, at sizes on both sides of each rule.

Tolerance: J sums fluxes c_f rho sqrt(R T) |S_f| of either sign over faces, velocities and steps; two
summation orders differ by a few 1e-16 of that size a step, 1e-13 of it is the bar.  The gradient's
terms do not cancel like that: 1e-11 of its largest entry (its parity with the host build is 1e-14 to
1e-13 on the small cases)."""
import numpy as np
import pytest

from adjoint_cases import random_problem
from adjoint_host import HostAdjoint
from dugksfoam_amd import cases
from dugksfoam_amd.adjoint import Adjoint

pytestmark = pytest.mark.gpu

SHAPES = {
    "64_lanes": lambda: cases.cavity(46, 8),
    "64_lanes_81": lambda: cases.cavity(46, 9),
    "128_lanes_few_points": lambda: cases.cavity(6, 9),
    "128_lanes": lambda: cases.cavity(33, 12),
    "256_lanes": lambda: cases.channel(8, 4, 2.0, 1.0, nv=12),
    "256_lanes_tail": lambda: cases.pressure_channel(6, 4, nv=17),
    "rows_in_lds_2025": lambda: cases.symmetry_cavity(3, 6, nv=45),
    "rows_in_memory_2116": lambda: cases.symmetry_cavity(3, 6, nv=46, kind="symmetryPlane"),
    "rows_in_memory_channel": lambda: cases.channel(6, 3, 2.0, 1.0, nv=46),
    "rows_in_memory_3d": lambda: cases.cavity(3, 13, dim=3, K=2),
}


@pytest.mark.parametrize("which", list(SHAPES))
def test_shapes_match_the_host_build(which):
    print(which, flush=True)
    c = SHAPES[which]()
    coef, _ = random_problem(c)
    steps = 4
    with Adjoint(c) as A:
        J, g = A.run(steps, 1, coef, checkpoint_every=2)
        m = A.macro()
    H = HostAdjoint(c)
    Jh, gh = H.run(steps, 1, coef, checkpoint_every=2)
    c0 = np.sqrt(c.R * np.max(c.T0))
    size = steps * np.max(c.rho0) * c0 * float(np.sum(np.abs(coef) * np.linalg.norm(c.Sf, axis=1)))
    assert abs(J - Jh) <= 1e-13 * size
    assert np.max(np.abs(g - gh)) <= 1e-11 * np.max(np.abs(gh))
    mh = H.macro()
    for k, s in (("rho", np.max(c.rho0)), ("U", c0), ("T", np.max(c.T0))):
        assert np.max(np.abs(m[k] - mh[k])) <= 1e-12 * s
