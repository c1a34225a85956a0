"""1D levels in units where the sound speed's floor is above 1 (smallc = 1e3,
speeds of 1e5), against the CPU oracle: within the one-launch path's sizes (both
cells-per-thread variants) and beyond, and with the floor in effect.

Bar: that of the 1D tests in units of order one, 1e-12 relative per conserved
variable after five steps, dt and time to 1e-13."""
import numpy as np
import pytest

from ramses2_amd import HydroParams, UniformLevel, UniformMesh, ic
from tests.helpers import oracle_params, oracle_uniform, rel_err_per_var

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("speed", [1e5, 10.0])
@pytest.mark.parametrize("riemann", ["llf", "hll", "hllc"])
@pytest.mark.parametrize("ncell", [64, 1000, 1026])
def test_smallc_above_one(ncell, riemann, speed):
    p = HydroParams(gamma=1.4, courant_factor=0.8, slope_type=1, riemann=riemann, smallc=1e3)
    mesh = UniformMesh.for_cells(1, ncell)
    cells = ic.sod_1d(ncell)
    cells[1:4] *= speed
    cells[4] *= speed ** 2
    lev = UniformLevel(mesh, cells, p, periodic=False)
    om = oracle_uniform(mesh, lev.state(), periodic=False)
    po = oracle_params(p)
    t = 0.0
    for _ in range(5):
        dt = om.courant_fine(mesh.level, po)[4]
        om.set_unew(mesh.level)
        om.godunov_fine(mesh.level, dt, po)
        om.set_uold(mesh.level)
        t += dt
    got = lev.run_device(5)
    assert abs(got[0] - dt) <= 1e-13 * dt and abs(got[1] - t) <= 1e-13 * t
    err = rel_err_per_var(lev.state(), om.uold)
    assert np.all(err < 1e-12), err
