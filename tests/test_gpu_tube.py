"""Small 1D levels stepped in one launch (rh_tube.hip) against the CPU oracle:
both cells-per-thread variants at their edges, one wave, outflow, reflexive and
periodic ends, every solver and slope, gravity, a fixed dt.

Bar: 1e-12 relative per conserved variable after five steps (the rounding of
some hundred operations per cell and step), dt and time to 1e-13.
"""
import numpy as np
import pytest

from ramses2_amd import HydroParams, UniformLevel, UniformMesh, ic
from tests.helpers import oracle_params, oracle_uniform, rel_err_per_var

pytestmark = pytest.mark.gpu


def _run(ncell, p, ends, nsteps=5, gravity=0.0, dt_fixed=0.0, seed=1):
    mesh = UniformMesh.for_cells(1, ncell)
    cells = ic.random_state((ncell,), np.random.default_rng(seed), vscale=0.5)
    periodic = ends == "periodic"
    bound = 1 if ends == "reflexive" else 2
    lev = UniformLevel(mesh, cells, p, periodic=periodic, bound_type=bound)
    om = oracle_uniform(mesh, lev.state(), periodic=periodic, bound_type=bound)
    om.m.constant_gravity[0] = gravity
    po = oracle_params(p)
    t = 0.0
    for _ in range(nsteps):
        c = om.courant_fine(mesh.level, po)
        dt = dt_fixed or c[4]
        om.set_unew(mesh.level)
        om.godunov_fine(mesh.level, dt, po)
        om.set_uold(mesh.level)
        t += dt
    got = lev.run_device(nsteps, dt_fixed=dt_fixed, gravity=(gravity, 0.0, 0.0))
    assert np.array_equal(lev.state(), lev.hh.transfer_unew_host())
    err = rel_err_per_var(lev.state(), om.uold)
    assert np.all(err < 1e-12), err
    assert abs(got[0] - dt) <= 1e-13 * dt and abs(got[1] - t) <= 1e-13 * t
    if not dt_fixed:
        assert np.allclose(got[2][:3], c[:3], rtol=1e-12, atol=0)


@pytest.mark.parametrize("ends", ["outflow", "reflexive", "periodic"])
@pytest.mark.parametrize("ncell", [8, 64, 1022, 1024, 1026, 2000, 2002])
def test_sizes_and_ends(ncell, ends):
    _run(ncell, HydroParams(gamma=1.4, courant_factor=0.8, slope_type=1, riemann="hllc"), ends)


@pytest.mark.parametrize("slope", [0, 1, 2])
@pytest.mark.parametrize("riemann", ["llf", "hll", "hllc"])
def test_solvers_and_slopes(riemann, slope):
    p = HydroParams(gamma=1.4, courant_factor=0.5, slope_type=slope, riemann=riemann)
    _run(130, p, "outflow", gravity=0.3)
    _run(130, p, "reflexive", dt_fixed=1e-4)


def test_long_call_equals_short_ones():
    """More steps than one launch takes, split anywhere, end on the same bits."""
    p = HydroParams(gamma=1.4, courant_factor=0.8, slope_type=1, riemann="hllc")
    mesh = UniformMesh(1, 7)
    a, b = (UniformLevel(mesh, ic.sod_1d(128), p, periodic=False) for _ in range(2))
    a.run_device(4100)
    for k in (1, 99, 4000):
        b.run_device(k, use_graph=True)
    assert np.array_equal(a.state(), b.state())
