"""The FP64 brick kernel (rh_brick64.h) at the sizes where it can go wrong,
against the CPU oracle: boxes smaller than a brick, one oct over a multiple of
a brick, bricks of one oct layer (whose split halves hold none), interior-wave
and row-major thread orders, every solver with every one-dimensional slope, the
general body (gravity) beside the specialised one.

Bar: 1e-12 relative per conserved variable for one step (a few hundred rounding
errors of 1e-16 on values of order one), as the other FP64 parity tests.
"""
import numpy as np
import pytest

from ramses2_amd import HydroParams, UniformLevel, UniformMesh, ic
from ramses2_amd.autotune import DEFAULT_SHAPE
from ramses2_amd.hydro import HipHydro
from tests.helpers import oracle_params, oracle_uniform, rel_err_per_var

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _steps(ncell, p, brick, seed, nsteps=2, gravity=(0.0, 0.0, 0.0)):
    """(device-resident steps, oracle steps) of a random box from the same state."""
    mesh = UniformMesh.for_cells(3, ncell)
    cells = ic.random_state((ncell,) * 3, np.random.default_rng(seed), gamma=p.gamma)
    HipHydro.set_brick_shape(*brick)
    try:
        lev = UniformLevel(mesh, cells, p)
    finally:
        HipHydro.set_brick_shape(*DEFAULT_SHAPE)
    om = oracle_uniform(mesh, lev.state())
    for d in range(3):
        om.m.constant_gravity[d] = gravity[d]
    po = oracle_params(p)
    for _ in range(nsteps):
        dt = om.courant_fine(mesh.level, po)[4]
        om.set_unew(mesh.level)
        om.godunov_fine(mesh.level, dt, po)
        om.set_uold(mesh.level)
    lev.run_device(nsteps, gravity=gravity)
    return lev.state(), om.uold


@pytest.mark.parametrize("brick", [(8, 6, 8), (4, 4, 4), (7, 7, 4), (3, 3, 8)])
@pytest.mark.parametrize("ncell", [4, 18, 26])
def test_partial_bricks(brick, ncell):
    p = HydroParams(gamma=1.4, courant_factor=0.5, slope_type=2, riemann="hllc")
    g, o = _steps(ncell, p, brick, ncell)
    assert np.all(rel_err_per_var(g, o) < TOL), rel_err_per_var(g, o)


@pytest.mark.parametrize("riemann", ["llf", "hll", "hllc"])
@pytest.mark.parametrize("slope", [0, 1, 2])
@pytest.mark.parametrize("brick", [(8, 6, 8), (7, 7, 8)])
def test_solvers_and_slopes(brick, slope, riemann):
    p = HydroParams(gamma=5.0 / 3.0, courant_factor=0.8, slope_type=slope, riemann=riemann)
    g, o = _steps(20, p, brick, 7 * slope + len(riemann))
    assert np.all(rel_err_per_var(g, o) < TOL), rel_err_per_var(g, o)


@pytest.mark.parametrize("riemann", ["llf", "hll", "hllc"])
def test_gravity_runs_the_general_body(riemann):
    p = HydroParams(gamma=1.4, courant_factor=0.5, slope_type=2, riemann=riemann)
    g, o = _steps(20, p, (8, 6, 8), 3, gravity=(0.5, -0.25, 0.125))
    assert np.all(rel_err_per_var(g, o) < TOL), rel_err_per_var(g, o)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("brick", [(8, 6, 8), (4, 4, 4)])
def test_parts_of_a_brick_give_the_whole_bricks_bits(brick, precision):
    """A batch of few bricks cuts each into parts along z, a batch that fills
    the chip does not (zsplit_for): the same job steps bit for bit alike in
    both, its sums to rounding."""
    from ramses2_amd.serving import HipEngine, JobSpec
    eng = HipEngine(precision=precision, brick=brick)
    job = JobSpec(0, 0.0, 34, 1, (1.0, 1e-3, 400.0, 16.0, 0.0), 3)
    big = JobSpec(1, 0.0, 128, 1, (1.0, 1e-2, 100.0, 63.0, 0.0), 3)
    alone, mixed, filler = eng.open(job), eng.open(job), eng.open(big)
    try:
        for _ in range(3):
            eng.step([alone])
            eng.step([filler, mixed])
        assert np.array_equal(eng.state(alone, job), eng.state(mixed, job))
        a, m = eng.status(alone), eng.status(mixed)
        assert a["t"] == m["t"] and a["dt_next"] == m["dt_next"]
        for k in ("mass", "ekin", "eint"):
            assert abs(a[k] - m[k]) <= 1e-13 * abs(m[k])
    finally:
        for h in (alone, mixed, filler):
            eng.close(h)
        eng.close_all()


@pytest.mark.parametrize("brick", [(4, 4, 4), (3, 3, 8), (8, 6, 8), (1, 1, 1)])
@pytest.mark.parametrize("deterministic", [True, False])
def test_refined_mesh_body_without_boundary_code(brick, deterministic):
    """A refined block that is not aligned with the bricks, on a periodic mesh:
    the body without boundary ghosts and the general one do the same arithmetic
    (same bits where the refluxes have a fixed order), and meet the oracle."""
    from ramses2_amd._lib import call
    from ramses2_amd.hydro import AmrHierarchy
    from tests.amr_cases import oracle_mesh, oracle_step, restrict_all, smooth_state, two_level_mesh
    am = two_level_mesh(region=(4, 10), offset=(2, 0, 8))
    om = oracle_mesh(am, smooth_state(am, 5, blast=True), 0, 2)
    restrict_all(am, om)
    p = HydroParams(gamma=1.4, courant_factor=0.5, slope_type=2, riemann="hllc")
    states = []
    try:
        for spec in (1, 0):
            call("rh_set_specialized", spec)
            HipHydro.set_brick_shape(*brick)
            gpu = AmrHierarchy(am, om.uold.copy(), p, interpol_var=0, interpol_type=2, deterministic=deterministic)
            gpu.run_device(2)
            states.append(gpu.state())
    finally:
        call("rh_set_specialized", 1)
        call("rh_set_deterministic", 0)
        HipHydro.set_brick_shape(*DEFAULT_SHAPE)
    if deterministic:
        assert np.array_equal(states[0], states[1])
    for _ in range(2):
        oracle_step(am, om, p)
    for s in states:
        assert np.all(rel_err_per_var(s, om.uold) < TOL)
