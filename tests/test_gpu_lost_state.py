"""dt of a level that has lost its state: a NaN cell fails the compares of cmpdt
(hydro/godunov_utils.f90:228-337) and drops out of the minimum, so a level whose
cells are all NaN keeps the initial bound dx/smallc of courant_fine
(hydro/courant_fine.f90:60-75), in every precision, solver, body and step loop.

Exact: the bound is one quotient of two numbers of the host."""
import numpy as np
import pytest

from ramses2_amd import HydroParams, UniformLevel, UniformMesh
from ramses2_amd._lib import call
from ramses2_amd.autotune import DEFAULT_SHAPE
from ramses2_amd.hydro import AmrHierarchy, HipHydro
from ramses2_amd.mesh import prim_to_cons
from tests.amr_cases import two_level_mesh

pytestmark = pytest.mark.gpu


def _params(slope, riemann):
    return HydroParams(gamma=1.4, courant_factor=0.5, slope_type=slope, riemann=riemann)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("gravity", [0.0, 0.5])
@pytest.mark.parametrize("slope,riemann", [(2, "hllc"), (1, "llf"), (2, "hll"), (3, "hllc")])
@pytest.mark.parametrize("brick", [(8, 6, 8), (4, 4, 4), (7, 7, 8)])
def test_lost_level(brick, slope, riemann, gravity, precision):
    p = _params(slope, riemann)
    mesh = UniformMesh.for_cells(3, 20)
    HipHydro.set_brick_shape(*brick)
    try:
        lev = UniformLevel(mesh, np.full((5, 20, 20, 20), np.nan), p)
    finally:
        HipHydro.set_brick_shape(*DEFAULT_SHAPE)
    dt, t, _, _ = lev.run_device(3, precision=precision, gravity=(gravity, 0.0, 0.0))
    bound = mesh.dx / np.sqrt(p.smallc ** 2)
    assert dt == bound and t == 3 * bound


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("ncell", [64, 1024, 2048])
def test_lost_tube(ncell, precision):
    p = _params(1, "hllc")
    mesh = UniformMesh.for_cells(1, ncell)
    lev = UniformLevel(mesh, np.full((5, ncell), np.nan), p, periodic=False)
    dt, t, _, _ = lev.run_device(3, precision=precision)
    bound = mesh.dx / np.sqrt(p.smallc ** 2)
    assert dt == bound and t == 3 * bound


@pytest.mark.parametrize("precision", [0, 1])
def test_lost_refined_mesh(precision):
    p = _params(2, "hllc")
    am = two_level_mesh(region=(4, 8))
    gpu = AmrHierarchy(am, np.full((am.ngrid, 5, 8), np.nan), p, precision=precision)
    dt, _, _, _ = gpu.run_device(2)
    assert dt == am.dx(am.levelmax) / np.sqrt(p.smallc ** 2)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("brick", [(8, 6, 8), (4, 4, 4)])
def test_lost_job(brick, precision):
    from ramses2_amd.serving import HipEngine, JobSpec
    eng = HipEngine(_params(2, "hllc"), precision=precision, brick=brick)
    job = JobSpec(0, 0.0, 32, 1, (np.nan, np.nan, np.nan, 15.0, 0.0), 3)
    h = eng.open(job)
    try:
        eng.step([h], 3)
        st = eng.status(h)
    finally:
        eng.close(h)
        eng.close_all()
        call("rh_set_brick_shape", *DEFAULT_SHAPE)
    bound = (1.0 / 32) / np.sqrt(1e-10 ** 2)
    assert st["dt_next"] == bound and st["t"] == 3 * bound


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("slope", [1, 2])
@pytest.mark.parametrize("ndim,axis,brick", [(1, 0, (8, 6, 8)), (3, 0, (8, 6, 8)), (3, 1, (7, 7, 8)), (3, 2, (4, 4, 4))])
def test_lost_cell_in_a_supersonic_stream(ndim, axis, brick, slope, sign, precision):
    """HLLC takes the upwind state of a supersonic face, whatever lies downstream: a
    lost cell loses no cell upstream of it, and those further off than its
    neighbours' slopes reach keep their bits."""
    n, at, nsteps = 32, 16, 4
    rng = np.random.default_rng(8)
    full = (n,) * ndim
    vel = [np.zeros(full)] * 3
    vel[axis] = sign * (8.0 + rng.random(full))
    cells = prim_to_cons(0.5 + rng.random(full), vel, 0.5 + rng.random(full), 1.4)
    ax = ndim - axis  # of a (5, ...) array
    out = []
    for lost in (True, False):
        c = cells.copy()
        if lost:
            c[(slice(None),) + (at,) * ndim] = np.nan
        HipHydro.set_brick_shape(*brick)
        try:
            lev = UniformLevel(UniformMesh.for_cells(ndim, n), c, _params(slope, "hllc"))
        finally:
            HipHydro.set_brick_shape(*DEFAULT_SHAPE)
        lev.run_device(nsteps, dt_fixed=0.5 / (n * 12.0), precision=precision)
        out.append(np.moveaxis(lev.cells(), ax, 1))
    up = [at - sign * k for k in range(1, 9)]
    assert np.isnan(out[0][:, at]).any()
    assert np.all(np.isfinite(out[0][:, up]))
    far = up[nsteps + 1:]
    assert np.array_equal(out[0][:, far], out[1][:, far])
