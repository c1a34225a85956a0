"""Planar flows in 3D stay planar to the last bit: the fluxes through the two
faces of a transverse direction are equal, and their difference is taken before
it is added to the cell, so the transverse momenta stay 0.  Exact, in both
precisions, for every solver and thread order of the bricks."""
import numpy as np
import pytest

from ramses2_amd import HydroParams, UniformLevel, UniformMesh
from ramses2_amd.autotune import DEFAULT_SHAPE
from ramses2_amd.hydro import HipHydro
from ramses2_amd.mesh import prim_to_cons

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("riemann", ["llf", "hll", "hllc"])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("brick", [(8, 6, 8), (4, 4, 4), (7, 7, 8)])
def test_transverse_momenta_stay_zero(brick, axis, riemann, precision):
    n = 20
    left = np.arange(n) < n // 2
    shape = [1, 1, 1]
    shape[2 - axis] = n
    rho, p = (np.broadcast_to(np.where(left, a, b).reshape(shape), (n, n, n)) for a, b in ((1.0, 0.37), (0.7, 0.11)))
    z = np.zeros((n, n, n))
    mesh = UniformMesh.for_cells(3, n)
    HipHydro.set_brick_shape(*brick)
    try:
        lev = UniformLevel(mesh, prim_to_cons(rho, (z, z, z), p, 1.4),
                           HydroParams(gamma=1.4, courant_factor=0.5, slope_type=2, riemann=riemann))
    finally:
        HipHydro.set_brick_shape(*DEFAULT_SHAPE)
    lev.run_device(5, precision=precision)
    mom = lev.cells()[1:4]
    for d in range(3):
        if d != axis:
            assert not mom[d].any(), (d, np.abs(mom[d]).max())
    assert np.abs(mom[axis]).max() > 0.01
