"""Flags of one level's octs (rh_get_flag1) against the whole mesh's
(rh_transfer_flag1_host), whole numbers: every level of a refined mesh and a
level of more octs than one grid of the count covers in a single round."""
import numpy as np
import pytest

from ramses2_amd import HydroParams, _lib
from ramses2_amd._lib import HipError, call, ptr
from ramses2_amd.hydro import AmrHierarchy
from tests.amr_cases import oracle_mesh, restrict_all, smooth_state, three_level_mesh, two_level_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh", ["three", "large"])
def test_level_flags_are_the_mesh_flags(mesh):
    am = three_level_mesh() if mesh == "three" else two_level_mesh(lo=6, region=(16, 50))
    om = oracle_mesh(am, smooth_state(am, 3, blast=True), 0, 1)
    restrict_all(am, om)
    p = HydroParams(gamma=1.4, courant_factor=0.5, slope_type=2, riemann="hllc")
    gpu = AmrHierarchy(am, om.uold.copy(), p)
    for l in am.levels:
        f, n = gpu.hh.hydro_flag(am.head[l], am.noct[l], p, 0.1, 0.1)
        whole = np.zeros((am.ngrid, 8), dtype=np.int32)
        call("rh_transfer_flag1_host", ptr(whole, _lib._ip), am.ngrid)
        assert f.shape == (am.noct[l], 8)
        assert np.array_equal(f, whole[am.head[l] - 1:am.head[l] - 1 + am.noct[l]])
        assert n == np.count_nonzero(f)
    with pytest.raises(HipError):
        call("rh_get_flag1", am.ngrid, 2, ptr(whole, _lib._ip))
