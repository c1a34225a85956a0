"""dt of the batched AMR step under gravity (each cell's own dt is formed and the
smallest taken) against the per-level Courant calls on the state it leaves.

Bar: 1e-14 in FP64 (a dozen roundings of 1.1e-16); 1e-6 in mixed precision, whose
signal speed and dt take about ten FP32 operations of 6e-8."""
import numpy as np
import pytest

from ramses2_amd import HydroParams
from ramses2_amd.hydro import AmrHierarchy
from tests.amr_cases import smooth_state, two_level_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [(0, 1e-14), (1, 1e-6)])
@pytest.mark.parametrize("interpol_var", [0, 1])
@pytest.mark.parametrize("gravity", [(0.5, -0.25, 0.125), (40.0, 0.0, -30.0)])
def test_batched_dt_under_gravity(gravity, interpol_var, precision, tol):
    am = two_level_mesh(region=(4, 11))
    p = HydroParams(gamma=1.4, courant_factor=0.5, slope_type=2, riemann="hllc")
    gpu = AmrHierarchy(am, smooth_state(am, 11), p, interpol_var=interpol_var, interpol_type=2, precision=precision)
    dt, _, sums, _ = gpu.run_device(2, gravity=gravity)
    c = [gpu.hh.cmpdt(am.head[l], am.noct[l], am.dx(l), p, gravity=gravity) for l in am.levels]
    want = min(x["dt"] for x in c)
    assert abs(dt - want) <= tol * want
    tot = np.array([[x[k] for k in ("mass", "ekin", "eint")] for x in c]).sum(axis=0)
    assert np.all(np.abs(np.array(sums[:3]) - tot) <= 1e-12 * np.abs(tot))
