"""The batched AMR step's joint restriction and Courant pass on a level of more
octs than its blocks take in one round (262,144 of level 7, 65,536 of them per
round), and on one that ends inside a round, against the per-level calls, which
restrict and reduce in passes of their own.

Bar: 1e-12 per conserved variable after two steps (refluxes by atomics), dt to
1e-14, the sums to 1e-12, as the other batched-step tests."""
import numpy as np
import pytest

from ramses2_amd import HydroParams
from ramses2_amd.hydro import AmrHierarchy
from tests.amr_cases import smooth_state, two_level_mesh
from tests.helpers import rel_err_per_var

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lo,region", [(7, (32, 49)), (4, (4, 11))])
def test_batched_step_matches_the_calls(lo, region):
    am = two_level_mesh(lo=lo, region=region)
    u = smooth_state(am, 9, blast=True)
    p = HydroParams(gamma=1.4, courant_factor=0.5, slope_type=2, riemann="hllc")
    calls = AmrHierarchy(am, u.copy(), p, interpol_var=0, interpol_type=2)
    for _ in range(2):
        dt_used = calls.step()
    want = calls.state()
    per = np.array([[c[k] for k in ("mass", "ekin", "eint", "emag", "dt")] for c in map(calls.courant, am.levels)])
    dt_next = per[:, 4].min()
    batched = AmrHierarchy(am, u.copy(), p, interpol_var=0, interpol_type=2)
    dt, t, sums, _ = batched.run_device(2)
    assert np.all(rel_err_per_var(batched.state(), want) < 1e-12)
    assert abs(dt - dt_next) <= 1e-14 * dt_next
    assert np.all(np.abs(np.array(sums[:3]) - per[:, :3].sum(axis=0)) <= 1e-12 * np.abs(per[:, :3]).sum(axis=0))
    assert dt_used < t
