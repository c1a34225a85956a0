"""The conservation sums of a job do not depend on the other jobs of its batch, bit
for bit, however the batch is cut into workgroups: alone (bricks in parts along z),
beside another small job, and beside one that fills the chip (whole bricks); by
status and by fence, and against the host's sums of the state."""
import ctypes
import math

import numpy as np
import pytest

from ramses2_amd import HydroParams
from ramses2_amd._lib import call, ptr
from ramses2_amd.serving import HipEngine, JobSpec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("slope,riemann", [(2, "hllc"), (1, "llf"), (2, "hll"), (3, "hllc")])
@pytest.mark.parametrize("brick", [(8, 6, 8), (4, 4, 4), (7, 7, 8), (15, 7, 8), (3, 3, 4), (1, 1, 1)])
@pytest.mark.parametrize("kind,ic", [(1, (1.0, 1e-3, 400.0, 16.0, 0.0)), (2, (1.3, 0.7, 0.3, 0.11, 2.0))])
def test_sums_do_not_depend_on_the_batch(kind, ic, brick, slope, riemann, precision):
    p = HydroParams(gamma=1.4, courant_factor=0.5, slope_type=slope, riemann=riemann)
    eng = HipEngine(p, precision=precision, brick=brick)
    job = JobSpec(0, 0.0, 34, kind, ic, 5)
    small, big = (JobSpec(1, 0.0, n, 1, (1.0, 1e-2, 100.0, n // 2 - 1.0, 0.0), 5) for n in (40, 128))
    batches = [[], [small], [big]]
    opened, res = [], []
    try:
        for others in batches:
            ids = [eng.open(s) for s in [job] + others]
            opened += ids
            for _ in range(5):
                eng.step(ids)
            st = eng.status(ids[0])
            assert eng.wait(eng.fence(ids[:1])) == [st]
            res.append((st, eng.state(ids[0], job)))
    finally:
        for h in opened:
            eng.close(h)
        eng.close_all()
    for st, u in res[1:]:
        assert np.array_equal(u, res[0][1])
        assert st == res[0][0]
    vol = eng._mesh_for(34)[0].dx ** 3
    mass, energy = (math.fsum(res[0][1][v].ravel()) * vol for v in (0, 4))
    # 39304 terms, added in 256 threads, their waves and blocks: far fewer roundings than 1e-13 allows
    assert abs(res[0][0]["mass"] - mass) <= 1e-13 * mass and abs(res[0][0]["ekin"] - energy) <= 1e-13 * energy


def test_status_after_another_call_is_of_that_call():
    """After a cut batch a status re-adds the job's sums only until another call
    reduces or rebuilds: then it is what that call left, as before."""
    eng = HipEngine(precision=0, brick=(8, 6, 8))
    job = JobSpec(0, 0.0, 34, 1, (1.0, 1e-3, 400.0, 16.0, 0.0), 3)
    h = eng.open(job)
    try:
        eng.step([h], 3)
        mesh = eng._mesh_for(34)[0]
        call("rh_ctx_select", h)
        out = [ctypes.c_double() for _ in range(5)]
        g = np.zeros(3)
        half = mesh.noct // 2
        call("rh_cmpdt", 1, half, mesh.dx, 1.4, 1e-10, 1e-20, 0.5, ptr(g), *[ctypes.byref(x) for x in out])
        call("rh_ctx_select", 0)
        st = eng.status(h)
    finally:
        call("rh_ctx_select", 0)
        eng.close(h)
        eng.close_all()
    assert [st[k] for k in ("mass", "ekin", "eint")] == [x.value for x in out[:3]]
