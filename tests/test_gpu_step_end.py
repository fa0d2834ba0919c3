"""The end of a step inside its last pass over the cells: launches of one
workgroup, fewer, as many and more than the sixteen arrival counters, dense and
sparse steps, with and without a topography pass behind, in captured sequences,
the remainder and runs that stop at an output time.  Against the oracle: equal
steps and times and, from the state a run leaves, an equal next time step and
count of active cells."""
import numpy as np
import pytest

from imex_sflow2d_v2_amd import decks
from imex_sflow2d_v2_amd.solver import Solver
from oracle import Oracle

pytestmark = pytest.mark.gpu

# With N_RK = 3 and two or three classes a run may reach the NaN trap
# (src/solver_2d.f90:1379-1394), where the reference stops: at an x face whose mass
# flux cancels to exactly zero and one of whose classes has no flux, the cap on the
# solid fluxes (:2832-3047) is 0 / 0.  Whether it does hangs on the last bit of the
# initial state.  Both sides reach it then, and nothing after it is compared
# (beside a NaN the device's limited slope is zero, the oracle's is NaN).  One class
# has no such face.


@pytest.mark.parametrize("kw", [{}, dict(erosion=True, topo_change=True),
                                dict(rheology_model=6, friction_factor=2e-3),
                                dict(n_rk=3), dict(n_rk=3, n_solid=1),
                                dict(n_rk=3, n_solid=3)])
@pytest.mark.parametrize("n,ny", [(8, 8), (31, 31), (33, 31), (130, 33)])
@pytest.mark.parametrize("sparse", [False, True])
def test_step_end(n, ny, kw, sparse):
    print("step end", n, ny, kw, sparse, flush=True)
    d = decks.small_2d(n=n, ny=ny, seed=3, **kw)
    orc = Oracle(d.params, fresh=True).load_deck(d)
    dev = Solver(d.params).load_deck(d)
    dev.set_tuning(target_strips=1 << 20 if sparse else 1)
    trap = kw.get("n_rk") == 3 and kw.get("n_solid") != 1
    for steps, t_out in ((1, 1e30), (61, 1e30), (1 << 20, None), (1 << 20, None), (27, 1e30)):
        t_out = orc.t + 0.21 if t_out is None else t_out
        a = orc.run(steps, dt0=d.dt0, t_end=1e30, t_output=t_out)
        b = dev.advance(steps, dt0=d.dt0, t_end=1e30, t_output=t_out)
        if trap and orc.counters()["nan"]:
            assert dev.stats()["nan_events"] > 0
            return
        assert b == a
        assert dev.t == orc.t and dev.get_dt() == orc.dt_last[0]
        q, ref = dev.q(), orc.q()
        for v in range(ref.shape[0]):
            assert np.abs(q[v] - ref[v]).max() <= 1e-13 * max(np.abs(ref[v]).max(), 1e-300), v
    assert dev.timestep() == orc.timestep()
    assert dev.check_solve(False, t=orc.t) == orc.check_solve(False)
