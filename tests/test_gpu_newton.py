"""The Newton solve's real chain and column derivatives (implicit_real,
implicit_col) where they can leave the usual form: layers at rest or nearly
so (the perturbed speed's square no longer vanishes and implicit_c takes
over; the residual is then the rounding of a large energy), thin layers below
eps_sing with desingularised velocities, momenta of one direction only, in
the one-lane and the four-lane solver and for both drag laws.  Against the
oracle: the operations are the same, so states within 1e-13 of each variable's
largest value and equal counts of Newton solves and iterations."""
import numpy as np
import pytest

from imex_sflow2d_v2_amd import decks
from imex_sflow2d_v2_amd.solver import Solver
from oracle import Oracle

pytestmark = pytest.mark.gpu


def deck(speed, depth, model, **kw):
    d = decks.small_2d(n=47, ny=33, seed=9, wet_floor=0.05, rheology_model=model,
                       friction_factor=1e-3 if model == 6 else -1.0, **kw)
    d.B_cent[:] = 0.0
    d.q[:] = d.q * depth
    # uniform and at the given fraction of the seeded velocities on one half,
    # along x only on the other
    d.q[:, :20, :] = d.q[:, :1, :1]
    d.q[1] *= speed
    d.q[2] *= speed
    d.q[2, 25:, :] = 0.0
    return d


@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("speed,depth,kw", [
    (0.0, 500.0, {}), (1e-15, 500.0, {}), (1e-9, 500.0, {}), (1e-5, 20.0, {}),
    (1.0, 1.0, {}), (1.0, 1e-10, {}), (1.0, 1e-13, {}),
    (1.0, 1.0, dict(slope_correction=True, curvature=True, energy=False)),
    (1e-8, 300.0, dict(n_solid=0)), (1.0, 1e-4, dict(n_solid=3, alpha=True))])
def test_newton_edges(sparse, speed, depth, kw):
    run(deck(speed, depth, 1, **kw), sparse)


@pytest.mark.parametrize("speed,depth", [(0.0, 500.0), (1e-9, 500.0), (1.0, 1.0), (1.0, 1e-12)])
def test_newton_edges_model6(speed, depth):
    run(deck(speed, depth, 6, slope_correction=True), False)


def run(d, sparse):
    orc = Oracle(d.params, fresh=True).load_deck(d)
    dev = Solver(d.params).load_deck(d)
    # the computed-cell count against the strip target decides the form
    dev.set_tuning(target_strips=1 << 20 if sparse else 1)
    assert dev.advance(24, dt0=1e-3) == orc.run(24, dt0=1e-3)
    q, ref = dev.q(), orc.q()
    for v in range(ref.shape[0]):
        assert np.abs(q[v] - ref[v]).max() <= 1e-13 * max(np.abs(ref[v]).max(), 1e-300)
    st, co = dev.stats(), orc.counters()
    for k in ("newton_cells", "newton_iters"):
        assert st[k] == co[k], k
