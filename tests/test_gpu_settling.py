"""settling_velocity over its range: a grain of zero or vanishing size, the
Stokes range, the turbulent range above Re = 1000 (no iteration), the whole
twenty rounds, and a grain lighter than the gas; the deposit of a wet layer
against the oracle, which evaluates the plain operations."""
import numpy as np
import pytest

from imex_sflow2d_v2_amd import decks
from imex_sflow2d_v2_amd.solver import Solver
from oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("diam,rho", [(0.0, 2500.0), (1e-150, 2500.0), (1e-12, 2500.0), (1e-7, 2500.0),
                                      (3e-5, 2500.0), (1.1e-3, 2500.0), (0.05, 2700.0), (1e-3, 0.3)])
def test_settling_range(diam, rho, sparse):
    d = decks.small_2d(n=35, ny=18, seed=8, wet_floor=0.3, n_solid=2)
    d.params.diam_s[1] = diam
    d.params.rho_s[1] = rho
    orc = Oracle(d.params, fresh=True).load_deck(d)
    dev = Solver(d.params).load_deck(d)
    dev.set_tuning(target_strips=1 << 20 if sparse else 1)
    assert dev.advance(6, dt0=1e-3) == orc.run(6, dt0=1e-3)
    for a, b in ((dev.q(), orc.q()), (dev.erosion_state()[1], orc.erosion_state()[1])):
        assert np.array_equal(np.isnan(a), np.isnan(b))
        assert np.nanmax(np.abs(a - b)) <= 1e-13 * np.nanmax(np.abs(b))
