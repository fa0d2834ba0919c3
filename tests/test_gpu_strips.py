"""The strips of the dense stencil pass against the oracle: the fixed heights of
imexsw_set_tuning at the edges of tiles, and the default's, whole-column strips
(every tile listed) and tile strips of the fitted height (a dry corner); and an
ensemble with the fitted height against the fixed ones.  The faces are the same
operations in every cut, so the bar is 1e-13 of each variable's largest value
against the oracle and equality between cuts."""
import numpy as np
import pytest

from imex_sflow2d_v2_amd import decks
from imex_sflow2d_v2_amd.solver import Ensemble, Solver
from oracle import Oracle

pytestmark = pytest.mark.gpu


def state(d, tuning, steps):
    s = Solver(d.params).load_deck(d)
    if tuning:
        s.set_tuning(*tuning)
    s.advance(steps, dt0=d.dt0)
    return s.q()


@pytest.mark.parametrize("wet", [0.5, 0.0])
@pytest.mark.parametrize("nx,ny,kw", [
    (2, 3, {}), (59, 16, {}), (60, 17, dict(limiter=3)), (61, 33, dict(limiter=[1, 2, 1, 3, 5, 1])),
    (122, 31, dict(source=True)), (63, 47, dict(slope_correction=True, curvature=True)),
    (181, 5, dict(n_solid=1, alpha=True))])
def test_strip_cuts(nx, ny, kw, wet):
    d = decks.small_2d(n=nx, ny=ny, seed=3, wet_floor=wet, **kw)
    # the smallest target leaves the dense form, in tile strips of at most 16, 1
    # and 4 rows (the default's strips: test_default_strips, test_default_strips_rich)
    cuts = [state(d, t, 21) for t in ((16, 1), (1, 1), (4, 1))]
    orc = Oracle(d.params, fresh=True).load_deck(d)
    orc.run(21, dt0=d.dt0)
    ref = orc.q()
    for q in cuts:
        assert np.array_equal(q, cuts[0])
        for v in range(ref.shape[0]):
            assert np.abs(q[v] - ref[v]).max() <= 1e-13 * max(np.abs(ref[v]).max(), 1e-300)


@pytest.mark.parametrize("nx,ny,dry", [(601, 420, False), (540, 513, False), (600, 470, True)])
def test_default_strips(nx, ny, dry):
    """Above 53 248 computed cells (one class) the default takes the dense form,
    with column strips (all tiles wet) or fitted tile strips (a dry corner)."""
    d = decks.small_2d(n=nx, ny=ny, seed=4, wet_floor=0.5, n_solid=1)
    if dry:
        d.q[:, -70:, -20:] = 0.0
    a = state(d, None, 5)
    assert np.array_equal(a, state(d, (8, 1), 5))
    orc = Oracle(d.params, fresh=True).load_deck(d)
    orc.run(5, dt0=d.dt0)
    ref = orc.q()
    for v in range(ref.shape[0]):
        assert np.abs(a[v] - ref[v]).max() <= 1e-13 * max(np.abs(ref[v]).max(), 1e-300)


# Grids of 47 000 to 50 000 cells, above the line of two and three classes, with a
# last tile of one column (241) or one row (193 = 12 * 16 + 1) and strips that do
# not divide the rows
@pytest.mark.parametrize("dry", [False, True])
@pytest.mark.parametrize("nx,ny,kw", [
    (241, 207, dict(source=True)), (260, 193, dict(slope_correction=True, curvature=True)),
    (241, 193, dict(limiter=[1, 2, 1, 3, 5, 1])), (259, 191, dict(limiter=4, n_solid=3)),
    (300, 161, dict(n_solid=3, alpha=True, erosion=True, topo_change=True))])
def test_default_strips_rich(nx, ny, kw, dry):
    print("default strips", nx, ny, kw, dry, flush=True)
    d = decks.small_2d(n=nx, ny=ny, seed=6, wet_floor=0.5, **kw)
    if dry:
        d.q[:, -70:, -25:] = 0.0
    s = Solver(d.params).load_deck(d)
    s.advance(6, dt0=d.dt0)
    assert s.stats()["sparse_steps"] == 0
    a = s.q()
    assert np.array_equal(a, state(d, (4, 1), 6))
    orc = Oracle(d.params, fresh=True).load_deck(d)
    orc.run(6, dt0=d.dt0)
    ref = orc.q()
    for v in range(ref.shape[0]):
        assert np.abs(a[v] - ref[v]).max() <= 1e-13 * max(np.abs(ref[v]).max(), 1e-300)


def test_ensemble_fitted_strips():
    ds = decks.ensemble_members(count=5, seed=6, sizes=[61, 33, 180, 97, 250])
    out = []
    for h in (None, 4, 16):
        e = Ensemble([d.params for d in ds]).load(ds)
        if h:
            e.set_tuning(strip_rows=h)
        e.advance(30, dt0=1e-3)
        out.append([m.q() for m in e.members])
        e.close()
    for o in out[1:]:
        assert all(np.array_equal(x, y) for x, y in zip(o, out[0]))
