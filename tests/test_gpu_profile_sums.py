"""The profile sums and the pass over face sides where they can go wrong: more
quadrature points than the mean speed's iteration keeps (20), slow flow whose
solid exponents leave the exponential's ordinary range in some lanes and not in
others, and layers that cover some of the 60 x 16 tiles only, so that sides are
formed for cells of tiles without a computed cell.  Same operations in the same
order as the oracle: conversions to the bit, runs within 1e-13 of each
variable's largest value."""
import numpy as np
import pytest

from imex_sflow2d_v2_amd import decks
from imex_sflow2d_v2_amd.solver import Solver
from oracle import Oracle

pytestmark = pytest.mark.gpu


def convert(p, qp):
    return Oracle(p).qp_to_qc(qp)


@pytest.mark.parametrize("ns,n_quad,slope", [(1, 7, True), (2, 21, True), (2, 33, False),
                                             (3, 20, True)])
def test_conversions(ns, n_quad, slope):
    p = decks.profile_channel(nx=8, ny=8, n_solid=ns, n_quad=n_quad, slope_correction=slope,
                              convert=convert).params
    print("conversions", ns, n_quad, slope, flush=True)
    rng = np.random.default_rng(ns + n_quad)
    n, nv = 300, p.n_vars
    qp = np.zeros((nv + 2, n))
    qp[0] = 10 ** rng.uniform(-2.0, 2.0, n)
    u = 10 ** rng.uniform(-5.0, 1.3, n)
    a = rng.uniform(0, 2 * np.pi, n)
    qp[nv], qp[nv + 1] = u * np.cos(a), u * np.sin(a)
    qp[1], qp[2] = qp[0] * qp[nv], qp[0] * qp[nv + 1]
    qp[3] = rng.uniform(300, 700, n)
    for i in range(ns):
        qp[4 + i] = rng.uniform(0.001, 0.04, n) * qp[0]
    bx, by = rng.uniform(-0.3, 0.3, (2, n))
    dev, orc = Solver(p), Oracle(p)
    qc = orc.qp_to_qc(qp)
    assert np.array_equal(dev.qp_to_qc(qp), qc, equal_nan=True)
    assert np.array_equal(dev.qc_to_qp(qc), orc.qc_to_qp(qc), equal_nan=True)
    assert np.array_equal(dev.flux_coeffs(qp, bx, by), orc.flux_coeffs(qp, bx, by),
                          equal_nan=True)


@pytest.mark.parametrize("nx,ny,x0,x1,y0,y1", [(130, 40, 0, 59, 0, 40), (130, 40, 61, 70, 17, 30),
                                               (121, 33, 30, 60, 0, 16)])
def test_partly_covered(nx, ny, x0, x1, y0, y1):
    print("partly covered", nx, ny, x0, x1, y0, y1, flush=True)
    d = decks.profile_channel(nx=nx, ny=ny, convert=convert)
    keep = np.zeros((nx, ny), bool)
    keep[x0:x1, y0:y1] = True
    d.q[:, ~keep] = 0.0
    orc, dev = Oracle(d.params, fresh=True).load_deck(d), Solver(d.params).load_deck(d)
    assert dev.advance(27, dt0=d.dt0) == orc.run(27, dt0=d.dt0)
    q, ref = dev.q(), orc.q()
    assert np.array_equal(np.isnan(q), np.isnan(ref))
    for v in range(ref.shape[0]):
        big = np.nanmax(np.abs(ref[v]))
        assert np.nanmax(np.abs(q[v] - ref[v])) <= 1e-13 * max(big, 1e-300), v
