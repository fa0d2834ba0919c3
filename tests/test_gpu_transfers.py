"""Uploads and downloads: states whose size lies around the pinned chunks'
(direct copy, part of a chunk, a whole number of chunks, an odd rest, several
threads), planes of odd widths, and contexts downloading from several threads
at once.  What was uploaded comes back bit for bit."""
import threading

import numpy as np
import pytest

from imex_sflow2d_v2_amd.params import make_params
from imex_sflow2d_v2_amd.solver import Solver

pytestmark = pytest.mark.gpu


def make(nx, ny, ns=2):
    return Solver(make_params(nx, ny, 1.0, ns, rho_s=(2500.0,) * ns, diam_s=(1e-3,) * ns,
                              sp_heat_s=(1617.0,) * ns))


def field(shape, seed):
    return np.asfortranarray(np.random.default_rng(seed).random(shape).transpose())


@pytest.mark.parametrize("nx,ny,ns", [
    (3, 2, 0), (73, 75, 2), (74, 74, 2),              # 262 144 bytes, the least through the chunks
    (256, 512, 0), (257, 512, 0), (127, 1032, 0),     # 4 MiB, a row more, a value less
    (512, 512, 0), (1000, 701, 2), (1500, 901, 3)])
def test_state_round_trip(nx, ny, ns):
    s = make(nx, ny, ns)
    for seed in (1, 2):
        q = field((ny, nx, 4 + ns), seed)
        s.upload_q(q)
        assert np.array_equal(s.q(), q)
    B = field((ny, nx), 3)
    s.set_topography(B)
    if ns:
        er = field((ny, nx, ns), 4)
        dep, ers = (np.asfortranarray(field((ny, nx), 5 + i)[:, :, None].repeat(ns, 2)) for i in (0, 1))
        s.upload_erosion(er, dep, ers)
        got = s.erosion_state()
        for a, b in zip(got, (er, dep, ers, B)):
            assert np.array_equal(a, b)


def test_downloads_from_several_threads():
    runs = []
    for i in range(4):
        s = make(500 + 37 * i, 600, 2)
        q = field((600, 500 + 37 * i, 6), 10 + i)
        s.upload_q(q)
        runs.append((s, q))
    bad = []

    def work(s, q):
        for _ in range(5):
            if not np.array_equal(s.q(), q):
                bad.append(s.nx)

    ts = [threading.Thread(target=work, args=r) for r in runs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
