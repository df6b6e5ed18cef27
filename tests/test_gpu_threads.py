"""Calls on one context from several threads: reading a build's results is safe
while others read them, and while the next orbitals are uploaded; different
contexts are independent."""
import threading

import numpy as np
import pytest

from pgxc import XCBuilder, basis, grid, systems
from pgxc.xc import BF16X3, FP32, FP64, PBE

pytestmark = pytest.mark.gpu


def run(*loops):
    """The loops at once, each in a thread; the first exception is raised."""
    errors = []

    def guard(f):
        try:
            f()
        except BaseException as e:  # noqa: BLE001
            errors.append(e)
    ts = [threading.Thread(target=guard, args=(f,)) for f in loops]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    if errors:
        raise errors[0]


@pytest.fixture(scope="module", params=[1, 2])
def built(request):
    els, xyz = systems.water_cluster(16, seed=3)
    b = basis.seeded_basis(els, xyz, seed=4, shell_set="medium")
    g = grid.molecular_grid(els, xyz, nrad=6, nang=194)
    C = systems.random_orbitals(b.nbas, 40, seed=5)[0]
    occ = np.ones(40)
    if request.param == 2:
        C, occ = np.asfortranarray(np.stack([C, C[:, ::-1]], axis=2)), np.ones((40, 2))
    with XCBuilder(b, g) as xc:
        xc.set_orbitals(C, occ)
        yield xc, C, occ, xc.build(PBE, FP64)


def same(r, ref):
    assert np.array_equal(r[0], ref[0]) and r[1:] == ref[1:]


def test_results_read_by_several_threads(built):
    xc, _, _, ref = built

    def read():
        for _ in range(60):
            same(xc.result(), ref)
    run(read, read, read)


def test_results_read_while_orbitals_are_set(built):
    xc, C, occ, ref = built
    half = C * 0.5

    def read():
        for _ in range(60):
            same(xc.result(), ref)

    def upload():
        for _ in range(30):
            xc.set_orbitals(half, occ)
            xc.set_orbitals(C, occ)
    run(read, upload, read)
    xc.set_orbitals(C, occ)
    same(xc.build(PBE, FP64), ref)


def test_contexts_in_threads_of_their_own():
    def work(i, out):
        els, xyz = systems.random_molecule(4 + i, seed=i)
        b = basis.seeded_basis(els, xyz, seed=6, shell_set="small")
        g = grid.molecular_grid(els, xyz, nrad=12, nang=194, partition="gpu")
        C, occ = systems.random_orbitals(b.nbas, 4, seed=1)
        with XCBuilder(b, g, chunk_points=2048) as xc:
            for prec in (FP64, FP32, BF16X3):
                xc.set_orbitals(C, occ)
                out[i, prec] = xc.build(PBE, prec)
    alone, together = {}, {}
    for i in range(4):
        work(i, alone)
    run(*[lambda i=i: work(i, together) for i in range(4)])
    for k, v in alone.items():
        same(together[k], v)
