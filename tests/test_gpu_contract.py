"""The contractions at the edges of their shares, blocks and lists: function
counts around 16, 64, 96, 128 and 256 columns, point counts that leave part of a
tile, chunk and split, tiles of many functions (wide split-BF16 items), and
partials that do not all fit (summed while the build runs)."""
import numpy as np
import pytest

import oracle
from pgxc import XCBuilder, basis, grid, systems
from pgxc.basis import Basis, Shell

pytestmark = pytest.mark.gpu


def _basis(n, rng):
    """n functions on a line of atoms: s shells of up to 12 functions and, from
    the second atom on, a p shell where it fits."""
    shells, xyz, left = [], [], n
    while left > 0:
        a = len(xyz)
        xyz.append((1.9 * a, 0.3 * (a % 3), 0.2 * (a % 2)))
        k = min(left, 12)
        shells.append(Shell(a, 0, np.sort(np.exp(rng.uniform(np.log(0.2), np.log(30.0), k))), k, np.zeros((k, 0))))
        left -= k
        if a and left >= 3:
            shells.append(Shell(a, 1, np.array([rng.uniform(0.2, 2.0)]), 1, np.zeros((1, 0))))
            left -= 3
    b = Basis(np.array(xyz))
    b.shells = shells
    assert b.nbas == n
    return b


def _grid(b, npts, rng):
    own = rng.integers(0, b.n_atoms, npts)
    d = rng.normal(size=(npts, 3))
    r = rng.uniform(0.1, 3.0, npts)
    pts = b.atom_xyz[own] + r[:, None] * d / np.linalg.norm(d, axis=1)[:, None]
    return np.asfortranarray(np.column_stack([pts, rng.uniform(0.01, 0.1, npts)]))


def _check(got, ref, rel):
    v = np.max(np.abs(ref[0]))
    # FP64: sums of some hundred points and functions; the mixed contractions of
    # a full density carry their operands' rounding (2^-24, 2^-17) into V
    assert abs(got[1] - ref[1]) <= 1e-9 + rel * abs(ref[1])
    assert np.max(np.abs(got[0] - ref[0])) <= 1e-10 + 10 * rel * v
    assert abs(got[2] - ref[2]) <= 1e-9 + rel * abs(ref[2])


@pytest.mark.parametrize("n,npts", [(1, 129), (15, 31), (16, 300), (17, 1000), (64, 700), (65, 700),
                                    (95, 257), (97, 511), (127, 300), (128, 300), (129, 640),
                                    (193, 300), (257, 385), (420, 300)])
@pytest.mark.parametrize("spins", [1, 2])
def test_function_counts(n, npts, spins):
    rng = np.random.default_rng(1000 * n + spins)
    b = _basis(n, rng)
    g = _grid(b, npts, rng)
    m = max(1, n // 6)
    C = [np.linalg.qr(rng.normal(size=(n, m)))[0] for _ in range(spins)]
    P = C[0] @ C[0].T if spins == 1 else np.stack([c @ c.T for c in C], axis=2)
    ref = {f: oracle.xc_build(b, g, mask, P=P, nthreads=4, ispin=spins)
           for f, mask in (("PBE", oracle.MASK_PBE), ("LDA", oracle.MASK_LDA))}
    for screen in (True, False):
        with XCBuilder(b, g, screen=screen) as xc:
            xc.set_density(P)
            for f in ("PBE", "LDA"):
                for prec, rel in (("fp64", 0.0), ("fp32", 2e-6), ("bf16x3", 5e-5)):
                    _check(xc.build(f, prec), ref[f], rel)


@pytest.mark.parametrize("tile", [64, 96, 128])
@pytest.mark.parametrize("variant", [0, 1, 2])
def test_tiles_and_variants(tile, variant):
    rng = np.random.default_rng(10 * tile + variant)
    b = _basis(150, rng)
    g = _grid(b, 5000, rng)
    C = np.linalg.qr(rng.normal(size=(150, 20)))[0]
    ref = oracle.xc_build(b, g, oracle.MASK_PBE, C=C, occ=np.ones(20), nthreads=4)
    with XCBuilder(b, g, tile=tile, variants=(variant, variant), chunk_points=2048) as xc:
        xc.set_orbitals(C, np.ones(20))
        for prec, rel in (("fp64", 0.0), ("fp32", 2e-6), ("bf16x3", 5e-5)):
            _check(xc.build("PBE", prec), ref, rel)


@pytest.mark.parametrize("lanes", [1, 2])
def test_partials_summed_during_the_build(lanes):
    """Without screening every split holds every function and the partials of
    all chunks pass 4 GiB, so they are summed as they fill their slots; with
    screening they fit.  Both are the same sums."""
    els, xyz = systems.water_cluster(45, seed=3, jitter_a=0.2)
    b = basis.seeded_basis(els, xyz, seed=12, shell_set="medium")
    g = grid.molecular_grid(els, xyz, nrad=16, nang=302, partition="gpu")
    C, occ = systems.random_orbitals(b.nbas, 40, seed=5)
    out = []
    for screen in (True, False):
        with XCBuilder(b, g, screen=screen, chunk_points=4096, basis_cache=False) as xc:
            xc.set_lanes(lanes)
            lay = xc.layout()
            if not screen:
                assert 8.0 * b.nbas ** 2 * lay["npad"] / 2048 > 4 * 2 ** 30
            xc.set_orbitals(C, occ)
            out.append(xc.build("PBE", "fp64"))
    (h0, e0, q0), (h1, e1, q1) = out
    assert np.max(np.abs(h0 - h1)) <= 1e-10 and abs(e0 - e1) <= 1e-9 and abs(q0 - q1) <= 1e-9


@pytest.mark.parametrize("n,nocc", [(1, 1), (3, 0), (17, 5), (63, 15), (64, 16), (65, 17), (130, 33), (200, 1)])
@pytest.mark.parametrize("spins", [1, 2])
def test_density_from_orbitals(n, nocc, spins):
    """P formed on the device from orbitals and occupations (tiles of 64, 16
    orbitals a step, caller order) gives the builds of the same P as a matrix."""
    rng = np.random.default_rng(n + 7 * nocc)
    b = _basis(n, rng)
    g = _grid(b, 200, rng)
    shape = (n, nocc) if spins == 1 else (n, nocc, 2)
    C, occ = rng.normal(size=shape) / np.sqrt(n), rng.uniform(0.1, 2.0, shape[1:])
    if spins == 1:
        P = (C * occ) @ C.T
    else:
        P = np.stack([(C[:, :, s] * occ[:, s]) @ C[:, :, s].T for s in range(2)], axis=2)
    with XCBuilder(b, g) as xc:
        xc.set_density(P)
        h0, e0, q0 = xc.build("PBE", "fp64")
        xc.set_orbitals(C, occ)
        h1, e1, q1 = xc.build("PBE", "fp64")
    # sums of at most 33 products of order 1 in both: P to some 1e-15
    assert np.max(np.abs(h0 - h1)) <= 1e-12 * max(1.0, np.max(np.abs(h0)))
    assert abs(e0 - e1) <= 1e-12 * max(1.0, abs(e0)) and abs(q0 - q1) <= 1e-12 * max(1.0, abs(q0))


def _shell_basis(lmax, rng):
    """Three atoms; the first with the most shells an atom may have: 1 to 9
    primitives (blocks of 4 and their remainders), 0 to 8 contractions."""
    shells = []
    for a, count in ((0, 16), (1, 3), (2, 1)):
        for s in range(count):
            ne, nc = 1 + (5 * s + a) % 9, (3 * s + 2 * a) % 9
            nu = 1 if nc == 0 else s % 2
            l = s % (lmax + 1)
            ex = np.sort(np.exp(rng.uniform(np.log(0.3), np.log(20.0), ne)))[::-1].copy()
            shells.append(Shell(a, l, ex, min(nu, ne), rng.uniform(-0.6, 0.6, (ne, nc))))
    b = Basis(np.array([(0.0, 0.0, 0.0), (1.1, 0.2, -0.3), (-0.4, 1.3, 0.9)]))
    b.shells = shells
    return b


@pytest.mark.parametrize("lmax", [0, 2, 3, 4])
@pytest.mark.parametrize("spins", [1, 2])
def test_shell_tables(lmax, spins):
    """Every count of primitives and contractions a block of a shell's table can
    end with, on both tiles of a block, in the basis, W and gradient stages."""
    from test_gpu_gradient import check, fd_gradient
    rng = np.random.default_rng(31 * lmax + spins)
    b = _shell_basis(lmax, rng)
    g = _grid(b, 300, rng)
    n, m = b.nbas, 3
    C = [np.linalg.qr(rng.normal(size=(n, m)))[0] for _ in range(spins)]
    P = C[0] @ C[0].T if spins == 1 else np.stack([c @ c.T for c in C], axis=2)
    with XCBuilder(b, g) as xc:
        xc.set_density(P)
        for f, mask in (("LDA", oracle.MASK_LDA), ("PBE", oracle.MASK_PBE)):
            ref = oracle.xc_build(b, g, mask, P=P, nthreads=4, ispin=spins)
            for prec, rel in (("fp32", 2e-6), ("bf16x3", 5e-5), ("fp64", 0.0)):
                _check(xc.build(f, prec), ref, rel)
            if spins == 1 and lmax in (2, 4):
                check(xc.gradient(), fd_gradient(b, g, mask, P=P))


def test_partials_of_uneven_chunks(monkeypatch, capfd):
    """Chunks of different sizes laid one behind the other in a lane's share of
    the partials: one lane and two, which sum them after different chunks, agree
    with the sums over every function (all chunks the same size)."""
    monkeypatch.setenv("PGXC_DEBUG", "1")
    els, xyz = systems.water_cluster(64, seed=4, jitter_a=0.2)
    b = basis.seeded_basis(els, xyz, seed=13, shell_set="medium")
    g = grid.molecular_grid(els, xyz, nrad=40, nang=302, partition="gpu")
    C, occ = systems.random_orbitals(b.nbas, 40, seed=6)
    out = []
    for screen, lanes in ((True, 1), (True, 2), (False, 2)):
        with XCBuilder(b, g, screen=screen, chunk_points=16384, basis_cache=False) as xc:
            if screen:
                said = [l for l in capfd.readouterr().err.splitlines() if "sums" in l][-1].split()
                one, two = int(said[said.index("sums") + 1]), int(said[-3])
                assert one > 1 and two > 2, said
            xc.set_lanes(lanes)
            xc.set_orbitals(C, occ)
            out.append(xc.build("PBE", "fp64"))
    for h, e, q in out[1:]:
        assert np.max(np.abs(h - out[0][0])) <= 1e-10
        assert abs(e - out[0][1]) <= 1e-9 and abs(q - out[0][2]) <= 1e-9
