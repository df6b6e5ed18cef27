"""Becke weights on the GPU at the sizes where their kernel takes another way:
fewer centres than it keeps as nearest ones, as many, a few more, and enough
that most are left out of the sum; against the numpy partition in FP64."""
import numpy as np
import pytest

from pgxc import becke_weights, grid, systems

pytestmark = pytest.mark.gpu


def _points(rng, xyz, npts):
    """Points at and near centres, between them and far outside."""
    own = rng.integers(0, len(xyz), npts).astype(np.int32)
    r = 10.0 ** rng.uniform(-6, 2, npts)
    d = rng.normal(size=(npts, 3))
    pts = xyz[own] + r[:, None] * d / np.linalg.norm(d, axis=1)[:, None]
    pts[:len(xyz)] = xyz[own[:len(xyz)]]                      # at a nucleus
    pts[len(xyz)] = 0.5 * (xyz[0] + xyz[-1])                  # halfway
    return pts, own


@pytest.mark.parametrize("na,npts", [(1, 70), (2, 63), (3, 257), (7, 300), (8, 300), (9, 1025),
                                     (13, 511), (60, 700)])
def test_weights_match_numpy(na, npts):
    if na <= 8:
        xyz = systems.random_molecule(9, seed=5)[1][:na]
    else:
        xyz = systems.random_molecule(na, seed=na)[1]
    rng = np.random.default_rng(na)
    pts, own = _points(rng, xyz, npts)
    wat = rng.uniform(0.1, 2.0, npts)
    ref = wat if na == 1 else grid.becke_numpy(xyz, pts, own, wat)
    got = becke_weights(xyz, pts, own, wat)
    # each weight is w times a quotient of products of na factors in [0, 1]
    # that both sides form in FP64 from distances of up to 100 bohr over
    # separations of about 2: 1e-13 per factor's mu, steps of slope up to 27/16
    assert np.max(np.abs(got - ref) / wat) < 1e-13 * 27 / 16 * na
    assert np.all(got[:na] >= 0)


def test_equidistant_centres():
    """Eight centres on a cube and its middle: no centre is negligible."""
    xyz = np.array([[i, j, k] for i in (-2.0, 2.0) for j in (-2.0, 2.0) for k in (-2.0, 2.0)])
    own = np.arange(8, dtype=np.int32)
    w = becke_weights(xyz, np.zeros((8, 3)), own, np.full(8, 3.0))
    assert np.max(np.abs(w - 3.0 / 8)) < 1e-15


@pytest.mark.parametrize("na", [1, 2, 9, 40])
@pytest.mark.parametrize("spins", [1, 2])
def test_moving_grid_gradient_against_fixed_grid_sums(na, spins):
    """The moving-grid gradient where the Becke derivatives keep every centre,
    a few and a small part of them: it is invariant under translation of the
    molecule with its grid, exactly, and one centre alone has none at all."""
    from pgxc import XCBuilder, basis
    els, xyz = systems.random_molecule(na, seed=21) if na > 1 else (["O"], np.zeros((1, 3)))
    b = basis.seeded_basis(els, xyz, seed=22, shell_set="small")
    g = grid.molecular_grid(els, xyz, nrad=8, nang=194)
    own = grid.owners(els, 8, 194)
    rng = np.random.default_rng(na)
    n = max(2, b.nbas // 5)
    C = [np.linalg.qr(rng.normal(size=(b.nbas, n)))[0] for _ in range(spins)]
    with XCBuilder(b, g, chunk_points=4096) as xc:
        if spins == 1:
            xc.set_orbitals(C[0], np.ones(n))
        else:
            xc.set_orbitals(np.stack(C, axis=2), np.ones((n, 2)))
        xc.build("PBE", "fp64", fetch=False)
        f, again = xc.gradient_grid(own), xc.gradient_grid(own)
    assert np.array_equal(f, again)
    # the sum over atoms cancels terms of the size of the per-point sums (about
    # npts of order 1 to 10 each) to FP64 rounding
    assert np.max(np.abs(f.sum(axis=0))) < 1e-16 * 10 * len(own)


def test_lone_centre_takes_the_whole_weight():
    """One centre: its weights are the one-centre weights at every point, also
    where the distance overflows or is no number."""
    pts = np.zeros((70, 3))
    pts[1:6] = [[1e200, 0, 0], [0, -1e160, 2], [np.inf, 1, 1], [0, 0, np.nan], [1e-300, 0, 0]]
    wat = np.linspace(0.1, 2.0, 70)
    w = becke_weights(np.zeros((1, 3)), pts, np.zeros(70, dtype=np.int32), wat)
    assert np.array_equal(w, wat)


@pytest.mark.parametrize("na", [11, 12, 13, 14])
@pytest.mark.parametrize("npts", [1, 63, 257, 4097])
def test_weights_where_the_kernel_changes(na, npts):
    """Up to 12 centres every pair is formed, above that the near ones first."""
    xyz = systems.random_molecule(14, seed=3)[1][:na]
    rng = np.random.default_rng(100 * na + npts)
    pts, own = _points(rng, xyz, max(npts, na + 1))
    pts, own = pts[:npts], own[:npts]
    wat = rng.uniform(0.1, 2.0, npts)
    got = becke_weights(xyz, pts, own, wat)
    ref = grid.becke_numpy(xyz, pts, own, wat)
    assert np.max(np.abs(got - ref) / wat) < 1e-13 * 27 / 16 * na  # as above


@pytest.mark.parametrize("na", [12, 13])
@pytest.mark.parametrize("npts", [0, 1, (1 << 18) - 1, 1 << 18, (1 << 18) + 1, (1 << 19) + 130])
def test_weights_in_one_part_and_in_several(na, npts):
    """Grids above 2^18 points of more than 12 centres go through the device in
    parts: each part's weights are those of a call with its points alone, and
    the output array may be the input's."""
    import ctypes
    from pgxc import _lib
    xyz = np.ascontiguousarray(systems.random_molecule(14, seed=3)[1][:na])
    rng = np.random.default_rng(npts + na)
    n = max(npts, 64)
    own = rng.integers(0, na, n).astype(np.int32)[:npts]
    pts = np.asfortranarray(xyz[own] + rng.normal(size=(npts, 3)))
    wat = rng.uniform(0.1, 2.0, n)[:npts]
    got = becke_weights(xyz, pts, own, wat)
    per = 1 << 18
    for p in range(0, npts, per):
        q = slice(p, min(p + per, npts))
        assert np.array_equal(got[q], becke_weights(xyz, pts[q], own[q], wat[q]))
    io = wat.copy()
    dp, ip = ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_int32)
    P = lambda a: a.ctypes.data_as(dp)
    assert _lib.load().pgxc_becke_weights(na, P(xyz), npts, P(pts), own.ctypes.data_as(ip), P(io),
                                          P(io)) == 0
    assert np.array_equal(io, got)


@pytest.mark.parametrize("na", [1024, 1025, 1500])
def test_weights_of_many_centres(na):
    """Above 1024 centres what is left out of the sum shrinks with their number."""
    xyz = np.array([[i, j, k] for i in range(12) for j in range(12) for k in range(11)])[:na] * 2.5
    xyz = xyz + np.random.default_rng(na).uniform(-0.5, 0.5, xyz.shape)
    rng = np.random.default_rng(1)
    own = rng.integers(0, na, 130).astype(np.int32)
    pts = xyz[own] + rng.normal(size=(130, 3))
    D = np.linalg.norm(xyz[:, None] - xyz[None], axis=2) + np.eye(na)
    ref = np.empty(130)
    for p in range(130):
        r = np.linalg.norm(pts[p] - xyz, axis=1)
        mu = (r[:, None] - r[None]) / D
        for _ in range(3):
            mu = mu * (3.0 - mu * mu) / 2.0
        P = np.prod(np.where(np.eye(na, dtype=bool), 1.0, (1.0 - mu) / 2.0), axis=1)
        ref[p] = P[own[p]] / P.sum()
    got = becke_weights(xyz, pts, own, np.ones(130))
    assert np.max(np.abs(got - ref)) < 1e-13 * 27 / 16 * na  # as above
