"""Transfers of a context's calls through its pinned memory (two halves of 1 MiB):
orbitals that just fill it, results of just under, of and over a half."""
import numpy as np
import pytest

import oracle
from pgxc import XCBuilder, basis
from pgxc.xc import FP64, LDA

pytestmark = pytest.mark.gpu


def s_functions(n, seed):
    """n functions, ten s functions an atom on a cubic lattice, and 500 points."""
    rng = np.random.default_rng(seed)
    na = (n + 9) // 10
    side = int(np.ceil(na ** (1 / 3)))
    xyz = np.stack(np.unravel_index(np.arange(na), (side,) * 3), axis=1) * 2.5
    b = basis.Basis(xyz)
    for f in range(n):
        b.shells.append(basis.Shell(f // 10, 0, rng.uniform(0.2, 2.0, 1), 1, np.zeros((1, 0))))
    g = np.concatenate([rng.uniform(-1.0, 2.5 * side, (500, 3)), rng.uniform(0.1, 1.0, (500, 1))], axis=1)
    return b, g


# 511 functions: a packed V of 130 816 doubles, half a pair holds 131 072; 512: 131 328.
# 511 x 512 orbitals with their occupations: 262 144 doubles, the whole pair; 512 x 512 do not fit.
@pytest.mark.parametrize("n,nocc", [(1, 1), (33, 7), (511, 512), (512, 512), (740, 3)])
@pytest.mark.parametrize("ispin", [1, 2])
def test_orbitals_and_results_of_every_size(n, nocc, ispin):
    b, g = s_functions(n, seed=n)
    if ispin == 2:
        nocc = max(1, nocc // 2)
    rng = np.random.default_rng(n + ispin)
    C, occ = rng.normal(size=(n, nocc, 2)) / np.sqrt(n), rng.uniform(0.5, 2.0, (nocc, 2))
    C, occ = (C, occ) if ispin == 2 else (C[..., 0], occ[..., 0])
    hr, er, qr = oracle.xc_build(b, g, oracle.MASK_LDA, C=C, occ=occ, nthreads=4, ispin=ispin)
    with XCBuilder(b, g) as xc:
        for _ in range(2):
            xc.set_orbitals(C, occ)
            ham, e, q = xc.build(LDA, FP64)
            again = xc.result()
            # sums of up to 740^2 terms a point, of one sign but for the cross terms of P: 1e-12 of
            # the density, and less of its cube root; anything misplaced is of the order of V itself
            assert np.max(np.abs(ham - hr)) <= 1e-10 * np.max(np.abs(hr))
            assert abs(e - er) <= 1e-10 * abs(er) and abs(q - qr) <= 1e-10 * abs(qr)
            assert np.array_equal(again[0], ham) and again[1:] == (e, q)
