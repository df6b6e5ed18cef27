"""The moving-grid gradient (pgxc_gradient_grid) against its formula written out
over every pair of centres in numpy, for molecules large enough that the kernel
leaves most of the Becke cells out: LDA, whose terms need no more than the
oracle's basis values and gradients, closed and open shell."""
import numpy as np
import pytest

import oracle
from pgxc import XCBuilder, basis, grid, systems
from pgxc.xc import FP64, LDA

pytestmark = pytest.mark.gpu


def weight_part(xyz, own, pts, wf, keep=0.0):
    """sum_p wf_p d log w_p / dR: the Becke weights of points that move with their
    owners.  keep: a mistake to plant, cells below that share of the largest are
    left out."""
    na = len(xyz)
    out = np.zeros((na, 3))
    eye = np.eye(na, dtype=bool)
    dR = xyz[:, None] - xyz[None]
    R = np.linalg.norm(dR, axis=2) + eye
    for s0 in range(0, len(pts), 128):
        p, o, k0 = pts[s0:s0 + 128], own[s0:s0 + 128], wf[s0:s0 + 128]
        e = p[:, None] - xyz[None]
        r = np.linalg.norm(e, axis=2)
        e = e / np.where(r > 0, r, 1.0)[..., None]
        mu = (r[:, :, None] - r[:, None, :]) / R
        f1 = mu * (3 - mu * mu) / 2
        f2 = f1 * (3 - f1 * f1) / 2
        g = 1 - mu  # 1 - p(m) = (1 - m)^2 (2 + m) / 2, three times: no cancellation
        for _ in range(3):
            g = g * g * (3 - g) / 2
        sl = -(27.0 / 16.0) * (1 - f2 * f2) * (1 - f1 * f1) * (1 - mu * mu)
        sig = np.where(g > 0, 2 * sl / np.where(g > 0, g, 1.0), 0.0)  # s' / s, s = g / 2
        sig[:, eye] = 0.0
        g[:, eye] = 2.0
        P = np.prod(g / 2, axis=2)
        P = np.where(P >= keep * P.max(axis=1, keepdims=True), P, 0.0)
        k = -P / P.sum(axis=1, keepdims=True)
        k[np.arange(len(o)), o] += 1
        T = (k * k0[:, None])[:, :, None] * sig / R
        M = ((T * mu / R)[..., None] * dR[None])
        TC, TD = T[..., None] * e[:, :, None], T[..., None] * e[:, None]
        out += (TD + M).sum(axis=(0, 1)) - (TC + M).sum(axis=(0, 2))
        np.add.at(out, o, (TC - TD).sum(axis=(1, 2)))
    return out


def reference(b, g, own, P):
    """The gradient and a bound of its rounding: every term is a product of a few
    factors (FP64, 1e-15 of the term together); a pair's share of the weight
    derivatives is at most the step's slope over the centres' distance."""
    phi, gr = oracle.basis_eval(b, g[:, :3])
    w = g[:, 3]
    X = [p @ phi for p in P]
    rho = [np.einsum("ip,ip->p", phi, x) for x in X]
    if len(P) == 1:
        f, fr, _ = oracle.functional(oracle.MASK_LDA, rho[0], 0 * rho[0])
        fr = fr[:, None]
    else:
        z = 0 * rho[0]
        f, fr, _ = oracle.functional_spin(oracle.MASK_LDA, rho[0], rho[1], z, z, z)
    out, size = np.zeros((b.n_atoms, 3)), 0.0
    for s, x in enumerate(X):
        t = 2 * gr * x[:, None] * (w * fr[:, s])
        np.add.at(out, b.function_atoms(), -t.sum(axis=2))
        np.add.at(out, own, t.sum(axis=0).T)
        size += 2 * np.abs(t).sum()
    xyz = b.atom_xyz
    d = np.linalg.norm(xyz[:, None] - xyz[None], axis=2) + 1e9 * np.eye(len(xyz))
    size += np.abs(w * f).sum() * len(xyz) * (27 / 16) / d.min()
    return out, weight_part(xyz, own, g[:, :3], w * f), 1e-15 * size, w * f


def system(kind, n):
    els, xyz = systems.random_molecule(n, seed=9) if kind == "molecule" else systems.water_cluster(n, seed=5)
    b = basis.seeded_basis(els, xyz, seed=6, shell_set="small", exp_range=(0.1, 500.0))
    g = grid.molecular_grid(els, xyz, nrad=5, nang=194, partition="numpy")
    return b, g, grid.owners(els, 5, 194)


@pytest.mark.parametrize("kind,n", [("molecule", 8), ("molecule", 9), ("molecule", 13),
                                    ("molecule", 30), ("water", 7)])
@pytest.mark.parametrize("spins", [1, 2])
def test_gradient_is_the_sum_over_all_pairs(kind, n, spins):
    b, g, own = system(kind, n)
    rng = np.random.default_rng(n)
    m = b.nbas // 4
    C = [np.linalg.qr(rng.normal(size=(b.nbas, m)))[0] for _ in range(spins)]
    fixed, weights, tol, wf = reference(b, g, own, [c @ c.T for c in C])
    # the bound notices cells left out that are 1e-8 of the nearest one's
    assert np.max(np.abs(weight_part(b.atom_xyz, own, g[:, :3], wf, keep=1e-8) - weights)) > 10 * tol
    with XCBuilder(b, g, chunk_points=4096) as xc:
        if spins == 1:
            xc.set_orbitals(np.asfortranarray(C[0]), np.ones(m))
        else:
            xc.set_orbitals(np.asfortranarray(np.stack(C, axis=2)), np.ones((m, 2)))
        xc.build(LDA, FP64, fetch=False)
        got = xc.gradient_grid(own)
    err = np.max(np.abs(got - (fixed + weights)))
    print("max|g| %.3g of it weights %.3g error %.2e bound %.2e"
          % (np.max(np.abs(got)), np.max(np.abs(weights)), err, tol), flush=True)
    assert err <= tol
