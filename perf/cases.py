"""The work a user of this framework has it do, as timed cases.

Every case is one pass through the public entry points of `pgxc` (XCBuilder,
Batch, becke_weights) on host arrays, as a program around them calls them:

  full    a full FP64 XC build: orbitals (or the density matrix) in, packed
          V_xc, E_xc and the charge out: the first build of an SCF, and every
          build of one that stays in FP64
  step    two incremental builds in a mixed precision (||dP||_F = 1e-4 each,
          there and back): the later cycles of an SCF
  batch   FP64 builds of many molecules in one graph-replayed launch sequence
  post    after the SCF: the energy of every functional term and the nuclear
          gradient with the grid moving with the atoms (the default forces)
  force   the nuclear gradient on a fixed grid
  becke   the Becke weights of a molecular grid (a new geometry)

Systems are seeded: the molecule's geometry and its orbitals change with the
seed, the basis set is part of the case (as a basis-set library is).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "paragauss-gpl_amd"))

from pgxc import Batch, XCBuilder, basis, grid, systems  # noqa: E402
from pgxc.xc import becke_weights  # noqa: E402

DP_NORM = 1e-4   # ||dP||_F of one incremental step
NEIGHBOURS = 32  # centres in the input grids' partition

FULL = dict(kind="full", system="water", n=1, shells="small", basis_seed=1, nrad=75, nang=302,
            functional="PBE", spins=1, precision="fp64", cache=True, density="orbitals")


def _case(name, **kw):
    c = dict(FULL, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one water: the smallest call, where launches and copies count
        _case("h2o_full_fp64"),
        # the same in the later cycles of an SCF
        _case("h2o_step_bf16x3", kind="step", precision="bf16x3"),
        # an organic molecule of 23 atoms on the coarser grid, LDA, P given as a matrix
        _case("mol23_lda_full_fp64", system="molecule", n=23, basis_seed=5, nrad=55, nang=194,
              functional="LDA", density="matrix"),
        # a radical or triplet of 14 atoms: open shell
        _case("mol14_open_full_fp64", system="molecule", n=14, basis_seed=7, nrad=60, spins=2),
        # open-shell cluster in FP32 steps (the more careful mixed precision)
        _case("h2o8_open_step_fp32", kind="step", n=8, shells="medium", basis_seed=12, spins=2,
              precision="fp32"),
        # an SCF cycle of a mid-size cluster with the basis values kept on the device (the default)
        _case("h2o16_step_bf16x3", kind="step", n=16, shells="medium", basis_seed=12,
              precision="bf16x3"),
        # (H2O)32 with the basis evaluated in every build: the benchmark's workload, FP64 and mixed
        _case("h2o32_full_fp64", n=32, shells="medium", basis_seed=12, cache=False),
        _case("h2o32_step_bf16x3", kind="step", n=32, shells="medium", basis_seed=12,
              precision="bf16x3", cache=False),
        # the largest: (H2O)128 with a 40-atom solute beside it
        _case("water128_solute_step_bf16x3", kind="step", system="solute", n=128, shells="medium",
              basis_seed=42, nrad=72, precision="bf16x3", cache=False),
        # a screening run: 12 molecules of 3 to 36 atoms in one batch
        _case("batch12_fp64", kind="batch", n=12, nrad=55, nang=194, basis_seed=2000),
        # forces after the SCF, the grid moving with the atoms
        _case("h2o16_post_fp64", kind="post", n=16, shells="medium", basis_seed=12, cache=False),
        # the grid of a new geometry
        _case("h2o32_becke", kind="becke", n=32),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["full", "full", "step", "step", "step", "batch", "post", "force", "becke"])
    spins = rng.choice([1, 1, 1, 2])
    functional = rng.choice(["PBE", "PBE", "LDA"])
    water = rng.random() < 0.6
    kw = dict(kind=kind, spins=spins, functional=functional, basis_seed=rng.randrange(1, 100),
              nrad=rng.randrange(50, 76), nang=rng.choice([194, 302]),
              shells=rng.choice(["small", "medium"]), cache=rng.random() < 0.5)
    if kind == "becke":
        return _case(None, kind="becke", system="water" if water else "molecule",
                     n=_log_int(rng, 1, 40) if water else _log_int(rng, 3, 60),
                     nrad=kw["nrad"], nang=kw["nang"])
    if kind == "batch":
        return _case(None, kind="batch", n=rng.randrange(3, 13), nrad=rng.randrange(50, 60),
                     nang=194, basis_seed=2000 + rng.randrange(100), functional=functional)
    if kind == "step":
        kw["precision"] = rng.choice(["bf16x3", "bf16x3", "fp32"])
    if kind in ("post", "force"):
        return _case(None, system="water" if water else "molecule",
                     **dict(kw, n=_log_int(rng, 1, 16) if water else _log_int(rng, 3, 40), cache=False))
    if water:
        return _case(None, **dict(kw, n=_log_int(rng, 1, 24)))
    return _case(None, system="molecule", **dict(kw, n=_log_int(rng, 3, 60)),
                 density=rng.choice(["orbitals", "matrix"]))


# ------------------------------------------------------------------- inputs

def _geometry(case, seed):
    if case["system"] == "water":
        if case["n"] == 1:
            return systems.h2o(rot=systems.random_rotation(np.random.default_rng(seed)))
        return systems.water_cluster(case["n"], seed=seed, jitter_a=0.2)
    if case["system"] == "solute":  # a cluster and, 3 A beyond its extent, a 40-atom molecule
        ew, xw = systems.water_cluster(case["n"], seed=seed, jitter_a=0.2)
        es, xs = _molecule(40, case["basis_seed"] + 1, seed)
        xs = xs + np.array([xw[:, 0].max() - xs[:, 0].min() + 3.0 * systems.ANG, 0.0, 0.0])
        return list(ew) + list(es), np.vstack([xw, xs])
    return _molecule(case["n"], case["basis_seed"], seed)


def _molecule(n, which, seed):
    """A C/H/N/O molecule of its own per `which`, turned and with its atoms
    moved by up to 0.03 A along each axis by the seed."""
    els, xyz = systems.random_molecule(n, seed=which)
    rng = np.random.default_rng(seed)
    xyz = (xyz - xyz.mean(axis=0)) @ systems.random_rotation(rng).T
    return els, xyz + rng.uniform(-0.03, 0.03, size=xyz.shape) * systems.ANG


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _step(mu):
    for _ in range(3):
        mu = mu * (3.0 - mu * mu) / 2.0
    return (1.0 - mu) / 2.0


def _points(case, els, xyz):
    """Atomic grids, atom after atom: points, owner, one-centre weights (as
    grid.molecular_grid lays them out)."""
    proto = {e: grid.atomic_grid(np.zeros(3), case["nrad"], case["nang"], grid.RADIUS[e])
             for e in sorted(set(els))}
    pts = np.concatenate([proto[e][0] + x for e, x in zip(els, xyz)])
    wat = np.concatenate([proto[e][1] for e in els])
    own = np.repeat(np.arange(len(els), dtype=np.int32), [len(proto[e][1]) for e in els])
    return pts, own, wat


def _partition(xyz, pts, own, wat, near=NEIGHBOURS):
    """Becke partition over the owner's `near` nearest centres (all of them in
    small systems), so that making the input grid of a large one is cheap."""
    dev = _device()
    A = torch.as_tensor(np.asarray(xyz), device=dev)
    na = A.shape[0]
    k = min(near, na)
    if na == 1:
        return wat.copy()
    D = torch.cdist(A, A, compute_mode="donot_use_mm_for_euclid_dist")
    idx = D.topk(k, dim=1, largest=False).indices  # the owner first
    out = torch.empty(len(own), dtype=torch.float64, device=dev)
    P, O = torch.as_tensor(pts, device=dev), torch.as_tensor(own, device=dev).long()
    eye = torch.eye(k, dtype=torch.bool, device=dev)
    step = max(1, int(6e7) // (k * k))
    for s in range(0, len(own), step):
        near_a = idx[O[s:s + step]]
        r = (P[s:s + step, None, :] - A[near_a]).norm(dim=2)
        R = D[near_a[:, :, None], near_a[:, None, :]].masked_fill(eye, 1.0)
        cell = _step((r[:, :, None] - r[:, None, :]) / R).masked_fill(eye, 1.0).prod(dim=2)
        out[s:s + step] = cell[:, 0] / cell.sum(dim=1)
    return wat * out.cpu().numpy()


def _system(case, seed):
    els, xyz = _geometry(case, seed)
    b = basis.seeded_basis(els, xyz, seed=case["basis_seed"], shell_set=case["shells"])
    pts, own, wat = _points(case, els, xyz)
    w = _partition(xyz, pts, own, wat)
    return els, b, np.asfortranarray(np.column_stack([pts, w])), own


def _orbitals(case, nbas, nocc, seed):
    """Two sets of occupied orbitals with ||C1 C1^T - C0 C0^T||_F = DP_NORM to
    first order; (nbas, nocc[, 2]) as the library takes them, occupations 1."""
    sets = []
    for s in range(case["spins"]):
        rng = np.random.default_rng([seed, s])
        m = max(1, nocc - s)
        C = np.linalg.qr(rng.normal(size=(nbas, m)))[0]
        X = rng.normal(size=(nbas, m))
        X -= C @ (C.T @ X)
        C1 = C + X * (DP_NORM / (math.sqrt(2.0) * max(np.linalg.norm(X), 1e-300)))
        if m < nocc:  # the beta spin's missing orbital: unoccupied
            C, C1 = (np.concatenate([a, np.zeros((nbas, 1))], axis=1) for a in (C, C1))
        sets.append((C, C1))
    if case["spins"] == 1:
        return [np.asfortranarray(C) for C in sets[0]], np.ones(nocc)
    occ = np.ones((nocc, 2))
    if nocc > 1:
        occ[-1, 1] = 0.0
    return [np.asfortranarray(np.stack([sets[0][i], sets[1][i]], axis=2)) for i in range(2)], \
        np.asfortranarray(occ)


def _density(C, occ):
    if C.ndim == 2:
        return np.asfortranarray((C * occ) @ C.T)
    return np.asfortranarray(np.stack([(C[:, :, s] * occ[:, s]) @ C[:, :, s].T for s in range(2)], axis=2))


def _members(case, seed):
    """The molecules of a batch: 3 to 36 atoms, evenly spread."""
    n = case["n"]
    return [dict(case, kind="full", system="molecule", n=3 + (33 * i) // max(1, n - 1),
                 basis_seed=case["basis_seed"] + i) for i in range(n)], [seed * 1000 + i for i in range(n)]


def _nocc(els, nbas):
    return min(nbas // 2, max(1, sum({"H": 1, "C": 6, "N": 7, "O": 8}[e] for e in els) // 2))


def _one(case, seed, chunk_points=0):
    els, b, g, own = _system(case, seed)
    (C0, C1), occ = _orbitals(case, b.nbas, _nocc(els, b.nbas), seed)
    xc = XCBuilder(b, g, basis_cache=case["cache"], chunk_points=chunk_points)
    return dict(case=case, xc=xc, C0=C0, C1=C1, occ=occ, own=own)


def prepare(case, seed):
    if case["kind"] == "becke":
        els, xyz = _geometry(case, seed)
        pts, own, wat = _points(case, els, xyz)
        return dict(case=case, xyz=np.asarray(xyz), pts=np.asfortranarray(pts), own=own, wat=wat)
    if case["kind"] == "batch":
        mols = [_one(c, s, chunk_points=65536) for c, s in zip(*_members(case, seed))]
        return dict(case=case, mols=mols, batch=Batch([m["xc"] for m in mols]))
    st = _one(case, seed)
    if case["density"] == "matrix":
        st["P"] = _density(st["C0"], st["occ"])
    if case["kind"] in ("step", "post", "force"):
        st["xc"].set_orbitals(st["C0"], st["occ"])
        st["xc"].build(case["functional"], "fp64", fetch=False)
    return st


def run(state):
    case = state["case"]
    f, kind = case["functional"], case["kind"]
    if kind == "becke":
        return becke_weights(state["xyz"], state["pts"], state["own"], state["wat"])
    if kind == "batch":
        for m in state["mols"]:
            m["xc"].set_orbitals(m["C0"], m["occ"])
        state["batch"].build(f, "fp64", graph=True)
        return state["batch"].results()
    xc = state["xc"]
    if kind == "full":
        if case["density"] == "matrix":
            xc.set_density(state["P"])
        else:
            xc.set_orbitals(state["C0"], state["occ"])
        return xc.build(f, case["precision"])
    if kind == "step":
        out = []
        for C in (state["C1"], state["C0"]):
            xc.set_orbitals(C, state["occ"], incremental=True)
            out.append(xc.build(f, case["precision"]))
        return out
    if kind == "post":
        terms, charge = xc.energy(f, "fp64")
        return [terms, charge, xc.gradient_grid(state["own"])]
    return xc.gradient()


# --------------------------------------------------------------------- work

def work(case):
    """Points x functions that are not exactly zero there (sampled on the
    geometry of seed 0): the products and the evaluation no path can leave out."""
    if case["kind"] == "batch":
        parts = [work(c) for c in _members(case, 0)[0]]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    els, xyz = _geometry(case, 0)
    A = np.asarray(xyz)
    npt = {e: len(grid.radial_grid(grid.radial_shells(case["nrad"], grid.RADIUS[e]),
                                   grid.RADIUS[e])[0]) * case["nang"] for e in set(els)}
    npts = sum(npt[e] for e in els)
    if case["kind"] == "becke":
        # per pair of centres one step function (its mirror is 1 - s), 12 operations
        return {"bytes": npts * 44.0 + 24.0 * len(els), "flops": npts * 6.0 * len(els) ** 2}
    b = basis.seeded_basis(els, xyz, seed=case["basis_seed"], shell_set=case["shells"])
    rng = np.random.default_rng(0)
    sh_atom = np.array([s.atom for s in b.shells])
    reach = np.array([50.0 / s.exps.min() for s in b.shells])
    nf = np.array([s.nfunc for s in b.shells], dtype=float)
    n1 = n2 = wsum = 0.0
    for e in sorted(set(els)):
        pts, _ = grid.atomic_grid(np.zeros(3), case["nrad"], case["nang"], grid.RADIUS[e])
        atoms = [i for i, x in enumerate(els) if x == e]
        pick = rng.choice(atoms, 128)
        p = pts[rng.integers(0, len(pts), 128)] + A[pick]
        r2 = ((p[:, None, :] - A[None]) ** 2).sum(axis=2)[:, sh_atom]
        n = ((r2 < reach) * nf).sum(axis=1)
        n1 += n.mean() * npt[e] * len(atoms)
        n2 += (n * n).mean() * npt[e] * len(atoms)
        wsum += npt[e] * len(atoms)
    nbas, nocc, s = b.nbas, _nocc(els, b.nbas), case["spins"]
    gga = case["functional"] == "PBE"
    in_out = 8.0 * s * (nbas * nocc + nbas * (nbas + 1) / 2)
    build = s * (4.0 * n2 + 16.0 * n1) if gga else s * (4.0 * n2 + 4.0 * n1)
    if case["kind"] == "full":
        return {"bytes": 32.0 * npts + in_out, "flops": build}
    if case["kind"] == "step":  # two builds, each reading and writing the per-point state
        return {"bytes": 2 * (32.0 * npts + s * (128.0 if gga else 32.0) * npts + in_out),
                "flops": 2 * build}
    # gradients: the products of the values and, for GGA, of the gradients
    force = s * (2.0 * n2 * (4 if gga else 1) + 60.0 * n1)
    out = {"bytes": 32.0 * npts + s * 64.0 * npts + 24.0 * len(els), "flops": force}
    if case["kind"] == "post":
        out["bytes"] += 4.0 * npts + 8.0 * s * nbas * nocc
        out["flops"] += s * 2.0 * n2 + npts * 12.0 * len(els) ** 2
    return out


# -------------------------------------------------------------------- exact
# The same sums in torch FP64: basis values from closed forms (s, p, d), the
# functional differentiated by autograd, V by one product per block of points.

_DEPS = 1.0e-30


def _harmonics(x, y, z, l):
    """Racah-normalised solid harmonics of l, stacked last, in the order z-like,
    then the (x, y) pairs."""
    if l == 0:
        return torch.ones_like(x)[..., None]
    if l == 1:
        return torch.stack([z, x, y], dim=-1)
    q = math.sqrt(3.0)
    r2 = x * x + y * y + z * z
    return torch.stack([1.5 * z * z - 0.5 * r2, q * z * x, q * z * y,
                        0.5 * q * (x * x - y * y), q * x * y], dim=-1)


def _harmonics_grad(x, y, z, l):
    o, i = torch.zeros_like(x), torch.ones_like(x)
    if l == 0:
        return [torch.stack([o], dim=-1)] * 3
    if l == 1:
        return [torch.stack(t, dim=-1) for t in ([o, i, o], [o, o, i], [i, o, o])]
    q = math.sqrt(3.0)
    return [torch.stack(t, dim=-1) for t in (
        [-x, q * z, o, q * x, q * y], [-y, o, q * z, -q * y, q * x], [2.0 * z, q * x, q * y, o, o])]


def _tables(els, b, dev):
    """Shells grouped by (element, l): atoms, exponents, contraction matrix and
    the first function of each atom's shell."""
    groups, off = {}, 0
    for s in b.shells:
        groups.setdefault((els[s.atom], s.l, len(s.exps), s.n_unc), []).append((s, off))
        off += s.nfunc
    out = []
    for (e, l, ne, nu), members in sorted(groups.items()):
        s = members[0][0]
        M = np.zeros((ne, nu + s.n_contr))
        M[np.arange(nu), np.arange(nu)] = 1.0
        M[:, nu:] = s.contr
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
        out.append(dict(l=l, atoms=np.array([m[0].atom for m in members]),
                        offs=np.array([m[1] for m in members]), ex=t(s.exps),
                        M=t(M * s.norms[:, None]), reach=math.sqrt(50.0 / s.exps.min())))
    return out


def _block_basis(tabs, R, p, lo, hi, dev):
    """Values and gradients (n_points, n_live) of the functions that can be
    nonzero in the box [lo, hi], and their caller indices."""
    cols, vals, grads = [], [], [[], [], []]
    Rh = R.detach().cpu().numpy()
    for g in tabs:
        c = Rh[g["atoms"]]
        d = np.maximum(np.maximum(lo - c, c - hi), 0.0)
        live = np.flatnonzero((d * d).sum(axis=1) < g["reach"] ** 2)
        if not len(live):
            continue
        at = torch.as_tensor(g["atoms"][live], device=dev)
        v = p[:, None, :] - R[at][None]
        x, y, z = v[..., 0], v[..., 1], v[..., 2]
        r2 = x * x + y * y + z * z
        ar2 = r2[..., None] * g["ex"]
        prim = torch.where(ar2 < 50.0, torch.exp(-ar2), torch.zeros_like(ar2))
        R0, R1 = prim @ g["M"], (prim * (-2.0 * g["ex"])) @ g["M"]
        S, dS = _harmonics(x, y, z, g["l"]), _harmonics_grad(x, y, z, g["l"])
        n, nl = p.shape[0], len(live)
        val = S[..., :, None] * R0[..., None, :]
        nf = val.shape[2] * val.shape[3]
        vals.append(val.reshape(n, nl * nf))
        for k, xk in enumerate((x, y, z)):
            gk = dS[k][..., :, None] * R0[..., None, :] + (xk[..., None] * S)[..., :, None] * R1[..., None, :]
            grads[k].append(gk.reshape(n, nl * nf))
        cols.append((g["offs"][live][:, None] + np.arange(nf)).reshape(-1))
    if not cols:
        return None, None, None
    idx = torch.as_tensor(np.concatenate(cols), device=dev)
    return torch.cat(vals, 1), [torch.cat(t, 1) for t in grads], idx


def _pw92(n, z):
    """eps_c(n, zeta) with the reference's digits."""
    rs = (3.0 / (4.0 * math.pi)) ** (1.0 / 3.0) / n ** (1.0 / 3.0)
    s = rs.sqrt()

    def G(A, a1, b1, b2, b3, b4):
        q = 2.0 * A * (b1 * s + b2 * rs + b3 * rs * s + b4 * rs * rs)
        return -2.0 * A * (1.0 + a1 * rs) * torch.log1p(1.0 / q)

    eu = G(0.031091, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294)
    if z is None:
        return eu
    ep = G(0.015545, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517)
    ma = G(0.016887, 0.11125, 10.357, 3.6231, 0.88026, 0.49671)
    cf = 1.0 / (2.0 * 2.0 ** (1.0 / 3.0) - 2.0)
    f = ((1.0 + z + _DEPS) ** (4.0 / 3.0) + (1.0 - z + _DEPS) ** (4.0 / 3.0) - 2.0) * cf
    return eu + (ep - eu) * f * z ** 4 - ma * f * (1.0 - z ** 4) * (9.0 / (8.0 * cf))


def _terms(gga, na, nb, gaa, gbb, gab):
    """XAlpha, PWLDAc, PBEx, PBEc energy densities (na is nb: closed shell)."""
    closed = nb is None
    cx = -0.75 * (3.0 / math.pi) ** (1.0 / 3.0)
    mu, kappa = 0.066725 * math.pi ** 2 / 3.0, 0.804
    spins = [(2.0 * na, 4.0 * gaa)] if closed else [(2.0 * na, 4.0 * gaa), (2.0 * nb, 4.0 * gbb)]
    share = 1.0 / len(spins)
    ex = sum(share * cx * n ** (4.0 / 3.0) for n, _ in spins)
    n = 2.0 * na if closed else na + nb
    z = None if closed else (na - nb) / n
    ec = _pw92(n, z)
    if not gga:
        return [ex, n * ec, torch.zeros_like(n), torch.zeros_like(n)]
    kf2 = (3.0 * math.pi ** 2) ** (2.0 / 3.0)
    exg = 0.0
    for m, g in spins:
        s2 = g / (4.0 * kf2 * m ** (8.0 / 3.0))
        exg = exg + share * cx * m ** (4.0 / 3.0) * kappa * mu * s2 / (kappa + mu * s2)
    beta, gam = 0.066725, 0.03109069086965489503494086371
    fi = 1.0 if closed else ((na / n) ** (2.0 / 3.0) + (nb / n) ** (2.0 / 3.0)) / 2.0 ** (1.0 / 3.0)
    A = beta / gam / torch.expm1(-ec / (gam * fi ** 3))
    g2 = 4.0 * gaa if closed else gaa + gbb + 2.0 * gab
    t2 = math.pi / (16.0 * (3.0 * math.pi ** 2) ** (1.0 / 3.0)) * g2 / (fi ** 2 * n ** (7.0 / 3.0))
    x = A * t2
    H = gam * fi ** 3 * torch.log1p(beta / gam * t2 * (1.0 + x) / (1.0 + x + x * x))
    return [ex, n * ec, exg, n * H]


def _functional(case, rho, gr):
    """The terms per point and their derivatives: rho[s], gr[s] = (n, 3)."""
    ok = rho[0] > 1e-25
    for r in rho[1:]:
        ok = ok & (r > 1e-25)
    gga = case["functional"] == "PBE"
    with torch.enable_grad():
        q = [torch.where(ok, r, torch.ones_like(r)).detach().requires_grad_() for r in rho]
        G = [torch.where(ok[:, None], g, torch.zeros_like(g)).detach() for g in gr]
        if len(rho) == 1:
            gam = (G[0] * G[0]).sum(1).requires_grad_()
            e = _terms(gga, 0.5 * q[0], None, 0.25 * gam, None, None)
            d = torch.autograd.grad(sum(t.sum() for t in e), [q[0], gam], allow_unused=True)
            d = [t if t is not None else torch.zeros_like(gam) for t in d]
            b = [2.0 * d[1][:, None] * G[0]]
            a = [0.5 * d[0]]
        else:
            s = [(G[0] * G[0]).sum(1).requires_grad_(), (G[1] * G[1]).sum(1).requires_grad_(),
                 (G[0] * G[1]).sum(1).requires_grad_()]
            e = _terms(gga, q[0], q[1], *s)
            d = torch.autograd.grad(sum(t.sum() for t in e), q + s, allow_unused=True)
            d = [t if t is not None else torch.zeros_like(s[0]) for t in d]
            a = [0.5 * d[0], 0.5 * d[1]]
            b = [2.0 * d[2][:, None] * G[0] + d[4][:, None] * G[1],
                 2.0 * d[3][:, None] * G[1] + d[4][:, None] * G[0]]
    zero = lambda t: torch.where(ok if t.dim() == 1 else ok[:, None], t, torch.zeros_like(t)).detach()  # noqa: E731
    return [zero(t) for t in e], [zero(t) for t in a], [zero(t) for t in b]


def _blocks(pts, size):
    """Points in boxes of 5 bohr, cut into blocks of at most `size`."""
    c = np.floor(pts / 5.0).astype(np.int64)
    key = (c[:, 0] << 42) ^ ((c[:, 1] + (1 << 20)) << 21) ^ (c[:, 2] + (1 << 20))
    order = np.argsort(key, kind="stable")
    cuts = np.flatnonzero(np.diff(key[order])) + 1
    out, start = [], 0
    for end in list(cuts) + [len(order)]:
        for s in range(start, end, size):
            out.append(order[s:min(end, s + size)])
        start = end
    # neighbouring small boxes together
    merged, cur = [], []
    for o in out:
        if cur and sum(map(len, cur)) + len(o) > size // 4:
            merged.append(np.concatenate(cur))
            cur = []
        cur.append(o)
    if cur:
        merged.append(np.concatenate(cur))
    return merged


def _integrate(case, els, b, g, Ps, forces=None):
    """E terms, charge and V per spin of every density set in Ps (a list of
    lists of P per spin); forces: the atom of every point, adds dE/dR."""
    dev = _device()
    R = torch.as_tensor(b.atom_xyz, device=dev)
    tabs = _tables(els, b, dev)
    T = torch.as_tensor(np.ascontiguousarray(g), device=dev)
    gga, ns = case["functional"] == "PBE", case["spins"]
    e = [torch.zeros(5, dtype=torch.float64, device=dev) for _ in Ps]
    V = [[torch.zeros_like(p) for p in P] for P in Ps]
    F = torch.zeros_like(R)
    for sel in _blocks(g[:, :3], 8192 if forces is not None else 16384):
        i = torch.as_tensor(sel, device=dev)
        p, w = T[i, :3], T[i, 3]
        lo, hi = g[sel, :3].min(axis=0), g[sel, :3].max(axis=0)
        val, grd, idx = _block_basis(tabs, R, p, lo, hi, dev)
        if idx is None:
            continue
        for k, P in enumerate(Ps):
            sub = [q[idx][:, idx] for q in P]
            X = [val @ q for q in sub]
            rho = [(x * val).sum(1) for x in X]
            gr = [torch.stack([2.0 * (x * t).sum(1) for t in grd], 1) for x in X]
            t, a, bb = _functional(case, rho, gr)
            for j in range(4):
                e[k][j] += (t[j] * w).sum()
            e[k][4] += (sum(rho) * w).sum()
            for s in range(ns):
                W = (a[s] * w)[:, None] * val
                if gga:
                    for c in range(3):
                        W = W + (bb[s][:, c] * w)[:, None] * grd[c]
                H = val.T @ W
                V[k][s].view(-1).index_put_(((idx[:, None] * V[k][s].shape[0] + idx[None, :]).reshape(-1),),
                                            (H + H.T).reshape(-1), accumulate=True)
            if forces is not None:
                F += _block_forces(case, tabs, R, p, w, lo, hi, a, bb, sum(t), sub, idx, i, forces, dev)
    return e, V, F


def _block_forces(case, tabs, R, p, w, lo, hi, a, bb, f, sub, idx, i, forces, dev):
    """dE/dR of one block: sum_p w (dF/drho drho + dF/dgrad . dgrad) with the
    centres (and, when the grid moves, the points and their weights)."""
    with torch.enable_grad():
        Rv = R.clone().requires_grad_()
        own, moving = forces
        o = own[i]
        q = p + (Rv[o] - R[o]) if moving else p
        val, grd, idx2 = _block_basis(tabs, Rv, q, lo, hi, dev)
        assert torch.equal(idx, idx2)
        e = 0.0
        for s, P in enumerate(sub):
            X = val @ P
            e = e + (2.0 * a[s] * w * (X * val).sum(1)).sum()
            if case["functional"] == "PBE":
                for c in range(3):
                    e = e + (bb[s][:, c] * w * 2.0 * (X * grd[c]).sum(1)).sum()
        if moving:
            D = (Rv[:, None, :] - Rv[None, :, :])
            na = R.shape[0]
            eye = torch.eye(na, dtype=torch.bool, device=dev)
            D = (D * D).sum(2).masked_fill(eye, 1.0).sqrt()
            for s0 in range(0, len(i), 2048):
                qq = q[s0:s0 + 2048]
                r = ((qq[:, None, :] - Rv[None]) ** 2).sum(2).clamp_min(1e-300).sqrt()
                cell = _step((r[:, :, None] - r[:, None, :]) / D).masked_fill(eye, 1.0)
                lp = cell.clamp_min(1e-300).log().sum(2)
                lb = lp.gather(1, o[s0:s0 + 2048, None])[:, 0] - torch.logsumexp(lp, 1)
                wf = (w * f)[s0:s0 + 2048]
                e = e + (torch.where(wf != 0.0, lb, torch.zeros_like(lb)) * wf).sum()
        return torch.autograd.grad(e, Rv)[0].detach()


def _spins(P):
    dev = _device()
    return [torch.as_tensor(np.ascontiguousarray(P if P.ndim == 2 else P[:, :, s]), device=dev)
            for s in range(1 if P.ndim == 2 else 2)]


def _packed(V):
    n = V[0].shape[0]
    j, k = np.tril_indices(n)
    rows = [v.cpu().numpy()[j, k] for v in V]
    if len(rows) == 1:
        return rows[0]
    return np.stack(rows, axis=1).reshape(-1)


def _built(e, V):
    return _packed(V), float(e[:4].sum()), float(e[4])


def exact(case, seed):
    kind = case["kind"]
    if kind == "becke":
        els, xyz = _geometry(case, seed)
        pts, own, wat = _points(case, els, xyz)
        return _exact_becke(np.asarray(xyz), pts, own, wat)
    if kind == "batch":
        return [_exact_one(c, s) for c, s in zip(*_members(case, seed))]
    return _exact_one(case, seed)


def _exact_becke(xyz, pts, own, wat):
    return _partition(xyz, pts, own, wat, near=len(xyz))


def _exact_one(case, seed):
    els, b, g, own = _system(case, seed)
    (C0, C1), occ = _orbitals(case, b.nbas, _nocc(els, b.nbas), seed)
    P0 = _spins(_density(C0, occ))
    if case["kind"] == "full":
        e, V, _ = _integrate(case, els, b, g, [P0])
        return _built(e[0], V[0])
    if case["kind"] == "step":
        e, V, _ = _integrate(case, els, b, g, [_spins(_density(C1, occ)), P0])
        return [_built(x, v) for x, v in zip(e, V)]
    o = torch.as_tensor(own, device=_device()).long()
    e, _, F = _integrate(case, els, b, g, [P0], forces=(o, case["kind"] == "post"))
    force = F.cpu().numpy()
    if case["kind"] == "force":
        return force
    t = dict(zip(("xalpha", "pwldac", "pbex", "pbec"), [float(x) for x in e[0][:4]]))
    return [t, float(e[0][4]), force]
