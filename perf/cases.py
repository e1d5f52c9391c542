"""Performance cases: what a user of this engine has it do, through its public entry points.

Eight kinds of work, each over the sizes that the tests, the benchmark and its
configurations use (water clusters in cc-pVDZ and cc-pVTZ, Cartesian):

* ``fock``  one RHF Fock build, the step of every SCF cycle (1 to 64 waters);
* ``jk``    J and K of one density in a basis with f functions (1 to 8 waters, cc-pVTZ);
* ``multi`` J and K of two densities at once, the step of a UHF or ROHF cycle;
* ``batch`` J and K of several independent small molecules in one call;
* ``grad``  J/K as a differentiable operation: forward, energy, and backward to dE/dD and dE/dR;
* ``df``    the density-fitting integrals of one geometry: auxiliary metric and three-centre integrals;
* ``int1e`` the one-electron integrals and their contribution to the nuclear gradient;
* ``scf``   a whole ``run_hf_df`` call, from the molecule to the converged energy, density and orbital energies.

``mode`` is the precision the caller asks for: "mixed" (the default of the entry
points: small quartets in FP32), "f64", or "det" (bitwise reproducible).

Densities are D = 2 C C^T with C orthonormalised from orbitals localised on the
molecules, with tails that decay over a few Bohr, as those of an insulator do.
The seed makes both the geometry and the density.

``exact`` evaluates the same integrals in 64 bits by another method: the Gaussian
transform of 1/r12 integrated by Gauss-Legendre quadrature (no Rys roots, no
screening), in plain torch, with derivatives by torch's autograd.
"""

import math

import numpy as np
import torch

from asuka_amd import df, metrics
from asuka_amd.basis import build_ao_basis_cart, cartesian_components, ncart
from asuka_amd.frontend import build_int1e, run_hf_df
from asuka_amd.hf.direct_jk import (direct_fock_rhf, direct_JK, direct_JK_batched, direct_JK_multi,
                                    make_direct_jk_batch_context, make_direct_jk_context)
from asuka_amd.hf.grad import direct_jk_autograd, int1e_grad
from asuka_amd.molecule import Molecule, water_cluster_atoms_ang

DZ, TZ = "cc-pVDZ", "cc-pVTZ"


def listed():
    cases = [
        # one water: the smallest call, a dozen launches of a few workgroups each; what an SCF of a small
        # molecule repeats every cycle, in the default precision
        {"name": "fock 1 dz mixed", "kind": "fock", "n": 1, "basis": DZ, "mode": "mixed"},
        # a mid-sized molecule in plain FP64, as in the last cycles of an SCF and for reference results
        {"name": "fock 7 dz f64", "kind": "fock", "n": 7, "basis": DZ, "mode": "f64"},
        # a large cluster in FP64
        {"name": "fock 27 dz f64", "kind": "fock", "n": 27, "basis": DZ, "mode": "f64"},
        # the benchmark's size, 1600 AOs, in the default precision: the largest call
        {"name": "fock 64 dz mixed", "kind": "fock", "n": 64, "basis": DZ, "mode": "mixed"},
        # f functions on a small molecule, reproducible to the bit (regression baselines, debugging)
        {"name": "jk 2 tz det", "kind": "jk", "n": 2, "basis": TZ, "mode": "det"},
        # the benchmark's triple-zeta workload, 520 AOs, 55 class pairs
        {"name": "jk 8 tz mixed", "kind": "jk", "n": 8, "basis": TZ, "mode": "mixed"},
        # an open-shell cycle
        {"name": "multi 5 dz mixed", "kind": "multi", "n": 5, "basis": DZ, "mode": "mixed"},
        # many small molecules at once: conformers, fragments, data generation
        {"name": "batch 14 dz f64", "kind": "batch", "n": 14, "most": 9, "basis": DZ, "mode": "f64"},
        # a geometry step: energy forward, dE/dR and dE/dD backward
        {"name": "grad 9 dz f64", "kind": "grad", "n": 9, "basis": DZ, "mode": "f64"},
        # the density-fitting integrals of a geometry
        {"name": "df 6 dz", "kind": "df", "n": 6, "basis": DZ, "mode": "f64"},
        # overlap, kinetic and nuclear attraction, and their gradient term
        {"name": "int1e 16 dz", "kind": "int1e", "n": 16, "basis": DZ, "mode": "f64"},
        # the whole program of most users: one call, a molecule in and its RHF energy out
        {"name": "scf 3 dz mixed", "kind": "scf", "n": 3, "basis": DZ, "mode": "mixed"},
    ]
    return [dict(c, spacing=3.0) for c in cases]  # about the density of the liquid


# largest n of each kind (FP64 and reproducible builds cost more than mixed ones)
_MOST = {"fock": 27, "jk": 8, "multi": 12, "grad": 12, "df": 8, "int1e": 24, "scf": 4}


def draw(rng):
    kind = rng.choice(["fock", "fock", "jk", "multi", "batch", "grad", "df", "int1e", "scf"])
    mode = "f64" if kind in ("grad", "df", "int1e") else rng.choice(["mixed", "mixed", "f64"] + ["det"] * (kind in ("fock", "jk", "multi")))
    if kind == "scf" and mode == "det":
        mode = "f64"

    def size(most):
        return max(1, min(most, round(math.exp(rng.uniform(0.0, math.log(most + 0.49))))))

    spacing = round(rng.uniform(3.0, 4.0), 3)  # up to a gas of well separated molecules
    if kind == "batch":
        return {"kind": kind, "n": rng.randint(2, 24), "most": rng.randint(1, 10), "basis": DZ, "mode": mode, "spacing": spacing}
    most = 64 if (kind, mode) == ("fock", "mixed") else _MOST[kind]
    basis = TZ if kind == "jk" or (kind == "int1e" and rng.random() < 0.3) else DZ
    return {"kind": kind, "n": size(most), "basis": basis, "mode": mode, "spacing": spacing}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _molecules(case, seed):
    """The case's molecules: one cluster, or a batch of clusters of 1 to "most" waters, "spacing" angstrom apart."""

    def cluster(n, seed):
        return Molecule.from_atoms(water_cluster_atoms_ang(n, seed, spacing=case["spacing"]), unit="Angstrom",
                                   basis=case["basis"])

    if case["kind"] != "batch":
        return [cluster(case["n"], seed)]
    sizes = np.random.default_rng(case["n"]).integers(1, case["most"] + 1, case["n"])
    return [cluster(int(k), 1000 * seed + i) for i, k in enumerate(sizes)]


def _density(ao, mol, seed, scale=2.0, drop=0):
    """scale C C^T of five occupied orbitals a water (less `drop`), localised on it with decaying tails."""
    dev, n = _device(), mol.natm // 3
    at = np.repeat(np.asarray(ao.shell_cxyz), [ncart(int(l)) for l in ao.shell_l], axis=0)
    owner = np.repeat(mol.coords_bohr[::3], 5, axis=0)[: 5 * n - drop]
    far = np.linalg.norm(at[:, None, :] - owner[None, :, :], axis=2)
    C = np.random.default_rng(seed).standard_normal(far.shape) * np.exp(-far / 2.0)
    Q = torch.linalg.qr(torch.as_tensor(C, device=dev)).Q
    D = scale * (Q @ Q.T)
    return 0.5 * (D + D.T)


def _symmetric(n, seed):
    X = torch.as_tensor(np.random.default_rng(seed).standard_normal((n, n)), device=_device())
    return 0.5 * (X + X.T)


def _inputs(case, seed):
    """Molecules, bases and densities of a case (everything but the engine's contexts)."""
    kind, mols = case["kind"], _molecules(case, seed)
    if kind == "scf":
        return {"mol": mols[0]}
    aos = [build_ao_basis_cart(m)[0] for m in mols]
    Ds = [_density(a, m, seed + 17 * i) for i, (a, m) in enumerate(zip(aos, mols))]
    if kind == "batch":
        return {"aos": aos, "Ds": Ds}
    mol, ao, D = mols[0], aos[0], Ds[0]
    st = {"mol": mol, "ao": ao, "D": D}
    if kind == "multi":  # spin densities that differ by two electrons
        st["D"], st["Db"] = 0.5 * D, _density(ao, mol, seed + 1, scale=1.0, drop=2)
    if kind == "grad":
        st["R"] = torch.tensor(mol.coords_bohr, device=_device())
    if kind == "df":
        st["aux"] = df.build_aux_basis_cart(mol)
    if kind == "int1e":  # an energy-weighted density of the usual size
        st["W"] = -0.5 * _density(ao, mol, seed + 1)
    if kind == "fock":
        st["h"] = -5.0 * torch.eye(ao.nao, dtype=torch.float64, device=_device()) + 0.1 * _symmetric(ao.nao, seed + 2)
    return st


def prepare(case, seed):
    """Inputs, and the context (screened shell-pair tables of the geometry) that a program keeps over its builds."""
    st = _inputs(case, seed)
    kind = st["kind"] = case["kind"]
    st["prec"] = {"mixed_precision": case["mode"] == "mixed"}
    if kind in ("fock", "jk", "multi"):
        st["prec"]["deterministic"] = case["mode"] == "det"
    if kind == "batch":
        st["ctx"] = make_direct_jk_batch_context(st["aos"])
    elif kind == "df":
        st["ctx"] = df.make_df_context(st["ao"], st["aux"])
    elif kind != "scf":
        st["ctx"] = make_direct_jk_context(st["ao"], atom_coords_bohr=st["mol"].coords_bohr,
                                           atom_charges=st["mol"].charges)
    return st


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def run(st):
    kind = st["kind"]
    if kind == "fock":
        return direct_fock_rhf(st["ctx"], st["D"], st["h"], **st["prec"])
    if kind == "jk":
        return direct_JK(st["ctx"], st["D"], **st["prec"])
    if kind == "multi":
        return direct_JK_multi(st["ctx"], st["D"], st["Db"], **st["prec"])
    if kind == "batch":
        return direct_JK_batched(st["ctx"], st["Ds"], **st["prec"])
    if kind == "grad":
        D = st["D"].clone().requires_grad_(True)
        R = st["R"].clone().requires_grad_(True)
        J, K = direct_jk_autograd(st["ctx"], D, R, **st["prec"])
        E = 0.5 * (D * J).sum() - 0.25 * (D * K).sum()
        E.backward()
        return {"E": E.detach(), "dR": R.grad, "dD": D.grad}
    if kind == "df":
        return {"V": st["ctx"].metric(), "X": st["ctx"].int3c2e_Q()}
    if kind == "int1e":
        i = build_int1e(st["ctx"])
        return {"S": i.S, "T": i.T, "V": i.V, "g": int1e_grad(st["ctx"], Dh=st["D"], Ws=st["W"])}
    r = run_hf_df(st["mol"], two_e_backend="direct", conv_tol=1e-9, conv_tol_dm=1e-7, **st["prec"])
    return {"e": r.scf.e_tot, "dm": r.scf.dm, "mo_energy": r.scf.mo_energy}


# ---------------------------------------------------------------------------
# Work and tolerances
# ---------------------------------------------------------------------------


def _pair_bounds(ao):
    """Per pair class (la, lb): log10 of an estimate of every primitive pair's bound, sqrt((p|p)) of the s part."""
    prim = [(int(ao.shell_l[s]), ao.shell_cxyz[s], ao.prim_exp[k], ao.prim_coef[k])
            for s in range(ao.nshell) for k in range(ao.shell_prim_start[s], ao.shell_prim_start[s] + ao.shell_nprim[s])
            if ao.prim_coef[k] != 0.0]
    ls, xyz, ex, co = (np.array([p[i] for p in prim]) for i in range(4))
    out = {}
    for la in sorted(set(ls)):
        for lb in range(la + 1):
            i, j = np.nonzero(ls == la)[0], np.nonzero(ls == lb)[0]
            a, b = ex[i][:, None], ex[j][None, :]
            r2 = ((xyz[i][:, None, :] - xyz[j][None, :, :]) ** 2).sum(2)
            lg = np.log10(np.abs(co[i][:, None] * co[j][None, :])) - a * b / (a + b) * r2 / math.log(10.0) \
                + 0.5 * math.log10(34.99 / math.sqrt(2.0)) - 1.25 * np.log10(a + b)
            lg = lg[np.tril_indices(len(i))] if la == lb else lg.ravel()
            out[(int(la), lb)] = lg
    return out


def _quartet_flops(ao, flop, eps=-12.0):
    """Floating-point operations of the primitive quartets whose estimated bound reaches 10^eps."""
    edges = np.arange(-16.0, 8.1, 0.25)
    hist = {c: np.histogram(np.clip(v[v > -16.0], -16.0, 8.0), edges)[0].astype(float) for c, v in _pair_bounds(ao).items()}
    mid = 0.5 * (edges[1:] + edges[:-1])
    keep = (mid[:, None] + mid[None, :]) >= eps
    cls, total = sorted(hist), 0.0
    for x in cls:
        for y in cls:
            if y <= x:
                total += float(hist[x] @ keep @ hist[y]) * (0.5 if x == y else 1.0) * flop(*x, *y, 1)
    return total


def work(case):
    """Operations: the screened primitive quartets at the engine's counting convention (asuka_amd.metrics), estimated from
    the primitive pairs' sizes on a geometry of fixed seed. Bytes: matrices in and out."""
    kind, mols = case["kind"], _molecules(case, 1)
    aos = [build_ao_basis_cart(m)[0] for m in mols]
    n2 = float(sum(a.nao ** 2 for a in aos)) * 8.0
    if kind == "df":
        aux = df.build_aux_basis_cart(mols[0])
        pairs = {c: len(v[v > -12.0]) for c, v in _pair_bounds(aos[0]).items()}
        ints = sum(k * float(metrics.flop_eri(*c, int(l), 0, 1)) for c, k in pairs.items() for l in aux.shell_l)
        return {"bytes": 8.0 * (aux.nao * aos[0].nao ** 2 + aux.nao ** 2), "flops": ints}
    if kind == "int1e":
        pairs = {c: len(v[v > -12.0]) for c, v in _pair_bounds(aos[0]).items()}
        return {"bytes": 5 * n2, "flops": sum(5.0 * k * mols[0].natm * metrics.flop_eri(*c, 0, 0, 1) for c, k in pairs.items())}
    flops = sum(_quartet_flops(a, metrics.flop_eri) for a in aos)
    if kind == "grad":
        flops = 2 * flops + _quartet_flops(aos[0], metrics.flop_grad)
    if kind == "scf":  # about a dozen Fock builds
        flops *= 12
    return {"bytes": n2 * {"multi": 6, "grad": 5}.get(kind, 3), "flops": flops}


def tolerance(case):
    """About four times what was seen against `exact`. The builds' differences come from the density screening (K of a
    density with decaying tails is off by up to 1e-8, in FP64 as in mixed builds); an SCF's from its convergence
    threshold; the one-electron and density-fitting integrals are unscreened sums in FP64."""
    if case["kind"] == "scf":
        return {"rel": 3e-5, "max": 1e-3}
    if case["kind"] in ("df", "int1e"):
        return {"rel": 1e-12, "max": 1e-9}
    return {"rel": 4e-8, "max": 2e-6}


# ---------------------------------------------------------------------------
# The same results by another method, in 64 bits
# ---------------------------------------------------------------------------

_NODES, _WEIGHTS = np.polynomial.legendre.leggauss(40)


class _Shells:
    """Shells with a differentiable copy of their centres."""

    def __init__(self, bases, xyz=None):
        dev = _device()
        self.l, self.ao, self.prims, cen, self.n = [], [], [], [], []
        for b in bases:
            if b is None:  # the constant function 1, for three- and two-centre integrals
                self.l.append(0), self.ao.append(0), self.prims.append(([0.0], [1.0])), cen.append(np.zeros(3))
                continue
            for s in range(b.nshell):
                k = slice(b.shell_prim_start[s], b.shell_prim_start[s] + b.shell_nprim[s])
                keep = b.prim_coef[k] != 0.0
                self.l.append(int(b.shell_l[s])), self.ao.append(int(b.shell_ao_start[s]))
                self.prims.append((b.prim_exp[k][keep], b.prim_coef[k][keep])), cen.append(b.shell_cxyz[s])
        self.xyz = torch.as_tensor(np.array(cen), device=dev) if xyz is None else xyz

    def pairs(self, which):
        """{(la, lb): (shell pairs, and of each primitive pair: a, b, coefficient, shells A and B, pair)}, la >= lb."""
        out, X = {}, self.xyz.detach().cpu().numpy()
        for A, B in which:
            if self.l[A] < self.l[B]:
                A, B = B, A
            sp, pp = out.setdefault((self.l[A], self.l[B]), ([], []))
            r2 = float(((X[A] - X[B]) ** 2).sum())
            for a, ca in zip(*self.prims[A]):
                for b, cb in zip(*self.prims[B]):
                    if a * b / (a + b) * r2 < 45.0:
                        pp.append((a, b, ca * cb, A, B, len(sp)))
            sp.append((A, B))
        return {c: (sp, torch.as_tensor(np.array(pp, dtype=np.float64).reshape(-1, 6), device=_device()))
                for c, (sp, pp) in out.items()}


def _one_axis(p, q, x, PA, QC, PQ, AB, CD, l):
    """1-D integrals (i j|k m) on one axis, i <= la .. m <= ld, over the last dimension of nodes x = t^2."""
    la, lb, lc, ld = l
    s = p + q
    b0 = 0.5 * x / s
    b1, b1p = 0.5 * (1 - x * q / s) / p, 0.5 * (1 - x * p / s) / q
    c, cp = PA - q / s * x * PQ, QC + p / s * x * PQ
    G = [[None] * (lc + ld + 1) for _ in range(la + lb + 1)]
    G[0][0] = torch.ones_like(x)
    for i in range(la + lb):
        G[i + 1][0] = c * G[i][0] + (i * b1 * G[i - 1][0] if i else 0.0)
    for k in range(lc + ld):
        for i in range(la + lb + 1):
            G[i][k + 1] = cp * G[i][k] + (k * b1p * G[i][k - 1] if k else 0.0) + (i * b0 * G[i - 1][k] if i else 0.0)

    def shift(T, lo, up, d):  # T[i], i <= lo + up  ->  S[i][j], i <= lo, j <= up
        rows, out = list(T), [[None] * (up + 1) for _ in range(lo + 1)]
        for j in range(up + 1):
            for i in range(lo + 1):
                out[i][j] = rows[i]
            rows = [rows[i + 1] + d * rows[i] for i in range(len(rows) - 1)]
        return out

    ket = [shift(G[i], lc, ld, CD) for i in range(la + lb + 1)]
    full = {}
    for k in range(lc + 1):
        for m in range(ld + 1):
            S = shift([ket[i][k][m] for i in range(la + lb + 1)], la, lb, AB)
            for i in range(la + 1):
                for j in range(lb + 1):
                    full[i, j, k, m] = S[i][j]
    return full


def _tiles(sh, bra, ket, lb_, lk_):
    """sum over primitives of (ab|cd) for all products of bra and ket shell pairs, as chunks (rows of the bra's
    primitive pairs): yields (bra pair, ket pair, values [quartets, NAB, NCD]) of primitive quartets."""
    nodes = torch.as_tensor(0.5 * (_NODES + 1.0), device=_device())
    wts = torch.as_tensor(0.5 * _WEIGHTS, device=_device())
    l = (*lb_, *lk_)
    comps = [[(u, v) for u in cartesian_components(x) for v in cartesian_components(y)] for x, y in (lb_, lk_)]
    table = 3 * (l[0] + 1) * (l[1] + 1) * (l[2] + 1) * (l[3] + 1) + 3 * len(comps[1]) + 40
    step = max(1, int(6e8 / (len(_NODES) * table)) // max(1, len(ket[1])))
    kstep = max(1, int(6e8 / (len(_NODES) * table)))
    for r0 in range(0, len(bra[1]), step):
        for c0 in range(0, len(ket[1]), kstep):
            X, Y = bra[1][r0:r0 + step], ket[1][c0:c0 + kstep]
            nx, ny = len(X), len(Y)
            X, Y = X.repeat_interleave(ny, 0), Y.repeat(nx, 1)
            cen = [sh.xyz[Z[:, i].long()] for Z, i in ((X, 3), (X, 4), (Y, 3), (Y, 4))]
            a, b, c, d = X[:, 0], X[:, 1], Y[:, 0], Y[:, 1]
            p, q = a + b, c + d
            P = (a[:, None] * cen[0] + b[:, None] * cen[1]) / p[:, None]
            Q = (c[:, None] * cen[2] + d[:, None] * cen[3]) / q[:, None]
            AB, CD, PQ = cen[0] - cen[1], cen[2] - cen[3], P - Q
            pre = 2 * math.pi ** 2.5 / (p * q * (p + q).sqrt()) * X[:, 2] * Y[:, 2] * torch.exp(
                -a * b / p * (AB ** 2).sum(1) - c * d / q * (CD ** 2).sum(1))
            T = p * q / (p + q) * (PQ ** 2).sum(1)
            top = (46.0 / T.detach().clamp_min(46.0)).sqrt()  # exp(-T t^2) ends there
            t = top[:, None] * nodes
            x = t * t
            w = pre[:, None] * top[:, None] * wts * torch.exp(-T[:, None] * x)
            ax = [_one_axis(p[:, None], q[:, None], x, (P - cen[0])[:, k:k + 1], (Q - cen[2])[:, k:k + 1],
                            PQ[:, k:k + 1], AB[:, k:k + 1], CD[:, k:k + 1], l) for k in range(3)]
            rows = []
            for u, v in comps[0]:
                f = [torch.stack([ax[k][u[k], v[k], i[k], j[k]] for i, j in comps[1]], 1) for k in range(3)]
                rows.append((f[0] * f[1] * f[2] * w[:, None, :]).sum(2))
                del f
            yield X[:, 5].long(), Y[:, 5].long(), torch.stack(rows, 1)


def _places(sh, sp, second=True):
    """AO indices (first, second) of every component of every shell pair: [pairs, components]."""
    first, snd = [], []
    for A, B in sp:
        na, nb = ncart(sh.l[A]), ncart(sh.l[B])
        first.append(np.repeat(sh.ao[A] + np.arange(na), nb))
        snd.append(np.tile(sh.ao[B] + np.arange(nb), na))
    t = [torch.as_tensor(np.array(v), device=_device()) for v in (first, snd)]
    return t if second else t[0]


def _all_pairs(n):
    return [(i, j) for i in range(n) for j in range(i + 1)]


def _sum_tiles(sh, bra, ket, lb_, lk_):
    nb, nk = ncart(lb_[0]) * ncart(lb_[1]), ncart(lk_[0]) * ncart(lk_[1])
    out = torch.zeros((len(bra[0]) * len(ket[0]), nb * nk), dtype=torch.float64, device=_device())
    for i, j, v in _tiles(sh, bra, ket, lb_, lk_):
        out.index_add_(0, i * len(ket[0]) + j, v.reshape(len(v), -1))
    return out.reshape(len(bra[0]), len(ket[0]), nb, nk)


def _eri(ao):
    """(ab|cd), dense."""
    sh, n = _Shells([ao]), ao.nao
    P = sh.pairs(_all_pairs(ao.nshell))
    out = torch.zeros((n, n, n, n), dtype=torch.float64, device=_device())
    cls = sorted(P)
    for x in cls:
        for y in cls:
            if y > x:
                continue
            v = _sum_tiles(sh, P[x], P[y], x, y).permute(0, 2, 1, 3)  # [pair, NAB, pair, NCD]
            i, j = _places(sh, P[x][0])
            k, m = _places(sh, P[y][0])
            i, j, k, m = i[:, :, None, None], j[:, :, None, None], k[None, None], m[None, None]
            for s, t in ((i, j), (j, i)):
                for u, w in ((k, m), (m, k)):
                    out[s, t, u, w] = v
                    out[u, w, s, t] = v
    return out


def _jk(G, D):
    n = len(D)
    J = (G.reshape(n * n, n * n) @ D.reshape(-1)).reshape(n, n)
    K = (G.permute(0, 2, 1, 3).reshape(n * n, n * n) @ D.reshape(-1)).reshape(n, n)
    return J, K


def _grad2e(mol, ao, D):
    """d/dR of 1/2 Tr D J(D) - 1/4 Tr D K(D) at fixed D, chunk by chunk."""
    R = torch.tensor(mol.coords_bohr, device=_device())
    g = torch.zeros_like(R)
    at = torch.as_tensor(ao.shell_atom, device=_device()).long()
    base = _Shells([ao])
    P = base.pairs(_all_pairs(ao.nshell))
    for x in sorted(P):
        for y in sorted(P):
            if y > x:
                continue
            (i, j), (k, m) = _places(base, P[x][0]), _places(base, P[y][0])
            twice = [torch.tensor([1.0 if A == B else 2.0 for A, B in P[c][0]], device=_device(), dtype=torch.float64) for c in (x, y)]
            Rv = R.clone().requires_grad_(True)
            sh = _Shells([ao], Rv[at])
            for p, q, v in _tiles(sh, P[x], P[y], x, y):
                I, J, K, M = i[p][:, :, None], j[p][:, :, None], k[q][:, None, :], m[q][:, None, :]
                bar = 0.5 * D[I, J] * D[K, M] - 0.125 * (D[I, K] * D[J, M] + D[I, M] * D[J, K])
                f = twice[0][p] * twice[1][q] * (1.0 if x == y else 2.0)
                g += torch.autograd.grad((v * bar * f[:, None, None]).sum(), Rv, retain_graph=True)[0]
    return g


def _int1e(mol, ao, D=None, W=None):
    """(S, T, V, g): overlap, kinetic energy and nuclear attraction, and d/dR [Tr D (T + V) - Tr W S]."""
    R = torch.tensor(mol.coords_bohr, device=_device())
    at = torch.as_tensor(ao.shell_atom, device=_device()).long()
    Z = torch.as_tensor(mol.charges, device=_device())
    nodes, wts = torch.as_tensor(0.5 * (_NODES + 1.0), device=_device()), torch.as_tensor(0.5 * _WEIGHTS, device=_device())
    S, T, V = (torch.zeros((ao.nao, ao.nao), dtype=torch.float64, device=_device()) for _ in range(3))
    g = torch.zeros_like(R)
    P = _Shells([ao]).pairs(_all_pairs(ao.nshell))
    for (la, lb), (sp, pp) in P.items():
        first, snd = _places(_Shells([ao]), sp)
        twice = torch.tensor([1.0 if A == B else 2.0 for A, B in sp], device=_device(), dtype=torch.float64)
        comps = [(u, v) for u in cartesian_components(la) for v in cartesian_components(lb)]
        step = max(1, int(1e8 / (mol.natm * len(_NODES) * (3 * (la + 1) * (lb + 3) + 8))))
        for r0 in range(0, len(pp), step):
            X = pp[r0:r0 + step]
            Rv = R.clone().requires_grad_(D is not None)
            xyz = Rv[at]
            A, B = xyz[X[:, 3].long()], xyz[X[:, 4].long()]
            a, b = X[:, 0], X[:, 1]
            p, AB = a + b, A - B
            C = (a[:, None] * A + b[:, None] * B) / p[:, None]
            pre = X[:, 2] * torch.exp(-a * b / p * (AB ** 2).sum(1))
            # 1-D overlaps s[k][i][j] up to j = lb + 2, in units of sqrt(pi / p)
            s = []
            for k in range(3):
                PA = (C - A)[:, k]
                m = [torch.ones_like(p)]
                for i in range(la + lb + 2):
                    m.append(PA * m[i] + (i * 0.5 / p * m[i - 1] if i else 0.0))
                rows, t = m, [[None] * (lb + 3) for _ in range(la + 1)]
                for j in range(lb + 3):
                    for i in range(la + 1):
                        t[i][j] = rows[i]
                    rows = [rows[i + 1] + AB[:, k] * rows[i] for i in range(len(rows) - 1)]
                s.append(t)

            def kin(k, i, j):
                return (-2 * b * b * s[k][i][j + 2] + b * (2 * j + 1) * s[k][i][j]
                        - (0.5 * j * (j - 1) * s[k][i][j - 2] if j > 1 else 0.0))

            PN = C[:, None, :] - Rv[None, :, :]  # [pairs, atoms, 3]
            U = p[:, None] * (PN ** 2).sum(2)
            top = (46.0 / U.detach().clamp_min(46.0)).sqrt()
            x = (top[:, :, None] * nodes) ** 2
            w = -Z[None, :, None] * top[:, :, None] * wts * torch.exp(-U[:, :, None] * x)
            v = []
            for k in range(3):
                c, b1 = (C - A)[:, k, None, None] - x * PN[:, :, k, None], 0.5 * (1 - x) / p[:, None, None]
                m = [torch.ones_like(x)]
                for i in range(la + lb):
                    m.append(c * m[i] + (i * b1 * m[i - 1] if i else 0.0))
                rows, t = m, [[None] * (lb + 1) for _ in range(la + 1)]
                for j in range(lb + 1):
                    for i in range(la + 1):
                        t[i][j] = rows[i]
                    rows = [rows[i + 1] + AB[:, k, None, None] * rows[i] for i in range(len(rows) - 1)]
                v.append(t)
            o, n = pre * (math.pi / p) ** 1.5, pre * 2 * math.pi / p
            ints = [[], [], []]
            for (ux, uy, uz), (wx, wy, wz) in comps:
                sx, sy, sz = s[0][ux][wx], s[1][uy][wy], s[2][uz][wz]
                ints[0].append(o * sx * sy * sz)
                ints[1].append(o * (kin(0, ux, wx) * sy * sz + sx * kin(1, uy, wy) * sz + sx * sy * kin(2, uz, wz)))
                ints[2].append(n * (w * v[0][ux][wx] * v[1][uy][wy] * v[2][uz][wz]).sum((1, 2)))
            ints = [torch.stack(t, 1) for t in ints]
            row = X[:, 5].long()
            I, J = first[row], snd[row]
            if D is not None:
                tot = ((D[I, J] * (ints[1] + ints[2]) - W[I, J] * ints[0]) * twice[row][:, None]).sum()
                g += torch.autograd.grad(tot, Rv)[0]
            for out, t in zip((S, T, V), ints):
                out.index_put_((I, J), t.detach(), accumulate=True)
    low = torch.zeros_like(S, dtype=torch.bool)
    for (la, lb), (sp, _) in P.items():
        i, j = _places(_Shells([ao]), sp)
        low[i, j] = True
    S, T, V = (torch.where(low, X, X.T) for X in (S, T, V))
    return S, T, V, g


def _df(ao, aux):
    sh = _Shells([ao, aux, None])
    na, unit = ao.nshell, ao.nshell + aux.nshell
    AO, AX = sh.pairs(_all_pairs(na)), sh.pairs([(na + i, unit) for i in range(aux.nshell)])
    X = torch.zeros((aux.nao, ao.nao, ao.nao), dtype=torch.float64, device=_device())
    V = torch.zeros((aux.nao, aux.nao), dtype=torch.float64, device=_device())
    for y in AX:
        k = _places(sh, AX[y][0], second=False)
        for x in AO:
            v = _sum_tiles(sh, AO[x], AX[y], x, y).permute(1, 3, 0, 2)
            i, j = _places(sh, AO[x][0])
            X[k[:, :, None, None], i[None, None], j[None, None]] = v
            X[k[:, :, None, None], j[None, None], i[None, None]] = v
        for x in AX:
            i = _places(sh, AX[x][0], second=False)
            V[i[:, :, None, None], k[None, None]] = _sum_tiles(sh, AX[x], AX[y], x, y).permute(0, 2, 1, 3)
    return {"V": V, "X": X}


def _scf(mol, ao):
    """RHF to convergence with dense integrals, Roothaan cycles with DIIS."""
    S, T, V, _ = _int1e(mol, ao)
    h, G, nocc = T + V, _eri(ao), mol.nelectron // 2
    e, U = torch.linalg.eigh(S)
    X = (U * e.rsqrt()) @ U.T

    def occupied(F):
        e, C = torch.linalg.eigh(X @ F @ X)
        C = X @ C[:, :nocc]
        return e, 2.0 * C @ C.T

    eps, D = occupied(h)
    Fs, es = [], []
    for _ in range(200):
        J, K = _jk(G, D)
        F = h + J - 0.5 * K
        err = X @ (F @ D @ S - S @ D @ F) @ X
        if float(err.abs().max()) < 1e-11:
            break
        Fs, es = (Fs + [F])[-8:], (es + [err])[-8:]
        m = len(Fs)
        M = torch.ones((m + 1, m + 1), dtype=torch.float64, device=S.device)
        M[m, m] = 0.0
        M[:m, :m] = torch.stack([torch.stack([(a * b).sum() for b in es]) for a in es])
        M[:m, :m] /= M[:m, :m].diagonal().max()
        r = torch.zeros(m + 1, dtype=torch.float64, device=S.device)
        r[m] = 1.0
        c = torch.linalg.lstsq(M.cpu(), r.cpu()[:, None]).solution[:m, 0].tolist()
        eps, D = occupied(sum(x * f for x, f in zip(c, Fs)))
    eps, _ = occupied(F)
    return {"e": float(0.5 * (D * (h + F)).sum()) + mol.energy_nuc(), "dm": D, "mo_energy": eps}


def exact(case, seed):
    """Every output by quadrature; None where that would take too long (more than a few molecules)."""
    kind, n = case["kind"], case["n"]
    most = {"fock": 5, "multi": 5, "grad": 2, "df": 2, "int1e": 4, "scf": 3, "batch": 0, "jk": 2}[kind]
    if kind == "int1e" and case["basis"] == TZ:
        most = 2
    if (n > most) if kind != "batch" else (case["most"] > 3 or n > 8):
        return None
    st = _inputs(case, seed)
    if kind == "int1e":
        return dict(zip("STVg", _int1e(st["mol"], st["ao"], st["D"], st["W"])))
    if kind == "df":
        return _df(st["ao"], st["aux"])
    if kind == "scf":
        return _scf(st["mol"], build_ao_basis_cart(st["mol"])[0])
    if kind == "batch":
        return [_jk(_eri(a), D) for a, D in zip(st["aos"], st["Ds"])]
    G = _eri(st["ao"])
    J, K = _jk(G, st["D"])
    if kind == "fock":
        return st["h"] + J - 0.5 * K
    if kind == "jk":
        return J, K
    if kind == "multi":
        return J, K, *_jk(G, st["Db"])
    E = 0.5 * (st["D"] * J).sum() - 0.25 * (st["D"] * K).sum()
    # E is quadratic in D: dE/dD = J - K/2
    return {"E": E, "dR": _grad2e(st["mol"], st["ao"], st["D"]), "dD": J - 0.5 * K}
