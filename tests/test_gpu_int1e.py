"""One-electron kernels where their work split can go wrong: the lanes of a
wave are divided into groups over the nuclei (a power of two up to 64) and
primitive pairs (64 at a time), so numbers of nuclei around those borders,
contractions of one and of more than 64 primitive pairs (with zero
coefficients among them), and every class up to (ff|, against the oracle.

S, T, V: the sums have at most a few thousand terms of the size of the largest
element, so 1e-12 of it bounds their rounding. The gradient is compared with
five-point differences of the oracle's integrals (step 5e-3 Bohr): their
truncation, h^4 times a fifth derivative, is below 1e-6 of the largest entry
for the exponents used."""

import numpy as np
import pytest

from asuka_amd.basis import pack_cart_basis, parse_basis_dict

pytestmark = pytest.mark.gpu

# nine primitives in two columns (81 primitive pairs, some of them zero) and one shell of each higher l
EXPS = [40.0, 18.0, 9.0, 5.0, 2.6, 1.4, 0.8, 0.45, 0.2]
FULL = {"O": [[0] + [[e, 0.1 + 0.05 * k, 0.0 if k % 2 else 0.3] for k, e in enumerate(EXPS)],
              [1, [1.3, 0.4, 0.0], [0.4, 0.7, 1.0]], [2, [0.9, 1.0]], [3, [1.1, 1.0]]],
        "H": [[0, [0.9, 1.0]]]}
SMALL = {"O": [[0, [1.1, 1.0]], [1, [0.7, 1.0]]], "H": [[0, [0.6, 1.0]]]}


def _atoms(n, seed):
    rng = np.random.default_rng(seed)
    xyz = rng.uniform(-2.0, 2.0, size=(n, 3)) * max(1.0, n / 8.0) ** (1.0 / 3.0)
    return [("O" if i == 0 else "H", x) for i, x in enumerate(xyz)]


def _build(atoms, spec):
    ao = pack_cart_basis(atoms, parse_basis_dict(spec, sorted({s for s, _ in atoms})))
    return ao, np.array([x for _, x in atoms]), np.array([8.0 if s == "O" else 1.0 for s, _ in atoms])


def _ctx(ao, xyz, Z):
    from asuka_amd.hf.direct_jk import make_direct_jk_context

    return make_direct_jk_context(ao, atom_coords_bohr=xyz, atom_charges=Z)


@pytest.mark.parametrize("natm,spec", [(1, FULL), (2, FULL), (5, FULL), (64, SMALL), (65, SMALL)])
def test_int1e_against_oracle(gpu, oracle, natm, spec):
    from asuka_amd.frontend import build_int1e

    ao, xyz, Z = _build(_atoms(natm, natm), spec)
    i = build_int1e(_ctx(ao, xyz, Z))
    for got, ref in zip((i.S, i.T, i.V), oracle.int1e(ao, xyz, Z)):
        g = got.cpu().numpy()
        assert np.array_equal(g, g.T)
        assert np.abs(g - ref).max() < 1e-12 * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("natm,spec", [(2, FULL), (5, FULL), (65, SMALL)])
def test_int1e_grad_against_differences(gpu, oracle, natm, spec):
    from asuka_amd.hf.grad import int1e_grad

    atoms = _atoms(natm, natm + 1)
    ao, xyz, Z = _build(atoms, spec)
    rng = np.random.default_rng(3)
    Dh, Ws = (0.5 * (X + X.T) for X in rng.standard_normal((2, ao.nao, ao.nao)))
    ctx = _ctx(ao, xyz, Z)
    g = int1e_grad(ctx, Dh=Dh, Ws=Ws).cpu().numpy()
    assert np.abs(g.sum(axis=0)).max() < 1e-10 * np.abs(g).max()  # translational invariance

    def L(x):
        a = [(s, p) for (s, _), p in zip(atoms, x)]
        S, T, V = oracle.int1e(_build(a, spec)[0], x, Z)
        return float((Dh * (T + V)).sum() - (Ws * S).sum())

    h = 5e-3
    for k in rng.choice(3 * natm, 4, replace=False):
        e = np.zeros((natm, 3))
        e.flat[k] = h
        d = (8.0 * (L(xyz + e) - L(xyz - e)) - (L(xyz + 2 * e) - L(xyz - 2 * e))) / (12.0 * h)
        assert abs(d - g.flat[k]) < 1e-6 * np.abs(g).max(), (k, d, g.flat[k])
    # one of the two matrices alone
    both = int1e_grad(ctx, Dh=Dh).cpu().numpy() + int1e_grad(ctx, Ws=Ws).cpu().numpy()
    assert np.abs(both - g).max() < 1e-11 * np.abs(g).max()


def test_int1e_grad_beyond_the_lds_sums(gpu, oracle):
    """513 nuclei, one more than the LDS sums of the nuclei's forces hold: they
    go to the output one by one. Most are point charges without functions."""
    from asuka_amd.hf.grad import int1e_grad

    atoms = _atoms(3, 11)
    ao, xyz, Z = _build(atoms, FULL)
    rng = np.random.default_rng(12)
    far = rng.uniform(-1.0, 1.0, size=(510, 3))
    far *= (4.0 + 8.0 * rng.random((510, 1))) / np.linalg.norm(far, axis=1, keepdims=True)
    Dh, Ws = (0.5 * (X + X.T) for X in rng.standard_normal((2, ao.nao, ao.nao)))
    x0, Z = np.vstack([xyz, far]), np.concatenate([Z, np.full(510, 0.1)])
    grads = [int1e_grad(_ctx(ao, x0[:n], Z[:n]), Dh=Dh, Ws=Ws).cpu().numpy() for n in (513, 512)]
    assert np.abs(grads[0].sum(axis=0)).max() < 1e-10 * np.abs(grads[0]).max()
    # the last charge on its own: what it adds to the others, and its force
    Zl = np.where(np.arange(513) == 512, Z, 0.0)
    last = int1e_grad(_ctx(ao, x0, Zl), Dh=Dh).cpu().numpy()
    rest = int1e_grad(_ctx(ao, x0, 0.0 * Z), Dh=Dh).cpu().numpy()
    diff = grads[0] - np.vstack([grads[1], np.zeros((1, 3))])
    assert np.abs(diff - (last - rest)).max() < 1e-11 * np.abs(grads[0]).max()

    def L(x):
        S, T, V = oracle.int1e(_build([(s, p) for (s, _), p in zip(atoms, x)], FULL)[0], x, Z)
        return float((Dh * (T + V)).sum() - (Ws * S).sum())

    h = 5e-3
    for k in (0, 7, 3 * 200 + 1, 3 * 512 + 2):
        e = np.zeros((513, 3))
        e.flat[k] = h
        d = (8.0 * (L(x0 + e) - L(x0 - e)) - (L(x0 + 2 * e) - L(x0 - 2 * e))) / (12.0 * h)
        assert abs(d - grads[0].flat[k]) < 1e-6 * np.abs(grads[0]).max(), k
