"""Wave units cut into slices of their primitive quartets (small contexts):
contractions that leave only the bra, only the ket, both or neither to cut,
counts around the cut sizes, with and without primitive screening, in J/K
(FP64, FP32, mixed and reproducible) and in the derivative kernels, against the
oracle. 1e-10 as in the other J/K tests: the slices only regroup sums, and
default mixed builds of contexts this small run all of it in FP64. With
tau_mixed = 1e3 every quartet of the register kernels is FP32: roundings of 6e-8
along chains of a few dozen operations, 2e-6."""

import numpy as np
import pytest

from asuka_amd.basis import pack_cart_basis, parse_basis_dict

pytestmark = pytest.mark.gpu


def _contraction(l, n, lo=0.25, ratio=1.9):
    return [l] + [[lo * ratio ** k, 0.2 + 0.6 / (1 + k)] for k in range(n)]


def _case(ns, np_, nd):
    """Two centres: s, p and d shells of ns, np_ and nd primitives, and an uncontracted s."""
    spec = {"O": [_contraction(0, ns), _contraction(1, np_)] + ([_contraction(2, nd, 0.7)] if nd else []),
            "H": [_contraction(0, 1, 0.4), _contraction(0, ns, 0.3, 2.3)]}
    atoms = [("O", np.array([0.1, -0.2, 0.05])), ("H", np.array([0.3, 0.4, 1.6]))]
    return pack_cart_basis(atoms, parse_basis_dict(spec, ["H", "O"])), np.array([x for _, x in atoms])


CASES = [(1, 1, 0), (3, 2, 1), (7, 1, 0), (8, 5, 0), (17, 3, 2)]


@pytest.mark.parametrize("ns,np_,nd", CASES)
@pytest.mark.parametrize("eps", [0.0, 1e-14])
def test_sliced_jk(gpu, oracle, ns, np_, nd, eps):
    from asuka_amd.hf.direct_jk import direct_JK, make_direct_jk_context

    ao, _ = _case(ns, np_, nd)
    n = ao.nao
    D = np.random.default_rng(n).standard_normal((n, n))
    D = 0.5 * (D + D.T)
    octx = oracle.make_context(ao)
    Jr, Kr = oracle.dense_JK(oracle.dense_eri(octx), D)
    ctx = make_direct_jk_context(ao, eps_schwarz=eps, eps_density=0.0)
    ctx32 = make_direct_jk_context(ao, eps_schwarz=eps, eps_density=0.0, tau_mixed=1e3)
    scale = max(1.0, np.abs(Jr).max())
    for c, kw, tol in ((ctx, {"mixed_precision": False}, 1e-10), (ctx, {"deterministic": True}, 1e-10),
                       (ctx, {"mixed_precision": True}, 1e-10), (ctx32, {"mixed_precision": True}, 2e-6)):
        stats = {}
        J, K = direct_JK(c, D, stats=stats, **kw)
        err = max(np.abs(J.cpu().numpy() - Jr).max(), np.abs(K.cpu().numpy() - Kr).max()) / scale
        assert err < tol
        # the counters take a quartet by its first slice alone
        assert stats["direct_jk_evaluated"] == c.ntasks
        for q in stats["class_counts"]:  # all FP32 or none, in the register kernels' classes
            if q["prim_quartets_evaluated"]:
                assert q["quartets_fp32"] == (q["bins"].sum() if c is ctx32 else 0)


@pytest.mark.parametrize("ns,np_,nd", CASES)
def test_sliced_gradient(gpu, oracle, ns, np_, nd):
    from asuka_amd.hf.direct_jk import make_direct_jk_context
    from asuka_amd.hf.grad import direct_jk_grad

    ao, xyz = _case(ns, np_, nd)
    n = ao.nao
    rng = np.random.default_rng(n)
    D, WJ, WK = (0.5 * (X + X.T) for X in rng.standard_normal((3, n, n)))
    ref = oracle.grad2e(oracle.make_context(ao), D, WJ, WK, ao.shell_atom, 2, hp=False, threads=0)
    for eps in (0.0, 1e-14):
        ctx = make_direct_jk_context(ao, eps_schwarz=eps, eps_density=0.0, atom_coords_bohr=xyz,
                                     atom_charges=np.array([8.0, 1.0]))
        g = direct_jk_grad(ctx, D, WJ, WK).cpu().numpy()
        assert np.abs(g - ref).max() < 1e-10 * max(1.0, np.abs(ref).max())


def test_slices_skip_the_same_primitive_quartets(gpu):
    """A 4-water cluster alone (cut into slices) and beside a 12-water one in a
    batch (whose units are longer, so it is cut less) leave out the same
    primitive quartets in FP64. The sums then differ by their order alone: fewer
    than 1e5 terms into elements below 1e2, whose roundings (1.4e-14 each at
    most) add up as their square root, under 5e-12."""
    import torch

    from asuka_amd.basis import build_ao_basis_cart
    from asuka_amd.hf.direct_jk import direct_JK_batched, make_direct_jk_batch_context, make_direct_jk_context
    from asuka_amd.molecule import water_cluster

    aos, Ds = [], []
    for n, seed in ((4, 3), (12, 17)):
        ao, _ = build_ao_basis_cart(water_cluster(n, 1000 + seed, "cc-pVDZ"))
        C, _ = np.linalg.qr(np.random.default_rng(2000 + seed).standard_normal((ao.nao, 5 * n)))
        aos.append(ao)
        Ds.append(torch.tensor(2.0 * C @ C.T, device="cuda"))
    batch = direct_JK_batched(make_direct_jk_batch_context(aos, eps_schwarz=1e-12), Ds, mixed_precision=False)
    alone = direct_JK_batched([make_direct_jk_context(ao, eps_schwarz=1e-12) for ao in aos], Ds, mixed_precision=False)
    for a, b in zip(batch, alone):
        for x, y in zip(a, b):
            assert float((x - y).abs().max()) < 2e-12  # well inside that
