"""The autotuner and tuning tables (asuka_jk_autotune, asuka_jk_tuning_get/set).

Launch shapes change only how work is cut and where it is summed, never
which quartets are evaluated, so every shape must reproduce the oracle's
golden J/K to the FP64 bar (1e-10 absolute): the tuned shapes, and two
forced extremes applied to every class pair (8 wavefronts per workgroup, 8
wave units per task, no LDS accumulators; 4 wavefronts, 64 units, LDS
accumulators where they fit).
"""

import os

import numpy as np
import pytest

from asuka_amd.basis import build_ao_basis_cart
from asuka_amd.molecule import water_cluster

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
CASES = {"h2o2_tz": (2, 2, "cc-pVTZ"), "h2o4_dz": (4, 4, "cc-pVDZ")}


def _ctx(mol, **kw):
    from asuka_amd.hf.direct_jk import make_direct_jk_context

    ao, _ = build_ao_basis_cart(mol)
    return ao, make_direct_jk_context(ao, atom_coords_bohr=mol.coords_bohr, atom_charges=mol.charges, **kw)


@pytest.fixture(scope="module")
def jk_golden():
    return dict(np.load(os.path.join(HERE, "golden", "jk_golden.npz"), allow_pickle=False))


def _check(ctx, D, golden, case):
    from asuka_amd.hf.direct_jk import direct_JK

    J, K = direct_JK(ctx, D)
    assert np.max(np.abs(J.cpu().numpy() - golden[f"{case}_J_scr"])) < 1e-10
    assert np.max(np.abs(K.cpu().numpy() - golden[f"{case}_K_scr"])) < 1e-10


@pytest.mark.parametrize("case", sorted(CASES))
def test_autotune_keeps_parity(gpu, jk_golden, case):
    n, seed, basis = CASES[case]
    mol = water_cluster(n, seed, basis)
    D = jk_golden[f"{case}_D"]
    _, ctx = _ctx(mol, eps_schwarz=1e-12)
    table = ctx.autotune(D, reps=1)
    assert len(table) > 0 and all(t["tuned_ms"] > 0 for t in table)
    assert {t["waves_per_group"] for t in table} <= {4, 8}
    assert all(t["units_per_task"] in (16, 32, 64, 128) for t in table)  # a candidate or the default cut
    _check(ctx, D, jk_golden, case)
    # the table carries over to a fresh context of the same molecule
    _, ctx2 = _ctx(mol, eps_schwarz=1e-12)
    ctx2.set_tuning(table)
    t2 = ctx2.tuning()
    assert [(t["class"], t["waves_per_group"], t["units_per_task"]) for t in t2] == \
        [(t["class"], t["waves_per_group"], t["units_per_task"]) for t in table]
    _check(ctx2, D, jk_golden, case)


@pytest.mark.parametrize("case", sorted(CASES))
def test_forced_launch_shapes(gpu, jk_golden, case):
    n, seed, basis = CASES[case]
    mol = water_cluster(n, seed, basis)
    D = jk_golden[f"{case}_D"]
    _, ctx = _ctx(mol, eps_schwarz=1e-12)
    classes = [t["class"] for t in ctx.tuning()]
    for wpg, tu, acc in ((8, 8, False), (4, 64, True), (8, 32, True), (4, 16, False)):
        ctx.set_tuning([{"class": c, "waves_per_group": wpg, "units_per_task": tu, "lds_accumulators": acc,
                         "tuned_ms": 0.0} for c in classes])
        _check(ctx, D, jk_golden, case)


def test_tuning_errors(gpu):
    mol = water_cluster(2, 3, "cc-pVDZ")
    _, ctx = _ctx(mol)
    c = ctx.tuning()[0]["class"]
    with pytest.raises(ValueError, match="must be"):
        ctx.set_tuning([{"class": c, "waves_per_group": 6, "units_per_task": 16, "lds_accumulators": True,
                         "tuned_ms": 0.0}])
    with pytest.raises(ValueError, match="must be"):
        ctx.set_tuning([{"class": c, "waves_per_group": 4, "units_per_task": 0, "lds_accumulators": True,
                         "tuned_ms": 0.0}])
    with pytest.raises(ValueError, match="must be"):
        ctx.autotune(np.zeros((3, 3)))


def test_graph_of_mixed_build_survives_retuning(gpu):
    """A mixed build captured under one table replays unchanged after tables
    with fewer and with more row tasks (lists that replaced the captured ones in
    place would hand its kernels other class pairs' units). Replays and eager
    builds differ by the order of their sums: fewer than 1e5 terms below 10 in
    elements below 1e2, 1e-12."""
    from asuka_amd.hf.direct_jk import direct_JK

    torch = gpu
    ao, ctx = _ctx(water_cluster(3, 5, "cc-pVDZ"), tau_mixed=1e-3)
    C = np.linalg.qr(np.random.default_rng(7).standard_normal((ao.nao, 15)))[0]
    D = torch.tensor(2.0 * C @ C.T, device="cuda")
    default = ctx.tuning()

    def units(n):
        return [dict(t, units_per_task=n) for t in default]

    ctx.set_tuning(units(1))  # as many tasks as units
    stats = {}
    ref = direct_JK(ctx, D, mixed_precision=True, stats=stats)
    assert 0 < sum(c["quartets_fp32"] for c in stats["class_counts"]) < stats["direct_jk_evaluated"]
    out = tuple(torch.empty_like(x) for x in ref)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        direct_JK(ctx, D, mixed_precision=True, out=out)
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        direct_JK(ctx, D, mixed_precision=True, out=out)
    for table in (default, units(4), units(1), default):
        ctx.set_tuning(table)
        eager = direct_JK(ctx, D, mixed_precision=True)
        for x in out:
            x.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for x, y, r in zip(out, eager, ref):
            assert float((x - r).abs().max()) < 1e-12 and float((y - r).abs().max()) < 1e-12


def test_autotune_mixed_builds(gpu):
    """Tuning for mixed builds runs each class pair as such a build does (one
    FP64 launch, or the two routed ones) and leaves J and K what they were but
    for the order of the sums (as above, 1e-12); tables that name the same cut
    differently, and a fresh context under the table, likewise."""
    from asuka_amd.hf.direct_jk import direct_JK

    ao, ctx = _ctx(water_cluster(3, 5, "cc-pVDZ"), tau_mixed=1e-3)
    C = np.linalg.qr(np.random.default_rng(7).standard_normal((ao.nao, 15)))[0]
    D = 2.0 * C @ C.T
    ref = direct_JK(ctx, D, mixed_precision=True)
    ref64 = direct_JK(ctx, D, mixed_precision=False)
    assert max(float((x - y).abs().max()) for x, y in zip(ref, ref64)) > 1e-11  # FP32 units among them
    table = ctx.autotune(D, mixed_precision=True, reps=1)
    assert all(t["tuned_ms"] > 0 for t in table)
    _, fresh = _ctx(water_cluster(3, 5, "cc-pVDZ"), tau_mixed=1e-3)
    fresh.set_tuning(table)
    builds = [direct_JK(c, D, mixed_precision=True) for c in (ctx, fresh)]
    for wpg, units in ((4, 1000), (8, 1000), (4, 2), (8, 2)):
        ctx.set_tuning([dict(t, waves_per_group=wpg, units_per_task=units) for t in table])
        builds.append(direct_JK(ctx, D, mixed_precision=True))
    for got in builds:
        assert all(float((x - y).abs().max()) < 1e-12 for x, y in zip(got, ref))
