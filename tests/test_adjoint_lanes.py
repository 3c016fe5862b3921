"""The adjoint's split over lanes: adhesion energy by the lanes of a metal atom, the carbon transpose by
four lanes per atom, and the adhesion record of steps whose closing is folded into the next.

Tolerances: both sides evaluate the same expressions in FP64, so they differ by summation order: n terms,
n u sum|x| <= 1e-12 of the energy for the <= 1e4 pairs here (all of one sign near the well) and 1e-9 of the
summed magnitudes for the transpose, as the force-VJP parity test."""
import numpy as np
import pytest

import oracle
import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


def _system(ux, uy, metal, seed=4):
    s = sg.make_system(regime=2, ux=ux, uy=uy, n_metal=metal, temperature=600.0, geometry="sphere", gap=2.2, seed=seed)
    r = s.r.astype(np.float64)
    r[:, :3] += 0.02 * np.random.default_rng(metal).standard_normal((s.n, 3))
    return s, r


@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("ux,uy,metal", [(3, 3, 0), (3, 2, 1), (4, 4, 16), (4, 4, 17), (6, 7, 257)])
def test_adhesion_energy_by_lanes(gpu, ux, uy, metal, lanes):
    s, r = _system(ux, uy, metal)
    o = oracle.Oracle(s.params, "f64")
    err, nn, nbl = o.neighbour_list(r)
    assert err == 0
    with sg.Engine(s.params, precision="mixed", metal_lanes=lanes) as eng:
        eng.upload(r)
        eng.bin()
        eng.build_nebr()
        e = eng.adhesion_energy()
    want = o.adhesion(r, nn, nbl)
    assert (want != 0.0) == (metal > 0)
    assert abs(e - want) <= 1e-12 * abs(want)


@pytest.mark.parametrize("metal", [0, 31])
def test_force_vjp_with_broken_bonds(gpu, metal):
    """Carbons with 0 to 2 bonds left, beside whole ones: some are lifted out of the sheet.  (Pushed
    within it they would bring the reference's neighbour-angle cosine, which divides by |e|^2, past 1,
    where the force law has no value.)"""
    s, r = _system(4, 3, metal)
    rng = np.random.default_rng(8)
    away = s.n_metal + rng.choice(s.n - s.n_metal, 25, replace=False)
    r[away, 2] -= 1.3
    o = oracle.Oracle(s.params, "f64")
    err, nn, nbl = o.neighbour_list(r)
    assert err == 0
    abar = rng.standard_normal((s.n, 3))
    with sg.Engine(s.params, precision="mixed") as eng:
        eng.upload(r)
        eng.bin()
        eng.build_nebr()
        rbar, pbar = eng.force_vjp(abar, 0.3)
    dirs = rng.standard_normal((oracle.ND, s.n, 3))
    _, dacc, _, dadh = o.tangent_forces(r, nn, nbl, rdir=dirs)
    for k in range(oracle.ND):
        want = np.sum(abar * dacc[k]) + 0.3 * dadh[k]
        got = np.sum(rbar * dirs[k])
        assert abs(got - want) <= 1e-9 * max(np.abs(abar * dacc[k]).sum(), np.abs(rbar * dirs[k]).sum())
    if metal:
        _, dacc, _, dadh = o.tangent_forces(r, nn, nbl, pdir=np.eye(4))
        want = np.einsum("nx,knx->k", abar, dacc) + 0.3 * dadh
        assert np.allclose(pbar, want, rtol=1e-9, atol=1e-12 * np.abs(want).max())


def test_adhesion_record_of_folded_steps(gpu):
    """Segments of one step fold nothing; longer ones fold most steps: same observables, bit for bit."""
    s, r = _system(5, 6, 147)
    out = []
    for every in (1, 2, 9, 30):
        with sg.Engine(s.params, precision="mixed", rebuild_every=6) as eng:
            eng.upload(r, s.v.astype(np.float64))
            o = eng.adjoint_forward(30, every, records=True)
            out.append((o["adhesion"], o["height"], o["records"]))
    assert all(x == out[0] for x in out[1:])
