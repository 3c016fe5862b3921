"""A step that only a shear or a deposition follows, closed by the next step's first kernel, must leave the
records and the state of the step closed by its own launches, bit for bit.  A run in chunks of one step
folds nothing; longer chunks fold an even number of steps."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


def _run(s, prec, chunks, graphs=True, rdf_every=0):
    with sg.Engine(s.params, precision=prec, rebuild_every=7, use_graphs=graphs) as eng:
        eng.upload(s.r, s.v, s.a)
        eng.set_run_state(0, 1, 0.0)
        if s.params.iRegime == 1:
            assert eng.lib.sgk_set_deposited(eng.h, 0) == 0
        recs = []
        for n in chunks:
            recs += eng.run(n, rdf_every=rdf_every)
        return recs, list(eng.download())


def _same(s, prec, steps, rdf_every=0):
    want_recs, want = _run(s, prec, [1] * steps, True, rdf_every)
    assert sum(r["rebuilt"] for r in want_recs) >= 2
    for chunks, graphs in (([steps], True), ([steps // 2, steps - steps // 2], True), ([3, steps - 3], False)):
        recs, got = _run(s, prec, chunks, graphs, rdf_every)
        assert recs == want_recs, chunks
        for a, b in zip(got, want):
            assert np.array_equal(a, b), chunks
    return want_recs


# 13 to 72 partials, and 1,031 and 1,043: beyond the 1,024 that k_lf1_next takes
@pytest.mark.parametrize("ux,uy,metal,prec,rdf_every", [
    (7, 5, 55, "fp32", 0), (7, 5, 55, "mixed", 5), (8, 8, 13, "mixed", 0), (20, 21, 13, "fp32", 0), (22, 23, 13, "mixed", 0),
    (88, 93, 13, "fp32", 0),
])
def test_sheared_steps(gpu, ux, uy, metal, prec, rdf_every):
    s = sg.make_system(regime=2, ux=ux, uy=uy, n_metal=metal, temperature=600.0, geometry="sphere", seed=3,
                       velocities="maxwell", step_equil=0, step_cool=4, delta_f=1e-4)
    s.v[:metal, 0] -= s.v[:metal, 0].mean() + 0.5  # the increment grows while the cluster is slow
    recs = _same(s, prec, 27, rdf_every)
    assert recs[-1]["shear"] > 0 and any(r["shearCount"] > 0 for r in recs)


@pytest.mark.parametrize("ux,uy,metal,prec,deposit", [
    (6, 7, 40, "fp32", 5), (6, 7, 40, "mixed", 3), (11, 13, 307, "fp32", 6), (23, 23, 30, "mixed", 5),
    (90, 92, 30, "fp32", 5),
])
def test_deposition_steps(gpu, ux, uy, metal, prec, deposit):
    s = sg.make_system(regime=1, ux=ux, uy=uy, n_metal=metal, material=2, temperature=600.0, seed=3, velocities="maxwell", depos_energy=2.0,
                       step_equil=2, step_deposit=deposit, n_to_deposit=3)
    recs = _same(s, prec, 27)
    assert recs[-1]["nMolDeposited"] > 3
