"""A step whose closing (skin rule, record, state) is folded into the next step must leave the records and
the state of the step closed by its own launches, bit for bit.  A run in chunks of one step folds
nothing; longer chunks fold an even number of the steps that nothing else follows."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


def _run(s, prec, chunks, rdf_every, graphs=True, msd=False):
    with sg.Engine(s.params, precision=prec, rebuild_every=7, use_graphs=graphs) as eng:
        if msd:
            eng.diffusion_enable(4)
        eng.upload(s.r, s.v, s.a)
        eng.set_run_state(0, 1, 0.0)
        recs = []
        for n in chunks:
            recs += eng.run(n, rdf_every=rdf_every)
        out = list(eng.download())
        if rdf_every:
            out.append(eng.rdf())
        return recs, out


# nMol: 1,161 atoms have one chunk of partials, 32,960 have 3, 130,880 have 11 (reduced by the closing workgroup);
# 268,192 have more than the 1,024 partials it takes (k_reduce1 first)
@pytest.mark.parametrize("ux,uy,metal,prec,rdf_every,steps", [
    (5, 6, 201, "mixed", 0, 31), (5, 6, 201, "fp32", 5, 30), (30, 34, 320, "mixed", 9, 29), (64, 62, 3904, "fp32", 0, 12),
    (84, 98, 4768, "mixed", 0, 9), (84, 98, 4768, "fp32", 4, 8), (6, 5, 0, "mixed", 0, 12),
])
def test_folded_closing_equals_single_steps(gpu, ux, uy, metal, prec, rdf_every, steps):
    s = sg.make_system(regime=2, ux=ux, uy=uy, n_metal=metal, temperature=900.0, geometry="sphere", seed=9,
                       velocities="maxwell", tauPs=0.1, step_equil=0, delta_f=0.0)
    print(f"[closing] {s.n} atoms {prec}", flush=True)
    want_recs, want = _run(s, prec, [1] * steps, rdf_every)
    assert sum(r["rebuilt"] for r in want_recs) >= 2
    for chunks, graphs in (([steps], True), ([steps // 2, steps - steps // 2], True), ([3, steps - 3], False)):
        recs, got = _run(s, prec, chunks, rdf_every, graphs)
        assert recs == want_recs, chunks
        for a, b in zip(got, want):
            assert np.array_equal(a, b), chunks


def test_folded_closing_reports_a_capacity(gpu):
    """A flag raised inside a folded run of steps reaches the host: cells of 8 overflow at the second
    rebuild's binning or at the first, whichever chunk length holds them."""
    s = sg.config_system("small", "reference")
    with sg.Engine(s.params, precision="mixed", cell_capacity=8, rebuild_every=2) as eng:
        eng.upload(s.r, s.v, s.a)
        eng.set_run_state(0, 1, 0.0)
        with pytest.raises(RuntimeError, match="cell capacity"):
            eng.run(12)
