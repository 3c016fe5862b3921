"""Diffusion samples, which need a step closed by its own launches, between steps that the next one's kernels
close: the tables, records and states of single steps, whether samples fall on every other step or on each tenth."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("every,steps", [(2, 60), (10, 120)])
def test_tables_of_long_chunks(gpu, every, steps, prec):
    s = sg.make_system(regime=2, ux=5, uy=6, n_metal=201, temperature=800.0, geometry="sphere", seed=9,
                       velocities="maxwell", step_equil=0, delta_f=0.0)
    s.params.stepDiffuse, s.params.nValDiffuse, s.params.nBuffDiffuse, s.params.limitDiffuseAv = every, 4, 2, 2
    out = []
    for chunks, graphs in (([1] * steps, True), ([steps], True), ([7, steps - 7], False)):
        with sg.Engine(s.params, precision=prec, rebuild_every=7, use_graphs=graphs) as eng:
            eng.diffusion_enable(8)
            eng.upload(s.r, s.v, s.a)
            eng.set_run_state(0, 1, 0.0)
            recs = [r for n in chunks for r in eng.run(n)]
            count, tables = eng.diffusion_tables(8)
            out.append((recs, count, tables, *eng.download()))
    assert out[0][1] >= 2 and np.abs(out[0][2]).max() > 0
    for got in out[1:]:
        assert got[0] == out[0][0] and got[1] == out[0][1]
        assert all(np.array_equal(x, y) for x, y in zip(got[2:], out[0][2:]))
