"""A shear that plain precision cannot hold exactly, with no increment per step: the reference adds the
increment 0 in its own precision while the cluster is slow, so the first record after the cooling phase
holds the rounded shear, whichever launch closes that step.  Mixed precision holds it exactly."""
import ctypes

import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cool", [0, 3])
@pytest.mark.parametrize("prec,want", [("fp32", float(np.float32(0.1))), ("mixed", 0.1)])
def test_rounded_at_its_step(gpu, prec, want, cool):
    s = sg.make_system(regime=2, ux=7, uy=5, n_metal=55, temperature=300.0, geometry="sphere", seed=3,
                       velocities="maxwell", step_equil=0, step_cool=cool, delta_f=0.0)
    s.v[:55, 0] -= s.v[:55, 0].mean() + 0.5  # slow: the rule applies
    for chunks in ([1] * 7, [7], [3, 4], [2, 5]):
        with sg.Engine(s.params, precision=prec) as eng:
            eng.upload(s.r, s.v, s.a)
            eng.set_run_state(0, 1, 0.0)
            assert eng.lib.sgk_set_shear_state(eng.h, ctypes.c_double(0.1), ctypes.c_double(0.0), ctypes.c_double(0.0)) == 0
            recs = [r for n in chunks for r in eng.run(n)]
        assert [r["shear"] for r in recs] == [0.1] * cool + [want] * (7 - cool), chunks
