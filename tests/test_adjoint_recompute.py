"""The recomputed segments of the adjoint: whatever the segment length - one step, an odd or even number, a
remainder, the whole window, with thermostat steps and rebuilds inside - the recomputed end states are those of
the forward (no mismatches) and the gradients agree.  The sweep's sums are made by FP64 atomics in any order:
n terms of u = 1.1e-16 each with cancellation to ~1e-3 of their sum stay below 1e-8 of the largest component."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ux,uy,metal,tau", [(6, 6, 55, 0.1), (8, 7, 147, 0.0)])
def test_gradients_do_not_depend_on_the_segments(gpu, ux, uy, metal, tau):
    kw = dict(tauPs=tau) if tau else {}
    s = sg.make_system(regime=2, ux=ux, uy=uy, n_metal=metal, temperature=600.0, geometry="icosahedron", gap=3.0, seed=4,
                       velocities="maxwell", step_equil=0, delta_f=0.0, **kw)
    steps, want = 23, None
    for every in (23, 1, 2, 5, 8):
        with sg.Engine(s.params, precision="mixed", rebuild_every=6) as eng:
            eng.upload(s.r, s.v, s.a)
            eng.set_run_state(0, 1, 0.0)
            eng.adjoint_forward(steps, every)
            end = eng.download()
            g, dr0, dv0 = eng.adjoint_backward([1.0, 0.25], initial_state=True)
            assert eng.adjoint_info()["mismatches"] == 0, every
            assert all(np.array_equal(x, y) for x, y in zip(end, eng.download())), every  # left where the forward ended
        if want is None:
            want = (g, dr0, dv0)
        for x, y in zip((g, dr0, dv0), want):
            assert np.abs(x - y).max() <= 1e-8 * np.abs(y).max(), every
