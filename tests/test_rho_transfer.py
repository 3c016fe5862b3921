"""The densities as they come back through the pinned stage, which serves the other transfers too, against
the FP64 oracle, atom by atom.  Bound: the mixed form's densities differ from the oracle's by up to 1e-6
of the largest."""
import ctypes

import numpy as np
import pytest

import oracle
import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metal", [1, 201, 32767, 32768])
def test_every_density(gpu, metal):
    s = sg.make_system(regime=2, ux=24, uy=26, n_metal=metal, temperature=300.0, geometry="sphere", seed=3)
    r = s.r.astype(np.float64)
    r[:metal, :3] += 0.03 * np.random.default_rng(1).standard_normal((metal, 3))
    o = oracle.Oracle(s.params, "f64")
    err, nn, nbl = o.neighbour_list(r)
    assert err == 0
    want = o.rho(r, nn, nbl)[:metal]
    with sg.Engine(s.params, precision="mixed") as eng:
        eng.upload(r)
        eng.bin()
        eng.build_nebr()
        eng.compute_forces()
        eng.download()
        out = np.full(metal + 2, -7.0)
        assert eng.lib.sgk_get_rho(eng.h, out[1:].ctypes.data_as(ctypes.c_void_p)) == 0
    assert out[0] == out[-1] == -7.0
    assert np.abs(out[1:-1] - want).max() <= 1e-6 * max(np.abs(want).max(), 1e-30)
