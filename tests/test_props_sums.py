"""The evaluation of the current state (one partial sum per 256 atoms) against sums over the state itself: one
partial, a wave of them, 256 and 257 (a second one per thread), a thousand.  Bound: a sum of n terms in any order,
n u sum|x|, doubled for the terms' own products."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["mixed", "fp32"])
# partials: 1, 5, 64, 65, 256, 257, 1,024
@pytest.mark.parametrize("ux,uy,metal", [(2, 2, 13), (5, 6, 201), (15, 34, 13), (16, 32, 13), (15, 136, 13), (32, 64, 13),
                                         (88, 93, 13)])
def test_against_the_state(gpu, ux, uy, metal, prec):
    s = sg.make_system(regime=2, ux=ux, uy=uy, n_metal=metal, temperature=500.0, geometry="sphere", seed=7,
                       velocities="maxwell")
    with sg.Engine(s.params, precision=prec) as eng:
        eng.upload(s.r, s.v, s.a)
        eng.set_run_state(0, 1, 0.0)
        eng.run(1)
        rec = eng.props()
        r, v, _ = eng.download()
    m = np.ones(s.n)
    m[:metal] = s.params.massMe
    w, vm = v.copy(), v.copy()
    w[:metal, 0] -= v[:metal, 0].mean()
    vm[:metal, 0] *= s.params.massMe
    u = 2.0 * s.n * (2.0 ** -53 if prec == "mixed" else 2.0 ** -24)
    assert abs(rec["uSum"] - r[:, 3].sum()) <= u * np.abs(r[:, 3]).sum()
    assert abs(rec["vvSum"] - (m * (w * w).sum(1)).sum()) <= 2 * u * (m * (v * v).sum(1)).sum()
    for d in range(3):
        assert abs(rec["vSum"][d] - vm[:, d].sum()) <= u * np.abs(vm[:, d]).sum()
        assert abs(rec["comSum"][d] - r[:metal, d].sum()) <= u * np.abs(r[:metal, d]).sum()
        assert abs(rec["cmVelSum"][d] - v[:metal, d].sum()) <= u * np.abs(v[:metal, d]).sum()
        assert rec["bboxMin"][d] == min(0.0, r[:metal, d].min()) and rec["bboxMax"][d] == max(0.0, r[:metal, d].max())
    assert abs(rec["vvMax"] - (v * v).sum(1).max()) <= 4 * u / s.n * rec["vvMax"]
