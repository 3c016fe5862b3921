"""The sums of a step's record, reduced by the force pass, against sums over the state the step left,
for every number of lanes per metal atom, workgroups only partly filled, and systems without metal or
with a single metal atom.  A record's sums are those of the downloaded state when no thermostat
follows the step.  Bound: sums of n terms in FP64 (mixed) or FP32 (plain), any order:
n u sum|x|, with u the unit roundoff of the accumulation, doubled for the terms' own products."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("ux,uy,metal", [(3, 2, 13), (5, 6, 201), (5, 5, 1), (4, 4, 0), (9, 11, 561)])
def test_record_sums_equal_the_states(gpu, ux, uy, metal, lanes, prec):
    s = sg.make_system(regime=2, ux=ux, uy=uy, n_metal=metal, temperature=700.0, geometry="sphere", seed=11)
    p = s.params
    with sg.Engine(p, precision=prec, metal_lanes=lanes) as eng:
        eng.upload(s.r, s.v, s.a)
        eng.set_run_state(0, 1, 0.0)
        rec = eng.run(3)[-1]
        r, v, _ = eng.download()
    m = np.ones(s.n)
    m[:metal] = p.massMe
    c = v[:metal, 0].mean() if metal else 0.0
    w = v.copy()
    w[:metal, 0] -= c
    u = 2.0 * s.n * (2.0 ** -53 if prec == "mixed" else 2.0 ** -24)
    vm = v.copy()
    vm[:metal, 0] *= p.massMe
    for name, terms in (("uSum", r[:, 3]), ("vvSum", m * (w * w).sum(1))):
        assert abs(rec[name] - terms.sum()) <= u * (np.abs(terms).sum() + (m * (v * v).sum(1)).sum() * (name == "vvSum")), name
    for d in range(3):
        assert abs(rec["vSum"][d] - vm[:, d].sum()) <= u * np.abs(vm[:, d]).sum()
        # positions of the record: before the next step's drift, which the last step of a run does not make
        assert abs(rec["comSum"][d] - r[:metal, d].sum()) <= u * np.abs(r[:metal, d]).sum()
        assert abs(rec["cmVelSum"][d] - v[:metal, d].sum()) <= u * np.abs(v[:metal, d]).sum()
        lo, hi = (min(0.0, r[:metal, d].min()), max(0.0, r[:metal, d].max())) if metal else (0.0, 0.0)
        assert rec["bboxMin"][d] == lo and rec["bboxMax"][d] == hi
    assert abs(rec["vvMax"] - (v * v).sum(1).max()) <= 4 * u / s.n * rec["vvMax"]
