"""The sums that close a step, where the reduction of the force pass's partial sums changes: rows of 16
partials, chunks of 64, more rows than groups of threads, and 1,024 against 1,025 partials (the latter
by way of chunk totals).  One partial per 256 carbons, one for the 13 metal atoms.  Bound: a sum of n
terms in any order, n u sum|x|, doubled for the terms' own products; a replica
closes as the system alone (atoms in launch order; an unset count of deposited atoms differs outside regime 1)."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu

# partials: 15, 16, 17, 64, 65, 193, 1,024, 1,025
SIZES = [(8, 14), (10, 12), (8, 16), (21, 24), (16, 32), (32, 48), (88, 93), (64, 128)]


def _system(ux, uy):
    return sg.make_system(regime=2, ux=ux, uy=uy, n_metal=13, temperature=700.0, geometry="sphere", seed=11,
                          velocities="maxwell")


@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("ux,uy", SIZES)
def test_record_sums(gpu, ux, uy, prec):
    s = _system(ux, uy)
    p = s.params
    with sg.Engine(p, precision=prec, metal_lanes=16) as eng:
        eng.upload(s.r, s.v, s.a)
        eng.set_run_state(0, 1, 0.0)
        rec = eng.run(2)[-1]
        r, v, _ = eng.download()
    m = np.ones(s.n)
    m[:13] = p.massMe
    w, vm = v.copy(), v.copy()
    w[:13, 0] -= v[:13, 0].mean()
    vm[:13, 0] *= p.massMe
    u = 2.0 * s.n * (2.0 ** -53 if prec == "mixed" else 2.0 ** -24)
    assert abs(rec["uSum"] - r[:, 3].sum()) <= u * np.abs(r[:, 3]).sum()
    assert abs(rec["vvSum"] - (m * (w * w).sum(1)).sum()) <= 2 * u * (m * (v * v).sum(1)).sum()
    for d in range(3):
        assert abs(rec["vSum"][d] - vm[:, d].sum()) <= u * np.abs(vm[:, d]).sum()
        assert abs(rec["comSum"][d] - r[:13, d].sum()) <= u * np.abs(r[:13, d]).sum()
        assert abs(rec["cmVelSum"][d] - v[:13, d].sum()) <= u * np.abs(v[:13, d]).sum()
        assert rec["bboxMin"][d] == min(0.0, r[:13, d].min()) and rec["bboxMax"][d] == max(0.0, r[:13, d].max())
    assert abs(rec["vvMax"] - (v * v).sum(1).max()) <= 4 * u / s.n * rec["vvMax"]


@pytest.mark.parametrize("prec", ["mixed", "fp32"])
def test_replicas_close_as_alone(gpu, prec):
    systems = [_system(*SIZES[k]) for k in (2, 4, 7)]
    with sg.Batch([s.params for s in systems], precision=prec, metal_lanes=16, xcd_map=0) as b:
        for k, s in enumerate(systems):
            b.upload(k, s.r, s.v, s.a)
            b.set_run_state(k, 0, 1, 0.0)
        got = b.run(4)
    for k, s in enumerate(systems):
        with sg.Engine(s.params, precision=prec, metal_lanes=16, xcd_map=0) as eng:
            eng.upload(s.r, s.v, s.a)
            eng.set_run_state(0, 1, 0.0)
            alone = eng.run(4)
        for x, y in zip(got[k], alone):
            assert {q: v for q, v in x.items() if q != "nMolDeposited"} == {q: v for q, v in y.items() if q != "nMolDeposited"}
