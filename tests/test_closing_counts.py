"""The sums that close a step at exactly the numbers of partials where their reduction changes: rows of 16, chunks
of 64, and the 1,024 that one workgroup takes directly against 1,025 by way of chunk totals.  Without XCD ranges
the metal workgroups are not padded, so 13 atoms at 16 lanes are one partial and a sheet of 256 k carbons
the others; by default they are padded to eight with identities.  Bounds: a sum of n terms in any order, n u sum|x|, doubled for the
terms' own products."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu

# carbon workgroups: 15, 16, 63, 64, 127, 1,016, 1,023, 1,024
SHEETS = [(8, 15), (8, 16), (18, 28), (16, 32), (8, 127), (64, 127), (88, 93), (64, 128)]


@pytest.mark.parametrize("xcd_map", [0, 2])
@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("ux,uy", SHEETS)
def test_record_sums(gpu, ux, uy, prec, xcd_map):
    s = sg.make_system(regime=2, ux=ux, uy=uy, n_metal=13, temperature=700.0, geometry="sphere", seed=11,
                       velocities="maxwell")
    p = s.params
    assert (s.n - 13 + 255) // 256 == {120: 15, 128: 16, 504: 63, 512: 64, 1016: 127, 8128: 1016, 8184: 1023, 8192: 1024}[ux * uy]
    with sg.Engine(p, precision=prec, metal_lanes=16, xcd_map=xcd_map) as eng:
        eng.upload(s.r, s.v, s.a)
        eng.set_run_state(0, 1, 0.0)
        rec = eng.run(3)[-1]
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
@pytest.mark.parametrize("ux,uy", [(18, 28), (16, 32), (88, 93)])
def test_folded_record_sums(gpu, ux, uy, prec):
    """The record of a step in the middle of a chunk, against the state a run of that many steps leaves."""
    s = sg.make_system(regime=2, ux=ux, uy=uy, n_metal=13, temperature=700.0, geometry="sphere", seed=12,
                       velocities="maxwell")
    out = []
    for n in (3, 7):
        with sg.Engine(s.params, precision=prec, metal_lanes=16, xcd_map=0) as eng:
            eng.upload(s.r, s.v, s.a)
            eng.set_run_state(0, 1, 0.0)
            out.append((eng.run(n)[2], eng.download()))
    rec, (r, v, _) = out[1][0], out[0][1]
    u = 2.0 * s.n * (2.0 ** -53 if prec == "mixed" else 2.0 ** -24)
    assert abs(rec["uSum"] - r[:, 3].sum()) <= u * np.abs(r[:, 3]).sum()
    vm = v.copy()
    vm[:13, 0] *= s.params.massMe
    for d in range(3):
        assert abs(rec["vSum"][d] - vm[:, d].sum()) <= u * np.abs(vm[:, d]).sum()
    assert abs(rec["vvMax"] - (v * v).sum(1).max()) <= 4 * u / s.n * rec["vvMax"]
