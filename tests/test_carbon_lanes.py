"""Four lanes per carbon (small systems) against one lane per carbon (batches of many carbons): the same
systems alone and in a batch that a large replica fills give the same bits, per-atom results and record
sums alike.  Carbon counts around a wave's 16 and a workgroup's 64 carbons per launch form, sheets whose
carbons have under three bonds at the edge, long and empty LJ lists, no metal at all."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu

CASES = [  # ux, uy, metal, temperature
    (3, 2, 13, 300.0),    # 192 carbons: 3 workgroups of 64
    (5, 5, 1, 900.0),     # 800: the last workgroup half full
    (4, 4, 0, 700.0),     # no metal
    (5, 6, 201, 1200.0),  # long lists under the cluster
    (9, 11, 561, 600.0),
]


@pytest.mark.parametrize("prec,fp64", [("mixed", 1), ("mixed", 0), ("fp32", 0)])
def test_four_lanes_equal_one(gpu, prec, fp64):
    systems = [sg.make_system(regime=2, ux=ux, uy=uy, n_metal=m, temperature=t, geometry="sphere", seed=5,
                              velocities="maxwell", delta_f=0.0) for ux, uy, m, t in CASES]
    # 65,536 carbons: with it in the batch, every replica takes one lane
    filler = sg.make_system(regime=2, ux=64, uy=32, n_metal=13, temperature=300.0, geometry="sphere", seed=5, delta_f=0.0)
    kw = dict(precision=prec, rebuild_every=5, metal_lanes=8, xcd_map=0, pair_fp64=fp64)
    with sg.Batch([s.params for s in systems + [filler]], **kw) as b:
        for k, s in enumerate(systems + [filler]):
            b.upload(k, s.r, s.v, s.a)
            b.set_run_state(k, 0, 1, 0.0)
        recs = b.run(12)
        states = [b.download(k) for k in range(len(systems))]
    for k, s in enumerate(systems):
        with sg.Engine(s.params, **kw) as eng:
            eng.upload(s.r, s.v, s.a)
            eng.set_run_state(0, 1, 0.0)
            alone = eng.run(12)
            for x, y in zip(eng.download(), states[k]):
                assert np.array_equal(x, y), CASES[k]
        for x, y in zip(recs[k], alone):
            assert {q: v for q, v in x.items() if q != "nMolDeposited"} == {q: v for q, v in y.items() if q != "nMolDeposited"}
