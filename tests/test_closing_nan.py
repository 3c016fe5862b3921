"""Steps of a trajectory that has lost atoms to NaN: a NaN takes part in no maximum and no minimum, so the
skin rule and the records are the same whichever launch closes a step, chunk by chunk or step by step.
All atoms lost: v^2 maximum 0 and the box of the padding, as a record of no atoms has.  One lost: the
maximum of the others.  The lists are built before the velocities are lost and the skin rule asks for no
other within these steps.  65 partials (a second chunk of them), and one to five.
vvMax: a product and two sums per atom, 4 u."""
import json

import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu

SIZES = [(21, 24, 13), (5, 6, 201), (4, 4, 0)]


def _system(ux, uy, metal):
    return sg.make_system(regime=2, ux=ux, uy=uy, n_metal=metal, temperature=100.0, geometry="sphere", seed=4,
                          velocities="maxwell", step_equil=0, delta_f=0.0)


def _lose(s, v, lost):
    v = np.array(v, np.float64)
    v[:] = np.nan if lost == "all" else v
    if lost != "all":
        v[int(lost * (s.n - 1))] = np.nan
    return v


def _largest(v):
    vv = (v * v).sum(1)
    return vv[~np.isnan(vv)].max(initial=0.0)


@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("lost", ["all", 0.0, 0.5, 1.0])
@pytest.mark.parametrize("ux,uy,metal", SIZES)
def test_one_system(gpu, ux, uy, metal, lost, prec):
    s = _system(ux, uy, metal)
    text = []
    for chunks, graphs in (([1] * 6, True), ([6], True), ([2, 4], True), ([3, 3], False)):
        with sg.Engine(s.params, precision=prec, use_graphs=graphs) as eng:
            eng.upload(s.r, _lose(s, s.v, lost), s.a)
            eng.bin()
            eng.build_nebr()
            eng.compute_forces()
            eng.set_run_state(0, 0, 0.0)
            recs = [r for n in chunks for r in eng.run(n)]
            v = eng.download()[1]
            box = eng.props()
        text.append(json.dumps(recs))
        assert not any(r["rebuilt"] for r in recs)
        for r in (recs[-1], box):
            assert abs(r["vvMax"] - _largest(v)) <= 4 * 2.0 ** -24 * r["vvMax"]
            assert np.isfinite([r["dispHi"]] + r["bboxMin"] + r["bboxMax"]).all()
            if lost == "all":
                assert r["dispHi"] == 0.0 and r["bboxMin"] == r["bboxMax"] == [0.0] * 3
    assert text[1:] == text[:1] * 3


@pytest.mark.parametrize("sync", [0, 1])
@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("lost", ["all", 0.5, 1.0])
def test_batch(gpu, lost, prec, sync):
    systems = [_system(*size) for size in SIZES]
    text = []
    for chunks in ([1] * 6, [6], [2, 4]):
        with sg.Batch([s.params for s in systems], precision=prec, sync_rebuilds=sync) as b:
            for k, s in enumerate(systems):
                b.upload(k, s.r, s.v, s.a)
                b.set_run_state(k, 0, 1, 0.0)
            b.run(1, records=False)
            for k, s in enumerate(systems):
                r, v, a = b.download(k)
                b.upload(k, r, _lose(s, v, lost), a)
                b.set_run_state(k, 1, 0, 0.0)
            recs = [[] for _ in systems]
            for n in chunks:
                for k, x in enumerate(b.run(n)):
                    recs[k] += x
            for k in range(len(systems)):
                v = b.download(k)[1]
                assert abs(recs[k][-1]["vvMax"] - _largest(v)) <= 4 * 2.0 ** -24 * recs[k][-1]["vvMax"]
        text.append(json.dumps(recs))
    assert text[1:] == text[:1] * 2
