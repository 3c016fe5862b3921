"""Reference-stencil RDF at the sizes where its split over lanes and workgroups changes: eight atoms at
a time (27 lanes each), one group a workgroup up to 4,096 metal atoms, more groups above.  Counts are
integers: equal to the oracle's, bin for bin, on a single system and in a batch."""
import numpy as np
import pytest

import oracle
import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


def _system(metal, seed):
    side = 6 if metal < 700 else 24
    s = sg.make_system(regime=2, ux=side, uy=side, n_metal=metal, temperature=600.0, geometry="sphere", seed=seed,
                       rangeRdfAngstrom=5.0)
    r = s.r.astype(np.float64)
    r[:, :3] += 0.03 * np.random.default_rng(metal).standard_normal((s.n, 3))
    return s, r


def _expected(s, r):
    o = oracle.Oracle(s.params, "f64")
    err, cell_of, cnt, slots = o.bin(r)
    assert err == 0
    return o.rdf(r, cell_of, cnt, slots)[0]


@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("metal", [1, 7, 8, 9, 201, 4096, 4111])
def test_rdf_equals_the_oracle(gpu, metal, prec):
    s, r = _system(metal, 2)
    if prec == "fp32":
        r = r.astype(np.float32).astype(np.float64)
    print(f"[rdf] {metal} metal atoms, {prec}", flush=True)
    with sg.Engine(s.params, precision=prec) as eng:
        eng.upload(r)
        eng.bin()
        eng.rdf_clear()
        eng.rdf_accumulate()
        assert np.array_equal(eng.rdf(), _expected(s, r))


def test_rdf_of_a_batch_equals_each_run_alone(gpu):
    """Replicas whose metal atoms fill a group, leave one over, or are none at all."""
    systems = [_system(m, 3)[0] for m in (8, 9, 0, 201, 33)]
    with sg.Batch([s.params for s in systems], precision="mixed", rebuild_every=2) as b:
        for k, s in enumerate(systems):
            b.upload(k, s.r, s.v, s.a)
            b.set_run_state(k, 0, 1, 0.0)
        b.run(4, rdf_every=2, records=False)
        got = [b.rdf(k) for k in range(len(systems))]
    for k, s in enumerate(systems):
        with sg.Engine(s.params, precision="mixed", rebuild_every=2, xcd_map=0) as eng:
            eng.upload(s.r, s.v, s.a)
            eng.set_run_state(0, 1, 0.0)
            eng.run(4, rdf_every=2, records=False)
            assert np.array_equal(eng.rdf(), got[k]), k
