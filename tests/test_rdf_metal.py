"""Reference-stencil RDF where a workgroup takes more than one group of eight atoms: from 8,193 metal atoms on, in
turn with the others, to the last, ragged group; in a batch by the metal atoms of all replicas.  Counts are integers:
equal to the oracle's, bin for bin."""
import numpy as np
import pytest

import oracle
import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


def _system(metal):
    s = sg.make_system(regime=2, ux=24, uy=24, n_metal=metal, temperature=600.0, geometry="sphere", seed=2,
                       rangeRdfAngstrom=5.0)
    r = s.r.astype(np.float64)
    r[:, :3] += 0.03 * np.random.default_rng(metal).standard_normal((s.n, 3))
    return s, r


def _expected(s, r):
    o = oracle.Oracle(s.params, "f64")
    err, cell_of, cnt, slots = o.bin(r)
    assert err == 0
    return o.rdf(r, cell_of, cnt, slots)[0]


@pytest.mark.parametrize("metal", [8192, 8193, 8200, 8201, 16385, 40007])
def test_rdf_equals_the_oracle(gpu, metal):
    s, r = _system(metal)
    print(f"[rdf] {metal} metal atoms", flush=True)
    with sg.Engine(s.params, precision="mixed") as eng:
        eng.upload(r)
        eng.bin()
        eng.rdf_clear()
        eng.rdf_accumulate()
        assert np.array_equal(eng.rdf(), _expected(s, r))


def test_rdf_of_a_batch_equals_each_run_alone(gpu):
    """12,321 metal atoms in all: two groups a workgroup, one workgroup each for the smallest."""
    systems = [_system(m)[0] for m in (8201, 4111, 9)]
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
