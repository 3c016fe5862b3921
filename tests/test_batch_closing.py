"""Batched steps closed by the next step's kernels leave the records and states of steps closed by their own
launch, bit for bit, with and without synchronised rebuilds: a run in chunks of one step folds nothing,
longer chunks an even number of steps.  One, few and 70 replicas (more than a wave), one and four lanes per
carbon, a replica with more than 1,024 partials (nothing is folded then)."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu

SMALL = [(4, 4, 13), (5, 6, 201), (4, 5, 0)]
SETS = {
    "one": SMALL[1:2],
    "few": SMALL,
    "many": [SMALL[k % 3] for k in range(70)],
    "one lane per carbon": SMALL + [(40, 42, 55)],
    "not folded": [SMALL[0], (88, 93, 13)],
}


@pytest.mark.parametrize("sync", [0, 1])
@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("name", list(SETS))
def test_folded_batch_equals_single_steps(gpu, name, prec, sync):
    systems = [sg.make_system(regime=2, ux=ux, uy=uy, n_metal=m, temperature=800.0 + 40.0 * (k % 9), geometry="sphere",
                              seed=2 + k, velocities="maxwell", tauPs=0.1, step_equil=0, delta_f=0.0)
               for k, (ux, uy, m) in enumerate(SETS[name])]
    print(f"[batch closing] {name} {prec} sync {sync}", flush=True)

    def run(chunks, rdf_every=0):
        with sg.Batch([s.params for s in systems], precision=prec, rebuild_every=0, sync_rebuilds=sync) as b:
            for k, s in enumerate(systems):
                b.upload(k, s.r, s.v, s.a)
                b.set_run_state(k, 0, 1, 0.0)
            recs = [[] for _ in systems]
            for n in chunks:
                for k, x in enumerate(b.run(n, rdf_every=rdf_every)):
                    recs[k] += x
            return recs, [b.download(k) for k in range(len(systems))]

    want_recs, want = run([1] * 40)
    assert all(sum(r["rebuilt"] for r in x) >= 2 for x in want_recs)
    for chunks, rdf_every in (([40], 0), ([40], 5), ([9, 31], 0)):
        recs, got = run(chunks, rdf_every)
        for k in range(len(systems)):
            assert recs[k] == want_recs[k], (chunks, k)
            assert all(np.array_equal(x, y) for x, y in zip(got[k], want[k])), (chunks, k)
