"""Batches of more replicas than one pass of a workgroup looks at: one, 257 (a second pass for the synchronised
rebuild), the 1,024 whose synchronised steps are closed by the next one's kernels, and one more.  Long
chunks leave the records and states of single steps, and with synchronised rebuilds the whole batch
rebuilds when the one hot replica, first, in the middle or last, asks for it."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sync", [0, 1])
@pytest.mark.parametrize("prec,nrep,hot", [("fp32", 257, 256), ("mixed", 257, 0), ("fp32", 1024, 700), ("fp32", 1025, 1024)])
def test_long_chunks_equal_single_steps(gpu, nrep, hot, prec, sync):
    make = lambda t: sg.make_system(regime=2, ux=3, uy=2, n_metal=13, temperature=t, geometry="sphere", seed=5,
                                    velocities="maxwell", step_equil=0, delta_f=0.0)
    cold, warm = make(10.0), make(1500.0)
    systems = [warm if k == hot else cold for k in range(nrep)]

    def run(chunks):
        with sg.Batch([s.params for s in systems], precision=prec, sync_rebuilds=sync) as b:
            for k, s in enumerate(systems):
                b.upload(k, s.r, s.v, s.a)
                b.set_run_state(k, 0, 1, 0.0)
            recs = [[] for _ in systems]
            for n in chunks:
                for k, x in enumerate(b.run(n)):
                    recs[k] += x
            return recs, [b.download(k) for k in range(0, nrep, 64)] + [b.download(hot), b.download(nrep - 1)]

    want_recs, want = run([1] * 24)
    asked = [r["rebuilt"] for r in want_recs[hot]]
    other = [r["rebuilt"] for r in want_recs[hot - 1 if hot else 1]]
    assert sum(asked) >= 3 and (other == asked if sync else sum(other) < sum(asked))
    recs, got = run([24])
    assert recs == want_recs
    assert all(np.array_equal(x, y) for g, w in zip(got, want) for x, y in zip(g, w))
