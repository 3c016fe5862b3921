"""Batches with a replica of more than 1,024 partials (1,035 carbon workgroups and the metal's): no step is
closed by the next one's kernels, fused drifts go on.  Long chunks leave the records and states of
single steps, bit for bit; and a replica of exactly 1,024, which is folded, beside it in size."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu

SETS = {"1,036 partials": [(4, 4, 13), (92, 90, 13)], "1,024 partials": [(88, 93, 13)], "1,025 partials": [(64, 128, 13)]}


@pytest.mark.parametrize("sync", [0, 1])
@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("name", list(SETS))
def test_long_chunks_equal_single_steps(gpu, name, prec, sync):
    systems = [sg.make_system(regime=2, ux=ux, uy=uy, n_metal=m, temperature=900.0, geometry="sphere", seed=2 + k,
                              velocities="maxwell", step_equil=0, delta_f=0.0) for k, (ux, uy, m) in enumerate(SETS[name])]
    print(f"[batch unfolded] {name} {prec} sync {sync}", flush=True)

    def run(chunks):
        with sg.Batch([s.params for s in systems], precision=prec, sync_rebuilds=sync) as b:
            for k, s in enumerate(systems):
                b.upload(k, s.r, s.v, s.a)
                b.set_run_state(k, 0, 1, 0.0)
            recs = [[] for _ in systems]
            for n in chunks:
                for k, x in enumerate(b.run(n)):
                    recs[k] += x
            return recs, [b.download(k) for k in range(len(systems))]

    want_recs, want = run([1] * 30)
    assert all(sum(r["rebuilt"] for r in x) >= 2 for x in want_recs)
    for chunks in ([30], [9, 21]):
        recs, got = run(chunks)
        assert recs == want_recs, chunks
        assert all(np.array_equal(x, y) for g, w in zip(got, want) for x, y in zip(g, w)), chunks
