"""The list build where much metal takes it from nine lanes per atom to four: bulk metal of up to 28,672 atoms,
clusters of up to 131,072 beside carbons.  Both sides of each line equal the per-atom scheme (nl_scheme 0), which the
parity tests tie to the oracle, entry for entry; and so do replicas of bulk metal that pass the line together,
their trajectories those of the replicas alone."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


def _bulk(nx, ny, nz):
    return sg.make_system(regime=0, material=3, ux=nx, uy=ny, uz=nz, temperature=300.0, geometry="reference", seed=3)


def _lists(s, r, scheme, cap):
    with sg.Engine(s.params, precision="mixed", nl_scheme=scheme, nl_capacity=cap, keep_full_nl=True) as eng:
        eng.upload(r)
        eng.bin()
        eng.build_nebr()
        return [*eng.get_nebr(), *eng.carbon_lists().values()] if s.n > s.n_metal else list(eng.get_nebr())


# atoms: 500, 28,672 (nine lanes), 28,800 (four), 32,000
@pytest.mark.parametrize("cells", [(5, 5, 5), (16, 16, 28), (15, 16, 30), (20, 20, 20)])
def test_bulk(gpu, cells):
    s = _bulk(*cells)
    assert s.n == s.n_metal == 4 * cells[0] * cells[1] * cells[2]
    r = s.r.astype(np.float64)
    r[:, :3] += 0.04 * np.random.default_rng(s.n).standard_normal((s.n, 3))
    half = 0.5 * np.array([s.params.region.x, s.params.region.y, s.params.region.z])
    r[:, :3] = (r[:, :3] + half) % (2 * half) - half
    for a, b in zip(_lists(s, r, 0, 160), _lists(s, r, 3, 160)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("metal", [131072, 131073])
def test_cluster(gpu, metal):
    s = sg.make_system(regime=2, ux=20, uy=22, n_metal=metal, temperature=600.0, geometry="sphere", seed=5)
    r = s.r.astype(np.float64)
    r[:, :3] += 0.02 * np.random.default_rng(metal).standard_normal((s.n, 3))
    for a, b in zip(_lists(s, r, 0, 128), _lists(s, r, 3, 128)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("count", [2, 3])
def test_replicas_of_bulk_metal(gpu, count):
    """13,500 atoms each: two stay on nine lanes, three do not."""
    systems = [sg.make_system(regime=0, material=3, ux=15, uy=15, uz=15, temperature=300.0 + 50.0 * k, geometry="reference",
                              seed=3 + k, velocities="maxwell") for k in range(count)]
    with sg.Batch([s.params for s in systems], precision="mixed", metal_lanes=8, rebuild_every=4) as b:
        for k, s in enumerate(systems):
            b.upload(k, s.r, s.v, s.a)
            b.set_run_state(k, 0, 1, 0.0)
        b.run(12, records=False)
        got = [b.download(k) for k in range(count)]
    for s, state in zip(systems, got):
        with sg.Engine(s.params, precision="mixed", metal_lanes=8, rebuild_every=4, xcd_map=0) as eng:
            eng.upload(s.r, s.v, s.a)
            eng.set_run_state(0, 1, 0.0)
            eng.run(12)
            for x, y in zip(eng.download(), state):
                assert np.array_equal(x, y)
