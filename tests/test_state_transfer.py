"""State to and from the device at the sizes where the transfer changes: one copy for everything (below
256 KiB of positions), two overlapped pinned slots, several host threads (8 MiB and more), with
ragged last pieces and arrays left out.  Values are moved and rounded once, so they come back exactly."""
import ctypes as C

import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu

# atoms: 397, 3,211 (103 KB a position array), 8,393 (269 KB), 34,273, 104,993 (8.4 MB in all, FP64), 138,407
SIZES = [(3, 4, 13), (10, 10, 11), (16, 16, 201), (33, 32, 481), (60, 54, 1313), (65, 66, 1127)]


def _state(n):
    rng = np.random.default_rng(n)
    return rng.standard_normal((n, 4)), rng.standard_normal((n, 3)), rng.standard_normal((n, 3))


@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("ux,uy,metal", SIZES)
def test_state_comes_back(gpu, ux, uy, metal, prec):
    s = sg.make_system(regime=2, ux=ux, uy=uy, n_metal=metal, temperature=300.0, geometry="sphere", seed=1)
    n = s.n
    state = _state(n)
    stored = [x if prec == "mixed" else x.astype(np.float32).astype(np.float64) for x in state]
    narrow = [x.astype(np.float32) for x in state]
    with sg.Engine(s.params, precision=prec) as eng:
        for _ in range(2):
            eng.upload(*state)
            for a, b in zip(eng.download(), stored):
                assert np.array_equal(a, b)
        acc, e, _ = eng.forces()
        assert np.array_equal(acc, stored[2]) and np.array_equal(e, stored[0][:, 3])
        # float arrays both ways, one array at a time; the others keep their values
        p = [x.ctypes.data_as(C.c_void_p) for x in narrow]
        assert eng.lib.sgk_upload(eng.h, None, p[1], None) == 0
        got = eng.download()
        assert np.array_equal(got[0], stored[0]) and np.array_equal(got[1], narrow[1].astype(np.float64))
        out = [np.full_like(x, np.nan) for x in narrow]
        q = [x.ctypes.data_as(C.c_void_p) for x in out]
        assert eng.lib.sgk_download(eng.h, None, None, q[2]) == 0
        assert eng.lib.sgk_download(eng.h, q[0], q[1], None) == 0
        assert all(np.array_equal(a, b) for a, b in zip(out, narrow))


@pytest.mark.parametrize("prec", ["mixed", "fp32"])
def test_replica_states_come_back(gpu, prec):
    systems = [sg.make_system(regime=2, ux=ux, uy=uy, n_metal=m, temperature=300.0, geometry="sphere", seed=1)
               for ux, uy, m in (SIZES[0], SIZES[2], SIZES[4])]
    with sg.Batch([s.params for s in systems], precision=prec) as b:
        states = [_state(s.n) for s in systems]
        for k, st in enumerate(states):
            b.upload(k, *st)
        b.upload(1, states[1][0][:, :3])  # three columns: the energies become 0
        for k, st in enumerate(states):
            want = [x if prec == "mixed" else x.astype(np.float32).astype(np.float64) for x in st]
            if k == 1:
                want[0] = want[0] * np.array([1.0, 1.0, 1.0, 0.0])
            for x, y in zip(b.download(k), want):
                assert np.array_equal(x, y)
        with pytest.raises(ValueError):
            b.upload(0, states[1][0])


def test_records_as_dicts(gpu):
    s = sg.config_system("small", "config")
    with sg.Engine(s.params, precision="mixed") as eng:
        eng.upload(s.r, s.v, s.a)
        eng.set_run_state(0, 1, 0.0)
        recs = eng.run(7)
        one = eng.props()
    assert [r["step"] for r in recs] == list(range(1, 8)) and set(one) == set(recs[0])
    assert all(type(r["step"]) is int and type(r["totEnergy"]) is float and type(r["comSum"]) is list and
               len(r["comSum"]) == 3 and type(r["comSum"][0]) is float for r in recs)
