"""List build at the sizes where its lane mapping changes or runs out: nine lanes per atom up to
2^18 atoms (one per column of the atom's 27 cells, 32 or 64 candidates as bits, the rest one by one),
one lane per carbon and four per metal atom above.  The lists are integers: every case must equal
the per-atom scheme (nl_scheme 0), which the parity tests tie to the oracle, entry for entry."""
import numpy as np
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


def _lists(s, r, scheme, cap, full):
    with sg.Engine(s.params, precision="mixed", nl_scheme=scheme, nl_capacity=cap, keep_full_nl=full) as eng:
        eng.upload(r)
        eng.bin()
        eng.build_nebr()
        out = eng.carbon_lists()
        if full:
            out["nn"], out["nbl"] = eng.get_nebr()
        eng.compute_forces()
        out["acc"] = eng.forces()[0]
    return out


# scale: the cluster compressed about its centre, for crowded cells (at 0.8, up to ~110 candidates in a
# column and ~150 neighbours)
@pytest.mark.parametrize("ux,uy,metal,scale", [
    (3, 2, 13, 1.0),      # grid axes of a few cells: every column wraps
    (4, 5, 1, 1.0),       # one metal atom: a workgroup with one used group of nine lanes
    (5, 6, 201, 1.0),
    (7, 5, 252, 0.93),    # exactly 9 workgroups of 28 metal atoms, and a slightly compressed cluster
    (9, 9, 561, 0.8),     # more than 64 candidates in a column
    (18, 14, 1289, 0.85),
])
def test_nine_lane_lists_equal_the_per_atom_scheme(gpu, ux, uy, metal, scale):
    s = sg.make_system(regime=2, ux=ux, uy=uy, n_metal=metal, temperature=600.0, geometry="sphere", seed=3)
    r = s.r.astype(np.float64)
    rng = np.random.default_rng(ux * 100 + uy)
    c = r[:metal, :3].mean(0)
    r[:metal, :3] = c + scale * (r[:metal, :3] - c)
    r[:, :3] += 0.02 * rng.standard_normal((s.n, 3))
    print(f"[nl] {ux}x{uy} sheet, {metal} metal, scale {scale}", flush=True)
    want, got = _lists(s, r, 0, 248, True), _lists(s, r, 3, 248, True)
    assert scale > 0.82 or want["nn"].max() > 128
    for k in want:
        assert np.array_equal(want[k], got[k]), k


@pytest.mark.parametrize("metal", [2911, 2975])
def test_lists_either_side_of_the_lane_threshold(gpu, metal):
    """262,111 atoms (nine lanes) and 262,175 (one lane per carbon): both equal the per-atom scheme."""
    s = sg.make_system(regime=2, ux=90, uy=90, n_metal=metal, temperature=900.0, geometry="sphere", seed=5)
    assert (s.n <= 1 << 18) == (metal == 2911)
    r = s.r.astype(np.float64)
    r[:, :3] += 0.02 * np.random.default_rng(metal).standard_normal((s.n, 3))
    print(f"[nl] {s.n} atoms", flush=True)
    want, got = _lists(s, r, 0, 128, False), _lists(s, r, 3, 128, False)
    for k in want:
        assert np.array_equal(want[k], got[k]), k


def test_nine_lane_lists_at_their_capacities(gpu):
    """Lists cut at a capacity report it and leave counts within it (the entries kept are the first)."""
    s = sg.make_system(regime=2, ux=5, uy=6, n_metal=201, temperature=300.0, geometry="sphere", seed=1)
    for cfg, word in ((dict(nl_capacity=40), "neighbour-list"), (dict(lj_capacity=8), "metal-neighbour"),
                      (dict(close_capacity=8), "close-neighbour")):
        print(f"[nl] {cfg}", flush=True)
        with sg.Engine(s.params, precision="mixed", **cfg) as eng:
            eng.upload(s.r.astype(np.float64))
            eng.bin()
            with pytest.raises(RuntimeError, match=word):
                eng.build_nebr()
            out = eng.carbon_lists()
            assert out["n_lj"].max() <= eng.cfg.lj_capacity and out["n_close"].max() <= eng.cfg.close_capacity
