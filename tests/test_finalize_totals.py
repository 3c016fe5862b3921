"""A step closed by its own launches: up to 256 partials by one workgroup, more by chunk totals.  Its record is that of the same
step closed by the next one's kernels, which take up to 1,024 directly, bit for bit, on both sides of the line: for
bulk metal (16 lanes an atom, 16 atoms a partial, padded to eight) and for sheets."""
import pytest

import surfacegrowthconsole_amd as sg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("cells", [(8, 8, 16), (5, 5, 41), (10, 10, 20), (16, 16, 16)])  # 256, 264, 500, 1,024 partials
def test_bulk(gpu, cells, prec):
    s = sg.make_system(regime=0, material=3, ux=cells[0], uy=cells[1], uz=cells[2], temperature=300.0,
                       geometry="reference", velocities="maxwell", seed=4)
    _same(s, prec, 16)


@pytest.mark.parametrize("prec", ["mixed", "fp32"])
@pytest.mark.parametrize("ux,uy", [(31, 64), (8, 249), (32, 62), (88, 92)])  # 248, 249, 248 and 1,012 of carbon
def test_sheets(gpu, ux, uy, prec):
    _same(sg.make_system(regime=2, ux=ux, uy=uy, n_metal=13, temperature=300.0, geometry="sphere", velocities="maxwell",
                         seed=4), prec, 16)


def _same(s, prec, lanes):
    out = []
    for chunks in ([1] * 9, [9]):
        with sg.Engine(s.params, precision=prec, metal_lanes=lanes) as eng:
            eng.upload(s.r, s.v, s.a)
            eng.set_run_state(0, 1, 0.0)
            out.append([r for n in chunks for r in eng.run(n)])
    assert out[0] == out[1]
