"""Replicas that a batch refuses before it touches a device, as a system alone is refused."""
import pytest

import surfacegrowthconsole_amd as sg


@pytest.mark.parametrize("cells,capacity", [((1024, 1024, 32), 64), ((2048, 1024, 128), 8), ((1 << 12, 1 << 12, 1 << 12), 16)])
@pytest.mark.parametrize("where", [0, 1])
def test_cell_grid_beyond_32_bits(cells, capacity, where):
    params = [sg.make_system(regime=2, ux=4, uy=4, n_metal=13).params for _ in range(2)]
    params[where].cells.x, params[where].cells.y, params[where].cells.z = cells
    with pytest.raises(RuntimeError, match=f"replica {where}: cell grid too large"):
        sg.Batch(params, cell_capacity=capacity)
