"""The search of one scene in parts of 2,048 cells, and the WCSPH passes of few
tiles with two lanes a particle, against the FP64 oracle over three steps, for
grids of less than one part up to fifteen; the search's other form on the same
scenes is compared bit for bit by the tests of the search forms."""
import numpy as np
import pytest

from graphics_amd import scenes, sphgpu as sg
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


# boxes from under one part to fifteen parts of cells
@pytest.mark.parametrize("n,box", [((6, 5, 4), (0.16, 0.14, 0.12)), ((10, 9, 8), (0.44, 0.44, 0.4)),
                                   ((25, 9, 8), (0.92, 0.8, 0.8)), ((40, 12, 10), (1.2, 1.2, 1.0))])
def test_lists_after_steps(gpu, n, box):
    print(f"[parts] {n} {box}", flush=True)
    sc = scenes.small_dam(sg.WCSPH, n=n, box=box)
    sim = scenes.make_simulation(sc)
    for _ in range(3):
        sim.step()
    o = orc.from_scene(sc, 64)
    for _ in range(3):
        o.step()
    # three steps of 1e-4 s: FP32 rounding of the step, as in the single-step tests
    x, ref = sim.get(sg.F_POS), o.get_by_id(orc.F_POS)[1]
    assert np.abs(x - ref).max() <= 1e-5 * np.abs(ref).max()
    rho, ref = sim.get(sg.F_RHO), o.get_by_id(orc.F_RHO)[1]
    assert np.abs(rho - ref).max() <= 1e-5 * np.abs(ref).max()
    sim.close()
    o.close()
