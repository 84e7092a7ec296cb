"""The window builds give each particle two lanes, which add its terms in list
order: the same bits as the gathers' one lane, on packed tiles, on tiles with
32-bit lists (rows so short that a tile spans more than three) and on both at
once, with one and two phases, moving boundaries and a ragged last tile."""
import numpy as np
import pytest

from graphics_amd import scenes, sphgpu as sg

pytestmark = pytest.mark.gpu


def _run(sc, on, steps=4):
    sim = scenes.make_simulation(sc)
    sim.set_lds_windows(on)
    st = [sim.step() for _ in range(steps)]
    form = sim.list_form()
    out = [sim.get(f).tobytes() for f in (sg.F_POS, sg.F_VEL, sg.F_RHO)]
    its = [(s["iter_density"], s["iter_divergence"], s["density_err"], s["divergence_err"]) for s in st]
    sim.close()
    return out, its, form


@pytest.mark.parametrize("solver", [sg.DFSPH, sg.IISPH])
@pytest.mark.parametrize("n,box", [((97, 6, 7), (2.1, 0.3, 0.3)), ((5, 12, 37), (0.2, 0.4, 0.9)),
                                   ((33, 9, 11), (0.9, 0.4, 0.4)), ((3, 3, 3), (0.2, 0.2, 0.2))])
@pytest.mark.parametrize("phases", [1, 2])
def test_two_lanes_equal_one(gpu, solver, n, box, phases):
    print(f"[lanes] solver={solver} n={n} phases={phases}", flush=True)
    make = scenes.two_layer if phases == 2 else scenes.small_dam
    runs = [_run(make(solver, n=n, box=box), on) for on in (1, 0)]
    assert runs[0][:2] == runs[1][:2]
    form = runs[0][2]
    if n[0] == 97:
        assert form["packed_tiles"] > 0
    if n[0] == 5:
        assert form["packed_tiles"] < form["tiles"]


@pytest.mark.parametrize("on", [0, 1])
def test_partial_sums_in_particle_order(gpu, on):
    """The error of a loop is the FP64 sum over the particles in a fixed order:
    two runs of each build, and the two builds, report the same doubles."""
    sc = scenes.small_dam(sg.DFSPH, n=(41, 7, 9), box=(1.0, 0.3, 0.3))
    a, b = _run(sc, on), _run(sc, 1 - on)
    assert a[1] == b[1] and np.isfinite([v for s in a[1] for v in s]).all()
