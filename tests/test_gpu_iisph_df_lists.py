"""The IISph DF_* boundary particles' own neighbour lists against the FP64
oracle: wall particles with no other solid near them, with a few particles of
one (listed), and with more than the list holds (those scan their cells)."""
import numpy as np
import pytest

from graphics_amd import scenes, sphgpu as sg
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# the single-step bar of the solvers' parity tests
FIELD_TOL = 1e-5


@pytest.mark.parametrize("other", [0, 5, 16, 18])
def test_wall_particles_with_another_solid(gpu, other):
    sc = scenes.small_dam(sg.IISPH_DF, n=(11, 9, 10), density_tol=0.0, min_iter_density=3, max_iter_density=3,
                          divergence_tol=0.0, min_iter_div=1, max_iter_div=1)
    sc.domains[0] = ((-0.02, -0.1, -0.02), sc.domains[0][1])
    x = sc.fluids[0][2]
    rng = np.random.default_rng(other)
    sc.beta = rng.uniform(0.9, 1.1, len(x)).astype(np.float32)
    sc.velocity = (-2.0 * (x - x.mean(0)) + rng.normal(0.0, 0.02, x.shape)).astype(np.float32)
    if other:
        # below the floor, out of the fluid's reach (0.04), within the floor's
        # (few enough that no list of the oracle reaches its cap of 48)
        c = np.array([0.1, -0.031, 0.1]) + rng.uniform(-0.002, 0.002, (other, 3))
        sc.solids.append((0, c.astype(np.float32), 0.01))
    sim = scenes.make_simulation(sc)
    print(f"[iisph_df lists] {other} of another solid", flush=True)
    sim.step()
    o = orc.from_scene(sc, 64)
    o.step()
    for f, of in ((sg.F_POS, orc.F_POS), (sg.F_VEL, orc.F_VEL), (sg.F_RHO, orc.F_RHO), (sg.F_ALPHA, orc.F_ALPHA)):
        a, b = sim.get(f).astype(np.float64), np.asarray(o.get_by_id(of)[1], np.float64)
        assert np.abs(a - b).max() / max(np.abs(b).max(), 1e-30) < FIELD_TOL, f
    sim.close()
    o.close()
