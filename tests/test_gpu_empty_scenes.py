"""Scenes without fluid: a handle that starts empty and is filled by an emitter,
and a handle with fewer tiles than scenes, whose loops' tests have no block for
every scene.  Every scene's loop ends at its smallest count where there is
nothing to solve, and the filled scene steps to the same bytes as alone."""
import numpy as np
import pytest

from graphics_amd import sphgpu as sg

pytestmark = pytest.mark.gpu

S = 0.02
ITER = dict(min_iter_density=3, max_iter_density=9, min_iter_div=2, max_iter_div=8)
SOLVERS = [sg.WCSPH, sg.DFSPH, sg.IISPH, sg.PCISPH, sg.IISPH_DF]


def _fluid():
    rng = np.random.default_rng(5)
    g = np.stack(np.meshgrid(*(np.arange(k) for k in (6, 5, 4)), indexing="ij"), -1).reshape(-1, 3)
    return ((g + 1.5 + rng.uniform(-0.01, 0.01, g.shape)) * S).astype(np.float32)


def _sim(solver, scenes, fill):
    sim = sg.Simulation(sg.default_params(solver=solver, spacing_r=S, smooth_radius_h=2 * S, dt=1e-4,
                                          num_scenes=scenes, fluid_capacity=600, boundary_density=1000.0,
                                          space_min=(-0.1,) * 3, space_max=(0.4,) * 3, **ITER))
    sim.add_phase(1000.0, 0.01)
    for s in range(scenes):
        sim.set_scene_domain(s, (-0.1,) * 3, (0.4,) * 3)
        sim.add_solid(np.array([[0.0, 0.0, 0.0], [S, 0.0, 0.0]], np.float32), 0.01, scene=s)
    if fill is not None:
        sim.add_fluid(_fluid(), scene=fill)
    return sim


def _state(sim):
    return [sim.get(f).tobytes() for f in (sg.F_POS, sg.F_VEL, sg.F_RHO)]


def _counts(solver, st):
    if solver == sg.WCSPH:
        return []
    return [st["iter_density"]] + ([st["iter_divergence"]] if solver in (sg.DFSPH, sg.IISPH_DF) else [])


@pytest.mark.parametrize("solver", SOLVERS)
@pytest.mark.parametrize("scenes", [1, 3])
def test_step_of_an_empty_handle_then_append(gpu, solver, scenes):
    print(f"[empty] solver {solver} scenes {scenes}", flush=True)
    sim, ref = _sim(solver, scenes, None), _sim(solver, 1, 0)
    st = sim.step()
    assert st["num_fluid"] == 0
    for s in range(scenes):
        assert _counts(solver, sim.scene_stats(s)) == [3, 2][:len(_counts(solver, st))]
    sim.append_fluid(_fluid(), scene=scenes - 1)
    for _ in range(2):
        a, b = sim.step(), ref.step()
        assert a["num_fluid"] == len(_fluid())
        assert _counts(solver, sim.scene_stats(scenes - 1)) == _counts(solver, b)
        assert _state(sim) == _state(ref)
    sim.close()
    ref.close()


@pytest.mark.parametrize("solver", SOLVERS)
@pytest.mark.parametrize("fill", [0, 2])
def test_fewer_tiles_than_scenes(gpu, solver, fill):
    print(f"[few tiles] solver {solver} scene {fill}", flush=True)
    sim, ref = _sim(solver, 3, fill), _sim(solver, 1, 0)
    for _ in range(2):
        sim.step()
        b = ref.step()
        for s in range(3):
            want = _counts(solver, b) if s == fill else [3, 2][:len(_counts(solver, b))]
            assert _counts(solver, sim.scene_stats(s)) == want, s
        assert _state(sim) == _state(ref)
    sim.close()
    ref.close()
