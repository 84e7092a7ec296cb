"""A WCSPH scene alone and beside a larger one in the same handle: the number of
tiles decides how many lanes a particle has, and the results are the same bytes.
One and two phases, walls in reach, packed lists and lists of crowded tiles."""
import numpy as np
import pytest

from graphics_amd import sphgpu as sg

pytestmark = pytest.mark.gpu

S = 0.02


def _lattice(rng, n, spread=0.1):
    g = np.stack(np.meshgrid(*(np.arange(k) for k in n), indexing="ij"), -1).reshape(-1, 3)
    return ((g + 1.0 + rng.uniform(-spread, spread, g.shape)) * S).astype(np.float32)


def _walls(n):
    a, b, c = n
    p = [(i, j, k) for i in range(a) for j in range(b) for k in range(c) if 0 in (i, j, k)]
    return (np.array(p) * S).astype(np.float32)


def _run(beside, kind, graph):
    rng = np.random.default_rng(3)
    dt = 1e-7 if kind == "crowded" else 1e-4
    sim = sg.Simulation(sg.default_params(solver=sg.WCSPH, spacing_r=S, smooth_radius_h=2 * S, dt=dt, gamma=7.0,
                                          sound_speed=20.0, num_scenes=2 if beside else 1, use_graph=int(graph)))
    sim.add_phase(1000.0, 0.01)
    sim.add_phase(2000.0, 0.05)
    sim.set_scene_domain(0, (-0.1,) * 3, (0.6,) * 3)
    if kind == "crowded":
        x = rng.uniform(0.02, 0.2, (3000, 3)).astype(np.float32)
    else:
        x = _lattice(rng, (13, 12, 11))
    v = rng.uniform(-0.5, 0.5, x.shape).astype(np.float32)
    if kind == "phases":
        half = len(x) // 2
        sim.add_fluid(x[:half], v[:half], phase=0)
        sim.add_fluid(x[half:], v[half:], phase=1)
    else:
        sim.add_fluid(x, v)
    sim.add_solid(_walls((15, 14, 13)), 0.02)
    if beside:   # more than 320 tiles
        sim.set_scene_domain(1, (-0.1,) * 3, (2.2, 0.7, 0.7))
        sim.add_fluid(_lattice(rng, (100, 29, 29)), scene=1)
    out = []
    for k in range(4):
        st = sim.step()
        out += [sim.get(f)[:len(x)].tobytes() for f in (sg.F_RHO, sg.F_ACC, sg.F_VEL, sg.F_POS)]
    assert (sim.num_fluid() > 320 * 256) == beside and st["removed"] == 0
    sim.close()
    return out


@pytest.mark.parametrize("kind", ["one", "phases", "crowded"])
@pytest.mark.parametrize("graph", [False, True])
def test_same_bits_alone_and_in_a_batch(gpu, kind, graph):
    print(f"[wcsph bits] {kind} graph {graph}", flush=True)
    alone, batch = _run(False, kind, graph), _run(True, kind, graph)
    same = [a == b for a, b in zip(alone, batch)]
    assert all(same), same
