"""The list builder of small scenes (a block takes a quarter of a tile, a wave
one row run) against the builder of large ones: the same particles in a domain
stretched until the search takes its other form, which the large builder
follows, step to the same bytes and have the same lists and counters.  Sizes
at the edges of a quarter and a tile, runs of more than 64 candidates, lists
past their width, tiles of more than three rows and of one, rows with gaps,
and the two sides of the size from which the large builder takes over.  (The
step is short, so that no particle leaves the smaller domain.)"""
import numpy as np
import pytest

from graphics_amd import sphgpu as sg

pytestmark = pytest.mark.gpu

S = 0.02


def _run(x, wall, far):
    sim = sg.Simulation(sg.default_params(solver=sg.WCSPH, spacing_r=S, smooth_radius_h=2 * S, dt=1e-9,
                                          space_min=(-0.2, -0.2, -0.2),
                                          space_max=(13.0, 13.0, 13.0) if far else (2.2, 0.6, 0.6)))
    sim.add_phase(1000.0, 0.01)
    sim.add_fluid(x)
    sim.add_solid(wall, 0.01)
    sim.init()
    st = [sim.step() for _ in range(3)][-1]
    counts, kinds, ids, dis = sim.neighbours(112)
    out = [sim.get(sg.F_POS).tobytes(), sim.get(sg.F_VEL).tobytes(), sim.get(sg.F_RHO).tobytes(), counts.tobytes(),
           kinds.tobytes(), ids.tobytes(), dis.tobytes()]
    out += [st[k] for k in ("zero_dis", "too_many_neigb", "list_overflow")]
    form = sim.list_form()
    sim.close()
    return out, form, counts


@pytest.mark.parametrize("n,size,kind", [
    (1, (0.3, 0.3, 0.3), "uniform"), (63, (0.2, 0.1, 0.1), "uniform"), (64, (1.0, 0.02, 0.02), "uniform"),
    (65, (0.2, 0.1, 0.1), "uniform"), (256, (2.0, 0.03, 0.03), "uniform"), (257, (0.3, 0.3, 0.3), "uniform"),
    (900, (0.11, 0.11, 0.11), "uniform"),           # runs of more than 64, lists past 64
    (700, (2.0, 0.05, 0.05), "gaps"), (5000, (0.4, 0.4, 0.4), "uniform"),
    (81920, (2.0, 0.4, 0.4), "lattice"), (81921, (2.0, 0.4, 0.4), "lattice"),   # 320 tiles and one more
])
def test_quarters_equal_tiles(gpu, n, size, kind):
    print(f"[quarters] n={n} {kind}", flush=True)
    rng = np.random.default_rng(n)
    if kind == "lattice":
        g = np.stack(np.meshgrid(*(np.arange(k) for k in (100, 29, 29)), indexing="ij"), -1).reshape(-1, 3)[:n]
        x = (g * 0.019 + rng.uniform(-0.002, 0.002, (n, 3))).astype(np.float32)
    else:
        x = (rng.uniform(0.0, 1.0, (n, 3)) * np.asarray(size)).astype(np.float32)
        if kind == "gaps":
            x = x[(x[:, 0] % 0.7 < 0.15) | (rng.uniform(size=n) < 0.02)]
        for _ in range(n // 100):
            x[rng.integers(len(x))] = x[rng.integers(len(x))]
    wall = (rng.uniform(0.0, 1.0, (max(n // 8, 1), 3)) * np.asarray(size)).astype(np.float32)
    wall[:, 1] = 0.0
    near, form, counts = _run(x, wall, False)
    far, _, _ = _run(x, wall, True)
    assert [a == b for a, b in zip(near, far)] == [True] * len(near)
    if (n, kind) == (256, "uniform"):
        assert form["packed_tiles"] == form["tiles"]
    if (n, kind) == (5000, "uniform"):
        assert form["packed_tiles"] < form["tiles"]
    if n == 900:
        assert counts.max() > 64
