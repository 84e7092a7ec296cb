"""The isotropic node field on the two sides of the line from which it is summed in
blocks of nodes, against the sum in 64 bits, with the tolerance of the tiled
field's test; and the blocks' sums, which are the same every run."""
import numpy as np
import pytest

from graphics_amd import sphgpu as sg
from test_gpu_surface_tiles import RH, RP, _reference

pytestmark = pytest.mark.gpu


def _particles(n, lo):
    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, 1.0, (n, 3)) * (0.3, 0.25, 0.2) + 0.002
    if lo:
        x[:40] = rng.uniform(-0.035, 0.005, (40, 3))     # at and past the lower corner
    return x.astype(np.float32)


@pytest.mark.parametrize("n,cell", [
    (7812, 0.0025), (7813, 0.0025),      # 8 nodes a radius: 4,000,000 / 512
    (18519, 0.0031),                     # 6.45 nodes
    (62500, 0.005),                      # 4 nodes, a node a lane's edge
])
def test_isotropic_field(gpu, n, cell):
    print(f"[spheres] n={n} cell={cell}", flush=True)
    x = _particles(n, True)
    s = sg.Surfacer((0.0,) * 3, (0.31, 0.26, 0.21), RP, RH, cell)
    s.isotro(x)
    f = s.field()
    ref = _reference(s.grid_min, s.grid_num, s.cell, x, np.broadcast_to(np.eye(3), (n, 3, 3)), np.ones(n), int(RH / s.cell))
    top = np.abs(ref).max()
    print(f"[spheres] {np.abs(f - ref).max() / top:.2e}", flush=True)
    assert np.abs(f - ref).max() <= 2e-5 * top
    s.close()


@pytest.mark.parametrize("n,cell", [(7813, 0.0025), (18519, 0.0031)])
def test_blocks_give_the_same_sums_every_run(gpu, n, cell):
    print(f"[spheres] again n={n}", flush=True)
    x = _particles(n, False)                 # (all in the grid: none is added by atomics)
    s = sg.Surfacer((0.0,) * 3, (0.31, 0.26, 0.21), RP, RH, cell)
    s.isotro(x)
    f = s.field()
    for _ in range(4):
        s.isotro(x[::-1])                    # (another field in between)
        s.isotro(x)
        assert s.field().tobytes() == f.tobytes()
    s.close()
