"""The node field on the two sides of the line from which it is summed in
blocks of nodes, with whole and fractional node counts a kernel radius (boxes
that hold their ellipsoid and boxes that cut it) and particles at and outside
the grid's lower faces: against the same sum in 64 bits over the device's own
ellipsoids, with the tolerance of the tiled field's test."""
import numpy as np
import pytest

from graphics_amd import sphgpu as sg
from test_gpu_surface_tiles import RH, RP, _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cell,aniso", [
    (3906, 0.0025, True), (3907, 0.0025, True), (3907, 0.0025, False),      # 8 nodes: 2,000,000 / 512
    (9260, 0.0031, True), (9260, 0.0031, False),                            # 6.45 nodes
    (16001, 0.0039, True),                                                  # 5.13 nodes
    (31250, 0.005, True),                                                   # 4 nodes, a node a lane's edge
])
def test_field_blocks(gpu, n, cell, aniso):
    print(f"[blocks] n={n} cell={cell} aniso={aniso}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, 1.0, (n, 3)) * (0.3, 0.25, 0.2)
    k = n // 3
    x[:k, 1] = 0.05 + rng.normal(0.0, 2e-4, k)           # a thin sheet: flat, wide ellipsoids
    x[k:k + 40] = rng.uniform(-0.035, 0.005, (40, 3))    # at and past the lower corner
    x = x.astype(np.float32)
    s = sg.Surfacer((0.0, 0.0, 0.0), (0.31, 0.26, 0.21), RP, RH, cell)
    (s.aniso if aniso else s.isotro)(x)
    f = s.field()
    again = s.field()
    assert np.array_equal(f, again)
    if aniso:
        xb, G, det, _ = s.particles(n)
    else:
        xb, G, det = x, np.broadcast_to(np.eye(3), (n, 3, 3)), np.ones(n)
    ref = _reference(s.grid_min, s.grid_num, s.cell, xb, G, det, int(RH / s.cell))
    top = np.abs(ref).max()
    print(f"[blocks] {np.abs(f - ref).max() / top:.2e}", flush=True)
    assert np.abs(f - ref).max() <= 2e-5 * top
    s.close()
