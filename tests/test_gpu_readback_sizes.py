"""Particles read back whole at every remainder of a 16-byte word and at the edges of
the handle's own bytes (64 KB), a stage's sizes and a chunk (2 MB): what was put in
comes out, bit for bit, and nothing past it is written."""
import ctypes as C

import numpy as np
import pytest

from graphics_amd import sphgpu as sg

pytestmark = pytest.mark.gpu

S = 0.02


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 1723, 5461, 5462, 16383, 16384, 16385, 43690, 43691, 65537,
                               174762, 174763, 524287, 524288, 524289])
def test_every_byte_arrives(gpu, n):
    print(f"[sizes] {n}", flush=True)
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = ((g + 1.0) * S).astype(np.float32)
    v = rng.uniform(-1, 1, x.shape).astype(np.float32)
    sim = sg.Simulation(sg.default_params(solver=sg.WCSPH, spacing_r=S, smooth_radius_h=2 * S, dt=1e-4,
                                          space_min=(-0.05,) * 3, space_max=((m + 3) * S,) * 3))
    sim.add_phase(1000.0, 0.01)
    sim.add_fluid(x, v)
    sim.init()
    assert sim.num_fluid() == n
    for _ in range(3):                               # plain, and through pinned bytes
        for field, want in ((sg.F_POS, x), (sg.F_VEL, v)):
            a = np.full(3 * n + 4, -7.25, np.float32)
            assert sim.lib.sphgpu_get_fluid(sim.h, field, a.ctypes.data_as(C.POINTER(C.c_float))) == 0
            assert np.array_equal(a[:3 * n].reshape(n, 3), want)
            assert np.all(a[3 * n:] == -7.25)
        ids = np.full(n + 4, -3, np.int64)
        assert sim.lib.sphgpu_get_fluid_ids(sim.h, ids.ctypes.data_as(C.POINTER(C.c_longlong))) == 0
        assert np.array_equal(ids[:n], np.arange(n)) and np.all(ids[n:] == -3)
    del sim
