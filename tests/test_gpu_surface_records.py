"""sphgpu_surfacer_particles gives the last anisotropic call's ellipsoids, also
after an isotropic field of the same particles, in either form of the field
kernel, and nothing after one of another number of particles."""
import numpy as np
import pytest

from graphics_amd import sphgpu as sg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,fine", [(900, 4), (1500, 2), (8000, 4), (64000, 2)])   # few nodes, and (the last two) blocks of nodes
def test_ellipsoids_stay_over_an_isotropic_field(gpu, n, fine):
    print(f"[records] n={n} fine={fine}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, 0.2, (n, 3)).astype(np.float32)
    x[: n // 2, 1] *= 0.1
    s = sg.Surfacer((0.0,) * 3, (0.2,) * 3, 0.01, 0.02, 0.01 / fine)
    s.aniso(x)
    first = s.particles(n)
    assert np.abs(first[1] - np.eye(3)).max() > 0.1 and first[3].max() > 0
    s.isotro(x)
    for a, b in zip(first, s.particles(n)):
        assert a.tobytes() == b.tobytes()
    more = rng.uniform(0.0, 0.2, (n + 2000, 3)).astype(np.float32)   # (more than the buffers hold)
    s.isotro(more)
    assert not any(a.any() for a in s.particles(n + 2000))
    s.aniso(x)
    for a, b in zip(first, s.particles(n)):
        assert a.tobytes() == b.tobytes()
    s.close()
