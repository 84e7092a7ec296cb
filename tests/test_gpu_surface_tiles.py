"""The tiled node field at its edges (tile remainders, boxes over tile and
cell borders, boxes reaching past one cell, particles outside the grid)
against the same sum in 64 bits over the device's own ellipsoids.

Tolerance: a node's offset from an ellipsoid is rounded at coordinates up to
0.3 (3e-8), stretched by |G| <= 6 over the radius 0.02 (1e-5 of it), and the
spline's slope is at most 3 of its peak a radius, in mean about a third of
that over the support; the signs of some ten contributions mix."""
import numpy as np
import pytest

from graphics_amd import sphgpu as sg

pytestmark = pytest.mark.gpu

RP, RH = 0.01, 0.02


def _reference(grid_min, num, cell, xbar, G, det, hcells):
    """det W(|G (p - xbar)|) over the box p - ext .. p + ext + 1 of each particle."""
    f = np.zeros(num[::-1])
    gm, c32 = grid_min.astype(np.float32), np.float32(cell)
    for x, g, d in zip(xbar, G.astype(np.float64), det):
        sig0 = 1.0 / np.linalg.eigvalsh(g).min()
        ext = int(hcells * sig0 * (1.0 + 1e-7))
        p = ((x - gm) / c32).astype(int)
        lo, hi = np.maximum(p - ext, 0), np.minimum(p + ext + 1, np.array(num) - 1)
        if (hi < lo).any():
            continue
        ax = [gm[a].astype(np.float64) + np.arange(lo[a], hi[a] + 1) * float(c32) - float(x[a]) for a in range(3)]
        x_, y_, z_ = ax[0], ax[1][:, None], ax[2][:, None, None]
        m = g @ g                        # |G d|^2 = d^T G^2 d
        plane = m[0, 0] * x_ * x_ + m[1, 1] * y_ * y_ + 2.0 * m[0, 1] * x_ * y_
        r2 = plane[None] + (z_ * (2.0 * (m[0, 2] * x_ + m[1, 2] * y_))[None]) + m[2, 2] * z_ * z_
        at = np.nonzero(r2 <= RH * RH)
        r = np.sqrt(np.maximum(r2[at], 0.0)) / RH
        w = np.where(r < 0.5, 8 * (1 - 6 * r ** 2 + 6 * r ** 3), 16 * (1 - r) ** 3)
        f[at[0] + lo[2], at[1] + lo[1], at[2] + lo[0]] += w * (RP ** 3 / (np.pi * RH ** 3) * d)
    return f


@pytest.mark.parametrize("n,cell,aniso", [
    # one block per particle
    (0, 0.0025, True),
    (1, 0.0025, True),
    (40, 0.0025, False),
    (600, 0.003, True),       # a sheet and loose particles
    (600, 0.0061, True),      # few nodes a kernel radius
    (300, 0.05, False),       # node spacing over the kernel radius
    # tiles (25 and 40 nodes a kernel radius), not in line with the cells
    (520, 0.0008, True),      # the smaller tiles
    (126, 0.0005, True),      # the larger tiles
    (126, 0.0005, False),
])
def test_field_tiles(gpu, n, cell, aniso):
    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, 0.1, (n, 3))
    x[: n // 3, 1] = 0.05 + rng.normal(0.0, 2e-4, n // 3)      # a thin sheet: flat, wide ellipsoids
    if n > 1:
        x[-1] = (0.31, 0.02, 0.02)                             # outside the grid
    x = x.astype(np.float32)
    s = sg.Surfacer((0.0, 0.0, 0.0), (0.11, 0.1, 0.13), RP, RH, cell)
    (s.aniso if aniso else s.isotro)(x)
    f = s.field()
    if aniso and n:
        xb, G, det, _ = s.particles(n)
    else:
        xb, G, det = x, np.broadcast_to(np.eye(3), (n, 3, 3)), np.ones(n)
    ref = _reference(s.grid_min, s.grid_num, s.cell, xb, G, det, int(RH / s.cell))
    top = max(np.abs(ref).max(), 1e-30)
    print(f"[tiles] n={n} cell={cell} aniso={aniso}: {np.abs(f - ref).max() / top:.2e}", flush=True)
    assert np.abs(f - ref).max() <= 2e-5 * top
    # the atomics of the splat and of boxes past one cell change the order of a
    # node's additions, no more
    (s.aniso if aniso else s.isotro)(x)
    assert np.abs(s.field() - f).max() <= 1e-6 * top
    s.close()
