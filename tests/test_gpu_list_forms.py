"""The list builder of scenes past 320 tiles (and of sparse grids at any size), one
thread a particle, against brute force with the reference's FP32 predicate: entries
past its LDS stage (48 packed and 24 32-bit ones with six groups, 64 and 32 with
eight) and past the list width, with the table of either search; and the window
lists it writes, by passes with their LDS windows on and off."""
import numpy as np
import pytest
import torch

from graphics_amd import sphgpu as sg

pytestmark = pytest.mark.gpu

S = np.float32(0.02)


def _sim(x, wall, top, groups, solver=sg.WCSPH, **kw):
    sim = sg.Simulation(sg.default_params(solver=solver, spacing_r=S, smooth_radius_h=2 * S, dt=1e-20,
                                          space_min=(-0.1, -0.1, -0.1), space_max=top, **kw))
    sim.add_phase(1000.0, 0.01)
    sim.add_fluid(x)
    sim.add_solid(wall, 0.01)
    sim.set_tuning(stage_groups=groups)
    return sim


def _pairs(a, b, same):
    """(i, j) of the pairs within h, in order of i then j, and the number of coincident ones."""
    a, b = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    h2 = float((S + S) * (S + S))
    out, zero = [], 0
    for i0 in range(0, len(a), 1024):
        d = a[i0:i0 + 1024, None, :] - b[None, :, :]
        l2 = (d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2]
        hit = l2 < h2
        if same:
            k = torch.arange(len(hit), device="cuda")
            hit[k, k + i0] = False
        zero += int((hit & (l2 == 0)).sum())
        ij = hit.nonzero()
        ij[:, 0] += i0
        out.append(ij.cpu().numpy())
    return np.concatenate(out), zero


def _check(x, wall, top, groups, min_tiles):
    n = len(x)
    f, zf = _pairs(x, x, True)
    b, zb = _pairs(x, wall, False)
    nf, nb = np.bincount(f[:, 0], minlength=n), np.bincount(b[:, 0], minlength=n)
    sim = _sim(x, wall, top, groups)
    sim.init()
    sim.step()                           # (its counters include the autotuner's list builds)
    st = sim.step()
    form = sim.list_form()
    print(f"[list forms] n={n} groups {groups} most {nf.max()} fluid {nb.max()} wall, {form}", flush=True)
    assert np.abs(sim.get(sg.F_POS) - x).max() < 1e-30
    assert form["tiles"] >= min_tiles
    assert st["zero_dis"] == zf + zb
    assert st["too_many_neigb"] == np.maximum(nf + nb - 48, 0).sum()
    assert st["list_overflow"] == np.maximum(nf - 64, 0).sum() + np.maximum(nb - 48, 0).sum()
    sim.close()
    sim = _sim(x, wall, top, groups)     # the sets themselves, at x
    counts, kinds, ids, dis = sim.neighbours(112)
    sim.close()
    assert np.array_equal(counts, np.minimum(nf, 64) + np.minimum(nb, 48))
    listed = np.arange(112)[None, :] < counts[:, None]
    for kind, pairs, full, width in ((0, f, nf, 64), (1, b, nb, 48)):
        i, k = np.nonzero(listed & (kinds == kind))
        got = np.stack([i, ids[i, k]], 1)
        fits = full <= width
        assert np.array_equal(got[fits[got[:, 0]]], pairs[fits[pairs[:, 0]]])
        over = set(map(tuple, got[~fits[got[:, 0]]].tolist()))       # a full list keeps some of them
        assert over <= set(map(tuple, pairs[~fits[pairs[:, 0]]].tolist()))
        assert len(over) == width * np.count_nonzero(~fits)
    return nf, nb, form


@pytest.mark.parametrize("groups", [6, 8])
@pytest.mark.parametrize("n,size,twins", [
    (1, (0.3, 0.3, 0.3), 0),
    (255, (0.3, 0.3, 0.3), 3),
    (257, (2.0, 0.05, 0.05), 4),
    (1500, (2.0, 0.08, 0.08), 20),       # packed, past 48 entries
    (700, (0.13, 0.13, 0.13), 8),        # 32-bit, past 24 and 32
    (1300, (0.12, 0.12, 0.12), 5),       # past the list width
])
def test_sparse_grid(gpu, n, size, twins, groups):
    rng = np.random.default_rng(n)
    x = rng.uniform(0.02, 1.0, (n, 3)).astype(np.float32) * np.asarray(size, np.float32)
    for _ in range(twins):
        x[rng.integers(n)] = x[rng.integers(n)]
    wall = rng.uniform(0.0, 1.0, (n // 4 + 1, 3)).astype(np.float32) * np.asarray(size, np.float32)
    wall[:, 1] = 0.0
    if n > 1:
        x[0] = wall[0]
    # (34 million cells: the radix search, which the quarter builder cannot follow)
    _check(x, wall, (13.0, 13.0, 13.0), groups, 1)


def _crowd():
    rng = np.random.default_rng(2)
    n, size = 90000, np.array([2.0, 0.62, 0.62])
    x = rng.uniform(0.0, 1.0, (n, 3)) * size + 0.01
    x[:3000, 0] = 0.5 + 0.06 * x[:3000, 0]               # a denser stretch
    for _ in range(200):
        x[rng.integers(n)] = x[rng.integers(n)]
    wall = rng.uniform(0.0, 1.0, (9000, 3)) * size
    wall[:, 1] = 0.005
    return x.astype(np.float32), wall.astype(np.float32)


@pytest.mark.parametrize("groups", [6, 8])
def test_dense_grid_past_320_tiles(gpu, groups):
    x, wall = _crowd()
    nf, nb, form = _check(x, wall, (2.2, 0.8, 0.8), groups, 321)
    assert form["packed_tiles"] > 300 and np.count_nonzero(nf > 48) > 100 and nf.max() > 64


@pytest.mark.parametrize("groups", [6, 8])
@pytest.mark.parametrize("top", [(2.2, 0.8, 0.8), (13.0, 13.0, 13.0)])
def test_window_lists(gpu, groups, top):
    print(f"[list forms] windows groups {groups} {top}", flush=True)
    x, wall = _crowd()
    got = []
    for on in (False, True):
        sim = _sim(x, wall, top, groups, sg.DFSPH, min_iter_density=2, max_iter_density=2, min_iter_div=2, max_iter_div=1)
        sim.set_lds_windows(on)
        sim.step()
        got.append([sim.get(f).tobytes() for f in (sg.F_VEL, sg.F_RHO, sg.F_ALPHA, sg.F_KAPPA_SUM, sg.F_KAPPAV_SUM)])
        sim.close()
    assert got[0] == got[1]
