"""A borrowed pinned stage of up to a chunk has the size of the transfer's next
power of two: transfers that outgrow it, and smaller ones after them, through
objects that share it."""
import numpy as np
import pytest

from graphics_amd import sphgpu as sg

pytestmark = pytest.mark.gpu


# past the object's own 64 KB, 128 KB and a node more, up to 1 MB, a chunk of
# 2 MB, a node row past it, and back
SIZES = [(26, 26, 25), (32, 32, 32), (33, 32, 32), (64, 64, 63), (128, 64, 64), (129, 64, 64), (32, 32, 33), (26, 26, 25)]


@pytest.mark.parametrize("sizes", [SIZES, SIZES[::-1]])
def test_growing_and_smaller_transfers(gpu, sizes):
    cell, alive, want = 0.0025, [], []
    for k, n in enumerate(sizes):
        print(f"[small stages] {n}", flush=True)
        sf = sg.Surfacer((0.0, 0.0, 0.0), tuple((m - 0.5) * cell - 0.03 for m in n), 0.01, 0.02, cell)
        f = np.random.default_rng(k).normal(size=sf.grid_num[::-1]).astype(np.float32)
        sf.set_field(f)
        alive.append(sf)
        want.append(f)
        for s, g in zip(alive, want):
            assert np.array_equal(s.field(), g)
    for s in alive:
        s.close()
