"""Large transfers borrow a pinned stage that the process's objects share: fields
of several sizes through objects in several threads at once, and through an
object made after the last one that used a stage is gone."""
import threading

import numpy as np
import pytest

from graphics_amd import sphgpu as sg

pytestmark = pytest.mark.gpu


def _round_trip(n, seed, out):
    cell = 0.0025
    sf = sg.Surfacer((0.0, 0.0, 0.0), tuple((k - 0.5) * cell - 0.03 for k in n), 0.01, 0.02, cell)
    f = np.random.default_rng(seed).normal(size=sf.grid_num[::-1]).astype(np.float32)
    for _ in range(3):
        sf.set_field(f)
        g = f.copy()
        f[:] = 0.0                           # (the source is free once the call returns)
        out.append(np.array_equal(sf.field(), g))
        f[:] = g
    sf.close()


# 1 MB and a node more, one chunk of 2 MB and a node more, more than all slots
@pytest.mark.parametrize("n", [(64, 64, 64), (65, 64, 64), (128, 64, 64), (129, 64, 64), (211, 160, 131)])
def test_one_object_after_another(gpu, n):
    print(f"[stages] {n}", flush=True)
    out = []
    _round_trip(n, 1, out)
    _round_trip(n, 2, out)
    assert out == [True] * 6


def test_several_threads(gpu):
    out = []
    threads = [threading.Thread(target=_round_trip, args=((97 + 20 * k, 90, 80), k, out)) for k in range(5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert out == [True] * 15
