"""The gradient kernel and its slices at the sizes where
their splits change: below, at and above one tile of 16 samples, one slice of
64, and the line where the slices go from 64 to 128 samples; and inputs that
pass through the staging ring in one and in several pieces."""
import numpy as np
import pytest

from graphics_amd import sphgpu as sg
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def _data(n, seed):
    rng = np.random.default_rng(seed)
    feat = rng.normal(size=(n, 8)).astype(np.float32)
    tgt = (np.sin(feat[:, 0]) + 0.5 * feat[:, 1] * feat[:, 2]).astype(np.float32)
    return feat, tgt


# 512 slices of 64 up to 32,768 samples, from there on slices of 128
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 129, 32768, 32769, 40000])
def test_gradient_at_split_edges(gpu, n):
    """Gradient and loss against FP64 with the same BF16 rounding points; the
    tolerances are those the whole-batch gradient test of the kernels holds."""
    print(f"[mlp batches] n={n}", flush=True)
    feat, tgt = _data(n, n)
    m = sg.Mlp(40000, seed=7)
    m.set_loss(2.0)
    p = m.get_params().astype(np.float64)
    g, loss = m.gradient(feat, tgt)
    gref, lref = mo.gradient(p, feat, tgt, bf=True, over=2.0)
    assert loss == pytest.approx(lref, rel=2e-3)
    assert np.linalg.norm(g - gref) / np.linalg.norm(gref) < 2e-2
    again, loss2 = m.gradient(feat, tgt)
    assert np.array_equal(g, again) and loss == loss2
    m.close()


@pytest.mark.parametrize("cap,n", [(1000, 1000), (1000, 2500), (700000, 600001)])
def test_forward_through_the_ring(gpu, cap, n):
    """Every row of a batch that is cut by the capacity (2,500 rows in pieces
    of 1,000) or by the ring's chunks (19 MB of features): equal to the row
    evaluated in a batch of its own, bit for bit."""
    print(f"[mlp batches] forward cap={cap} n={n}", flush=True)
    feat, _ = _data(n, 3)
    m = sg.Mlp(cap, seed=9)
    y = m.forward(feat)
    for a in (0, n // 2, max(0, n - 100)):
        assert np.array_equal(y[a:a + 100], m.forward(feat[a:a + 100]))
    m.close()
