"""Matrices near the partial-sum slots of the no-allocation power method's fixed
workspace (PWM_NOALLOC_MAX_SLOTS) stay within them.

CRS_MERGE, rows of 27 entries and one of 64: a slot of the merge kernels is a tile
of 2048 merge items, 211 919 slots for the 419 M entries here; the wave tiles that
such rows take must not need more than the workspace holds.

BlockCOH in one band: 32 768 entries a task would make 23 463 slots of the 769 M
entries here; tasks of 4096 entries and pieces of 2048 rows make 263 K."""
import numpy as np
import pytest

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu


def test_short_rows():
    n, L = 15_500_000, 27
    lens = np.full(n, L)
    lens[0] = 64
    rs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = np.concatenate([np.arange(64), (np.minimum(np.arange(1, n), n - L)[:, None] + np.arange(L)).ravel()])
    m = pw.CRSMergeHip(values="f32")
    m.loadCRS(n, n, rs, ci.astype(np.int32), np.ones(len(ci)))
    assert m.info()["kernels"] == 1  # the wave tiles
    x, y = (pw.DeviceVector(n, np.float32) for _ in range(2))
    x.fill(1.0)
    lam, norm, k = m.power_method_device_noalloc(x, y, 1)
    # whole row sums; one rounding of the norm's square root
    assert k == 1 and lam == len(ci) / n
    assert abs(norm - np.sqrt(float(L * L * (n - 1) + 64 * 64))) <= 2.0 ** -52 * norm
    ref = (x.download(), y.download())
    x.fill(1.0)
    assert (lam, norm, k) == m.power_method_device(x, y, 1)
    assert np.array_equal(x.download(), ref[0]) and np.array_equal(y.download(), ref[1])


def test_one_band():
    m, n = 12400, 12400
    A = pw.BlockCOHHip(1, "bf16")
    A.generatePoissonMatrix(m, n)
    assert A.info()["threads"] == 1
    x, y = (pw.DeviceVector(m * n, np.float32) for _ in range(2))
    x.fill(1.0)
    lam, norm, k = A.power_method_device_noalloc(x, y, 1)
    # A 1 is the number of missing neighbours: 1 on the edges, 2 in the corners
    assert k == 1 and lam == 2.0 * (m + n) / (m * n)
    assert abs(norm ** 2 - (2 * (m + n - 4) + 16)) <= 1e-12 * norm ** 2
    g = y.download().reshape(n, m)  # divided by its norm: the power method's result
    assert not g[1:-1, 1:-1].any() and np.allclose(g[0, 1:-1] * norm, 1.0, rtol=1e-6)
