"""Power steps whose norms the next step adds up, against steps with a reduction.

A fixed number of steps (tol < 0) defers the norms where a step has at most 1280
partial-sum slots; with a stop test (tol = 0, which positive data does not meet)
every step reduces its own.  The two add the same slots in another order: with
positive values a step's scale differs by at most about 64 roundings, its row
sums (LDS sums take any order) by L, so x, y, lambda and the norm agree within
its (L + 64) 2^-52.  Sizes below and above each change of the block size and the
last size that defers."""
import numpy as np
import pytest

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu

L = 5
# tiles of 249 entries: 2048 tiles at 101990 rows, 10240 at 509952
SIZES = [9000, 101990, 102100, 509900, 510100]


@pytest.mark.parametrize("values", ["f64", "f32"])
@pytest.mark.parametrize("cls", [pw.CRSHip, pw.CRSMergeHip, pw.CSBHip, pw.BlockCOHHip], ids=lambda c: c.__name__)
@pytest.mark.parametrize("n", SIZES)
def test_deferred_norms(cls, n, values):
    rng = np.random.default_rng(n)
    rs = (np.arange(n + 1) * L).astype(np.int32)
    ci = np.sort((np.arange(n)[:, None] + rng.integers(-40, 40, (n, L))) % n, axis=1).astype(np.int32).ravel()
    vt = np.float64 if values == "f64" else np.float32
    v = rng.uniform(0.5, 1.5, n * L).astype(vt).astype(np.float64)
    x0 = rng.uniform(0.5, 1.5, n).astype(vt)
    A = cls(values=values)
    A.loadCRS(n, n, rs, ci, v)
    u = 2.0 ** -52 if values == "f64" else 2.0 ** -23
    for its in (1, 2, 7):
        out = []
        for tol in (-1.0, 0.0):
            xd, yd = pw.DeviceVector.from_array(x0, vt), pw.DeviceVector(n, vt)
            r = A.power_method_device(xd, yd, its, tol)
            out.append((list(r), xd.download().astype(np.float64), yd.download().astype(np.float64)))
        (ra, xa, ya), (rb, xb, yb) = out
        tol = its * (L + 64) * u
        assert np.all(np.abs(np.array(ra, float) - np.array(rb, float)) <= tol * np.abs(np.array(rb, float))), (ra, rb)
        assert np.all(np.abs(xa - xb) <= tol * np.abs(xb)) and np.all(np.abs(ya - yb) <= tol * np.abs(yb))
