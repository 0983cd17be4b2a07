"""When CRS and CRS_MERGE handles keep swept slabs beside their CRS arrays."""
import numpy as np
import pytest

import oracle

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu
CLASSES = pytest.mark.parametrize("cls", [pw.CRSHip, pw.CRSMergeHip], ids=lambda c: c.__name__)


def _swept(m):
    """A second copy of the entries is held (a CRS entry takes 12 bytes, the plans less than 4)."""
    i = m.info()
    return i["device_bytes"] >= 20 * i["nnz"]


@CLASSES
def test_asked_for_on_a_generated_matrix(cls):
    m, ref = cls(csb_layout=4), cls(csb_layout=1)
    for a in (m, ref):
        a.generatePoissonMatrix(300, 200)
    assert _swept(m) and not _swept(ref)
    x = np.random.default_rng(1).standard_normal(60000)
    y, z = np.zeros(60000), np.zeros(60000)
    m.mv(x, y)
    ref.mv(x, z)
    # five products each, added in another order
    P = oracle.poisson_crs(300, 200)
    P.data = np.abs(P.data)
    assert np.all(np.abs(y - z) <= 6 * 2.0 ** -52 * oracle.crs_mv(P, np.abs(x)))


def _scattered(n, L, seed):
    """Rows of L columns, a random one in each L-th of x."""
    rng = np.random.default_rng(seed)
    cols = (rng.integers(0, n // L, (n, L)) + np.arange(L) * (n // L)).astype(np.int32)
    v = rng.choice([-2.0, -0.5, 0.25, 1.0, 3.0], (n, L))  # exact in every type
    return (np.arange(n + 1) * L).astype(np.int32), cols, v


@pytest.mark.parametrize("values", ["f64", "f32", "bf16"])
@CLASSES
def test_scattered_columns(cls, values):
    # 9.6 MB of x in FP64 and 12 MB in FP32, where the sweep takes less than half the time
    n, L = (1200000, 16) if values == "f64" else (3000000, 16)
    rs, cols, v = _scattered(n, L, 3)
    m = cls(values=values)
    m.loadCRS(n, n, rs, cols.ravel(), v.ravel())
    es = 4 + {"f64": 8, "f32": 4, "bf16": 2}[values]
    assert m.info()["device_bytes"] >= 1.9 * es * n * L, m.info()
    vt = m.vector_dtype
    x = np.random.default_rng(4).standard_normal(n).astype(vt)
    xd, yd = pw.DeviceVector.from_array(x, vt), pw.DeviceVector(n, vt)
    yd.fill(5.0)
    m.mv_device(xd, yd)
    got = yd.download()
    p = v * x.astype(np.float64)[cols]
    ref, mag = p.sum(axis=1), np.abs(p).sum(axis=1)
    # FP64 sums in two orders; FP32: products (exact but for 3.0) and the result rounded
    bound = (L + 1) * 2.0 ** -52 * mag + (0 if values == "f64" else 2.0 ** -24 * (1 + 2.0 ** -20) * (np.abs(ref) + mag))
    assert np.all(np.abs(got - ref) <= bound)
    for _ in range(3):
        m.mv_device(xd, yd)
        assert np.array_equal(yd.download(), got)


@CLASSES
def test_not_kept_where_memory_is_taken(cls):
    n, L = 1200000, 16
    rs, cols, v = _scattered(n, L, 5)
    taken = pw.DeviceVector(10_000_000_000)  # 80 GB of 288
    m = cls()
    m.loadCRS(n, n, rs, cols.ravel(), v.ravel())
    assert not _swept(m)
    taken.free()
    again = cls()
    again.loadCRS(n, n, rs, cols.ravel(), v.ravel())
    assert _swept(again)
