"""FP32 row sums of the wave tiles and the one-workgroup power method.

Rows of up to 15 entries are FP64 sums of FP32 products: with the products'
rounding and the result's, within u (sum |a x| + |y|), u = 2^-24.  Of longer
rows 16 entries at a time go through two FP32 additions each: 2 u sum |a x|
more.  All data positive, where a left-to-right FP32 sum drifts furthest."""
import numpy as np
import pytest

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu

U = 2.0 ** -24 * (1 + 2.0 ** -20)


def _matrix(n, L, seed):
    rng = np.random.default_rng(seed)
    ci = np.sort(rng.integers(0, n, (n, L)), axis=1).astype(np.int32)
    v = rng.uniform(0.5, 1.5, (n, L)).astype(np.float32).astype(np.float64)
    x = rng.uniform(0.5, 1.5, n).astype(np.float32)
    rs = (np.arange(n + 1) * L).astype(np.int32)
    return rs, ci, v, x, (v * x.astype(np.float64)[ci]).sum(axis=1)


@pytest.mark.parametrize("L", [5, 15, 16, 37, 64])
@pytest.mark.parametrize("cls", [pw.CRSHip, pw.CRSMergeHip], ids=lambda c: c.__name__)
def test_wave_tiles(cls, L):
    n = min(40000, 500000 // L)  # small: the wave tiles run whatever L is
    rs, ci, v, x, ref = _matrix(n, L, L)
    m = cls(values="f32")
    m.loadCRS(n, n, rs, ci.ravel(), v.ravel())
    xd, yd = pw.DeviceVector.from_array(x, np.float32), pw.DeviceVector(n, np.float32)
    m.mv_device(xd, yd)
    assert m.info()["kernels"] == 1 and m.info()["group_size"] == 0
    err = np.abs(yd.download() - ref) / ref
    print(cls.__name__, L, "largest error", err.max(), flush=True)
    assert err.max() <= (2 if L < 16 else 4) * U


@pytest.mark.parametrize("n,L", [(1500, 15), (300, 64)])
@pytest.mark.parametrize("cls", [pw.CRSHip, pw.CRSMergeHip, pw.CSBHip, pw.BlockCOHHip], ids=lambda c: c.__name__)
def test_small_power_step(cls, n, L):
    rs, ci, v, x, ref = _matrix(n, L, L)
    m = cls(values="f32")
    m.loadCRS(n, n, rs, ci.ravel(), v.ravel())
    xd, yd = pw.DeviceVector.from_array(x, np.float32), pw.DeviceVector(n, np.float32)
    _, norm, _ = m.power_method_device(xd, yd, 1)
    # one more rounding: y is left divided by its norm, which is the FP64 norm
    # of the rounded sums and exact to far less than u
    err = np.abs(yd.download().astype(np.float64) * norm - ref) / ref
    print(cls.__name__, L, "largest error", err.max(), flush=True)
    assert err.max() <= (3 if L < 16 else 5) * U
