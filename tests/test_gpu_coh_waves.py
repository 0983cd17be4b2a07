"""BlockCOH tasks by workgroups of 8 waves or by single waves: the option
coh_occ8 chooses (reported as high_occupancy), by default the faster is kept.

Rows of L columns, one random one in each L-th of x, 24 M entries.  Single waves
are a quarter faster at L = 6 (x of 32 MB) and an eighth slower at L = 16 (12 MB).
y within (L + 1) 2^-52 sum |a x| of FP64 sums in another order."""
import numpy as np
import pytest

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,waves8", [(6, 0), (16, 1)])
def test_faster_one_is_kept(L, waves8):
    n = 24_000_000 // L
    rng = np.random.default_rng(L)
    cols = (rng.integers(0, n // L, (n, L)) + np.arange(L) * (n // L)).astype(np.int32)
    vals = rng.uniform(-1, 1, (n, L))
    rs = (np.arange(n + 1, dtype=np.int64) * L).astype(np.int32)
    x = rng.uniform(-1, 1, n)
    p = vals * x[cols]
    ref, bound = p.sum(axis=1), (L + 1) * 2.0 ** -52 * np.abs(p).sum(axis=1)
    xd, yd = pw.DeviceVector.from_array(x), pw.DeviceVector(n)
    for option in (-1, 0, 1):
        m = pw.BlockCOHHip(coh_occ8=option)
        m.loadCRS(n, n, rs, cols.ravel(), vals.ravel())
        assert m.info()["high_occupancy"] == (waves8 if option < 0 else option)
        yd.fill(9.0)
        m.mv_device(xd, yd)
        assert np.all(np.abs(yd.download() - ref) <= bound)
        del m
