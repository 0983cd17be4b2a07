"""Rows of up to 64 entries: the wave tiles run where they are the fastest.

Of 64 entries near the diagonal a lane's serial sums take twice the vector
kernel's time (CRS, FP64: 40 against 19 us) and a third more than the merge
kernel's (CRS_MERGE: 40 against 28); of 9 they are the fastest.  FP64 y within
(L + 1) 2^-52 sum |a x| of the oracle's, whose products another order adds up."""
import numpy as np
import pytest

import oracle

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,wave_tiles", [(9, True), (64, False)])
@pytest.mark.parametrize("cls", [pw.CRSHip, pw.CRSMergeHip], ids=lambda c: c.__name__)
def test_kernel_for_the_row_length(cls, L, wave_tiles):
    n = 150000
    rng = np.random.default_rng(L)
    ci = np.sort((np.arange(n)[:, None] + rng.integers(-100, 100, (n, L))) % n, axis=1).astype(np.int32)
    rs = (np.arange(n + 1) * L).astype(np.int32)
    A = oracle.CRSMatrix(n, n, rs, ci.ravel(), rng.uniform(0.1, 1.1, n * L))
    m = cls()
    m.loadCRS(n, n, rs, A.col_ind, A.data)
    info = m.info()
    if cls is pw.CRSMergeHip:
        assert info["kernels"] == (1 if wave_tiles else 2)
    else:
        assert (info["threads"] == -(-n * L // (253 - (L - 1)))) == wave_tiles, info
    x = rng.uniform(0.5, 1.5, n)
    xd, yd = pw.DeviceVector.from_array(x), pw.DeviceVector(n)
    m.mv_device(xd, yd)
    ref = oracle.crs_mv(A, x)
    assert np.all(np.abs(yd.download() - ref) <= (L + 1) * 2.0 ** -52 * ref)
    y = pw.DeviceVector(n)
    lam, _, k = m.power_method_device(xd, y, 12)
    xr, yr = oracle.crs_power_iteration(A, x, 12)
    assert k == 12 and np.max(np.abs(xd.download() - xr)) <= 1e-12 and np.max(np.abs(y.download() - yr)) <= 1e-12
