"""BlockCOH power steps with deferred norms divide every row by the same norm.

A multiple of the identity, padded with stored zeros, keeps a constant vector
constant: its rows must stay equal bit for bit, those of a band that is cut
into atomic tasks (the last row, 12 001 entries) and those of LDS bands, for
single waves and workgroups of 8, whose blocks add the slots in other orders."""
import numpy as np
import pytest

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("option", [0, 1])
@pytest.mark.parametrize("threads", [70, 500, 1200])
def test_constant_vector_stays_constant(threads, option):
    n, L = 20000, 4
    rng = np.random.default_rng(threads)
    cols = (np.arange(n)[:, None] + np.arange(L)) % n
    vals = np.zeros((n, L))
    vals[:, 0] = 0.7
    order = np.argsort(cols, axis=1)
    cols, vals = np.take_along_axis(cols, order, 1), np.take_along_axis(vals, order, 1)
    ci = np.concatenate([cols[:-1].ravel(), np.arange(n - 12001, n)]).astype(np.int32)
    v = np.concatenate([vals[:-1].ravel(), np.zeros(12000), [0.7]])
    rs = np.concatenate([np.arange(n) * L, [len(ci)]]).astype(np.int32)
    m = pw.BlockCOHHip(threads, coh_occ8=option)
    m.loadCRS(n, n, rs, ci, v)
    info = m.info()
    assert info["kernels"] == 2 and info["high_occupancy"] == option  # a band is cut
    for its in (2, 3, 20):
        x, y = pw.DeviceVector.from_array(np.full(n, rng.uniform(0.1, 1.0))), pw.DeviceVector(n)
        m.power_method_device(x, y, its)
        for z in (x.download(), y.download()):
            assert np.all(z == z[0])
