"""Matrices without entries, and with long stretches of rows without any: y is
written, with zeros, on every format (BlockCOH puts more empty rows than its LDS
window holds into bands that have no task of their own)."""
import numpy as np
import pytest

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("values", ["f64", "f32"])
@pytest.mark.parametrize("nor,full", [(4096, 0), (4097, 0), (8193, 0), (30000, 0), (30000, 5), (30000, 29995)])
@pytest.mark.parametrize("cls,threads", [(pw.CRSHip, -1), (pw.CRSMergeHip, -1), (pw.CSBHip, -1), (pw.BlockCOHHip, -1),
                                         (pw.BlockCOHHip, 1)], ids=lambda v: getattr(v, "__name__", str(v)))
def test_rows_without_entries(cls, threads, nor, full, values):
    noc = 700
    lens = np.zeros(nor, np.int64)
    lens[:full] = 1 if full > 5 else 300
    rs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = (np.arange(rs[-1]) % 300).astype(np.int32)
    m = cls(threads, values)
    m.loadCRS(nor, noc, rs, ci, np.ones(rs[-1]))
    vt = m.vector_dtype
    x, y = pw.DeviceVector(noc, vt), pw.DeviceVector(nor, vt)
    x.fill(1.0)
    for _ in range(2):
        y.fill(7.0)
        m.mv_device(x, y)
        assert np.array_equal(y.download(), lens.astype(vt))
