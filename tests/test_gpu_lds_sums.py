"""CSB and BlockCOH with FP32 storage: rows are summed in LDS in FP64.

y is then the FP64 sum of the FP32-rounded products, rounded once: within
2^-24 |sum| of it, plus the FP64 sums' own L 2^-52 sum |a x|.  Swept slabs with
more rows than fit in FP64 sum in FP32: (L + 1) 2^-24 sum |a x|."""
import numpy as np
import pytest

import oracle

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu


def _matrix(n, noc, lens, seed):
    rng = np.random.default_rng(seed)
    rs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    r = np.repeat(np.arange(n), lens)
    ci = rng.integers(0, noc, rs[-1])
    ci = ci[np.lexsort((ci, r))].astype(np.int32)
    v = rng.standard_normal(rs[-1]).astype(np.float32)
    x = rng.standard_normal(noc).astype(np.float32)
    p = (v * x[ci]).astype(np.float64)  # FP32 products
    y = np.zeros(n)
    np.add.at(y, r, p)
    mag = np.zeros(n)
    np.add.at(mag, r, np.abs(p))
    return rs, ci, v.astype(np.float64), x, y, mag


LAYOUTS = [("csb", pw.CSBHip, {"csb_layout": k, "csb_groups": 1}) for k in (1, 2, 3)] + \
          [("csb_swept", pw.CSBHip, {"csb_layout": 4}), ("csb_swept_rows", pw.CSBHip, {"csb_layout": 4, "csb_sweep_order": 0}),
           ("coh", pw.BlockCOHHip, {})]


# a band of BlockCOH with threads = 1 holds all rows: 4096 and 8192 are the
# most an LDS window takes; 30000 rows fill several CSB slabs of 4096
@pytest.mark.parametrize("n,threads", [(4096, 1), (8192, 1), (30000, -1)])
@pytest.mark.parametrize("name,cls,opt", LAYOUTS, ids=[f"{l[0]}{l[2].get('csb_layout', '')}" for l in LAYOUTS])
def test_fp32_rows_are_summed_in_fp64(name, cls, opt, n, threads):
    lens = np.random.default_rng(n).integers(0, 8 if threads == 1 else 40, n)
    lens[5] = 3000
    rs, ci, v, x, ref, mag = _matrix(n, 5000, lens, 11)
    m = cls(threads, values="f32", **opt)
    m.loadCRS(n, 5000, rs, ci, v)
    xd, yd = pw.DeviceVector.from_array(x, np.float32), pw.DeviceVector(n, np.float32)
    m.mv_device(xd, yd)
    if name == "coh" and threads == 1 and len(ci) > 16 * 2048:
        pytest.skip("the band is too long for one LDS task")
    got = yd.download().astype(np.float64)
    assert np.all(np.abs(got - ref) <= 2.0 ** -24 * np.abs(ref) + lens * 2.0 ** -52 * mag + 1e-45)


@pytest.mark.parametrize("n", [5177344, 5300000])
def test_swept_slabs_beyond_the_fp64_rows(n):
    """256 slabs of 20224 FP64 rows hold 5 177 344 rows; more take FP32 sums."""
    lens = np.ones(n, np.int64)
    lens[::1000] = 9
    rs, ci, v, x, ref, mag = _matrix(n, 70000, lens, 3)
    m = pw.CSBHip(values="f32", csb_layout=4)
    m.loadCRS(n, 70000, rs, ci, v)
    assert m.info()["layout"] == 4
    xd, yd = pw.DeviceVector.from_array(x, np.float32), pw.DeviceVector(n, np.float32)
    m.mv_device(xd, yd)
    got = yd.download().astype(np.float64)
    assert np.all(np.abs(got - ref) <= (lens + 1) * 2.0 ** -24 * mag + 1e-45)
