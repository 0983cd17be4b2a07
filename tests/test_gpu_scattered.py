"""The CRS formats' sweep over scattered columns: swept slabs beside the CRS
arrays (csb_layout = 4 asks for them), the waves adding in turn.

FP64 y within (L + 1) 2^-52 sum |a x| of the oracle's (two sums of L products in
different orders), FP32 within 2^-24 |sum| more (FP64 sums of FP32 products);
every repetition equal bit for bit; the CRS arrays still exported."""
import numpy as np
import pytest

import oracle

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu


def _crs(lens, noc, seed, cols=None):
    rng = np.random.default_rng(seed)
    lens = np.asarray(lens)
    rs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    r = np.repeat(np.arange(len(lens)), lens)
    ci = rng.integers(0, noc, rs[-1]) if cols is None else cols(rng, rs[-1])
    ci = ci[np.lexsort((ci, r))].astype(np.int32)  # duplicates kept
    v = rng.standard_normal(rs[-1]).astype(np.float32).astype(np.float64)
    return oracle.CRSMatrix(len(lens), noc, rs, ci, v)


def _cases():
    rng = np.random.default_rng(1)
    yield "one entry", [1], 1, None
    yield "one window", rng.integers(0, 9, 5000), 4000, None
    yield "wide", rng.integers(1, 40, 60000), 600000, None
    yield "tall", rng.integers(0, 12, 300000), 70000, None
    # a row longer than a slab's share, beside empty ones
    yield "long row", [90000] + [0] * 500 + [3] * 20000 + [50000], 150000, None
    # every entry in the last columns of a window, and windows without entries
    yield "one column band", [20] * 30000, 500000, lambda g, n: 262100 + g.integers(0, 60, n)
    # runs of several rounds of 16 x 512 entries
    yield "many rounds", [600] * 9000, 131072, None


CASES = list(_cases())


@pytest.mark.parametrize("values", ["f64", "f32"])
@pytest.mark.parametrize("cls", [pw.CRSHip, pw.CRSMergeHip], ids=lambda c: c.__name__)
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_sweep_in_turns(case, cls, values):
    name, lens, noc, cols = case
    A = _crs(lens, noc, 7, cols)
    m = cls(values=values, csb_layout=4)
    m.loadCRS(A.nor, A.noc, A.row_start, A.col_ind, A.data)
    assert m.info()["kernels"] == 1 and m.info()["device_bytes"] >= 24 * len(A.data) * (1 if values == "f64" else 0.6)
    x = np.random.default_rng(2).standard_normal(noc).astype(np.float32).astype(np.float64)
    vt = np.float64 if values == "f64" else np.float32
    xd, yd = pw.DeviceVector.from_array(x, vt), pw.DeviceVector(A.nor, vt)
    yd.fill(5.0)
    m.mv_device(xd, yd)
    got, ref = yd.download(), oracle.crs_mv(A, x)
    mag = oracle.crs_mv(oracle.CRSMatrix(A.nor, A.noc, A.row_start, A.col_ind, np.abs(A.data)), np.abs(x))
    L = np.diff(A.row_start)
    bound = (L + 1) * 2.0 ** -52 * mag
    if values == "f32":
        bound = bound + 2.0 ** -24 * (np.abs(ref) + mag) * (1 + 2.0 ** -20)
    assert np.all(np.abs(got - ref) <= bound)
    for _ in range(10):
        m.mv_device(xd, yd)
        assert np.array_equal(yd.download(), got)
    rs, ci, dv = m.crs_export()
    assert np.array_equal(rs, A.row_start) and np.array_equal(ci, A.col_ind) and np.array_equal(dv, A.data)


@pytest.mark.parametrize("cls", [pw.CRSHip, pw.CRSMergeHip], ids=lambda c: c.__name__)
def test_sweep_power_steps(cls):
    A = _crs(np.random.default_rng(3).integers(1, 30, 20000), 20000, 8)
    A.data = np.abs(A.data) + 0.1
    m = cls(csb_layout=4)
    m.loadCRS(A.nor, A.noc, A.row_start, A.col_ind, A.data)
    x0 = np.random.default_rng(4).uniform(0.5, 1.5, A.nor)
    xr, yr = oracle.crs_power_iteration(A, x0, 7)
    first = None
    for _ in range(3):
        x, y = pw.DeviceVector.from_array(x0), pw.DeviceVector(A.nor)
        lam, yn, k = m.power_method_device(x, y, 7)
        # nonnegative sums: (L + 4) u per step on either side, and the norms
        bound = 2 * (34 * 7 + 8 + A.nor) * 2.0 ** -53
        for got, ref in ((x.download(), xr), (y.download(), yr)):
            assert np.max(np.abs(got - ref) / np.where(ref > 0, ref, 1.0)) <= bound
        res = (lam, yn, k, x.download().tobytes())
        assert first in (None, res)
        first = res


def test_scattered_columns_are_swept_and_banded_ones_are_not():
    n = 1 << 20
    for cls in (pw.CRSHip, pw.CRSMergeHip):
        A = _crs([100] * (n // 20), n, 5)
        m = cls()
        m.loadCRS(A.nor, A.noc, A.row_start, A.col_ind, A.data)
        swept = m.info()["device_bytes"] >= 24 * len(A.data)
        off = cls(csb_layout=1)
        off.loadCRS(A.nor, A.noc, A.row_start, A.col_ind, A.data)
        assert off.info()["device_bytes"] < 20 * len(A.data)
        x, y, z = (pw.DeviceVector.from_array(np.random.default_rng(1).standard_normal(k)) for k in (n, A.nor, A.nor))
        m.mv_device(x, y)
        off.mv_device(x, z)
        print(cls.__name__, "swept", swept, m.info(), flush=True)
        assert np.max(np.abs(y.download() - z.download())) <= 1e-13 * np.max(np.abs(z.download()))
        P = oracle.poisson_crs(1000, 800)
        p = cls()
        p.loadCRS(P.nor, P.noc, P.row_start, P.col_ind, P.data)
        assert p.info()["device_bytes"] < 20 * len(P.data)
