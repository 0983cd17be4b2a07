"""Infinities and NaN in x reach the rows that use them and no others.

Every kernel gathers x for entries that it then drops: those of a tile's
neighbours, lanes past a tile's or band's end, padding of windows and blocks.
x is special at the first and last columns, at the first columns of blocks and
windows and at a few more; the rows without a special column must equal those
of the same x with zeros in the special places, bit for bit where the kernel
adds in a fixed order, the others the oracle's infinities and NaN."""
import numpy as np
import pytest

import oracle

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu

KINDS = [("wave tiles", pw.CRSHip, {}), ("wave tiles merge", pw.CRSMergeHip, {}),
         ("ordered sweep", pw.CRSHip, {"csb_layout": 4}), ("sweep", pw.CSBHip, {"csb_layout": 4}),
         ("streams", pw.CSBHip, {"csb_layout": 2}), ("pieces", pw.CSBHip, {"csb_layout": 1}),
         ("coh", pw.BlockCOHHip, {"coh_occ8": 1}), ("coh single waves", pw.BlockCOHHip, {"coh_occ8": 0})]


def _matrix(n, seed):
    """Rows of 1 to 20 entries; every 7th row of the first half without entries."""
    rng = np.random.default_rng(seed)
    lens = rng.integers(1, 21, n)
    lens[:n // 2:7] = 0
    rs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    r = np.repeat(np.arange(n), lens)
    ci = rng.integers(0, n, rs[-1])
    ci = ci[np.lexsort((ci, r))].astype(np.int32)
    return oracle.CRSMatrix(n, n, rs, ci, rng.choice([-1.5, -0.5, 0.5, 1.0, 2.0], rs[-1])), r


def _special_columns(n):
    cols = {0, 1, n // 3, n - 2, n - 1}
    for bits in (10, 12, 13, 17):
        cols |= set(range(0, n, 1 << bits))
    return np.array(sorted(c for c in cols if c < n))


@pytest.mark.parametrize("values", ["f64", "f32"])
@pytest.mark.parametrize("name,cls,opt", KINDS, ids=[k[0] for k in KINDS])
@pytest.mark.parametrize("n", [1500, 40000, 300000])
def test_only_the_rows_that_use_them(n, name, cls, opt, values):
    A, r = _matrix(n, n)
    m = cls(values=values, **opt)
    m.loadCRS(n, n, A.row_start, A.col_ind, A.data)
    vt = m.vector_dtype
    x = np.random.default_rng(2).standard_normal(n).astype(vt)
    sp = _special_columns(n)
    clean, dirty = x.copy(), x.copy()
    clean[sp] = 0
    dirty[sp] = np.resize([np.inf, -np.inf, np.nan], len(sp))
    out = []
    for v in (clean, dirty):
        xd, yd = pw.DeviceVector.from_array(v, vt), pw.DeviceVector(n, vt)
        yd.fill(9.0)
        m.mv_device(xd, yd)
        out.append(yd.download().astype(np.float64))
    uses = np.zeros(n, bool)
    uses[r[np.isin(A.col_ind, sp)]] = True
    assert uses.any() and not uses.all()
    ref = oracle.crs_mv(A, dirty.astype(np.float64))
    assert np.all(np.isfinite(out[0]))
    if cls is not pw.BlockCOHHip and cls is not pw.CSBHip:
        assert np.array_equal(out[1][~uses], out[0][~uses])
    else:  # LDS sums in any order
        mag = oracle.crs_mv(oracle.CRSMatrix(n, n, A.row_start, A.col_ind, np.abs(A.data)), np.abs(clean.astype(np.float64)))
        u = 2.0 ** -52 if values == "f64" else 2.0 ** -23
        assert np.all(np.abs(out[1] - out[0])[~uses] <= 22 * u * mag[~uses])
    assert np.array_equal(np.isnan(out[1]), np.isnan(ref)) and np.array_equal(np.isinf(out[1]), np.isinf(ref))
    inf = np.isinf(ref)
    assert np.array_equal(out[1][inf], ref[inf])


@pytest.mark.parametrize("values", ["f64", "f32"])
@pytest.mark.parametrize("cls", [pw.CRSHip, pw.CRSMergeHip, pw.CSBHip, pw.BlockCOHHip], ids=lambda c: c.__name__)
def test_small_power_step(cls, values):
    """The one-workgroup power method: an infinite norm divides every finite row to
    zero and leaves NaN where a row was infinite; NaN anywhere in y makes all of it
    NaN.  Entries beyond the matrix's last gather column 0."""
    n = 40
    rs = np.arange(n + 1, dtype=np.int32)
    ci = np.roll(np.arange(n), -1).astype(np.int32)  # row i takes x[i + 1]
    m = cls(values=values)
    m.loadCRS(n, n, rs, ci, np.ones(n))
    vt = m.vector_dtype
    x0 = np.ones(n)
    x0[0] = np.inf
    x, y = pw.DeviceVector.from_array(x0, vt), pw.DeviceVector(n, vt)
    m.power_method_device(x, y, 1)
    got = y.download()
    assert np.isnan(got[n - 1]) and np.all(got[:n - 1] == 0)
    x0[0] = np.nan
    x, y = pw.DeviceVector.from_array(x0, vt), pw.DeviceVector(n, vt)
    m.power_method_device(x, y, 1)
    assert np.all(np.isnan(y.download()))
