"""Wave tiles (k_rows) of CRS and CRS_MERGE handles: SpMV against the oracle.

A lane sums a row's products left to right in the vector's type, as the
oracle does in FP64, so FP64 results are equal bit for bit.  FP32: products and
L additions, each rounded, stay within (L + 1) 2^-24 sum |a x| (L entries in the
row; x and the values are exact in FP32)."""
import numpy as np
import pytest

import oracle

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu


def _crs(lens, noc, seed=5):
    rng = np.random.default_rng(seed)
    lens = np.asarray(lens)
    rs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = rng.integers(0, noc, rs[-1])
    r = np.repeat(np.arange(len(lens)), lens)
    ci = ci[np.lexsort((ci, r))].astype(np.int32)  # duplicates kept
    v = rng.standard_normal(rs[-1]).astype(np.float32).astype(np.float64)
    return oracle.CRSMatrix(len(lens), noc, rs, ci, v)


def _cases():
    rng = np.random.default_rng(9)
    yield "one row", [7], 5, True
    yield "one entry", [1], 1, True
    yield "longest row taken", [64] * 40, 1000, True
    yield "row too long", [64] * 40 + [65], 1000, False
    yield "128 rows a tile", [2] * 5000, 5000, True
    yield "more rows than a tile takes", [1] * 5000, 5000, False
    yield "empty rows", np.where(rng.random(20000) < 0.4, 0, rng.integers(4, 20, 20000)), 300, True
    yield "empty tail", [9] * 1000 + [0] * 60, 77, True
    yield "mixed", rng.integers(1, 65, 9001), 12345, True
    # whole stretches of 8 x 256 tiles and a remainder; one tile less, one more
    yield "block order", [5] * (50 * 2048 + 777), 4001, True
    yield "stretch", [8] * (31 * 2048), 4001, True
    yield "stretch and one", [8] * (31 * 2048 + 1), 4001, True


CASES = list(_cases())


@pytest.mark.parametrize("values", ["f64", "f32"])
@pytest.mark.parametrize("nt", [0, 1])
@pytest.mark.parametrize("cls", [pw.CRSHip, pw.CRSMergeHip], ids=lambda c: c.__name__)
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_wave_tiles(case, cls, nt, values):
    name, lens, noc, taken = case
    A = _crs(lens, noc)
    x = np.random.default_rng(2).standard_normal(noc).astype(np.float32).astype(np.float64)
    m = cls(values=values, crs_nt=nt)
    m.loadCRS(A.nor, A.noc, A.row_start, A.col_ind, A.data)
    info = m.info()
    if cls is pw.CRSHip:
        step = 253 - (int(np.max(lens)) - 1)
        assert info["threads"] == -(-len(A.data) // step) or not taken, info
    assert (info["kernels"] == 1 and info["non_temporal"] == nt and info["group_size"] == 0) or not taken, info
    vt = np.float64 if values == "f64" else np.float32
    xd, yd = pw.DeviceVector.from_array(x, vt), pw.DeviceVector(A.nor, vt)
    yd.fill(3.0)
    m.mv_device(xd, yd)
    got, ref = yd.download(), oracle.crs_mv(A, x)
    if values == "f64" and taken:
        assert np.array_equal(got, ref)
        return
    bound = oracle.crs_mv(oracle.CRSMatrix(A.nor, A.noc, A.row_start, A.col_ind, np.abs(A.data)), np.abs(x))
    u = 2.0 ** -24 if values == "f32" else 2.0 ** -52
    assert np.all(np.abs(got - ref) <= (np.diff(A.row_start) + 1) * u * bound)
