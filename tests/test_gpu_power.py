"""The power method's device loop against the oracle's powerIteration, on
nonnegative matrices and positive start vectors.

No sum cancels there, so every element of an iterate carries a relative error
of at most (L + 4) u per step (L entries in the longest row: one rounding per
product, L - 1 per sum, the rest for the scale), u the unit roundoff of the
vectors: after K steps and the final division (L + 4) K u + 8 u on each side,
oracle and device."""
import numpy as np
import pytest

import oracle

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu


def _matrix(kind, n, seed=3):
    rng = np.random.default_rng(seed)
    if kind == "poisson":
        A = oracle.poisson_crs(*n)
        return oracle.CRSMatrix(A.nor, A.noc, A.row_start, A.col_ind, np.abs(A.data))
    if kind == "rows":  # the given row lengths, random columns
        lens = np.asarray(n)
    else:  # "ragged": n rows, some empty, one as long as allowed
        lens = rng.integers(0, 9, n)
        lens[n // 2] = min(n, 900)
    N = len(lens)
    cols = [np.sort(rng.choice(N, k, replace=False)) for k in lens]
    rs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = np.concatenate(cols).astype(np.int32) if rs[-1] else np.zeros(0, np.int32)
    return oracle.CRSMatrix(N, N, rs, ci, rng.uniform(0.5, 1.5, rs[-1]))


# The one-workgroup loop: matrices of one row and one partial wave, just below
# and above one entry per thread, at the last FP64 and FP32 sizes that fit its
# registers or LDS and the first that do not, empty rows and a long row
SMALL = [("poisson", (1, 1)), ("poisson", (3, 1)), ("poisson", (37, 29)), ("rows", [1] * 1024), ("rows", [1] * 1025),
         ("rows", [16] * 1024), ("rows", [16] * 1024 + [1]), ("poisson", (52, 51)), ("poisson", (53, 53)),
         ("rows", [6] * 4096), ("rows", [6] * 4096 + [1]), ("poisson", (75, 75)), ("ragged", 1500)]


@pytest.mark.parametrize("values", ["f64", "f32"])
@pytest.mark.parametrize("kind,n", SMALL, ids=lambda v: str(v) if isinstance(v, (str, int, tuple)) else str(len(v)))
def test_small_power_method(kind, n, values):
    A = _matrix(kind, n)
    if values == "f32":
        A = oracle.CRSMatrix(A.nor, A.noc, A.row_start, A.col_ind, A.data.astype(np.float32).astype(np.float64))
    x0 = np.random.default_rng(1).uniform(0.5, 1.5, A.nor).astype(np.float32).astype(np.float64)
    u = 2.0 ** -53 if values == "f64" else 2.0 ** -24
    L = int(np.max(np.diff(A.row_start)))
    vt = np.float64 if values == "f64" else np.float32
    for cls in (pw.CRSHip, pw.CRSMergeHip, pw.CSBHip, pw.BlockCOHHip):
        m = cls(values=values)
        m.loadCRS(A.nor, A.noc, A.row_start, A.col_ind, A.data)
        # one step, an odd and an even count, and more than one launch's 4096
        for its in (1, 2, 25) + ((4097,) if A.nor <= 1200 and kind == "poisson" else ()):
            print(f"{cls.__name__} {kind} N={A.nor} nnz={len(A.data)} {values} its={its}", flush=True)
            xr, yr = oracle.crs_power_iteration(A, x0, its)
            x, y = pw.DeviceVector.from_array(x0, vt), pw.DeviceVector(A.nor, vt)
            lam, yn, k = m.power_method_device(x, y, its)
            bound = (L + 4) * its * (u + 2.0 ** -53) + 8 * (u + 2.0 ** -53)
            assert k == its
            for got, ref in ((x.download(), xr), (y.download(), yr)):
                if its == 1 and np.array_equal(ref, x0):
                    assert np.array_equal(got, x0.astype(vt))  # the start vector stays
                    continue
                assert np.max(np.abs(got - ref) / np.where(ref > 0, ref, 1.0)) <= bound
            # lambda and |y| of the last step, from the oracle's iterate before it
            v = xr if its % 2 else yr
            w = oracle.crs_mv(A, v)
            tol = 4 * bound + A.nor * 2.0 ** -52
            assert abs(lam - v @ w / (v @ v)) <= tol * abs(lam)
            assert abs(yn - np.linalg.norm(w) / (np.linalg.norm(v) if its > 1 else 1.0)) <= tol * yn
    # a stop test: the same steps as the fixed count it stops at
    x, y = pw.DeviceVector.from_array(x0, vt), pw.DeviceVector(A.nor, vt)
    lam, yn, k = m.power_method_device(x, y, 300, 1e-5)
    x2, y2 = pw.DeviceVector.from_array(x0, vt), pw.DeviceVector(A.nor, vt)
    lam2, yn2, k2 = m.power_method_device(x2, y2, k)
    assert k2 == k and abs(lam - lam2) <= 1e-5 * abs(lam)
    if k < 300 and k > 2:
        x3, y3 = pw.DeviceVector.from_array(x0, vt), pw.DeviceVector(A.nor, vt)
        lam3 = m.power_method_device(x3, y3, k - 1)[0]
        assert abs(lam2 - lam3) <= 1.1e-5 * abs(lam2)


# The general loop's norms: partial-sum slots of every kernel within one
# workgroup's reach, and more of them than that (wave tiles: one slot per 8
# tiles of about 250 entries; merge path and tiles: one slot a tile)
GENERAL = [("crs", pw.CRSHip, {}), ("tiles", pw.CRSHip, {"crs_kernel": 2}), ("vector", pw.CRSHip, {"crs_kernel": 1}),
           ("merge", pw.CRSMergeHip, {}), ("csb", pw.CSBHip, {}), ("coh", pw.BlockCOHHip, {})]


@pytest.mark.parametrize("side", [(80, 77), (331, 300), (2100, 2000)], ids=str)
@pytest.mark.parametrize("name,cls,opt", GENERAL, ids=[g[0] for g in GENERAL])
def test_power_steps(name, cls, opt, side):
    A = _matrix("poisson", side)
    x0 = np.random.default_rng(4).uniform(0.5, 1.5, A.nor)
    m = cls(**opt)
    m.loadCRS(A.nor, A.noc, A.row_start, A.col_ind, A.data)
    its, u = 5, 2.0 ** -53
    xr, yr = oracle.crs_power_iteration(A, x0, its)
    x, y = pw.DeviceVector.from_array(x0), pw.DeviceVector(A.nor)
    lam, yn, k = m.power_method_device(x, y, its)
    bound = 2 * (9 * its + 8) * u + 2 * A.nor * u  # the norms: N squares added in any order
    assert k == its
    for got, ref in ((x.download(), xr), (y.download(), yr)):
        assert np.max(np.abs(got - ref) / ref) <= bound
    w = oracle.crs_mv(A, xr)
    assert abs(lam - xr @ w / (xr @ xr)) <= 4 * bound * lam
    assert abs(yn - np.linalg.norm(w)) <= 4 * bound * yn
    lam2, yn2, k2 = m.power_method_device(*(pw.DeviceVector.from_array(v) for v in (x0, x0)), 40, 1e-3)
    assert 2 <= k2 <= 40 and abs(lam2 - lam) <= 0.05 * lam
