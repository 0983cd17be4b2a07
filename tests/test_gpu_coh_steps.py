"""BlockCOH: steps of 256 entries per wave, sums in LDS or in the band's FP64 rows.

Cases where the steps' bookkeeping can go wrong: bands that begin off a multiple
of 4 entries, a step within one row, more blocks than are kept in LDS, a band cut
into atomic tasks (rows beyond the window, or many times the others' entries),
empty bands, bands of one wave each (scattered columns, x beyond 10 MB in FP64).
y is the FP64 sum of the products, rounded once; the products are
formed in the vectors' type, so against exact products each adds its own
rounding: |err| <= u_x (|y| + sum |a x|) + L 2^-52 sum |a x|, with u_x = 2^-24 for
FP32 vectors (BF16 storage too) and 2^-53 for FP64."""
import numpy as np
import pytest

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu


def _lens(kind, rng):
    if kind == "last_band":  # 64-entry rows, then a band that closes late
        lens = rng.integers(1, 40, 40000)
        lens[::97] = 1500
        return lens
    if kind == "one_row":
        lens = rng.integers(0, 5, 5000)
        lens[1234] = 40003
        return lens
    if kind == "gaps":  # empty rows around full ones
        lens = np.zeros(6000, np.int64)
        lens[5::50] = rng.integers(1, 700, 120)
        return lens
    return np.full({"tiny": 9, "blocks": 700, "wide": 120000, "waves": 66000}[kind],
                   {"tiny": 3, "blocks": 11, "wide": 4, "waves": 9}[kind])


CASES = [("tiny", 7, -1), ("blocks", 10000000, 1), ("wide", 300000, 1), ("wide", 300000, 3), ("last_band", 30011, -1),
         ("one_row", 60000, -1), ("one_row", 60000, 2), ("gaps", 4099, -1), ("gaps", 4099, 5), ("waves", 1500000, 1100)]


@pytest.mark.parametrize("values", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("kind,noc,threads", CASES, ids=lambda v: str(v))
def test_blockcoh_steps(kind, noc, threads, values):
    rng = np.random.default_rng(noc)
    lens = _lens(kind, rng)
    n = len(lens)
    rs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    r = np.repeat(np.arange(n), lens)
    ci = rng.integers(0, noc, rs[-1])
    ci = ci[np.lexsort((ci, r))].astype(np.int32)
    v = rng.standard_normal(rs[-1])
    x = rng.standard_normal(noc)
    if values == "bf16":  # values exact in BF16
        v = (v.astype(np.float32).view(np.uint32) & 0xffff0000).view(np.float32).astype(np.float64)
    vt = np.float64 if values == "f64" else np.float32
    v, x = v.astype(vt).astype(np.float64), x.astype(vt)
    p = v * x[ci]
    ref, mag = np.zeros(n), np.zeros(n)
    np.add.at(ref, r, p)
    np.add.at(mag, r, np.abs(p))
    u = 2.0 ** -53 if values == "f64" else 2.0 ** -24
    tol = u * (np.abs(ref) + mag) + 2 * lens * 2.0 ** -52 * mag + 1e-45
    m = pw.BlockCOHHip(threads, values=values)
    m.loadCRS(n, noc, rs, ci, v)
    xd, yd = pw.DeviceVector.from_array(x, vt), pw.DeviceVector(n, vt)
    for _ in range(3):
        m.mv_device(xd, yd)
        assert np.all(np.abs(yd.download().astype(np.float64) - ref) <= tol)


@pytest.mark.parametrize("threads", [-1, 1, 3])
def test_blockcoh_power_with_atomic_bands(threads):
    """Steps whose norms come from LDS bands and from the rows of atomic bands."""
    n = 40000
    rng = np.random.default_rng(2)
    lens = _lens("last_band", rng)
    rs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    r = np.repeat(np.arange(n), lens)
    ci = rng.integers(0, n, rs[-1])
    ci = ci[np.lexsort((ci, r))].astype(np.int32)
    v = rng.uniform(0.5, 1.5, rs[-1])
    x0 = rng.uniform(0.5, 1.5, n)
    m = pw.BlockCOHHip(threads)
    m.loadCRS(n, n, rs, ci, v)
    ref = pw.CRSHip(crs_kernel=2)
    ref.loadCRS(n, n, rs, ci, v)
    for its in (4, 5):
        out = []
        for A in (m, ref):
            xd, yd = pw.DeviceVector.from_array(x0), pw.DeviceVector(n)
            out.append((A.power_method_device(xd, yd, its), xd.download(), yd.download()))
        (a, xa, ya), (b, xb, yb) = out
        # positive terms: a step's relative error is about (longest row + n) 2^-53
        tol = 2 * its * (lens.max() + 512) * 2.0 ** -53
        assert abs(a[0] - b[0]) <= tol * abs(b[0])
        assert np.all(np.abs(xa - xb) <= tol * np.abs(xb)) and np.all(np.abs(ya - yb) <= tol * np.abs(yb))
