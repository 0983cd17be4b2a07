"""mv and powerIteration on host arrays against the same call on device vectors.

The transfers are staged through pinned buffers: lengths up to and above what
the calling thread copies alone (1 MB), chunks and their remainders, one 64 MB
buffer, and more than both buffers hold.  CRS results repeat bit for bit,
so the two calls' agree exactly; the guards around y stay."""
import numpy as np
import pytest

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu

GRIDS = [(1, 1), (127, 129), (256, 512), (257, 512), (512, 512), (513, 513), (1025, 1024), (2049, 2048), (4096, 2048),
         (4097, 2049), (4200, 4100)]


@pytest.mark.parametrize("values", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("m,n", GRIDS, ids=lambda v: str(v))
def test_mv_on_host_arrays(m, n, values):
    N = m * n
    if values == "bf16" and N > 1 << 20:
        pytest.skip("BF16 vectors are FP32: the FP32 case covers their transfers")
    A = pw.CRSHip(values=values, crs_nt=0)
    A.generatePoissonMatrix(m, n)
    rng = np.random.default_rng(N)
    vt = np.float64 if values == "f64" else np.float32
    for _ in range(2):
        x = rng.standard_normal(N)
        buf = np.full(N + 64, 7.0)
        A.mv(x, buf[32:32 + N])
        xd, yd = pw.DeviceVector.from_array(x, vt), pw.DeviceVector(N, vt)
        A.mv_device(xd, yd)
        assert np.array_equal(buf[32:32 + N], yd.download().astype(np.float64))
        assert np.all(buf[:32] == 7.0) and np.all(buf[32 + N:] == 7.0)


@pytest.mark.parametrize("m,n", [(128, 129), (1025, 1024)], ids=lambda v: str(v))
def test_power_iteration_on_host_arrays(m, n):
    A = pw.CRSHip(crs_nt=0)
    A.generatePoissonMatrix(m, n)
    x0 = np.random.default_rng(1).uniform(0.5, 1.5, m * n)
    for its in (4, 5):
        x, y = x0.copy(), np.zeros(m * n)
        A.powerIteration(x, y, its)
        xd, yd = pw.DeviceVector.from_array(x0), pw.DeviceVector(m * n)
        A.power_method_device(xd, yd, its)
        assert np.array_equal(x, xd.download()) and np.array_equal(y, yd.download())


def test_transfers_from_two_threads():
    """Two handles in two threads share the staging buffers and the host pool."""
    import threading
    out = {}

    def work(k):
        A = pw.CRSHip(crs_nt=0)
        A.generatePoissonMatrix(700 + k, 900)
        x = np.random.default_rng(k).standard_normal((700 + k) * 900)
        xd, yd = pw.DeviceVector.from_array(x), pw.DeviceVector(len(x))
        A.mv_device(xd, yd)
        ref, y = yd.download(), np.zeros(len(x))
        ok = True
        for _ in range(20):
            y[:] = 0
            A.mv(x, y)
            ok = ok and np.array_equal(y, ref)
        out[k] = ok

    ts = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert out == {0: True, 1: True, 2: True}
