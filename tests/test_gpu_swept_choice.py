"""When CRS and CRS_MERGE handles keep swept slabs beside their CRS arrays."""
import numpy as np
import pytest

import oracle

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu
CLASSES = pytest.mark.parametrize("cls", [pw.CRSHip, pw.CRSMergeHip], ids=lambda c: c.__name__)


def _swept(m):
    """A second copy of the entries is held (a CRS entry takes 12 bytes, the plans less than 4)."""
    i = m.info()
    return i["device_bytes"] >= 20 * i["nnz"]


@CLASSES
def test_asked_for_on_a_generated_matrix(cls):
    m, ref = cls(csb_layout=4), cls(csb_layout=1)
    for a in (m, ref):
        a.generatePoissonMatrix(300, 200)
    assert _swept(m) and not _swept(ref)
    x = np.random.default_rng(1).standard_normal(60000)
    y, z = np.zeros(60000), np.zeros(60000)
    m.mv(x, y)
    ref.mv(x, z)
    # five products each, added in another order
    P = oracle.poisson_crs(300, 200)
    P.data = np.abs(P.data)
    assert np.all(np.abs(y - z) <= 6 * 2.0 ** -52 * oracle.crs_mv(P, np.abs(x)))
