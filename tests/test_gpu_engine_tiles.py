"""The batch engine's tiles of 256 x 16 merge items, run by 512 threads of 8
items each (FP64: 256 of 16): instances whose items end just before, at and after a tile, rows
around the 64 entries up to which a tile is summed row by row, and rows around
the 1024 entries from which a tile's cut may split them.

One step from the start vector x, y = A x / |A x|, against FP64.  A row of m
entries carries at most m + 3 roundings of its sum of |a||x|, and |A x| one of
its own: (m + 3) eps sum|a||x| / |A x| + 4 eps |y|, eps the rounding unit of
the sums (2^-53, 2^-24)."""
import numpy as np
import pytest

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu


def _matrix(rng, lens, n):
    lens = np.asarray(lens)
    rs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = np.concatenate([np.sort(rng.choice(n, m, replace=False)) for m in lens] + [np.zeros(0, int)]).astype(np.int32)
    return rs, ci, (rng.random(rs[-1]) + 0.5).astype(np.float32).astype(np.float64)


def _lens(kind):
    if kind.startswith("items"):  # rows of 5: 6 items each, n + nnz around a cut (3072) or a full tile (4096)
        total = int(kind[5:])
        lens = [5] * (total // 6)
        return lens[:-1] + [5 + total % 6]
    if kind == "short":  # a row per thread and more
        return [1] * 1500 + [0] * 700 + [2] * 900
    m = int(kind[4:])  # rows of about m entries among short ones
    return ([3] * 40 + [m - 1, m, m + 1]) * 3 + [0, 3]


@pytest.mark.parametrize("values,eps", [("f64", 2.0**-53), ("f32", 2.0**-24)])
@pytest.mark.parametrize("kind", ["items3071", "items3072", "items3073", "items4096", "items4097", "items9216", "short",
                                  "rows64", "rows512", "rows1024", "rows3072", "rows4096"])
def test_tile_edges(values, eps, kind):
    rng = np.random.default_rng(len(kind))
    lens = _lens(kind)
    n = len(lens)
    if n < max(lens):  # room for the columns of the longest row
        lens = lens + [1] * (max(lens) + 2 - n)
        n = len(lens)
    rs, ci, v = _matrix(rng, lens, n)
    for opt in ([{}, {"bf16_when_exact": 1}] if values == "f32" else [{}]):
        b = pw.Batch(values, items_per_thread=16, **opt)
        b.add_crs(rs, ci, v)
        b.solve(1, -1.0, seed=2)
        got, _ = b.vector(0, n)
        x = b.start_vector(0, n, seed=2)
        rows = np.repeat(np.arange(n), lens)
        y = np.bincount(rows, v * x[ci], n)
        mag = np.bincount(rows, np.abs(v * x[ci]), n)
        norm = np.linalg.norm(y)
        bound = (np.asarray(lens) + 3) * eps * mag / norm + 4 * eps * np.abs(y) / norm
        bound += np.linalg.norm((np.asarray(lens) + 3) * eps * mag) / norm * np.abs(y) / norm  # |A x| from the rounded y
        assert np.all(np.abs(got - y / norm) <= bound), (kind, np.max(np.abs(got - y / norm) - bound))
