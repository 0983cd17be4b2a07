"""Start vectors and final scaling of a batch, written for up to 64 instances
per launch: instance counts around the group size, with one instance longer
than one pass of its group's grid (16384 / 64 blocks of 256 rows) at either
end of the list.

After two steps every instance's vector is checked against the FP64 oracle
(CRS::powerIteration, Matrix/CRS.hpp:118-130).  Tolerance: a step rounds a row
sum of at most 5 products (7 units in the last place) and divides by |Ax|, at
least 0.76 |x| on the small grids (lambda_min of 4 x 4) against row sums of at
most 8 |x|, so an error grows by at most 11 per step: 7 * 132 units, 1.1e-13 in
FP64 and 5.6e-5 in FP32.  On the 90 000 row grid |Ax| is about 4.4 |x| for a
random x and the growth at most 2."""
import numpy as np
import pytest

import oracle

pw = pytest.importorskip("thesis_spmv_amd")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("values,tol", [("f64", 1.1e-13), ("f32", 5.6e-5)])
@pytest.mark.parametrize("count,long_at", [(1, None), (2, 0), (63, 62), (64, 0), (65, 64), (65, 0), (129, 128)])
def test_group_edges(values, tol, count, long_at):
    rng = np.random.default_rng(count)
    sizes = [(int(rng.integers(1, 5)), int(rng.integers(1, 5))) for _ in range(count)]
    if long_at is not None:
        sizes[long_at] = (300, 300)
    b = pw.Batch(values)
    for m, n in sizes:
        b.add_poisson(m, n)
    for seed in (5, 6):  # a second solve starts from its own vectors
        lam, its, _ = b.solve(2, -1.0, seed=seed)
        assert np.all(its == 2)
        for i, (m, n) in enumerate(sizes):
            A = oracle.poisson_crs(m, n)
            xr, _ = oracle.crs_power_iteration(A, b.start_vector(i, A.nor, seed=seed), 2)
            v, _ = b.vector(i, A.nor)
            assert np.max(np.abs(v - xr)) <= tol, (values, count, i, m, n)


@pytest.mark.parametrize("its", [1, 31, 32, 33, 64, 70])
def test_tail_of_a_chunk(its):
    """Steps around multiples of the 32-step chunk: full chunks replay a graph,
    a shorter last one is launched step by step; the same bits either way, with
    other work between the solves."""
    out = []
    for graph in (1, 0):
        b = pw.Batch("f32", graph=graph)
        sizes = [(3, 4), (70, 61), (300, 9)]
        for m, n in sizes:
            b.add_poisson(m, n)
        for rep in range(3):
            lam, k, _ = b.solve(its, -1.0, seed=7)
            assert np.all(k == its)
            out.append((lam, [b.vector(i, m * n)[0] for i, (m, n) in enumerate(sizes)]))
    for lam, vecs in out[1:]:
        assert np.array_equal(lam, out[0][0])
        for v, w in zip(vecs, out[0][1]):
            assert np.array_equal(v, w)
