"""Timed cases: SpMV, the power method, loading and batched solves as a user's program runs them.

A case is a dict of plain values:

  op      "mv"         y = A x on device vectors (mv_device)
          "power"      `its` fused power steps on device vectors (power_method_device)
          "mv_host"    the drop-in mv(x, y) on host arrays
          "power_host" the drop-in powerIteration(x, y, its) on host arrays
          "load"       a new handle: loadFromTriplets, then the first SpMV
          "batch"      many power methods solved together (Batch.solve)
  format  "crs", "merge", "csb" or "coh" (the four GPU classes)
  values  "f64", "f32" or "bf16" (storage of the matrix values)
  matrix  "poisson" (m x n grid), "stencil9" (9-point stencil on side x side
          plus 2 random entries per row) or "powerlaw" (rows x cols, row
          lengths of a power law with mean about 16)

Device vectors are torch tensors handed to the handle by address.  Vectors
and random matrices are drawn from the seed; the Poisson matrix has no random
part.
"""
import math

import numpy as np
import torch

import thesis_spmv_amd as pw

CLASSES = {"crs": pw.CRSHip, "merge": pw.CRSMergeHip, "csb": pw.CSBHip, "coh": pw.BlockCOHHip}
POWERLAW_MEAN = 16.0  # nonzeros per row of the power law below


def listed():
    return [
        # the smallest call: one SpMV on a matrix of about a thousand rows, the
        # size of the test collection's small matrices; launch latency
        dict(name="mv_crs_poisson_1k", op="mv", format="crs", values="f64", matrix="poisson", m=33, n=31),
        # 100 power iterations on such a matrix (the reference's own test sizes
        # and iteration count): the cost of a step beside its launches
        dict(name="power_merge_poisson_1k", op="power", format="merge", values="f64", matrix="poisson", m=37, n=29,
             its=100),
        # SpMV on the 1024 x 1024 Poisson grid
        dict(name="mv_csb_poisson_1m", op="mv", format="csb", values="f64", matrix="poisson", m=1024, n=1024),
        # the reference's headline run: 100 power iterations, m = 5000
        dict(name="power_crs_poisson_25m", op="power", format="crs", values="f64", matrix="poisson", m=5000, n=5000,
             its=100),
        # graph-like matrices with scattered columns, x beyond an L2: CSB, the
        # format for them, and the two CRS formats a user has at hand
        dict(name="mv_csb_powerlaw_2m", op="mv", format="csb", values="f64", matrix="powerlaw", rows=2097152,
             cols=2097152),
        dict(name="mv_merge_powerlaw_1m", op="mv", format="merge", values="f64", matrix="powerlaw", rows=1200007,
             cols=1200007),
        dict(name="mv_crs_powerlaw_f32", op="mv", format="crs", values="f32", matrix="powerlaw", rows=3000001,
             cols=3000001),
        # a discretised operator with a little long-range coupling, in CRS and
        # in the block format
        dict(name="mv_crs_stencil_2m", op="mv", format="crs", values="f64", matrix="stencil9", side=1448),
        dict(name="mv_coh_stencil_1m", op="mv", format="coh", values="f64", matrix="stencil9", side=1001),
        # the drop-in interface on host arrays, transfers included
        dict(name="mv_host_csb_poisson_1m", op="mv_host", format="csb", values="f64", matrix="poisson", m=1000, n=999),
        # a new matrix: 8 M shuffled triplets to a CRS handle, then its first SpMV
        dict(name="load_crs_powerlaw_8m", op="load", format="crs", values="f64", matrix="powerlaw", rows=500009,
             cols=500009),
        # 24 independent power methods of mixed sizes in one batch
        dict(name="batch_f32_24", op="batch", values="f32", instances=24, max_rows=300000, its=100, bf16=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_matrix(rng, lo, hi, square):
    kind = rng.choice(["poisson", "poisson", "powerlaw", "powerlaw", "stencil9"])
    rows = _log(rng, lo, hi)
    if kind == "poisson":
        m = max(2, _log(rng, max(2, math.isqrt(rows) // 4), math.isqrt(rows) * 4))
        return dict(matrix=kind, m=m, n=max(1, rows // m))
    if kind == "stencil9":
        return dict(matrix=kind, side=max(3, math.isqrt(min(rows, 4000000))))
    rows = min(rows, 3000000)
    cols = rows if square else rng.choice([rows, rows, max(64, rows // 2), rows * 2])
    return dict(matrix=kind, rows=max(64, rows), cols=max(64, min(cols, 4000000)))


def draw(rng):
    op = rng.choice(["mv"] * 8 + ["power"] * 4 + ["mv_host"] * 2 + ["power_host"] + ["load"] * 2 + ["batch"] * 2)
    if op == "batch":
        return dict(op=op, values=rng.choice(["f32", "f32", "f64"]), instances=rng.randint(2, 24),
                    max_rows=_log(rng, 2000, 300000), its=rng.randint(10, 100), bf16=rng.choice([False, True]))
    fmt = rng.choice(["crs", "merge", "csb", "coh"])
    if op == "load":
        return dict(op=op, format=fmt, values=rng.choice(["f64", "f64", "f32"]),
                    **_draw_matrix(rng, 1000, 400000, False))
    power = op.startswith("power")
    hi = {"mv": 9000000, "power": 9000000, "mv_host": 4000000, "power_host": 2000000}[op]
    c = dict(op=op, format=fmt, **_draw_matrix(rng, 300, hi, power))
    c["values"] = rng.choice(["f64", "f64", "f32"] + (["bf16"] if c["matrix"] == "poisson" else []))
    if power:
        c["its"] = rng.randint(5, 100)
    return c


# ------------------------------------------------------------ matrices


def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt) % (1 << 62))
    return g


def _coo(rows, cols, r, c, v):
    """Sorted (row, col) without duplicates."""
    key, order = torch.sort(r * cols + c, stable=True)
    keep = torch.ones_like(key, dtype=torch.bool)
    keep[1:] = key[1:] != key[:-1]
    key, v = key[keep], v[order][keep]
    return rows, cols, torch.div(key, cols, rounding_mode="floor"), key % cols, v


def _powerlaw(rows, cols, seed, positive):
    """Row lengths floor(7.3333 U^(-1/1.8)) (capped at 50 000 and at an eighth
    of the columns), uniform columns, N(0,1) values (their magnitudes when
    `positive`, the weights a power iteration meets)."""
    g = _gen(seed, 1)
    u = 1.0 - torch.rand(rows, generator=g, device="cuda", dtype=torch.float64)
    length = torch.clamp(torch.floor(7.3333 * u ** (-1.0 / 1.8)), max=min(50000, cols // 8)).to(torch.int64)
    r = torch.repeat_interleave(torch.arange(rows, device="cuda"), length)
    c = torch.randint(0, cols, (r.numel(),), generator=g, device="cuda")
    v = torch.randn(r.numel(), generator=g, device="cuda", dtype=torch.float64)
    return _coo(rows, cols, r, c, v.abs() + 1e-3 if positive else v)


def _stencil9(side, seed):
    """9-point stencil (8 / -1) and two random entries per row, U(-1, 1)."""
    g = _gen(seed, 2)
    n = side * side
    i = torch.arange(n, device="cuda")
    y, x = torch.div(i, side, rounding_mode="floor"), i % side
    rs, cs, vs = [], [], []
    for dy in (-1, 0, 1):
        for dx in (-1, 0, 1):
            ok = (y + dy >= 0) & (y + dy < side) & (x + dx >= 0) & (x + dx < side)
            rs.append(i[ok])
            cs.append((i + dy * side + dx)[ok])
            vs.append(torch.full((int(ok.sum()),), 8.0 if dy == dx == 0 else -1.0, device="cuda", dtype=torch.float64))
    for _ in range(2):
        rs.append(i)
        cs.append(torch.randint(0, n, (n,), generator=g, device="cuda"))
        vs.append(torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * 2 - 1)
    return _coo(n, n, torch.cat(rs), torch.cat(cs), torch.cat(vs))


def _coo_of(case, seed):
    if case["matrix"] == "powerlaw":
        return _powerlaw(case["rows"], case["cols"], seed, case["op"].startswith("power"))
    if case["matrix"] == "stencil9":
        return _stencil9(case["side"], seed)
    m, n = case["m"], case["n"]
    i = torch.arange(m * n, device="cuda")
    rs, cs, vs = [], [], []
    for d, v, ok in ((-m, -1.0, i >= m), (-1, -1.0, i % m != 0), (0, 4.0, i >= 0), (1, -1.0, i % m != m - 1),
                     (m, -1.0, i < m * n - m)):
        rs.append(i[ok])
        cs.append((i + d)[ok])
        vs.append(torch.full((int(ok.sum()),), v, device="cuda", dtype=torch.float64))
    return _coo(m * n, m * n, torch.cat(rs), torch.cat(cs), torch.cat(vs))


def _crs_of(coo):
    rows, cols, r, c, v = coo
    rs = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
    rs[1:] = torch.cumsum(torch.bincount(r, minlength=rows), 0)
    return rs, c, v


def _host(t, dtype):
    return np.ascontiguousarray(t.cpu().numpy(), dtype=dtype)


def _sizes(case):
    """Rows, columns and (expected) nonzeros."""
    if case["matrix"] == "poisson":
        m, n = case["m"], case["n"]
        return m * n, m * n, 5 * m * n - 2 * m - 2 * n
    if case["matrix"] == "stencil9":
        s = case["side"]
        return s * s, s * s, (3 * s - 2) ** 2 + 2 * s * s
    return case["rows"], case["cols"], int(POWERLAW_MEAN * case["rows"])


def _instances(case, seed):
    """The batch's matrices: Poisson grids and positive power-law matrices in
    turn, sizes spread over [max_rows / 30, max_rows] in log scale."""
    k, top = case["instances"], case["max_rows"]
    out = []
    for i in range(k):
        rows = max(64, int(top / 30 * 30 ** (i / max(k - 1, 1))))
        if i % 2 == 0:
            m = max(2, math.isqrt(rows) - i % 3)
            out.append(dict(op="power", matrix="poisson", m=m, n=max(2, rows // m)))
        else:
            out.append(dict(op="power", matrix="powerlaw", rows=rows, cols=rows))
    return [(c, seed * 64 + i) for i, c in enumerate(out)]


# ------------------------------------------------------------ the work


class _Vec:
    """A device vector of the framework's device entry points: its address."""

    def __init__(self, t):
        self.t, self.ptr = t, pw.C.c_void_p(t.data_ptr())


def _start(n, seed, dtype):
    return (torch.rand(n, generator=_gen(seed, 3), device="cuda", dtype=torch.float64) * 2 - 1).to(dtype)


def _vector_dtype(case):
    return torch.float64 if case["values"] == "f64" else torch.float32


def prepare(case, seed):
    op = case["op"]
    if op == "batch":
        b = pw.Batch(values=case["values"], bf16_when_exact=int(case["bf16"] and case["values"] == "f32"))
        for c, s in _instances(case, seed):
            if c["matrix"] == "poisson":
                b.add_poisson(c["m"], c["n"])
            else:
                rs, ci, v = _crs_of(_coo_of(c, s))
                b.add_crs(_host(rs, np.int32), _host(ci, np.int32), _host(v, np.float64))
        return dict(case=case, batch=b, seed=seed)
    rows, cols, _ = _sizes(case)
    state = dict(case=case)
    if op == "load":
        coo = _coo_of(case, seed)
        order = torch.randperm(coo[2].numel(), generator=_gen(seed, 4), device="cuda")
        state["triplets"] = pw.Triplet(rows, cols, _host(coo[2][order], np.int32), _host(coo[3][order], np.int32),
                                       _host(coo[4][order], np.float64))
    else:
        A = CLASSES[case["format"]](values=case["values"])
        if case["matrix"] == "poisson":
            A.generatePoissonMatrix(case["m"], case["n"])
        else:
            rs, ci, v = _crs_of(_coo_of(case, seed))
            A.loadCRS(rows, cols, _host(rs, np.int32), _host(ci, np.int32), _host(v, np.float64))
        state["A"] = A
    x = _start(cols, seed, _vector_dtype(case))
    if op.endswith("_host"):
        state["x"], state["y"] = _host(x, np.float64), np.zeros(rows)
    else:
        state["x"], state["y"] = _Vec(x), _Vec(torch.zeros(rows, device="cuda", dtype=x.dtype))
    torch.cuda.synchronize()  # the library works on streams of its own
    return state


def _single(case, v):
    """What FP32 vectors hold, as FP32 (the library hands it out as double)."""
    return v if case["values"] == "f64" else np.float32(v)


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "mv":
        state["A"].mv_device(state["x"], state["y"])
        return state["y"].t
    if op == "power":
        lam, norm, _ = state["A"].power_method_device(state["x"], state["y"], case["its"])
        return [state["x"].t, state["y"].t, _single(case, lam), _single(case, norm)]
    if op == "mv_host":
        state["A"].mv(state["x"], state["y"])
        return _single(case, state["y"])
    if op == "power_host":
        state["A"].powerIteration(state["x"], state["y"], case["its"])
        return [_single(case, state["x"]), _single(case, state["y"])]
    if op == "load":
        A = CLASSES[case["format"]](values=case["values"])
        A.loadFromTriplets(state["triplets"])
        A.mv_device(state["x"], state["y"])
        return state["y"].t
    b = state["batch"]
    lam, its, _ = b.solve(case["its"], -1.0, state["seed"])
    return [_single(case, lam), its] + [_single(case, b.vector(i)[0]) for i in range(case["instances"])]


def work(case):
    vb = {"f64": 8, "f32": 4, "bf16": 2}[case["values"]]
    xb = 8 if case["values"] == "f64" else 4
    if case["op"] == "batch":
        nbytes = flops = 0
        for c, _ in _instances(case, 0):
            n, _, z = _sizes(c)
            b = 2 if case["bf16"] and case["values"] == "f32" and c["matrix"] == "poisson" else vb
            nbytes += case["its"] * ((b + 4) * z + 4 * (n + 1) + 2 * xb * n)
            flops += case["its"] * 2 * z
        return {"bytes": nbytes, "flops": flops}
    rows, cols, z = _sizes(case)
    step = (vb + 4) * z + 4 * (rows + 1) + xb * (rows + cols)
    its = case.get("its", 1)
    if case["op"] == "load":  # the triplets in, the matrix out, the matrix in
        return {"bytes": 16 * z + (vb + 4) * z + 4 * (rows + 1) + step, "flops": 2 * z}
    return {"bytes": its * step, "flops": 2 * its * z}


# ------------------------------------------------------------ the same in 64 bits


def _operator(case, seed):
    """x -> A x in torch, FP64."""
    if case["matrix"] == "poisson":
        m, n = case["m"], case["n"]

        def mul(x):
            x = x.view(n, m)
            y = 4.0 * x
            y[1:] -= x[:-1]
            y[:-1] -= x[1:]
            y[:, 1:] -= x[:, :-1]
            y[:, :-1] -= x[:, 1:]
            return y.reshape(-1)

        return mul
    rows, cols, _ = _sizes(case)
    rs, ci, v = _crs_of(_coo_of(case, seed))
    a = torch.sparse_csr_tensor(rs, ci, v, size=(rows, cols))
    return lambda x: (a @ x.unsqueeze(1)).squeeze(1)


def _power(mul, x, its):
    """The last iterate, the one before it, the Rayleigh quotient and the norm of the last step."""
    lam = norm = None
    prev = x
    for k in range(its):
        prev = x if k == 0 else x / norm
        x = mul(prev)
        lam = torch.dot(prev, x) / torch.dot(prev, prev)
        norm = torch.linalg.vector_norm(x)
    return x / norm, prev, float(lam), float(norm)


def _batch_start(n, seed, i):
    """Batch.solve's documented start vector: U[-1, 1) hashed from (seed, id, row)."""
    with np.errstate(over="ignore"):
        z = np.uint64(seed) * np.uint64(0x9e3779b97f4a7c15) + (np.uint64(i) << np.uint64(32))
        z = z + np.arange(n, dtype=np.uint64) + np.uint64(0x632be59bd9b4e019)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xbf58476d1ce4e5b9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94d049bb133111eb)
        z = z ^ (z >> np.uint64(31))
    return torch.from_numpy((z >> np.uint64(11)).astype(np.float64) * 2.0 ** -53 * 2.0 - 1.0).cuda()


def exact(case, seed):
    op = case["op"]
    if op == "batch":
        lam, vec = [], []
        for i, (c, s) in enumerate(_instances(case, seed)):
            v, _, l, _ = _power(_operator(c, s), _batch_start(_sizes(c)[0], seed, i), case["its"])
            lam.append(l)
            vec.append(v)
        return [np.array(lam), None] + vec
    mul = _operator(case, seed)
    x = _start(_sizes(case)[1], seed, _vector_dtype(case)).double()
    if not op.startswith("power"):
        return mul(x)
    last, prev, lam, norm = _power(mul, x, case["its"])
    xy = [last, prev] if case["its"] % 2 == 0 else [prev, last]
    return xy if op == "power_host" else xy + [lam, norm]
