"""Performance cases: the work that programs have this library do, through its
public entry points, each with its inputs, its ideal traffic, the agreement
between correct implementations and a plain 64-bit computation of its result.

The matrices are the library's own workloads: the cqmat generator (rows of c
entries, a share q of them rewired to random columns), the 7-point Poisson
problem with a smoothed log-normal coefficient, symmetrised cqmat systems,
and edge lists with hub rows as a file import delivers them.
"""
import math

import numpy as np
import torch

import tbsla_amd as T
from tbsla_amd import learned as LP

DEV = "cuda"

FORMATS = {"CSR": T.CSR, "ELL": T.ELL, "COO": T.COO, "SCOO": T.SCOO}


# ---- the cases ---------------------------------------------------------------


def listed():
    return [
        # one SpMV of a small graph inside somebody's own iteration: launch and call latency
        {"name": "spmv_small", "kind": "spmv", "format": "CSR", "n": 2003, "c": 10, "q": 0.1,
         "layout": "default"},
        # an ordinary SpMV on a matrix as it was filled, nothing tuned, ragged size
        {"name": "spmv_csr", "kind": "spmv", "format": "CSR", "n": 1000003, "c": 17, "q": 0.1,
         "layout": "default"},
        # the headline SpMV: many products with one large matrix, its layout chosen once
        {"name": "spmv_large", "kind": "spmv", "format": "CSR", "n": 4194304, "c": 32, "q": 0.1,
         "layout": "diagonal"},
        # building the transition matrix of a web graph: generation, column sums, normalisation
        {"name": "build_graph", "kind": "build", "n": 1500007, "c": 16, "q": 0.1},
        # an imported edge list (columns in file order, hub rows) becomes a CSR block
        {"name": "convert", "kind": "convert", "n": 300007, "nnz": 4800000, "order": "columns"},
        # PageRank of a mid-size graph to convergence
        {"name": "page_rank", "kind": "page_rank", "n": 200003, "c": 12, "q": 0.1},
        # personalised PageRank, 64 teleports as one dense block
        {"name": "ppr", "kind": "ppr", "n": 500009, "c": 24, "q": 0.1, "iterations": 24},
        # the sparse attention step: fused row softmax of the scores, product with the values
        {"name": "attention", "kind": "attention", "n": 200003, "c": 10, "k": 512},
        # one PDE solve, Jacobi-preconditioned CG in FP64
        {"name": "cg_jacobi", "kind": "cg", "nx": 64, "ny": 64, "nz": 64, "precision": "fp64",
         "preconditioner": "jacobi", "layout": "diagonal"},
        # many independent uneven SPD systems in one call, mixed precision
        {"name": "cg_batched", "kind": "cg_batched", "systems": 96, "q": 0.1},
        # a PDE solve with the learned factor: network inference, then factored CG
        {"name": "learned_solve", "kind": "cg", "nx": 101, "ny": 97, "nz": 100,
         "precision": "mixed", "preconditioner": "learned", "layout": "diagonal"},
        # one training step's loss and gradient of the preconditioner network
        {"name": "learned_train", "kind": "train", "side": 64, "probes": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spmv", "spmv", "spmv", "build", "convert", "page_rank", "ppr",
                       "attention", "cg", "cg", "cg_batched", "train"])
    q = round(rng.uniform(0.02, 0.3), 3)
    if kind == "spmv":
        fmt = rng.choice(["CSR", "CSR", "CSR", "ELL", "COO", "SCOO"])
        n, c = _log_int(rng, 1500, 3500000), rng.randint(5, 36)
        layout = "diagonal" if fmt == "CSR" and n > 100000 and rng.random() < 0.4 else "default"
        return {"kind": kind, "format": fmt, "n": n, "c": c, "q": q, "layout": layout}
    if kind == "build":
        return {"kind": kind, "n": _log_int(rng, 3000, 1500000), "c": rng.randint(5, 16), "q": q}
    if kind == "convert":
        n = _log_int(rng, 3000, 300000)
        return {"kind": kind, "n": n, "nnz": n * rng.randint(4, 16) + rng.randint(0, n - 1),
                "order": rng.choice(["columns", "random", "rows"])}
    if kind == "page_rank":
        return {"kind": kind, "n": _log_int(rng, 3000, 600000), "c": rng.randint(5, 24), "q": q}
    if kind == "ppr":
        return {"kind": kind, "n": _log_int(rng, 5000, 450000), "c": rng.randint(6, 24), "q": q,
                "iterations": rng.randint(8, 24)}
    if kind == "attention":
        n = _log_int(rng, 1024, 190000)
        return {"kind": kind, "n": n, "c": rng.randint(4, 40),
                "k": min(rng.choice([32, 64, 100, 128, 200, 256, 333, 512]), 30000000 // n)}
    if kind == "cg":
        side = [_log_int(rng, 12, 96) for _ in range(1)][0]
        nx, ny, nz = (max(8, side + rng.randint(-4, 4)) for _ in range(3))
        pre = rng.choice(["none", "jacobi", "jacobi", "learned"])
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz,
                "precision": rng.choice(["fp64", "mixed"]), "preconditioner": pre,
                "layout": rng.choice(["default", "diagonal"])}
    if kind == "cg_batched":
        return {"kind": kind, "systems": rng.randint(8, 90), "q": q}
    return {"kind": kind, "side": rng.randint(16, 63), "probes": rng.choice([4, 8, 16])}


# ---- helpers -----------------------------------------------------------------


class _Array:
    """Device memory of the library's, as torch reads foreign arrays; the
    tensor keeps this object, and so the memory's owner, alive."""

    def __init__(self, owner, ptr, n, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": kind, "data": (ptr, False),
                                         "version": 2}


def _view(owner, n, ptr=None, kind="<f8"):
    """A tensor over n elements of a DeviceBuffer, or of a matrix's array at ptr."""
    return torch.as_tensor(_Array(owner, owner.ptr if ptr is None else ptr, n, kind), device=DEV)


def _csr_views(m):
    g = m.geometry()
    a, b, v = m.device_arrays()
    return [_view(m, g.ln_row + 1, a, "<i4"), _view(m, g.stored, b, "<i4"), _view(m, g.stored, v)]


def _mult(seed):
    """The generator's seed multiplier for an input seed."""
    return 1 + seed % 65521


def _stochastic(case, seed):
    m = T.Matrix(T.CSR).fill_cqmat(case["n"], case["n"], case["c"], case["q"], _mult(seed),
                                   value_seed=seed)
    s = T.DeviceBuffer(case["n"] * 8)
    T.check(T.lib().tbsla_hip_memcpy_htod(s.ptr, np.zeros(case["n"]).ctypes.data, case["n"] * 8,
                                          None))
    T.check(T.lib().tbsla_hip_make_stochastic(m.h, s.ptr, None))
    return m


def _batch_sizes(case):
    """Uneven system sizes, the same for every seed (log-uniform 2^12 .. 2^16)."""
    rng = np.random.default_rng(case["systems"])
    return (np.floor(2.0 ** rng.uniform(12, 16, case["systems"])).astype(np.int64),
            rng.integers(8, 33, case["systems"]))


def _triplets(case, seed):
    """An edge list with uneven rows: half of the entries uniform, half drawn towards row 0."""
    rng = np.random.default_rng(seed)
    n, nnz = case["n"], case["nnz"]
    r = rng.integers(0, n, nnz).astype(np.int32)
    half = nnz // 2
    r[:half] = (n * rng.random(half) ** 2).astype(np.int32)
    c = rng.integers(0, n, nnz).astype(np.int32)
    v = rng.random(nnz)
    if case["order"] == "random":
        return r, c, v
    p = np.argsort(c if case["order"] == "columns" else r, kind="stable")
    return r[p], c[p], v[p]


def _mid_training(seed):
    """Parameters some way from the trained ones: at those the gradient has
    cancelled to its rounding errors, which no step of a training run sees."""
    theta = np.fromfile(LP.WEIGHTS, dtype="<f4")
    noise = np.random.default_rng(seed).standard_normal(theta.size)
    return (theta * (1.0 + 0.2 * noise)).astype(np.float32)


def _solver_options(A, case, G=None, GT=None):
    mixed = case["precision"] == "mixed"
    pre = {"none": T.PRECOND_NONE, "jacobi": T.PRECOND_JACOBI,
           "learned": T.PRECOND_FACTORED}[case["preconditioner"]]
    return A.cg_options(20000, 1e-8, True, T.CG_MIXED if mixed else T.CG_FP64, pre,
                        50 if mixed else 0, factor=G, factor_t=GT)


# ---- inputs ------------------------------------------------------------------


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind == "spmv":
        n = case["n"]
        m = T.Matrix(FORMATS[case["format"]]).fill_cqmat(n, n, case["c"], case["q"], _mult(seed),
                                                         value_seed=seed)
        if case["layout"] == "diagonal":
            m.set_csr_layout(T.CSR_DIAG, 65536, 8)
        s.update(m=m, x=T.uniform_vector(n, seed + 1), y=T.DeviceBuffer(n * 8))
        s["out"] = _view(s["y"], n)
    elif kind == "build":
        s.update(seed=seed, zero=torch.zeros(case["n"], dtype=torch.float64, device=DEV))
    elif kind == "convert":
        r, c, v = _triplets(case, seed)
        n = case["n"]
        geom = {"n_row": n, "n_col": n, "f_row": 0, "f_col": 0, "ln_row": n, "ln_col": n, "pr": 0,
                "pc": 0, "NR": 1, "NC": 1, "nnz": case["nnz"]}
        s["m"] = T.Matrix.from_arrays(T.COO, geom, r, c, v)
    elif kind == "page_rank":
        s.update(m=_stochastic(case, seed), b=T.DeviceBuffer(case["n"] * 8))
        s["out"] = _view(s["b"], case["n"])
    elif kind == "ppr":
        n = case["n"]
        s.update(m=_stochastic(case, seed), X=T.DeviceBuffer(n * 64 * 8),
                 src=np.random.default_rng(seed).choice(n, 64, replace=False).astype(np.int32))
        s["out"] = _view(s["X"], n * 64)
    elif kind == "attention":
        n, k = case["n"], case["k"]
        s["m"] = T.Matrix(T.CSR).fill_cqmat(n, n, case["c"], 1.0, _mult(seed), value_seed=seed)
        s.update(mx=T.DeviceBuffer(n * 8), sm=T.DeviceBuffer(n * 8),
                 B=T.uniform_vector(n * k, seed + 1, -1.0, 1.0), C=T.DeviceBuffer(n * k * 8))
        s["out"] = [_view(s["mx"], n), _view(s["sm"], n), _csr_views(s["m"])[2],
                    _view(s["C"], n * k)]
    elif kind == "cg":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        n = nx * ny * nz
        A = T.Matrix(T.CSR).fill_poisson3d(nx, ny, nz, T.lognormal_field(nx, ny, nz, seed=seed))
        if case["layout"] == "diagonal":
            A.set_csr_layout(T.CSR_DIAG, 65536, 8)
        s.update(A=A, rhs=T.uniform_vector(n, seed + LP.RHS_SEED_OFFSET, -1.0, 1.0),
                 x=T.DeviceBuffer(n * 8))
        if case["preconditioner"] == "learned":
            s.update(net=T.PrecondNet(), G=T.Matrix(T.CSR), GT=T.Matrix(T.CSR))
            LP.load_weights(s["net"])
        s["out"] = _view(s["x"], n)
    elif kind == "cg_batched":
        n, c = _batch_sizes(case)
        parts = [T.Matrix(T.CSR).fill_sym_cqmat(int(n[k]), int(c[k]), case["q"],
                                                _mult(seed + k), value_seed=seed + k)
                 for k in range(len(n))]
        A = T.Matrix.block_diag(parts)
        offs = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
        rows = int(offs[-1])
        s.update(A=A, offs=offs, rhs=T.uniform_vector(rows, seed + 17, -1.0, 1.0),
                 x=T.DeviceBuffer(rows * 8), res=(T.CGResult * len(n))(),
                 opt=A.cg_options(5000, 1e-8, True, T.CG_MIXED, T.PRECOND_NONE, 50))
        s["out"] = _view(s["x"], rows)
    elif kind == "train":
        net = T.PrecondNet()
        net.set_params(_mid_training(seed))
        s.update(net=net, A=LP.poisson_problem(case["side"], seed)[0], seed=seed)
    else:
        raise ValueError(kind)
    return s


# ---- one pass ----------------------------------------------------------------


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "spmv":
        s["m"].spmv_device(s["y"], s["x"])
        return s["out"]
    if kind == "build":
        m = T.Matrix(T.CSR).fill_cqmat(case["n"], case["n"], case["c"], case["q"],
                                       _mult(s["seed"]), value_seed=s["seed"])
        sums = s["zero"].clone()
        T.check(T.lib().tbsla_hip_make_stochastic(m.h, sums.data_ptr(), None))
        return _csr_views(m) + [sums]
    if kind == "convert":
        return _csr_views(s["m"].to(T.CSR))
    if kind == "page_rank":
        it, err = T.C.c_int(), T.C.c_double()
        T.check(T.lib().tbsla_hip_page_rank(s["m"].h, 0.85, 1e-10, 10000, s["b"].ptr,
                                            T.C.byref(it), T.C.byref(err), None))
        return s["out"]
    if kind == "ppr":
        s["m"].personalized_page_rank(s["src"], 0.85, 1e-10, case["iterations"], out=s["X"])
        return s["out"]
    if kind == "attention":
        T.check(T.lib().tbsla_hip_softmax_rows(s["m"].h, -1, s["mx"].ptr, s["sm"].ptr, None))
        T.check(T.lib().tbsla_hip_spmm(s["m"].h, s["B"].ptr, s["C"].ptr, case["k"], None))
        return s["out"]
    if kind == "cg":
        G = GT = None
        if case["preconditioner"] == "learned":
            G, GT = s["G"], s["GT"]
            T.check(T.lib().tbsla_hip_precond_net_apply(s["net"].h, s["A"].h, G.h, GT.h, None))
        s["A"].cg_device(s["rhs"], s["x"], _solver_options(s["A"], case, G, GT))
        return s["out"]
    if kind == "cg_batched":
        T.check(T.lib().tbsla_hip_cg_batched(
            s["A"].h, len(s["res"]), s["offs"].ctypes.data_as(T._ip), None, s["rhs"].ptr,
            s["x"].ptr, T.C.byref(s["opt"]), s["res"], None))
        return s["out"]
    loss, grad = s["net"].loss_grad(s["A"], case["probes"], s["seed"])
    return [loss, grad]


# ---- ideal traffic -----------------------------------------------------------


def _nnz(case):
    return case["n"] * case["c"]


def work(case):
    kind = case["kind"]
    if kind == "spmv":
        n, nnz = case["n"], _nnz(case)
        entry = 12 if case["format"] in ("CSR", "ELL") else 16
        return {"bytes": entry * nnz + 4 * (n + 1) + 16 * n, "flops": 2 * nnz}
    if kind == "build":  # the block and its column sums written once
        n, nnz = case["n"], _nnz(case)
        return {"bytes": 12 * nnz + 12 * n, "flops": 2 * nnz}
    if kind == "convert":  # triplets read once, the block written once
        return {"bytes": 28 * case["nnz"] + 4 * case["n"], "flops": 0}
    if kind == "page_rank":  # some 60 iterations: matrix, old and new iterate
        n, nnz = case["n"], _nnz(case)
        return {"bytes": 60 * (12 * nnz + 4 * n + 16 * n), "flops": 60 * (2 * nnz + 4 * n)}
    if kind == "ppr":
        n, nnz = case["n"], _nnz(case)
        return {"bytes": case["iterations"] * (12 * nnz + 4 * n + 2 * 8 * 64 * n),
                "flops": case["iterations"] * 64 * (2 * nnz + 4 * n)}
    if kind == "attention":  # scores read and written, then B, the block and C
        n, nnz, k = case["n"], _nnz(case), case["k"]
        return {"bytes": 16 * nnz + 12 * nnz + 4 * n + 16 * n + 2 * 8 * n * k,
                "flops": 2 * nnz * k + 4 * nnz}
    if kind == "cg":
        # iterations grow with the grid's side: 51 a cell without a
        # preconditioner, 4.7 with Jacobi's, 2.5 with the learned factor; each
        # reads the diagonals and reads and writes x, r, p once
        n = case["nx"] * case["ny"] * case["nz"]
        side = n ** (1 / 3)
        its = {"none": 51, "jacobi": 4.7, "learned": 2.5}[case["preconditioner"]] * side
        val = 4 if case["precision"] == "mixed" else 8
        per = 7 * val + 6 * 8 + {"none": 0, "jacobi": 8, "learned": 8 * val}[
            case["preconditioner"]]
        return {"bytes": int(its * per * n), "flops": int(its * n * 30)}
    if kind == "cg_batched":  # about 24 iterations of FP32 values and columns
        n, c = _batch_sizes(case)
        nnz = int((2 * n * c).sum())
        return {"bytes": 24 * (8 * nnz + 52 * int(n.sum())), "flops": 24 * 2 * nnz}
    # three layers of 64 x 128 products forward, twice that backward; the
    # matrix read and the activations written and read once, in FP32
    n = case["side"] ** 3
    return {"bytes": n * (7 * 12 + 2 * 4 * (64 * 3 + 128 * 3)), "flops": 3 * 3 * 2 * n * 64 * 128}


# ---- agreement ---------------------------------------------------------------


def tolerance(case):
    kind = case["kind"]
    if kind in ("build", "convert"):  # sums and sorts in a defined order
        return "exact"
    if kind in ("spmv", "attention"):  # FP64 sums of some tens of terms
        return {"rel": 1e-14, "max": 1e-12}
    if kind in ("page_rank", "ppr"):  # FP64 iterates in another order of summation
        return {"rel": 1e-12, "max": 1e-10}
    if kind in ("cg", "cg_batched"):
        # two solutions whose residuals pass 1e-8: the condition number is
        # what lets them differ by more
        return {"rel": 1e-6, "max": 1e-4} if kind == "cg" else {"rel": 5e-8, "max": 5e-6}
    # BF16 operands, FP32 sums: values on a rounding edge move by one BF16 step
    return {"rel": 2e-3, "max": 0.05}


# ---- the results in 64 bits, in plain torch ----------------------------------


def _i64(v):
    return v - (1 << 64) if v >= 1 << 63 else v


def _mix64(z):
    z = z + _i64(0x9E3779B97F4A7C15)
    z = (z ^ ((z >> 30) & ((1 << 34) - 1))) * _i64(0xBF58476D1CE4E5B9)
    z = (z ^ ((z >> 27) & ((1 << 37) - 1))) * _i64(0x94D049BB133111EB)
    return z ^ ((z >> 31) & ((1 << 33) - 1))


def _unit(seed, k):
    """The uniform value of index k (int64 tensor) under a seed: splitmix64."""
    h = _mix64(_mix64(torch.tensor(seed, dtype=torch.int64, device=DEV)) ^ k)
    return ((h >> 11) & ((1 << 53) - 1)).double() * 2.0 ** -53


def _rand_r(seed):
    """glibc's rand_r on a tensor of 32-bit states: (value, next state)."""
    m = (1 << 32) - 1
    s = (seed * 1103515245 + 12345) & m
    v = (s >> 16) & 2047
    for _ in range(2):
        s = (s * 1103515245 + 12345) & m
        v = (v << 10) ^ ((s >> 16) & 1023)
    return v, s


def _cqmat(n, c, q, mult, value_seed):
    """A square cqmat as (columns, values), n x c; short rows end in zeros."""
    full = n - c + 1
    row = torch.arange(n, device=DEV)
    length = torch.where(row < full, torch.full_like(row, c), c - 1 - (row - full))
    start = torch.cumsum(length, 0) - length
    j = torch.arange(c, device=DEV)[None, :]
    inside = j < length[:, None]
    k = torch.where(inside, start[:, None] + j, torch.zeros_like(j))
    v, state = _rand_r((k * mult) & ((1 << 32) - 1))
    col2, _ = _rand_r(state)
    tail = (row >= full)[:, None]
    rewired = torch.where(tail, (v // 2147483647).double() < q, v.double() / 2147483647.0 < q)
    del v, state
    cols = torch.where(rewired, col2 % n, row[:, None] + j)
    del col2, rewired
    return torch.where(inside, cols, torch.zeros_like(cols)), _unit(value_seed, k) * inside, length


def _product(cols, vals, x):
    """A x for one vector or a block of them, by column slots."""
    y = torch.zeros(cols.shape[0], *x.shape[1:], dtype=torch.float64, device=DEV)
    for j in range(cols.shape[1]):
        v = vals[:, j] if x.dim() == 1 else vals[:, j, None]
        y += v * x[cols[:, j]]
    return y


def _column_sums(cols, vals):
    return torch.zeros(cols.shape[0], dtype=torch.float64, device=DEV).index_add_(
        0, cols.reshape(-1), vals.reshape(-1))


def _exact_stochastic(case, seed):
    cols, vals, length = _cqmat(case["n"], case["c"], case["q"], _mult(seed), seed)
    sums = _column_sums(cols, vals)
    return cols, vals / torch.where(sums > 0, sums, torch.ones_like(sums))[cols], length, sums


def _rows(cols, vals, length):
    """rowptr, columns and values of the entries that are there."""
    inside = torch.arange(cols.shape[1], device=DEV)[None, :] < length[:, None]
    ptr = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEV), torch.cumsum(length, 0)])
    return ptr.int(), cols[inside].int(), vals[inside]


def _field(nx, ny, nz, seed, corr=4.0):
    """exp of a smoothed unit-variance Gaussian field, indexed [z, y, x]."""
    i = torch.arange(nx * ny * nz, device=DEV)
    z = torch.sqrt(-2.0 * torch.log(1.0 - _unit(seed, 2 * i))) * torch.cos(
        6.283185307179586 * _unit(seed, 2 * i + 1))
    z = z.reshape(nz, ny, nx)
    radius = math.ceil(3.0 * corr)
    w = [math.exp(-0.5 * (d / corr) ** 2) for d in range(-radius, radius + 1)]
    total = sum(w)
    w = [v / total for v in w]
    for axis in (2, 1, 0):
        size = z.shape[axis]
        out = torch.zeros_like(z)
        for d in range(-radius, radius + 1):
            j = (torch.arange(size, device=DEV) + d) % (2 * size)
            out += w[d + radius] * z.index_select(axis, torch.where(j >= size, 2 * size - 1 - j, j))
        z = out
    return torch.exp(z / sum(v * v for v in w) ** 1.5)


class _Poisson:
    """-div(k grad u) on the grid, matrix free."""

    def __init__(self, k):
        self.k, self.faces, self.diag = k, [], torch.zeros_like(k)
        for axis in (0, 1, 2):
            size = k.shape[axis]
            a, b = k.narrow(axis, 0, size - 1), k.narrow(axis, 1, size - 1)
            f = 2.0 * a * b / (a + b)
            self.faces.append(f)
            self.diag.narrow(axis, 0, size - 1).add_(f)
            self.diag.narrow(axis, 1, size - 1).add_(f)
            self.diag.select(axis, 0).add_(k.select(axis, 0))
            self.diag.select(axis, size - 1).add_(k.select(axis, size - 1))

    def __call__(self, u):
        y = self.diag * u
        for axis, f in enumerate(self.faces):
            size = u.shape[axis]
            y.narrow(axis, 0, size - 1).sub_(f * u.narrow(axis, 1, size - 1))
            y.narrow(axis, 1, size - 1).sub_(f * u.narrow(axis, 0, size - 1))
        return y


def _solve(apply, diag, b, tol=1e-13, most=6000):
    """Jacobi-PCG far past the tolerance of the measured solves."""
    x, r = torch.zeros_like(b), b.clone()
    z = r / diag
    p, rz, stop = z.clone(), (r * z).sum(), tol * b.norm()
    for it in range(most):
        q = apply(p)
        alpha = rz / (p * q).sum()
        x += alpha * p
        r -= alpha * q
        if it % 32 == 31 and bool(r.norm() < stop):
            break
        z = r / diag
        new = (r * z).sum()
        p = z + (new / rz) * p
        rz = new
    return x


def _exact_batched(case, seed):
    sizes, cs = _batch_sizes(case)
    rows, cols, vals, diags, base = [], [], [], [], 0
    for k, (n, c) in enumerate(zip(sizes, cs)):
        n, c = int(n), int(c)
        bc, bv, length = _cqmat(n, c, case["q"], _mult(seed + k), seed + k)
        r = torch.arange(n, device=DEV)[:, None].expand_as(bc)
        keep = (bc != r) & (torch.arange(c, device=DEV)[None, :] < length[:, None])
        i, j, v = r[keep], bc[keep], bv[keep] * 0.5
        key, where = torch.unique(torch.cat([i * n + j, j * n + i]), return_inverse=True)
        a = torch.zeros(key.numel(), dtype=torch.float64, device=DEV).index_add_(
            0, where, torch.cat([v, v]))
        i, j = key // n, key % n
        diags.append(1.0 + torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, i, a.abs()))
        rows.append(i + base)
        cols.append(j + base)
        vals.append(a)
        base += n
    i, j, a, d = (torch.cat(t) for t in (rows, cols, vals, diags))
    b = -1.0 + 2.0 * _unit(seed + 17, torch.arange(base, device=DEV))
    return _solve(lambda p: (d * p).index_add_(0, i, a * p[j]), d, b)


# the network's tensors, in the order of its parameter vector
_SHAPES = [("W0", (8, 64)), ("b0", (64,)), ("W1", (64, 128)), ("b1", (64,)), ("W2", (64, 128)),
           ("b2", (64,)), ("V", (64, 128)), ("ve", (64,)), ("c", (64,)), ("wo", (64,)),
           ("bo", (1,)), ("wd", (64,)), ("bd", (1,))]


def _exact_train(case, seed):
    """The preconditioner network's loss and gradient, by automatic
    differentiation, without its BF16 roundings."""
    side, probes = case["side"], case["probes"]
    n = side ** 3
    theta = torch.from_numpy(_mid_training(seed)).double().to(DEV)
    theta.requires_grad_(True)
    p, at = {}, 0
    for name, shape in _SHAPES:
        size = math.prod(shape)
        p[name] = theta[at:at + size].reshape(shape)
        at += size
    A = _Poisson(_field(side, side, side, seed))
    s = 1.0 / torch.sqrt(A.diag)
    index = torch.arange(n, device=DEV).reshape(side, side, side)
    er, ec, ev = [], [], []
    for axis, f in enumerate(A.faces):
        lo, hi = index.narrow(axis, 0, side - 1), index.narrow(axis, 1, side - 1)
        e = -f * s.narrow(axis, 0, side - 1) * s.narrow(axis, 1, side - 1)
        er += [hi.reshape(-1), lo.reshape(-1)]
        ec += [lo.reshape(-1), hi.reshape(-1)]
        ev += [e.reshape(-1)] * 2
    er, ec, ev = torch.cat(er), torch.cat(ec), torch.cat(ev)

    def edges(u):  # E u
        return torch.zeros_like(u).index_add(0, er, ev[:, None] * u[ec])

    one = torch.ones(n, dtype=torch.float64, device=DEV)
    degree = torch.zeros_like(one).index_add(0, er, torch.ones_like(ev))
    feats = torch.stack([one, torch.zeros_like(one).index_add(0, er, ev.abs()),
                         torch.zeros_like(one).scatter_reduce(0, er, ev.abs(), "amax"),
                         degree / 8], 1)
    h = torch.relu(torch.cat([feats, edges(feats)], 1) @ p["W0"] + p["b0"])
    for w, b in (("W1", "b1"), ("W2", "b2")):
        u = h @ p[w]
        h = torch.relu(u[:, :64] + edges(u[:, 64:]) + p[b])
    u = h @ p["V"]
    low = ec < er
    lr, lc, le = er[low], ec[low], ev[low]
    g = torch.relu(u[lr, :64] + u[lc, 64:] + le[:, None] * p["ve"] + p["c"]) @ p["wo"] + p["bo"]
    gd = torch.exp(h @ p["wd"] + p["bd"])
    i = torch.arange(n * probes, device=DEV)
    Z = torch.where(_unit(seed, i) < 0.5, -1.0, 1.0).double().reshape(n, probes)
    U = gd[:, None] * Z + torch.zeros_like(Z).index_add(0, lr, g[:, None] * Z[lc])
    V = U + edges(U)
    W = gd[:, None] * V + torch.zeros_like(V).index_add(0, lc, g[:, None] * V[lr])
    loss = ((Z - W) ** 2).sum() / (n * probes)
    loss.backward()
    return [float(loss.detach()), theta.grad.cpu().numpy()]


def exact(case, seed):
    kind = case["kind"]
    if kind == "spmv":
        cols, vals, _ = _cqmat(case["n"], case["c"], case["q"], _mult(seed), seed)
        return _product(cols, vals, _unit(seed + 1, torch.arange(case["n"], device=DEV)))
    if kind == "build":
        cols, vals, length, sums = _exact_stochastic(case, seed)
        return list(_rows(cols, vals, length)) + [sums]
    if kind == "convert":
        r, c, v = _triplets(case, seed)
        p = np.lexsort((c, r))
        ptr = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=case["n"]))])
        return [ptr.astype(np.int32), c[p], v[p]]
    if kind == "page_rank":
        n = case["n"]
        cols, vals, _, _ = _exact_stochastic(case, seed)
        b = torch.ones(n, dtype=torch.float64, device=DEV)
        for _ in range(10000):
            old, total = b, b.sum()
            b = (0.85 * _product(cols, vals, old) + total * ((1 - 0.85) / n)) / total
            if float((b - old).abs().sum()) < 1e-10:
                break
        return b / b.sum()
    if kind == "ppr":
        n = case["n"]
        cols, vals, _, _ = _exact_stochastic(case, seed)
        src = np.random.default_rng(seed).choice(n, 64, replace=False)
        one = torch.zeros(n, 64, dtype=torch.float64, device=DEV)
        one[torch.from_numpy(src).to(DEV), torch.arange(64, device=DEV)] = 1.0
        X = torch.ones(n, 64, dtype=torch.float64, device=DEV)
        for _ in range(case["iterations"]):
            old, total = X, X.sum(0)
            X = (0.85 * _product(cols, vals, old) + (1 - 0.85) * total * one) / total
            if float((X - old).abs().sum(0).max()) < 1e-10:
                break
        return (X / X.sum(0)).reshape(-1)
    if kind == "attention":
        n, k = case["n"], case["k"]
        cols, vals, length = _cqmat(n, case["c"], 1.0, _mult(seed), seed)
        inside = torch.arange(case["c"], device=DEV)[None, :] < length[:, None]
        top = vals.abs().amax(1)
        w = torch.exp(vals - top[:, None]) * inside
        total = w.sum(1)
        prob = w / torch.where(total == 0, torch.ones_like(total), total)[:, None]
        B = -1.0 + 2.0 * _unit(seed + 1, torch.arange(n * k, device=DEV)).reshape(n, k)
        return [top, total, prob[inside], _product(cols, prob, B).reshape(-1)]
    if kind == "cg":
        shape = (case["nz"], case["ny"], case["nx"])
        A = _Poisson(_field(case["nx"], case["ny"], case["nz"], seed))
        b = -1.0 + 2.0 * _unit(seed + LP.RHS_SEED_OFFSET,
                               torch.arange(math.prod(shape), device=DEV)).reshape(shape)
        return _solve(A, A.diag, b).reshape(-1)
    if kind == "cg_batched":
        return _exact_batched(case, seed)
    return _exact_train(case, seed)
