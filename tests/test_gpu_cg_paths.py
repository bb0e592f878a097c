"""The CG engine's first kernel on every path it can take: stencils of 3, 5 and
7 diagonals and others in the diagonal layout, rows of 0 to 200 entries under
every lane count, one and two passes.  A few iterations from a known start
against numpy's CG in float64 (the iterates then differ by rounding only), and
the two passes of K1 bit for bit."""
import numpy as np
import pytest

import tbsla_amd as T

pytestmark = pytest.mark.gpu


def matrix(A):
    n = A.shape[0]
    rows, cols = np.nonzero(A)
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))])
    geom = dict(n_row=n, n_col=n, f_row=0, f_col=0, ln_row=n, ln_col=n, pr=0, pc=0, NR=1, NC=1,
                nnz=len(rows))
    return T.Matrix.from_arrays(T.CSR, geom, rp, cols, A[rows, cols])


def dense(m):
    rp, ci, va = m.arrays()
    A = np.zeros((len(rp) - 1,) * 2)
    A[np.repeat(np.arange(len(rp) - 1), np.diff(rp)), ci] = va
    return A


def reference(A, b, its, dinv):
    x, r = np.zeros_like(b), b.copy()
    z = r * dinv
    p, rz = z.copy(), r @ z
    for _ in range(its):
        q = A @ p
        alpha = rz / (p @ q)
        x, r = x + alpha * p, r - alpha * q
        z = r * dinv
        new = r @ z
        p, rz = z + new / rz * p, new
    return x


def check(m, A, its=4, **kw):
    b = np.random.default_rng(1).standard_normal(A.shape[0])
    jac = kw.get("preconditioner") == T.PRECOND_JACOBI
    want = reference(A, b, its, 1.0 / np.diag(A) if jac else np.ones(len(b)))
    x, it, _ = m.cg(b, max_iterations=its, tolerance=1e-300, relative=True, **kw)
    assert it == its
    # FP64: a handful of roundings per step; mixed: FP32 matrix values and sums
    bound = 1e-12 if kw.get("precision", T.CG_FP64) == T.CG_FP64 else 1e-5
    assert np.linalg.norm(x - want) <= bound * np.linalg.norm(want)
    return x


@pytest.mark.parametrize("precision", [T.CG_FP64, T.CG_MIXED])
@pytest.mark.parametrize("pre", [T.PRECOND_NONE, T.PRECOND_JACOBI])
# 3, 5 and 7 diagonals; row counts at and around one and two rows per thread
@pytest.mark.parametrize("grid", [(255, 1, 1), (256, 1, 1), (513, 1, 1), (16, 16, 1), (31, 33, 1),
                                  (2, 2, 2), (8, 8, 8), (9, 10, 11)])
def test_stencils_in_the_diagonal_layout(grid, pre, precision):
    m = T.Matrix(T.CSR).fill_poisson3d(*grid, kappa=T.lognormal_field(*grid, seed=3))
    A = dense(m)
    its = 4 if A.shape[0] > 8 else 2
    m.set_csr_layout(T.CSR_DIAG, 65536, 8)
    assert m.get_csr_layout()["remote"] == 0
    check(m, A, its, preconditioner=pre, precision=precision)


@pytest.mark.parametrize("precision", [T.CG_FP64, T.CG_MIXED])
@pytest.mark.parametrize("at", [(1, 0), (0, 1), (299, 300), (511, 510)])
def test_one_entry_off_symmetry(at, precision):
    """Not read as half of a symmetric matrix, before or after the entry changes."""
    m = T.Matrix(T.CSR).fill_poisson3d(512, 1, 1, kappa=T.lognormal_field(512, 1, 1, seed=3))
    A = dense(m)
    rp, ci, va = m.arrays()
    m.set_csr_layout(T.CSR_DIAG, 65536, 8)
    check(m, A, precision=precision)
    A[at] *= 1.25
    k = rp[at[0]] + int(np.flatnonzero(ci[rp[at[0]]:rp[at[0] + 1]] == at[1])[0])
    va = va.copy()
    va[k] *= 1.25
    T.check(T.lib().tbsla_hip_memcpy_htod(m.device_arrays()[2], va.ctypes.data, va.nbytes, None))
    m.values_changed()
    check(m, A, precision=precision)


@pytest.mark.parametrize("offsets", [(0,), (0, 3), (0, 1, 2, 7), (0, 1, 5, 6, 40, 41)])
def test_other_diagonal_counts(offsets):
    n = 700
    A = sum(np.diag(np.full(n - o, -1.0 / (1 + o)), o) for o in offsets if o)
    A = A + A.T if len(offsets) > 1 else np.zeros((n, n))
    A += np.diag(np.abs(A).sum(1) + 1.0 + np.arange(n) % 5)
    m = matrix(A)
    m.set_csr_layout(T.CSR_DIAG, 64, 8)
    assert m.get_csr_layout()["remote"] == 0
    check(m, A)


def ragged_spd(n=600, seed=2):
    """Symmetric, with rows of one entry, of a few, and of some 200."""
    rng = np.random.default_rng(seed)
    A = np.zeros((n, n))
    for i, k in [(0, 200), (299, 200), (n - 1, 200)]:
        A[i, rng.choice(n, k, replace=False)] = rng.standard_normal(k)
    for i in range(0, n, 3):
        k = i % 70
        A[i, rng.choice(n, k, replace=False)] = rng.standard_normal(k)
    A = A + A.T
    A[5, :] = A[:, 5] = A[n - 2, :] = A[:, n - 2] = 0.0
    np.fill_diagonal(A, np.abs(A).sum(1) + 1.0)
    return A


@pytest.mark.parametrize("precision", [T.CG_FP64, T.CG_MIXED])
@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16, 32, 64])
def test_ragged_rows_under_every_lane_count(lanes, precision):
    A = ragged_spd()
    m = matrix(A)
    x = [check(m, A, lanes_per_row=lanes, precision=precision, spmv_passes=p) for p in (1, 2)]
    assert np.array_equal(x[0], x[1])


@pytest.mark.parametrize("precision", [T.CG_FP64, T.CG_MIXED])
@pytest.mark.parametrize("pre", [T.PRECOND_NONE, T.PRECOND_JACOBI])
def test_two_passes_of_uneven_systems(pre, precision):
    """Systems of 1 to 236 workgroups that finish at different iterations, so that a
    launch meets running systems, the one it ends and those ended before: bit for
    bit as in one pass, and each as it is alone."""
    sizes = [(60401, 6), (300, 9), (9000, 40), (1, 3), (33000, 17), (5003, 2)]
    parts = [T.Matrix(T.CSR).fill_sym_cqmat(n, c, 0.1, 1, value_seed=k)
             for k, (n, c) in enumerate(sizes)]
    bd = T.Matrix.block_diag(parts)
    offs = np.concatenate([[0], np.cumsum([n for n, _ in sizes])]).astype(np.int32)
    rhs = np.random.default_rng(2).standard_normal(int(offs[-1]))
    kw = dict(tolerance=1e-10, relative=True, precision=precision, preconditioner=pre,
              lanes_per_row=4, replace_every=20 if precision == T.CG_MIXED else 0,
              max_blocks_per_system=256, max_iterations=300)
    x, res = bd.cg_batched(offs, rhs, bd.cg_options(spmv_passes=2, **kw))
    assert len({r.iterations for r in res}) >= 4
    x1, res1 = bd.cg_batched(offs, rhs, bd.cg_options(spmv_passes=1, **kw))
    of = [[(r.status, r.iterations, r.res_norm) for r in rs] for rs in (res, res1)]
    assert of[0] == of[1]
    assert np.array_equal(x, x1)
    for k, p in enumerate(parts):
        xs, its, rs = p.cg(rhs[offs[k]:offs[k + 1]], spmv_passes=2, **kw)
        assert (res[k].iterations, res[k].res_norm) == (its, rs)
        assert np.array_equal(x[offs[k]:offs[k + 1]], xs)
