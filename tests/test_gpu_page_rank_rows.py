"""PageRank with product and update in one kernel, on every row kernel that has
the form, at the edges of its 256-row tiles and of the wavefront's share of one:
against the batched solve of the same block as one instance, which multiplies
and updates in two kernels, bit for bit, and against numpy's iteration."""
import numpy as np
import pytest

import tbsla_amd as T

pytestmark = pytest.mark.gpu

KERNELS = ([(1, lanes) for lanes in (2, 4, 8, 16, 32, 64)] + [(2, lanes) for lanes in (4, 8, 16, 32)] +
           [(4, lanes) for lanes in (4, 8, 16)])


def ragged(n, seed=7):
    rng = np.random.default_rng(seed)
    length = rng.integers(0, 9, n)
    length[[0, n - 1]] = 3 * n // 4 + 1  # long first and last rows
    length[5:9] = 0
    rp = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
    nnz = int(rp[-1])
    ci = rng.integers(0, n, nnz).astype(np.int32)
    ci[:min(n, nnz)] = np.arange(min(n, nnz))  # no column without entries
    va = rng.random(nnz) + 0.1
    sums = np.zeros(n)
    np.add.at(sums, ci, va)
    va /= sums[ci]
    geom = dict(n_row=n, n_col=n, f_row=0, f_col=0, ln_row=n, ln_col=n, pr=0, pc=0, NR=1, NC=1,
                nnz=nnz)
    return T.Matrix.from_arrays(T.CSR, geom, rp, ci, va), (rp, ci, va)


@pytest.mark.parametrize("vec, lanes", KERNELS)
@pytest.mark.parametrize("n", [64, 255, 256, 257, 1000])
def test_page_rank_on_rows(n, vec, lanes):
    m, (rp, ci, va) = ragged(n)
    m.set_csr_kernel(lanes, 1, vec, 0)
    its = 5
    b, it, _ = m.page_rank(0.85, 0.0, its)
    assert it == its
    alone, it_b, _ = m.page_rank_batched([0, n], 0.85, 0.0, its)
    assert it_b[0] == its and np.array_equal(b, alone)
    A = np.zeros((n, n))
    np.add.at(A, (np.repeat(np.arange(n), np.diff(rp)), ci), va)
    x = np.ones(n)
    for _ in range(its):
        s = x.sum()
        x = (0.85 * (A @ x) + s * 0.15 / n) / s
    x /= x.sum()
    # positive terms: a row's sum carries at most its length + 3 roundings a
    # step, S at most n, each step again what came before
    bound = 4 * its * n * np.finfo(float).eps
    assert np.all(np.abs(b - x) <= bound * x)
