"""The row kernel picked from the mean row length, on either side of every line
of the rule, for CSR and for COO triplets; rows from empty to ten times the mean."""
import numpy as np
import pytest

import tbsla_amd as T

pytestmark = pytest.mark.gpu

LINES = [2, 2.5, 4, 10, 15, 20, 28, 32, 48, 128]


@pytest.mark.parametrize("fmt", [T.CSR, T.COO])
@pytest.mark.parametrize("mean", [m + d for m in LINES for d in (-0.05, 0.05)])
def test_products_of_ragged_rows(fmt, mean):
    n = 1003
    rng = np.random.default_rng(int(100 * mean))
    weight = rng.exponential(1.0, n)
    weight[[0, n - 1]] = 10.0  # a long first and last row
    weight[5:9] = 0.0
    nnz = int(mean * n)
    length = np.bincount(rng.choice(n, nnz, p=weight / weight.sum()), minlength=n)
    rows = np.repeat(np.arange(n), length).astype(np.int32)
    rp = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
    ci, va, x = rng.integers(0, n, nnz).astype(np.int32), rng.random(nnz), rng.random(n)
    geom = dict(n_row=n, n_col=n, f_row=0, f_col=0, ln_row=n, ln_col=n, pr=0, pc=0, NR=1, NC=1,
                nnz=nnz)
    m = (T.Matrix.from_arrays(T.CSR, geom, rp, ci, va) if fmt == T.CSR
         else T.Matrix.from_arrays(T.COO, geom, rows, ci, va))
    want = np.zeros(n)
    np.add.at(want, rows, va * x[ci])
    # positive terms: both sums are within (length) roundings of the exact one
    bound = 2 * (length + 1) * np.finfo(float).eps * np.abs(want)
    assert np.all(np.abs(m.spmv(x) - want) <= bound)
