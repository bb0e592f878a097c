"""Infinities and NaN in x reach the rows that have an entry in their column, and
no other, on every CSR row kernel: ragged rows, so that a lane's load covers
entries of its neighbours, at both ends of the arrays too."""
import numpy as np
import pytest

import tbsla_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vec, lanes", [(1, 1), (1, 2), (1, 8), (1, 64), (2, 4), (2, 32), (4, 4),
                                        (4, 8), (4, 16)])
@pytest.mark.parametrize("rows", [1, 2])
def test_rows_take_no_other_rows_entries(vec, lanes, rows):
    n = 517
    rng = np.random.default_rng(3)
    length = rng.integers(0, 40, n)
    length[[0, 3, n - 1]] = 0, 200, 1
    rp = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
    ci, va = rng.integers(0, n, rp[-1]).astype(np.int32), rng.random(rp[-1])
    va[::7] = 0.0  # 0 times an infinity is NaN: only where the entry is the row's own
    geom = dict(n_row=n, n_col=n, f_row=0, f_col=0, ln_row=n, ln_col=n, pr=0, pc=0, NR=1, NC=1,
                nnz=int(rp[-1]))
    m = T.Matrix.from_arrays(T.CSR, geom, rp, ci, va)
    m.set_csr_kernel(lanes, rows, vec, 0)
    owner = np.repeat(np.arange(n), length)
    for where in (0, int(ci[5]), int(ci[rp[200]]), int(ci[-1])):
        for bad in (np.inf, np.nan):
            x = rng.random(n)
            x[where] = bad
            want = np.zeros(n)
            with np.errstate(invalid="ignore"):
                np.add.at(want, owner, va * x[ci])
            got = m.spmv(x)
            assert np.array_equal(np.isnan(got), np.isnan(want))
            assert np.array_equal(np.isinf(got), np.isinf(want))
            ok = np.isfinite(want)
            assert np.allclose(got[ok], want[ok], rtol=1e-13)
