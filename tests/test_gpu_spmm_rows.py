"""SpMM rows at the edges of the 16 entries that a row's lanes hold at a time, for
every alignment's lane count, in a block whose column filter drops entries:
bit for bit the loop of separate products and sums."""
import numpy as np
import pytest

import tbsla_amd as T

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 2, 7, 8, 9, 15, 16, 17, 23, 24, 25, 31, 32, 33, 100, 0]


@pytest.mark.parametrize("k", [1, 2, 15, 16, 17, 18, 32, 33, 34, 96])
def test_row_lengths(k):
    rng = np.random.default_rng(k)
    n_row, f_col, ln_col = len(LENGTHS), 40, 200
    rp = np.concatenate([[0], np.cumsum(LENGTHS)]).astype(np.int32)
    ci = (f_col + rng.integers(0, ln_col, rp[-1])).astype(np.int32)
    va = rng.standard_normal(rp[-1])
    geom = dict(n_row=n_row, n_col=300, f_row=0, f_col=f_col, ln_row=n_row, ln_col=ln_col, pr=0,
                pc=0, NR=1, NC=1, nnz=int(rp[-1]))
    m = T.Matrix.from_arrays(T.CSR, geom, rp, ci, va)
    B = rng.standard_normal((ln_col, k))
    want = np.zeros((n_row, k))
    for i in range(n_row):
        for j in range(rp[i], rp[i + 1]):
            want[i] += va[j] * B[ci[j] - f_col]
    assert np.array_equal(m.spmm(B), want)
