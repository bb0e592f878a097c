"""Column sums whose last digit is sorted by the workgroup that adds: column
counts at which the sort's passes and that digit's bits change, with hub columns
over several chunks, against the entry-by-entry sums."""
import numpy as np
import pytest

import tbsla_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_col", [2, 3, 511, 512, 65535, 65536, 131071, 300000])
@pytest.mark.parametrize("nnz", [63, 4096, 50011])
@pytest.mark.parametrize("hub", [False, True])
def test_sums_in_storage_order(n_col, nnz, hub):
    rng = np.random.default_rng(n_col + nnz)
    n_row = 700
    r = np.sort(rng.integers(0, n_row, nnz)).astype(np.int32)
    c = rng.integers(0, n_col, nnz).astype(np.int32)
    if hub:
        c[rng.random(nnz) < 0.5] = n_col - 1
    v = rng.random(nnz) - 0.25
    rp = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n_row))]).astype(np.int32)
    geom = dict(n_row=n_row, n_col=n_col, f_row=0, f_col=0, ln_row=n_row, ln_col=n_col, pr=0, pc=0,
                NR=1, NC=1, nnz=nnz)
    m = T.Matrix.from_arrays(T.CSR, geom, rp, c, v)
    want = rng.random(n_col)
    got = m.get_col_sums(want)
    np.add.at(want, c, v)  # unbuffered: entry by entry, in order
    assert np.array_equal(got, want)
