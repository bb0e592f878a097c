"""Conversion of triplets that the import found in column order (sorted by row
alone), of the same after their arrays were written to, and the prefix sum on
both sides of one and of 2048 tiles of 2048 counts: against numpy."""
import numpy as np
import pytest

import tbsla_amd as T

pytestmark = pytest.mark.gpu


def geom(n, nnz):
    return {"n_row": n, "n_col": n, "f_row": 0, "f_col": 0, "ln_row": n, "ln_col": n, "pr": 0,
            "pc": 0, "NR": 1, "NC": 1, "nnz": nnz}


def expect(m, r, c, v, n):
    rp, ci, va = m.to(T.CSR).arrays()
    p = np.lexsort((c, r))  # stable
    assert np.array_equal(rp, np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]))
    assert np.array_equal(ci, c[p]) and np.array_equal(va, v[p])


@pytest.mark.parametrize("n", [7, 255, 256, 70001, 3000000])
@pytest.mark.parametrize("nnz", [1, 64, 8191, 8193, 30011])
def test_column_ordered(n, nnz):
    rng = np.random.default_rng(nnz)
    r = rng.integers(0, n, nnz).astype(np.int32)
    c = np.sort(rng.integers(0, n, nnz)).astype(np.int32)
    c[nnz // 2:] = c[nnz // 2]  # a long tie, kept in its order
    v = rng.random(nnz)
    m = T.Matrix.from_arrays(T.COO, geom(n, nnz), r, c, v)
    expect(m, r, c, v, n)
    # and no longer in column order, after a write through the device arrays
    c = rng.permutation(c).astype(np.int32)
    T.check(T.lib().tbsla_hip_memcpy_htod(m.device_arrays()[1], c.ctypes.data, c.nbytes, None))
    m.values_changed()
    expect(m, r, c, v, n)


@pytest.mark.parametrize("n", [2047, 2048, 2049, 2048 * 2048, 2048 * 2048 + 1])
def test_prefix_sum_of_row_lengths(n):
    """A tridiagonal's row pointer, summed from its row lengths."""
    rp = T.Matrix(T.CSR).fill_poisson3d(n, 1, 1).arrays()[0]
    want = 3 * np.arange(n + 1, dtype=np.int64)
    want[1:] -= 1
    want[n] -= 1
    assert np.array_equal(rp, want)
