"""The radix sort behind the conversions, the column sums and the transpose, at the
edges of its tiles (4096 entries of a conversion, 8192 32-bit keys of the sums, 4096
64-bit keys of the transpose) and of the column sums' chunks (4096 entries of 256
columns), against numpy's stable sort and serial sums."""
import numpy as np
import pytest

import tbsla_amd as T

pytestmark = pytest.mark.gpu


def geom(n_row, n_col, nnz):
    return {"n_row": n_row, "n_col": n_col, "f_row": 0, "f_col": 0, "ln_row": n_row,
            "ln_col": n_col, "pr": 0, "pc": 0, "NR": 1, "NC": 1, "nnz": nnz}


def triplets(n_row, n_col, nnz, hub, seed=3):
    rng = np.random.default_rng(seed)
    r = rng.integers(0, n_row, nnz).astype(np.int32)
    c = rng.integers(0, n_col, nnz).astype(np.int32)
    if hub:  # most entries in one row and one column
        r[rng.random(nnz) < 0.7] = n_row - 1
        c[rng.random(nnz) < 0.7] = 0
    return r, c, rng.random(nnz)


@pytest.mark.parametrize("hub", [False, True])
@pytest.mark.parametrize("n", [7, 40000, 3000000])  # one, two and three passes an index
@pytest.mark.parametrize("nnz", [1, 63, 64, 65, 4095, 4096, 4097, 8191, 8192, 8193, 20011])
def test_convert_sorts_stably(n, nnz, hub):
    r, c, v = triplets(n, n, nnz, hub)
    m = T.Matrix.from_arrays(T.COO, geom(n, n, nnz), r, c, v)
    rp, ci, va = m.to(T.CSR).arrays()
    p = np.lexsort((c, r))  # stable
    assert np.array_equal(rp, np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]))
    assert np.array_equal(ci, c[p])
    assert np.array_equal(va, v[p])


@pytest.mark.parametrize("hub", [False, True])
@pytest.mark.parametrize("n_col", [1, 255, 256, 257, 1000])
@pytest.mark.parametrize("nnz", [1, 4095, 4097, 30011])
@pytest.mark.parametrize("fmt", ["CSR", "SCOO", "ELL"])
def test_col_sums_serial_order(fmt, nnz, n_col, hub):
    n_row = 300
    r, c, v = triplets(n_row, n_col, nnz, hub)
    m = T.Matrix.from_arrays(T.COO, geom(n_row, n_col, nnz), r, c, v - 0.25).to(T.FORMATS[fmt])
    s0 = np.random.default_rng(5).random(n_col)
    got = m.get_col_sums(s0)
    want = s0.copy()
    if fmt == "CSR":
        rp, cols, vals = m.arrays()
    elif fmt == "SCOO":
        _, cols, vals = m.arrays()
    else:  # only positive values are added (MatrixELL.cpp:809-815)
        cols, vals = (a.reshape(-1) for a in m.arrays())
        cols, vals = cols[vals > 0], vals[vals > 0]
    np.add.at(want, cols, vals)  # unbuffered: entry by entry, in order
    assert np.array_equal(got, want)


@pytest.mark.parametrize("nnz", [1, 4095, 4096, 4097, 8193])
def test_transpose_at_a_tiles_edges(nnz):
    n_row, n_col = 3000, 700
    r, c, v = triplets(n_row, n_col, nnz, True)
    g = T.Matrix.from_arrays(T.COO, geom(n_row, n_col, nnz), r, c, v).to(T.CSR)
    trp, tci, tva = g.transpose().arrays()
    p = np.lexsort((r, c))  # by column, then row, then the triplets' order
    assert np.array_equal(trp, np.concatenate([[0], np.cumsum(np.bincount(c, minlength=n_col))]))
    assert np.array_equal(tci, r[p]) and np.array_equal(tva, v[p])


def test_transpose_and_row_sums_past_one_tile():
    n, c = 5000, 11
    g = T.Matrix(T.CSR).fill_cqmat(n, n, c, 0.4, 3, value_seed=2)
    rp, ci, va = g.arrays()
    rows = np.repeat(np.arange(n), np.diff(rp))
    trp, tci, tva = g.transpose().arrays()
    p = np.lexsort((rows, ci))
    assert np.array_equal(trp, np.concatenate([[0], np.cumsum(np.bincount(ci, minlength=n))]))
    assert np.array_equal(tci, rows[p]) and np.array_equal(tva, va[p])
    r, cc, v = triplets(n, n, 20011, True)
    got = T.Matrix.from_arrays(T.SCOO, geom(n, n, len(r)), r, cc, v).get_row_sums()
    want = np.zeros(n)
    np.add.at(want, r, v)
    assert np.array_equal(got, want)
