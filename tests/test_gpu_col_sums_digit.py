"""Column sums whose last digit is sorted by the workgroup that adds: column
counts at which the sort's passes and that digit's bits change, with hub columns
over several chunks, against the entry-by-entry sums; and blocks whose slots are
mostly ones that the sums skip."""
import time

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


def few_long_rows(n_row, n_col, width, seed=0):
    """ELL: one row of `width` entries, the others of one: nearly all slots padding."""
    rng = np.random.default_rng(seed)
    r = np.concatenate([np.arange(n_row), np.full(width - 1, n_row // 2)]).astype(np.int32)
    c = rng.integers(0, n_col, len(r)).astype(np.int32)
    v = rng.random(len(r)) - 0.25
    geom = dict(n_row=n_row, n_col=n_col, f_row=0, f_col=0, ln_row=n_row, ln_col=n_col, pr=0, pc=0,
                NR=1, NC=1, nnz=len(r))
    return T.Matrix.from_arrays(T.COO, geom, r, c, v).to(T.ELL)


# on and off a multiple of a bucket's columns, in one bucket, and with as many
# buckets as the sort's bits can and cannot tell apart beside the skipped one
@pytest.mark.parametrize("n_col", [1, 2, 255, 256, 257, 4096, 5000, 65280, 65281, 65535, 65536])
@pytest.mark.parametrize("width", [1, 37, 700])
def test_padding_is_skipped(n_col, width):
    m = few_long_rows(777, n_col, width, seed=n_col)
    want = np.random.default_rng(1).random(n_col)
    got = m.get_col_sums(want)
    cols, vals = (a.reshape(-1) for a in m.arrays())  # slots row by row
    np.add.at(want, cols[vals > 0], vals[vals > 0])
    assert np.array_equal(got, want)


def test_padding_costs_no_more_than_entries():
    """16 M slots: one long row takes no longer than rows that are all entries (0.3
    and 0.7 ms; 30 when one workgroup read the skipped slots 4096 at a time)."""
    n, width = 16384, 1024

    def seconds(m):
        s = T.DeviceBuffer(n * 8)
        best = np.inf
        for _ in range(5):
            t = time.perf_counter()
            T.check(T.lib().tbsla_hip_get_col_sums(m.h, s.ptr, None))  # waits for the sums
            best = min(best, time.perf_counter() - t)
        return best

    full = seconds(T.Matrix(T.ELL).fill_cqmat(n, n, width, 0.5, 1, value_seed=3))
    assert seconds(few_long_rows(n, n, width)) < 3 * full
