"""SpMM at the edges of its column chunks (16 and 32 columns, pairs and single
doubles), of its two grid orders, and at every remainder of its entry steps:
bit-exact with the products added in entry order."""
import numpy as np
import pytest

import tbsla_amd as T

pytestmark = pytest.mark.gpu


def ragged(n_row, n_col, seed=4):
    """Rows of 0, 1, 2, ... 17, 0, 1, ... entries at random columns."""
    rng = np.random.default_rng(seed)
    length = np.arange(n_row) % 18
    rp = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
    return rp, rng.integers(0, n_col, rp[-1]).astype(np.int32), rng.standard_normal(rp[-1])


def product(rp, ci, va, B):
    C = np.zeros((len(rp) - 1, B.shape[1]))
    for s in range(17):  # slot by slot: every row adds its entries in order
        rows = np.nonzero(rp[1:] - rp[:-1] > s)[0]
        j = rp[rows] + s
        C[rows] = C[rows] + va[j, None] * B[ci[j]]
    return C


def check(n_row, n_col, k, shift=0):
    rp, ci, va = ragged(n_row, n_col)
    geom = dict(n_row=n_row, n_col=n_col, f_row=0, f_col=0, ln_row=n_row, ln_col=n_col, pr=0, pc=0,
                NR=1, NC=1, nnz=len(ci))
    m = T.Matrix.from_arrays(T.CSR, geom, rp, ci, va)
    B = np.random.default_rng(k).standard_normal((n_col, k))
    dB = T.DeviceBuffer(8 * (B.size + 2))
    dC = T.DeviceBuffer(8 * (n_row * k + 2))
    T.check(T.lib().tbsla_hip_memcpy_htod(dB.ptr + shift, B.ctypes.data, B.nbytes, None))
    T.check(T.lib().tbsla_hip_spmm(m.h, dB.ptr + shift, dC.ptr + shift, k, None))
    got = np.empty((n_row, k))
    T.check(T.lib().tbsla_hip_memcpy_dtoh(got.ctypes.data, dC.ptr + shift, got.nbytes, None))
    assert np.array_equal(got, product(rp, ci, va, B))


# 1, 2, 4, 8, 9, 16 and 17 chunks of 32, and both chunk widths' edges
@pytest.mark.parametrize("k", [1, 2, 15, 16, 17, 18, 31, 32, 33, 34, 63, 64, 66, 127, 128, 130, 256,
                               288, 512, 544])
@pytest.mark.parametrize("n_row", [1, 17, 333])
def test_chunk_edges(n_row, k):
    check(n_row, 300, k)


@pytest.mark.parametrize("k", [16, 64, 256])
def test_operands_off_a_16_byte_boundary(k):
    check(333, 300, k, shift=8)


@pytest.mark.parametrize("n_col", [65536, 65537])
def test_both_grid_orders(n_col):
    check(5000, n_col, 64)
