"""cqmat blocks as wide as the matrix, filled without a counting pass: CSR and
SCOO bit-exact with the oracle at the edges of the rows' lengths, of the tail
rows and of the rewiring test."""
import numpy as np
import pytest

import oracle as O
import tbsla_amd as T

pytestmark = pytest.mark.gpu


def same(fmt, args, kw):
    g = T.Matrix(fmt).fill_cqmat(*args, **kw)
    o = O.fill_cqmat(fmt, *args, **kw)
    assert g.geom == o.geom, (args, kw)
    for a, b in zip(g.arrays(), o.arrays()):
        assert np.array_equal(a, b) or (a.size == 0 and b.size == 0), (args, kw)


@pytest.mark.parametrize("fmt", [T.CSR, T.SCOO])
@pytest.mark.parametrize("c", [1, 2, 3, 4, 5, 7, 8, 31, 33, 64, 255, 499, 500])
def test_row_lengths_and_tails(fmt, c):
    for n_row, n_col in [(500, 500), (511, 500), (480, 500)]:
        for pr, NR in [(0, 1), (0, 3), (2, 3), (6, 7)]:
            same(fmt, (n_row, n_col, c, 0.3, 1, pr, 0, NR, 1), dict(value_seed=3))


@pytest.mark.parametrize("q", [0.0, 1e-9, 0.25, 0.999999999, 1.0, 1.5, -1.0])
@pytest.mark.parametrize("seed_mult", [0, 1, 40507, 4294967295])
def test_rewiring(q, seed_mult):
    same(T.CSR, (3001, 3001, 13, q, seed_mult, 0, 0, 1, 1), dict(value_seed=-1))
