"""Handles built and dropped over and over, from several threads at once: the
device memory that one leaves behind serves the next, and every result is that
of a fresh block."""
import threading

import numpy as np
import pytest

import oracle as O
import tbsla_amd as T

pytestmark = pytest.mark.gpu


def build_and_check(seed, sizes, errors):
    try:
        for n, c in sizes:
            g = T.Matrix(T.CSR).fill_cqmat(n, n, c, 0.2, 0, value_seed=seed)
            o = O.fill_cqmat(O.CSR, n, n, c, 0.2, 0, value_seed=seed)
            assert np.array_equal(g.make_stochastic(), o.make_stochastic())
            for a, b in zip(g.arrays(), o.arrays()):
                assert np.array_equal(a, b)
            x = O.unit_vector(seed, n)
            y = o.spmv(x)
            assert np.max(np.abs(g.spmv(x) - y)) <= 1e-12 * np.max(np.abs(y))
            del g
    except BaseException as e:  # noqa: BLE001 (reported by the test)
        errors.append(e)


@pytest.mark.parametrize("threads", [1, 4])
def test_reused_memory_gives_fresh_results(threads):
    # growing, shrinking and repeated sizes: blocks are reused, or too small
    sizes = [(500, 3), (40000, 16), (500, 3), (41000, 16), (9000, 31), (40000, 16), (200, 200)]
    errors = []
    ts = [threading.Thread(target=build_and_check, args=(k, sizes[k:] + sizes[:k], errors))
          for k in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors[0]
