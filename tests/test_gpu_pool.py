"""Handles built and dropped over and over, from several threads at once: the
device memory that one leaves behind serves the next, and every result is that
of a fresh block.  What is left behind goes back to the device when asked for."""
import threading

import numpy as np
import pytest
import torch

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


def test_idle_memory_goes_back_to_the_device():
    n, c = 1000000, 16
    held = 12 * n * c  # an int and a double an entry
    T.Matrix(T.CSR).fill_cqmat(1000, 1000, 3, 0.2, 0).spmv(np.ones(1000))  # code is loaded
    T.release_memory()
    free = torch.cuda.mem_get_info()[0]
    g = T.Matrix(T.CSR).fill_cqmat(n, n, c, 0.2, 0)
    del g
    assert torch.cuda.mem_get_info()[0] <= free - held  # kept
    assert T.release_memory() >= held
    assert torch.cuda.mem_get_info()[0] >= free
    assert T.release_memory() == 0


def test_release_while_others_build():
    errors = []
    sizes = [(500, 3), (40000, 16), (9000, 31), (41000, 16)]
    ts = [threading.Thread(target=build_and_check, args=(k, sizes[k:] + sizes[:k], errors))
          for k in range(3)]
    for t in ts:
        t.start()
    while any(t.is_alive() for t in ts):
        T.release_memory()
        ts[0].join(0.001)
    for t in ts:
        t.join()
    assert not errors, errors[0]
