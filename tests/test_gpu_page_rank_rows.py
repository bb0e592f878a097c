"""PageRank with product and update in one kernel, on every row kernel that has
the form, at the edges of its 256-row tiles and of the wavefront's share of one:
against the batched solve of the same block as one instance, which multiplies
and updates in two kernels, bit for bit, and against numpy's iteration.  And
instances of a batch whose entries start anywhere, each as it is alone."""
import numpy as np
import pytest

import tbsla_amd as T

pytestmark = pytest.mark.gpu

KERNELS = ([(1, lanes) for lanes in (2, 4, 8, 16, 32, 64)] + [(2, lanes) for lanes in (4, 8, 16, 32)] +
           [(4, lanes) for lanes in (4, 8, 16)])


def ragged(n, seed=7):
    rng = np.random.default_rng(seed)
    length = rng.integers(0, 9, n)
    length[[0, n - 1]] = 3 * n // 4 + 1  # long first and last rows
    length[5:9] = 0
    rp = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
    nnz = int(rp[-1])
    ci = rng.integers(0, n, nnz).astype(np.int32)
    ci[:min(n, nnz)] = np.arange(min(n, nnz))  # no column without entries
    va = rng.random(nnz) + 0.1
    sums = np.zeros(n)
    np.add.at(sums, ci, va)
    va /= sums[ci]
    geom = dict(n_row=n, n_col=n, f_row=0, f_col=0, ln_row=n, ln_col=n, pr=0, pc=0, NR=1, NC=1,
                nnz=nnz)
    return T.Matrix.from_arrays(T.CSR, geom, rp, ci, va), (rp, ci, va)


@pytest.mark.parametrize("vec, lanes", KERNELS)
@pytest.mark.parametrize("n", [64, 255, 256, 257, 1000])
def test_page_rank_on_rows(n, vec, lanes):
    m, (rp, ci, va) = ragged(n)
    m.set_csr_kernel(lanes, 1, vec, 0)
    its = 5
    b, it, _ = m.page_rank(0.85, 0.0, its)
    assert it == its
    alone, it_b, _ = m.page_rank_batched([0, n], 0.85, 0.0, its)
    assert it_b[0] == its and np.array_equal(b, alone)
    A = np.zeros((n, n))
    np.add.at(A, (np.repeat(np.arange(n), np.diff(rp)), ci), va)
    x = np.ones(n)
    for _ in range(its):
        s = x.sum()
        x = (0.85 * (A @ x) + s * 0.15 / n) / s
    x /= x.sum()
    # positive terms: a row's sum carries at most its length + 3 roundings a
    # step, S at most n, each step again what came before
    bound = 4 * its * n * np.finfo(float).eps
    assert np.all(np.abs(b - x) <= bound * x)


@pytest.mark.parametrize("vec, lanes", [(2, 4), (2, 32), (4, 4), (4, 16), (0, 0)])
@pytest.mark.parametrize("rows", [1, 2])
def test_instances_as_they_are_alone(rows, vec, lanes):
    """Small and large instances whose first entries lie on three or four remainders of 4, many
    of them in one wavefront's rows; vec 0: the default kernel, on blocks of one mean."""
    sizes = [257, 64, 65, 1000, 66, 67] + ([3, 5, 7, 1, 2] * 9 if vec else [])
    if vec:
        parts = [ragged(n, seed=k)[0] for k, n in enumerate(sizes)]
    else:  # 15 entries to a row, and one row of 13 or 14: the same default for all
        parts = []
        for k, n in enumerate(sizes):
            length = np.full(n, 15)
            length[n // 2] = 14 - k % 2
            rp = np.concatenate([[0], np.cumsum(length)]).astype(np.int32)
            ci = np.random.default_rng(k).integers(0, n, rp[-1]).astype(np.int32)
            ci[:n] = np.arange(n)
            va = (1.0 / np.bincount(ci, minlength=n))[ci]
            geom = dict(n_row=n, n_col=n, f_row=0, f_col=0, ln_row=n, ln_col=n, pr=0, pc=0, NR=1,
                        NC=1, nnz=int(rp[-1]))
            parts.append(T.Matrix.from_arrays(T.CSR, geom, rp, ci, va))
    bd = T.Matrix.block_diag(parts)
    rp = bd.arrays()[0]
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    assert len(set(rp[offs[:-1]] % 4)) >= 3
    if vec:
        bd.set_csr_kernel(lanes, rows, vec, 0)
    b, its, errs = bd.page_rank_batched(offs, 0.85, 1e-12, 40)
    for k, m in enumerate(parts):
        if vec:
            m.set_csr_kernel(lanes, rows, vec, 0)
        else:
            mine, batch = m.get_csr_kernel(), bd.get_csr_kernel()
            assert mine["vec"] == batch["vec"] == 4 and mine["lanes"] == batch["lanes"]
        alone, it, err = m.page_rank(0.85, 1e-12, 40)
        assert (its[k], errs[k]) == (it, err)
        assert np.array_equal(b[offs[k]:offs[k + 1]], alone)
