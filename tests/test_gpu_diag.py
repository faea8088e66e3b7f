"""Diagonal factor of the blocked factorizations (16-column pieces).

Bars: the factor against the oracle's blocked loop within 1e-12 (the bar of
the blocked path; rounding order differs), integer problems exactly, a
failing column with the state the reference leaves, an infinite pivot as the
reference treats it.  Block widths at the edges of the 16-column pieces.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import elemental_amd as E  # noqa: E402
from elemental_amd import inputs  # noqa: E402

pytestmark = pytest.mark.gpu


def host(M):
    torch.cuda.synchronize()
    return M.to_numpy()


@pytest.mark.parametrize("nb", [1, 2, 15, 16, 17, 32, 33, 48, 63, 100, 112, 127, 128])
def test_block_widths(oracle, nb):
    n = 2 * nb + 3
    A = inputs.gram_host(n, seed=nb)
    ref = A.copy(order="F")
    assert oracle.lvar3(ref, nb) == 0
    M = E.Matrix.from_numpy(A, ldim=n + 3)
    E.Cholesky(E.LOWER, M, nb=nb)
    got = host(M)
    assert np.linalg.norm(np.tril(got - ref)) <= 1e-12 * np.linalg.norm(np.tril(ref))
    assert np.array_equal(np.triu(got, 1), np.triu(A, 1))
    Ai, L0 = inputs.integer_factor(n, seed=nb)
    M = E.Matrix.from_numpy(Ai)
    E.Cholesky(E.LOWER, M, nb=nb)
    assert np.array_equal(np.tril(host(M)), L0)


@pytest.mark.parametrize("dtype,tol", [("f64", 1e-12), ("f32", 2e-5)])
@pytest.mark.parametrize("col", [0, 1, 15, 16, 40, 111, 127, 128, 150])
def test_failing_column_state(oracle, col, dtype, tol):
    n, nb = 300, 128
    A = inputs.gram_host(n, seed=5)
    L = np.linalg.cholesky(A)
    A[col, col] -= 1.5 * L[col, col] ** 2
    if dtype == "f32":
        A = np.asfortranarray(A.astype(np.float32))
    ref = np.asfortranarray(A.astype(np.float64))
    assert oracle.lvar3(ref, nb) == col + 1
    M = E.Matrix.from_numpy(A)
    with pytest.raises(E.LogicError) as ei:
        E.Cholesky(E.LOWER, M, nb=nb)
    assert ei.value.column == col
    # the failing block: columns before `col` factored, the rest updated by them
    k0 = col // nb * nb
    k1 = min(k0 + nb, n)
    got = host(M).astype(np.float64)[k0:k1, k0:k1]
    want = ref[k0:k1, k0:k1]
    assert np.linalg.norm(np.tril(got - want)) <= tol * np.linalg.norm(np.tril(want))


@pytest.mark.parametrize("col", [0, 20, 127])
def test_infinite_pivot_goes_on(oracle, col):
    n = 160
    A = inputs.gram_host(n, seed=8)
    A[col, col] = np.inf
    ref = A.copy(order="F")
    assert oracle.lvar3(ref, 128) == 0
    M = E.Matrix.from_numpy(A)
    E.Cholesky(E.LOWER, M)
    got, want = np.tril(host(M)), np.tril(ref)
    assert np.array_equal(np.isinf(got), np.isinf(want)) and not np.isnan(got).any()
    fin = np.isfinite(want)
    assert np.linalg.norm(got[fin] - want[fin]) <= 1e-12 * np.linalg.norm(want[fin])


@pytest.mark.parametrize("n", [16, 33, 128, 129, 200, 515])
def test_float_factor(n):
    A = inputs.gram_host(n, seed=n).astype(np.float32)
    M = E.Matrix.from_numpy(np.asfortranarray(A))
    E.Cholesky(E.LOWER, M)
    L = np.tril(host(M)).astype(np.float64)
    A64 = A.astype(np.float64)
    # backward error of a float factorization: c n u with u = 2^-24
    assert np.linalg.norm(np.tril(L @ L.T - A64)) <= 4 * n * 2.0**-24 * np.linalg.norm(A64)
