"""Triangular solves (chain of 16-row tiles): block and tile edges, one to many
right-hand sides, both directions, both storages, unit diagonals, both types.

Bars: against a 64-bit reference, n u of the triangular solve's componentwise
growth (|T^-1| |T| |X| row by row); integer problems exactly.
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


def triangle(n, upper, unit, seed):
    T = inputs.normal_host(n, n, seed) / np.sqrt(n)
    T = np.triu(T, 1) if upper else np.tril(T, -1)
    d = 1.0 + 0.5 * np.abs(inputs.normal_host(n, 1, seed + 1)[:, 0])
    stored = T + np.diag(np.full(n, 7.0) if unit else d)  # a unit diagonal is never read
    return np.asfortranarray(stored), T + np.diag(np.ones(n) if unit else d)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 129, 320, 449])
@pytest.mark.parametrize("k", [1, 4, 5, 8, 9, 16, 17, 33])
@pytest.mark.parametrize("uplo,trans,unit", [("L", "N", False), ("L", "T", True), ("U", "N", True), ("U", "T", False)])
def test_trsm_shapes(n, k, uplo, trans, unit):
    stored, T = triangle(n, uplo == "U", unit, seed=n)
    B = inputs.normal_host(n, k, seed=3)
    Ad, Bd = E.Matrix.from_numpy(stored, ldim=n + 1), E.Matrix.from_numpy(B, ldim=n + 2)
    E.Trsm(E.LEFT, E.UPPER if uplo == "U" else E.LOWER, E.TRANSPOSE if trans == "T" else E.NORMAL,
           E.UNIT if unit else E.NON_UNIT, 1.0, Ad, Bd)
    M = T.T if trans == "T" else T
    X = np.linalg.solve(M, B)
    bound = (n + 4) * 2.0**-53 * (np.abs(np.linalg.inv(M)) @ (np.abs(M) @ np.abs(X)))
    assert (np.abs(host(Bd) - X) <= 4 * bound).all()


@pytest.mark.parametrize("n,k", [(70, 300), (400, 1100), (1100, 150), (2100, 300)])
def test_many_columns(n, k):
    """Several slabs a launch and several launches: every column as alone."""
    stored, T = triangle(n, False, False, seed=n)
    B = inputs.normal_host(n, k, seed=3)
    Ad, Bd = E.Matrix.from_numpy(stored, ldim=n + 1), E.Matrix.from_numpy(B)
    E.Trsm(E.LEFT, E.LOWER, E.TRANSPOSE, E.NON_UNIT, 1.0, Ad, Bd)
    X = host(Bd)
    for c0 in range(0, k, 16):
        one = E.Matrix.from_numpy(np.asfortranarray(B[:, c0:c0 + 16]))
        E.Trsm(E.LEFT, E.LOWER, E.TRANSPOSE, E.NON_UNIT, 1.0, Ad, one)
        assert np.array_equal(host(one), X[:, c0:c0 + 16])



@pytest.mark.parametrize("n,k", [(2500, 130), (1000, 300)])
def test_many_columns_integer_exact(n, k):
    A, L0 = inputs.integer_factor(n, seed=n)
    X0 = np.asfortranarray(np.random.default_rng(n).integers(-4, 5, (n, k)).astype(float))
    Ld, Bd = E.Matrix.from_numpy(L0), E.Matrix.from_numpy(A @ X0)
    E.SolveAfter(E.LOWER, E.NORMAL, Ld, Bd)
    assert np.array_equal(host(Bd), X0)


@pytest.mark.parametrize("n", [1, 16, 63, 130, 700])
@pytest.mark.parametrize("k", [1, 8, 20])
@pytest.mark.parametrize("uplo", ["L", "U"])
def test_float_solves(n, k, uplo):
    A = inputs.gram_host(n, seed=n).astype(np.float32)
    L = np.linalg.cholesky(A.astype(np.float64)).astype(np.float32)
    F = np.asfortranarray(L.T if uplo == "U" else L)
    B = inputs.normal_host(n, k, seed=4).astype(np.float32)
    Fd, Bd = E.Matrix.from_numpy(F), E.Matrix.from_numpy(B)
    E.SolveAfter(E.UPPER if uplo == "U" else E.LOWER, E.NORMAL, Fd, Bd)
    L64 = L.astype(np.float64)
    Y = np.linalg.solve(L64, B.astype(np.float64))
    X = np.linalg.solve(L64.T, Y)
    Li = np.abs(np.linalg.inv(L64))
    fwd = Li @ (np.abs(L64) @ np.abs(Y))
    bound = (n + 4) * 2.0**-24 * (Li.T @ (np.abs(L64.T) @ np.abs(X) + fwd))
    assert (np.abs(host(Bd) - X) <= 4 * bound).all()
