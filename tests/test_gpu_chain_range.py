"""Triangular solves whose coefficients or right-hand sides leave the range in
which a tile's multipliers l_ck / l_kk are ordinary numbers.

Bars: rows scaled by powers of two give the unscaled system's solution within
its own bound, n u of |T^-1| |T| |X|; an entry that is not finite leaves the
rows solved before it, and the other columns, bit for bit what they were.
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


def triangle(n, upper, seed):
    T = inputs.normal_host(n, n, seed) / np.sqrt(n)
    T = np.triu(T, 1) if upper else np.tril(T, -1)
    return np.asfortranarray(T + np.diag(1.0 + 0.5 * np.abs(inputs.normal_host(n, 1, seed + 1)[:, 0])))


def trsm(T, B, uplo, trans):
    Td, Bd = E.Matrix.from_numpy(T, ldim=T.shape[0] + 1), E.Matrix.from_numpy(B)
    E.Trsm(E.LEFT, E.UPPER if uplo == "U" else E.LOWER, E.TRANSPOSE if trans == "T" else E.NORMAL, E.NON_UNIT, 1.0,
           Td, Bd)
    return host(Bd)


FORMS = [("L", "N"), ("L", "T"), ("U", "N"), ("U", "T")]


def test_two_rows():
    for l, b, x in [([[1e-200, 0.0], [1e150, 1.0]], [1e-200, 1e150], [1.0, 0.0]),
                    ([[1e200, 0.0], [1e-150, 1e-150]], [1e200, 2e-150], [1.0, 1.0])]:
        X = trsm(np.asfortranarray(l), np.asfortranarray(np.array(b)[:, None]), "L", "N")[:, 0]
        assert np.abs(X - x).max() <= 4 * 2.0**-53
    Ld = E.Matrix.from_numpy(np.asfortranarray(np.array([[1e-18, 0.0], [1e21, 1.0]], np.float32)))
    Bd = E.Matrix.from_numpy(np.asfortranarray(np.array([[1e-18], [1e21]], np.float32)))
    E.SolveAfter(E.LOWER, E.NORMAL, Ld, Bd)  # forward [1, 0], backward [1e18, 0]
    assert np.abs(host(Bd)[:, 0] - [1e18, 0.0]).max() <= 8 * 2.0**-24 * 1e18


@pytest.mark.parametrize("uplo,trans", FORMS)
@pytest.mark.parametrize("n,k", [(7, 1), (16, 5), (130, 9), (449, 20)])
def test_scaled_rows(n, k, uplo, trans):
    T = triangle(n, uplo == "U", seed=n)
    B = inputs.normal_host(n, k, seed=3)
    D = np.ldexp(1.0, np.random.default_rng(n).integers(-600, 601, n))
    Ts = T * D[None, :] if trans == "T" else T * D[:, None]  # op(T)'s rows
    X = trsm(np.asfortranarray(Ts), np.asfortranarray(B * D[:, None]), uplo, trans)
    M = T.T if trans == "T" else T
    ref = np.linalg.solve(M, B)
    bound = (n + 4) * 2.0**-53 * (np.abs(np.linalg.inv(M)) @ (np.abs(M) @ np.abs(ref)))
    assert (np.abs(X - ref) <= 4 * bound).all()


@pytest.mark.parametrize("n,k", [(40, 3), (200, 17)])
@pytest.mark.parametrize("uplo", ["L", "U"])
def test_scaled_rows_float(n, k, uplo):
    L = triangle(n, False, seed=n).astype(np.float32)
    B = inputs.normal_host(n, k, seed=4).astype(np.float32)
    D = np.ldexp(np.float32(1.0), np.random.default_rng(n).integers(-45, 46, n)).astype(np.float32)
    D[::3] *= np.float32(2.0**-20)  # ratios beyond 2^127 and below 2^-126 among neighbours
    D[1::3] = np.ldexp(np.float32(1.0), 70)
    Ls = (L * D[:, None]).astype(np.float32)
    F = np.asfortranarray(Ls.T if uplo == "U" else Ls)
    Fd, Bd = E.Matrix.from_numpy(F), E.Matrix.from_numpy(np.asfortranarray(B * D[:, None]))
    E.SolveAfter(E.UPPER if uplo == "U" else E.LOWER, E.NORMAL, Fd, Bd)
    Z = host(Bd).astype(np.float64) * D.astype(np.float64)[:, None]
    L64 = L.astype(np.float64)
    Y = np.linalg.solve(L64, B.astype(np.float64))
    X = np.linalg.solve(L64.T, Y)
    Li = np.abs(np.linalg.inv(L64))
    bound = (n + 4) * 2.0**-24 * (Li.T @ (np.abs(L64.T) @ np.abs(X) + Li @ (np.abs(L64) @ np.abs(Y))))
    assert (np.abs(Z - X) <= 4 * bound).all()


@pytest.mark.parametrize("uplo,trans", FORMS)
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("n,row", [(5, 3), (30, 13), (130, 47), (700, 640)])
def test_not_finite(n, row, value, uplo, trans):
    T = triangle(n, uplo == "U", seed=n)
    B = inputs.normal_host(n, 6, seed=3)
    X0 = trsm(T, np.asfortranarray(B), uplo, trans)
    B[row, 2] = value
    X = trsm(T, np.asfortranarray(B), uplo, trans)
    forward = (uplo == "L") == (trans == "N")
    before = slice(0, row) if forward else slice(row + 1, n)
    assert np.array_equal(np.delete(X, 2, 1), np.delete(X0, 2, 1))
    assert np.array_equal(X[before, 2], X0[before, 2])
    assert np.array_equal(X[row, 2], value / T[row, row], equal_nan=True)


def test_overflow_on_the_way():
    n = 100
    T = np.asfortranarray(np.eye(n) - 2.0**40 * np.eye(n, k=-1))
    B = np.asfortranarray(np.eye(n, 1))
    X = trsm(T, B, "L", "N")[:, 0]
    assert np.array_equal(X[:26], np.ldexp(1.0, 40 * np.arange(26)))
    assert X[26] == np.inf and not np.isfinite(X[26:]).any()


def test_zero_diagonal():
    T = triangle(20, False, seed=20)
    B = inputs.normal_host(20, 2, seed=3)
    X0 = trsm(T, np.asfortranarray(B), "L", "N")
    T[9, 9] = 0.0
    X = trsm(T, np.asfortranarray(B), "L", "N")
    assert np.array_equal(X[:9], X0[:9]) and np.isinf(X[9]).all() and not np.isfinite(X[9:]).any()
