"""Products in 64 x 64 tiles (and 128 x 128 ones for the largest): every
orientation at tile and chunk edges, padded leading dimensions, each kind of
beta, triangles, an operand that C overlaps.

Bars: whole-number operands and scales, so every sum is exact.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import elemental_amd as E  # noqa: E402

pytestmark = pytest.mark.gpu

FORMS = [(E.NORMAL, E.NORMAL), (E.NORMAL, E.TRANSPOSE), (E.TRANSPOSE, E.NORMAL), (E.TRANSPOSE, E.TRANSPOSE)]


def ints(rng, r, c):
    return np.asfortranarray(rng.integers(-4, 5, (r, c)).astype(np.float64))


def stored(op, M):
    return np.asfortranarray(M if op is E.NORMAL else M.T)


@pytest.mark.parametrize("oa,ob", FORMS)
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (15, 65, 17), (64, 63, 16), (65, 64, 15), (130, 17, 33), (64, 128, 48), (200, 129, 0)])
@pytest.mark.parametrize("beta", [0.0, 1.0, -2.0])
def test_gemm(oa, ob, m, n, k, beta):
    rng = np.random.default_rng(m + 7 * n + k)
    A, B, C = ints(rng, m, k), ints(rng, k, n), ints(rng, m, n)
    Am = E.Matrix.from_numpy(stored(oa, A), ldim=max(1, stored(oa, A).shape[0]) + 3)
    Bm = E.Matrix.from_numpy(stored(ob, B), ldim=max(1, stored(ob, B).shape[0]) + 1)
    Cm = E.Matrix.from_numpy(C, ldim=m + 2)
    E.Gemm(oa, ob, -3.0, Am, Bm, beta, Cm)
    torch.cuda.synchronize()
    assert np.array_equal(Cm.to_numpy(), beta * C - 3.0 * (A @ B))


@pytest.mark.parametrize("oa,ob", FORMS)
def test_large(oa, ob):
    n, k = 4100, 24
    rng = np.random.default_rng(1)
    A, B = ints(rng, n, k), ints(rng, k, n)
    Cm = E.Matrix(n, n)
    E.Gemm(oa, ob, 1.0, E.Matrix.from_numpy(stored(oa, A)), E.Matrix.from_numpy(stored(ob, B)), 0.0, Cm)
    torch.cuda.synchronize()
    assert np.array_equal(Cm.to_numpy(), A @ B)


@pytest.mark.parametrize("uplo", [E.LOWER, E.UPPER])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 200])
def test_triangles(uplo, n):
    rng = np.random.default_rng(n)
    A, B, C = ints(rng, n, 20), ints(rng, 20, n), ints(rng, n, n)
    Cm = E.Matrix.from_numpy(C)
    E.Trrk(uplo, E.TRANSPOSE, E.NORMAL, 2.0, E.Matrix.from_numpy(stored(E.TRANSPOSE, A)), E.Matrix.from_numpy(B), 1.0, Cm)
    torch.cuda.synchronize()
    mask = np.tril(np.ones((n, n), bool)) if uplo is E.LOWER else np.triu(np.ones((n, n), bool))
    assert np.array_equal(Cm.to_numpy(), np.where(mask, C + 2.0 * (A @ B), C))


@pytest.mark.parametrize("m", [100, 300])
def test_operand_in_place(m):
    rng = np.random.default_rng(5)
    A, B = ints(rng, m, 100), ints(rng, 100, 100)
    Am = E.Matrix.from_numpy(A)
    E.Gemm(E.NORMAL, E.NORMAL, 1.0, Am, E.Matrix.from_numpy(B), 0.0, Am)
    torch.cuda.synchronize()
    assert np.array_equal(Am.to_numpy(), A @ B)


@pytest.mark.parametrize("n", [129, 192, 300, 513])
@pytest.mark.parametrize("nb", [32, 100, 128])
def test_inverse_blocks(n, nb):
    rng = np.random.default_rng(n)
    G = rng.standard_normal((n, n))
    A = np.asfortranarray(G @ G.T / n + np.eye(n))
    M = E.Matrix.from_numpy(A, ldim=n + 1)
    E.HPDInverse(E.LOWER, M, nb=nb)
    torch.cuda.synchronize()
    X = np.tril(M.to_numpy())
    X = X + np.tril(X, -1).T
    # condition below 6: n u of A times its inverse, with room for the sums
    assert np.abs(X @ A - np.eye(n)).max() <= 8 * n * 2.0**-53 * np.abs(A).sum(1).max() * np.abs(X).sum(1).max()
