"""Diagonal factor of the blocked factorizations with infinities and NaN.

Bars: LVar3Unb's loop (a pivot that is not positive fails, NaN among them)
decides which column fails and which entries of the factored block are finite;
those agree within 1e-12 (float storage 2e-5, as for finite matrices).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import elemental_amd as E  # noqa: E402
from elemental_amd import inputs  # noqa: E402

pytestmark = pytest.mark.gpu

TYPES = [("f64", 1e-12), ("f32", 2e-5)]


def host(M):
    torch.cuda.synchronize()
    return M.to_numpy()


def matrix(n, dtype, seed):
    A = inputs.gram_host(n, seed=seed)
    return np.asfortranarray(A.astype(np.float32)) if dtype == "f32" else A


def unblocked(A):
    """LVar3Unb on A (lower triangle): the failing column or None, and its state."""
    A = A.copy()
    for j in range(len(A)):
        if not A[j, j] > 0:
            return j, A
        A[j, j] = np.sqrt(A[j, j])
        A[j + 1:, j] /= A[j, j]
        A[j + 1:, j + 1:] -= np.tril(np.outer(A[j + 1:, j], A[j + 1:, j]))
    return None, A


@pytest.mark.parametrize("dtype,tol", TYPES)
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("row,col", [(17, 0), (40, 7), (100, 85), (127, 15), (110, 99)])
def test_entry_below_the_diagonal(row, col, value, dtype, tol):
    n, nb = 160, 128
    A = matrix(n, dtype, 5)
    A[row, col] = value
    with np.errstate(all="ignore"):
        fails, ref = unblocked(A.astype(np.float64)[:nb, :nb])
    assert fails == row
    M = E.Matrix.from_numpy(A)
    with pytest.raises(E.LogicError) as ei:
        E.Cholesky(E.LOWER, M, nb=nb)
    assert ei.value.column == row
    got, want = (np.tril(X.astype(np.float64)[:nb, :nb]) for X in (host(M), ref))
    fin = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fin)
    assert np.linalg.norm(got[fin] - want[fin]) <= tol * np.linalg.norm(want[fin])


@pytest.mark.parametrize("col", [3, 20, 47, 112, 140])
def test_infinite_pivot_float(oracle, col):
    n = 300
    A = matrix(n, "f32", 8)
    A[col, col] = np.inf
    ref = np.asfortranarray(A.astype(np.float64))
    assert oracle.lvar3(ref, 128) == 0
    M = E.Matrix.from_numpy(A)
    E.Cholesky(E.LOWER, M)
    got, want = np.tril(host(M).astype(np.float64)), np.tril(ref)
    assert np.array_equal(np.isinf(got), np.isinf(want)) and not np.isnan(got).any()
    fin = np.isfinite(want)
    assert np.linalg.norm(got[fin] - want[fin]) <= 2e-5 * np.linalg.norm(want[fin])
