"""Products of blocks of one matrix: views that interleave in memory without
sharing an element need no copy, and products of up to 128 rows or columns
may be in place.

Bars: whole-number operands, so every sum is exact; free device memory is what
it was after a product of views.
"""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import elemental_amd as E  # noqa: E402

pytestmark = pytest.mark.gpu


def ints(rng, r, c):
    return np.asfortranarray(rng.integers(-4, 5, (r, c)).astype(np.float64))


def host(M):
    torch.cuda.synchronize()
    return M.to_numpy()


def test_row_blocks_take_no_memory():
    m, n = 128, 200000
    P = E.Matrix(2 * m, n)
    P.tensor()[:] = torch.randint(-4, 5, (2 * m, n), device="cuda").double()
    A = E.Matrix.from_numpy(ints(np.random.default_rng(0), m, m))
    C, B = E.View(P, 0, 0, m, n), E.View(P, m, 0, m, n)
    want = A.tensor() @ B.tensor()[:, :64] + C.tensor()[:, :64]
    below = B.tensor()[:, -64:].clone()
    small = E.Matrix(m, m)
    E.Gemm(E.NORMAL, E.NORMAL, 1.0, A, A, 0.0, small)  # (the stream's own state exists)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    E.Gemm(E.NORMAL, E.NORMAL, 1.0, A, B, 1.0, C)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] < 64 << 20
    assert torch.equal(C.tensor()[:, :64], want) and torch.equal(B.tensor()[:, -64:], below)


@pytest.mark.parametrize("m,n,k", [(100, 100, 40), (64, 300, 64), (300, 128, 128), (100, 300, 70), (70, 90, 200)])
@pytest.mark.parametrize("where", ["first", "second", "apart"])
def test_operands_inside_the_result(m, n, k, where):
    rng = np.random.default_rng(m + n + k)
    rows, cols = max(m, k) + 5, max(n, k) + 130
    P = ints(rng, rows, cols)
    Pd = E.Matrix.from_numpy(P, ldim=rows + 1)
    C = E.View(Pd, 2, 1, m, n)
    if where == "first":  # A shares columns with C
        A, B = E.View(Pd, 2, 1, m, k), E.Matrix.from_numpy(ints(rng, k, n))
    elif where == "second":  # B shares rows with C
        A, B = E.Matrix.from_numpy(ints(rng, m, k)), E.View(Pd, 2, 1, k, n)
    else:  # beside it
        A, B = E.Matrix.from_numpy(ints(rng, m, 100)), E.Matrix.from_numpy(ints(rng, 100, n))
        if n + 101 <= cols:
            A = E.View(Pd, 2, n + 1, m, 100)
    want = C.to_numpy() - A.to_numpy() @ B.to_numpy()
    E.Gemm(E.NORMAL, E.NORMAL, -1.0, A, B, 1.0, C)
    assert np.array_equal(host(C), want)


@pytest.mark.parametrize("uplo", [E.LOWER, E.UPPER])
@pytest.mark.parametrize("n", [64, 65, 100, 128])
def test_triangles_in_place(n, uplo):
    rng = np.random.default_rng(n)
    mask = np.tril(np.ones((n, n), bool)) if uplo is E.LOWER else np.triu(np.ones((n, n), bool))
    C0 = ints(rng, n, n)
    for oa in (E.NORMAL, E.TRANSPOSE):
        C = E.Matrix.from_numpy(C0)
        E.Herk(uplo, oa, -1.0, C, 2.0, C)
        P = C0 @ C0.T if oa is E.NORMAL else C0.T @ C0
        assert np.array_equal(host(C), np.where(mask, 2.0 * C0 - P, C0))
        C = E.Matrix.from_numpy(C0)
        E.Trrk(uplo, oa, E.NORMAL, 1.0, C, C, 1.0, C)
        P = (C0 if oa is E.NORMAL else C0.T) @ C0
        assert np.array_equal(host(C), np.where(mask, C0 + P, C0))


@pytest.mark.parametrize("n", [64, 100, 128])
def test_float_triangle_in_place(n):
    C0 = ints(np.random.default_rng(n), n, n).astype(np.float32)
    C = E.Matrix.from_numpy(C0)
    rc = E.lib().elemamd_herk_f32(1, n, n, -1.0, C.ptr(), C.LDim(), 2.0, C.ptr(), C.LDim(),
                                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    assert np.array_equal(host(C), np.where(np.tril(np.ones((n, n), bool)), 2.0 * C0 - C0 @ C0.T, C0))
