"""Products and updates in 64 x 64 tiles: sizes at the edges of the tiles, of
the K chunks (16 in FP64, 32 in FP32) and of the leading dimension.

Bar, entry by entry: |err| <= (k + 4) u (|alpha| |A||B| + |beta| |C|), the
bound of any order of k + 1 additions and products in the working precision.
"""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import elemental_amd as E  # noqa: E402
from elemental_amd import inputs  # noqa: E402
from elemental_amd._lib import lib  # noqa: E402

pytestmark = pytest.mark.gpu


def host(M):
    torch.cuda.synchronize()
    return M.to_numpy()


def check(got, A, B, C, alpha, beta, u, part):
    A, B, C = (x.astype(np.longdouble) for x in (A, B, C))
    k = A.shape[1]
    want = alpha * (A @ B) + (beta * C if beta else 0)
    bound = (k + 4) * u * (abs(alpha) * (np.abs(A) @ np.abs(B)) + abs(beta) * np.abs(C))
    err = np.abs(got.astype(np.longdouble) - want)
    assert (err <= bound)[part].all()


@pytest.mark.parametrize("n", [1, 31, 63, 64, 65, 128, 200])
@pytest.mark.parametrize("k", [0, 1, 15, 16, 17, 31, 32, 33, 70])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_herk_tiles(n, k, dtype):
    t, u = (np.float64, 2.0**-53) if dtype == "f64" else (np.float32, 2.0**-24)
    for alpha, beta in ((-1.0, 1.0), (0.5, 0.0), (2.0, -0.25)):
        A = inputs.normal_host(n, max(k, 1), seed=n + k).astype(t)[:, :k]
        C = inputs.normal_host(n, n, seed=7).astype(t)
        Ad = E.Matrix.from_numpy(A, ldim=n + 1) if k else E.Matrix(n, 0, n + 1, dtype=torch.float64)
        Cd = E.Matrix.from_numpy(C, ldim=n + 3)
        if dtype == "f64":
            E.Herk(E.LOWER, E.NORMAL, alpha, Ad, beta, Cd)
        else:
            s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
            assert lib().elemamd_herk_f32(1, n, k, alpha, Ad.ptr(), Ad.LDim(), beta, Cd.ptr(), Cd.LDim(), s) == 0
        got = host(Cd)
        check(got, A, A.T, C, alpha, beta, u, np.tril(np.ones((n, n), bool)))
        assert np.array_equal(np.triu(got, 1), np.triu(C, 1))
