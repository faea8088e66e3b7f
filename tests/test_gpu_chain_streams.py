"""Triangular solves with many right-hand sides on several streams at once:
their chains leave room for the helpers that they wait for.

Bar: every solve is bit for bit what it is alone.
"""
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import elemental_amd as E  # noqa: E402
from elemental_amd import inputs  # noqa: E402

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]


@pytest.mark.parametrize("n,k", [(300, 2100), (400, 1100)])
def test_four_streams(n, k):
    T = np.asfortranarray(np.tril(inputs.normal_host(n, n, 1) / np.sqrt(n), -1) + 1.5 * np.eye(n))
    B = np.asfortranarray(inputs.normal_host(n, k, 2))
    Td = E.Matrix.from_numpy(T)
    alone = E.Matrix.from_numpy(B)
    E.Trsm(E.LEFT, E.LOWER, E.NORMAL, E.NON_UNIT, 1.0, Td, alone)
    torch.cuda.synchronize()
    want = alone.to_numpy()
    right = [E.Matrix.from_numpy(B) for _ in range(4)]
    torch.cuda.synchronize()
    errors = []

    def solve(M):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                E.Trsm(E.LEFT, E.LOWER, E.NORMAL, E.NON_UNIT, 1.0, Td, M)
                torch.cuda.current_stream().synchronize()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=solve, args=(M,)) for M in right]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for M in right:
        assert np.array_equal(M.to_numpy(), want)
