"""Panel solves (16-column tiles) and trailing tiles of 64: block widths whole
and partial, row remainders, single matrices and batches.

Bars: the factor against the oracle's blocked loop within 1e-12 (the bar of the
blocked path), integer problems exactly; batches by the FP64 normwise backward
error, 4 n u.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import elemental_amd as E  # noqa: E402
from elemental_amd import batch as EB  # noqa: E402
from elemental_amd import inputs  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [8, 16, 24, 47, 100, 112, 128])
@pytest.mark.parametrize("m", [1, 15, 17, 64, 130])
def test_rows_and_widths(oracle, nb, m):
    n = nb + m
    A = inputs.gram_host(n, seed=n)
    ref = A.copy(order="F")
    assert oracle.lvar3(ref, nb) == 0
    M = E.Matrix.from_numpy(A, ldim=n + 1)
    E.Cholesky(E.LOWER, M, nb=nb)
    torch.cuda.synchronize()
    assert np.linalg.norm(np.tril(M.to_numpy() - ref)) <= 1e-12 * np.linalg.norm(np.tril(ref))
    Ai, L0 = inputs.integer_factor(n, seed=n)
    M = E.Matrix.from_numpy(Ai)
    E.Cholesky(E.LOWER, M, nb=nb)
    torch.cuda.synchronize()
    assert np.array_equal(np.tril(M.to_numpy()), L0)


def test_leading_dimension_past_32_bits(oracle):
    n, ld = 131, 1 << 27
    if torch.cuda.mem_get_info()[0] < 8 * n * ld + (8 << 30):
        pytest.skip("needs 140 GB")
    A = inputs.gram_host(n, seed=3)
    ref = A.copy(order="F")
    assert oracle.lvar3(ref, 128) == 0
    M = E.Matrix(n, n, ld)
    M.tensor().copy_(torch.from_numpy(A))
    E.Cholesky(E.LOWER, M, nb=128)
    got = M.tensor().cpu().numpy()
    del M
    torch.cuda.empty_cache()
    assert np.linalg.norm(np.tril(got - ref)) <= 1e-12 * np.linalg.norm(np.tril(ref))


@pytest.mark.parametrize("nb", [16, 40, 100, 128])
def test_batch(nb):
    n = [nb + d for d in (1, 15, 16, 63, 64, 65, 127, 129, 193)]
    plan = EB.BatchPlan(n, [2] * len(n), "f64", [(1 << 30, nb, 0)])
    A, B = plan.empty_a(), plan.empty_b()
    EB.fill_gram(plan, A, B, 9)
    A0, B0 = A.clone(), B.clone()
    plan.solve(A, B, use_graph=False)
    assert (plan.results()[0] == 0).all()
    eta = plan.backward_error(A0, B, B0)
    assert (eta <= 4 * np.array(n) * 2.0**-53).all(), eta
