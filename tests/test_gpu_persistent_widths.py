"""The persistent launch's panel solve at block widths around its 64-column form.

Bar: bit for bit the stepwise form's result, as for every width.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from elemental_amd import batch as EB  # noqa: E402

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("nb", [1, 15, 16, 17, 33, 48, 63, 64, 65])
def test_equals_stepwise(precision, nb):
    n = [nb + d for d in (0, 1, 15, 64, 65, 130)]
    got = []
    for grid in (0, 4):
        plan = EB.BatchPlan(n, [2] * len(n), precision, [(1 << 30, nb, grid)])
        A, B = plan.empty_a(), plan.empty_b()
        EB.fill_gram(plan, A, B, 9)
        A0, B0 = A.clone(), B.clone()
        plan.solve(A, B, use_graph=False)
        assert (plan.results()[0] == 0).all()
        eta = plan.backward_error(A0, B, B0)
        assert (eta <= np.maximum(4 * np.maximum(n, 8) * 2.0**-53, 1e-14)).all(), eta
        got.append((A, B))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
