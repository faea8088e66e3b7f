"""A matrix of a batch that is not HPD, in both launch forms.

Bars: the first failing column is reported; the bad matrix is left as the
reference leaves it when LVar3 throws (1e-12 against the oracle's blocked
loop; float storage 2e-5), equal bit for bit between the stepwise and the
persistent form; the batch's other matrices are what they are without it.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from elemental_amd import batch as EB  # noqa: E402

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]

N = [40, 256, 300, 130, 300]
K = [2, 3, 1, 4, 2]
BAD = {1: None, 2: None, 4: (70, 200)}  # -I twice, two bad pivots in different blocks


def run(precision, nb, grid, spoil):
    plan = EB.BatchPlan(N, K, precision, [(1 << 30, nb, grid)])
    A, B = plan.empty_a(), plan.empty_b()
    EB.fill_gram(plan, A, B, 31)
    for i, cols in BAD.items() if spoil else ():
        V = plan.a_view(A, i)
        if cols is None:
            V.copy_(-torch.eye(N[i], dtype=V.dtype, device=V.device))
        else:
            for c in cols:
                V[c, c] = -5.0
    A0 = A.clone()
    plan.solve(A, B, use_graph=False)
    info, _, _ = plan.results()
    # the factor's storage: A itself, or the float copy at the workspace's start
    F = A if precision == "f64" else plan._work[:4 * plan.a_total].view(torch.float32)
    factors = [torch.tril(plan.a_view(F, i)).cpu().numpy() for i in range(len(N))]
    return plan, info, A0, factors, B


@pytest.mark.parametrize("precision,tol", [("f64", 1e-12), ("f32", 2e-5), ("bf16x3", 1e-4)])
@pytest.mark.parametrize("nb", [32, 128])
def test_not_hpd(oracle, precision, tol, nb):
    forms = [run(precision, nb, grid, True) for grid in (0, 3)]
    good = run(precision, nb, 0, False)
    for plan, info, A0, factors, B in forms:
        assert info.tolist() == [0, 1, 1, 0, 71]
        for i in range(len(N)):
            if i in BAD:
                ref = np.array(plan.a_view(A0, i).cpu().numpy(), order="F", copy=True)
                assert oracle.lvar3(ref, nb) == info[i]
                want, got = np.tril(ref), factors[i].astype(np.float64)
                assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want), i
            else:
                assert np.array_equal(factors[i], good[3][i])
                assert torch.equal(plan.b_view(B, i), plan.b_view(good[4], i))
    for a, b in zip(forms[0][3], forms[1][3]):
        assert np.array_equal(a, b)
