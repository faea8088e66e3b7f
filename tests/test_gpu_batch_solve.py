"""Solves of a batch (one workgroup per matrix): block and tile edges, and
matrices beyond the solved blocks that LDS holds (12, 20 or 32 blocks of 64
rows), one to several slabs of right-hand sides, buckets merged and apart.

Bars: FP64 normwise backward error within 4 n u (the factorization's and the
two solves' own bound, n u each at most, with room for the sums); FP32 with
refinement converges to 1e-14 in four sweeps.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from elemental_amd import batch as EB  # noqa: E402

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="no GPU")]

EDGES = [1, 2, 15, 16, 17, 63, 64, 65, 128, 129, 200]


def run(n, k, precision, buckets=None):
    plan = EB.BatchPlan(n, k, precision, buckets)
    A, B = plan.empty_a(), plan.empty_b()
    EB.fill_gram(plan, A, B, 5)
    A0, B0 = A.clone(), B.clone()
    plan.solve(A, B, use_graph=False)
    info, eta, _ = plan.results()
    assert (info == 0).all()
    return plan.backward_error(A0, B, B0)


@pytest.mark.parametrize("n,k", [(EDGES + [830, 1000], 17), (EDGES + [1281, 1400], 7), (EDGES + [2049, 2200], 3)])
@pytest.mark.parametrize("buckets", [None, [(128, 128, 0), (1 << 30, 64, 0)]])
def test_fp64(n, k, buckets):
    ks = [k - i % 3 for i in range(len(n))]
    eta = run(n, ks, "f64", buckets)
    assert (eta <= 4 * np.maximum(n, 8) * 2.0**-53).all(), eta


@pytest.mark.parametrize("k", [1, 16, 17])
def test_fp32_refined(k):
    n = EDGES + [1281, 1400]
    eta = run(n, [k] * len(n), "f32")
    assert (eta <= 1e-14).all(), eta
