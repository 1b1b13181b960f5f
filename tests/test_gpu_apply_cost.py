"""What applyJacobian costs at column counts on either side of its kernels'
change: a few row-major columns are summed over the entries of a cell's rows
(fewer than 8) or taken over the lanes (8 and more), and fewer columns of the
same Jacobian cost no more than many.  Five columns move under half the bytes
of twelve; the bar is one and a half times their time, against three times
when the sums of the entry kernel were chosen by a searched index."""
import time

import pytest

import pressiodemoapps_amd as pda

pytestmark = pytest.mark.gpu
S = pda.InviscidFluxReconstruction


@pytest.mark.parametrize("enum,n,scheme,st,few", [
    (pda.AdvectionDiffusion2d.BurgersPeriodic, (500, 512), S.FirstOrder, 3, 5),
    (pda.AdvectionDiffusion2d.BurgersPeriodic, (500, 512), S.Weno3, 5, 5),
    (pda.Euler2d.PeriodicSmooth, (300, 310), S.FirstOrder, 3, 3),
])
def test_few_columns_cost_no_more_than_many(enum, n, scheme, st, few):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    print(f"[gpu-apply-cost] {enum!r} {n} {scheme.name}", flush=True)
    prob = pda.create_problem(pda.create_structured_mesh(n, (-1.0, 1.0, -1.0, 1.0), st, True), enum, scheme)
    U = prob.initialCondition()

    def cost(cols):
        B = torch.rand(prob.totalDofStencilMesh(), cols, dtype=torch.float64, device="cuda")
        AJ = prob.createApplyJacobianResult(B)
        best = float("inf")
        for _ in range(6):
            torch.cuda.synchronize()
            t = time.perf_counter()
            for _ in range(10):
                prob.applyJacobian(U, B, 0.0, AJ)
            torch.cuda.synchronize()
            best = min(best, (time.perf_counter() - t) / 10 * 1e6)
        return best

    a, b = cost(few), cost(12)
    print(f"[gpu-apply-cost] {few} columns {a:.1f} us, 12 columns {b:.1f} us", flush=True)
    assert a <= 1.5 * b
