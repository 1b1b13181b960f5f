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


def _cost(prob, U, cols):
    import torch
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


def test_odd_columns_cost_little_more_than_even():
    """33 columns, one to a lane, against 32, two to a lane: 1.03 times the bytes
    in twice the accesses, at most 1.8 times the time (2.3 times with the lanes
    rounded up to a power of two)."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    mesh = pda.create_structured_mesh((600, 500), (0.0, 1.0, 0.0, 1.0), 3)
    prob = pda.create_problem(mesh, pda.AdvectionDiffusionReaction2d.ProblemA, S.FirstOrder)
    U = torch.rand(prob.totalDofStencilMesh(), dtype=torch.float64, device="cuda")
    a, b = _cost(prob, U, 33), _cost(prob, U, 32)
    print(f"[gpu-apply-cost] 33 columns {a:.1f} us, 32 columns {b:.1f} us", flush=True)
    assert a <= 1.8 * b


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

    a, b = _cost(prob, U, few), _cost(prob, U, 12)
    print(f"[gpu-apply-cost] {few} columns {a:.1f} us, 12 columns {b:.1f} us", flush=True)
    assert a <= 1.5 * b
