"""The implicit stepper where device memory is short: with less than twice its
second matrix left, it keeps the iteration's matrix in the Jacobian's place.  The
same steps must come out: to the same tolerance, with as many Newton and (to the
rounding of the sums) linear iterations.  Most of the device's memory is taken by
a few allocations meanwhile; what is left holds the stepper without its second
matrix and half of that matrix again."""
import pytest

import pressiodemoapps_amd as pda

pytestmark = pytest.mark.gpu
S = pda.InviscidFluxReconstruction


PROBLEMS = [
    (pda.AdvectionDiffusion2d.BurgersPeriodic, (700, 701), (-1.0, 1.0) * 2, S.Weno5, 7, 1, True),
    (pda.Swe2d.SlipWall, (400, 403), (-5.0, 5.0) * 2, S.Weno3, 5, 1, ()),
    (pda.Euler3d.SedovSymmetry, (40, 41, 42), (0.0, 1.2) * 3, S.FirstOrder, 3, None, ()),
]


def test_steps_with_little_memory_left():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    dt = 2e-4

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    def take(leave):
        """allocations that leave that much (one of nearly everything leaves more)"""
        held = []
        for _ in range(8):
            over = free() - leave
            if over < 24 << 20:
                break
            held.append(torch.empty(over, dtype=torch.uint8, device="cuda"))
        return held

    def run(prob):
        """(memory, state, statistics) of a stepper's three steps"""
        before = free()
        ip = pda.ImplicitStepper(prob, pda.ImplicitScheme.BDF1)
        size = before - free()
        ip.set_options(pda.StopRule.Residual, 1e-9, 12, 1e-12, 0)
        U, out = prob.initialCondition(), []
        for k in range(3):
            out.append(ip.step(U, k * dt, dt))
        return size, U, out

    cases = []
    for enum, n, bounds, scheme, st, ic, periodic in PROBLEMS:
        print(f"[gpu-implicit-memory] {enum!r} {n}", flush=True)
        args = (pda.create_structured_mesh(n, bounds, st, periodic), enum, scheme) + (() if ic is None else (ic,))
        prob = pda.create_problem(*args)
        prob.rightHandSide(prob.initialCondition(), 0.0, prob.createRightHandSide())  # the problem's own tables
        cases.append((prob, *run(prob)))
    most = take(1 << 30)
    for prob, full, U, stats in cases:
        second = 8 * prob.nonZeros() * 0.85  # its second matrix is a little less than the Jacobian
        rest = take(int(full - 0.5 * second))
        little, V, few = run(prob)
        del rest
        torch.cuda.empty_cache()
        most += take(1 << 30)
        print(f"[gpu-implicit-memory] stepper {full / 1e6:.0f} MB and {little / 1e6:.0f} MB; linear "
              f"{[s['linear_iters'] for s in stats]} {[s['linear_iters'] for s in few]}", flush=True)
        assert little < full - 0.7 * second
        for a, b in zip(stats, few):
            assert b["converged"] and b["residual_norm"] <= 1e-9
            assert a["newton_iters"] == b["newton_iters"] and abs(a["linear_iters"] - b["linear_iters"]) <= 2
        # both states solve R = 0 to 1e-9 in the l2 norm, with a Jacobian I - dt df/dy
        # whose inverse is below 2 for these steps
        assert float(torch.linalg.vector_norm(U - V)) <= 3 * 2 * 2e-9
    del most
    torch.cuda.empty_cache()
