"""How many linear iterations the implicit stepper queues between two looks at
the convergence flag.  An easy step after a hard one must cost about what it
costs by itself: the hard solve's iterations are not all queued again.  One
hard step stops at the iteration limit (3,000) and fails; the other converges
in a long solve.  The bar is a factor of 6 on the easy step's time (60 when the
count was queued without a bound), and the state is a fresh stepper's, bit for
bit."""
import time

import pytest

import pressiodemoapps_amd as pda

pytestmark = pytest.mark.gpu


def _stepper(prob, options):
    ip = pda.ImplicitStepper(prob, pda.ImplicitScheme.BDF1)
    ip.set_options(*options)
    return ip


@pytest.mark.parametrize("hard_dt,options,fails", [
    (1e4, (pda.StopRule.Residual, 1e-9, 2, 1e-12, 3000), True),
    (3.0, (pda.StopRule.Correction, 1e30, 4, 1e-14, 0), False),
])
def test_easy_step_after_a_hard_one(hard_dt, options, fails):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    print(f"[gpu-implicit-polls] hard step of {hard_dt:g}", flush=True)
    mesh = pda.create_structured_mesh((64, 64), (-1.0, 1.0, -1.0, 1.0), 7, True)
    prob = pda.create_problem(mesh, pda.AdvectionDiffusion2d.BurgersPeriodic, pda.InviscidFluxReconstruction.Weno5, 1,
                              {"diffusion": 5e-3})
    U0 = prob.initialCondition()

    def step(ip, dt):
        U = U0.clone()
        torch.cuda.synchronize()
        t = time.perf_counter()
        st = ip.step(U, 0.0, dt)
        return (time.perf_counter() - t) * 1e6, U, st

    fresh = _stepper(prob, options)
    step(fresh, 1e-4)
    alone = min(step(fresh, 1e-4)[0] for _ in range(5))
    want = step(_stepper(prob, options), 1e-4)[1]
    ip = _stepper(prob, options)
    step(ip, 1e-4)
    after = float("inf")
    for _ in range(4):
        if fails:
            with pytest.raises(pda.PdaError, match="did not converge"):
                step(ip, hard_dt)
        else:
            hard = step(ip, hard_dt)[2]
            print(f"[gpu-implicit-polls] hard: {hard['linear_iters']} iterations", flush=True)
            assert hard["linear_iters"] > 200
        us, U, _ = step(ip, 1e-4)
        after = min(after, us)
        assert torch.equal(U, want)
    print(f"[gpu-implicit-polls] easy step {alone:.0f} us alone, {after:.0f} us after the hard one", flush=True)
    assert after <= 6 * alone
