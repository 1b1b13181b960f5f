"""States of very large magnitude.  With every cell difference far above the
WENO schemes' epsilon (1e-6), the Euler right hand side is homogeneous of
degree one in the state, Burgers' of degree two and the linear problem's of
degree one, and a power of two in the state is the same power (or its square)
in the results, bit for bit but for terms below the last place.  The results at
2^100 are in every kernel's range; those at the larger scales must be theirs.
(Moderate states have their parity tests.)"""
import numpy as np
import pytest

import cases
import pressiodemoapps_amd as pda

pytestmark = pytest.mark.gpu
S = pda.InviscidFluxReconstruction
BASE = 100
NAMES = ["euler1d-sod", "euler1d-periodic", "euler2d-riemann", "euler2d-periodic", "burgers-periodic",
         "burgers-outflow", "adr-probA", "euler3d-sedov"]
CASES = [c for c in cases.CASES if c[0].rsplit("-", 1)[0] in NAMES and c[2] != S.FirstOrder]


def _problem(case, sample):
    mesh, prob = cases.make(case)
    if sample:
        n = mesh.sampleMeshSize()
        gids = np.arange(0, n, 3) if mesh.dimensionality() == 1 else np.sort(
            np.random.default_rng(3).choice(n, size=n // 5, replace=False))
        mesh = pda.create_sample_mesh(mesh, gids)
        prob = pda.create_problem(mesh, case[1], case[2], case[7], case[8])
    return mesh, prob


def _cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


@pytest.mark.parametrize("sample", [False, True], ids=["full", "sample"])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_jacobian_at_large_magnitudes(case, sample):
    """to 2^130 (1.4e39), to which the reference's gradients hold"""
    torch = _cuda()
    print(f"[gpu-wide] jacobian {case[0]} sample={sample}", flush=True)
    mesh, prob = _problem(case, sample)
    U = cases.perturbed_state(prob, 4)
    J = prob.createJacobian()

    def at(scale):
        prob.jacobian(torch.from_numpy(U * 2.0 ** scale).cuda(), 0.0, J)
        return J.values.cpu().numpy().copy()

    base = at(BASE)
    assert np.isfinite(base).all()
    degree = 1 if case[0].startswith("burgers") else 0
    for scale in (115, 124, 130):
        got = at(scale) * 2.0 ** (-degree * (scale - BASE))
        assert np.isfinite(got).all(), scale
        assert cases.rel_err(got, base) <= 1e-14, scale


ROWS = [c for c in CASES if c[0].startswith("euler1d")]


def _scales(case):
    return (114, 140, 170) if case[2] == S.Weno5 else (114, 170, 240)


@pytest.mark.parametrize("case,sample", [(c, False) for c in ROWS] + [(c, True) for c in CASES],
                         ids=[f"{c[0]}-full" for c in ROWS] + [f"{c[0]}-sample" for c in CASES])
def test_velocity_rows_at_large_magnitudes(case, sample):
    """to 2^170 (1.5e51) with WENO5 and 2^240 (1.8e72) with WENO3: the rows outside
    the structured boxes, alone and with the Jacobian's"""
    torch = _cuda()
    print(f"[gpu-wide] velocity {case[0]} sample={sample}", flush=True)
    _, prob = _problem(case, sample)
    U = cases.perturbed_state(prob, 4)
    V, J = prob.createRightHandSide(), prob.createJacobian()

    def at(scale, with_jacobian):
        Ud = torch.from_numpy(U * 2.0 ** scale).cuda()
        if with_jacobian:
            prob.rightHandSideAndJacobian(Ud, 0.0, V, J)
        else:
            prob.rightHandSide(Ud, 0.0, V)
        return V.cpu().numpy() * 2.0 ** (-degree * (scale - BASE))

    degree = 2 if case[0].startswith("burgers") else 1
    base = at(BASE, False)
    assert np.isfinite(base).all()
    for scale in _scales(case):
        got = at(scale, False)
        assert np.isfinite(got).all(), scale
        assert cases.rel_err(got, base) <= 1e-14, scale
    base = at(BASE, True)
    for scale in (114, 130):  # as far as the gradients beside it hold
        got = at(scale, True)
        assert np.isfinite(got).all(), scale
        assert cases.rel_err(got, base) <= 1e-14, scale


@pytest.mark.parametrize("name", ["SSPRK3", "RK4", "ForwardEuler"])
@pytest.mark.parametrize("case", ROWS, ids=[c[0] for c in ROWS])
def test_steps_at_large_magnitudes(case, name):
    """the 1D steps in one launch, and the stages row by row"""
    torch = _cuda()
    print(f"[gpu-wide] steps {case[0]} {name}", flush=True)
    _, prob = _problem(case, False)
    U = cases.perturbed_state(prob, 4)

    def at(scale):
        Ud = torch.from_numpy(U * 2.0 ** scale).cuda()
        pda.ExplicitStepper(prob, getattr(pda.StepScheme, name)).advance(Ud, 1e-4, 13)
        return Ud.cpu().numpy() * 2.0 ** -(scale - BASE)

    base = at(BASE)
    assert np.isfinite(base).all() and not np.array_equal(base, U * 2.0 ** BASE)
    for scale in _scales(case):
        got = at(scale)
        assert np.isfinite(got).all(), scale
        assert cases.rel_err(got, base) <= 1e-14, scale
