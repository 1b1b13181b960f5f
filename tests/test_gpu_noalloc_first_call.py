"""pda_apply_jacobian_noalloc after any evaluation, as its header says: the
product reads the block tables alone, which the first evaluation uploads."""
import ctypes

import pytest

import cases
import pressiodemoapps_amd as pda

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", ["velocity", "jacobian", "pattern", "apply", "implicit"])
def test_accepted_after_any_evaluation(first):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    print(f"[no-alloc] after {first}", flush=True)
    case = [c for c in cases.CASES if c[0] == "swe-slipwall-Weno3"][0]
    _, prob = cases.make(case)
    _, other = cases.make(case)
    L, s = pda.lib(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    f = L.pda_apply_jacobian_noalloc
    vp = ctypes.c_void_p
    f.argtypes, f.restype = [vp, vp, ctypes.c_double, vp, ctypes.c_int64, ctypes.c_int, vp, vp], ctypes.c_int
    U = torch.from_numpy(cases.perturbed_state(prob, 3)).cuda()
    B = torch.rand(prob.totalDofStencilMesh(), 3, dtype=torch.float64, device="cuda")
    out, want = (torch.full((prob.totalDofSampleMesh(), 3), float("nan"), dtype=torch.float64, device="cuda")
                 for _ in range(2))
    if first == "velocity":
        prob.rightHandSide(U, 0.0, prob.createRightHandSide())
    elif first == "jacobian":  # through the C interface: the values alone
        J = torch.empty(prob.nonZeros(), dtype=torch.float64, device="cuda")
        assert L.pda_jacobian(prob.handle, vp(U.data_ptr()), ctypes.c_double(0.0), vp(J.data_ptr()), None, s) == 0
    elif first == "pattern":
        n = [ctypes.c_int64(), ctypes.c_int64(), vp(), vp()]
        assert L.pda_jacobian_pattern(prob.handle, *[ctypes.byref(x) for x in n]) == 0
    elif first == "apply":
        prob.applyJacobian(U, B, 0.0, want)
    else:
        pda.ImplicitStepper(prob, pda.ImplicitScheme.BDF1)
    rc = f(prob.handle, vp(U.data_ptr()), 0.0, vp(B.data_ptr()), 3, 1, vp(out.data_ptr()), s)
    assert rc == 0, L.pda_last_error()
    other.applyJacobian(U, B, 0.0, want)
    torch.cuda.synchronize()
    assert torch.equal(out, want)
