"""applyJacobian against the CSR product of the same problem's jacobian():
every block size, full and sample meshes (merged columns among them), the
column counts at which the kernels change (one column, row-major from 8 on,
two columns a lane, more columns than a wavefront's lanes), column-major and
row-major, and operands that are only 8-byte aligned.  Tolerance: a row sums at
most 13 blocks of 4 or 19 of 5 products, so two summation orders differ by
less than 2 * 95 ulps of the sum of the products' magnitudes."""
import numpy as np
import pytest

import cases
import pressiodemoapps_amd as pda

pytestmark = pytest.mark.gpu

S = pda.InviscidFluxReconstruction
MERGED = ("burgers-merged-Weno5", pda.AdvectionDiffusion2d.BurgersPeriodic, S.Weno5, (5, 6), (-1, 1, -1, 1), 7,
          True, 1, {"diffusion": 1e-3})
NAMES = ["euler1d-sod-Weno5", "euler2d-riemann-Weno5", "swe-slipwall-Weno3", "burgers-outflow-FirstOrder",
         "adr-probA-Weno5", "euler3d-sedov-FirstOrder"]
CASES = [c for c in cases.CASES if c[0] in NAMES] + [MERGED]


@pytest.mark.parametrize("sample", [False, True], ids=["full", "sample"])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_apply_jacobian_columns_and_layouts(case, sample):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    print(f"[gpu-apply] {case[0]} sample={sample}", flush=True)
    mesh, prob = cases.make(case)
    rng = np.random.default_rng(3)
    if sample:
        if case is MERGED or mesh.dimensionality() == 1:
            gids = np.arange(0, mesh.sampleMeshSize(), 3)
        else:
            n = mesh.sampleMeshSize()
            gids = np.sort(rng.choice(n, size=n // 5, replace=False))
        mesh = pda.create_sample_mesh(mesh, gids)
        prob = pda.create_problem(mesh, case[1], case[2], case[7], case[8])
    U = torch.from_numpy(cases.perturbed_state(prob, 4)).cuda()
    J = prob.createJacobian()
    prob.jacobian(U, 0.0, J)
    A = J.to_scipy()
    nst = prob.totalDofStencilMesh()
    for ncols in (1, 2, 3, 7, 8, 9, 32, 33, 130):
        B = rng.standard_normal((nst, ncols))
        ref, mag = A @ B, abs(A) @ abs(B)
        flat = torch.empty(nst * ncols + 1, dtype=torch.float64, device="cuda")
        odd = flat[1:].view(nst, ncols)  # 8-byte aligned
        odd.copy_(torch.from_numpy(B))
        rowm = torch.from_numpy(B).cuda()
        colm = torch.from_numpy(np.ascontiguousarray(B.T)).cuda().t()
        for what, Bt in (("row", rowm), ("odd", odd), ("column", colm)):
            AJ = prob.createApplyJacobianResult(Bt)
            prob.applyJacobian(U, Bt, 0.0, AJ)
            err = np.abs(AJ.cpu().numpy() - ref)
            assert (err <= 2 * 95 * 2.3e-16 * mag + 1e-300).all(), (what, ncols, err.max())
    b = torch.from_numpy(B[:, 0].copy()).cuda()
    out = prob.createApplyJacobianResult(b)
    prob.applyJacobian(U, b, 0.0, out)
    assert (np.abs(out.cpu().numpy() - ref[:, 0]) <= 2 * 95 * 2.3e-16 * mag[:, 0] + 1e-300).all()
