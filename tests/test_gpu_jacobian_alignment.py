"""Jacobian values written to memory that is only 8-byte aligned (a slice of a
caller's buffer): the same bits as to an aligned array, and nothing beside them.
The kernels that copy whole rows in 16-byte stores: the staged first-order rows
of sample meshes, the near-boundary rows of WENO problems, the 2D and 3D box
marches, the tiled and staged WENO rows."""
import ctypes

import numpy as np
import pytest

import cases
import pressiodemoapps_amd as pda

pytestmark = pytest.mark.gpu
NAMES = ["euler2d-riemann-FirstOrder", "euler2d-riemann-Weno5", "euler2d-periodic-Weno3", "euler3d-sedov-FirstOrder",
         "euler3d-sedov-Weno3", "euler3d-sedov-big-FirstOrder", "euler1d-sod-Weno5", "swe-slipwall-Weno3",
         "adr-probA-Weno5"]
CASES = [c for c in cases.CASES + cases.BIG_CASES if c[0] in NAMES]


@pytest.mark.parametrize("sample", [False, True], ids=["full", "sample"])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_values_at_an_odd_multiple_of_eight_bytes(case, sample):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    print(f"[gpu-alignment] {case[0]} sample={sample}", flush=True)
    mesh, prob = cases.make(case)
    if sample:
        n = mesh.sampleMeshSize()
        gids = np.arange(0, n, 3) if mesh.dimensionality() == 1 else np.sort(
            np.random.default_rng(3).choice(n, size=n // 4, replace=False))
        mesh = pda.create_sample_mesh(mesh, gids)
        prob = pda.create_problem(mesh, case[1], case[2], case[7], case[8])
    U = torch.from_numpy(cases.perturbed_state(prob, 4)).cuda()
    n = prob.nonZeros()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for with_velocity in (False, True):
        V = prob.createRightHandSide() if with_velocity else None

        def values(offset):
            buf = torch.full((n + 8,), -7.0, dtype=torch.float64, device="cuda")
            assert buf.data_ptr() % 16 == 0
            rc = pda.lib().pda_jacobian(prob.handle, ctypes.c_void_p(U.data_ptr()), ctypes.c_double(0.0),
                                        ctypes.c_void_p(buf.data_ptr() + 8 * offset),
                                        ctypes.c_void_p(V.data_ptr()) if with_velocity else None, s)
            assert rc == 0, pda.lib().pda_last_error()
            torch.cuda.synchronize()
            return buf.cpu().numpy()

        want, got = values(2), values(3)
        assert np.array_equal(got[3:3 + n], want[2:2 + n])
        assert (got[:3] == -7.0).all() and (got[3 + n:] == -7.0).all()
