"""The Navier-Stokes residual by own parts and neighbours' halves (k_ns_own, k_ns_add) at element counts that leave
both kernels' last workgroups part full, with turned element frames, against the oracle.

Tolerances: FP64 as the residual's own test (1e-12 of the largest value); FP32 and the mixed form to the bound of their
test on the 4x4 mesh, 2e-4 and 5e-6, times two for the 7 to 9 times smaller differences within an element on FP32
values of the same size.
"""
import numpy as np
import pytest

import pyoracle as O
from dpgsolver_amd import mesh as M

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

MU, PR = 0.02, 0.72


@pytest.mark.parametrize("p,shape", [(1, (13, 11)), (2, (9, 7)), (3, (7, 7)), (4, (7, 5)), (5, (5, 3))])
def test_part_full_workgroups_match_oracle(p, shape):
    from dpgsolver_amd import _lib

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    prim = M.freestream_prim(2)

    def curve(q):
        return np.stack([q[..., 0] + 0.03 * np.sin(2 * np.pi * q[..., 1]), q[..., 1] + 0.03 * np.sin(2 * np.pi * q[..., 0])], -1)

    mesh = M.structured_tp_mesh(2, p, shape, (0.0, 0.0), (1.0, 1.0), (True, True), curve=curve,
                                rotate=np.random.default_rng(p).integers(0, 4, shape[0] * shape[1]))
    x = M.nodes_xyz(mesh)
    pert = 0.05 * np.sin(2 * np.pi * x[..., 0]) * np.cos(2 * np.pi * x[..., 1])
    u = M.pack_state(M.prim_to_cons(prim[None, None, :] * (1.0 + np.stack([pert, pert, -pert, 0.5 * pert], -1)), 2))
    for flux in (M.FLUX_ROE, M.FLUX_LF):
        ref = O.Oracle(mesh, M.PDE_EULER, flux, bc_prim=prim, viscous=(MU, PR)).rhs_ns(u)
        ctx = _lib.Context(2, p, M.PDE_NAVIER_STOKES, flux, mu=MU, Pr=PR, bc_prim=prim)
        ctx.set_stream(torch.cuda.current_stream().cuda_stream)
        ctx.upload_mesh(mesh.xyz, mesh.faces)
        ud = torch.from_numpy(u).cuda()
        u32 = ud.float()
        r = torch.full_like(ud, float("nan"))
        r32, rmx = torch.full_like(u32, float("nan")), torch.full_like(u32, float("nan"))
        ctx.compute_rhs(ud.data_ptr(), r.data_ptr())
        ctx.compute_rhs_f32(u32.data_ptr(), r32.data_ptr())
        ctx.compute_rhs_mixed(ud.data_ptr(), rmx.data_ptr())
        torch.cuda.synchronize()
        scale = np.abs(ref).max()
        for got, tol in ((r, 1e-12), (r32, 4e-4), (rmx, 1e-5)):
            err = np.abs(got.double().cpu().numpy() - ref).max() / scale
            print(f"p={p} flux={flux}: {err:.2e} of {tol:.0e}", flush=True)
            assert err < tol
        ctx.close()
