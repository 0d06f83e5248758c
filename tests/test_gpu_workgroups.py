"""The residual kernels at the edges of their workgroups: element counts that leave the last workgroup part full, with
boundary faces on some elements (a branch that the face items of each order, type and direction meet in another lane
order).  FP64 to 1e-12 of max |R| and J v to 1e-12 of max |J v| (the bounds of these calls on other meshes); the mixed form
to 2e-5; FP32 to 64 units of rounding (2^-24) of the largest volume term, which the face terms cancel to R (a term passes
through some 30 multiply-adds: three sweeps, flux, divergence, lift)."""
import numpy as np
import pytest

import pyoracle as O
from dpgsolver_amd import mesh as M

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

R, W = M.BC_RIEMANN, M.BC_SLIPWALL


@pytest.mark.parametrize("d,p,n", [(2, 1, (7, 5)), (2, 1, (13, 10)), (2, 2, (5, 3)), (2, 2, (11, 9)), (2, 3, (5, 5)), (2, 4, (4, 3)),
                                   (2, 5, (5, 3)), (3, 1, (3, 3, 3)), (3, 1, (5, 4, 7)), (3, 2, (3, 3, 1)), (3, 2, (4, 3, 3)),
                                   (3, 3, (2, 2, 1)), (3, 4, (3, 1, 1))])
def test_part_full_workgroups_with_boundaries(d, p, n):
    from dpgsolver_amd import _lib

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    prim = M.freestream_prim(d)
    mesh = M.structured_tp_mesh(d, p, n, (0.0,) * d, (1.0,) * d, (False, False, True)[:d], bc_low=(R, W, R), bc_high=(R, W, R))
    x = M.nodes_xyz(mesh)
    pert = 0.05 * np.sin(2 * np.pi * x[..., 0] + 0.4) * np.cos(2 * np.pi * x[..., -1])
    u = M.pack_state(M.prim_to_cons(prim * (1.0 + np.stack([pert, pert, -pert, 0.5 * pert, pert][:d + 2], -1)), d))
    v = np.random.default_rng(p).standard_normal(u.size)
    for flux in (M.FLUX_ROE, M.FLUX_LF):
        orc = O.Oracle(mesh, M.PDE_EULER, flux, bc_prim=prim)
        ref = orc.rhs(u)
        ctx = _lib.Context(d, p, M.PDE_EULER, flux, bc_prim=prim)
        ctx.set_stream(torch.cuda.current_stream().cuda_stream)
        ctx.upload_mesh(mesh.xyz, mesh.faces)
        ud, vd = torch.from_numpy(u).cuda(), torch.from_numpy(v).cuda()
        u32 = ud.float()
        r, jv = torch.full_like(ud, float("nan")), torch.full_like(ud, float("nan"))
        r32, rmx = torch.full_like(u32, float("nan")), torch.full_like(u32, float("nan"))
        ctx.compute_rhs(ud.data_ptr(), r.data_ptr())
        ctx.compute_rhs_f32(u32.data_ptr(), r32.data_ptr())
        ctx.compute_rhs_mixed(ud.data_ptr(), rmx.data_ptr())
        torch.cuda.synchronize()
        scale = np.abs(ref).max()
        e64, emx, e32 = (np.abs(a.double().cpu().numpy() - ref).max() for a in (r, rmx, r32))
        tol32 = 64 * 2.0 ** -24 * np.abs(orc.rhs(u, "volume")).max()
        print(f"d={d} p={p} {n} flux={flux}: {e64 / scale:.1e} {emx / scale:.1e} FP32 {e32:.1e} of {tol32:.1e}", flush=True)
        assert e64 < 1e-12 * scale
        assert emx < 2e-5 * scale
        assert e32 < tol32
        if d == 3 or p <= 4:
            jref = orc.rhs_complex(u, 1e-30 * v)[1] / 1e-30
            ctx.jacobian_vector(ud.data_ptr(), vd.data_ptr(), jv.data_ptr())
            torch.cuda.synchronize()
            assert np.abs(jv.cpu().numpy() - jref).max() <= 1e-12 * np.abs(jref).max()
        ctx.close()
