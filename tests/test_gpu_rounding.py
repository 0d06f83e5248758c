"""Roundings of the FP32 and mixed residuals.

The mixed Navier-Stokes residual by own parts and halves rounds no more than the gradient-trace kernels, which compute the
same elements on a mesh with one element of another order: the 2-norm of its error against FP64, over the elements that do
not touch that one, is at most 1.005 times theirs (two error sums over 360000 and more values of independent roundings
agree to 0.2%)."""
import numpy as np
import pytest

from dpgsolver_amd import mesh as M

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,n", [(1, 200), (2, 150)])
def test_mixed_error_is_that_of_the_gradient_trace_kernels(p, n):
    from dpgsolver_amd import _lib

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    E, nv, Np = n * n, 4, (p + 1) ** 2
    uni = M.structured_tp_mesh(2, p, (n, n), (0.0, 0.0), (1.0, 1.0), (True, True))
    state = lambda x: M.prim_to_cons(M.smooth_state_3d(x), 2)      # noqa: E731
    u = M.pack_state(state(M.nodes_xyz(uni)))
    pe = np.full(E, p, dtype=np.int32)
    odd = E - 1                                                    # (the groups come in order of p: it stays last)
    pe[odd] = p + 1
    mesh = M.structured_hp_mesh(pe, (n, n), (0.0, 0.0), (1.0, 1.0), (True, True))
    uh = M.hp_state(mesh, state)
    k = (E - 1) * nv * Np
    err = []
    for hp in (True, False):
        ctx = _lib.Context(2, p + 1 if hp else p, M.PDE_NAVIER_STOKES, M.FLUX_ROE, mu=0.02, Pr=0.72)
        ctx.set_stream(torch.cuda.current_stream().cuda_stream)
        ctx.upload_mesh_hp(mesh) if hp else ctx.upload_mesh(uni.xyz, uni.faces)
        ud = torch.from_numpy(uh if hp else u).cuda()
        r, rm = torch.empty_like(ud), torch.empty(ud.shape, dtype=torch.float32, device="cuda:0")
        ctx.compute_rhs(ud.data_ptr(), r.data_ptr())
        ctx.compute_rhs_mixed(ud.data_ptr(), rm.data_ptr())
        torch.cuda.synchronize()
        assert torch.equal(ud[:k].cpu(), torch.from_numpy(u[:k]))
        far = torch.ones(E - 1, dtype=torch.bool, device="cuda:0")
        x, y = odd % n, odd // n
        for i, j in ((x - 1, y), ((x + 1) % n, y), (x, y - 1), (x, (y + 1) % n)):
            far[i + n * j] = False
        d = (rm[:k].double() - r[:k]).reshape(E - 1, nv * Np)[far]
        err.append(float(d.norm()))
        ctx.close()
    print(f"p={p}: {err[1] / err[0]:.4f}", flush=True)
    assert err[1] <= 1.005 * err[0]


@pytest.mark.parametrize("flux,ieee", [(M.FLUX_ROE, 2.048e-5), (M.FLUX_LF, 2.176e-5)])
def test_fp32_faces_of_tri_quad_meshes_take_rounded_normals(flux, ieee):
    """The faces with a TRI side normalise n J_f with the correctly rounded square root and quotient in FP32 too: the 2-norm
    of the error of the Euler residual against FP64 (of the same FP32 state) is then `ieee`; the hardware's approximations
    gave 1.02 times that."""
    from dpgsolver_amd import _lib

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mesh = M.config4_mixed_mesh(90, 60)
    u32 = torch.from_numpy(M.config4_mixed_state(mesh)).cuda().float()
    u = u32.double()
    ctx = _lib.Context(2, 5, M.PDE_EULER, flux)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    ctx.upload_mesh_mixed(mesh)
    r, r32 = torch.empty_like(u), torch.empty_like(u32)
    ctx.compute_rhs(u.data_ptr(), r.data_ptr())
    ctx.compute_rhs_f32(u32.data_ptr(), r32.data_ptr())
    torch.cuda.synchronize()
    err = float((r32.double() - r).norm() / r.norm())
    print(f"flux {flux}: {err:.3e}", flush=True)
    assert err <= 1.01 * ieee
    ctx.close()
