"""Block SGS solves on the reduced system of two-coloured meshes (compact vectors on one colour): the packed face-node
kernels of QUAD Euler at p = 1..4, with boundary faces and turned element frames, and the general form (HEX, and the
Navier-Stokes solve with its full face blocks).

The solution of one Newton step x satisfies |b - A x| <= 1.1 gmres_rtol |b|, b and A x from dgx_compute_rhs and
dgx_newton_operator (the estimate that ends GMRES is the full system's residual; the FP32 Krylov basis adds about 1e-6
to it), and the same holds for the full system that block SGS with FP32-stored blocks solves.  x is the difference of the
states, so the step must be small enough that neither the relaxation nor the limiter of the update acts.
"""
import numpy as np
import pytest

from dpgsolver_amd import mesh as M

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _case(kind, p):
    if kind == "walls":                        # slip walls and Riemann faces, odd element counts
        R, W = M.BC_RIEMANN, M.BC_SLIPWALL
        curve = lambda x: x + 0.03 * (np.sin(2 * np.pi * x[..., :1]) * np.sin(np.pi * x[..., 1:]))      # noqa: E731
        mesh = M.structured_tp_mesh(2, p, (7, 5), (0, 0), (1, 1), (False, False), curve=curve, bc_low=(R, W), bc_high=(R, W))
    else:                                      # turned frames, curved
        d, n = (3, (4, 2, 2)) if kind == "hex" else (2, (6, 4))
        curve = lambda x: x + 0.03 * np.sin(2 * np.pi * x[..., ::-1])      # noqa: E731
        mesh = M.structured_tp_mesh(d, p, n, (0,) * d, (1,) * d, (True,) * d, curve=curve,
                                    rotate=np.random.default_rng(p).integers(0, 4 * d - 4, int(np.prod(n))))
    d = mesh.d
    x = M.nodes_xyz(mesh)
    prim = M.freestream_prim(d)
    pert = 0.02 * np.sin(2 * np.pi * x[..., 0] + 0.3) * np.cos(2 * np.pi * x[..., 1])
    u = M.pack_state(M.prim_to_cons(prim * (1.0 + np.stack([pert, pert, -pert, 0.5 * pert, pert][:d + 2], -1)), d))
    return mesh, u, prim


@pytest.mark.parametrize("kind,p", [(k, p) for k in ("walls", "turned") for p in (1, 2, 3, 4)] +
                         [("hex", 1), ("hex", 2), ("ns", 1), ("ns", 3)])
def test_linear_residual_of_a_newton_step(kind, p):
    from dpgsolver_amd import _lib

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    mesh, u, prim = _case(kind, p)
    if kind == "ns":
        ctx = _lib.Context(2, p, M.PDE_NAVIER_STOKES, M.FLUX_ROE, mu=0.02, Pr=0.72)
    else:
        ctx = _lib.Context(mesh.d, p, M.PDE_EULER, M.FLUX_ROE, bc_prim=prim)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    ctx.upload_mesh(mesh.xyz, mesh.faces)
    ud = torch.from_numpy(u).to("cuda:0")
    b = torch.empty_like(ud)
    inv_dt = torch.empty(mesh.E, dtype=torch.float64, device="cuda:0")
    ctx.compute_rhs(ud.data_ptr(), b.data_ptr())
    ctx.cfl_dt(ud.data_ptr(), 20.0, inv_dt.data_ptr())
    for pc, rtol, restart in ((_lib.PC_BLOCK_SGS, 1e-5, 60), (_lib.PC_BLOCK_SGS, 1e-9, 7), (_lib.PC_BLOCK_SGS32, 1e-5, 60)):
        un = ud.clone()
        st = ctx.solve_implicit(un.data_ptr(), cfl_initial=20.0, exit_tol=1e-14, max_newton=1, gmres_restart=restart,
                                gmres_rtol=rtol, gmres_max_iter=1000, precond=pc, raise_on_error=False)
        x, ax = un - ud, torch.empty_like(ud)
        ctx.newton_operator(ud.data_ptr(), inv_dt.data_ptr(), x.data_ptr(), ax.data_ptr())
        torch.cuda.synchronize()
        rel = float((b + ax).norm() / b.norm())
        print(f"{kind} p={p} pc {pc}: {rel:.2e} of {rtol:.0e} after {st['gmres_iters']} iterations", flush=True)
        assert float(x.abs().max()) < 0.1
        assert st["gmres_not_converged"] == 0 and rel <= 1.1 * rtol
    ctx.close()
