"""Block SGS on two-coloured meshes whose elements are their own neighbours (one element across a periodic direction).

* dgx_precond_apply does not depend on what its output buffer held and equals the sweeps run in numpy from z = 0 over
  the assembled blocks (self-coupling faces included) to 1e-11 (FP32-stored blocks: 1e-5), the bounds of the sweeps on
  other meshes.
* The linear residual that solve_implicit leaves, |b - A x| / |b| with b and A x from dgx_compute_rhs and
  dgx_newton_operator, is at most 1.1 times the gmres_rtol it was asked for (the FP32 Krylov basis adds about 1e-6).
"""
import numpy as np
import pytest

from dpgsolver_amd import mesh as M

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def _case(name):
    ns = name.startswith("ns")
    d, p, n = {"quad_4x1_p3": (2, 3, (4, 1)), "quad_2x1_p2": (2, 2, (2, 1)), "hex_4x1x1_p1": (3, 1, (4, 1, 1)),
               "ns_4x1_p2": (2, 2, (4, 1))}[name]
    mesh = M.structured_tp_mesh(d, p, n, (0.0,) * d, tuple(0.5 * k for k in n), (True,) * d)
    x = M.nodes_xyz(mesh)
    prim = M.freestream_prim(d)
    k = np.pi * np.array([4.0 / n[0]] + [4.0] * (d - 1))
    pert = 0.03 * np.sin(k[0] * x[..., 0] + 0.3) * np.cos(k[1] * x[..., 1])
    u = M.pack_state(M.prim_to_cons(prim * (1.0 + np.stack([pert, pert, -pert, 0.5 * pert, pert][:d + 2], -1)), d))
    return mesh, u, (dict(pde=M.PDE_NAVIER_STOKES, kw=dict(mu=0.02, Pr=0.72)) if ns else dict(pde=M.PDE_EULER, kw={}))


def _context(mesh, pde, kw):
    from dpgsolver_amd import _lib

    ctx = _lib.Context(mesh.d, mesh.p, pde, M.FLUX_ROE, **kw)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    ctx.upload_mesh(mesh.xyz, mesh.faces)
    return ctx


NAMES = ["quad_4x1_p3", "quad_2x1_p2", "hex_4x1x1_p1", "ns_4x1_p2"]


@pytest.mark.parametrize("name", NAMES)
def test_sgs_apply_starts_from_zero(dev, name):
    from dpgsolver_amd import _lib

    mesh, u, how = _case(name)
    ctx = _context(mesh, **how)
    nb, nf, E = ctx.Np * ctx.nv, 2 * mesh.d, mesh.E
    ud = torch.from_numpy(u).to(dev)
    inv_dt = torch.empty(E, dtype=torch.float64, device=dev)
    ctx.cfl_dt(ud.data_ptr(), 5.0, inv_dt.data_ptr())
    fb = torch.zeros(E * nf * nb * nb, dtype=torch.float64, device=dev)
    db = torch.zeros(E * nb * nb, dtype=torch.float64, device=dev)
    ctx.assemble_face_blocks(ud.data_ptr(), fb.data_ptr())
    ctx.assemble_diag_blocks(ud.data_ptr(), inv_dt.data_ptr(), db.data_ptr())
    v = np.random.default_rng(23).standard_normal(u.size)
    vd = torch.from_numpy(v).to(dev)
    out = {}
    for pc in (_lib.PC_BLOCK_SGS, _lib.PC_BLOCK_SGS32):
        z = torch.full_like(ud, float("nan"))
        ctx.precond_apply(pc, ud.data_ptr(), inv_dt.data_ptr(), vd.data_ptr(), z.data_ptr())
        torch.cuda.synchronize()
        out[pc] = z.cpu().numpy()
    F, D, V = fb.cpu().numpy().reshape(E, nf, nb, nb), db.cpu().numpy().reshape(E, nb, nb), v.reshape(E, nb)
    nbr = {}
    for eL, fL, eR, fR, _, _ in mesh.faces:
        nbr[(eL, fL)], nbr[(eR, fR)] = eR, eL
    assert any(n == e for (e, _), n in nbr.items())
    col = np.arange(E) % 2                       # a chain of an even number of elements
    z = np.zeros_like(V)
    for k in (0, 1, 0):                          # the last colour's update is not repeated
        zold = z.copy()
        for e in np.flatnonzero(col == k):
            z[e] = np.linalg.solve(D[e], V[e] - sum(F[e, lf] @ zold[nbr[(e, lf)]] for lf in range(nf)))
    scale = np.abs(z).max()
    e64 = np.abs(out[_lib.PC_BLOCK_SGS] - z.ravel()).max() / scale
    e32 = np.abs(out[_lib.PC_BLOCK_SGS32] - z.ravel()).max() / scale
    print(f"{name}: {e64:.2e} {e32:.2e}", flush=True)
    assert e64 < 1e-11 and e32 < 1e-5
    ctx.close()


@pytest.mark.parametrize("name", NAMES)
def test_linear_residual_is_what_gmres_reports(dev, name):
    from dpgsolver_amd import _lib

    mesh, u, how = _case(name)
    ctx = _context(mesh, **how)
    ud = torch.from_numpy(u).to(dev)
    b = torch.empty_like(ud)
    inv_dt = torch.empty(mesh.E, dtype=torch.float64, device=dev)
    ctx.compute_rhs(ud.data_ptr(), b.data_ptr())
    ctx.cfl_dt(ud.data_ptr(), 20.0, inv_dt.data_ptr())
    for pc in (_lib.PC_BLOCK_SGS, _lib.PC_BLOCK_SGS32, _lib.PC_BLOCK_JACOBI):
        un = ud.clone()
        st = ctx.solve_implicit(un.data_ptr(), cfl_initial=20.0, exit_tol=1e-14, max_newton=1, gmres_restart=60,
                                gmres_rtol=1e-5, gmres_max_iter=400, precond=pc, raise_on_error=False)
        x, ax = un - ud, torch.empty_like(ud)
        ctx.newton_operator(ud.data_ptr(), inv_dt.data_ptr(), x.data_ptr(), ax.data_ptr())
        torch.cuda.synchronize()
        rel = float((b + ax).norm() / b.norm())
        print(f"{name} pc {pc}: linear residual {rel:.2e} after {st['gmres_iters']} iterations", flush=True)
        assert st["gmres_not_converged"] == 0 and rel <= 1.1e-5
    ctx.close()
