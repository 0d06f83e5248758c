"""GPU parity of the 3-D (HEX, Euler) linearisation and implicit solve against the oracle.

* J v (dgx_jacobian_vector: the fused residual kernel in dual numbers, 3-D) equals the oracle's complex step of
  the residual to 1e-12 relative on curved periodic HEX meshes with rotated element numberings (every face
  orientation), p = 1..4, Lax-Friedrichs and Roe.
* The diagonal blocks (dgx_assemble_diag_blocks) equal the oracle's complex-step blocks, the reference's own
  linearisation check (test_integration_linearization.c:377), with and without the -s_e M_e term.
* dgx_newton_operator equals dgx_jacobian_vector followed by dgx_mass_sub; the pseudo-time step has its closed
  form on a uniform state.
* A steady solve on a 3-D box with Riemann faces (p = 1; block-Jacobi, block SGS with FP64 and FP32-stored
  blocks, and no preconditioner; p = 2 with block-Jacobi and block SGS over 135 x 135 blocks) reaches max |R|
  < 1e-10 from a perturbed free stream; the oracle's residual of the result agrees, and block SGS takes fewer GMRES iterations
  than block-Jacobi.
* The 3-D face blocks, the block-sparse export and the SGS sweeps are checked against the oracle and numpy with
  the 2-D ones (test_gpu_solvers.py, the hex_* cases).
* 3-D paths with no counterpart here (FP32 J v, blocks beyond the batched inverse and LU: p >= 3) return
  DGX_ERR_UNSUPPORTED.
"""
import numpy as np
import pytest

import pyoracle as O
from dpgsolver_amd import mesh as M

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def _rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


def _ctx(mesh, flux, bc_prim=None):
    from dpgsolver_amd import _lib

    ctx = _lib.Context(3, mesh.p, M.PDE_EULER, flux, bc_prim=bc_prim)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    ctx.upload_mesh(mesh.xyz, mesh.faces)
    return ctx


def _curved(p, n, seed):
    curve = lambda pts: pts + 0.03 * np.sin(2 * np.pi * pts[..., [1, 2, 0]])
    mesh = M.structured_tp_mesh(3, p, (n, n, n), (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), (True, True, True), curve=curve,
                                rotate=np.random.default_rng(seed).integers(0, 8, n ** 3))
    u = M.pack_state(M.prim_to_cons(M.smooth_state_3d(M.nodes_xyz(mesh)), 3))
    return mesh, u


CASES = [(p, flux) for p in (1, 2, 3, 4) for flux in (M.FLUX_LF, M.FLUX_ROE)]


@pytest.mark.parametrize("p,flux", CASES, ids=[f"p{p}_{'lf' if f == M.FLUX_LF else 'roe'}" for p, f in CASES])
def test_jacobian_vector_3d_matches_complex_step(dev, p, flux):
    mesh, u = _curved(p, 2, p)
    print(f"HEX p={p} flux={flux}", flush=True)
    ctx = _ctx(mesh, flux)
    v = np.random.default_rng(9).standard_normal(u.size)
    ud, vd = torch.from_numpy(u).to(dev), torch.from_numpy(v).to(dev)
    jv = torch.full_like(ud, float("nan"))
    ctx.jacobian_vector(ud.data_ptr(), vd.data_ptr(), jv.data_ptr())
    torch.cuda.synchronize()
    h = 1e-30
    _, im = O.Oracle(mesh, M.PDE_EULER, flux).rhs_complex(u, h * v)
    err = _rel(jv.cpu().numpy(), im / h)
    print(f"  J v rel err {err:.1e}", flush=True)
    assert err < 1e-12
    sc = np.random.default_rng(19).uniform(0.5, 30.0, mesh.E)
    sd = torch.from_numpy(sc).to(dev)
    a = torch.full_like(ud, float("nan"))
    ctx.newton_operator(ud.data_ptr(), sd.data_ptr(), vd.data_ptr(), a.data_ptr())
    ctx.mass_sub(vd.data_ptr(), sd.data_ptr(), jv.data_ptr())
    torch.cuda.synchronize()
    assert _rel(a.cpu().numpy(), jv.cpu().numpy()) < 1e-13
    ctx.close()


@pytest.mark.parametrize("p", [1, 2])
def test_diag_blocks_3d_match_complex_step(dev, p):
    mesh, u = _curved(p, 2, 10 + p)
    ctx = _ctx(mesh, M.FLUX_ROE)
    nb = ctx.Np * ctx.nv
    ud = torch.from_numpy(u).to(dev)
    blocks = torch.full((mesh.E * nb * nb,), float("nan"), dtype=torch.float64, device=dev)
    ctx.assemble_diag_blocks(ud.data_ptr(), None, blocks.data_ptr())
    torch.cuda.synchronize()
    g = blocks.cpu().numpy().reshape(mesh.E, nb, nb)
    orc = O.Oracle(mesh, M.PDE_EULER, M.FLUX_ROE)
    ref = orc.diag_blocks(u)
    for e in range(mesh.E):
        assert np.abs(g[e] - ref[e]).max() <= 1e-12 * np.abs(ref[e]).max(), e
    s = np.linspace(0.5, 2.0, mesh.E)
    sd = torch.from_numpy(s).to(dev)
    ctx.assemble_diag_blocks(ud.data_ptr(), sd.data_ptr(), blocks.data_ptr())
    torch.cuda.synchronize()
    g2 = blocks.cpu().numpy().reshape(mesh.E, nb, nb)
    for e in (0, mesh.E - 1):
        Mm = np.kron(np.eye(ctx.nv), orc.mass(e))
        assert np.abs(g2[e] - (ref[e] - s[e] * Mm)).max() <= 1e-12 * np.abs(ref[e]).max()
    ctx.close()


def test_cfl_dt_3d_closed_form(dev):
    mesh = M.structured_tp_mesh(3, 2, (3, 2, 2), (0.0, 0.0, 0.0), (1.5, 0.8, 0.6), (True, True, True))
    prim = M.freestream_prim(3)
    ctx = _ctx(mesh, M.FLUX_ROE)
    ud = torch.from_numpy(M.uniform_state(mesh, prim)).to(dev)
    inv = torch.empty(mesh.E, dtype=torch.float64, device=dev)
    ctx.cfl_dt(ud.data_ptr(), 7.0, inv.data_ptr())
    torch.cuda.synchronize()
    ws = abs(prim[1]) + np.sqrt(1.4 * prim[4] / prim[0])
    np.testing.assert_allclose(inv.cpu().numpy(), ws / (7.0 * 0.3), rtol=1e-13)   # h_min = 0.6 / 2
    ctx.close()


def _box(p=1):
    prim = M.freestream_prim(3)
    R = M.BC_RIEMANN
    mesh = M.structured_tp_mesh(3, p, (4, 3, 3), (0.0, 0.0, 0.0), (1.0, 0.75, 0.75), (False, True, True),
                                bc_low=(R, R, R), bc_high=(R, R, R))
    x = M.nodes_xyz(mesh)
    pert = 0.02 * np.sin(3 * x[..., 0]) * np.cos(2 * x[..., 1]) * np.cos(x[..., 2])
    u = M.pack_state(M.prim_to_cons(prim[None, None, :] * (1.0 + np.stack([pert, pert, -pert, pert, 0.5 * pert], -1)), 3))
    return mesh, u, prim


def test_steady_box_3d_newton_gmres(dev):
    from dpgsolver_amd import _lib

    mesh, u0, prim = _box()
    ctx = _ctx(mesh, M.FLUX_ROE, bc_prim=prim)
    its = {}
    for pc in (_lib.PC_BLOCK_JACOBI, _lib.PC_NONE, _lib.PC_BLOCK_SGS, _lib.PC_BLOCK_SGS32):
        ud = torch.from_numpy(u0).to(dev)
        st = ctx.solve_implicit(ud.data_ptr(), cfl_initial=5.0, cfl_max=300.0, exit_tol=1e-10, max_newton=60,
                                precond=pc)
        print("3-D box, precond", pc, "newton", st["newton_steps"], "gmres", st["gmres_iters"], st["seconds"],
              flush=True)
        assert st["converged"] == 1 and st["max_rhs"] < 1e-10
        its[pc] = st["gmres_iters"]
        r = O.Oracle(mesh, M.PDE_EULER, M.FLUX_ROE, bc_prim=prim).rhs(ud.cpu().numpy())
        assert np.abs(r).max() < 1e-9
    assert its[_lib.PC_BLOCK_SGS] < its[_lib.PC_BLOCK_JACOBI]
    ctx.close()


def test_steady_box_3d_p2_block_jacobi_and_sgs(dev):
    """p = 2 (nb = 135): block-Jacobi and block SGS over batched inverses of 146 KB blocks (270 face dofs per
    element in the SGS sweep)."""
    from dpgsolver_amd import _lib

    mesh, u0, prim = _box(2)
    ctx = _ctx(mesh, M.FLUX_ROE, bc_prim=prim)
    its = {}
    for pc in (_lib.PC_BLOCK_JACOBI, _lib.PC_BLOCK_SGS):
        ud = torch.from_numpy(u0).to(dev)
        st = ctx.solve_implicit(ud.data_ptr(), cfl_initial=5.0, cfl_max=300.0, exit_tol=1e-10, max_newton=60,
                                precond=pc)
        print("3-D box p=2, precond", pc, "newton", st["newton_steps"], "gmres", st["gmres_iters"], st["seconds"],
              flush=True)
        assert st["converged"] == 1 and st["max_rhs"] < 1e-10
        its[pc] = st["gmres_iters"]
        r = O.Oracle(mesh, M.PDE_EULER, M.FLUX_ROE, bc_prim=prim).rhs(ud.cpu().numpy())
        assert np.abs(r).max() < 1e-9
    assert its[_lib.PC_BLOCK_SGS] < its[_lib.PC_BLOCK_JACOBI]
    ctx.close()


def test_3d_unsupported_paths_are_refused(dev):
    from dpgsolver_amd import _lib

    mesh, u0, prim = _box()
    ctx = _ctx(mesh, M.FLUX_ROE, bc_prim=prim)
    ud = torch.from_numpy(u0).to(dev)
    with pytest.raises(_lib.DgxError, match="UNSUPPORTED"):
        ctx.solve_implicit(ud.data_ptr(), precond=_lib.PC_BLOCK_JACOBI, jvp_fp32=True)
    ctx.close()
    mesh3, u3 = _curved(3, 2, 3)    # nb = 320: more than the batched LU and inverse take
    ctx = _ctx(mesh3, M.FLUX_ROE)
    ud = torch.from_numpy(u3).to(dev)
    for pc in (_lib.PC_BLOCK_JACOBI, _lib.PC_BLOCK_SGS, _lib.PC_BLOCK_SGS32):
        with pytest.raises(_lib.DgxError, match="UNSUPPORTED"):
            ctx.solve_implicit(ud.data_ptr(), precond=pc)
    ctx.close()
