"""Element blocks of the Newton matrix and their batched inverse at the edges of the kernels' tilings.

* dgx_block_inverse against numpy: block sizes around the tile (8 x 8 and 16 x 16 lanes) and wavefront boundaries,
  matrices that need row exchanges.  Tolerance: Gauss-Jordan's forward error is bounded by a small multiple of
  nb eps cond(A) |A^-1|; 32 nb eps cond(A) is asked.
* The diagonal and face blocks of every QUAD order and equation, applied to a vector, against the exact J v.
"""
import numpy as np
import pytest

from dpgsolver_amd import mesh as M

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


@pytest.mark.parametrize("nb", [1, 7, 8, 9, 16, 36, 63, 64, 65, 80, 81, 100, 135, 142])
def test_block_inverse_matches_numpy(dev, nb):
    from dpgsolver_amd import _lib

    E = 5
    rng = np.random.default_rng(nb)
    A = rng.standard_normal((E, nb, nb))
    A[1, np.arange(nb), np.arange(nb)] = 0.0 if nb > 1 else 1.0    # every pivot off the diagonal
    A[2] = A[2][::-1] * 1e-8                                       # small entries
    A[3] += 1e3 * np.eye(nb)[rng.permutation(nb)]                  # dominant permutation
    ctx = _lib.Context(2, 1, M.PDE_EULER, M.FLUX_LF)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    b = torch.from_numpy(A.copy()).to(dev)
    ctx.block_inverse(b.data_ptr(), E, nb)
    torch.cuda.synchronize()
    got = b.cpu().numpy().transpose(0, 2, 1)
    for e in range(E):
        ref = np.linalg.inv(A[e])
        tol = 32 * nb * EPS * np.linalg.cond(A[e]) * np.abs(ref).max()
        assert np.abs(got[e] - ref).max() <= tol, e
    ctx.close()


@pytest.mark.parametrize("pde,flux", [("euler", M.FLUX_LF), ("euler", M.FLUX_ROE), ("advection", M.FLUX_UPWIND)])
@pytest.mark.parametrize("p", [1, 2, 3, 4])
def test_quad_blocks_times_vector_equal_the_exact_product(dev, p, pde, flux):
    """5 x 3 QUADs with turned local frames (both face orientations): sum of the blocks times v = J v to 1e-12."""
    from dpgsolver_amd import _lib

    curve = lambda x: x + 0.04 * np.sin(2 * np.pi * x[..., ::-1])      # noqa: E731
    m = M.structured_tp_mesh(2, p, (5, 3), (0, 0), (1, 1), (True, True), curve=curve,
                             rotate=np.random.default_rng(p).integers(0, 4, 15))
    if pde == "euler":
        ctx = _lib.Context(2, p, M.PDE_EULER, flux)
        u = M.pack_state(M.prim_to_cons(M.smooth_state_3d(M.nodes_xyz(m)), 2))
    else:
        ctx = _lib.Context(2, p, M.PDE_ADVECTION, flux, b_adv=(1.0, 0.5, 0.0))
        u = np.random.default_rng(3).standard_normal(m.E * m.Np)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    ctx.upload_mesh(m.xyz, m.faces)
    nb = ctx.Np * ctx.nv
    v = np.random.default_rng(8).standard_normal(u.size)
    ud, vd = torch.from_numpy(u).to(dev), torch.from_numpy(v).to(dev)
    jv = torch.empty_like(ud)
    db = torch.zeros((m.E, nb, nb), dtype=torch.float64, device=dev)
    fb = torch.zeros((m.E, 4, nb, nb), dtype=torch.float64, device=dev)
    ctx.assemble_diag_blocks(ud.data_ptr(), None, db.data_ptr())
    ctx.assemble_face_blocks(ud.data_ptr(), fb.data_ptr())
    ctx.jacobian_vector(ud.data_ptr(), vd.data_ptr(), jv.data_ptr())
    torch.cuda.synchronize()
    V = v.reshape(m.E, nb)
    y = np.einsum("eij,ej->ei", db.cpu().numpy(), V)
    F = fb.cpu().numpy()
    for eL, fL, eR, fR, _, _ in m.faces:
        y[eL] += F[eL, fL] @ V[eR]
        y[eR] += F[eR, fR] @ V[eL]
    ref = jv.cpu().numpy()
    assert np.abs(y.ravel() - ref).max() <= 1e-12 * np.abs(ref).max()
    ctx.close()
