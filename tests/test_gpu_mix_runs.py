"""The mixed faces' single launch (k_mix_faces) where some face-point counts are absent and where a run of faces takes
several workgroups with the last part full: orders drawn from a subset, FP64 against oracle/mixed_oracle.py at the mixed
residual's own bound (1e-12 of the larger of max |R| and max |volume term|), Euler and Navier-Stokes.
"""
import numpy as np
import pytest

import mixed_oracle as MO
from dpgsolver_amd import mesh as M

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

MU, PR = 0.02, 0.72


@pytest.mark.parametrize("orders,n", [((1,), (9, 8)), ((1, 5), (8, 5)), ((2, 4), (7, 6)), ((3, 5), (6, 5)), ((1, 2, 3), (11, 7))])
def test_subsets_of_face_point_counts_match_oracle(orders, n):
    from dpgsolver_amd import _lib

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(sum(orders))
    split = rng.random(n[0] * n[1]) < 0.4
    p = rng.choice(orders, int(n[0] * n[1] + split.sum())).astype(np.int32)
    mesh = M.structured_mixed_mesh(n, split, p)
    u = M.mixed_state(mesh, lambda x: M.prim_to_cons(M.smooth_state_3d(x), 2))
    for flux in (M.FLUX_ROE, M.FLUX_LF):
        for ns in (False, True):
            orc = MO.MixedOracle(mesh, flux, viscous=(MU, PR)) if ns else MO.MixedOracle(mesh, flux)
            ref = orc.rhs_ns(u) if ns else orc.rhs(u)
            visc = dict(mu=MU, Pr=PR) if ns else {}
            ctx = _lib.Context(2, max(orders), M.PDE_NAVIER_STOKES if ns else M.PDE_EULER, flux, **visc)
            ctx.set_stream(torch.cuda.current_stream().cuda_stream)
            ctx.upload_mesh_mixed(mesh)
            ud = torch.from_numpy(u).cuda()
            rd = torch.full_like(ud, float("nan"))
            ctx.compute_rhs(ud.data_ptr(), rd.data_ptr())
            torch.cuda.synchronize()
            scale = max(np.abs(orc.rhs(u, "volume")).max(), np.abs(ref).max())
            err = np.abs(rd.cpu().numpy() - ref).max() / scale
            print(f"orders {orders} flux={flux} ns={ns}: {err:.2e}", flush=True)
            assert err < 1e-12
            ctx.close()
