"""Graphs of variable-order and TRI / QUAD residuals above the sizes from which their phases run on the side streams: every
replay equals the eager call on one stream bit for bit, with eager work and synchronisations between the replays and a
changed state for each, also where the caller captures the call into a graph of its own."""
import pytest

from dpgsolver_amd import mesh as M

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CASES = [("hp", "ns", (20, 16)), ("hp", "euler", (150, 140)), ("tri", "ns", (16, 15)), ("tri", "euler", (150, 110))]


def _context(kind, pde, n):
    from dpgsolver_amd import _lib

    mesh = M.config4_hp_mesh(*n) if kind == "hp" else M.config4_mixed_mesh(*n)
    u = M.config4_hp_state(mesh) if kind == "hp" else M.config4_mixed_state(mesh)
    if pde == "ns":
        ctx = _lib.Context(2, 5, M.PDE_NAVIER_STOKES, M.FLUX_ROE, mu=0.02, Pr=0.72)
    else:
        ctx = _lib.Context(2, 5, M.PDE_EULER, M.FLUX_ROE)
    (ctx.upload_mesh_hp if kind == "hp" else ctx.upload_mesh_mixed)(mesh)
    return ctx, torch.from_numpy(u).to("cuda:0")


@pytest.mark.parametrize("kind,pde,n", CASES, ids=["-".join(c[:2]) for c in CASES])
def test_replays_equal_the_eager_call(kind, pde, n):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ctx, u64 = _context(kind, pde, n)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    u32 = u64.float()
    calls = [(ctx.compute_rhs, 0, u64, torch.float64), (ctx.compute_rhs_f32, 1, u32, torch.float32)]
    if kind == "hp":
        calls.append((ctx.compute_rhs_mixed, 2, u64, torch.float32))
    runs = [(fn, ui, torch.empty(ui.shape, dtype=dt, device="cuda:0"), torch.empty(ui.shape, dtype=dt, device="cuda:0"))
            for fn, _, ui, dt in calls]
    graphs = [ctx.graph_rhs(k, ui.data_ptr(), out.data_ptr()) for (_, k, ui, _), (_, _, _, out) in zip(calls, runs)]
    for rep in range(4):
        for g, (fn, ui, ref, out) in zip(graphs, runs):
            out.fill_(float("nan"))
            g.launch(2)
            g.sync()
            fn(ui.data_ptr(), ref.data_ptr())
            torch.cuda.synchronize()
            assert torch.equal(out, ref), rep
        u64.mul_(1.0 + 1e-3)
        u32.copy_(u64)
    for g in graphs:
        g.close()
    ctx.close()


def test_capture_by_the_caller():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ctx, u = _context("hp", "ns", (20, 16))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    ctx.set_stream(s.cuda_stream)
    ref, out = torch.empty_like(u), torch.empty_like(u)
    ctx.compute_rhs(u.data_ptr(), ref.data_ptr())
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        ctx.compute_rhs(u.data_ptr(), out.data_ptr())
    for rep in range(3):
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), rep
        u.mul_(1.0 + 1e-3)
        torch.cuda.synchronize()
        ctx.compute_rhs(u.data_ptr(), ref.data_ptr())
        s.synchronize()
    ctx.close()
