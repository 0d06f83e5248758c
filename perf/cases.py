"""The calls that a user of this framework makes, as measurable cases.

A case is a dict of plain values.  ``prepare`` builds what a program has in hand before the call (mesh uploaded, state
on the GPU, recorded graph), ``run`` is one pass through the public entry points, ``work`` what such a pass cannot do
without, and ``exact`` the same outputs in plain float64 torch.  Kinds of case:

* ``residual``         R(u) on a uniform-order QUAD / HEX mesh (Euler or Navier-Stokes; FP64, FP32 or mixed);
* ``mixed_residual``   R(u) on a mixed TRI / QUAD mesh with an order per element;
* ``time_steps``       SSP-RK3 steps (advection, or Euler with the positivity limiter);
* ``newton_operator``  (dR/du - M/dt) v, the product inside every Krylov iteration;
* ``block_inverse``    assembly and inversion of the element diagonal blocks, once per Newton step;
* ``steady``           a whole pseudo-time Newton-GMRES solve to max|R| < 1e-11 (a decade below the usual 1e-10, so
                       that the states of two solvers that round differently agree far better than they are used);
* ``train``            one epoch of the learned preconditioner's training.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from dpgsolver_amd import _lib
from dpgsolver_amd import mesh as M

DEV = "cuda:0"
GAMMA, GM1, EPS_PHYS = 1.4, 0.4, 1e-13
NS_MU, NS_PR = 0.28 / 100.0, 0.72            # Re 100 on the velocity amplitude 0.28 and unit length
FLUX = {"lf": M.FLUX_LF, "roe": M.FLUX_ROE}
PRECOND = {"sgs": _lib.PC_BLOCK_SGS, "sgs32": _lib.PC_BLOCK_SGS32}


# ----------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest job: 100 steps of linear advection on 16 x 16 QUADs, every kernel a few microseconds long
        {"name": "advection_16_rk3", "kind": "time_steps", "pde": "advection", "p": 2, "n0": 16, "n1": 16, "steps": 100,
         "api": "graph"},
        # one FP64 residual call of the 128 x 128 isentropic vortex: a user's own time integrator or monitor
        {"name": "vortex_128_residual", "kind": "residual", "pde": "euler", "d": 2, "p": 3, "n0": 128, "n1": 128, "n2": 1,
         "flux": "roe", "dtype": "f64"},
        # the explicit time loop on the same vortex: SSP-RK3 with the positivity limiter after every stage
        {"name": "vortex_128_rk3", "kind": "time_steps", "pde": "euler", "p": 3, "n0": 128, "n1": 128, "steps": 10,
         "api": "graph"},
        # the headline: 3-D Euler on 64^3 curved HEXes, the inner residual (FP64 state, FP32 contractions)
        {"name": "hex_64_mixed", "kind": "residual", "pde": "euler", "d": 3, "p": 4, "n0": 64, "n1": 64, "n2": 64,
         "flux": "lf", "dtype": "mixed"},
        # the outer FP64 residual of the same flow on a grid of ordinary size
        {"name": "hex_32_f64", "kind": "residual", "pde": "euler", "d": 3, "p": 4, "n0": 32, "n1": 32, "n2": 32,
         "flux": "lf", "dtype": "f64"},
        # an odd-sized 3-D grid of lower order in plain FP32, Roe flux
        {"name": "hex_odd_f32", "kind": "residual", "pde": "euler", "d": 3, "p": 3, "n0": 37, "n1": 23, "n2": 29,
         "flux": "roe", "dtype": "f32"},
        # Navier-Stokes (BR2) on the 448 x 448 QUAD grid, FP64
        {"name": "ns_448_f64", "kind": "residual", "pde": "ns", "d": 2, "p": 3, "n0": 448, "n1": 448, "n2": 1,
         "flux": "roe", "dtype": "f64"},
        # Navier-Stokes on the 200 k element TRI / QUAD mesh with orders 1..5 drawn per element, FP64
        {"name": "ns_tri_quad_f64", "kind": "mixed_residual", "pde": "ns", "n0": 500, "n1": 300, "dtype": "f64"},
        # one operator product of the 64 x 64 channel's Newton system, as a Krylov method calls it thousands of times
        {"name": "channel_64_operator", "kind": "newton_operator", "p": 3, "n0": 64, "n1": 64},
        # the block-Jacobi set-up of the same system: 4096 diagonal blocks of 64 x 64, assembled and inverted
        {"name": "channel_64_blocks", "kind": "block_inverse", "p": 3, "n0": 64, "n1": 64},
        # the whole steady solve of the channel with the block SGS preconditioner: time to a converged FP64 residual
        {"name": "channel_64_steady", "kind": "steady", "p": 3, "n0": 64, "n1": 64, "precond": "sgs"},
        # an epoch of the learned preconditioner's training: mini-batches of 256 captured blocks
        {"name": "train_kron8", "kind": "train", "p": 3, "structure": "kron", "rank": 8, "hidden": 256, "samples": 8192,
         "batch": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["residual2", "residual2", "residual3", "residual3", "ns", "mixed_residual", "time_steps",
                       "time_steps", "newton_operator", "block_inverse", "steady", "train"])
    if kind == "residual2":
        return {"kind": "residual", "pde": "euler", "d": 2, "p": rng.randint(1, 5), "n0": _log_int(rng, 8, 400),
                "n1": _log_int(rng, 8, 400), "n2": 1, "flux": rng.choice(["lf", "roe"]),
                "dtype": rng.choice(["f64", "mixed", "f32"])}
    if kind == "residual3":
        return {"kind": "residual", "pde": "euler", "d": 3, "p": rng.randint(1, 4), "n0": _log_int(rng, 3, 48),
                "n1": _log_int(rng, 3, 48), "n2": _log_int(rng, 3, 48), "flux": rng.choice(["lf", "roe"]),
                "dtype": rng.choice(["f64", "mixed", "f32"])}
    if kind == "ns":
        return {"kind": "residual", "pde": "ns", "d": 2, "p": rng.randint(1, 5), "n0": _log_int(rng, 8, 400),
                "n1": _log_int(rng, 8, 400), "n2": 1, "flux": rng.choice(["lf", "roe"]),
                "dtype": rng.choice(["f64", "f64", "mixed"])}
    if kind == "mixed_residual":
        return {"kind": "mixed_residual", "pde": rng.choice(["euler", "ns"]), "n0": _log_int(rng, 8, 300),
                "n1": _log_int(rng, 8, 200), "dtype": "f64"}
    if kind == "time_steps":
        euler = rng.random() < 0.6
        return {"kind": "time_steps", "pde": "euler" if euler else "advection", "p": rng.randint(1, 5),
                "n0": _log_int(rng, 16, 200), "n1": _log_int(rng, 16, 200), "steps": rng.randint(1, 20),
                "api": rng.choice(["graph", "call"])}
    if kind == "newton_operator":
        return {"kind": kind, "p": rng.randint(1, 4), "n0": _log_int(rng, 8, 160), "n1": _log_int(rng, 8, 160)}
    if kind == "block_inverse":
        return {"kind": kind, "p": rng.randint(1, 4), "n0": _log_int(rng, 8, 64), "n1": _log_int(rng, 8, 64)}
    if kind == "steady":
        return {"kind": kind, "p": rng.randint(2, 3), "n0": _log_int(rng, 16, 48), "n1": _log_int(rng, 16, 48),
                "precond": rng.choice(["sgs", "sgs32"])}
    structure = rng.choice(["kron", "lowrank"])
    batch = rng.choice([64, 128, 200, 256, 512])
    return {"kind": "train", "p": rng.randint(2, 3), "structure": structure,
            "rank": rng.choice([4, 8]) if structure == "kron" else 8, "hidden": rng.choice([64, 128, 256]),
            "samples": batch * rng.randint(2, 4096 // batch) + rng.randint(0, batch - 1), "batch": batch}


# --------------------------------------------------------------------------------------------------- the inputs
@functools.lru_cache(maxsize=3)
def _tp_mesh(d, p, n, curved, lo, hi):
    """Periodic structured mesh; curved: the sinusoidal 3-D map, or its 2-D counterpart."""
    curve = None
    if curved and d == 3:
        curve = M.curve3d(0.05)
    return M.structured_tp_mesh(d, p, n, (lo,) * d, (hi,) * d, (True,) * d, curve=curve)


@functools.lru_cache(maxsize=2)
def _channel(n0, n1, p):
    return M.channel_mesh(n0, n1, p)


@functools.lru_cache(maxsize=2)
def _mixed_mesh(n0, n1):
    return M.config4_mixed_mesh(n0, n1)


def _phases(seed, n):
    return np.random.RandomState(seed & 0x7FFFFFFF).uniform(0.0, 2.0 * math.pi, n)


def _smooth(xyz, seed):
    """Conserved smooth state (E, d + 2, Np) at nodes xyz (E, d, Np): density and pressure within 10 % of 1, velocity
    components up to 0.28, every variable a product of sines of unit period with seeded phases."""
    d = xyz.shape[1]
    ph = _phases(seed, 15).reshape(5, 3)
    s = []
    for k in range(5):
        v = None
        for c in range(d):
            t = torch.sin(2.0 * math.pi * xyz[:, c] + float(ph[k, c]))
            v = t if v is None else v * t
        s.append(v)
    rho, p = 1.0 + 0.1 * s[0], 1.0 + 0.1 * s[4]
    vel = [0.28 * s[1 + c] for c in range(d)]
    ke = sum(v * v for v in vel)
    return torch.stack([rho] + [rho * v for v in vel] + [p / GM1 + 0.5 * rho * ke], 1)


def _vortex(xyz, seed):
    """Isentropic vortex of strength 5 on a Mach 0.5 stream plus a seeded uniform 1e-3 perturbation."""
    dx, dy = xyz[:, 0] - 5.0, xyz[:, 1] - 5.0
    r2 = dx * dx + dy * dy
    rho = (1.0 - GM1 * 25.0 / (8.0 * GAMMA * math.pi ** 2) * torch.exp(1.0 - r2)) ** (1.0 / GM1)
    p = rho ** GAMMA
    f = 5.0 / (2.0 * math.pi) * torch.exp(0.5 * (1.0 - r2))
    u, v = 0.5 * math.sqrt(GAMMA) - f * dy, f * dx
    cons = torch.stack([rho, rho * u, rho * v, p / GM1 + 0.5 * rho * (u * u + v * v)], 1)
    g = torch.Generator(device=xyz.device).manual_seed(seed)
    return cons + 1e-3 * (2.0 * torch.rand(cons.shape, generator=g, device=xyz.device, dtype=torch.float64) - 1.0)


def _channel_state(mesh, seed, amp=0.02):
    """The free stream with a smooth seeded variation of relative size amp: a state on the way to the steady one."""
    xyz = torch.from_numpy(mesh.xyz).to(DEV)
    ph = _phases(seed, 8)
    w = torch.stack([torch.sin(2.1 * xyz[:, 0] + float(ph[2 * k])) * torch.sin(4.0 * xyz[:, 1] + float(ph[2 * k + 1]))
                     for k in range(4)], 1)
    prim = M.freestream_prim(2)
    rho = prim[0] * (1.0 + amp * w[:, 0])
    u, v, p = prim[1] * (1.0 + amp * w[:, 1]), amp * w[:, 2], prim[3] * (1.0 + amp * w[:, 3])
    return torch.stack([rho, rho * u, rho * v, p / GM1 + 0.5 * rho * (u * u + v * v)], 1).reshape(-1)


def _context(*args, **kw):
    ctx = _lib.Context(*args, **kw)
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    return ctx


def _uniform_mesh(case):
    if case["kind"] == "residual":
        d = case["d"]
        n = (case["n0"], case["n1"], case["n2"])[:d]
        hi = 10.0 if case["pde"] == "euler" and d == 2 else 1.0
        return _tp_mesh(d, case["p"], n, d == 3, 0.0, hi)
    if case["kind"] == "time_steps":
        if case["pde"] == "advection":
            return _tp_mesh(2, case["p"], (case["n0"], case["n1"]), False, -1.0, 1.0)
        return _tp_mesh(2, case["p"], (case["n0"], case["n1"]), False, 0.0, 10.0)
    return _channel(case["n0"], case["n1"], case["p"])


def _uniform_state(case, mesh, seed):
    if case["kind"] == "residual":
        xyz = torch.from_numpy(mesh.xyz).to(DEV)
        if case["d"] == 2 and case["pde"] == "euler":
            return _vortex(xyz, seed).reshape(-1)
        return _smooth(xyz, seed).reshape(-1)
    if case["kind"] == "time_steps":
        xyz = torch.from_numpy(mesh.xyz).to(DEV)
        if case["pde"] == "euler":
            return _vortex(xyz, seed).reshape(-1)
        ph = _phases(seed, 2)
        return (torch.sin(math.pi * xyz[:, 0] + float(ph[0])) * torch.sin(math.pi * xyz[:, 1] + float(ph[1]))).reshape(-1)
    return _channel_state(mesh, seed, 0.002 if case["kind"] == "steady" else 0.02)


def _time_step(case):
    h = (2.0 if case["pde"] == "advection" else 10.0) / max(case["n0"], case["n1"])
    return 0.2 * h / ((2 * case["p"] + 1) * (1.0 if case["pde"] == "advection" else 2.0))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mixed_residual":
        mesh = _mixed_mesh(case["n0"], case["n1"])
        if case["pde"] == "ns":
            ctx = _context(2, 5, M.PDE_NAVIER_STOKES, M.FLUX_ROE, mu=NS_MU, Pr=NS_PR)
        else:
            ctx = _context(2, 5, M.PDE_EULER, M.FLUX_ROE)
        ctx.upload_mesh_mixed(mesh)
        u = torch.from_numpy(M.config4_mixed_state(mesh, seed)).to(DEV)
        return {"case": case, "ctx": ctx, "u": u, "r": torch.empty_like(u)}
    if kind == "train":
        return _prepare_training(case, seed)
    mesh = _uniform_mesh(case)
    u = _uniform_state(case, mesh, seed)
    if kind == "residual":
        if case["pde"] == "ns":
            ctx = _context(case["d"], case["p"], M.PDE_NAVIER_STOKES, FLUX[case["flux"]], mu=NS_MU, Pr=NS_PR)
        else:
            ctx = _context(case["d"], case["p"], M.PDE_EULER, FLUX[case["flux"]])
        ctx.upload_mesh(mesh.xyz, mesh.faces)
        if case["dtype"] == "f32":
            u = u.float()
        r = torch.empty(u.numel(), dtype=torch.float64 if case["dtype"] == "f64" else torch.float32, device=DEV)
        return {"case": case, "ctx": ctx, "u": u, "r": r}
    if kind == "time_steps":
        euler = case["pde"] == "euler"
        if euler:
            ctx = _context(2, case["p"], M.PDE_EULER, M.FLUX_ROE)
        else:
            ctx = _context(2, case["p"], M.PDE_ADVECTION, M.FLUX_UPWIND, b_adv=(1.0, 0.5, 0.0))
        ctx.upload_mesh(mesh.xyz, mesh.faces)
        st = {"case": case, "ctx": ctx, "u0": u, "u": u.clone(), "dt": _time_step(case), "euler": euler}
        if case["api"] == "graph":
            st["graph"] = ctx.graph_rk3(st["u"].data_ptr(), st["dt"], positivity=euler)
        return st
    prim = M.freestream_prim(2)
    ctx = _context(2, case["p"], M.PDE_EULER, M.FLUX_ROE, bc_prim=prim)
    ctx.upload_mesh(mesh.xyz, mesh.faces)
    st = {"case": case, "ctx": ctx, "u": u, "E": mesh.E, "nb": 4 * mesh.Np}
    if kind == "steady":
        st["u0"], st["u"] = u, u.clone()
        return st
    st["inv_dt"] = torch.empty(mesh.E, dtype=torch.float64, device=DEV)
    ctx.cfl_dt(u.data_ptr(), 30.0, st["inv_dt"].data_ptr())
    if kind == "newton_operator":
        g = torch.Generator(device=DEV).manual_seed(seed + 1)
        st["v"] = torch.randn(u.numel(), generator=g, device=DEV, dtype=torch.float64)
        st["out"] = torch.empty_like(u)
    else:
        st["blocks"] = torch.empty((mesh.E, st["nb"], st["nb"]), dtype=torch.float64, device=DEV)
    return st


def _prepare_training(case, seed):
    """Blocks, features and scales of the solver's own systems: the channel of 64 x 64 elements at seeded states and
    CFL numbers along the ramp."""
    mesh = _channel(64, 64, case["p"])
    nb, n = 4 * mesh.Np, case["samples"]
    ctx = _context(2, case["p"], M.PDE_EULER, M.FLUX_ROE, bc_prim=M.freestream_prim(2))
    ctx.upload_mesh(mesh.xyz, mesh.faces)
    mlp = _lib.MLP(nb, mesh.Np, hidden=case["hidden"], rank=case["rank"],
                   kind=_lib.MLP_KRON if case["structure"] == "kron" else _lib.MLP_LOWRANK)
    sets = -(-n // mesh.E)
    blocks = torch.empty((sets, mesh.E, nb, nb), dtype=torch.float64, device=DEV)
    feat = torch.empty((sets, mesh.E, mlp.nf), dtype=torch.float32, device=DEV)
    sigma = torch.empty((sets, mesh.E), dtype=torch.float32, device=DEV)
    inv_dt = torch.empty(mesh.E, dtype=torch.float64, device=DEV)
    for k in range(sets):
        u = _channel_state(mesh, seed + 1000 * k)
        ctx.cfl_dt(u.data_ptr(), (3.0, 60.0)[k % 2], inv_dt.data_ptr())
        ctx.assemble_diag_blocks(u.data_ptr(), inv_dt.data_ptr(), blocks[k].data_ptr())
        mlp.features(ctx, u.data_ptr(), inv_dt.data_ptr(), feat[k].data_ptr(), sigma[k].data_ptr())
        torch.cuda.synchronize()
    ctx.close()
    return {"case": case, "mlp": mlp, "w0": mlp.get_params(), "blocks": blocks.reshape(-1, nb, nb)[:n].contiguous(),
            "feat": feat.reshape(-1, mlp.nf)[:n].contiguous(), "sigma": sigma.reshape(-1)[:n].contiguous()}


# ------------------------------------------------------------------------------------------------------ one pass
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind in ("residual", "mixed_residual"):
        fn = {"f64": st["ctx"].compute_rhs, "f32": st["ctx"].compute_rhs_f32,
              "mixed": st["ctx"].compute_rhs_mixed}[case["dtype"]]
        fn(st["u"].data_ptr(), st["r"].data_ptr())
        return st["r"]
    if kind == "time_steps":
        st["u"].copy_(st["u0"])
        if case["api"] == "graph":
            st["graph"].launch(case["steps"])
            return st["u"]
        for _ in range(case["steps"]):
            mx = st["ctx"].ssp_rk3_step(st["u"].data_ptr(), st["dt"], positivity=st["euler"])
        return st["u"], mx
    if kind == "newton_operator":
        st["ctx"].newton_operator(st["u"].data_ptr(), st["inv_dt"].data_ptr(), st["v"].data_ptr(), st["out"].data_ptr())
        return st["out"]
    if kind == "block_inverse":
        ctx = st["ctx"]
        ctx.assemble_diag_blocks(st["u"].data_ptr(), st["inv_dt"].data_ptr(), st["blocks"].data_ptr())
        ctx.block_inverse(st["blocks"].data_ptr(), st["E"], st["nb"])
        return st["blocks"]
    if kind == "steady":
        st["u"].copy_(st["u0"])
        st["ctx"].solve_implicit(st["u"].data_ptr(), cfl_initial=1.0, cfl_max=300.0, exit_tol=1e-11, max_newton=100,
                                 gmres_restart=60, gmres_rtol=1e-4, gmres_max_iter=1000,
                                 precond=PRECOND[case["precond"]])
        return st["u"]
    st["mlp"].train(st["feat"].data_ptr(), st["sigma"].data_ptr(), st["blocks"].data_ptr(), case["samples"],
                    epochs=1, batch=case["batch"], lr=1e-4)
    return st["mlp"].get_params()


# ------------------------------------------------------------------------------------------- what a pass needs
def _residual_work(d, p, nv, E, sin, sout, sgeo, viscous=False, dual=1):
    """Bytes: state in, residual out, metrics (and det J where the gradient needs it), n J_f of the owned faces.
    Flops: three sum-factorised sweeps per direction, the trace interpolations, pointwise fluxes."""
    N, Np, NF = p + 1, (p + 1) ** d, (p + 1) ** (d - 1)
    per = nv * Np * (sin + sout) + Np * (d * d + (1 if viscous else 0)) * sgeo + d * NF * d * sgeo
    flops = nv * Np * 3 * d * 2 * N + 2 * d * (d - 1) * nv * NF * 2 * N + Np * 20 * d + d * NF * 130
    if viscous:
        flops += nv * Np * d * 2 * N + Np * 90 + 2 * d * d * nv * NF * 2 * N + d * NF * 120
    return {"bytes": float(E * per), "flops": float(dual * E * flops)}


def work(case):
    kind, p = case["kind"], case.get("p")
    if kind == "residual":
        E = case["n0"] * case["n1"] * case["n2"]
        sin = 4 if case["dtype"] == "f32" else 8
        sout = 8 if case["dtype"] == "f64" else 4
        return _residual_work(case["d"], p, case["d"] + 2, E, sin, sout, sout, case["pde"] == "ns")
    if kind == "mixed_residual":
        # a third of the cells is two TRIs; orders 1..5 equally often
        cells, tot = case["n0"] * case["n1"], {"bytes": 0.0, "flops": 0.0}
        for q in range(1, 6):
            w = _residual_work(2, q, 4, 1, 8, 8, 8, case["pde"] == "ns")
            tri = ((q + 1) * (q + 2) / 2.0) / (q + 1) ** 2
            for k in tot:
                tot[k] += w[k] * cells / 5.0 * (2.0 / 3.0 + 2.0 / 3.0 * tri)
        return tot
    if kind == "time_steps":
        E, nv = case["n0"] * case["n1"], 4 if case["pde"] == "euler" else 1
        w = _residual_work(2, p, nv, E, 8, 8, 8, True)      # det J: the mass inverse
        stage = 8.0 * E * nv * (p + 1) ** 2                 # the step's initial state, read once a stage
        return {"bytes": 3.0 * case["steps"] * (w["bytes"] + stage), "flops": 3.0 * case["steps"] * w["flops"]}
    E = case.get("n0", 64) * case.get("n1", 64)
    Np = (p + 1) ** 2
    nb = 4 * Np
    if kind == "newton_operator":
        w = _residual_work(2, p, 4, E, 16, 8, 8, False, dual=3)
        return {"bytes": w["bytes"] + 8.0 * E * (Np + 1), "flops": w["flops"]}
    if kind == "block_inverse":
        w = _residual_work(2, p, 4, E, 8, 0, 8)
        return {"bytes": w["bytes"] + 8.0 * E * nb * nb, "flops": E * (2.0 * nb ** 3 + 2.0 * 16 * 4 * Np * Np * (p + 1))}
    if kind == "steady":
        # about 18 Newton steps and, on n elements across, 90 n GMRES iterations; per step the blocks once, per
        # iteration the stored blocks read once, the operator and one basis pass
        its = max(case["n0"], case["n1"]) * 90.0
        nfv = 4 * (p + 1)
        stored = E * (nb * nb + 4 * nfv * nfv)
        size = 4.0 if case["precond"] == "sgs32" else 8.0
        op = _residual_work(2, p, 4, E, 16, 8, 8, False, dual=3)
        return {"bytes": 18 * 8.0 * stored + its * (size * stored + op["bytes"] + 30 * 4.0 * E * nb),
                "flops": 18 * E * 2.0 * nb ** 3 + its * (2.0 * stored + op["flops"] + 4 * 30 * 2.0 * E * nb)}
    nf, h, n = -(-(nb + Np + 1) // 16) * 16, case["hidden"], case["samples"]
    no = case["rank"] * (16 + Np * Np) if case["structure"] == "kron" else nb + 2 * nb * case["rank"]
    gemm = 2.0 * (nf * h + h * h + h * no)
    nparam = nf * h + h * h + h * no
    steps = -(-n // case["batch"])
    # training pass over the blocks, then the loss of the whole set
    return {"bytes": n * (2.0 * 8 * nb * nb + 2 * 4 * nf) + steps * 28.0 * nparam,
            "flops": n * (3 * gemm + gemm + 6.0 * nb ** 3)}


# --------------------------------------------------------------------------------- the same in float64 torch
def _legendre_nodes(n):
    x, w = np.polynomial.legendre.leggauss(n)
    return 0.5 * (x - x[::-1]), 0.5 * (w + w[::-1])


def _lobatto_nodes(n):
    c = np.polynomial.legendre.Legendre.basis(n - 1)
    x = np.concatenate([[-1.0], np.sort(c.deriv().roots().real), [1.0]])
    for _ in range(4):
        x[1:-1] -= c.deriv()(x[1:-1]) / c.deriv(2)(x[1:-1])
    return 0.5 * (x - x[::-1])


def _lagrange(xin, xout):
    """Values and derivatives of the Lagrange basis on xin at xout: (out, in) matrices."""
    n = len(xin)
    V, D = np.zeros((len(xout), n)), np.zeros((len(xout), n))
    for j in range(n):
        others = np.delete(xin, j)
        poly = np.polynomial.Polynomial.fromroots(others) / np.prod(xin[j] - others) if n > 1 else np.polynomial.Polynomial([1.0])
        V[:, j], D[:, j] = poly(xout), poly.deriv()(xout)
    return V, D


class _Plain:
    """R(u) of the DG weak form on a uniform-order tensor-product mesh, dense one-dimensional operators in float64."""

    def __init__(self, mesh, pde, flux="roe", bc_prim=None, b=(1.0, 0.5), mu=NS_MU, Pr=NS_PR):
        self.d, self.N, self.E = mesh.d, mesh.p + 1, mesh.xyz.shape[0]
        self.pde, self.flux, self.mu, self.Pr, self.b = pde, flux, mu, Pr, b
        self.nv = 1 if pde == "advection" else self.d + 2
        self.prim = None if bc_prim is None else [float(v) for v in bc_prim]
        t = lambda a: torch.tensor(a, dtype=torch.float64, device=DEV)       # noqa: E731
        gl, w = _legendre_nodes(self.N)
        gll = _lobatto_nodes(self.N)
        V, D = _lagrange(gll, gl)
        ends, _ = _lagrange(gl, np.array([-1.0, 1.0]))
        self.I, self.DI, self.w, self.ends = t(V), t(D), t(w), t(ends)
        self.Dgll = t(_lagrange(gll, gll)[1])
        bern = np.stack([math.comb(self.N - 1, k) * (0.5 * (1 + gll)) ** k * (0.5 * (1 - gll)) ** (self.N - 1 - k)
                         for k in range(self.N)], 1)
        self.bern, self.bern_inv = t(bern), t(np.linalg.inv(bern))
        wd = self.w
        for _ in range(self.d - 1):
            wd = wd.unsqueeze(-1) * self.w
        self.wvol = wd                                                        # (N,) * d
        self.wface = self.w if self.d == 2 else self.w[:, None] * self.w
        faces = torch.from_numpy(np.asarray(mesh.faces, dtype=np.int64)).to(DEV)
        self.eL, self.fL, self.eR, self.fR, self.ord, self.bc = (faces[:, k] for k in range(6))
        if bool((self.ord[self.eR >= 0] != 0).any()):
            raise ValueError("aligned faces only")
        self._geometry(torch.from_numpy(mesh.xyz).to(DEV))

    # arrays hold one axis per direction after the variable axis, the last axis the first direction
    def _ax(self, k):
        return -1 - k

    def _apply(self, A, u, k):
        return torch.movedim(torch.tensordot(u, A, dims=([u.dim() - 1 - k], [1])), -1, self._ax(k))

    def _all(self, A, u, dirs=None):
        for k in range(self.d) if dirs is None else dirs:
            u = self._apply(A, u, k)
        return u

    def _geometry(self, xyz):
        d, N = self.d, self.N
        X = xyz.reshape((self.E, d) + (N,) * d)
        J = torch.stack([self._apply(self.Dgll, X, k) for k in range(d)], 2)  # (E, i, k, ...)
        if d == 2:
            met = torch.stack([torch.stack([J[:, 1, 1], -J[:, 1, 0]], 1), torch.stack([-J[:, 0, 1], J[:, 0, 0]], 1)], 1)
        else:
            # conservative symmetric curl form of the cofactors, met[:, i, j] = J dxi_j / dx_i
            rows = []
            for a, b in ((1, 2), (2, 0), (0, 1)):
                cols = []
                for c in range(3):
                    k1, k2 = (c + 1) % 3, (c + 2) % 3
                    curl = lambda p, q: (self._apply(self.Dgll, X[:, p] * J[:, q, k2], k1)      # noqa: E731
                                         - self._apply(self.Dgll, X[:, p] * J[:, q, k1], k2))
                    cols.append(0.5 * (curl(a, b) - curl(b, a)))
                rows.append(torch.stack(cols, 1))
            met = torch.stack(rows, 1)
        self.met = self._all(self.I, met)
        if d == 2:                                                            # (only 2-D cases need det J)
            Jc = self._all(self.I, J)
            self.detJ = Jc[:, 0, 0] * Jc[:, 1, 1] - Jc[:, 0, 1] * Jc[:, 1, 0]
        # n J_f from the left element, interpolated from its face nodes
        nJ = torch.zeros((len(self.eL), d) + (N,) * (d - 1), dtype=torch.float64, device=DEV)
        for lf in range(2 * d):
            sel = (self.fL == lf).nonzero().squeeze(1)
            if len(sel):
                m = met[self.eL[sel], :, lf // 2]
                tr = m.select(m.dim() - 1 - lf // 2, N - 1 if lf % 2 else 0)
                nJ[sel] = (1.0 if lf % 2 else -1.0) * self._all(self.I, tr, range(d - 1))
        self.nJ = nJ
        self.Jf = torch.sqrt((nJ * nJ).sum(1, keepdim=True))
        self.n = nJ / self.Jf

    def _traces(self, a, e, f):
        """Values of (E, c, ...) nodal a on local faces f of elements e: (len(e), c, face nodes)."""
        out = torch.zeros((len(e), a.shape[1]) + (self.N,) * (self.d - 1), dtype=a.dtype, device=DEV)
        for lf in range(2 * self.d):
            sel = (f == lf).nonzero().squeeze(1)
            if len(sel):
                pick = a.select(a.dim() - 1 - lf // 2, self.N - 1 if lf % 2 else 0)
                out = out.index_copy(0, sel, pick[e[sel]])
        return out

    def _lift(self, out, x, e, f):
        """out[e] += x at the face nodes of local face f."""
        for lf in range(2 * self.d):
            sel = (f == lf).nonzero().squeeze(1)
            if len(sel):
                acc = torch.zeros((self.E,) + tuple(x.shape[1:]), dtype=x.dtype, device=DEV)
                acc = acc.index_add(0, e[sel], x[sel]).unsqueeze(-1 - lf // 2)
                rest = acc.new_zeros(tuple(self.N - 1 if k == acc.dim() - 1 - lf // 2 else n
                                           for k, n in enumerate(acc.shape)))
                out = out + torch.cat([rest, acc] if lf % 2 else [acc, rest], dim=acc.dim() - 1 - lf // 2)
        return out

    def _prims(self, s):
        d = self.d
        rho = s[:, 0]
        vel = s[:, 1:1 + d] / rho.unsqueeze(1)
        V2 = (vel * vel).sum(1)
        return rho, vel, V2, GM1 * (s[:, d + 1] - 0.5 * rho * V2)

    def _euler_flux(self, s):
        """(n, d, nv, ...)"""
        d = self.d
        rho, vel, V2, p = self._prims(s)
        rows = []
        for k in range(d):
            mom = [s[:, 1 + i] * vel[:, k] + (p if i == k else 0.0) for i in range(d)]
            rows.append(torch.stack([s[:, 1 + k]] + mom + [(s[:, d + 1] + p) * vel[:, k]], 1))
        return torch.stack(rows, 1)

    def _viscous_flux(self, s, g):
        """Negated viscous flux (n, 2, 4, ...) for gradients g (n, 2, 4, ...)."""
        rho, vel, V2, p = self._prims(s)
        E = s[:, 3]
        du = [[(g[:, j, 1 + k] - vel[:, k] * g[:, j, 0]) / rho for j in range(2)] for k in range(2)]
        div = du[0][0] + du[1][1]
        tau = [[self.mu * (du[i][j] + du[j][i]) - (2.0 / 3.0 * self.mu * div if i == j else 0.0) for j in range(2)]
               for i in range(2)]
        rows = []
        for j in range(2):
            dT = (g[:, j, 3] * rho - E * g[:, j, 0]) / rho ** 2 - (vel[:, 0] * du[0][j] + vel[:, 1] * du[1][j])
            q = GAMMA / self.Pr * self.mu * dT + vel[:, 0] * tau[j][0] + vel[:, 1] * tau[j][1]
            rows.append(torch.stack([torch.zeros_like(rho), -tau[0][j], -tau[1][j], -q], 1))
        return torch.stack(rows, 1)

    def _numflux(self, L, R):
        n, d = self.n, self.d
        if self.pde == "advection":
            bn = sum(self.b[k] * n[:, k] for k in range(d)).unsqueeze(1)
            return bn * torch.where(bn > 0, L, R)
        rL, vL, V2L, pL = self._prims(L)
        rR, vR, V2R, pR = self._prims(R)
        FL = (self._euler_flux(L) * n.unsqueeze(2)).sum(1)
        FR = (self._euler_flux(R) * n.unsqueeze(2)).sum(1)
        if self.flux == "lf":
            lam = torch.maximum(torch.sqrt(V2L) + torch.sqrt(GAMMA * pL / rL), torch.sqrt(V2R) + torch.sqrt(GAMMA * pR / rR))
            return 0.5 * (FL + FR + lam.unsqueeze(1) * (L - R))
        # Roe-Pike with the entropy fix on the acoustic waves
        VnL, VnR = (vL * n).sum(1), (vR * n).sum(1)
        HL, HR = (L[:, d + 1] + pL) / rL, (R[:, d + 1] + pR) / rR
        r = torch.sqrt(rR / rL)
        rho, H = r * rL, (r * HR + HL) / (r + 1.0)
        vel = (r.unsqueeze(1) * vR + vL) / (r + 1.0).unsqueeze(1)
        Vn, V2 = (vel * n).sum(1), (vel * vel).sum(1)
        c2 = GM1 * (H - 0.5 * V2)
        c = torch.sqrt(c2)
        l1 = torch.minimum((VnL - c).abs(), (Vn - c).abs())
        l5 = torch.maximum((VnR + c).abs(), (Vn + c).abs())
        l2 = Vn.abs()
        dp, dVn = pR - pL, VnR - VnL
        a1, a2 = 0.5 * (l5 + l1) - l2, 0.5 * (l5 - l1)
        d1 = a1 * dp / c2 + a2 * rho * dVn / c
        d2 = a1 * rho * dVn + a2 * dp / c
        wave = torch.cat([torch.ones_like(rho).unsqueeze(1), vel, H.unsqueeze(1)], 1) * d1.unsqueeze(1)
        wave2 = torch.cat([torch.zeros_like(rho).unsqueeze(1), n * d2.unsqueeze(1), (d2 * Vn).unsqueeze(1)], 1)
        return 0.5 * (FL + FR - (l2.unsqueeze(1) * (R - L) + wave + wave2))

    def _boundary(self, L):
        """Right state of the boundary faces (Riemann invariants or slip wall), L elsewhere unused."""
        d, n = self.d, self.n
        mVn = (L[:, 1:1 + d] * n).sum(1, keepdim=True)
        slip = torch.cat([L[:, :1], L[:, 1:1 + d] - 2.0 * mVn * n, L[:, d + 1:]], 1)
        rl, vl, V2l, pl = self._prims(L)
        rr, pr = self.prim[0], self.prim[d + 1]
        vr = torch.stack([torch.full_like(rl, self.prim[1 + k]) for k in range(d)], 1)
        cl, cr = torch.sqrt(GAMMA * pl / rl), math.sqrt(GAMMA * pr / rr)
        Vnl, Vnr = (vl * n).sum(1), (vr * n).sum(1)
        Rl, Rr = Vnl + 2.0 / GM1 * cl, Vnr - 2.0 / GM1 * cr
        Vn, c = 0.5 * (Rl + Rr), 0.25 * GM1 * (Rl - Rr)
        if bool((Vn.abs() >= c.abs())[self.bc == M.BC_RIEMANN].any()):
            raise ValueError("subsonic far field only")
        inlet = Vn < 0
        s = torch.where(inlet, torch.full_like(rl, pr / rr ** GAMMA), pl / rl ** GAMMA)
        rho = (c * c / (GAMMA * s)) ** (1.0 / GM1)
        vt = torch.where(inlet.unsqueeze(1), vr - Vnr.unsqueeze(1) * n, vl - Vnl.unsqueeze(1) * n)
        vel = Vn.unsqueeze(1) * n + vt
        p = c * c * rho / GAMMA
        far = torch.cat([rho.unsqueeze(1), rho.unsqueeze(1) * vel,
                         (p / GM1 + 0.5 * rho * (vel * vel).sum(1)).unsqueeze(1)], 1)
        is_slip = (self.bc == M.BC_SLIPWALL).reshape((-1,) + (1,) * (L.dim() - 1))
        return torch.where(is_slip, slip, far)

    def _face_states(self, u):
        d = self.d
        L = self._all(self.I, self._traces(u, self.eL, self.fL), range(d - 1))
        R = self._all(self.I, self._traces(u, self.eR.clamp(min=0), self.fR.clamp(min=0)), range(d - 1))
        if bool((self.eR < 0).any()):
            edge = (self.eR < 0).reshape((-1,) + (1,) * (L.dim() - 1))
            return L, torch.where(edge, self._boundary(L), R)
        return L, R

    def _scatter(self, FL, FR):
        """- sum over faces of phi J_f F: FL tested by the left element, FR (the same flux) by the right one."""
        out = torch.zeros((self.E, self.nv) + (self.N,) * self.d, dtype=torch.float64, device=DEV)
        it = self.I.T.contiguous()
        gl = self._all(it, self.wface * FL, range(self.d - 1))
        out = self._lift(out, -gl, self.eL, self.fL)
        inner = (self.eR >= 0).nonzero().squeeze(1)
        gr = self._all(it, self.wface * FR[inner], range(self.d - 1))
        return self._lift(out, gr, self.eR[inner], self.fR[inner])

    def _volume(self, F):
        """sum over directions of (d phi / d xi_j) w sum_i met[i, j] F_i"""
        out = None
        for j in range(self.d):
            x = self.wvol * sum(self.met[:, i, j].unsqueeze(1) * F[:, i] for i in range(self.d))
            for k in range(self.d):
                x = self._apply((self.DI if k == j else self.I).T.contiguous(), x, k)
            out = x if out is None else out + x
        return out

    def _shape(self, u):
        return u.reshape((self.E, self.nv) + (self.N,) * self.d)

    def residual(self, u):
        u = self._shape(u)
        s = self._all(self.I, u)
        if self.pde == "ns":
            return self._residual_ns(u, s)
        if self.pde == "advection":
            F = torch.stack([self.b[k] * s for k in range(self.d)], 1)
        else:
            F = self._euler_flux(s)
        r = self._volume(F)
        del F, s
        f = self.Jf * self._numflux(*self._face_states(u))
        return (r + self._scatter(f, f)).reshape(-1)

    def _residual_ns(self, u, s):
        """BR2: volume gradient plus lifted jumps, face gradients with eta = 1.01 x 4 (2-D, aligned faces)."""
        N = self.N
        d0, d1 = (self._apply(self.DI, self._apply(self.I, u, 1), 0), self._apply(self.DI, self._apply(self.I, u, 0), 1))
        Ji = 1.0 / self.detJ
        g = torch.stack([(self.met[:, i, 0] * Ji).unsqueeze(1) * d0 + (self.met[:, i, 1] * Ji).unsqueeze(1) * d1
                         for i in range(2)], 1)                               # (E, 2, 4, N, N)
        L, R = self._face_states(u)
        q = self.nJ.unsqueeze(2) * (0.5 * (R - L)).unsqueeze(1)               # (F, 2, 4, N)
        gs = []
        full = g
        for e, f in ((self.eL, self.fL), (self.eR, self.fR)):
            tr = torch.zeros_like(q)
            kap = torch.zeros((len(e), N), dtype=torch.float64, device=DEV)
            for lf in range(4):
                sel = (f == lf).nonzero().squeeze(1)
                if not len(sel):
                    continue
                end = self.ends[lf % 2]
                ax = -1 - lf // 2
                tr[sel] = torch.movedim(g[e[sel]], ax, -1) @ end
                wj = torch.movedim(self.detJ[e[sel]], ax, -1)                 # (n, N face, N normal)
                kap[sel] = (end ** 2 / (self.w * wj)).sum(-1)
                coef = end / (self.w * wj)
                add = torch.movedim(q[sel].unsqueeze(-1) * coef[:, None, None], -1, ax)
                full = full.index_add(0, e[sel], add)
            gs.append(tr + 1.01 * 4.0 * kap[:, None, None] * q)
        r = self._volume(self._euler_flux(s) + self._viscous_flux(s, full))
        vis = 0.5 * (self._viscous_flux(L, gs[0]) + self._viscous_flux(R, gs[1]))
        f = self.Jf * (self._numflux(L, R) + (vis * self.n.unsqueeze(2)).sum(1))
        return (r + self._scatter(f, f)).reshape(-1)

    def mass(self, x):
        """M x with the collocated mass matrix."""
        y = self._all(self.I, self._shape(x)) * (self.wvol * self.detJ).unsqueeze(1)
        return self._all(self.I.T.contiguous(), y).reshape(-1)

    def mass_inverse(self, r):
        inv = torch.linalg.inv(self.I)
        y = self._all(inv.T.contiguous(), self._shape(r)) / (self.wvol * self.detJ).unsqueeze(1)
        return self._all(inv, y).reshape(-1)

    def jacobian_vector(self, u, v):
        return torch.func.jvp(self.residual, (u,), (v,))[1]

    def diagonal_blocks(self, u):
        """dR_e / du_e, the neighbours held fixed: (E, nb, nb)."""
        u = self._shape(u)
        nb = self.nv * self.N ** self.d
        blocks = torch.empty((self.E, nb, nb), dtype=torch.float64, device=DEV)
        edge = (self.eR < 0).reshape((-1,) + (1,) * self.d)
        L0, R0 = self._face_states(u)

        def own(x):
            r = self._volume(self._euler_flux(self._all(self.I, x)))
            L, R = self._face_states(x)
            left = self.Jf * self._numflux(L, torch.where(edge, R, R0))
            right = self.Jf * self._numflux(L0, R)
            return r + self._scatter(left, right)

        for c in range(nb):
            seed = torch.zeros((self.E, nb), dtype=torch.float64, device=DEV)
            seed[:, c] = 1.0
            blocks[:, :, c] = torch.func.jvp(own, (u,), (seed.reshape(u.shape),))[1].reshape(self.E, nb)
        return blocks

    def mass_blocks(self):
        n = self.N ** self.d
        out = torch.empty((self.E, n, n), dtype=torch.float64, device=DEV)
        keep, self.nv = self.nv, 1
        for c in range(n):
            x = torch.zeros((self.E, n), dtype=torch.float64, device=DEV)
            x[:, c] = 1.0
            out[:, :, c] = self.mass(x.reshape(-1)).reshape(self.E, n)
        self.nv = keep
        return out

    def limit(self, u):
        """The positivity limiter on Bezier coefficients of the primitive variables."""
        d = self.d
        c = self._all(self.bern_inv, self._shape(u)).reshape(self.E, self.nv, -1)
        rho, vel, V2, p = self._prims(c)
        prim = torch.cat([rho.unsqueeze(1), vel, p.unsqueeze(1)], 1)
        for k in (0, self.nv - 1):
            avg, low = prim[:, k].mean(1), prim[:, k].min(1).values
            phi = torch.where(low < EPS_PHYS, ((avg - EPS_PHYS) / (avg - low)).clamp(0.0, 1.0), torch.ones_like(avg))
            mean = prim.mean(2, keepdim=True)
            prim = torch.where((low < EPS_PHYS)[:, None, None], phi[:, None, None] * prim + (1 - phi)[:, None, None] * mean, prim)
        rho, vel, p = prim[:, 0], prim[:, 1:1 + d], prim[:, d + 1]
        cons = torch.cat([rho.unsqueeze(1), rho.unsqueeze(1) * vel, (p / GM1 + 0.5 * rho * (vel * vel).sum(1)).unsqueeze(1)], 1)
        return self._all(self.bern, self._shape(cons)).reshape(-1)

    def rk3(self, u, dt, steps, limiter):
        fix = self.limit if limiter else (lambda x: x)
        rate = lambda x: self.mass_inverse(self.residual(x))                  # noqa: E731
        for _ in range(steps):
            a = fix(u + dt * rate(u))
            b = fix(0.25 * (3.0 * u + a + dt * rate(a)))
            last = rate(b)
            u = fix((u + 2.0 * b + 2.0 * dt * last) / 3.0)
        return u, float(last.abs().max())


def _exact_training(case, seed):
    """One epoch of Adam on the float64 network with the weights rounded to bfloat16 for every product."""
    st = _prepare_training(case, seed)
    nb, n, batch, h = st["blocks"].shape[1], case["samples"], case["batch"], case["hidden"]
    Np, R = nb // 4, case["rank"]
    nf = st["feat"].shape[1]
    X, sig = st["feat"].double(), st["sigma"].double()
    w = torch.from_numpy(st["w0"]).double().to(DEV)
    no = R * (16 + Np * Np) if case["structure"] == "kron" else nb + 2 * nb * R
    sizes = [(h, nf), (h,), (h, h), (h,), (no, h), (no,)]

    def loss_of(wb, lo, hi):
        parts, at = [], 0
        for s in sizes:
            k = math.prod(s)
            parts.append(wb[at:at + k].reshape(s))
            at += k
        y = torch.tanh(X[lo:hi] @ parts[0].T + parts[1])
        y = torch.tanh(y @ parts[2].T + parts[3])
        o = y @ parts[4].T + parts[5]
        if case["structure"] == "kron":
            S, Q = o[:, :R * 16].reshape(-1, R, 4, 4), o[:, R * 16:].reshape(-1, R, Np, Np)
            P = (S.reshape(-1, R, 16).transpose(1, 2) @ Q.reshape(-1, R, Np * Np)).reshape(-1, 4, 4, Np, Np)
            P = P.permute(0, 1, 3, 2, 4).reshape(-1, nb, nb)
        else:
            U, V = o[:, nb:nb + nb * R].reshape(-1, nb, R), o[:, nb + nb * R:].reshape(-1, nb, R)
            P = torch.diag_embed(o[:, :nb]) + U @ V.transpose(1, 2)
        res = sig[lo:hi, None, None] * (P @ st["blocks"][lo:hi]) - torch.eye(nb, dtype=torch.float64, device=DEV)
        return (res ** 2).sum((1, 2)).mean() / nb

    # mini-batches are visited in the order of a seeded Fisher-Yates shuffle (splitmix64)
    mask, s = (1 << 64) - 1, 0x5EED
    order = list(range(-(-n // batch)))
    for i in range(len(order) - 1, 0, -1):
        s = (s + 0x9E3779B97F4A7C15) & mask
        z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        j = (z ^ (z >> 31)) % (i + 1)
        order[i], order[j] = order[j], order[i]
    m, v = torch.zeros_like(w), torch.zeros_like(w)
    rounded = lambda x: x.float().bfloat16().double()                         # noqa: E731
    for step, k in enumerate(order, 1):
        wb = rounded(w).requires_grad_(True)
        g, = torch.autograd.grad(loss_of(wb, k * batch, min(n, (k + 1) * batch)), wb)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        w = w - 1e-4 * (m / (1 - 0.9 ** step)) / (torch.sqrt(v / (1 - 0.999 ** step)) + 1e-8)
    return w


def exact(case, seed):
    kind = case["kind"]
    if kind == "mixed_residual":
        return None          # the symmetric TRI cubature rules exist only as the library's tables
    if kind == "steady":
        return None          # a float64 torch Newton-GMRES of this system takes minutes
    if kind == "train":
        return _exact_training(case, seed)
    mesh = _uniform_mesh(case)
    u = _uniform_state(case, mesh, seed)
    if kind == "residual":
        if case["dtype"] == "f32":
            u = u.float().double()
        return _Plain(mesh, case["pde"], case["flux"]).residual(u)
    if kind == "time_steps":
        u, mx = _Plain(mesh, case["pde"]).rk3(u, _time_step(case), case["steps"], case["pde"] == "euler")
        return u if case["api"] == "graph" else (u, mx)
    st = prepare(case, seed)
    plain = _Plain(mesh, "euler", "roe", bc_prim=M.freestream_prim(2))
    scale = st["inv_dt"]
    if kind == "newton_operator":
        jv = plain.jacobian_vector(st["u"], st["v"])
        return jv - (scale[:, None] * plain.mass(st["v"]).reshape(mesh.E, -1)).reshape(-1)
    blocks = plain.diagonal_blocks(st["u"])
    mass = scale[:, None, None] * plain.mass_blocks()
    n = mesh.Np
    for k in range(4):
        blocks[:, k * n:(k + 1) * n, k * n:(k + 1) * n] -= mass
    return torch.linalg.inv(blocks).transpose(1, 2).contiguous()
