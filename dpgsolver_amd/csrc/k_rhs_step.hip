// k_rhs_step.hip -- SSP-RK3 stages of uniform-order Euler and advection meshes, residual, M^-1, stage arithmetic and
// positivity limiter in one kernel (time_step_ssp_rk_33, solve_explicit.c:252-301).  A translation unit of its own: the
// residual kernels keep the register allocation they have in k_rhs64.hip.
#include "k_residual.h"

namespace dgx {

bool rk_fused(const Ctx& c)
{
	// Navier-Stokes takes two kernels for its residual.  A persistent grid chosen for the M^-1 R kernel is that kernel's alone:
	// it gains a few per cent where the fused stages halve the step (below).
	return c.cfg.pde != DGX_PDE_NAVIER_STOKES && !c.has_nonconforming;
}

// The three stages go u -> a -> b -> u: a stage never overwrites the state whose traces other elements still read, and
// the step's initial state stays in u until the last stage combines it, so nothing is copied.  What bounds a stage: on
// small meshes the latency of one launch (launches per step 9 or 12 before, with the max-norm slot's fill, the stage
// and the limiter kernels); on large ones one read of u and base and one write.  128 x 128 QUAD p = 3 Euler with the
// limiter: 169 us -> 65 us per step; 16 x 16 QUAD p = 2 advection: 46.1 -> 25.5 us.
hipError_t launch_rk3_fused(Ctx& c, double* u, double* ua, double* ub, double dt, bool positivity, int* status,
                            unsigned long long* dmax)
{
	RhsArgs<double, double> a{};
	a.met = c.metrics_vc;
	a.detJ = c.detJ_vc;
	a.nJ = c.nJ_fc;
	a.ef = c.elem_faces;
	a.order = c.order;
	a.ops = c.ops64;
	for (int k = 0; k < 5; ++k) a.bc_prim[k] = c.cfg.bc_prim[k];
	for (int k = 0; k < 3; ++k) a.b_adv[k] = c.cfg.b_adv[k];
	a.E = c.E;
	a.dt = dt;
	a.status = status;
	a.base = u;
	double* src[3] = { u, ua, ub };
	double* dst[3] = { ua, ub, u };
	for (int stage = 0; stage < 3; ++stage) {
		a.stage = stage;
		a.u = src[stage];
		a.out = dst[stage];
		a.dmax = stage == 2 ? dmax : nullptr;      // max |M^-1 R| of the last stage
		a.clear = stage == 0 ? dmax : nullptr;
		const int pde = c.cfg.pde, flux = c.cfg.num_flux;
		if (positivity && pde == DGX_PDE_EULER)
			DGX_HIP_CHECK((dispatch_rhs<double, double, MODE_RK_POS>(c.d, c.p, pde, flux, a, c.stream)));
		else
			DGX_HIP_CHECK((dispatch_rhs<double, double, MODE_RK>(c.d, c.p, pde, flux, a, c.stream)));
	}
	return hipSuccess;
}

}  // namespace dgx
