// dgx_implicit.hip -- pseudo-time Newton-GMRES for steady problems (solve_implicit.c:95-110, 232-281).
//
// Per Newton step: r = R(u); max|r| exit test (check_exit, solve_implicit.c:258-281); CFL-ramped
// per-element dt = cfl * h_min / max wave speed (compute_dt_cfl_constrained, solve_dg.c:284-319);
// linear system (dR/du - M/dt) du = -r (compute_CFL_ramping solve_dg.c:223-248, fill_petsc_Vec_b_dg
// :203-221) solved by right-preconditioned restarted GMRES (the reference uses PETSc GMRES(60),
// rtol 1e-4, external/petsc/options_files/petsc_options_gmres_default.txt) with a block-Jacobi LU or a
// learned preconditioner; update u += relax du with positivity under-relaxation (update_coef /
// compute_relaxation, solve_implicit.c:780-873).  The operator is matrix-free: exact J v by dual numbers,
// M v sum-factorised.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

#include "dgx_device.h"
#include "dgx_internal.h"

namespace dgx {

template <int D, int N>
__device__ inline void coords2(int n, int* c)
{
	c[0] = n % N;
	c[1] = (D > 1) ? (n / N) % N : 0;
	c[2] = (D > 2) ? n / (N * N) : 0;
}
template <int D, int N>
__device__ inline double apply1d_(const double* M, const double* buf, int n, int k)
{
	int c[3];
	coords2<D, N>(n, c);
	double acc = 0.0;
	for (int j = 0; j < N; ++j) {
		int cc[3] = { c[0], c[1], c[2] };
		cc[k] = j;
		acc += M[c[k] * N + j] * buf[cc[0] + N * (cc[1] + N * cc[2])];
	}
	return acc;
}

// y_e -= s_e * M_e x_e with M_e = Ibar^T diag(w J) Ibar per variable
template <int D, int N, int NV>
__global__ void __launch_bounds__(128) k_mass_sub(const double* __restrict__ x, const double* __restrict__ detJ,
                                                  const double* __restrict__ scale, const Ops1D<double>* ops, int E,
                                                  double* y)
{
	constexpr int Np = ipow(N, D);
	__shared__ double B0[NV * Np], B1[NV * Np], sI[N * N], sIT[N * N], sW[N];
	const int e = blockIdx.x, n = threadIdx.x;
	for (int i = threadIdx.x; i < N * N; i += blockDim.x) { sI[i] = ops->I[i]; sIT[i] = ops->IT[i]; }
	for (int i = threadIdx.x; i < N; i += blockDim.x) sW[i] = ops->w[i];
	for (int i = threadIdx.x; i < NV * Np; i += blockDim.x) B0[i] = x[(size_t)e * NV * Np + i];
	__syncthreads();
	double* cur = B0;
	double* nxt = B1;
	for (int pass = 0; pass < 2 * D; ++pass) {
		const double* M = pass < D ? sI : sIT;
		if (n < Np)
			for (int v = 0; v < NV; ++v) nxt[v * Np + n] = apply1d_<D, N>(M, cur + v * Np, n, pass % D);
		__syncthreads();
		if (pass == D - 1 && n < Np) {
			int c[3];
			coords2<D, N>(n, c);
			double wq = sW[c[0]] * sW[c[1]];
			if (D == 3) wq *= sW[c[2]];
			const double s = wq * detJ[(size_t)e * Np + n];
			for (int v = 0; v < NV; ++v) nxt[v * Np + n] *= s;
		}
		__syncthreads();
		double* t = cur; cur = nxt; nxt = t;
	}
	const double s = scale ? scale[e] : 1.0;
	for (int i = threadIdx.x; i < NV * Np; i += blockDim.x) y[(size_t)e * NV * Np + i] -= s * cur[i];
}

// per-element dt = cfl * min(h_min / max(|V| + c), h_min^2 / mu) over the Bezier coefficients (the viscous
// bound with mu > 0, the Navier-Stokes constant viscosity; solve_dg.c:284-319)
template <int D, int N>
__global__ void __launch_bounds__(128) k_cfl_dt(const double* __restrict__ u, const double* __restrict__ hmin,
                                                const Ops1D<double>* ops, int E, double cfl, double mu,
                                                int sutherland, double r_s, double* inv_dt)
{
	constexpr int Np = ipow(N, D), NV = D + 2;
	__shared__ double B0[NV * Np], B1[NV * Np], sBinv[N * N], sWs[Np], sMu[Np];
	const int e = blockIdx.x, n = threadIdx.x;
	for (int i = threadIdx.x; i < N * N; i += blockDim.x) sBinv[i] = ops->Binv[i];
	for (int i = threadIdx.x; i < NV * Np; i += blockDim.x) B0[i] = u[(size_t)e * NV * Np + i];
	__syncthreads();
	double* cur = B0;
	double* nxt = B1;
	for (int k = 0; k < D; ++k) {
		if (n < Np)
			for (int v = 0; v < NV; ++v) nxt[v * Np + n] = apply1d_<D, N>(sBinv, cur + v * Np, n, k);
		__syncthreads();
		double* t = cur; cur = nxt; nxt = t;
	}
	if (n < Np) {
		const double rho = cur[n], ri = 1.0 / rho;
		double V2 = 0.0;
		for (int k = 0; k < D; ++k) { const double w = cur[(1 + k) * Np + n] * ri; V2 += w * w; }
		const double p = kGM1 * (cur[(D + 1) * Np + n] - 0.5 * rho * V2);
		sWs[n] = sqrt(V2) + sqrt(kGamma * p * ri);
		// the largest viscosity over the coefficients (compute_viscosity, solve_dg.c:300-307)
		const double T = p * ri / r_s;
		sMu[n] = sutherland ? 8e-2 * mu * sqrt(T) / (1.0 + 112.0 / T) : mu;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		double m = 0.0, mmu = 0.0;
		for (int i = 0; i < Np; ++i) {
			m = fmax(m, sWs[i]);
			mmu = fmax(mmu, sMu[i]);
		}
		inv_dt[e] = fmax(m / (cfl * hmin[e]), mmu / (cfl * hmin[e] * hmin[e]));
	}
}

// u_e += relax_e du_e, relax halved until the Bezier-coefficient means of rho and p exceed EPS_PHYS
// (compute_relaxation, solve_implicit.c:823-873)
template <int D, int N>
__global__ void __launch_bounds__(128) k_relaxed_update(double* u, const double* __restrict__ du,
                                                       const Ops1D<double>* ops, int E, int* status,
                                                       double* relax_out)
{
	constexpr int Np = ipow(N, D), NV = D + 2;
	__shared__ double Bu[NV * Np], Bd[NV * Np], T[NV * Np], sBinv[N * N];
	__shared__ double sRelax;
	const int e = blockIdx.x, n = threadIdx.x;
	for (int i = threadIdx.x; i < N * N; i += blockDim.x) sBinv[i] = ops->Binv[i];
	for (int i = threadIdx.x; i < NV * Np; i += blockDim.x) {
		Bu[i] = u[(size_t)e * NV * Np + i];
		Bd[i] = du[(size_t)e * NV * Np + i];
	}
	__syncthreads();
	for (int arr = 0; arr < 2; ++arr) {
		double* X = arr == 0 ? Bu : Bd;
		for (int k = 0; k < D; ++k) {
			if (n < Np)
				for (int v = 0; v < NV; ++v) T[v * Np + n] = apply1d_<D, N>(sBinv, X + v * Np, n, k);
			__syncthreads();
			if (n < Np)
				for (int v = 0; v < NV; ++v) X[v * Np + n] = T[v * Np + n];
			__syncthreads();
		}
	}
	if (threadIdx.x == 0) {
		double relax = 1.0;
		for (;;) {
			double ar = 0.0, ap = 0.0;
			for (int i = 0; i < Np; ++i) {
				const double rho = Bu[i] + relax * Bd[i];
				double V2 = 0.0;
				for (int k = 0; k < D; ++k) {
					const double w = (Bu[(1 + k) * Np + i] + relax * Bd[(1 + k) * Np + i]) / rho;
					V2 += w * w;
				}
				ar += rho;
				ap += kGM1 * ((Bu[(D + 1) * Np + i] + relax * Bd[(D + 1) * Np + i]) - 0.5 * rho * V2);
			}
			ar /= Np;
			ap /= Np;
			if (!(ar < kEpsPhys || ap < kEpsPhys)) break;
			relax *= 0.5;
			if (relax < kEps) { atomicOr(status, 1); break; }
		}
		sRelax = relax;
		if (relax_out) relax_out[e] = relax;
	}
	__syncthreads();
	const double r = sRelax;
	for (int i = threadIdx.x; i < NV * Np; i += blockDim.x) u[(size_t)e * NV * Np + i] += r * du[(size_t)e * NV * Np + i];
}

// ------------------------------------------------------------------------------- BLAS-1 (deterministic)
// Krylov vectors are cut into at most kMaxChunks chunks of a multiple of kChunkUnit values, one workgroup each; a dot
// product is the sum of its chunks' partial sums in chunk order, so results do not depend on scheduling.  256 chunks
// are one workgroup per CU; 512 values are 8 per lane of the wavefront that owns a row.
constexpr int kChunkUnit = 512, kMaxChunks = 256, kMaxRows = 208;

struct Chunks {
	int count = 0;
	size_t size = 0;
};
static Chunks chunks_of(size_t n)
{
	const size_t units = (n + kChunkUnit - 1) / kChunkUnit;
	const size_t per = (units + kMaxChunks - 1) / kMaxChunks;
	Chunks c;
	c.size = (per > 0 ? per : 1) * kChunkUnit;
	c.count = (int)((n + c.size - 1) / c.size);
	return c;
}

// DPP wave reduction (no LDS round trips): sums within rows of 16 lanes, then across them; the total is lane 63's,
// returned in every lane
__device__ inline double wave_sum(double x)
{
#define DGX_DPP_ADD(ctrl, rows)                                                                                       \
	{                                                                                                                 \
		const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), ctrl, rows, 0xf, false);                     \
		const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), ctrl, rows, 0xf, false);                     \
		x += __hiloint2double(hi, lo);                                                                                \
	}
	DGX_DPP_ADD(0x111, 0xf)   // row_shr:1
	DGX_DPP_ADD(0x112, 0xf)   // row_shr:2
	DGX_DPP_ADD(0x114, 0xf)   // row_shr:4
	DGX_DPP_ADD(0x118, 0xf)   // row_shr:8
	DGX_DPP_ADD(0x142, 0xa)   // row_bcast:15
	DGX_DPP_ADD(0x143, 0xc)   // row_bcast:31
#undef DGX_DPP_ADD
	return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), 63), __builtin_amdgcn_readlane(__double2loint(x), 63));
}
// sum of partial[row][0 .. nc) over the chunks, by one wavefront
__device__ inline double row_sum(const double* __restrict__ partial, int row, int nc, int lane)
{
	double s = 0.0;
#pragma unroll
	for (int c = 0; c < kMaxChunks; c += 64) s += (c + lane < nc) ? partial[(size_t)row * kMaxChunks + c + lane] : 0.0;
	return wave_sum(s);
}

constexpr int kGsLanes = 1024;

// acc[row] += V_row . w over one unit of the chunk (w in LDS, zero beyond n), rows dealt to the wavefronts; a lane
// holds its eight values of w for all rows and loads two rows at a time
__device__ inline void unit_dots(const float* __restrict__ V, size_t ldv, int k, size_t base, size_t n, const double* sw,
                                 double* acc)
{
	constexpr int NW = kGsLanes / 64;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	double w[8];
#pragma unroll
	for (int q = 0; q < 8; ++q) w[q] = sw[(q >> 2) * 256 + 4 * lane + (q & 3)];
	if (base + kChunkUnit <= n && (ldv & 3) == 0) {
		for (int r = wave; r < k; r += 2 * NW) {
			const float* v0 = V + (size_t)r * ldv + base + 4 * lane;
			const float* v1 = V + (size_t)(r + NW < k ? r + NW : r) * ldv + base + 4 * lane;
			const float4 a = *reinterpret_cast<const float4*>(v0), b = *reinterpret_cast<const float4*>(v0 + 256);
			const float4 c = *reinterpret_cast<const float4*>(v1), d = *reinterpret_cast<const float4*>(v1 + 256);
			double s0 = (((double)a.x * w[0] + (double)a.y * w[1]) + ((double)a.z * w[2] + (double)a.w * w[3])) +
			            (((double)b.x * w[4] + (double)b.y * w[5]) + ((double)b.z * w[6] + (double)b.w * w[7]));
			double s1 = (((double)c.x * w[0] + (double)c.y * w[1]) + ((double)c.z * w[2] + (double)c.w * w[3])) +
			            (((double)d.x * w[4] + (double)d.y * w[5]) + ((double)d.z * w[6] + (double)d.w * w[7]));
			s0 = wave_sum(s0);
			s1 = wave_sum(s1);
			if (lane == 0) {
				acc[r] += s0;
				if (r + NW < k) acc[r + NW] += s1;
			}
		}
	} else {
		for (int r = wave; r < k; r += NW) {
			const float* v = V + (size_t)r * ldv + base;
			double s = 0.0;
#pragma unroll
			for (int q = 0; q < 8; ++q) {
				const int o = (q >> 2) * 256 + 4 * lane + (q & 3);
				if (base + o < n) s += (double)v[o] * w[q];
			}
			s = wave_sum(s);
			if (lane == 0) acc[r] += s;
		}
	}
}

// One step of the Gram-Schmidt chain on one chunk:
//   SUB:  w -= V h, h = the k row sums of `in` (the previous step's partial sums);
//   DOTS: out[row][chunk] = V_row . w of the updated w; otherwise out[0][chunk] = |w|^2.
// Bound by the latency of reading V once (FP32 basis, in the caches) and by launches: with the subtraction and the next
// dot products in one kernel an Arnoldi step takes four launches where it took seven, and w is read and written once
// per pass instead of once per row.  Sixteen wavefronts a workgroup, since one workgroup per CU is all there is: each
// wavefront takes every sixteenth row of the dot products, each quarter of the lanes every fourth row of V h.
template <bool SUB, bool DOTS>
__global__ void __launch_bounds__(kGsLanes) k_gs(const float* __restrict__ V, size_t ldv, int k, double* w, size_t n,
                                                 size_t chunk, int nc, const double* __restrict__ in, double* out)
{
	constexpr int NW = kGsLanes / 64;
	__shared__ double sh[kMaxRows], acc[kMaxRows], sw[kChunkUnit], sp[SUB ? 3 : 1][SUB ? kChunkUnit : 1];
	const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
	if constexpr (SUB)
		for (int r = wave; r < k; r += NW) {
			const double h = row_sum(in, r, nc, lane);
			if (lane == 0) sh[r] = h;
		}
	for (int r = t; r < kMaxRows; r += kGsLanes) acc[r] = 0.0;
	__syncthreads();
	const size_t lo = (size_t)blockIdx.x * chunk;
	const size_t hi = lo + chunk < n ? lo + chunk : n;
	double nrm = 0.0;
	for (size_t base = lo; base < hi; base += kChunkUnit) {
		if constexpr (SUB) {
			// value pair 2 (t mod 256), rows t / 256, t / 256 + 4, ...
			const int part = t >> 8, o = 2 * (t & 255);
			double s0 = 0.0, s1 = 0.0;
			if (base + kChunkUnit <= n && (ldv & 1) == 0) {
#pragma unroll 8
				for (int r = part; r < k; r += 4) {
					const float2 v = *reinterpret_cast<const float2*>(V + (size_t)r * ldv + base + o);
					s0 += (double)v.x * sh[r];
					s1 += (double)v.y * sh[r];
				}
			} else {
				for (int r = part; r < k; r += 4) {
					if (base + o < hi) s0 += (double)V[(size_t)r * ldv + base + o] * sh[r];
					if (base + o + 1 < hi) s1 += (double)V[(size_t)r * ldv + base + o + 1] * sh[r];
				}
			}
			if (part > 0) {
				sp[part - 1][o] = s0;
				sp[part - 1][o + 1] = s1;
			} else {
				sw[o] = s0;
				sw[o + 1] = s1;
			}
			__syncthreads();
		}
		if (t < kChunkUnit) {
			const size_t i = base + t;
			double x = i < hi ? w[i] : 0.0;
			if constexpr (SUB) {
				x -= (sw[t] + sp[0][t]) + (sp[1][t] + sp[2][t]);
				if (i < hi) w[i] = x;
				else x = 0.0;
			}
			nrm += x * x;
			sw[t] = x;
		}
		if constexpr (DOTS) {
			__syncthreads();
			unit_dots(V, ldv, k, base, n, sw, acc);
		}
		__syncthreads();
	}
	if constexpr (DOTS) {
		for (int r = t; r < k; r += kGsLanes) out[(size_t)r * kMaxChunks + blockIdx.x] = acc[r];
	} else {
		nrm = wave_sum(nrm);
		if (lane == 0) acc[wave] = nrm;
		__syncthreads();
		if (t == 0) {
			double s = 0.0;
			for (int q = 0; q < NW; ++q) s += acc[q];
			out[blockIdx.x] = s;
		}
	}
}
// out[0] = the sum of the nc partial sums
__global__ void __launch_bounds__(64) k_sum_final(const double* __restrict__ partial, int nc, double* out)
{
	const double s = row_sum(partial, 0, nc, threadIdx.x);
	if (threadIdx.x == 0) out[0] = s;
}
// y = a x + b y
__global__ void k_axpby(double a, const double* __restrict__ x, double b, double* y, size_t n)
{
	for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
		y[i] = a * x[i] + (b == 0.0 ? 0.0 : b * y[i]);
}
// y = V c (k vectors), accumulate
template <typename TV>
__global__ void k_gemv_add(const TV* __restrict__ V, size_t ldv, const double* __restrict__ c, int k, double* y,
                           size_t n)
{
	for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
		double s = 0.0;
		for (int j = 0; j < k; ++j) s += (double)V[(size_t)j * ldv + i] * c[j];
		y[i] += s;
	}
}

static int grid_for(size_t n) { return (int)((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096); }

struct Blas {
	hipStream_t s;
	double* partial = nullptr;  // kMaxChunks * kmax
	double* partial2 = nullptr; // kMaxChunks * kmax: second Gram-Schmidt pass
	double* partialn = nullptr; // kMaxChunks: |w|^2
	double* dvec = nullptr;     // kmax
	hipError_t init(hipStream_t st, int k)
	{
		s = st;
		DGX_HIP_CHECK(hipMalloc(&partial, sizeof(double) * kMaxChunks * k));
		DGX_HIP_CHECK(hipMalloc(&partial2, sizeof(double) * kMaxChunks * k));
		DGX_HIP_CHECK(hipMalloc(&partialn, sizeof(double) * kMaxChunks));
		DGX_HIP_CHECK(hipMalloc(&dvec, sizeof(double) * k));
		return hipSuccess;
	}
	void release()
	{
		for (double* q : { partial, partial2, partialn, dvec })
			if (q) (void)hipFree(q);
		partial = partial2 = partialn = dvec = nullptr;
	}
	template <bool SUB, bool DOTS>
	hipError_t gs(const float* V, size_t ldv, int k, double* w, size_t n, const double* in, double* out)
	{
		const Chunks ch = chunks_of(n);
		hipLaunchKernelGGL((k_gs<SUB, DOTS>), dim3(ch.count), dim3(kGsLanes), 0, s, V, ldv, k, w, n, ch.size, ch.count, in,
		                   out);
		return hipGetLastError();
	}
	template <typename TV>
	hipError_t gemv_add(const TV* V, size_t ldv, const double* cc, int k, double* y, size_t n)
	{
		DGX_HIP_CHECK(hipMemcpyAsync(dvec, cc, sizeof(double) * k, hipMemcpyHostToDevice, s));
		hipLaunchKernelGGL(k_gemv_add<TV>, dim3(grid_for(n)), dim3(256), 0, s, V, ldv, dvec, k, y, n);
		return hipGetLastError();
	}
	hipError_t axpby(double a, const double* x, double b, double* y, size_t n)
	{
		hipLaunchKernelGGL(k_axpby, dim3(grid_for(n)), dim3(256), 0, s, a, x, b, y, n);
		return hipGetLastError();
	}
	// |x| on the host (synchronous)
	hipError_t norm(double* x, size_t n, double* out)
	{
		const Chunks ch = chunks_of(n);
		hipLaunchKernelGGL((k_gs<false, false>), dim3(ch.count), dim3(kGsLanes), 0, s, (const float*)nullptr, (size_t)0, 0, x,
		                   n, ch.size, ch.count, (const double*)nullptr, partialn);
		hipLaunchKernelGGL(k_sum_final, dim3(1), dim3(64), 0, s, partialn, ch.count, dvec);
		double v;
		DGX_HIP_CHECK(hipGetLastError());
		DGX_HIP_CHECK(hipMemcpyAsync(&v, dvec, sizeof(double), hipMemcpyDeviceToHost, s));
		DGX_HIP_CHECK(hipStreamSynchronize(s));
		*out = std::sqrt(v);
		return hipSuccess;
	}
};

// one workgroup per element, a lane per node (HEX p = 4: 128 lanes for its 125 nodes)
#define DGX_PER_ELEM2(KNAME, BLK, ...)                                                               \
	switch (c.d * 16 + c.N) {                                                                       \
	case 2 * 16 + 2: hipLaunchKernelGGL((KNAME<2, 2 __VA_ARGS__>), dim3(c.E), dim3(BLK), 0, c.stream, ARGS); break; \
	case 2 * 16 + 3: hipLaunchKernelGGL((KNAME<2, 3 __VA_ARGS__>), dim3(c.E), dim3(BLK), 0, c.stream, ARGS); break; \
	case 2 * 16 + 4: hipLaunchKernelGGL((KNAME<2, 4 __VA_ARGS__>), dim3(c.E), dim3(BLK), 0, c.stream, ARGS); break; \
	case 2 * 16 + 5: hipLaunchKernelGGL((KNAME<2, 5 __VA_ARGS__>), dim3(c.E), dim3(BLK), 0, c.stream, ARGS); break; \
	case 2 * 16 + 6: hipLaunchKernelGGL((KNAME<2, 6 __VA_ARGS__>), dim3(c.E), dim3(BLK), 0, c.stream, ARGS); break; \
	case 3 * 16 + 2: hipLaunchKernelGGL((KNAME<3, 2 __VA_ARGS__>), dim3(c.E), dim3(64), 0, c.stream, ARGS); break;  \
	case 3 * 16 + 3: hipLaunchKernelGGL((KNAME<3, 3 __VA_ARGS__>), dim3(c.E), dim3(64), 0, c.stream, ARGS); break;  \
	case 3 * 16 + 4: hipLaunchKernelGGL((KNAME<3, 4 __VA_ARGS__>), dim3(c.E), dim3(64), 0, c.stream, ARGS); break;  \
	case 3 * 16 + 5: hipLaunchKernelGGL((KNAME<3, 5 __VA_ARGS__>), dim3(c.E), dim3(128), 0, c.stream, ARGS); break; \
	default: return hipErrorInvalidValue;                                                       \
	}

hipError_t launch_mass_sub(Ctx& c, const double* x, const double* scale, double* y)
{
	if (c.E == 0) return hipSuccess;
	if (c.d != 2 && c.d != 3) return hipErrorInvalidValue;
#define ARGS x, c.detJ_vc, scale, c.ops64, c.E, y
	if (c.nv == 1) { DGX_PER_ELEM2(k_mass_sub, 64, , 1) }
	else if (c.nv == 4) { DGX_PER_ELEM2(k_mass_sub, 64, , 4) }
	else { DGX_PER_ELEM2(k_mass_sub, 64, , 5) }
#undef ARGS
	return hipGetLastError();
}

hipError_t launch_cfl_dt(Ctx& c, const double* u, double cfl, double* inv_dt)
{
	if (c.nv != c.d + 2) return hipErrorInvalidValue;   // Euler and Navier-Stokes
#define ARGS u, c.hmin, c.ops64, c.E, cfl, (c.cfg.pde == DGX_PDE_NAVIER_STOKES ? c.cfg.mu : 0.0),                   \
             (c.cfg.pde == DGX_PDE_NAVIER_STOKES && c.cfg.viscosity_type == DGX_VISC_SUTHERLAND) ? 1 : 0,          \
             (c.cfg.r_s > 0.0 ? c.cfg.r_s : 1.0), inv_dt
	DGX_PER_ELEM2(k_cfl_dt, 64, )
#undef ARGS
	return hipGetLastError();
}

hipError_t launch_relaxed_update(Ctx& c, double* u, const double* du, int* status)
{
	if (c.nv != c.d + 2) return hipErrorInvalidValue;
#define ARGS u, du, c.ops64, c.E, status, (double*)nullptr
	DGX_PER_ELEM2(k_relaxed_update, 64, )
#undef ARGS
	return hipGetLastError();
}

}  // namespace dgx

// ------------------------------------------------------------------------------- preconditioners
namespace dgx {

// 2-D face-node map: node of local face lf at face position a (faces r-, r+, s-, s+)
template <int D>
__device__ inline int sgs_face_node(int lf, int a, int N)
{
	const int fd = lf >> 1, fix = (lf & 1) ? N - 1 : 0;
	if constexpr (D == 2) return fd == 0 ? fix + N * a : a + N * fix;
	const int i = a % N, j = a / N;   // HEX face position a = i + N j over the two remaining directions
	if (fd == 0) return fix + N * (i + N * j);
	if (fd == 1) return i + N * (fix + N * j);
	return i + N * (j + N * fix);
}

// One element's block operation of the Gauss-Seidel sweeps:
//   r   = rhs_e (or 0) +- sum_faces A_e,n z_n          (faces < 0: minus, > 0: plus, 0: no face term)
//   out = A_ee^-1 r (inverse) or r.
// A_ee^-1 is stored transposed (nb x nb).  The face blocks A_e,n are stored transposed too: compactly on the
// nfv = nv N^(D-1) face-node rows and columns (the launch_offd_blocks layout), so a face costs an nfv x nfv mat-vec on
// the neighbour's trace; FULL (BR2: the neighbour's whole state enters through its lifted gradient, 2-D): nb x nb per
// face.  Elements of one colour share no face, so their updates are independent.  rhs and out are indexed by element,
// or by position in the colour's list (compact vectors).
// TB: the stored blocks' type (FP64, or FP32 with the products and sums in FP64).
// Bound by reading the blocks (QUAD p = 3: 40 KB an element, 84 MB a colour of the 64 x 64 channel, from the Infinity
// Cache): four wavefronts per element, a quarter of the columns each, keep four times the loads in flight of one
// wavefront with whole rows; sizes are compile-time, so index arithmetic takes no divisions and the column loops unroll
// into independent loads (QUAD p = 3, 2048 elements, faces and inverse: 14.7 -> 11.7 us in FP64, 8.1 in FP32).
struct SgsArgs {
	const int* elems;
	const ElemFace* ef;
	const double* rhs;
	const double* z;
	double* out;
	int faces;
	int inverse, rhs_compact, out_compact;
};
template <typename TB, int D, int N, bool FULL>
__global__ void __launch_bounds__(256) k_sgs(SgsArgs a, const TB* __restrict__ invT, const TB* __restrict__ offT)
{
	constexpr int NFACE = 2 * D, NV = D + 2, NF = ipow(N, D - 1), Np = NF * N, NB = Np * NV, NFV = NV * NF;
	constexpr int FB = FULL ? NB : NFV, G = FULL ? 1 : 64 / NFV;   // G column groups of a face product in a wavefront
	constexpr int KG = (NFV + G - 1) / G;
	constexpr int Q4 = (NB + 3) / 4, ROWS = (NB + 63) / 64;
	static_assert(NB <= kMaxInvBlock && G >= 1, "block sizes of the batched inverse");
	__shared__ double sz[NFACE * FB], sp[FULL ? 4 * NB : NFACE * 64], sr[4 * Q4], sq[4][NB];
	const int e = a.elems[blockIdx.x], t = threadIdx.x, l = t & 63, w = t >> 6;
	if (a.faces) {
		for (int it = t; it < NFACE * FB; it += 256) {   // neighbour values (traces in the neighbour's face-node order)
			const int lf = it / FB, c = it - lf * FB;
			const ElemFace f = a.ef[(size_t)e * NFACE + lf];
			double x = 0.0;
			if (f.en >= 0) {
				int src = c;
				if constexpr (!FULL) {
					const int v = c / NF;
					src = v * Np + sgs_face_node<D>(f.packed & 15, c - v * NF, N);
				}
				x = a.z[(size_t)f.en * NB + src];
			}
			sz[it] = x;
		}
		__syncthreads();
		for (int lf = w; lf < NFACE; lf += 4) {
			const TB* C = offT + ((size_t)e * NFACE + lf) * FB * FB;
			if constexpr (FULL) {
				for (int row = l; row < NB; row += 64) {
					double acc = 0.0;
#pragma unroll 16
					for (int c = 0; c < NB; ++c) acc += (double)C[(size_t)c * NB + row] * sz[lf * NB + c];
					sp[lf * NB + row] = acc;
				}
			} else if (l < G * NFV) {
				const int g = l / NFV, row = l - g * NFV;
				double acc = 0.0;
#pragma unroll
				for (int k = 0; k < KG; ++k)
					if (g + k * G < NFV) acc += (double)C[(size_t)(g + k * G) * NFV + row] * sz[lf * NFV + g + k * G];
				sp[lf * 64 + l] = acc;
			}
		}
		__syncthreads();
	}
	const double sgn = a.faces < 0 ? -1.0 : 1.0;
	for (int i = t; i < 4 * Q4; i += 256) {
		double r = (a.rhs && i < NB) ? a.rhs[(size_t)(a.rhs_compact ? (int)blockIdx.x : e) * NB + i] : 0.0;
		if (a.faces && i < NB) {
			double s = 0.0;
			if constexpr (FULL) {
				s = (sp[i] + sp[NB + i]) + (sp[2 * NB + i] + sp[3 * NB + i]);
			} else {
				const int v = i / Np, node = i - v * Np;
				const int cc[3] = { node % N, (node / N) % N, D == 3 ? node / (N * N) : 0 };
#pragma unroll
				for (int lf = 0; lf < NFACE; ++lf) {
					const int fd = lf >> 1;
					if (cc[fd] == ((lf & 1) ? N - 1 : 0)) {
						const int c0 = fd == 0 ? cc[1] : cc[0], c1 = fd == 2 ? cc[1] : cc[2];
						const double* q = sp + lf * 64 + v * NF + (D == 2 ? c0 : c0 + N * c1);
#pragma unroll
						for (int g = 0; g < G; ++g) s += q[g * NFV];
					}
				}
			}
			r += sgn * s;
		}
		if (a.inverse) sr[i] = r;
		else if (i < NB) a.out[(size_t)(a.out_compact ? (int)blockIdx.x : e) * NB + i] = r;
	}
	if (!a.inverse) return;
	__syncthreads();
	const TB* M = invT + (size_t)e * NB * NB;
#pragma unroll
	for (int rr = 0; rr < ROWS; ++rr) {   // quarter w of the columns of A_ee^-1 r (past the last: its values, times zero)
		const int row = l + 64 * rr;
		if (row < NB) {
			double acc = 0.0;
#pragma unroll
			for (int k = 0; k < Q4; ++k) acc += (double)M[(size_t)min(w * Q4 + k, NB - 1) * NB + row] * sr[w * Q4 + k];
			sq[w][row] = acc;
		}
	}
	__syncthreads();
	for (int i = t; i < NB; i += 256)
		a.out[(size_t)(a.out_compact ? (int)blockIdx.x : e) * NB + i] = (sq[0][i] + sq[1][i]) + (sq[2][i] + sq[3][i]);
}

// Position of node (i0, i1) of an N x N element among its 4 N - 4 face nodes (node order, interior nodes left out)
__device__ inline int face_pos(int i0, int i1, int N)
{
	if (i1 == 0) return i0;
	if (i1 == N - 1) return N + 2 * (N - 2) + i0;
	return N + 2 * (i1 - 1) + (i0 == 0 ? 0 : 1);
}
// and the node at a position
__device__ inline int face_node_at(int pos, int N)
{
	if (pos < N) return pos;
	const int q = pos - N;
	if (q < 2 * (N - 2)) return (q & 1 ? N - 1 : 0) + N * (1 + q / 2);
	return (q - 2 * (N - 2)) + N * (N - 1);
}

// The reduced operator's blocks on face nodes (QUAD, compact face blocks), R = nv (4 N - 4) rows, stored transposed:
//   colour 2:  B = A_22^-1 on face-node rows and columns            [col R][row R]
//   colour 1:  W = -A_11^-1 A_12 on face-node rows, one column per
//              neighbour-trace value                                [col 4 nfv][row R]
__global__ void __launch_bounds__(256) k_pack_reduced(const int* __restrict__ elems, const double* __restrict__ invT,
                                                      const double* __restrict__ offT, double* out, int N, int nv, int first)
{
	const int Np = N * N, nb = nv * Np, nfv = nv * N, nfn = 4 * N - 4, R = nv * nfn;
	const int e = elems[blockIdx.x];
	const double* M = invT + (size_t)e * nb * nb;
	if (!first) {
		double* B = out + (size_t)blockIdx.x * R * R;
		for (int it = threadIdx.x; it < R * R; it += 256) {
			const int c = it / R, r = it - c * R;
			const int gc = (c / nfn) * Np + face_node_at(c % nfn, N), gr = (r / nfn) * Np + face_node_at(r % nfn, N);
			B[it] = M[(size_t)gc * nb + gr];
		}
		return;
	}
	double* W = out + (size_t)blockIdx.x * 4 * nfv * R;
	for (int it = threadIdx.x; it < 4 * nfv * R; it += 256) {
		const int c = it / R, r = it - c * R, lf = c / nfv, cc = c - lf * nfv;
		const int gr = (r / nfn) * Np + face_node_at(r % nfn, N);
		const double* C = offT + (((size_t)e * 4 + lf) * nfv + cc) * nfv;
		double acc = 0.0;
		for (int b = 0; b < nfv; ++b) {
			const int v = b / N;
			acc -= M[(size_t)(v * Np + sgs_face_node<2>(lf, b - v * N, N)) * nb + gr] * C[b];
		}
		W[it] = acc;
	}
}

// One block product of the reduced operator per workgroup, on face-node vectors (R values an element):
//   GATHER = false: zf[e] = B v_pos  (v compact);   GATHER = true: zf[e] = W (neighbour traces of zf).
// Bound by reading the blocks: QUAD p = 3, 18 and 25 KB an element against the 32 and 40 KB of the whole inverse and
// the face blocks; two rows a lane (16-byte loads), as many column groups as 256 lanes hold, all loads of a lane in
// flight before the vector's own chain of loads (list, face record, neighbour values) begins.
template <int N, bool GATHER>
__global__ void __launch_bounds__(256) k_reduced_gemv(const int* __restrict__ elems, const ElemFace* __restrict__ ef,
                                                      const double* __restrict__ blocks, const double* v, double* zf)
{
	constexpr int NV = 4, NFV = NV * N, NFN = 4 * N - 4, R = NV * NFN, C = GATHER ? 4 * NFV : R;
	constexpr int L = R / 2, G = 256 / L, KC = (C + G - 1) / G;
	__shared__ double sx[KC * G], sp[G * R];
	const int t = threadIdx.x, g = t / L, row = 2 * (t - g * L);
	const int e = elems[blockIdx.x];
	const double* M = blocks + (size_t)blockIdx.x * C * R + row;
	double2 m[KC];   // (columns past the last: its values again, times zero)
#pragma unroll
	for (int k = 0; k < KC; ++k) m[k] = *reinterpret_cast<const double2*>(M + (size_t)min(g + k * G, C - 1) * R);
	for (int c = t; c < KC * G; c += 256) {
		double x = 0.0;
		if (c < C) {
			if constexpr (GATHER) {
				const int lf = c / NFV, cc = c - lf * NFV, w = cc / N;
				const ElemFace f = ef[(size_t)e * 4 + lf];
				if (f.en >= 0) {
					const int node = sgs_face_node<2>(f.packed & 15, cc - w * N, N);
					x = zf[(size_t)f.en * R + w * NFN + face_pos(node % N, node / N, N)];
				}
			} else {
				x = v[(size_t)blockIdx.x * R + c];
			}
		}
		sx[c] = x;
	}
	__syncthreads();
	if (g < G) {
		double a0 = 0.0, a1 = 0.0;
#pragma unroll
		for (int k = 0; k < KC; ++k) {
			const double x = sx[g + k * G];
			a0 += m[k].x * x;
			a1 += m[k].y * x;
		}
		sp[g * R + row] = a0;
		sp[g * R + row + 1] = a1;
	}
	__syncthreads();
	if (t < R) {
		double s = 0.0;
#pragma unroll
		for (int k = 0; k < G; ++k) s += sp[k * R + t];
		zf[(size_t)e * R + t] = s;
	}
}
// w_pos = v_pos + A_21 (traces of zf), face-node rows: one wavefront per local face
template <int N>
__global__ void __launch_bounds__(256) k_reduced_faces(const int* __restrict__ elems, const ElemFace* __restrict__ ef,
                                                       const double* __restrict__ offT, const double* __restrict__ v,
                                                       const double* __restrict__ zf, double* w)
{
	constexpr int NV = 4, NFV = NV * N, NFN = 4 * N - 4, R = NV * NFN, G = 64 / NFV, KC = (NFV + G - 1) / G;
	__shared__ double sz[4][KC * G], sp[4][64];
	const int t = threadIdx.x, l = t & 63, lf = t >> 6, g = l / NFV, row = l - g * NFV;
	const int e = elems[blockIdx.x];
	const double* C = offT + ((size_t)e * 4 + lf) * NFV * NFV + row;
	double m[KC];
#pragma unroll
	for (int k = 0; k < KC; ++k) m[k] = C[(size_t)min(g + k * G, NFV - 1) * NFV];
	const ElemFace f = ef[(size_t)e * 4 + lf];
	if (l < KC * G) {
		double x = 0.0;
		if (l < NFV && f.en >= 0) {
			const int vv = l / N, node = sgs_face_node<2>(f.packed & 15, l - vv * N, N);
			x = zf[(size_t)f.en * R + vv * NFN + face_pos(node % N, node / N, N)];
		}
		sz[lf][l] = x;
	}
	__syncthreads();
	if (g < G) {
		double acc = 0.0;
#pragma unroll
		for (int k = 0; k < KC; ++k) acc += m[k] * sz[lf][g + k * G];
		sp[lf][l] = acc;
	}
	__syncthreads();
	if (t < R) {
		const int vv = t / NFN, node = face_node_at(t - vv * NFN, N), i0 = node % N, i1 = node / N;
		double s = v[(size_t)blockIdx.x * R + t];
#pragma unroll
		for (int k = 0; k < G; ++k) {
			if (i0 == 0) s += sp[0][k * NFV + vv * N + i1];
			if (i0 == N - 1) s += sp[1][k * NFV + vv * N + i1];
			if (i1 == 0) s += sp[2][k * NFV + vv * N + i0];
			if (i1 == N - 1) s += sp[3][k * NFV + vv * N + i0];
		}
		w[(size_t)blockIdx.x * R + t] = s;
	}
}
// compact vectors of colour 2: whole elements (nb values) <-> face-node rows (R values, the others zero)
__global__ void __launch_bounds__(256) k_face_rows(const double* __restrict__ src, double* dst, int count, int N, int nv,
                                                   int expand)
{
	const int Np = N * N, nb = nv * Np, nfn = 4 * N - 4, R = nv * nfn;
	const size_t n = (size_t)count * (expand ? nb : R);
	for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
		if (expand) {
			const size_t p = i / nb;
			const int k = (int)(i - p * nb), v = k / Np, node = k - v * Np, i0 = node % N, i1 = node / N;
			const bool face = i0 == 0 || i0 == N - 1 || i1 == 0 || i1 == N - 1;
			dst[i] = face ? src[p * R + v * nfn + face_pos(i0, i1, N)] : 0.0;
		} else {
			const size_t p = i / R;
			const int k = (int)(i - p * R), v = k / nfn;
			dst[i] = src[p * nb + v * Np + face_node_at(k - v * nfn, N)];
		}
	}
}

struct PrecondIdentity : Precond {
	hipError_t setup(Ctx&, const double*, const double*) override { return hipSuccess; }
	hipError_t apply(Ctx& c, const double* v, double* z) override
	{
		return hipMemcpyAsync(z, v, sizeof(double) * (size_t)c.E * c.Np * c.nv, hipMemcpyDeviceToDevice, c.stream);
	}
};

// exact inverse (or LU) of the element diagonal blocks of (dR/du - M/dt): the block-Jacobi baseline
hipError_t launch_features(Ctx& c, const double* u, const double* inv_dt, float* feat, int nf, float* sigma);

struct PrecondBlockJacobi : Precond {
	double* blocks = nullptr;
	int* piv = nullptr;
	// optional training-set capture
	double* cap_blocks = nullptr;
	float* cap_feat = nullptr;
	float* cap_sigma = nullptr;
	long long cap_capacity = 0, cap_count = 0;
	~PrecondBlockJacobi() override
	{
		if (blocks) (void)hipFree(blocks);
		if (piv) (void)hipFree(piv);
	}
	hipError_t setup(Ctx& c, const double* u, const double* inv_dt) override
	{
		const int nb = c.Np * c.nv;
		if (!blocks) {
			DGX_HIP_CHECK(hipMalloc(&blocks, sizeof(double) * (size_t)c.E * nb * nb));
			DGX_HIP_CHECK(hipMalloc(&piv, sizeof(int) * (size_t)c.E * nb));
		}
		DGX_HIP_CHECK(launch_diag_blocks(c, u, inv_dt, blocks));
		if (cap_blocks && cap_feat && cap_sigma && cap_count + c.E <= cap_capacity) {
			const int nf = (nb + c.Np + 1 + 15) / 16 * 16;
			DGX_HIP_CHECK(hipMemcpyAsync(cap_blocks + (size_t)cap_count * nb * nb, blocks,
			                             sizeof(double) * (size_t)c.E * nb * nb, hipMemcpyDeviceToDevice, c.stream));
			DGX_HIP_CHECK(launch_features(c, u, inv_dt, cap_feat + (size_t)cap_count * nf, nf,
			                              cap_sigma + (size_t)cap_count));
			cap_count += c.E;
		}
		// blocks up to 142 x 142: explicit inverse (one coalesced mat-vec per application); larger: LU
		if (nb <= kMaxInvBlock) return launch_block_inverse(c.stream, blocks, c.E, nb, nullptr);
		return launch_block_lu(c.stream, blocks, piv, c.E, nb);
	}
	hipError_t apply(Ctx& c, const double* v, double* z) override
	{
		const int nb = c.Np * c.nv;
		if (nb <= kMaxInvBlock) return launch_block_inv_apply(c.stream, blocks, v, z, c.E, nb);
		DGX_HIP_CHECK(hipMemcpyAsync(z, v, sizeof(double) * (size_t)c.E * nb, hipMemcpyDeviceToDevice, c.stream));
		return launch_block_lu_solve(c.stream, blocks, piv, z, c.E, nb);
	}
};

// Multicolour block symmetric Gauss-Seidel on the block-sparse Jacobian (diagonal blocks with the -M/dt
// term, exact inverses; compact face blocks from the dual-number MODE_OFFD columns): forward over the
// colours, then backward, from z = 0.  A fixed linear operator, so plain right-preconditioned GMRES applies.
struct PrecondBlockSGS : Precond {
	PrecondBlockJacobi diag;   // assembles and inverts A_ee - M_e/dt
	double* offT = nullptr;    // E * 4 * nfv^2 compact transposed face blocks (Navier-Stokes: E * 4 * nb^2, full)
	bool fp32 = false;         // sweep over FP32 copies of the inverse and face blocks
	float* inv32 = nullptr;
	float* off32 = nullptr;
	// reduced operator on face nodes (QUAD, compact face blocks): see k_pack_reduced
	double* redB = nullptr;
	double* redW = nullptr;
	double* zf = nullptr;      // E x R face-node values
	double* tmp = nullptr;     // colour 2, whole elements
	explicit PrecondBlockSGS(bool use_fp32 = false) : fp32(use_fp32) {}
	~PrecondBlockSGS() override
	{
		for (double* p : { redB, redW, zf, tmp })
			if (p) (void)hipFree(p);
		if (offT) (void)hipFree(offT);
		if (inv32) (void)hipFree(inv32);
		if (off32) (void)hipFree(off32);
	}
	static bool full(const Ctx& c) { return c.cfg.pde == DGX_PDE_NAVIER_STOKES; }
	hipError_t setup(Ctx& c, const double* u, const double* inv_dt) override
	{
		const int nb = c.Np * c.nv, nf = 2 * c.d, nfv = c.nv * (c.d == 2 ? c.N : c.N * c.N);
		if ((c.d != 2 && c.d != 3) || (full(c) && c.d != 2) || nb > kMaxInvBlock || nf * nfv > kMaxSgsFace)
			return hipErrorInvalidValue;
		DGX_HIP_CHECK(diag.setup(c, u, inv_dt));
		// the face blocks: compact on the face nodes (Euler, advection), full for BR2
		const int fb = full(c) ? nb : nfv;
		if (!offT) DGX_HIP_CHECK(hipMalloc(&offT, sizeof(double) * (size_t)c.E * nf * fb * fb));
		if (full(c))
			for (int col = 0; col < nb; ++col) DGX_HIP_CHECK(launch_ns_offd_col(c, u, offT, col, true));
		else
			DGX_HIP_CHECK(launch_offd_blocks(c, u, offT));
		if (faces_only(c)) {
			const int R = rows(c);
			const size_t n1 = count(c, 0), n2 = count(c, 1);
			if (!redB) DGX_HIP_CHECK(hipMalloc(&redB, sizeof(double) * std::max<size_t>(n2, 1) * R * R));
			if (!redW) DGX_HIP_CHECK(hipMalloc(&redW, sizeof(double) * std::max<size_t>(n1, 1) * 4 * nfv * R));
			if (!zf) DGX_HIP_CHECK(hipMalloc(&zf, sizeof(double) * (size_t)c.E * R));
			if (!tmp) DGX_HIP_CHECK(hipMalloc(&tmp, sizeof(double) * std::max<size_t>(n2, 1) * nb));
			if (n1)
				hipLaunchKernelGGL(k_pack_reduced, dim3((unsigned)n1), dim3(256), 0, c.stream, c.color_elems + c.color_off[0],
				                   diag.blocks, offT, redW, c.N, c.nv, 1);
			if (n2)
				hipLaunchKernelGGL(k_pack_reduced, dim3((unsigned)n2), dim3(256), 0, c.stream, c.color_elems + c.color_off[1],
				                   diag.blocks, offT, redB, c.N, c.nv, 0);
			DGX_HIP_CHECK(hipGetLastError());
		}
		if (!fp32) return hipSuccess;
		const size_t ni = (size_t)c.E * nb * nb, no = (size_t)c.E * nf * fb * fb;
		if (!inv32) DGX_HIP_CHECK(hipMalloc(&inv32, sizeof(float) * ni));
		if (!off32) DGX_HIP_CHECK(hipMalloc(&off32, sizeof(float) * no));
		DGX_HIP_CHECK(launch_convert(diag.blocks, inv32, ni, c.stream));
		return launch_convert(offT, off32, no, c.stream);
	}
	// one block operation (see k_sgs) on every element of colour k
	hipError_t run(Ctx& c, int k, const double* rhs, bool rhs_compact, int faces, bool inverse, const double* z, double* out,
	               bool out_compact)
	{
		const int n0 = c.color_off[k], cnt = c.color_off[k + 1] - n0;
		if (cnt == 0) return hipSuccess;
		SgsArgs a{ c.color_elems + n0, c.elem_faces, rhs, z, out, faces, inverse, rhs_compact, out_compact };
		if (c.nv != c.d + 2) return hipErrorInvalidValue;
#define DGX_SGS(DD, NN, FULL)                                                                                            \
		if (c.d == DD && c.N == NN && full(c) == FULL) {                                                                 \
			if (fp32) hipLaunchKernelGGL((k_sgs<float, DD, NN, FULL>), dim3(cnt), dim3(256), 0, c.stream, a, inv32, off32); \
			else hipLaunchKernelGGL((k_sgs<double, DD, NN, FULL>), dim3(cnt), dim3(256), 0, c.stream, a, diag.blocks, offT); \
			return hipGetLastError();                                                                                  \
		}
		DGX_SGS(2, 2, false) DGX_SGS(2, 3, false) DGX_SGS(2, 4, false) DGX_SGS(2, 5, false)
		DGX_SGS(2, 2, true) DGX_SGS(2, 3, true) DGX_SGS(2, 4, true) DGX_SGS(2, 5, true)
		DGX_SGS(3, 2, false) DGX_SGS(3, 3, false)
#undef DGX_SGS
		return hipErrorInvalidValue;
	}
	hipError_t apply(Ctx& c, const double* v, double* z) override
	{
		const size_t n = (size_t)c.E * c.Np * c.nv;
		const int nc = (int)c.color_off.size() - 1;
		// with two colours every neighbour of the first still holds zero: no face terms, nothing to clear (not where an
		// element is its own neighbour: the sweeps then read z within a colour too)
		const bool two = nc == 2 && !c.self_neighbour;
		if (!two)
			DGX_HIP_CHECK(launch_fill_u64(c.stream, reinterpret_cast<unsigned long long*>(z), (int)n, 0ull));
		for (int k = 0; k < nc; ++k) DGX_HIP_CHECK(run(c, k, v, false, (two && k == 0) ? 0 : -1, true, z, z, false));
		// backward: the last colour's inputs have not changed since its forward update, so it is not redone
		for (int k = nc - 2; k >= 0; --k) DGX_HIP_CHECK(run(c, k, v, false, -1, true, z, z, false));
		return hipSuccess;
	}
	// Two colours (1, 2) without couplings inside a colour, FP64 blocks.  The backward half-sweep leaves row 1 of A z = v exactly solved, so with
	// M = the sweeps' operator, A M^-1 is the identity on colour 1 and maps a vector that vanishes there to
	//   v_2 + A_21 z_1,   z_1 = -A_11^-1 A_12 z_2,   z_2 = A_22^-1 v_2,
	// which vanishes on colour 1 again.  Once the right-hand side is cleared on colour 1 (one block solve), the whole
	// Krylov space therefore lives on colour 2: vectors of half the length, two block sweeps instead of three, and the
	// face blocks in place of the matrix-free product.  The residual norm is the full system's.
	// With compact face blocks A_21 reaches only the face nodes of colour 2, so the same holds there: a start that
	// solves colour 2, then colour 1, leaves a residual on those nodes alone, and only the face-node rows of z_1 and
	// z_2 are needed (k_pack_reduced).  QUAD p = 3: 105 MB of blocks an iteration on the 64 x 64 channel instead of the
	// three sweeps' 235 MB and the product's traffic.
	bool reducible(const Ctx& c) const override { return !fp32 && (int)c.color_off.size() == 3 && !c.self_neighbour; }
	static size_t count(const Ctx& c, int k) { return (size_t)(c.color_off[k + 1] - c.color_off[k]); }
	static int rows(const Ctx& c) { return c.nv * (4 * c.N - 4); }
	// the packed kernels' sizes: nv = 4, N <= 5 (the largest order that the batched inverse takes)
	bool faces_only(const Ctx& c) const { return reducible(c) && c.d == 2 && !full(c) && c.nv == 4 && c.N <= 5; }
	size_t reduced_size(const Ctx& c) const override { return count(c, 1) * (faces_only(c) ? rows(c) : c.Np * c.nv); }
	hipError_t face_rows(Ctx& c, const double* src, double* dst, bool expand)
	{
		const size_t n = count(c, 1) * (expand ? c.Np * c.nv : rows(c));
		if (n == 0) return hipSuccess;
		hipLaunchKernelGGL(k_face_rows, dim3(grid_for(n)), dim3(256), 0, c.stream, src, dst, (int)count(c, 1), c.N, c.nv,
		                   expand ? 1 : 0);
		return hipGetLastError();
	}
	hipError_t reduced_start(Ctx& c, const double* r, double* z, double* v2) override
	{
		const size_t n = (size_t)c.E * c.Np * c.nv;
		DGX_HIP_CHECK(launch_fill_u64(c.stream, reinterpret_cast<unsigned long long*>(z), (int)n, 0ull));
		if (!faces_only(c)) {   // z = (A_11^-1 r_1, 0), v_2 = r_2 - A_21 z_1
			DGX_HIP_CHECK(run(c, 0, r, false, 0, true, z, z, false));
			return run(c, 1, r, false, -1, false, z, v2, true);
		}
		// z_2 = A_22^-1 r_2, z_1 = A_11^-1 (r_1 - A_12 z_2), v_2 = r_2 - A_22 z_2 - A_21 z_1 = -A_21 z_1
		DGX_HIP_CHECK(run(c, 1, r, false, 0, true, z, z, false));
		DGX_HIP_CHECK(run(c, 0, r, false, -1, true, z, z, false));
		DGX_HIP_CHECK(run(c, 1, nullptr, false, -1, false, z, tmp, true));
		return face_rows(c, tmp, v2, false);
	}
	hipError_t reduced_solution(Ctx& c, const double* v2, double* z) override
	{
		if (faces_only(c)) {
			DGX_HIP_CHECK(face_rows(c, v2, tmp, true));
			v2 = tmp;
		}
		DGX_HIP_CHECK(run(c, 1, v2, true, 0, true, z, z, false));
		return run(c, 0, nullptr, false, -1, true, z, z, false);
	}
	hipError_t reduced_apply(Ctx& c, const double* v2, double* z, double* w2) override
	{
		if (!faces_only(c)) {
			DGX_HIP_CHECK(reduced_solution(c, v2, z));
			return run(c, 1, v2, true, 1, false, z, w2, true);
		}
		const unsigned n1 = (unsigned)count(c, 0), n2 = (unsigned)count(c, 1);
		const int *e1 = c.color_elems + c.color_off[0], *e2 = c.color_elems + c.color_off[1];
		if (c.nv != 4) return hipErrorInvalidValue;
#define DGX_REDUCED(NN)                                                                                                  \
		case NN:                                                                                                        \
			if (n2)                                                                                                     \
				hipLaunchKernelGGL((k_reduced_gemv<NN, false>), dim3(n2), dim3(256), 0, c.stream, e2, c.elem_faces, redB, v2, zf); \
			if (n1)                                                                                                     \
				hipLaunchKernelGGL((k_reduced_gemv<NN, true>), dim3(n1), dim3(256), 0, c.stream, e1, c.elem_faces, redW, v2, zf);  \
			if (n2)                                                                                                     \
				hipLaunchKernelGGL(k_reduced_faces<NN>, dim3(n2), dim3(256), 0, c.stream, e2, c.elem_faces, offT, v2, zf, w2);     \
			break;
		switch (c.N) {
		DGX_REDUCED(2) DGX_REDUCED(3) DGX_REDUCED(4) DGX_REDUCED(5)
		default: return hipErrorInvalidValue;
		}
#undef DGX_REDUCED
		return hipGetLastError();
	}
};


// ------------------------------------------------------------------------------- GMRES
constexpr int kMaxRestart = 200;

// The last kernel of an Arnoldi step.  Every workgroup: the next basis vector w / |w| (FP64 vcur, the preconditioner's
// input, and its FP32 copy).  Workgroup 0 also forms column j: H(0..j, j) = h1 + h2 (the two Gram-Schmidt passes),
// H(j+1, j) = |w|, the previous Givens rotations applied to the new column, the new rotation, and the residual
// estimate.  st[0] = |g(j+1)|, st[1] = first column count at which |g| <= tol (or -1), st[2] = |w|; host[0..2] is a
// copy in pinned memory.
// The rotation chain is sequential: the column and the rotations are staged in LDS by all lanes first, so the chain
// runs on LDS values instead of waiting on global loads at every step.
struct ArnoldiArgs {
	double *H, *cs, *sn, *g, *st, *host;
	const double *p1, *p2, *pn;
	int j, m, nc;
	double tol;
};
__global__ void __launch_bounds__(kGsLanes) k_arnoldi_step(ArnoldiArgs a, const double* __restrict__ w, float* v32,
                                                           double* vcur, size_t n, size_t chunk)
{
	__shared__ double sb[kMaxRows], so[kMaxRows], sc[kMaxRestart], ss[kMaxRestart], snrm;
	const int t = threadIdx.x, lane = t & 63, wave = t >> 6, j = a.j;
	if (wave == 0) {
		const double s = row_sum(a.pn, 0, a.nc, lane);
		if (lane == 0) snrm = s;
	}
	if (blockIdx.x == 0) {
		for (int i = wave; i <= j; i += kGsLanes / 64) {
			const double h = row_sum(a.p1, i, a.nc, lane) + row_sum(a.p2, i, a.nc, lane);
			if (lane == 0) sb[i] = h;
		}
		for (int i = t; i < j; i += kGsLanes) {
			sc[i] = a.cs[i];
			ss[i] = a.sn[i];
		}
	}
	__syncthreads();
	const double nv = snrm, inv = nv > 0.0 ? 1.0 / sqrt(nv) : 0.0;
	const size_t lo = (size_t)blockIdx.x * chunk, hi = lo + chunk < n ? lo + chunk : n;
	for (size_t i = lo + t; i < hi; i += kGsLanes) {
		const double v = inv * w[i];
		vcur[i] = v;
		v32[i] = (float)v;
	}
	if (blockIdx.x != 0) return;
	if (t == 0) {
		const double hn = sqrt(nv);
		double x = sb[0];
#pragma unroll 8
		for (int i = 0; i < j; ++i) {
			const double b = sb[i + 1], c = sc[i], d = ss[i];
			so[i] = c * x + d * b;
			x = -d * x + c * b;
		}
		const double b = hn;
		const double r = sqrt(x * x + b * b);
		const double c = r > 0 ? x / r : 1.0, sj = r > 0 ? b / r : 0.0;
		a.cs[j] = c;
		a.sn[j] = sj;
		so[j] = r;
		so[j + 1] = 0.0;
		const double gj = a.g[j];
		a.g[j + 1] = -sj * gj;
		a.g[j] = c * gj;
		const double est = fabs(sj * gj);
		double first = a.st[1];
		if (first < 0.0 && (est <= a.tol || hn == 0.0)) first = (double)(j + 1);
		a.st[0] = est;
		a.st[1] = first;
		a.st[2] = hn;
		a.host[0] = est;
		a.host[1] = first;
		a.host[2] = hn;
	}
	__syncthreads();
	double* col = a.H + (size_t)j * (a.m + 1);   // column j, rows 0..m
	for (int i = t; i <= j + 1; i += kGsLanes) col[i] = so[i];
}

// g = (beta, 0, ...), st = (beta, -1, 1) at the start of a restart cycle
__global__ void k_arnoldi_start(double* g, int m, double beta, double* st)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i <= m) g[i] = (i == 0) ? beta : 0.0;
	if (i == 0) { st[0] = beta; st[1] = -1.0; st[2] = 1.0; }
}

struct Gmres {
	int m = 60;
	static constexpr int kCheck = 4;   // Arnoldi steps between host convergence checks
	// Krylov basis (m+1) x n in FP32: the Gram-Schmidt passes read it three times per iteration, and FP32 halves
	// those bytes; every product and sum stays in FP64, and so do w, x and the newest basis vector vcur (the
	// preconditioner's input).  The Arnoldi relation then holds to FP32 rounding (~1e-7 relative), far below the
	// inner tolerance; the outer Newton residual decides convergence in FP64.
	float* V = nullptr;
	double* vcur = nullptr;
	double* w = nullptr;
	double* z = nullptr;
	double* x = nullptr;
	size_t n = 0;
	Blas blas;
	std::vector<double> y;
	double* dls = nullptr;    // device: H ((m+1) x m, column-major) | cs (m) | sn (m) | g (m+1) | st (3)
	double* host = nullptr;   // pinned: two slots of (residual estimate, converged column count, |w|)
	hipEvent_t seen[2] = { nullptr, nullptr };
	hipError_t init(Ctx& c, int restart)
	{
		m = restart;
		n = (size_t)c.E * c.Np * c.nv;
		DGX_HIP_CHECK(hipMalloc(&V, sizeof(float) * (size_t)(m + 1) * n));
		DGX_HIP_CHECK(hipMalloc(&vcur, sizeof(double) * n));
		DGX_HIP_CHECK(hipMalloc(&w, sizeof(double) * n));
		DGX_HIP_CHECK(hipMalloc(&z, sizeof(double) * n));
		DGX_HIP_CHECK(hipMalloc(&x, sizeof(double) * n));
		y.assign(m, 0.0);
		DGX_HIP_CHECK(hipMalloc(&dls, sizeof(double) * ls_size()));
		DGX_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&host), sizeof(double) * 6, hipHostMallocDefault));
		for (hipEvent_t& ev : seen) DGX_HIP_CHECK(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
		return blas.init(c.stream, m + 1);
	}
	void release()
	{
		if (V) (void)hipFree(V);
		V = nullptr;
		for (double* p : { vcur, w, z, x, dls })
			if (p) (void)hipFree(p);
		vcur = w = z = x = dls = nullptr;
		if (host) (void)hipHostFree(host);
		host = nullptr;
		for (hipEvent_t& ev : seen) {
			if (ev) (void)hipEventDestroy(ev);
			ev = nullptr;
		}
		blas.release();
	}
	size_t ls_size() const { return (size_t)(m + 1) * m + 2 * (size_t)m + (m + 1) + 3; }
	bool jvp32 = false;   // the operator in FP32 dual numbers
	// w = A v with A = dR/du(u) - M/dt
	hipError_t op(Ctx& c, const double* u, const double* inv_dt, const double* v, double* out)
	{
		// dual-number J v with the -M/dt term added in the same kernel (at the GL nodes, before Ibar^T)
		return jvp32 ? launch_jvp32(c, u, v, out, inv_dt) : launch_jvp(c, u, v, out, inv_dt);
	}
	// one Arnoldi step: w orthogonalised against the j + 1 basis vectors (classical Gram-Schmidt, twice), the next
	// basis vector and column j of the least-squares problem; nk values per vector
	hipError_t orthogonalise(hipStream_t st, int j, size_t nk, double tol, double* slot)
	{
		DGX_HIP_CHECK((blas.gs<false, true>(V, nk, j + 1, w, nk, nullptr, blas.partial)));
		DGX_HIP_CHECK((blas.gs<true, true>(V, nk, j + 1, w, nk, blas.partial, blas.partial2)));
		DGX_HIP_CHECK((blas.gs<true, false>(V, nk, j + 1, w, nk, blas.partial2, blas.partialn)));
		const Chunks ch = chunks_of(nk);
		ArnoldiArgs a{};
		a.H = dls;
		a.cs = a.H + (size_t)(m + 1) * m;
		a.sn = a.cs + m;
		a.g = a.sn + m;
		a.st = a.g + (m + 1);
		a.host = slot;
		a.p1 = blas.partial;
		a.p2 = blas.partial2;
		a.pn = blas.partialn;
		a.j = j;
		a.m = m;
		a.nc = ch.count;
		a.tol = tol;
		hipLaunchKernelGGL(k_arnoldi_step, dim3(ch.count), dim3(kGsLanes), 0, st, a, w, V + (size_t)(j + 1) * nk, vcur, nk,
		                   ch.size);
		return hipGetLastError();
	}
	// right-preconditioned restarted GMRES on A x = b, x0 = 0; returns iterations, sets converged.
	// The Hessenberg column and its Givens rotation are formed on the device.  Every kCheck steps the host looks at the
	// residual estimate of the check before, while the device works on the steps it has just queued (steps past
	// convergence only enlarge the Krylov space; the solution takes the first columns up to it), and it brings H and g
	// back once per restart cycle for the triangular solve.
	// With a reducible preconditioner the basis is built on the reduced vectors (see Precond).
	hipError_t solve(Ctx& c, const double* u, const double* inv_dt, const double* b, Precond& P, double rtol,
	                 int max_it, int* iters, bool* converged)
	{
		DGX_HIP_CHECK(blas.axpby(0.0, b, 0.0, x, n));
		double bnorm;
		DGX_HIP_CHECK(blas.axpby(1.0, b, 0.0, w, n));
		DGX_HIP_CHECK(blas.norm(w, n, &bnorm));
		*iters = 0;
		*converged = (bnorm == 0.0);
		if (*converged) return hipSuccess;
		const double tol = rtol * bnorm;
		double* dg = dls + (size_t)(m + 1) * m + 2 * (size_t)m;
		double* dst = dg + (m + 1);
		std::vector<double> hls(ls_size());
		const bool red = P.reducible(c);
		const size_t nk = red ? P.reduced_size(c) : n;
		int total = 0;
		while (total < max_it) {
			// w = r = b - A x  (x = 0 on the first cycle)
			if (total > 0) {
				DGX_HIP_CHECK(op(c, u, inv_dt, x, w));
				DGX_HIP_CHECK(blas.axpby(1.0, b, -1.0, w, n));
			}
			if (red) {
				DGX_HIP_CHECK(P.reduced_start(c, w, z, vcur));
				DGX_HIP_CHECK(blas.axpby(1.0, z, 1.0, x, n));
			} else {
				DGX_HIP_CHECK(blas.axpby(1.0, w, 0.0, vcur, n));
			}
			double beta;
			DGX_HIP_CHECK(blas.norm(vcur, nk, &beta));
			if (beta <= tol) { *converged = true; break; }
			DGX_HIP_CHECK(blas.axpby(1.0 / beta, vcur, 0.0, vcur, nk));
			DGX_HIP_CHECK(launch_convert(vcur, V, nk, c.stream));
			hipLaunchKernelGGL(k_arnoldi_start, dim3((m + 64) / 64), dim3(64), 0, c.stream, dg, m, beta, dst);
			DGX_HIP_CHECK(hipGetLastError());
			int j = 0, jconv = -1, check = 0, pending = -1, pending_total = 0;
			for (; j < m && total < max_it; ++j, ++total) {
				if (red) {
					DGX_HIP_CHECK(P.reduced_apply(c, vcur, z, w));
				} else {
					DGX_HIP_CHECK(P.apply(c, vcur, z));   // vcur = v_j in FP64
					DGX_HIP_CHECK(op(c, u, inv_dt, z, w));
				}
				DGX_HIP_CHECK(orthogonalise(c.stream, j, nk, tol, host + 3 * (check & 1)));
				const bool last = j + 1 == m || total + 1 >= max_it;
				if ((j + 1) % kCheck == 0 || last) {
					DGX_HIP_CHECK(hipEventRecord(seen[check & 1], c.stream));
					if (pending >= 0) {
						DGX_HIP_CHECK(hipEventSynchronize(seen[pending]));
						if (host[3 * pending + 1] >= 0.0) {
							jconv = (int)host[3 * pending + 1];
							total = pending_total;
							*converged = true;
							break;
						}
					}
					pending = check & 1;
					pending_total = total + 1;
					++check;
				}
			}
			if (!*converged && pending >= 0) {
				DGX_HIP_CHECK(hipEventSynchronize(seen[pending]));
				if (host[3 * pending + 1] >= 0.0) {
					jconv = (int)host[3 * pending + 1];
					*converged = true;
				}
			}
			// y = H^-1 g over the first jj columns, x += P^-1 (V y)
			const int jj = (jconv > 0) ? jconv : j;
			DGX_HIP_CHECK(hipMemcpyAsync(hls.data(), dls, sizeof(double) * hls.size(), hipMemcpyDeviceToHost, c.stream));
			DGX_HIP_CHECK(hipStreamSynchronize(c.stream));
			const double* Hh = hls.data();
			const double* gh = Hh + (size_t)(m + 1) * m + 2 * (size_t)m;
			for (int i = jj - 1; i >= 0; --i) {
				double sacc = gh[i];
				for (int k = i + 1; k < jj; ++k) sacc -= Hh[(size_t)k * (m + 1) + i] * y[k];
				y[i] = sacc / Hh[(size_t)i * (m + 1) + i];
			}
			DGX_HIP_CHECK(blas.axpby(0.0, b, 0.0, w, nk));
			DGX_HIP_CHECK(blas.gemv_add(V, nk, y.data(), jj, w, nk));
			if (red) DGX_HIP_CHECK(P.reduced_solution(c, w, z));
			else DGX_HIP_CHECK(P.apply(c, w, z));
			DGX_HIP_CHECK(blas.axpby(1.0, z, 1.0, x, n));
			if (*converged) break;
		}
		*iters = total;
		return hipSuccess;
	}
};

}  // namespace dgx

using dgx::Ctx;

// 3-D (HEX Euler): the FP64 J v, and no preconditioner, block-Jacobi with blocks the batched LU takes
// (nb = 5 (p + 1)^3 <= 143: p <= 2), or block SGS with blocks the batched inverse and the sweep take (p <= 2)
static bool implicit_3d_ok(const Ctx& c, int precond, int jvp_fp32)
{
	if (c.d != 3) return true;
	if (jvp_fp32) return false;
	if (precond == DGX_PC_NONE) return true;
	if (precond == DGX_PC_BLOCK_SGS || precond == DGX_PC_BLOCK_SGS32)   // batched inverses (nb <= 142: p <= 2)
		return c.Np * c.nv <= dgx::kMaxInvBlock && 6 * c.nv * c.N * c.N <= dgx::kMaxSgsFace;
	return precond == DGX_PC_BLOCK_JACOBI && c.Np * c.nv <= dgx::kMaxLuBlock;
}

extern "C" dgx_status dgx_precond_apply(dgx_ctx* h, int precond, const double* u, const double* inv_dt,
                                        const double* v, double* z)
{
	if (!h || !u || !inv_dt || !v || !z || v == z) return DGX_ERR_ARG;
	Ctx& c = h->c;
	if (!c.mesh_ready) return c.hp ? DGX_ERR_UNSUPPORTED : DGX_ERR_NO_MESH;
	if ((c.d != 2 && c.d != 3) || c.cfg.pde == DGX_PDE_ADVECTION) return DGX_ERR_UNSUPPORTED;
	// Navier-Stokes: no learned preconditioner (it is trained on Euler blocks)
	if (c.cfg.pde == DGX_PDE_NAVIER_STOKES && precond == DGX_PC_LEARNED) return DGX_ERR_UNSUPPORTED;
	if (!implicit_3d_ok(c, precond, 0)) return DGX_ERR_UNSUPPORTED;
	dgx::Precond* P = nullptr;
	if (precond == DGX_PC_NONE) P = new dgx::PrecondIdentity();
	else if (precond == DGX_PC_BLOCK_JACOBI) P = new dgx::PrecondBlockJacobi();
	else if (precond == DGX_PC_BLOCK_SGS) P = new dgx::PrecondBlockSGS();
	else if (precond == DGX_PC_BLOCK_SGS32) P = new dgx::PrecondBlockSGS(true);
	else if (precond == DGX_PC_LEARNED) P = dgx::make_learned_precond(c);
	if (!P) return precond == DGX_PC_LEARNED ? DGX_ERR_UNSUPPORTED : DGX_ERR_ARG;
	hipError_t e = P->setup(c, u, inv_dt);
	if (e == hipSuccess) e = P->apply(c, v, z);
	if (e == hipSuccess) e = hipStreamSynchronize(c.stream);   // the preconditioner's buffers go with it
	delete P;
	if (e == hipErrorInvalidValue) return DGX_ERR_UNSUPPORTED;
	return e == hipSuccess ? DGX_OK : DGX_ERR_HIP;
}

extern "C" dgx_status dgx_solve_implicit(dgx_ctx* h, double* u, const dgx_implicit_params* prm, dgx_implicit_stats* st)
{
	if (!h || !u || !prm || !st) return DGX_ERR_ARG;
	Ctx& c = h->c;
	if (!c.mesh_ready) return c.hp ? DGX_ERR_UNSUPPORTED : DGX_ERR_NO_MESH;
	if ((c.d != 2 && c.d != 3) || c.cfg.pde == DGX_PDE_ADVECTION) return DGX_ERR_UNSUPPORTED;
	// Navier-Stokes: no learned preconditioner (it is trained on Euler blocks)
	if (c.cfg.pde == DGX_PDE_NAVIER_STOKES && prm->precond == DGX_PC_LEARNED) return DGX_ERR_UNSUPPORTED;
	if (!implicit_3d_ok(c, prm->precond, prm->jvp_fp32)) return DGX_ERR_UNSUPPORTED;
	if (prm->gmres_restart < 1 || prm->gmres_restart > 200 || prm->max_newton < 1 || !(prm->cfl_initial > 0.0))
		return DGX_ERR_ARG;
	std::memset(st, 0, sizeof(*st));
	const auto t0 = std::chrono::steady_clock::now();
	const size_t n = (size_t)c.E * c.Np * c.nv;
	double *r = nullptr, *inv_dt = nullptr;
	int* status = nullptr;
	dgx::Gmres gm;
	dgx::Precond* P = nullptr;
	dgx::PrecondBlockJacobi* Pfb = nullptr;   // exact fallback of the learned preconditioner
	dgx_status ret = DGX_OK;
	auto fail = [&](dgx_status s) { ret = s; };
	do {
		if (hipMalloc(&r, sizeof(double) * n) != hipSuccess || hipMalloc(&inv_dt, sizeof(double) * c.E) != hipSuccess ||
		    hipMalloc(&status, sizeof(int)) != hipSuccess || gm.init(c, prm->gmres_restart) != hipSuccess) {
			fail(DGX_ERR_HIP);
			break;
		}
		gm.jvp32 = prm->jvp_fp32 != 0;
		if (prm->precond == DGX_PC_BLOCK_JACOBI) {
			auto* bj = new dgx::PrecondBlockJacobi();
			bj->cap_blocks = prm->capture_blocks;
			bj->cap_feat = prm->capture_features;
			bj->cap_sigma = prm->capture_sigma;
			bj->cap_capacity = prm->capture_capacity;
			P = bj;
		}
		else if (prm->precond == DGX_PC_BLOCK_SGS) P = new dgx::PrecondBlockSGS();
		else if (prm->precond == DGX_PC_BLOCK_SGS32) P = new dgx::PrecondBlockSGS(true);
		else if (prm->precond == DGX_PC_LEARNED) {
			P = dgx::make_learned_precond(c);
			if (prm->learned_fallback_iters > 0) Pfb = new dgx::PrecondBlockJacobi();
		}
		else P = new dgx::PrecondIdentity();
		if (!P) { fail(DGX_ERR_UNSUPPORTED); break; }
		double max_rhs0 = 0.0;
		for (int it = 0; it < prm->max_newton; ++it) {
			if (dgx::launch_rhs64(c, u, r, dgx::MODE_RHS, nullptr) != hipSuccess) { fail(DGX_ERR_HIP); break; }
			double mx = 0.0;
			if (dgx::launch_fill_u64(c.stream, c.dmax, 1, 0ull) != hipSuccess ||
			    dgx::launch_maxabs(c, r, n, c.dmax) != hipSuccess) { fail(DGX_ERR_HIP); break; }
			unsigned long long bits = 0;
			// read on the stream that wrote it (a non-blocking caller stream does not order with the null stream)
			if (hipMemcpyAsync(&bits, c.dmax, sizeof(bits), hipMemcpyDeviceToHost, c.stream) != hipSuccess ||
			    hipStreamSynchronize(c.stream) != hipSuccess) { fail(DGX_ERR_HIP); break; }
			std::memcpy(&mx, &bits, sizeof(mx));
			if (!(mx == mx) || mx > 1e300) { fail(DGX_ERR_NONFINITE); break; }
			if (it == 0) max_rhs0 = mx;
			if (it < DGX_HISTORY_MAX) st->history[it] = mx;
			st->newton_steps = it;
			st->max_rhs = mx;
			st->max_rhs0 = max_rhs0;
			if (mx < prm->exit_tol || (prm->exit_ratio > 0.0 && mx / max_rhs0 < prm->exit_ratio)) {
				st->converged = 1;
				break;
			}
			double cfl = prm->cfl_initial * (max_rhs0 / mx < 1.0 ? 1.0 : max_rhs0 / mx);
			if (prm->cfl_max > 0.0 && cfl > prm->cfl_max) cfl = prm->cfl_max;
			if (dgx::launch_cfl_dt(c, u, cfl, inv_dt) != hipSuccess) { fail(DGX_ERR_HIP); break; }
			// b = -r
			if (gm.blas.axpby(-1.0, r, 0.0, r, n) != hipSuccess) { fail(DGX_ERR_HIP); break; }
			if (P->setup(c, u, inv_dt) != hipSuccess) { fail(DGX_ERR_HIP); break; }
			int its = 0;
			bool conv = false;
			const int first_max = Pfb ? std::min(prm->learned_fallback_iters, prm->gmres_max_iter) : prm->gmres_max_iter;
			if (gm.solve(c, u, inv_dt, r, *P, prm->gmres_rtol, first_max, &its, &conv) != hipSuccess) {
				fail(DGX_ERR_HIP);
				break;
			}
			int step_its = its;
			if (Pfb && !conv) {
				// the learned preconditioner did not get there: exact block-Jacobi for this step
				st->fallback_steps += 1;
				if (Pfb->setup(c, u, inv_dt) != hipSuccess ||
				    gm.solve(c, u, inv_dt, r, *Pfb, prm->gmres_rtol, prm->gmres_max_iter, &its, &conv) != hipSuccess) {
					fail(DGX_ERR_HIP);
					break;
				}
				step_its += its;
			}
			its = step_its;
			if (it < DGX_HISTORY_MAX) st->gmres_per_step[it] = its;
			st->gmres_iters += its;
			if (!conv) st->gmres_not_converged += 1;  // KSP DIVERGED_ITS: warn and continue
			// s += relax * x, then the positivity limiter on every element (update_coef_s_v,
			// solve_implicit.c:723-732; enforce_positivity_highorder, solve.c:187-233)
			if (dgx::launch_fill_i32(c.stream, status, 1, 0) != hipSuccess ||
			    dgx::launch_relaxed_update(c, u, gm.x, status) != hipSuccess ||
			    dgx::launch_positivity(c, u, status) != hipSuccess) { fail(DGX_ERR_HIP); break; }
			int bad = 0;
			if (hipMemcpyAsync(&bad, status, sizeof(int), hipMemcpyDeviceToHost, c.stream) != hipSuccess ||
			    hipStreamSynchronize(c.stream) != hipSuccess) { fail(DGX_ERR_HIP); break; }
			if (bad) { fail(DGX_ERR_POSITIVITY); break; }
			st->newton_steps = it + 1;
		}
	} while (0);
	(void)hipStreamSynchronize(c.stream);
	if (prm->precond == DGX_PC_BLOCK_JACOBI && P) st->captured = static_cast<dgx::PrecondBlockJacobi*>(P)->cap_count;
	delete P;
	delete Pfb;
	gm.release();
	if (r) (void)hipFree(r);
	if (inv_dt) (void)hipFree(inv_dt);
	if (status) (void)hipFree(status);
	st->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
	if (ret == DGX_OK && !st->converged) ret = DGX_ERR_NOT_CONVERGED;
	return ret;
}
