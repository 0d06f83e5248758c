// k_blocks.hip -- element blocks of the Newton matrix on uniform-order QUAD meshes, each element's blocks in one
// workgroup, and the batched block inverse (gfx950).
//
// The diagonal block dR_e/du_e - s_e M_e (constructor_lhs_v_1_T compute_volume_rlhs_T.c:179-220, the lhs_ll / lhs_rr
// parts of constructor_lhs_f_1_T compute_face_rlhs_T.c:163-220, compute_CFL_ramping solve_dg.c:223-248) and the face
// blocks dR_e/du_n (lhs_lr / lhs_rl) follow from the pointwise Jacobians of the fluxes:
//   A[(eq,i),(v,j)] = sum_d sum_q (d phi_i / d xi_d)(q) J_d(q)[eq][v] phi_j(q) - s_e sum_q phi_i w J phi_j (eq = v)
//                     - sum_faces sum_a phi_i(a) H_f(a)[eq][v] phi_j(a),
// J_d the weighted contravariant flux Jacobian at the volume cubature and H_f the weighted numerical-flux Jacobian with
// respect to the own trace, both by dual numbers with one seed per variable.
#include <hip/hip_runtime.h>

#include "k_residual.h"

namespace dgx {

struct BlockArgs {
	const double* u;
	const double* scale;   // s_e of the -s_e M_e term (or NULL)
	double* diag;          // E x nb x nb, row-major (or NULL)
	double* off;           // E x 4 x nfv x nfv compact transposed face blocks [col][row] (or NULL)
	const double* met;
	const double* detJ;
	const double* nJ;
	const ElemFace* ef;
	const Ops1D<double>* ops;
	double bc_prim[5];
	double b_adv[3];
};

template <int N, int NV>
constexpr int block_threads()
{
	constexpr int items = NV * NV * N * N;
	return items >= 256 ? 256 : (items + 63) / 64 * 64;
}

// One workgroup per element.  What bounds it: the store of the nb x nb block (QUAD p = 3: 32 KB an element) and, per
// lane, N^3 + 2 N^2 multiply-adds; the pointwise Jacobians take NV dual evaluations per node.  A lane owns the outputs
// of one (eq, i1, v, j1): it contracts the Jacobians over q1 once (T0, T1), then forms the N x N outputs over (i0, j0),
// N contiguous values of a row each.  The face terms ride along: a face r- / r+ has i0 = j0 = 0 / N-1, a face s- / s+
// i1 = j1 = 0 / N-1, where it has the form of T1.  Against one residual launch in dual numbers per block column and a
// mass kernel: QUAD p = 3, 4096 elements, 1090 us -> 73 us.
template <int N, int PDE, int FLUX>
__global__ void __launch_bounds__(256) k_element_blocks(BlockArgs a)
{
	constexpr int Np = N * N, NV = (PDE == DGX_PDE_EULER) ? 4 : 1, NV2 = NV * NV, NFV = NV * N;
	__shared__ double sI[Np], sDI[Np], sW[N];
	__shared__ int sPerm[8][N];
	__shared__ double sU[NV * Np], sT[NV * Np], sTr[2][4][NV][N], sNb[4][NV][N];
	__shared__ double sJ[2][Np][NV2], sH[2][4][N][NV2], sM[Np];
	__shared__ ElemFace sEF[4];
	const int e = blockIdx.x, t = threadIdx.x, nt = blockDim.x;
	for (int i = t; i < Np; i += nt) {
		sI[i] = a.ops->I[i];
		sDI[i] = a.ops->DI[i];
		sM[i] = a.scale ? a.scale[e] * (a.ops->w[i % N] * a.ops->w[i / N] * a.detJ[(size_t)e * Np + i]) : 0.0;
	}
	for (int i = t; i < N; i += nt) sW[i] = a.ops->w[i];
	for (int i = t; i < 8 * N; i += nt) sPerm[i / N][i % N] = a.ops->perm[i / N][i % N];
	if (t < 4) sEF[t] = a.ef[(size_t)e * 4 + t];
	for (int i = t; i < NV * Np; i += nt) sU[i] = a.u[(size_t)e * NV * Np + i];
	for (int it = t; it < 4 * NV * N; it += nt) {   // the neighbours' face nodes, each in its own ordering
		const int lf = it / (NV * N), v = (it / N) % NV, b = it % N;
		const ElemFace f = a.ef[(size_t)e * 4 + lf];
		sNb[lf][v][b] = f.en >= 0 ? a.u[((size_t)f.en * NV + v) * Np + face_vol_node<2, N>(f.packed & 15, b)] : 0.0;
	}
	__syncthreads();
	for (int it = t; it < NV * Np; it += nt) {      // GLL -> GL along r
		const int q0 = it % N, row = it - q0;
		double acc = 0.0;
#pragma unroll
		for (int m = 0; m < N; ++m) acc += sI[q0 * N + m] * sU[row + m];
		sT[it] = acc;
	}
	for (int it = t; it < 8 * NV * N; it += nt) {   // face traces at the GL points, own then neighbour
		const int s = it / (4 * NV * N), lf = (it / (NV * N)) % 4, v = (it / N) % NV, q = it % N;
		double acc = 0.0;
#pragma unroll
		for (int m = 0; m < N; ++m)
			acc += sI[q * N + m] * (s == 0 ? sU[v * Np + face_vol_node<2, N>(lf, m)] : sNb[lf][v][m]);
		sTr[s][lf][v][q] = acc;
	}
	__syncthreads();
	// pointwise Jacobians, one seeded variable per item
	for (int it = t; it < Np * NV; it += nt) {
		const int q = it % Np, sv = it / Np, q0 = q % N, q1 = q / N;
		Dual s[NV], fr[2][NV];
#pragma unroll
		for (int v = 0; v < NV; ++v) {
			double acc = 0.0;
#pragma unroll
			for (int m = 0; m < N; ++m) acc += sI[q1 * N + m] * sT[v * Np + q0 + N * m];
			s[v] = Dual(acc, v == sv ? 1.0 : 0.0);
		}
		double m[4];
#pragma unroll
		for (int k = 0; k < 4; ++k) m[k] = a.met[((size_t)e * 4 + k) * Np + q];
		const double wq = sW[q0] * sW[q1];
		if constexpr (PDE == DGX_PDE_EULER) {
			euler_contravariant_flux<Dual, double, 2>(s, m, wq, fr);
		} else {
			fr[0][0] = wq * ((a.b_adv[0] * m[0] + a.b_adv[1] * m[1]) * s[0]);
			fr[1][0] = wq * ((a.b_adv[0] * m[2] + a.b_adv[1] * m[3]) * s[0]);
		}
#pragma unroll
		for (int eq = 0; eq < NV; ++eq) {
			sJ[0][q][eq * NV + sv] = fr[0][eq].d;
			sJ[1][q][eq * NV + sv] = fr[1][eq].d;
		}
	}
	const int sides = a.off ? 2 : 1;   // derivative with respect to the own trace, then the neighbour's
	for (int it = t; it < sides * 4 * N * NV; it += nt) {
		const int i = it % N, lf = (it / N) % 4, sv = (it / (4 * N)) % NV, which = it / (4 * N * NV);
		const ElemFace f = sEF[lf];
		const int side = (f.packed >> 4) & 1, ord = (f.packed >> 8) & 7, bc = (f.packed >> 12) & 15;
		const int pi = sPerm[ord][i], own = side == 0 ? i : pi, nb = side == 0 ? pi : i;
		Dual so[NV], sn[NV], nnf[NV], nu[2];
#pragma unroll
		for (int v = 0; v < NV; ++v) {
			so[v] = Dual(sTr[0][lf][v][own], (which == 0 && v == sv) ? 1.0 : 0.0);
			sn[v] = Dual(sTr[1][lf][v][nb], (which == 1 && v == sv) ? 1.0 : 0.0);
		}
		const double* np_ = a.nJ + ((size_t)f.f * N + i) * 2;
		const double Jf = tsqrt(np_[0] * np_[0] + np_[1] * np_[1]), Jfi = trcp(Jf);
		nu[0] = Dual(np_[0] * Jfi);
		nu[1] = Dual(np_[1] * Jfi);
		if constexpr (PDE == DGX_PDE_EULER) {
			if (f.en < 0) bc_state<Dual, 2>(bc, so, nu, a.bc_prim, sn);
			Dual sL[NV], sR[NV];
#pragma unroll
			for (int v = 0; v < NV; ++v) {
				sL[v] = side == 0 ? so[v] : sn[v];
				sR[v] = side == 0 ? sn[v] : so[v];
			}
			if constexpr (FLUX == DGX_FLUX_LF) numflux_lf<Dual, 2>(sL, sR, nu, nnf);
			else numflux_roe<Dual, 2>(sL, sR, nu, nnf);
		} else {
			const double bn = a.b_adv[0] * nu[0].v + a.b_adv[1] * nu[1].v;
			nnf[0] = ((bn > kEps) == (side == 0)) ? bn * so[0] : bn * sn[0];
		}
		const double scale = (side == 0 ? Jf : -Jf) * sW[own];
#pragma unroll
		for (int eq = 0; eq < NV; ++eq) sH[which][lf][own][eq * NV + sv] = scale * nnf[eq].d;
	}
	__syncthreads();
	if (a.diag) {
		constexpr int nb = NV * Np;
		double* out = a.diag + (size_t)e * nb * nb;
		const auto gI = as_constant(a.ops->I), gDI = as_constant(a.ops->DI);
		for (int it = t; it < NV2 * Np; it += nt) {
			const int j1 = it % N, v = (it / N) % NV, i1 = (it / (N * NV)) % N, eq = it / (Np * NV);
			const int ev = eq * NV + v;
			const bool lo = (i1 == 0 && j1 == 0), hi = (i1 == N - 1 && j1 == N - 1);
			double p[N], d[N], T0[N], T1[N], e0 = 0.0, e1 = 0.0;
#pragma unroll
			for (int q = 0; q < N; ++q) {
				const double ij = sI[q * N + j1];
				p[q] = sI[q * N + i1] * ij;
				d[q] = sDI[q * N + i1] * ij;
				e0 += p[q] * sH[0][0][q][ev];
				e1 += p[q] * sH[0][1][q][ev];
			}
#pragma unroll
			for (int q0 = 0; q0 < N; ++q0) {
				double x0 = 0.0, x1 = 0.0, xm = 0.0;
#pragma unroll
				for (int q1 = 0; q1 < N; ++q1) {
					const int q = q0 + N * q1;
					x0 += p[q1] * sJ[0][q][ev];
					x1 += d[q1] * sJ[1][q][ev];
					xm += p[q1] * sM[q];
				}
				if (eq == v) x1 -= xm;
				if (lo) x1 -= sH[0][2][q0][ev];
				if (hi) x1 -= sH[0][3][q0][ev];
				T0[q0] = x0;
				T1[q0] = x1;
			}
#pragma unroll
			for (int i0 = 0; i0 < N; ++i0) {
				double X[N];
#pragma unroll
				for (int q0 = 0; q0 < N; ++q0) X[q0] = gDI[q0 * N + i0] * T0[q0] + gI[q0 * N + i0] * T1[q0];
				double* row = out + (size_t)(eq * Np + i0 + N * i1) * nb + v * Np + N * j1;
#pragma unroll
				for (int j0 = 0; j0 < N; ++j0) {
					double acc = 0.0;
#pragma unroll
					for (int q0 = 0; q0 < N; ++q0) acc += gI[q0 * N + j0] * X[q0];
					if (i0 == 0 && j0 == 0) acc -= e0;
					if (i0 == N - 1 && j0 == N - 1) acc -= e1;
					row[j0] = acc;
				}
			}
		}
	}
	if (a.off) {
		double* out = a.off + (size_t)e * 4 * NFV * NFV;
		for (int it = t; it < 4 * NFV * NFV; it += nt) {
			const int b = it % N, eq = (it / N) % NV, c = (it / NFV) % N, w = (it / (NFV * N)) % NV, lf = it / (NFV * NFV);
			const ElemFace f = sEF[lf];
			double acc = 0.0;
			if (f.en >= 0) {
				const int side = (f.packed >> 4) & 1, ord = (f.packed >> 8) & 7;
#pragma unroll
				for (int i = 0; i < N; ++i) {
					const int pi = sPerm[ord][i], own = side == 0 ? i : pi, nb = side == 0 ? pi : i;
					acc -= sI[own * N + b] * sI[nb * N + c] * sH[1][lf][own][eq * NV + w];
				}
			}
			out[it] = acc;
		}
	}
}

static hipError_t run_element_blocks(Ctx& c, const BlockArgs& a)
{
	const int pde = c.cfg.pde, flux = c.cfg.num_flux;
#define DGX_BLOCKS(NN)                                                                                                   \
	if (c.N == NN) {                                                                                                      \
		if (pde == DGX_PDE_ADVECTION)                                                                                     \
			hipLaunchKernelGGL((k_element_blocks<NN, DGX_PDE_ADVECTION, DGX_FLUX_UPWIND>), dim3(c.E),                     \
			                   dim3(block_threads<NN, 1>()), 0, c.stream, a);                                             \
		else if (flux == DGX_FLUX_LF)                                                                                     \
			hipLaunchKernelGGL((k_element_blocks<NN, DGX_PDE_EULER, DGX_FLUX_LF>), dim3(c.E), dim3(block_threads<NN, 4>()), \
			                   0, c.stream, a);                                                                           \
		else                                                                                                              \
			hipLaunchKernelGGL((k_element_blocks<NN, DGX_PDE_EULER, DGX_FLUX_ROE>), dim3(c.E), dim3(block_threads<NN, 4>()), \
			                   0, c.stream, a);                                                                           \
		return hipGetLastError();                                                                                         \
	}
	DGX_BLOCKS(2) DGX_BLOCKS(3) DGX_BLOCKS(4) DGX_BLOCKS(5)
#undef DGX_BLOCKS
	return hipErrorInvalidValue;
}

static BlockArgs make_block_args(Ctx& c, const double* u)
{
	BlockArgs a{};
	a.u = u;
	a.met = c.metrics_vc;
	a.detJ = c.detJ_vc;
	a.nJ = c.nJ_fc;
	a.ef = c.elem_faces;
	a.ops = c.ops64;
	for (int k = 0; k < 5; ++k) a.bc_prim[k] = c.cfg.bc_prim[k];
	for (int k = 0; k < 3; ++k) a.b_adv[k] = c.cfg.b_adv[k];
	return a;
}

// QUAD Euler and advection: k_element_blocks; HEX meshes and the BR2 residual: one dual-number residual per column
// (their blocks couple whole elements or do not fit a workgroup's pointwise Jacobians at every order)
hipError_t launch_diag_blocks(Ctx& c, const double* u, const double* scale, double* blocks)
{
	if (c.has_nonconforming) return hipErrorInvalidValue;   // no linearisation of faces between orders
	if (c.E == 0) return hipSuccess;
	if (c.d == 2 && c.cfg.pde != DGX_PDE_NAVIER_STOKES) {
		BlockArgs a = make_block_args(c, u);
		a.scale = scale;
		a.diag = blocks;
		return run_element_blocks(c, a);
	}
	const int nb = c.Np * c.nv;
	for (int col = 0; col < nb; ++col) DGX_HIP_CHECK(launch_diag_col(c, u, blocks, col));
	return scale ? launch_sub_mass(c, blocks, scale, 0.0) : hipSuccess;
}

hipError_t launch_offd_blocks(Ctx& c, const double* u, double* offT)
{
	if (c.has_nonconforming) return hipErrorInvalidValue;
	if (c.E == 0) return hipSuccess;
	if (c.d == 2 && c.cfg.pde != DGX_PDE_NAVIER_STOKES) {
		BlockArgs a = make_block_args(c, u);
		a.off = offT;
		return run_element_blocks(c, a);
	}
	const int nfv = c.nv * (c.d == 2 ? c.N : c.N * c.N);
	for (int col = 0; col < nfv; ++col) DGX_HIP_CHECK(launch_offd_col(c, u, offT, col));
	return hipSuccess;
}

// ------------------------------------------------------------------------------- batched block inverse
// In-place inverse of every nb x nb block by Gauss-Jordan elimination with partial pivoting, stored transposed
// (out[j * nb + i] = (A^-1)[i][j]) so that the apply kernel reads it coalesced.
//
// One workgroup of G x G lanes per block; lane (ti, tj) holds rows ti + G r, columns tj + G c in registers.  Rows are
// never exchanged: step k takes the largest entry of column k among the rows not used yet as its pivot, and the
// permutation is applied to the addresses of the store.  What bounds it is instruction issue and the serial chain of a
// step (pivot column to LDS, its reduction, pivot row to LDS, rank-1 update), not the 2 nb^3 flops or the two passes
// over memory.  Hence one wavefront per block up to nb = 64 (G = 8: no barrier waits, and the work that every wavefront
// of a block repeats is done once; 16 x 16 lanes took 370 us where this takes 185), four wavefronts beyond, where one
// wavefront's registers do not hold the block.  With the block in LDS, a pivot search on one lane and an integer division per entry:
// 4096 blocks of 64 x 64 1700 us -> 185 us.
__device__ inline unsigned wave_max(unsigned x)   // the maximum over the 64 lanes, in every lane
{
	// within rows of 16 lanes, then across them; lanes without a source keep their own value
#define DGX_DPP_MAX(ctrl, rows)                                                                               \
	{                                                                                                          \
		const unsigned o = (unsigned)__builtin_amdgcn_update_dpp((int)x, (int)x, ctrl, rows, 0xf, false);      \
		x = o > x ? o : x;                                                                                     \
	}
	DGX_DPP_MAX(0x111, 0xf)   // row_shr:1
	DGX_DPP_MAX(0x112, 0xf)   // row_shr:2
	DGX_DPP_MAX(0x114, 0xf)   // row_shr:4
	DGX_DPP_MAX(0x118, 0xf)   // row_shr:8
	DGX_DPP_MAX(0x142, 0xa)   // row_bcast:15
	DGX_DPP_MAX(0x143, 0xc)   // row_bcast:31
#undef DGX_DPP_MAX
	return (unsigned)__builtin_amdgcn_readlane((int)x, 63);
}

template <int G, int TR>
__global__ void __launch_bounds__(G * G) k_block_inverse(double* blocks, int nb, int* status)
{
	constexpr int ROWS = G * TR;
	__shared__ double sCol[2][ROWS], sRow[2][ROWS];
	__shared__ int sStep[ROWS], sPivot[ROWS];   // step of a pivot row, pivot row of a step
	const int e = blockIdx.x, t = threadIdx.x, ti = t % G, tj = t / G, lane = t & 63;
	double* g = blocks + (size_t)e * nb * nb;
	double A[TR][TR];
#pragma unroll
	for (int r = 0; r < TR; ++r)
#pragma unroll
		for (int c = 0; c < TR; ++c) {
			const int i = ti + G * r, j = tj + G * c;
			A[r][c] = (i < nb && j < nb) ? g[(size_t)i * nb + j] : 0.0;
		}
	// rows already used as pivots (and rows beyond the block), one bit per r of row lane + 64 r
	unsigned used = 0;
#pragma unroll
	for (int r = 0; r < (ROWS + 63) / 64; ++r)
		if (lane + 64 * r >= nb) used |= 1u << r;
	int buf = 0;
#pragma unroll
	for (int kc = 0; kc < TR; ++kc) {
		const int kend = min(G, nb - G * kc);
		for (int kt = 0; kt < kend; ++kt, buf ^= 1) {
			const int k = G * kc + kt;
			if (tj == kt)
#pragma unroll
				for (int r = 0; r < TR; ++r) {
					sCol[buf][ti + G * r] = A[r][kc];
					A[r][kc] = 0.0;
				}
			__syncthreads();
			// the pivot row, found by every wavefront: the magnitudes' bits order like the magnitudes; the last eight of
			// the upper word give way to the row, so entries within 2^-12 of the largest count as equal (first row wins)
			unsigned key = 0;
#pragma unroll
			for (int r = 0; r < (ROWS + 63) / 64; ++r) {
				const int i = lane + 64 * r;
				if (!((used >> r) & 1u)) {
					const unsigned b = ((unsigned)__double2hiint(sCol[buf][i]) & 0x7fffff00u) | (unsigned)(255 - i);
					key = b > key ? b : key;
				}
			}
			key = wave_max(key);
			const int p = 255 - (int)(key & 255u);
			if (lane == (p & 63)) used |= 1u << (p >> 6);
			if (t == 0) {
				sStep[p] = k;
				sPivot[k] = p;
				if ((key >> 8) == 0 && status && !(fabs(sCol[buf][p]) > 0.0)) atomicOr(status, 1);
			}
			if (ti == p % G)
#pragma unroll
				for (int r = 0; r < TR; ++r)
					if (r == p / G)
#pragma unroll
						for (int c = 0; c < TR; ++c) {
							sRow[buf][tj + G * c] = A[r][c];
							A[r][c] = 0.0;
						}
			__syncthreads();
			const double inv = 1.0 / sCol[buf][p];
			double row[TR];
#pragma unroll
			for (int c = 0; c < TR; ++c) row[c] = sRow[buf][tj + G * c] * inv;
			if (tj == kt) row[kc] = inv;
			// the pivot row and column start from zero: the pivot row becomes 0 - (-1) row
#pragma unroll
			for (int r = 0; r < TR; ++r) {
				const double col = (ti + G * r == p) ? -1.0 : sCol[buf][ti + G * r];
#pragma unroll
				for (int c = 0; c < TR; ++c) A[r][c] -= col * row[c];
			}
		}
	}
	__syncthreads();
	// A^-1[step of row i][pivot row of column j] = A[i][j]
#pragma unroll
	for (int c = 0; c < TR; ++c) {
		const int j = tj + G * c;
		if (j >= nb) continue;
		double* orow = g + (size_t)sPivot[j] * nb;
#pragma unroll
		for (int r = 0; r < TR; ++r) {
			const int i = ti + G * r;
			if (i < nb) orow[sStep[i]] = A[r][c];
		}
	}
}

hipError_t launch_block_inverse(hipStream_t s, double* blocks, int E, int nb, int* status)
{
	if (E == 0) return hipSuccess;
	if (nb <= 0 || nb > kMaxInvBlock) return hipErrorInvalidValue;
#define DGX_INV(G, TR) \
	case TR: hipLaunchKernelGGL((k_block_inverse<G, TR>), dim3(E), dim3(G * G), 0, s, blocks, nb, status); break;
	if (nb <= 64) {
		switch ((nb + 7) / 8) {
		DGX_INV(8, 1) DGX_INV(8, 2) DGX_INV(8, 3) DGX_INV(8, 4) DGX_INV(8, 5) DGX_INV(8, 6) DGX_INV(8, 7) DGX_INV(8, 8)
		}
	} else {
		switch ((nb + 15) / 16) {
		DGX_INV(16, 5) DGX_INV(16, 6) DGX_INV(16, 7) DGX_INV(16, 8) DGX_INV(16, 9)
		}
	}
#undef DGX_INV
	return hipGetLastError();
}

}  // namespace dgx
