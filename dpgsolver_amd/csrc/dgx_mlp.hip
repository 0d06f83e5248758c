// dgx_mlp.hip -- learned block preconditioner: a 3-layer MLP (BF16 weights, FP32 accumulation on
// MFMA) maps per-element features to an approximate inverse P_e of the element diagonal block
// A_e = dR_e/du_e - M_e/dt_e of the pseudo-time Newton system, in one of two structures:
//   LOWRANK: P_e = sigma_e (diag(d_e) + U_e V_e^T), rank R (= 8);
//   KRON:    P_e = sigma_e sum_{r<R} S_r (x) Q_r, S_r nv x nv (variables), Q_r Np x Np (nodes), R = 4 or 8,
//            which follows the (variables) x (nodes) Kronecker structure of the DG block;
// sigma_e = 1 / (mean(w detJ)/dt_e + 0.25 h_e lambda_e) is analytic, so the network outputs stay O(1)
// along the CFL ramp.
// Training data are the solver's own blocks captured along its Newton iterations; the loss is
//   L = (1/B) sum_e ||P_e A_e - I||_F^2 / nb,
// minimised with Adam.  Forward, backward and the loss gradient are hand-written kernels; the GEMMs use
// v_mfma_f32_16x16x32_bf16, the loss's block products v_mfma_f32_16x16x4_f32.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "dgx_device.h"
#include "dgx_internal.h"

namespace dgx {

using bf16x8 = __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16;
using f32x4 = __attribute__((__vector_size__(4 * sizeof(float)))) float;

__device__ inline short f2bf(float x)
{
	// round-to-nearest-even float -> bf16 bits
	unsigned u = __float_as_uint(x);
	if ((u & 0x7f800000u) == 0x7f800000u) return (short)(u >> 16);  // inf/nan
	u += 0x7fffu + ((u >> 16) & 1u);
	return (short)(u >> 16);
}
__device__ inline float bf2f(short b) { return __uint_as_float(((unsigned)(unsigned short)b) << 16); }

// C[M x N] = A[M x K] B[K x N], A and B given as FP32 and rounded to bf16 on load, FP32 accumulation, then
//   + bias[col], tanh (act = 1), or times 1 - h^2 (h: the layer's tanh outputs, the derivative in the backward pass);
// rowsum (optional): the FP32 sums of A's rows over K, unrounded (a bias gradient, where A is a transposed gradient).
// A(i, k) = A[i lda + k] (ak = 1: K contiguous) or A[k lda + i];  B(k, j) = B[j ldb + k] (bk = 1) or B[k ldb + j].
struct GemmJob {
	const float *A, *B;
	float* C;
	const float *bias, *h;
	float* rowsum;
	int M, N, K, lda, ldb, ldc;
	int ak, bk, act;
	int avec, bvec;   // K-contiguous operand whose rows start on 16 bytes: 16-byte loads
	int tiles_m, tiles_n, splits, blocks;
};
struct GemmJobs {
	GemmJob job[2];   // independent products sharing a launch (tiles of the first, then of the second)
};

// Eight K values k0 + kq .. of one operand row; P points to the tile's first row at K = 0.  Everything but lane (the
// row's offset: row ld + kq, or row + kq ld) is uniform, so the loads take a scalar base and one lane offset, without a
// branch per lane.  left = K - k0 - kq: values from there on are zero (only in the last step).
__device__ inline void load8(const float* __restrict__ P, int ld, int lane, int k0, int kc, int vec, bool tail, int left,
                             float* v)
{
	if (kc && vec && !tail) {
		const float4* p = reinterpret_cast<const float4*>(P + k0 + lane);
		const float4 a = p[0], b = p[1];
		v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
		v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
	} else if (!tail) {
		const float* p = kc ? P + k0 : P + (size_t)k0 * ld;
		const int step = kc ? 1 : ld;
#pragma unroll
		for (int t = 0; t < 8; ++t) v[t] = p[(size_t)t * step + lane];
	} else {
		const float* p = kc ? P + k0 : P + (size_t)k0 * ld;
		const int step = kc ? 1 : ld;
#pragma unroll
		for (int t = 0; t < 8; ++t) v[t] = t < left ? p[(size_t)t * step + lane] : 0.f;
	}
}

// One output tile of 32 Q x 32 per workgroup of eight wavefronts: Q wavefronts above each other, each with a 32 x 32
// part, and 8 / Q of them along K (steps of 32 values dealt in turn), whose partial parts are added in a fixed order
// through LDS.  With splits > 1 a tile's K range is cut over that many workgroups and C receives their sums in planes of
// M ldc values (k_sum_planes adds them).
// The training products are small (256 x 2176 x 256 at most) and follow one another, so what bounds them is one tile's
// latency, about 4.5 us with launch and operand fetch, times the rounds of workgroups: 100 VGPRs let a CU hold two
// workgroups.  Hence no staging (operands go straight to registers, all loads of a step in flight), Q = 1 for outputs
// with few tiles (256 x 256: 64 workgroups, one step deep) and Q = 2, half the workgroups and two steps deep, where
// Q = 1 would need a second round (256 x 2176: 544 workgroups, 12.2 us; 272 with Q = 2, 12.3 too, with larger outputs 1.4x ahead).  64 x 64 tiles on four
// steps took 12.7, and letting the last workgroup of a split tile add the parts 60 (its fence writes the L2 back).
// Training step of 256 samples, hidden 256, 2176 outputs: eight products of 16.7 us (one wavefront per 16 x 16 tile,
// 4-byte loads) before, 51 us in all now.
constexpr int kGemmWaves = 8;
template <int Q>
__global__ void __launch_bounds__(64 * kGemmWaves, 4) k_gemm_bf16(GemmJobs jobs)
{
	constexpr int KW = kGemmWaves / Q, BT = 32 * Q;
	__shared__ float part[kGemmWaves][32 * 33], srow[kGemmWaves][32];
	const bool second = (int)blockIdx.x >= jobs.job[0].blocks;
	const GemmJob& g = jobs.job[second ? 1 : 0];
	const int idx = (int)blockIdx.x - (second ? jobs.job[0].blocks : 0);
	// Consecutive workgroups go to the eight XCDs in turn.  Each XCD takes a contiguous eighth of the tiles, counted along
	// the longer side of the output, so that its L2 fetches an eighth of the larger operand and not all of it; with
	// splits, the workgroups of one K range share an XCD instead.
	int tile, split = 0;
	if (g.splits > 1) {
		tile = idx / g.splits;
		split = idx - tile * g.splits;
	} else {
		tile = (idx & 7) * (g.blocks >> 3) + (idx >> 3);
	}
	if (tile >= g.tiles_m * g.tiles_n) return;
	const bool tall = g.tiles_m > g.tiles_n;
	const int minor = tall ? g.tiles_n : g.tiles_m, hi = tile / minor, lo = tile - hi * minor;
	const int tm = tall ? hi : lo, tn = tall ? lo : hi;
	const int t = threadIdx.x, l = t & 63, w = t >> 6, r16 = l & 15, kq = (l >> 4) * 8;
	const int qi = w / KW, kw = w - qi * KW;
	const int i0 = BT * tm + 32 * qi, j0 = 32 * tn;
	const bool sums = g.rowsum && tn == 0;
	// this workgroup's K range, in whole steps
	const int steps = (g.K + 31) / 32, s0 = (int)((long long)steps * split / g.splits), s1 = (int)((long long)steps * (split + 1) / g.splits);
	f32x4 acc[2][2] = {};
	float rs[2] = { 0.f, 0.f };
	// rows past the operand's last repeat it: their products are not stored
	const float* Ab = g.A + (g.ak ? (size_t)i0 * g.lda : (size_t)i0);
	const float* Bb = g.B + (g.bk ? (size_t)j0 * g.ldb : (size_t)j0);
	int la[2], lb[2];
#pragma unroll
	for (int f = 0; f < 2; ++f) {
		const int ra = max(0, min(16 * f + r16, g.M - 1 - i0)), rb = min(16 * f + r16, g.N - 1 - j0);
		la[f] = g.ak ? ra * g.lda + kq : ra + kq * g.lda;
		lb[f] = g.bk ? rb * g.ldb + kq : rb + kq * g.ldb;
	}
	if (i0 >= g.M) Ab = g.A;   // (Q = 2: the lower half of the last tile may lie beyond the output)
#pragma unroll 2
	for (int st = s0 + kw; st < s1; st += KW) {
		const int k0 = 32 * st;
		const bool tail = k0 + 32 > g.K;
		float a[2][8], b[2][8];
#pragma unroll
		for (int f = 0; f < 2; ++f) {
			load8(Ab, g.lda, la[f], k0, g.ak, g.avec, tail, g.K - k0 - kq, a[f]);
			load8(Bb, g.ldb, lb[f], k0, g.bk, g.bvec, tail, g.K - k0 - kq, b[f]);
		}
		bf16x8 ah[2], bh[2];
#pragma unroll
		for (int f = 0; f < 2; ++f)
#pragma unroll
			for (int q = 0; q < 8; ++q) {
				ah[f][q] = (__bf16)a[f][q];
				bh[f][q] = (__bf16)b[f][q];
			}
		if (sums)
#pragma unroll
			for (int f = 0; f < 2; ++f)
				rs[f] += ((a[f][0] + a[f][1]) + (a[f][2] + a[f][3])) + ((a[f][4] + a[f][5]) + (a[f][6] + a[f][7]));
#pragma unroll
		for (int fi = 0; fi < 2; ++fi)
#pragma unroll
			for (int fj = 0; fj < 2; ++fj)
				acc[fi][fj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[fi], bh[fj], acc[fi][fj], 0, 0, 0);
	}
#pragma unroll
	for (int fi = 0; fi < 2; ++fi)
#pragma unroll
		for (int fj = 0; fj < 2; ++fj)
#pragma unroll
			for (int q = 0; q < 4; ++q) part[w][(16 * fi + (l >> 4) * 4 + q) * 33 + 16 * fj + r16] = acc[fi][fj][q];
	if (sums)
#pragma unroll
		for (int f = 0; f < 2; ++f) {
			float x = rs[f];
			x += __shfl_xor(x, 16);
			x += __shfl_xor(x, 32);
			if (l < 16) srow[w][16 * f + l] = x;
		}
	__syncthreads();
	float* C = g.C + (size_t)split * g.M * g.ldc;
	for (int o = t; o < 32 * BT; o += 64 * kGemmWaves) {
		const int r = o >> 5, c = o & 31, i = BT * tm + r, j = j0 + c;
		if (i >= g.M || j >= g.N) continue;
		const float(*p)[32 * 33] = part + (r >> 5) * KW;
		float v = p[0][(r & 31) * 33 + c];
#pragma unroll
		for (int k = 1; k < KW; ++k) v += p[k][(r & 31) * 33 + c];
		if (g.bias) v += g.bias[j];
		if (g.act == 1) v = tanhf(v);
		const size_t at = (size_t)i * g.ldc + j;
		if (g.h) {
			const float h = g.h[at];
			v *= 1.f - h * h;
		}
		C[at] = v;
	}
	if (sums && t < BT && BT * tm + t < g.M) {
		const float(*p)[32] = srow + (t >> 5) * KW;
		float v = p[0][t & 31];
#pragma unroll
		for (int k = 1; k < KW; ++k) v += p[k][t & 31];
		g.rowsum[BT * tm + t] = v;
	}
}

// out = (sum of the planes, in order) times 1 - h^2
__global__ void __launch_bounds__(256) k_sum_planes(const float* __restrict__ planes, int count, const float* __restrict__ h,
                                                    float* out, size_t n)
{
	for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
		float v = planes[i];
		for (int k = 1; k < count; ++k) v += planes[(size_t)k * n + i];
		out[i] = v * (1.f - h[i] * h[i]);
	}
}

static GemmJob gemm_job(const float* A, int lda, int ak, const float* B, int ldb, int bk, float* C, int ldc, int M, int N, int K)
{
	GemmJob g{};
	g.A = A; g.B = B; g.C = C;
	g.M = M; g.N = N; g.K = K;
	g.lda = lda; g.ldb = ldb; g.ldc = ldc;
	g.ak = ak; g.bk = bk;
	g.avec = ak && lda % 4 == 0 && reinterpret_cast<uintptr_t>(A) % 16 == 0;
	g.bvec = bk && ldb % 4 == 0 && reinterpret_cast<uintptr_t>(B) % 16 == 0;
	g.splits = 1;
	return g;
}
static hipError_t gemm(hipStream_t s, const GemmJob& a, const GemmJob* b = nullptr)
{
	GemmJobs jobs{};
	jobs.job[0] = a;
	if (b) jobs.job[1] = *b;
	const int count = b ? 2 : 1;
	int grid = 0;
	auto shape = [&](int q) {
		grid = 0;
		for (int k = 0; k < count; ++k) {
			GemmJob& g = jobs.job[k];
			g.tiles_m = (g.M + 32 * q - 1) / (32 * q);
			g.tiles_n = (g.N + 31) / 32;
			g.blocks = g.splits > 1 ? g.tiles_m * g.tiles_n * g.splits : (g.tiles_m * g.tiles_n + 7) / 8 * 8;
			grid += g.blocks;
		}
	};
	// one round of two workgroups on each of the 256 CUs with 32 x 32 tiles; beyond it 64 x 32 ones
	shape(1);
	if (grid <= 512) {
		hipLaunchKernelGGL(k_gemm_bf16<1>, dim3(grid), dim3(64 * kGemmWaves), 0, s, jobs);
	} else {
		shape(2);
		hipLaunchKernelGGL(k_gemm_bf16<2>, dim3(grid), dim3(64 * kGemmWaves), 0, s, jobs);
	}
	return hipGetLastError();
}

// ------------------------------------------------------------------------------- loss and its gradient
// Per sample e the loss and, for the gradient, G = sigma dL/dP:
//   Rm = P A - I, L_e = ||Rm||_F^2 / nb,  G = sigma 2 Rm A^T / nb (times gscale, into P's place).
// One workgroup of sixteen wavefronts per sample; the two nb^3 products run on FP32 matrix instructions (FP32 inputs and
// sums, as before), one 16 x 16 tile per wavefront, blocks zero-padded to a multiple of 16 in LDS with rows of an odd
// number of words.  A training batch has about one sample per CU, so what bounds the kernel is one sample's latency:
// with four wavefronts and 4 x 4 register tiles of ordinary multiply-adds a batch of 256 took 21.8 us, now 12.4.
constexpr int kLossLanes = 1024;
template <int NB>
struct LossBlocks {
	static constexpr int T = (NB + 15) / 16, NP = 16 * T, LD = NP + 1;
	float A[NP * LD], P[NP * LD], R[NP * LD];
	double red[kLossLanes / 64];
};
// C tile (ti, tj) += X Y over NP columns; Y(k, j) = Y[k LD + j], or Y[j LD + k] (TRANS)
template <int NB, bool TRANS>
__device__ inline f32x4 loss_tile(const float* X, const float* Y, int ti, int tj, f32x4 acc)
{
	constexpr int NP = LossBlocks<NB>::NP, LD = LossBlocks<NB>::LD;
	const int l = threadIdx.x & 63, r16 = l & 15, kq = l >> 4;
#pragma unroll
	for (int k = 0; k < NP; k += 4) {
		const float x = X[(16 * ti + r16) * LD + k + kq];
		const float y = TRANS ? Y[(16 * tj + r16) * LD + k + kq] : Y[(k + kq) * LD + 16 * tj + r16];
		acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, acc, 0, 0, 0);
	}
	return acc;
}
// P and A in LDS (zero-padded); the loss to *loss, then (grad) P = gs Rm A^T
template <int NB>
__device__ inline void loss_core(LossBlocks<NB>& b, double* loss, bool grad, float gs)
{
	constexpr int T = LossBlocks<NB>::T, LD = LossBlocks<NB>::LD, NW = kLossLanes / 64;
	const int t = threadIdx.x, l = t & 63, w = t >> 6, r16 = l & 15, kq = l >> 4;
	double lsum = 0.0;
	for (int tile = w; tile < T * T; tile += NW) {
		const int ti = tile / T, tj = tile - ti * T;
		f32x4 acc;
#pragma unroll
		for (int q = 0; q < 4; ++q) {
			const int i = 16 * ti + 4 * kq + q, j = 16 * tj + r16;
			acc[q] = (i == j && i < NB) ? -1.f : 0.f;
		}
		acc = loss_tile<NB, false>(b.P, b.A, ti, tj, acc);
#pragma unroll
		for (int q = 0; q < 4; ++q) {
			b.R[(16 * ti + 4 * kq + q) * LD + 16 * tj + r16] = acc[q];
			lsum += (double)acc[q] * acc[q];
		}
	}
#pragma unroll
	for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off);
	if (l == 0) b.red[w] = lsum;
	__syncthreads();
	if (t == 0) {
		double s = 0.0;
		for (int q = 0; q < NW; ++q) s += b.red[q];
		*loss = s / NB;
	}
	if (!grad) return;
	for (int tile = w; tile < T * T; tile += NW) {
		const int ti = tile / T, tj = tile - ti * T;
		const f32x4 acc = loss_tile<NB, true>(b.R, b.A, ti, tj, f32x4{});
#pragma unroll
		for (int q = 0; q < 4; ++q) b.P[(16 * ti + 4 * kq + q) * LD + 16 * tj + r16] = acc[q] * gs;
	}
	__syncthreads();
}
template <int NB>
__device__ inline void loss_load(LossBlocks<NB>& b, const double* A)
{
	constexpr int NP = LossBlocks<NB>::NP, LD = LossBlocks<NB>::LD;
	for (int i = threadIdx.x; i < NP * NP; i += kLossLanes) {
		const int r = i / NP, c = i - r * NP;
		b.A[r * LD + c] = (r < NB && c < NB) ? (float)A[r * NB + c] : 0.f;
	}
}

// LOWRANK.  out = [d (nb) | U (nb x R, row-major) | V (nb x R)], P = sigma (diag(d) + U V^T);
// dd = diag(G), dU = G V, dV = G^T U.
template <int NB, int RK>
__global__ void __launch_bounds__(kLossLanes) k_block_loss(const float* __restrict__ out, const float* __restrict__ sigma,
                                                           const double* __restrict__ A, float* grad,
                                                           double* loss_partial, float gscale)
{
	constexpr int NO = NB + 2 * NB * RK, NP = LossBlocks<NB>::NP, LD = LossBlocks<NB>::LD;
	__shared__ LossBlocks<NB> b;
	__shared__ float sD[NB], sU[NB * RK], sV[NB * RK];
	const int e = blockIdx.x, t = threadIdx.x;
	const float sg = sigma ? sigma[e] : 1.f;
	const float* o = out + (size_t)e * NO;
	loss_load<NB>(b, A + (size_t)e * NB * NB);
	for (int i = t; i < NB; i += kLossLanes) sD[i] = o[i];
	for (int i = t; i < NB * RK; i += kLossLanes) { sU[i] = o[NB + i]; sV[i] = o[NB + NB * RK + i]; }
	__syncthreads();
	for (int ij = t; ij < NP * NP; ij += kLossLanes) {
		const int i = ij / NP, j = ij - i * NP;
		float p = 0.f;
		if (i < NB && j < NB) {
			p = (i == j) ? sD[i] : 0.f;
#pragma unroll
			for (int r = 0; r < RK; ++r) p += sU[i * RK + r] * sV[j * RK + r];
		}
		b.P[i * LD + j] = sg * p;
	}
	__syncthreads();
	loss_core<NB>(b, loss_partial + e, grad != nullptr, (2.0f / NB) * gscale * sg);
	if (!grad) return;
	float* g = grad + (size_t)e * NO;
	for (int i = t; i < NB; i += kLossLanes) g[i] = b.P[i * LD + i];
	for (int x = t; x < 2 * NB * RK; x += kLossLanes) {
		const bool u = x < NB * RK;
		const int ir = u ? x : x - NB * RK, i = ir / RK, r = ir - i * RK;
		float acc = 0.f;
		if (u)
			for (int j = 0; j < NB; ++j) acc += b.P[i * LD + j] * sV[j * RK + r];
		else
			for (int j = 0; j < NB; ++j) acc += b.P[j * LD + i] * sU[j * RK + r];
		g[NB + x] = acc;
	}
}

// z_e = sigma_e (d_e * v_e + U_e (V_e^T v_e))   (FP64 vectors, FP32 factors)
template <int NB, int RK>
__global__ void __launch_bounds__(64) k_lowrank_apply(const float* __restrict__ out, const float* __restrict__ sigma,
                                                      const double* __restrict__ v, double* z, int E)
{
	constexpr int NO = NB + 2 * NB * RK;
	__shared__ double sv[NB], sw[RK];
	const int e = blockIdx.x, t = threadIdx.x;
	const float* o = out + (size_t)e * NO;
	const double sg = sigma[e];
	for (int i = t; i < NB; i += blockDim.x) sv[i] = v[(size_t)e * NB + i];
	__syncthreads();
	for (int r = t; r < RK; r += blockDim.x) {
		double s = 0.0;
		for (int j = 0; j < NB; ++j) s += (double)o[NB + NB * RK + j * RK + r] * sv[j];
		sw[r] = s;
	}
	__syncthreads();
	for (int i = t; i < NB; i += blockDim.x) {
		double s = (double)o[i] * sv[i];
		for (int r = 0; r < RK; ++r) s += (double)o[NB + i * RK + r] * sw[r];
		z[(size_t)e * NB + i] = sg * s;
	}
}

// KRON structure.  out = [S_0 .. S_{RK-1} (NV x NV each) | Q_0 .. Q_{RK-1} (NPN x NPN each)], row-major;
// P[(a,i),(b,j)] = sigma sum_r S_r[a,b] Q_r[i,j] (rows var-major like the state).
// With G = sigma dL/dP: dS_r[a,b] = sum_ij G[(a,i),(b,j)] Q_r[i,j], dQ_r[i,j] = sum_ab G[(a,i),(b,j)] S_r[a,b].
template <int NV, int NPN, int RK>
__global__ void __launch_bounds__(kLossLanes) k_block_loss_kron(const float* __restrict__ out,
                                                                const float* __restrict__ sigma,
                                                                const double* __restrict__ A, float* grad,
                                                                double* loss_partial, float gscale)
{
	constexpr int NB = NV * NPN, NS = NV * NV, NQ = NPN * NPN, NO = RK * (NS + NQ);
	constexpr int NP = LossBlocks<NB>::NP, LD = LossBlocks<NB>::LD;
	__shared__ LossBlocks<NB> b;
	__shared__ float sO[NO];
	const int e = blockIdx.x, t = threadIdx.x;
	const float sg = sigma ? sigma[e] : 1.f;
	const float* o = out + (size_t)e * NO;
	loss_load<NB>(b, A + (size_t)e * NB * NB);
	for (int i = t; i < NO; i += kLossLanes) sO[i] = o[i];
	__syncthreads();
	const float* S = sO;
	const float* Q = sO + RK * NS;
	// a lane takes one (i, j) of a block column c for all block rows a: its Q values serve NV outputs
	for (int x = t; x < NPN * NB; x += kLossLanes) {
		const int i = x / NB, col = x - i * NB, c = col / NPN, j = col - c * NPN;
		float p[NV] = {};
#pragma unroll
		for (int r = 0; r < RK; ++r) {
			const float q = Q[r * NQ + i * NPN + j];
#pragma unroll
			for (int a = 0; a < NV; ++a) p[a] += S[r * NS + a * NV + c] * q;
		}
#pragma unroll
		for (int a = 0; a < NV; ++a) b.P[(a * NPN + i) * LD + col] = sg * p[a];
	}
	if constexpr (NP > NB)
		for (int x = t; x < NP * NP; x += kLossLanes) {
			const int row = x / NP, col = x - row * NP;
			if (row >= NB || col >= NB) b.P[row * LD + col] = 0.f;
		}
	__syncthreads();
	loss_core<NB>(b, loss_partial + e, grad != nullptr, (2.0f / NB) * gscale * sg);
	if (!grad) return;
	float* g = grad + (size_t)e * NO;
	// dS: eight lanes per entry, each every eighth (i, j)
	for (int x = t; x < 8 * RK * NS; x += kLossLanes) {
		const int y = x >> 3, r = y / NS, a = (y % NS) / NV, c = y % NV;
		float acc = 0.f;
		for (int ij = x & 7; ij < NQ; ij += 8) {
			const int i = ij / NPN, j = ij - i * NPN;
			acc += b.P[(a * NPN + i) * LD + c * NPN + j] * Q[r * NQ + ij];
		}
		acc += __shfl_xor(acc, 1);
		acc += __shfl_xor(acc, 2);
		acc += __shfl_xor(acc, 4);
		if ((x & 7) == 0) g[y] = acc;
	}
	// dQ: a lane takes one (i, j) for RG of the terms, its G values serve them all
	constexpr int RG = (RK * NQ >= 2 * kLossLanes) ? 2 : 1;
	for (int x = t; x < RK / RG * NQ; x += kLossLanes) {
		const int r = RG * (x / NQ), ij = x % NQ, i = ij / NPN, j = ij - i * NPN;
		float acc[RG] = {};
#pragma unroll
		for (int a = 0; a < NV; ++a)
#pragma unroll
			for (int c = 0; c < NV; ++c) {
				const float gp = b.P[(a * NPN + i) * LD + c * NPN + j];
#pragma unroll
				for (int q = 0; q < RG; ++q) acc[q] += gp * S[(r + q) * NS + a * NV + c];
			}
#pragma unroll
		for (int q = 0; q < RG; ++q) g[RK * NS + (r + q) * NQ + ij] = acc[q];
	}
}

// z_e[a,i] = sigma_e sum_r sum_b S_r[a,b] sum_j Q_r[i,j] v_e[b,j]   (FP64 vectors, FP32 factors)
template <int NV, int NPN, int RK>
__global__ void __launch_bounds__(64) k_kron_apply(const float* __restrict__ out, const float* __restrict__ sigma,
                                                   const double* __restrict__ v, double* z, int E)
{
	constexpr int NB = NV * NPN, NS = NV * NV, NQ = NPN * NPN, NO = RK * (NS + NQ);
	__shared__ float sO[NO];
	__shared__ double sv[NB], sW[RK * NB];
	const int e = blockIdx.x, t = threadIdx.x;
	const float* o = out + (size_t)e * NO;
	for (int i = t; i < NO; i += blockDim.x) sO[i] = o[i];
	for (int i = t; i < NB; i += blockDim.x) sv[i] = v[(size_t)e * NB + i];
	__syncthreads();
	const float* S = sO;
	const float* Q = sO + RK * NS;
	for (int x = t; x < RK * NB; x += blockDim.x) {   // W_r[b][i] = sum_j Q_r[i,j] v[b,j]
		const int r = x / NB, b = (x % NB) / NPN, i = x % NPN;
		double acc = 0.0;
		for (int j = 0; j < NPN; ++j) acc += (double)Q[r * NQ + i * NPN + j] * sv[b * NPN + j];
		sW[x] = acc;
	}
	__syncthreads();
	const double sg = sigma[e];
	for (int x = t; x < NB; x += blockDim.x) {
		const int a = x / NPN, i = x % NPN;
		double acc = 0.0;
		for (int r = 0; r < RK; ++r)
			for (int b = 0; b < NV; ++b) acc += (double)S[r * NS + a * NV + b] * sW[r * NB + b * NPN + i];
		z[(size_t)e * NB + x] = sg * acc;
	}
}

// features [u / u_ref (nb) | detJ / mean (Np) | log10(h inv_dt / lambda) | 0 pad] and sigma_e
template <int D, int N>
__global__ void __launch_bounds__(64) k_features(const double* __restrict__ u, const double* __restrict__ detJ,
                                                 const Ops1D<double>* ops, const double* __restrict__ hmin,
                                                 const double* __restrict__ inv_dt, int E, float* feat, int nf,
                                                 double uref0, double uref1, double uref2, float* sigma)
{
	constexpr int Np = ipow(N, D), NV = D + 2, nb = NV * Np;
	__shared__ double sWJ[Np], sWs[Np];
	const int e = blockIdx.x, t = threadIdx.x;
	for (int q = t; q < Np; q += blockDim.x) {
		const int c0 = q % N, c1 = (q / N) % N, c2 = (D == 3) ? q / (N * N) : 0;
		double w = ops->w[c0] * ops->w[c1];
		if (D == 3) w *= ops->w[c2];
		sWJ[q] = w * detJ[(size_t)e * Np + q];
		const double* ue = u + (size_t)e * nb;
		const double rho = ue[q], ri = 1.0 / rho;
		double V2 = 0.0;
		for (int k = 0; k < D; ++k) { const double w2 = ue[(1 + k) * Np + q] * ri; V2 += w2 * w2; }
		const double p = kGM1 * (ue[(D + 1) * Np + q] - 0.5 * rho * V2);
		sWs[q] = sqrt(V2) + sqrt(fmax(kGamma * p * ri, 0.0));
	}
	__syncthreads();
	__shared__ double mj, mdj, ws;
	if (t == 0) {
		double a = 0.0, b = 0.0, m = 0.0;
		for (int q = 0; q < Np; ++q) { a += sWJ[q]; b += detJ[(size_t)e * Np + q]; m = fmax(m, sWs[q]); }
		mj = a / Np;
		mdj = b / Np;
		ws = m;
		sigma[e] = (float)(1.0 / (mj * inv_dt[e] + 0.25 * hmin[e] * m));
	}
	__syncthreads();
	float* f = feat + (size_t)e * nf;
	for (int i = t; i < nb; i += blockDim.x) {
		const int v = i / Np;
		const double ref = (v == 0) ? uref0 : (v == NV - 1 ? uref2 : uref1);
		f[i] = (float)(u[(size_t)e * nb + i] / ref);
	}
	for (int i = t; i < Np; i += blockDim.x) f[nb + i] = (float)(detJ[(size_t)e * Np + i] / mdj);
	if (t == 0) f[nb + Np] = (float)log10(hmin[e] * inv_dt[e] / ws + 1e-30);
	for (int i = nb + Np + 1 + t; i < nf; i += blockDim.x) f[i] = 0.f;
}

// one Adam step on the FP32 master weights and the BF16 values of the result that the next forward pass takes
__global__ void __launch_bounds__(256) k_adam(float* w, const float* __restrict__ g, float* m, float* v, float* wb, size_t n,
                                              float lr, float b1, float b2, float c1, float c2, float eps)
{
	for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
		const float gi = g[i];
		const float mi = b1 * m[i] + (1.f - b1) * gi, vi = b2 * v[i] + (1.f - b2) * gi * gi;
		const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
		m[i] = mi;
		v[i] = vi;
		w[i] = wi;
		wb[i] = bf2f(f2bf(wi));
	}
}
// the forward pass always sees the BF16 values of the FP32 master weights
__global__ void k_round_bf16(const float* __restrict__ w, float* wb, size_t n)
{
	for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
		wb[i] = bf2f(f2bf(w[i]));
}

static int gridn(size_t n) { return (int)((n + 255) / 256 < 8192 ? (n + 255) / 256 : 8192); }

}  // namespace dgx

// ------------------------------------------------------------------------------- the model
struct dgx_mlp {
	int kind = 0;
	int nf = 0, nhid = 0, nout = 0, nb = 0, rank = 0, Np = 0;
	float* w = nullptr;   // FP32 master parameters W1,b1,W2,b2,W3,b3
	float* wb = nullptr;  // BF16-rounded copy used by the forward pass
	float* gw = nullptr;
	float* am = nullptr;
	float* av = nullptr;
	size_t nparam = 0;
	size_t off[6] = { 0, 0, 0, 0, 0, 0 };
	int step = 0;
	int cap = 0;
	float *h1 = nullptr, *h2 = nullptr, *o = nullptr, *go = nullptr, *gh2 = nullptr, *gh1 = nullptr;
	float* gpart = nullptr;   // planes of the product cut along K (see k_gemm_bf16), backward pass only
	int gcap = 0;             // samples that gpart holds
	double* lpart = nullptr;
	double* lall = nullptr;   // per-sample losses of a whole training set
	long long lall_cap = 0;
	hipStream_t s = nullptr;
};

namespace dgx {

constexpr int kSplits = 4;

static void mlp_free_work(dgx_mlp* m)
{
	for (float* p : { m->h1, m->h2, m->o, m->go, m->gh2, m->gh1, m->gpart })
		if (p) (void)hipFree(p);
	if (m->lpart) (void)hipFree(m->lpart);
	if (m->lall) (void)hipFree(m->lall);
	m->lall = nullptr;
	m->lall_cap = 0;
	m->h1 = m->h2 = m->o = m->go = m->gh2 = m->gh1 = m->gpart = nullptr;
	m->lpart = nullptr;
	m->cap = m->gcap = 0;
}

static hipError_t mlp_reserve(dgx_mlp* m, int B)
{
	if (B <= m->cap) return hipSuccess;
	mlp_free_work(m);
	DGX_HIP_CHECK(hipMalloc(&m->h1, sizeof(float) * (size_t)B * m->nhid));
	DGX_HIP_CHECK(hipMalloc(&m->h2, sizeof(float) * (size_t)B * m->nhid));
	DGX_HIP_CHECK(hipMalloc(&m->o, sizeof(float) * (size_t)B * m->nout));
	DGX_HIP_CHECK(hipMalloc(&m->go, sizeof(float) * (size_t)B * m->nout));
	DGX_HIP_CHECK(hipMalloc(&m->gh2, sizeof(float) * (size_t)B * m->nhid));
	DGX_HIP_CHECK(hipMalloc(&m->gh1, sizeof(float) * (size_t)B * m->nhid));
	DGX_HIP_CHECK(hipMalloc(&m->lpart, sizeof(double) * (size_t)B));
	m->cap = B;
	return hipSuccess;
}

static hipError_t mlp_forward(dgx_mlp* m, const float* X, int B, float* out = nullptr)
{
	DGX_HIP_CHECK(mlp_reserve(m, B));
	const float *W1 = m->wb + m->off[0], *W2 = m->wb + m->off[2], *W3 = m->wb + m->off[4];
	const int nf = m->nf, nh = m->nhid, no = m->nout;
	GemmJob g = gemm_job(X, nf, 1, W1, nf, 1, m->h1, nh, B, nh, nf);
	g.bias = m->wb + m->off[1];
	g.act = 1;
	DGX_HIP_CHECK(gemm(m->s, g));
	g = gemm_job(m->h1, nh, 1, W2, nh, 1, m->h2, nh, B, nh, nh);
	g.bias = m->wb + m->off[3];
	g.act = 1;
	DGX_HIP_CHECK(gemm(m->s, g));
	g = gemm_job(m->h2, nh, 1, W3, nh, 1, out ? out : m->o, no, B, no, nh);
	g.bias = m->wb + m->off[5];
	return gemm(m->s, g);
}

// gradients of the weights (transposed gradient times layer input, the bias gradient its row sums) and of the layer
// inputs; the two products that wait for the same gradient share a launch, the longer sum first
static hipError_t mlp_backward(dgx_mlp* m, const float* X, int B)
{
	const float *W2 = m->wb + m->off[2], *W3 = m->wb + m->off[4];
	const int nf = m->nf, nh = m->nhid, no = m->nout;
	if (B > m->gcap) {   // inference, over as many samples as there are elements, does without these planes
		if (m->gpart) (void)hipFree(m->gpart);
		m->gpart = nullptr;
		m->gcap = 0;
		DGX_HIP_CHECK(hipMalloc(&m->gpart, sizeof(float) * (size_t)B * nh * kSplits));
		m->gcap = B;
	}
	// the sum over the outputs is the one long K range: cut over kSplits workgroups a tile
	GemmJob gh = gemm_job(m->go, no, 1, W3, nh, 0, m->gpart, nh, B, nh, no);
	gh.splits = kSplits;
	GemmJob gw = gemm_job(m->go, no, 0, m->h2, nh, 0, m->gw + m->off[4], nh, no, nh, B);
	gw.rowsum = m->gw + m->off[5];
	DGX_HIP_CHECK(gemm(m->s, gh, &gw));
	const size_t nh2 = (size_t)B * nh;
	hipLaunchKernelGGL(k_sum_planes, dim3(gridn(nh2)), dim3(256), 0, m->s, m->gpart, kSplits, m->h2, m->gh2, nh2);
	DGX_HIP_CHECK(hipGetLastError());
	gh = gemm_job(m->gh2, nh, 1, W2, nh, 0, m->gh1, nh, B, nh, nh);
	gh.h = m->h1;
	gw = gemm_job(m->gh2, nh, 0, m->h1, nh, 0, m->gw + m->off[2], nh, nh, nh, B);
	gw.rowsum = m->gw + m->off[3];
	DGX_HIP_CHECK(gemm(m->s, gh, &gw));
	gw = gemm_job(m->gh1, nh, 0, X, nf, 0, m->gw + m->off[0], nf, nh, nf, B);
	gw.rowsum = m->gw + m->off[1];
	return gemm(m->s, gw);
}

// per-sample losses of the outputs in m->o to lpart (default: the model's buffer) and, with want_grad, their gradient
// to m->go; *loss (optional, synchronous): the mean
static hipError_t mlp_loss(dgx_mlp* m, const float* sigma, const double* A, int B, double* loss, float gscale,
                           bool want_grad, double* lpart = nullptr)
{
	float* g = want_grad ? m->go : nullptr;
	double* lp = lpart ? lpart : m->lpart;
	if (m->kind == DGX_MLP_LOWRANK && m->nb == 64 && m->rank == 8)
		hipLaunchKernelGGL((k_block_loss<64, 8>), dim3(B), dim3(kLossLanes), 0, m->s, m->o, sigma, A, g, lp, gscale);
	else if (m->kind == DGX_MLP_LOWRANK && m->nb == 36 && m->rank == 8)
		hipLaunchKernelGGL((k_block_loss<36, 8>), dim3(B), dim3(kLossLanes), 0, m->s, m->o, sigma, A, g, lp, gscale);
#define DGX_KRON_LOSS(NPN, RK)                                                                                  \
	else if (m->kind == DGX_MLP_KRON && m->Np == NPN && m->rank == RK)                                          \
		hipLaunchKernelGGL((k_block_loss_kron<4, NPN, RK>), dim3(B), dim3(kLossLanes), 0, m->s, m->o, sigma, A, g, lp, \
		                   gscale);
	DGX_KRON_LOSS(16, 4) DGX_KRON_LOSS(9, 4) DGX_KRON_LOSS(16, 8) DGX_KRON_LOSS(9, 8)
#undef DGX_KRON_LOSS
	else
		return hipErrorInvalidValue;
	DGX_HIP_CHECK(hipGetLastError());
	if (loss) {
		std::vector<double> host(B);
		DGX_HIP_CHECK(hipMemcpyAsync(host.data(), lp, sizeof(double) * B, hipMemcpyDeviceToHost, m->s));
		DGX_HIP_CHECK(hipStreamSynchronize(m->s));
		double sum = 0.0;
		for (double x : host) sum += x;
		*loss = sum / B;
	}
	return hipSuccess;
}

static hipError_t mlp_sync_bf16(dgx_mlp* m)
{
	hipLaunchKernelGGL(k_round_bf16, dim3(gridn(m->nparam)), dim3(256), 0, m->s, m->w, m->wb, m->nparam);
	return hipGetLastError();
}

struct PrecondLearned : Precond {
	dgx_mlp* mlp = nullptr;
	float* feat = nullptr;
	float* sigma = nullptr;
	~PrecondLearned() override
	{
		if (feat) (void)hipFree(feat);
		if (sigma) (void)hipFree(sigma);
	}
	hipError_t setup(Ctx& c, const double* u, const double* inv_dt) override;
	hipError_t apply(Ctx& c, const double* v, double* z) override
	{
		if (mlp->kind == DGX_MLP_KRON) {
#define DGX_KRON_APPLY(NPN, RK)                                                                                     \
			if (mlp->Np == NPN && mlp->rank == RK) {                                                                \
				hipLaunchKernelGGL((k_kron_apply<4, NPN, RK>), dim3(c.E), dim3(64), 0, c.stream, mlp->o, sigma, v, z, \
				                   c.E);                                                                            \
				return hipGetLastError();                                                                          \
			}
			DGX_KRON_APPLY(16, 4) DGX_KRON_APPLY(9, 4) DGX_KRON_APPLY(16, 8) DGX_KRON_APPLY(9, 8)
#undef DGX_KRON_APPLY
			return hipErrorInvalidValue;
		}
		if (mlp->nb == 64 && mlp->rank == 8)
			hipLaunchKernelGGL((k_lowrank_apply<64, 8>), dim3(c.E), dim3(64), 0, c.stream, mlp->o, sigma, v, z, c.E);
		else if (mlp->nb == 36 && mlp->rank == 8)
			hipLaunchKernelGGL((k_lowrank_apply<36, 8>), dim3(c.E), dim3(64), 0, c.stream, mlp->o, sigma, v, z, c.E);
		else
			return hipErrorInvalidValue;
		return hipGetLastError();
	}
};

hipError_t launch_features(Ctx& c, const double* u, const double* inv_dt, float* feat, int nf, float* sigma)
{
	if (c.d != 2 || c.nv != 4) return hipErrorInvalidValue;
	const double* bp = c.cfg.bc_prim;
	const double rho = bp[0] > 0 ? bp[0] : 1.0;
	const double vel = std::sqrt(bp[1] * bp[1] + bp[2] * bp[2]);
	const double uref1 = rho * (vel > 0 ? vel : 1.0);
	const double pres = bp[3] > 0 ? bp[3] : 1.0;
	const double uref2 = pres / kGM1 + 0.5 * rho * vel * vel;
#define DGX_FEAT(NN)                                                                                              \
	if (c.N == NN) {                                                                                              \
		hipLaunchKernelGGL((k_features<2, NN>), dim3(c.E), dim3(64), 0, c.stream, u, c.detJ_vc, c.ops64, c.hmin,   \
		                   inv_dt, c.E, feat, nf, rho, uref1, uref2, sigma);                                       \
		return hipGetLastError();                                                                                 \
	}
	DGX_FEAT(2) DGX_FEAT(3) DGX_FEAT(4) DGX_FEAT(5) DGX_FEAT(6)
#undef DGX_FEAT
	return hipErrorInvalidValue;
}

hipError_t PrecondLearned::setup(Ctx& c, const double* u, const double* inv_dt)
{
	if (!feat) {
		DGX_HIP_CHECK(hipMalloc(&feat, sizeof(float) * (size_t)c.E * mlp->nf));
		DGX_HIP_CHECK(hipMalloc(&sigma, sizeof(float) * (size_t)c.E));
	}
	// inference runs on the solver's stream; the model keeps its own stream for training calls
	const hipStream_t saved = mlp->s;
	mlp->s = c.stream;
	hipError_t err = launch_features(c, u, inv_dt, feat, mlp->nf, sigma);
	if (err == hipSuccess) err = mlp_forward(mlp, feat, c.E);
	mlp->s = saved;
	return err;
}

Precond* make_learned_precond(Ctx& c)
{
	if (!c.mlp || c.mlp->nb != c.Np * c.nv || c.mlp->Np != c.Np) return nullptr;
	PrecondLearned* p = new PrecondLearned();
	p->mlp = c.mlp;
	return p;
}

static uint64_t splitmix64(uint64_t& s)
{
	uint64_t z = (s += 0x9E3779B97F4A7C15ull);
	z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
	z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
	return z ^ (z >> 31);
}

}  // namespace dgx

extern "C" {

dgx_status dgx_mlp_create(dgx_mlp** out, int kind, int nb, int Np, int hidden, int rank, unsigned long long seed)
{
	if (!out || hidden < 16 || hidden > 1024) return DGX_ERR_ARG;
	// 2-D Euler blocks: nv = 4 variables, p = 2 (Np = 9) or p = 3 (Np = 16)
	if (!((nb == 64 && Np == 16) || (nb == 36 && Np == 9))) return DGX_ERR_ARG;
	if (!((kind == DGX_MLP_LOWRANK && rank == 8) || (kind == DGX_MLP_KRON && (rank == 4 || rank == 8))))
		return DGX_ERR_ARG;
	const int nv = nb / Np;
	dgx_mlp* m = new dgx_mlp();
	m->kind = kind;
	m->nb = nb;
	m->Np = Np;
	m->rank = rank;
	m->nhid = hidden;
	m->nf = ((nb + Np + 1) + 15) / 16 * 16;
	m->nout = (kind == DGX_MLP_LOWRANK) ? nb + 2 * nb * rank : rank * (nv * nv + Np * Np);
	const size_t sizes[6] = { (size_t)m->nhid * m->nf, (size_t)m->nhid, (size_t)m->nhid * m->nhid, (size_t)m->nhid,
	                          (size_t)m->nout * m->nhid, (size_t)m->nout };
	size_t acc = 0;
	for (int i = 0; i < 6; ++i) { m->off[i] = acc; acc += sizes[i]; }
	m->nparam = acc;
	std::vector<float> w(acc, 0.f);
	uint64_t st = seed ? seed : 20261202ull;
	auto uni = [&](float a) { return (float)(((dgx::splitmix64(st) >> 11) * (1.0 / 9007199254740992.0)) * 2.0 - 1.0) * a; };
	const int fan[3][2] = { { m->nf, m->nhid }, { m->nhid, m->nhid }, { m->nhid, m->nout } };
	for (int l = 0; l < 3; ++l) {
		const float a = std::sqrt(6.0f / (fan[l][0] + fan[l][1])) * (l == 2 ? 0.1f : 1.0f);
		for (size_t i = 0; i < sizes[2 * l]; ++i) w[m->off[2 * l] + i] = uni(a);
	}
	// start from the (negative) scaled identity P = -sigma I
	if (kind == DGX_MLP_LOWRANK) {
		for (int i = 0; i < nb; ++i) w[m->off[5] + i] = -1.0f;
	} else {
		for (int a = 0; a < nv; ++a) w[m->off[5] + a * nv + a] = -1.0f;                         // S_0 = -I
		for (int i = 0; i < Np; ++i) w[m->off[5] + rank * nv * nv + i * Np + i] = 1.0f;          // Q_0 = I
	}
	if (hipMalloc(&m->w, sizeof(float) * acc) != hipSuccess || hipMalloc(&m->wb, sizeof(float) * acc) != hipSuccess ||
	    hipMalloc(&m->gw, sizeof(float) * acc) != hipSuccess || hipMalloc(&m->am, sizeof(float) * acc) != hipSuccess ||
	    hipMalloc(&m->av, sizeof(float) * acc) != hipSuccess) {
		dgx_mlp_destroy(m);
		return DGX_ERR_HIP;
	}
	std::vector<float> z(acc, 0.f);
	if (hipMemcpy(m->w, w.data(), sizeof(float) * acc, hipMemcpyHostToDevice) != hipSuccess ||
	    hipMemcpy(m->am, z.data(), sizeof(float) * acc, hipMemcpyHostToDevice) != hipSuccess ||
	    hipMemcpy(m->av, z.data(), sizeof(float) * acc, hipMemcpyHostToDevice) != hipSuccess ||
	    dgx::mlp_sync_bf16(m) != hipSuccess || hipStreamSynchronize(m->s) != hipSuccess) {
		dgx_mlp_destroy(m);
		return DGX_ERR_HIP;
	}
	*out = m;
	return DGX_OK;
}

dgx_status dgx_mlp_destroy(dgx_mlp* m)
{
	if (!m) return DGX_OK;
	dgx::mlp_free_work(m);
	for (float* p : { m->w, m->wb, m->gw, m->am, m->av })
		if (p) (void)hipFree(p);
	delete m;
	return DGX_OK;
}

dgx_status dgx_mlp_sizes(const dgx_mlp* m, int* nf, int* nout, long long* nparam)
{
	if (!m) return DGX_ERR_ARG;
	if (nf) *nf = m->nf;
	if (nout) *nout = m->nout;
	if (nparam) *nparam = (long long)m->nparam;
	return DGX_OK;
}

dgx_status dgx_mlp_get_params(dgx_mlp* m, float* host)
{
	if (!m || !host) return DGX_ERR_ARG;
	// on the model's stream: the training kernels that update m->w run there
	if (hipMemcpyAsync(host, m->w, sizeof(float) * m->nparam, hipMemcpyDeviceToHost, m->s) != hipSuccess ||
	    hipStreamSynchronize(m->s) != hipSuccess)
		return DGX_ERR_HIP;
	return DGX_OK;
}

dgx_status dgx_mlp_set_params(dgx_mlp* m, const float* host)
{
	if (!m || !host) return DGX_ERR_ARG;
	if (hipMemcpyAsync(m->w, host, sizeof(float) * m->nparam, hipMemcpyHostToDevice, m->s) != hipSuccess) return DGX_ERR_HIP;
	if (dgx::mlp_sync_bf16(m) != hipSuccess || hipStreamSynchronize(m->s) != hipSuccess) return DGX_ERR_HIP;
	return DGX_OK;
}

dgx_status dgx_mlp_features(dgx_ctx* h, const dgx_mlp* m, const double* u, const double* inv_dt, float* feat,
                            float* sigma)
{
	if (!h || !m || !u || !inv_dt || !feat || !sigma) return DGX_ERR_ARG;
	if (!h->c.mesh_ready) return h->c.hp ? DGX_ERR_UNSUPPORTED : DGX_ERR_NO_MESH;
	if (m->nb != h->c.Np * h->c.nv || m->Np != h->c.Np) return DGX_ERR_ARG;
	return dgx::launch_features(h->c, u, inv_dt, feat, m->nf, sigma) == hipSuccess ? DGX_OK : DGX_ERR_HIP;
}

dgx_status dgx_mlp_loss_grad(dgx_mlp* m, const float* feat, const float* sigma, const double* blocks, int B,
                             double* loss, float* grad_host)
{
	if (!m || !feat || !blocks || B <= 0) return DGX_ERR_ARG;
	if (dgx::mlp_forward(m, feat, B) != hipSuccess) return DGX_ERR_HIP;
	if (dgx::mlp_loss(m, sigma, blocks, B, loss, 1.0f / B, grad_host != nullptr) != hipSuccess) return DGX_ERR_HIP;
	if (grad_host) {
		if (dgx::mlp_backward(m, feat, B) != hipSuccess) return DGX_ERR_HIP;
		if (hipMemcpyAsync(grad_host, m->gw, sizeof(float) * m->nparam, hipMemcpyDeviceToHost, m->s) != hipSuccess ||
		    hipStreamSynchronize(m->s) != hipSuccess)
			return DGX_ERR_HIP;
	}
	return DGX_OK;
}

dgx_status dgx_mlp_train(dgx_mlp* m, const float* feat, const float* sigma, const double* blocks, long long n,
                         int epochs, int batch, float lr, double* loss)
{
	if (!m || !feat || !blocks || n <= 0 || epochs < 0 || batch <= 0 || !(lr > 0.f)) return DGX_ERR_ARG;
	const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
	const long long nbatch = (n + batch - 1) / batch;
	// the closing full-set loss runs in chunks of at least kLossChunk samples: work space for them from the start
	constexpr long long kLossChunk = 2048;
	const long long chunk = std::min<long long>(n, std::max<long long>(batch, kLossChunk));
	if (dgx::mlp_reserve(m, (int)std::min<long long>(n, loss ? chunk : batch)) != hipSuccess) return DGX_ERR_HIP;
	std::vector<long long> order(nbatch);
	for (long long i = 0; i < nbatch; ++i) order[i] = i;
	uint64_t rs = 0x5EEDull + (uint64_t)m->step;
	for (int ep = 0; ep < epochs; ++ep) {
		// visit the mini-batches (contiguous runs of samples) in a fresh seeded order each epoch
		for (long long i = nbatch - 1; i > 0; --i) {
			const long long j = (long long)(dgx::splitmix64(rs) % (uint64_t)(i + 1));
			const long long t = order[i];
			order[i] = order[j];
			order[j] = t;
		}
		for (long long oi = 0; oi < nbatch; ++oi) {
			const long long bi = order[oi];
			const long long s0 = bi * batch;
			const int B = (int)((s0 + batch <= n) ? batch : n - s0);
			const float* X = feat + (size_t)s0 * m->nf;
			const float* sg = sigma ? sigma + s0 : nullptr;
			const double* A = blocks + (size_t)s0 * m->nb * m->nb;
			if (dgx::mlp_forward(m, X, B) != hipSuccess) return DGX_ERR_HIP;
			if (dgx::mlp_loss(m, sg, A, B, nullptr, 1.0f / B, true) != hipSuccess) return DGX_ERR_HIP;
			if (dgx::mlp_backward(m, X, B) != hipSuccess) return DGX_ERR_HIP;
			++m->step;
			const float c1 = 1.f - std::pow(b1, (float)m->step), c2 = 1.f - std::pow(b2, (float)m->step);
			hipLaunchKernelGGL(dgx::k_adam, dim3(dgx::gridn(m->nparam)), dim3(256), 0, m->s, m->w, m->gw, m->am, m->av, m->wb,
			                   m->nparam, lr, b1, b2, c1, c2, eps);
			if (hipGetLastError() != hipSuccess) return DGX_ERR_HIP;
		}
	}
	if (loss) {
		// the per-sample losses come back in one copy
		if (m->lall_cap < n) {
			if (m->lall) (void)hipFree(m->lall);
			m->lall = nullptr;
			m->lall_cap = 0;
			if (hipMalloc(&m->lall, sizeof(double) * (size_t)n) != hipSuccess) return DGX_ERR_HIP;
			m->lall_cap = n;
		}
		bool ok = true;
		for (long long s0 = 0; s0 < n && ok; s0 += chunk) {
			const int B = (int)std::min<long long>(chunk, n - s0);
			ok = dgx::mlp_forward(m, feat + (size_t)s0 * m->nf, B) == hipSuccess &&
			     dgx::mlp_loss(m, sigma ? sigma + s0 : nullptr, blocks + (size_t)s0 * m->nb * m->nb, B, nullptr, 1.0f, false,
			                   m->lall + s0) == hipSuccess;
		}
		std::vector<double> host(ok ? (size_t)n : 0);
		ok = ok && hipMemcpyAsync(host.data(), m->lall, sizeof(double) * (size_t)n, hipMemcpyDeviceToHost, m->s) == hipSuccess;
		ok = (hipStreamSynchronize(m->s) == hipSuccess) && ok;
		if (!ok) return DGX_ERR_HIP;
		double tot = 0.0;
		for (double x : host) tot += x;
		*loss = tot / n;
	}
	return hipStreamSynchronize(m->s) == hipSuccess ? DGX_OK : DGX_ERR_HIP;
}

dgx_status dgx_mlp_predict(dgx_mlp* m, const float* feat, int B, float* out)
{
	if (!m || !feat || !out || B <= 0) return DGX_ERR_ARG;
	return dgx::mlp_forward(m, feat, B, out) == hipSuccess ? DGX_OK : DGX_ERR_HIP;
}

dgx_status dgx_attach_mlp(dgx_ctx* h, dgx_mlp* m)
{
	if (!h) return DGX_ERR_ARG;
	h->c.mlp = m;
	return DGX_OK;
}

}  // extern "C"
