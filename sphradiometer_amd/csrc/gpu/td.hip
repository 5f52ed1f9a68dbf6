/*
 * Time-domain correlator (correlator.c:325-400, 611-673, 820-858,
 * 967-984 of the reference) with the integration on the GPU.
 *
 * The reference integrates sample by sample: for each output sample t it
 * dots the two delay-tap projections with the series (sample_a(t) =
 * sum_k proj_a[k] a[t + k], sample_b likewise), multiplies the two polar
 * series (sh_series_product) and adds window[t] times the product to
 * power_1d.  As functions of x = cos theta, sample_a(t)(x) =
 * sum_k T^a_k(x) a[t + k] with T^a_k the synthesis of proj_a[k], and the
 * product's coefficient d is 2 pi int sample_a sample_b Pbar_d0 dx, which a
 * Gauss-Legendre rule of n_q = (a + b + P) / 2 + 1 nodes integrates
 * exactly.  Summed over t:
 *   power_1d[d] = sum_q 2 pi w_q Pbar_d0(x_q) U_q,
 *   U_q = sum_{k,k'} T^a_k(x_q) C[k][k'] T^b_k'(x_q),
 *   C[k][k'] = sum_t window[t] a[t + k] b[t + k'],
 * the same arithmetic up to rounding, with the per-sample work folded into
 * the windowed correlation matrix C (n_p x n_p, a GEMM over t with the
 * Hankel operands generated from the series in the tile loader, float64
 * MFMA), then Y = C T^b and its bilinear form with T^a in one pass
 * (k_td_yu) and the d sums (k_td_pw).  For a window that is flat over
 * most of the series, C comes from the samples where the window changes
 * (the same GEMM over that support gives the diagonal differences of C),
 * its first row and column, and a sum along each diagonal.
 * The rotation to the baseline direction and the network average run on
 * the device (k_rotsum) from the rows D^l_{0 m'} of the plan's rotation
 * plan, uploaded once when the plan is made; a call copies back only
 * power_1d and the rotated (or summed) series.
 *
 * The plan keeps the reference's struct (proj_a, proj_b, sample_a,
 * sample_b, product, power_1d, product_plan, rotation_plan) as the first
 * member of a larger allocation that holds the device tables.  After an
 * integration power_1d holds the axially symmetric power, as in the
 * reference; sample_a, sample_b and product are not updated.
 */
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <sphradiometer/correlator.h>
#include <sphradiometer/projection.h>
#include <sphradiometer/sh_series.h>
#include <sphradiometer/sphradiometer_gpu.h>
#include "../sphr_internal.h"
#include "kernels.h"
#include "runtime.h"

struct td_plan {
	struct correlator_plan_td pub;	/* the reference layout, first */
	int np, nq, P;
	double *d_Ta, *d_Tb;		/* [np][nq]: tap projections at the product nodes */
	double *d_WP;			/* [nq][P + 1]: 2 pi w_q Pbar_d0(x_q) */
	/* per-call device buffers, grown as needed */
	size_t cap_a, cap_b, cap_w, cap_part;
	double *d_a, *d_b, *d_w, *d_part, *d_C;
	double *d_U;			/* [ceil(np / 16)][nq]: partial bilinear forms */
	double *d_powc;			/* power_1d as P + 1 complex (imaginary parts 0) */
	double *d_rows;			/* (P + 1)^2 complex: D^l_{0 m'} of the rotation plan */
	size_t cap_out, cap_sv, cap_edge;
	double *d_sv;			/* a call's window differences on their support, baseline by baseline */
	double *d_edge;			/* first row and column of C, by chunk */
	double *d_out;			/* rotated series (or a network's partial sums) */
	/* a network's series and windows (kept on its first plan) */
	size_t cap_nts, cap_nws, cap_npow;
	double *d_nts, *d_nws, *d_npow;	/* npow: every baseline's power */
};

namespace {

/*
 * One baseline of a call.  The baselines of a network go through each
 * kernel together, blockIdx.z the baseline (at most TD_SET per launch): the
 * launches of one baseline leave the chip nearly idle, and one after the
 * other with a copy of each window's differences between them they were
 * 300 of the 780 us of three baselines over 65536 samples; together 50.
 */
#define TD_SET 8
struct td_item {
	const double *a, *b;	/* the series */
	const double *w;	/* the window, or NULL where sv describes it */
	const double *sv;	/* its nnz first differences: values, offsets, running sums */
	const double *Ta, *Tb, *WP;
	double *part, *edge, *C, *U, *pow;
	int sparse, nnz, nt, np, nq, P;
	int nk, nz, tpz, tiles;	/* correlation: terms, K splits, terms per split, tiles per side */
	int nch, spc;		/* first row and column: chunks, samples per chunk */
};

struct td_set {
	struct td_item it[TD_SET];
};

/*
 * partial[z][k][k'] = sum_{t in split z} w[t] a[s_t + k] b[s_t + k'],
 * k, k' < np, with s_t = t or, for a gathered support, s_t = sidx[t]
 * (reads at or past na, the series length, count as 0): 64 x 64 tiles of 4 waves (32 x 32 each) on
 * v_mfma_f64_16x16x4f64, t in chunks of TD_KC through LDS, the operands read
 * from the series (Hankel structure) with the next chunk's loads in flight
 * during the current chunk's MFMAs.  MFMA layout: A[i][k] in lane
 * i + 16 k, B[k][j] in lane j + 16 k, accumulator element e of lane
 * j + 16 q holds D[q + 4 e][j].
 */
#define TD_TILE 64
#define TD_KC 32
/* operand elements per thread per chunk */
#define TD_LR (TD_KC * TD_TILE / 256)
/* output samples per K split */
#define TD_TSPLIT 1024

__global__ void __launch_bounds__(256) k_td_corr(const struct td_set set, int na)
{
	const struct td_item &I = set.it[blockIdx.z];
	const int tiles = I.tiles, np = I.np, nt = I.nk, tpz = I.tpz;
	if((int) blockIdx.x >= tiles * tiles * I.nz)
		return;
	const double *__restrict__ a = I.a, *__restrict__ b = I.b, *__restrict__ w = I.sparse ? I.sv : I.w, *__restrict__ sidx = I.sparse ? I.sv + I.nnz : NULL;
	typedef double v4 __attribute__((ext_vector_type(4)));
	__shared__ double sA[TD_KC][TD_TILE + 4];	/* [t][k] */
	__shared__ double sB[TD_KC][TD_TILE + 4];	/* [t][k'] */
	const int tile = blockIdx.x % (tiles * tiles), z = blockIdx.x / (tiles * tiles);
	const int m0 = (tile % tiles) * TD_TILE, n0 = (tile / tiles) * TD_TILE;
	const int t0 = z * tpz, t1 = t0 + tpz < nt ? t0 + tpz : nt;
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int li = lane & 15, lk = lane >> 4;
	const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
	double ra[TD_LR], rb[TD_LR];
	auto load = [&](int c0) {
#pragma unroll
		for(int r = 0; r < TD_LR; r++) {
			const int e = tid + 256 * r;
			const int t = c0 + e / TD_TILE, k = e % TD_TILE;
			const bool ok = t < t1;
			/* sample offset of term t: t itself, or the t-th entry of a
			 * gathered support */
			const int st = sidx && ok ? (int) sidx[t] : t;
			ra[r] = ok && m0 + k < np && st + m0 + k < na ? w[t] * a[st + m0 + k] : 0.0;
			rb[r] = ok && n0 + k < np && st + n0 + k < na ? b[st + n0 + k] : 0.0;
		}
	};
	v4 acc[2][2];
#pragma unroll
	for(int i = 0; i < 2; i++)
#pragma unroll
		for(int j = 0; j < 2; j++)
			acc[i][j] = (v4) 0;
	if(t0 < t1)
		load(t0);
	for(int c0 = t0; c0 < t1; c0 += TD_KC) {
#pragma unroll
		for(int r = 0; r < TD_LR; r++) {
			const int e = tid + 256 * r;
			sA[e / TD_TILE][e % TD_TILE] = ra[r];
			sB[e / TD_TILE][e % TD_TILE] = rb[r];
		}
		__syncthreads();
		if(c0 + TD_KC < t1)
			load(c0 + TD_KC);
#pragma unroll
		for(int ks = 0; ks < TD_KC; ks += 4) {
			double af[2], bf[2];
#pragma unroll
			for(int i = 0; i < 2; i++)
				af[i] = sA[ks + lk][wm + 16 * i + li];
#pragma unroll
			for(int j = 0; j < 2; j++)
				bf[j] = sB[ks + lk][wn + 16 * j + li];
#pragma unroll
			for(int i = 0; i < 2; i++)
#pragma unroll
				for(int j = 0; j < 2; j++)
					acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[i], bf[j], acc[i][j], 0, 0, 0);
		}
		__syncthreads();
	}
	/* a single split is C itself */
	double *P = I.nz == 1 ? I.C : I.part + (size_t) z * np * np;
#pragma unroll
	for(int i = 0; i < 2; i++)
#pragma unroll
		for(int j = 0; j < 2; j++) {
			const int c = n0 + wn + 16 * j + li;
			if(c >= np)
				continue;
#pragma unroll
			for(int e = 0; e < 4; e++) {
				const int r = m0 + wm + 16 * i + lk + 4 * e;
				if(r < np)
					P[(size_t) r * np + c] = acc[i][j][e];
			}
		}
}

/* C = sum_z partial[z] where there are several */
__global__ void k_td_reduce(const struct td_set set)
{
	const struct td_item &I = set.it[blockIdx.z];
	const long i = (long) blockIdx.x * blockDim.x + threadIdx.x, n = (long) I.np * I.np;
	if(i >= n || I.nz == 1)
		return;
	double s = 0.0;
#pragma unroll 4
	for(int z = 0; z < I.nz; z++)
		s += I.part[(size_t) z * n + i];
	I.C[i] = s;
}

/*
 * part[c][j] = sum_{t in chunk c} w[t] a[t] b[t + j] and part[c][np + j] =
 * sum_{t in chunk c} w[t] a[t + j] b[t], j < np (the first row and column
 * of C, summed over the chunks by k_td_diag).  A workgroup takes a chunk
 * and TD_EJ offsets j, TD_EC samples at a time through LDS: each wave a
 * quarter of the samples, each lane four consecutive j, whose 2 x 4 shifted
 * samples slide through its registers, two LDS reads for eight
 * multiply-adds (with one j per thread the reads bounded it: three
 * baselines over 65536 samples 81 + 48 us with the sum over the chunks,
 * now 13, and the sum 4 of k_td_diag's 9).  The shifted samples lie with one double of padding after every
 * four (lanes four apart then read different banks).  The window is rebuilt
 * where it is staged from its differences: w[t] = -sum_{s <= t} v[s].
 */
#define TD_EC 256
#define TD_EJ 256
/* most chunks of a baseline: a longer series has longer chunks */
#define TD_NCH_MAX 1024
#define TD_EDGE_NP_MAX 1024
__global__ void __launch_bounds__(256) k_td_edge(const struct td_set set, int n)
{
	constexpr int NY = TD_EC + TD_EJ + 4;
	__shared__ double wa[TD_EC], wb[TD_EC], ya[NY + NY / 4], yb[NY + NY / 4], red[2][4][TD_EJ];
	const struct td_item &I = set.it[blockIdx.z];
	const int nt = I.nt, np = I.np, nnz = I.nnz, j0 = blockIdx.y * TD_EJ;
	if(!I.sparse || (int) blockIdx.x >= I.nch || j0 >= np)
		return;
	const double *__restrict__ a = I.a, *__restrict__ b = I.b, *__restrict__ sidx = I.sv + nnz, *__restrict__ cum = I.sv + 2 * (size_t) nnz;
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int c0 = blockIdx.x * I.spc, c1 = c0 + I.spc < nt ? c0 + I.spc : nt;
	double r[4] = { 0.0, 0.0, 0.0, 0.0 }, c[4] = { 0.0, 0.0, 0.0, 0.0 };
	for(int t0 = c0; t0 < c1; t0 += TD_EC) {
		__syncthreads();
		for(int i = tid; i < NY; i += 256) {
			const int t = t0 + j0 + i;
			ya[i + (i >> 2)] = t < n ? a[t] : 0.0;
			yb[i + (i >> 2)] = t < n ? b[t] : 0.0;
		}
		{
			const int t = t0 + tid;
			double x = 0.0, y = 0.0;
			if(t < c1) {
				int lo = 0, hi = nnz;
				while(lo < hi) {
					const int mid = (lo + hi) >> 1;
					if(sidx[mid] <= (double) t)
						lo = mid + 1;
					else
						hi = mid;
				}
				const double w = lo ? -cum[lo - 1] : 0.0;
				x = w * a[t];
				y = w * b[t];
			}
			wa[tid] = x;
			wb[tid] = y;
		}
		__syncthreads();
		/* samples t0 + s, s = 64 wave + ..: y index 4 lane + s + (0..3) */
		const int s0 = 64 * wave, y0 = 5 * lane + (s0 + (s0 >> 2));
		double va[8], vb[8];
#pragma unroll
		for(int i = 0; i < 4; i++) {
			va[i] = ya[y0 + i];
			vb[i] = yb[y0 + i];
		}
#pragma unroll 4
		for(int s = 0; s < 64; s += 4) {
#pragma unroll
			for(int i = 0; i < 4; i++) {
				va[4 + i] = ya[y0 + s / 4 * 5 + 5 + i];
				vb[4 + i] = yb[y0 + s / 4 * 5 + 5 + i];
			}
#pragma unroll
			for(int u = 0; u < 4; u++) {
				const double x = wa[s0 + s + u], y = wb[s0 + s + u];
#pragma unroll
				for(int i = 0; i < 4; i++) {
					r[i] = fma(x, vb[u + i], r[i]);
					c[i] = fma(y, va[u + i], c[i]);
				}
			}
#pragma unroll
			for(int i = 0; i < 4; i++) {
				va[i] = va[4 + i];
				vb[i] = vb[4 + i];
			}
		}
	}
#pragma unroll
	for(int i = 0; i < 4; i++) {
		red[0][wave][4 * lane + i] = r[i];
		red[1][wave][4 * lane + i] = c[i];
	}
	__syncthreads();
	if(j0 + tid < np) {
		double *o = I.edge + (size_t) blockIdx.x * 2 * np + j0 + tid;
		o[0] = (red[0][0][tid] + red[0][1][tid]) + (red[0][2][tid] + red[0][3][tid]);
		o[np] = (red[1][0][tid] + red[1][1][tid]) + (red[1][2][tid] + red[1][3][tid]);
	}
}

/* C from its first row and column (the chunk sums in edge) and the diagonal
 * differences D (in C on entry): C[k + 1][k' + 1] = C[k][k'] + D[k][k'].
 * One wave per diagonal k' - k: the lanes sum the chunks of its first
 * element, each lane sums a segment of D, a scan over the lanes gives each
 * segment's starting value, and the lanes then write their segments. */
__global__ void __launch_bounds__(256) k_td_diag(const struct td_set set)
{
	const struct td_item &I = set.it[blockIdx.z];
	const int np = I.np;
	const int lane = threadIdx.x & 63;
	const int d = (int) (blockIdx.x * 4 + (threadIdx.x >> 6)) - (np - 1);
	if(!I.sparse || d > np - 1)
		return;
	double *__restrict__ X = I.C;
	const double *__restrict__ edge = I.edge + (d >= 0 ? d : np - d);
	double e0 = 0.0;
#pragma unroll 4
	for(int c = lane; c < I.nch; c += 64)
		e0 += edge[(size_t) c * 2 * np];
	for(int o = 32; o; o >>= 1)
		e0 += __shfl_xor(e0, o);
	const int k0 = d >= 0 ? 0 : -d, kp0 = d >= 0 ? d : 0;
	const int len = np - (d >= 0 ? d : -d);
	const int seg = (len + 63) / 64, b0 = lane * seg, b1 = b0 + seg < len ? b0 + seg : len;
	const size_t step = (size_t) np + 1, base = (size_t) k0 * np + kp0;
	double sum = 0.0;
	for(int e = b0; e < b1; e++)
		sum += X[base + e * step];
	/* exclusive scan of the segment sums over the wave */
	double incl = sum;
	for(int o = 1; o < 64; o <<= 1) {
		const double u = __shfl_up(incl, o);
		if(lane >= o)
			incl += u;
	}
	double c = e0 + (incl - sum);
	for(int e = b0; e < b1; e++) {
		const double x = X[base + e * step];
		X[base + e * step] = c;
		c += x;
	}
}

/*
 * Upart[kb][q] = sum_{k in block kb} Ta[k][q] sum_k' C[k][k'] Tb[k'][q]:
 * Y = C Tb and its bilinear form with Ta in one pass, 16 k (block kb) by
 * 16 q per workgroup on v_mfma_f64_16x16x4f64, each of the four waves a
 * quarter of the k', their Y never added up: the form is linear in Y.
 * Bound by the latency of its operand loads (L2): many small tiles, eight
 * loads in flight per lane; one thread per (4 k, q) was a chain of 175
 * loads, 25 us a baseline at 233 taps and 351 nodes, now 11 for three.
 * Loads are clamped into the matrices, terms past the end multiply by 0.
 */
/* the product rule's node count that k_td_pw's LDS holds */
#define TD_NQ_MAX 7680
__global__ void __launch_bounds__(256) k_td_yu(const struct td_set set)
{
	typedef double v4 __attribute__((ext_vector_type(4)));
	__shared__ double red[4][16];
	const struct td_item &I = set.it[blockIdx.z];
	const int np = I.np, nq = I.nq, q0 = blockIdx.x * 16, kb = blockIdx.y, k0 = kb * 16;
	if(q0 >= nq || k0 >= np)
		return;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
	const int q = q0 + li < nq ? q0 + li : nq - 1, ka = k0 + li < np ? k0 + li : np - 1;
	const int per = (np + 15) / 16 * 4, cb = wave * per, ce = cb + per < np ? cb + per : np;
	const double *__restrict__ A = I.C + (size_t) ka * np, *__restrict__ B = I.Tb + q;
	v4 acc = (v4) 0;
	for(int c0 = cb; c0 < ce; c0 += 16) {
		double af[4], bf[4];
#pragma unroll
		for(int i = 0; i < 4; i++) {
			const int c = c0 + 4 * i + lk, cc = c < ce ? c : ce - 1;
			af[i] = A[cc];
			bf[i] = B[(size_t) cc * nq];
			af[i] = c < ce ? af[i] : 0.0;
			bf[i] = c < ce ? bf[i] : 0.0;
		}
#pragma unroll
		for(int i = 0; i < 4; i++)
			acc = __builtin_amdgcn_mfma_f64_16x16x4f64(af[i], bf[i], acc, 0, 0, 0);
	}
	double u = 0.0;
#pragma unroll
	for(int e = 0; e < 4; e++) {
		const int k = k0 + lk + 4 * e;
		const double t = I.Ta[(size_t) (k < np ? k : np - 1) * nq + q];
		u = k < np ? fma(t, acc[e], u) : u;
	}
	u += __shfl_xor(u, 16);
	u += __shfl_xor(u, 32);
	if(lk == 0)
		red[wave][li] = u;
	__syncthreads();
	if(threadIdx.x < 16 && q0 + li < nq)
		I.U[(size_t) kb * nq + q] = (red[0][li] + red[1][li]) + (red[2][li] + red[3][li]);
}

/* power[d] = sum_q U_q WP[q][d] with U_q = sum_kb Upart[kb][q] (stored as
 * the complex power[d] + 0 i): 16 d per workgroup, the q sum split 16
 * ways; every workgroup first sums U into LDS (nq doubles, dynamic).  Both
 * sums are chains of L2 loads, four in flight (14.5 us a baseline, now 8.6
 * for three). */
__global__ void __launch_bounds__(256) k_td_pw(const struct td_set set)
{
	extern __shared__ double Us[];
	__shared__ double red[16][16];
	const struct td_item &I = set.it[blockIdx.z];
	const int nq = I.nq, P = I.P, nkb = (I.np + 15) / 16;
	if((int) blockIdx.x * 16 > P)
		return;
	const double *__restrict__ Upart = I.U, *__restrict__ WP = I.WP;
	for(int q = threadIdx.x; q < nq; q += 256) {
		double u = 0.0;
#pragma unroll 4
		for(int kb = 0; kb < nkb; kb++)
			u += Upart[(size_t) kb * nq + q];
		Us[q] = u;
	}
	__syncthreads();
	const int di = threadIdx.x & 15, qs = threadIdx.x >> 4, d = blockIdx.x * 16 + di, dc = d <= P ? d : P;
	double s = 0.0;
#pragma unroll 4
	for(int q = qs; q < nq; q += 16)
		s = fma(Us[q], WP[(size_t) q * (P + 1) + dc], s);
	red[qs][di] = s;
	__syncthreads();
	if(qs == 0 && d <= P) {
		double t = 0.0;
		for(int g = 0; g < 16; g++)
			t += red[g][di];
		I.pow[2 * d] = t;
		I.pow[2 * d + 1] = 0.0;
	}
}

}	/* namespace */

/* ------------------------------------------------------------- the plan */

static void td_dev_free(struct td_plan *p)
{
	double *b[] = { p->d_Ta, p->d_Tb, p->d_WP, p->d_a, p->d_b, p->d_w, p->d_part, p->d_C, p->d_U, p->d_powc, p->d_rows, p->d_out, p->d_sv, p->d_edge, p->d_nts, p->d_nws, p->d_npow };
	for(unsigned i = 0; i < sizeof(b) / sizeof(b[0]); i++)
		if(b[i])
			(void) hipFree(b[i]);
}

/* correlator_plan_td_new (correlator.c:325-385) */
extern "C" struct correlator_plan_td *correlator_plan_td_new(const struct correlator_baseline *baseline, double delta_t)
{
	if(!baseline || delta_t <= 0. || sphr_gpu_ensure())
		return NULL;
	struct td_plan *p = (struct td_plan *) calloc(1, sizeof(*p));
	gsl_vector *dp = gsl_vector_alloc(3);
	double *R = sh_series_rot_matrix(baseline->theta, baseline->phi);
	double *Ta = NULL, *Tb = NULL, *WP = NULL, *rows = NULL;
	if(!p || !dp || !R)
		goto fail;
	{
		struct correlator_plan_td *t = &p->pub;
		const double D = vector_magnitude(baseline->d);
		const unsigned a_l = projection_matrix_l_max(D / 2, delta_t), b_l = projection_matrix_l_max(D / 2, delta_t);
		unsigned P = correlator_baseline_power_l_max(baseline, delta_t);
		if(P > a_l + b_l)
			P = a_l + b_l;
		t->sample_a = sh_series_new(a_l, 1);
		t->sample_b = sh_series_new(b_l, 1);
		t->product = sh_series_new(P, 1);
		t->power_1d = sh_series_new_zero(P, 1);
		if(!t->sample_a || !t->sample_b || !t->product || !t->power_1d)
			goto fail;
		/* d' = +D/2 z and -D/2 z */
		gsl_vector_set(dp, 0, 0);
		gsl_vector_set(dp, 1, 0);
		gsl_vector_set(dp, 2, +D / 2.);
		t->proj_a = projection_matrix_delay(projection_matrix_n_elements(vector_magnitude(dp), delta_t), a_l, dp, delta_t);
		gsl_vector_set(dp, 2, -D / 2.);
		t->proj_b = projection_matrix_delay(projection_matrix_n_elements(vector_magnitude(dp), delta_t), b_l, dp, delta_t);
		if(!t->proj_a || !t->proj_b)
			goto fail;
		t->product_plan = sh_series_product_plan_new(t->power_1d, t->sample_a, t->sample_b);
		t->rotation_plan = sh_series_rotation_plan_new(t->power_1d, R);
		if(!t->product_plan || !t->rotation_plan)
			goto fail;
		t->baseline = baseline;
		t->delta_t = delta_t;
		t->transient = correlator_transient(t->proj_a, t->proj_b);
		/* device tables on an exact product rule: degree a + b + P */
		/* the correlation kernel reads a[t + k] for t < n - 2 transient,
		 * k < n_p: in range when n_p = 2 transient + 1 (odd tap counts,
		 * projection.c's 2 (int) (60 + r / dt + 1) + 1) */
		if(t->proj_a->n != t->proj_b->n || t->proj_a->n != 2 * t->transient + 1) {
			sphr_set_error("correlator_plan_td_new: tap counts %d, %d with transient %d", t->proj_a->n, t->proj_b->n, t->transient);
			goto fail;
		}
		const int np = t->proj_a->n, nq = (int) ((a_l + b_l + P) / 2 + 1);
		/* k_td_pw holds the nq bilinear forms in LDS */
		if(nq > TD_NQ_MAX) {
			sphr_set_error("correlator_plan_td_new: %d product nodes exceed %d", nq, TD_NQ_MAX);
			goto fail;
		}
		p->np = np;
		p->nq = nq;
		p->P = (int) P;
		Ta = (double *) malloc((size_t) np * nq * sizeof(double));
		Tb = (double *) malloc((size_t) np * nq * sizeof(double));
		WP = (double *) malloc((size_t) nq * (P + 1) * sizeof(double));
		rows = (double *) malloc(2 * (size_t) (P + 1) * (P + 1) * sizeof(double));
		if(!Ta || !Tb || !WP || !rows || sphr_td_tables(t->proj_a, t->proj_b, nq, (int) P, Ta, Tb, WP))
			goto fail;
		sphr_polar_rows((int) P, sphr_rotation_blocks(t->rotation_plan), rows);
		if(sphr_rt_check(hipMalloc(&p->d_Ta, (size_t) np * nq * sizeof(double)), "hipMalloc")
		   || sphr_rt_check(hipMalloc(&p->d_Tb, (size_t) np * nq * sizeof(double)), "hipMalloc")
		   || sphr_rt_check(hipMalloc(&p->d_WP, (size_t) nq * (P + 1) * sizeof(double)), "hipMalloc")
		   || sphr_rt_check(hipMalloc(&p->d_C, (size_t) np * np * sizeof(double)), "hipMalloc")
		   || sphr_rt_check(hipMalloc(&p->d_U, (size_t) ((np + 15) / 16) * nq * sizeof(double)), "hipMalloc")
		   || sphr_rt_check(hipMalloc(&p->d_powc, 2 * (size_t) (P + 1) * sizeof(double)), "hipMalloc")
		   || sphr_rt_check(hipMalloc(&p->d_rows, 2 * (size_t) (P + 1) * (P + 1) * sizeof(double)), "hipMalloc")
		   || sphr_memcpy_htod(p->d_rows, rows, 2 * (size_t) (P + 1) * (P + 1) * sizeof(double))
		   || sphr_memcpy_htod(p->d_Ta, Ta, (size_t) np * nq * sizeof(double))
		   || sphr_memcpy_htod(p->d_Tb, Tb, (size_t) np * nq * sizeof(double))
		   || sphr_memcpy_htod(p->d_WP, WP, (size_t) nq * (P + 1) * sizeof(double)))
			goto fail;
	}
	free(Ta);
	free(Tb);
	free(WP);
	free(rows);
	free(R);
	gsl_vector_free(dp);
	return &p->pub;
fail:
	free(Ta);
	free(Tb);
	free(WP);
	free(rows);
	free(R);
	if(dp)
		gsl_vector_free(dp);
	if(p)
		correlator_plan_td_free(&p->pub);
	return NULL;
}

extern "C" void correlator_plan_td_free(struct correlator_plan_td *plan)
{
	if(!plan)
		return;
	struct td_plan *p = (struct td_plan *) plan;
	sh_series_rotation_plan_free(plan->rotation_plan);
	sh_series_product_plan_free(plan->product_plan);
	sh_series_free(plan->power_1d);
	sh_series_free(plan->product);
	sh_series_free(plan->sample_b);
	sh_series_free(plan->sample_a);
	sh_series_array_free(plan->proj_b);
	sh_series_array_free(plan->proj_a);
	td_dev_free(p);
	free(p);
}

static int grow(double **buf, size_t *cap, size_t need)
{
	if(need <= *cap)
		return 0;
	if(*buf)
		(void) hipFree(*buf);
	*buf = NULL;
	*cap = 0;	/* also where the new buffer cannot be had */
	if(sphr_rt_check(hipMalloc(buf, need * sizeof(double)), "hipMalloc"))
		return -1;
	*cap = need;
	return 0;
}

/* the number of nonzero first differences of the host window hw (nt
 * samples) when the flat-window route applies to a plan of np taps, their
 * offsets in off (room for nt / 2 + 1), else -1.  A flat window is read at
 * the speed of memory: the bits of 64 differences are collected without a
 * branch (a difference that is NaN counts, one of either zero does not), and
 * only blocks with a difference are gone through.  Counting them in the
 * blocks cost up to 18 of the 265 us of 16 s of three sites, by where the
 * linker had put the loop. */
static int td_window_nnz(const double *hw, int nt, int np, int *off)
{
	if(!hw || nt < 2 || np < 2 || np > TD_EDGE_NP_MAX)
		return -1;
	const int most = nt / 2;
	int nnz = 0;
	if(hw[0] != 0.0)
		off[nnz++] = 0;
	for(int s0 = 1; s0 < nt; s0 += 64) {
		const int s1 = s0 + 64 < nt ? s0 + 64 : nt;
		uint64_t bits = 0;
		for(int s = s0; s < s1; s++) {
			const double d = hw[s - 1] - hw[s];
			uint64_t u;
			memcpy(&u, &d, sizeof(u));
			bits |= u;
		}
		if(!(bits << 1))
			continue;
		if(nnz + (s1 - s0) <= most)
			for(int s = s0; s < s1; s++) {
				off[nnz] = s;
				nnz += hw[s - 1] - hw[s] != 0.0;
			}
		else
			for(int s = s0; s < s1; s++)
				if(hw[s - 1] - hw[s] != 0.0) {
					if(nnz == most)
						return -1;
					off[nnz++] = s;
				}
	}
	if(hw[nt - 1] != 0.0) {
		if(nnz + 1 > most)
			return -1;
		off[nnz++] = nt;
	}
	return nnz;
}

/* host memory on its way to the device: through a pinned buffer where the
 * call fits in one of TD_PIN_MAX bytes (the copies then run behind the
 * host's work: with the scan above 451 -> 274 us for 16 s of three sites),
 * otherwise copied directly.  The buffer belongs to the
 * runtime, is used under the drop-in lock and is free again once the call
 * has waited for its stream. */
#define TD_PIN_MAX ((size_t) 16 << 20)
struct td_stage {
	char *p;
	size_t at, cap;
};

static struct td_stage td_stage_new(size_t bytes)
{
	struct td_stage g = { bytes <= TD_PIN_MAX ? (char *) sphr_rt_pinned(0, bytes) : NULL, 0, bytes };
	return g;
}

static int td_upload(struct td_stage *g, double *dst, const double *src, size_t n)
{
	const size_t bytes = n * sizeof(double);
	if(!g->p || g->at + bytes > g->cap)
		return sphr_memcpy_htod(dst, src, bytes);
	memcpy(g->p + g->at, src, bytes);
	const int rc = sphr_rt_check(hipMemcpyAsync(dst, g->p + g->at, bytes, hipMemcpyHostToDevice, sphr_rt_stream()), "hipMemcpy HtoD");
	g->at += bytes;
	return rc ? -1 : 0;
}

/* one baseline of td_power_dev: its plan, device copies of its series,
 * its window in host memory and, where nnz (td_window_nnz) is -1, on the
 * device; pow takes P + 1 complex values */
struct td_call {
	struct td_plan *p;
	const double *a, *b, *hw, *w;
	double *pow;
	int nnz;
	const int *off;		/* the differences' offsets */
};

/*
 * The powers of m baselines over n samples.
 *
 * With v[s] = w[s - 1] - w[s] for s = 0..nt (w = 0 outside [0, nt)),
 * C[k + 1][k' + 1] - C[k][k'] = sum_s v[s] a[s + k] b[s + k'] exactly.  For
 * windows that are constant over most of the series (the square and
 * Tukey windows of the reference's stitching) v has few nonzeros: the
 * correlation kernel then runs over that support only, and C follows from
 * its first row and column along the diagonals.  The differences of all
 * windows go to the device in one copy, into owner's buffer; the kernels
 * then run back to back.
 */
static int td_power_dev(struct td_call *call, int m, int n, struct td_plan *owner, struct td_stage *stage)
{
	hipStream_t st = sphr_rt_stream();
	size_t nsv = 0;
	for(int k = 0; k < m; k++)
		nsv += call[k].nnz > 0 ? 3 * (size_t) call[k].nnz : 0;
	if(grow(&owner->d_sv, &owner->cap_sv, nsv ? nsv : 1))
		return -1;
	if(nsv) {
		/* values, offsets and running sums of each window's differences */
		double *hv = (double *) malloc(nsv * sizeof(double)), *v = hv;
		if(!hv)
			return -1;
		for(int k = 0; k < m; k++) {
			const double *hw = call[k].hw;
			const int nt = n - 2 * call[k].p->pub.transient, nnz = call[k].nnz;
			if(nnz <= 0)
				continue;
			double run = 0.0;
			for(int e = 0; e < nnz; e++) {
				const int s = call[k].off[e];
				const double x = (s > 0 ? hw[s - 1] : 0.0) - (s < nt ? hw[s] : 0.0);
				run += x;
				v[e] = x;
				v[nnz + e] = (double) s;
				v[2 * nnz + e] = run;
			}
			v += 3 * (size_t) nnz;
		}
		const int rc = td_upload(stage, owner->d_sv, hv, nsv);
		free(hv);
		if(rc)
			return -1;
	}
	const double *sv = owner->d_sv;
	for(int k0 = 0; k0 < m; k0 += TD_SET) {
		const int g = m - k0 < TD_SET ? m - k0 : TD_SET;
		struct td_set set;
		memset(&set, 0, sizeof(set));
		unsigned corr = 0, red = 0, nch = 0, jb = 0, diag = 0, qb = 0, kb = 0, db = 0;
		size_t lds = 0;
		for(int k = 0; k < g; k++) {
			const struct td_call *c = call + k0 + k;
			struct td_plan *p = c->p;
			struct td_item *I = &set.it[k];
			const int np = p->np;
			I->a = c->a;
			I->b = c->b;
			I->w = c->w;
			I->sparse = c->nnz >= 0;
			I->nnz = I->sparse ? c->nnz : 0;
			I->sv = sv;
			sv += 3 * (size_t) I->nnz;
			I->nt = n - 2 * p->pub.transient;
			I->np = np;
			I->nq = p->nq;
			I->P = p->P;
			I->nk = I->sparse ? I->nnz : I->nt;
			/* K splits of about TD_TSPLIT terms, enough workgroups on a
			 * short series; on a long one at most eight workgroups per
			 * CU's worth of splits, each then longer, so the partial sums
			 * (nz np^2 doubles) stay bounded whatever the stream's
			 * length */
			I->tiles = (np + TD_TILE - 1) / TD_TILE;
			int nz = (I->nk + TD_TSPLIT - 1) / TD_TSPLIT;
			const int nz_max = 8 * (sphr_rt_cus() > 0 ? sphr_rt_cus() : 256) / (I->tiles * I->tiles);
			if(nz > nz_max)
				nz = nz_max;
			if(nz < 1)
				nz = 1;
			I->tpz = ((I->nk + nz - 1) / nz + TD_KC - 1) / TD_KC * TD_KC;
			I->nz = I->nk > 0 ? (I->nk + I->tpz - 1) / I->tpz : 1;
			I->spc = ((I->nt + TD_NCH_MAX - 1) / TD_NCH_MAX + TD_EC - 1) / TD_EC * TD_EC;
			I->nch = I->sparse ? (I->nt + I->spc - 1) / I->spc : 0;
			if(grow(&p->d_part, &p->cap_part, I->nz > 1 ? (size_t) I->nz * np * np : 1) || grow(&p->d_edge, &p->cap_edge, (size_t) (I->nch ? I->nch : 1) * 2 * np))
				return -1;
			I->part = p->d_part;
			I->edge = p->d_edge;
			I->C = p->d_C;
			I->U = p->d_U;
			I->pow = c->pow;
			I->Ta = p->d_Ta;
			I->Tb = p->d_Tb;
			I->WP = p->d_WP;
			auto most = [](unsigned &x, unsigned y) { x = y > x ? y : x; };
			most(corr, (unsigned) (I->tiles * I->tiles * I->nz));
			if(I->nz > 1)
				most(red, (unsigned) (((long) np * np + 255) / 256));
			if(I->sparse) {
				most(nch, (unsigned) I->nch);
				most(jb, (unsigned) ((np + TD_EJ - 1) / TD_EJ));
				most(diag, (unsigned) ((2 * np - 1 + 3) / 4));
			}
			most(qb, (unsigned) ((p->nq + 15) / 16));
			most(kb, (unsigned) ((np + 15) / 16));
			most(db, (unsigned) ((p->P + 16) / 16));
			lds = (size_t) p->nq * sizeof(double) > lds ? (size_t) p->nq * sizeof(double) : lds;
		}
		hipLaunchKernelGGL(k_td_corr, dim3(corr, 1, g), dim3(256), 0, st, set, n);
		if(red)
			hipLaunchKernelGGL(k_td_reduce, dim3(red, 1, g), dim3(256), 0, st, set);
		if(nch)
			hipLaunchKernelGGL(k_td_edge, dim3(nch, jb, g), dim3(256), 0, st, set, n);
		if(diag)
			hipLaunchKernelGGL(k_td_diag, dim3(diag, 1, g), dim3(256), 0, st, set);
		hipLaunchKernelGGL(k_td_yu, dim3(qb, kb, g), dim3(256), 0, st, set);
		hipLaunchKernelGGL(k_td_pw, dim3(db, 1, g), dim3(256), lds, st, set);
	}
	return sphr_rt_check(hipGetLastError(), "time-domain correlator") ? -1 : 0;
}

/* the same from host series: copied into the plan's buffers first */
static int td_power_1d(const double *ta, const double *tb, const double *window, int n, struct td_plan *p)
{
	const int nt = n - 2 * p->pub.transient;
	if(grow(&p->d_a, &p->cap_a, (size_t) n) || grow(&p->d_b, &p->cap_b, (size_t) n) || grow(&p->d_w, &p->cap_w, (size_t) (nt > 0 ? nt : 1)))
		return -1;
	int *off = (int *) malloc(((size_t) (nt > 0 ? nt : 0) / 2 + 1) * sizeof(int));
	if(!off)
		return -1;
	const int nnz = td_window_nnz(window, nt, p->np, off);
	struct td_stage stage = td_stage_new((2 * (size_t) n + (nnz < 0 ? (size_t) nt : 3 * (size_t) nnz)) * sizeof(double));
	int rc = td_upload(&stage, p->d_a, ta, (size_t) n) || td_upload(&stage, p->d_b, tb, (size_t) n) || (nt > 0 && nnz < 0 && td_upload(&stage, p->d_w, window, (size_t) nt));
	struct td_call c = { p, p->d_a, p->d_b, window, p->d_w, p->d_powc, nnz, off };
	if(!rc)
		rc = td_power_dev(&c, 1, n, p, &stage);
	free(off);
	return rc ? -1 : 0;
}

/* power_1d of the plan set from its P + 1 complex values */
static void td_set_power(struct td_plan *p, const double *v)
{
	for(int d = 0; d <= p->P; d++)
		sh_series_set(p->pub.power_1d, d, 0, v[2 * d]);
}

/* correlator_baseline_integrate_power_td (correlator.c:648-673) */
extern "C" struct sh_series *correlator_baseline_integrate_power_td(const double *time_series_a, const double *time_series_b, const double *window, int n, struct correlator_plan_td *plan)
{
	if(!plan || !time_series_a || !time_series_b || !window)
		return NULL;
	if(n - 2 * plan->transient < 0)
		return NULL;
	struct td_plan *p = (struct td_plan *) plan;
	const int P = p->P;
	const size_t nsky = (size_t) (P + 1) * (P + 1);
	double *buf = (double *) malloc(2 * (size_t) (P + 1) * sizeof(double));
	struct sh_series *power_2d = sh_series_new(P, 0);
	int rc = !buf || !power_2d;
	pthread_mutex_lock(&sphr_dropin_lock);
	if(!rc)
		rc = td_power_1d(time_series_a, time_series_b, window, n, p) || grow(&p->d_out, &p->cap_out, 2 * nsky);
	if(!rc) {
		const cplx<double> *pw[1] = { (const cplx<double> *) p->d_powc }, *bk[1] = { (const cplx<double> *) p->d_rows };
		const int Lb[1] = { P }, pol[1] = { 1 };
		rc = launch_rotsum(1, pw, Lb, pol, bk, P, 1.0, (cplx<double> *) p->d_out, sphr_rt_stream());
		if(rc)
			sphr_set_error("rotation launch failed");
	}
	if(!rc)
		rc = sphr_memcpy_dtoh(buf, p->d_powc, 2 * (size_t) (P + 1) * sizeof(double));
	if(!rc)
		td_set_power(p, buf);
	if(!rc)
		rc = sphr_memcpy_dtoh(power_2d->coeff, p->d_out, 2 * nsky * sizeof(double));
	if(rc)
		(void) hipStreamSynchronize(sphr_rt_stream());
	pthread_mutex_unlock(&sphr_dropin_lock);
	free(buf);
	if(rc) {
		sh_series_free(power_2d);
		return NULL;
	}
	return power_2d;
}

/* correlator_network_plan_td_new / _free (correlator.c:820-858) */
extern "C" struct correlator_network_plan_td *correlator_network_plan_td_new(struct correlator_network_baselines *baselines, double delta_t)
{
	struct correlator_network_plan_td *n = (struct correlator_network_plan_td *) malloc(sizeof(*n));
	struct correlator_plan_td **plans = baselines ? (struct correlator_plan_td **) calloc(baselines->n_baselines, sizeof(*plans)) : NULL;
	if(!n || !plans) {
		free(n);
		free(plans);
		return NULL;
	}
	for(int i = 0; i < baselines->n_baselines; i++) {
		plans[i] = correlator_plan_td_new(baselines->baselines[i], delta_t);
		if(!plans[i]) {
			while(--i >= 0)
				correlator_plan_td_free(plans[i]);
			free(n);
			free(plans);
			return NULL;
		}
	}
	n->baselines = baselines;
	n->plans = plans;
	return n;
}

extern "C" void correlator_network_plan_td_free(struct correlator_network_plan_td *plan)
{
	if(plan) {
		for(int i = 0; i < plan->baselines->n_baselines; i++)
			correlator_plan_td_free(plan->plans[i]);
		free(plan->plans);
	}
	free(plan);
}

/* the powers (npow doubles, to buf and the plans) and n doubles of the sky:
 * through pinned memory the second half arrives as the host empties the
 * first (16 s of three sites, order 351: 274 us a call; thirds 282, quarters
 * 292, each copy starting 25 us after the last) */
#define TD_PARTS 2
static int td_fetch(struct correlator_network_plan_td *plan, struct td_plan *p0, double *buf, size_t npow, double *sky, size_t n)
{
	hipStream_t st = sphr_rt_stream();
	const size_t bytes = (npow + n) * sizeof(double);
	double *h = bytes <= TD_PIN_MAX ? (double *) sphr_rt_pinned(1, bytes) : NULL;
	hipEvent_t ev[TD_PARTS] = { 0 };
	int rc = 0, np = 0;
	if(!h)
		rc = sphr_memcpy_dtoh(buf, p0->d_npow, npow * sizeof(double)) || (n && sphr_memcpy_dtoh(sky, p0->d_out, n * sizeof(double)));
	else {
		np = n ? TD_PARTS : 1;
		rc = sphr_rt_check(hipMemcpyAsync(h, p0->d_npow, npow * sizeof(double), hipMemcpyDeviceToHost, st), "hipMemcpy DtoH") ? -1 : 0;
		for(int i = 0; i < np && !rc; i++) {
			const size_t a = n * i / np, b = n * (i + 1) / np;
			rc = (b > a && sphr_rt_check(hipMemcpyAsync(h + npow + a, p0->d_out + a, (b - a) * sizeof(double), hipMemcpyDeviceToHost, st), "hipMemcpy DtoH"))
			     || sphr_rt_check(hipEventCreateWithFlags(&ev[i], hipEventDisableTiming), "hipEventCreate") || sphr_rt_check(hipEventRecord(ev[i], st), "hipEventRecord");
		}
		for(int i = 0; i < np && !rc; i++) {
			const size_t a = n * i / np, b = n * (i + 1) / np;
			rc = sphr_rt_check(hipEventSynchronize(ev[i]), "hipEventSynchronize");
			if(!rc && i == 0)
				memcpy(buf, h, npow * sizeof(double));
			if(!rc)
				memcpy(sky + a, h + npow + a, (b - a) * sizeof(double));
		}
		for(int i = 0; i < np; i++)
			if(ev[i])
				(void) hipEventDestroy(ev[i]);
	}
	if(rc)
		return -1;
	const double *v = buf;
	for(int k = 0; k < plan->baselines->n_baselines; v += 2 * (size_t) (((struct td_plan *) plan->plans[k])->P + 1), k++)
		td_set_power((struct td_plan *) plan->plans[k], v);
	return 0;
}

/* correlator_network_integrate_power_td (correlator.c:967-984).  The
 * series go to the device once for all baselines, in the first plan's
 * buffers; each baseline's power stays on the device, and one k_rotsum
 * launch per SPHR_MAX_BASELINES baselines rotates and averages them.  As
 * in the reference (sh_series_add), a sky of lower order than a baseline's
 * power, or a polar sky, fails after the powers are computed. */
extern "C" struct sh_series *correlator_network_integrate_power_td(struct sh_series *sky, double **tseries, int tseries_length, double **windows, struct correlator_network_plan_td *plan)
{
	if(!sky || !tseries || !windows || !plan || !plan->baselines->n_baselines)
		return NULL;
	const int nb = plan->baselines->n_baselines;
	const int n_inst = instrument_array_len(plan->baselines->baselines[0]->instruments);
	int tmax = 0, Pmax = 0;
	size_t npow = 0;
	for(int k = 0; k < nb; k++) {
		const struct td_plan *p = (const struct td_plan *) plan->plans[k];
		npow += 2 * (size_t) (p->P + 1);
		tmax = p->pub.transient > tmax ? p->pub.transient : tmax;
		Pmax = p->P > Pmax ? p->P : Pmax;
	}
	sh_series_zero(sky);
	if(tseries_length - 2 * tmax < 0)
		return NULL;
	const int L = (int) sky->l_max;
	const size_t nsky = (size_t) (L + 1) * (L + 1);
	const int nchunk = (nb + SPHR_MAX_BASELINES - 1) / SPHR_MAX_BASELINES;
	double *buf = (double *) malloc(npow * sizeof(double));
	struct td_call *call = (struct td_call *) calloc(nb, sizeof(*call));
	double *part = nchunk > 1 ? (double *) malloc(2 * nsky * sizeof(double)) : NULL;
	struct td_plan *p0 = (struct td_plan *) plan->plans[0];
	int rc = !buf || !call || (nchunk > 1 && !part);
	pthread_mutex_lock(&sphr_dropin_lock);
	if(!rc)
		rc = grow(&p0->d_nts, &p0->cap_nts, (size_t) n_inst * tseries_length) || grow(&p0->d_nws, &p0->cap_nws, (size_t) nb * tseries_length)
		     || grow(&p0->d_npow, &p0->cap_npow, npow);
	double *dts = p0->d_nts, *dws = p0->d_nws;
	/* windows flat over most of the series are rebuilt on the device from
	 * their differences; the others are copied */
	const size_t ostr = (size_t) tseries_length / 2 + 1;
	int *off = rc ? NULL : (int *) malloc(nb * ostr * sizeof(int));
	size_t at = 0, up = (size_t) n_inst * tseries_length;
	int k = 0;
	if(!rc && !off)
		rc = -1;
	for(int i = 1; i < n_inst && !rc; i++)
		for(int j = 0; j < i; j++, k++) {
			struct td_plan *p = (struct td_plan *) plan->plans[k];
			const int nt = tseries_length - 2 * p->pub.transient;
			const int nnz = td_window_nnz(windows[k], nt, p->np, off + k * ostr);
			const struct td_call c = { p, dts + (size_t) i * tseries_length, dts + (size_t) j * tseries_length, windows[k], dws + (size_t) k * tseries_length, p0->d_npow + at, nnz, off + k * ostr };
			call[k] = c;
			at += 2 * (size_t) (p->P + 1);
			up += nnz < 0 ? (size_t) nt : 3 * (size_t) nnz;
		}
	struct td_stage stage = { NULL, 0, 0 };
	if(!rc)
		stage = td_stage_new(up * sizeof(double));
	for(int i = 0; i < n_inst && !rc; i++)
		rc = td_upload(&stage, dts + (size_t) i * tseries_length, tseries[i], (size_t) tseries_length);
	for(int c = 0; c < k && !rc; c++) {
		const int nt = tseries_length - 2 * call[c].p->pub.transient;
		rc = nt > 0 && call[c].nnz < 0 && td_upload(&stage, dws + (size_t) c * tseries_length, windows[c], (size_t) nt);
	}
	if(!rc)
		rc = td_power_dev(call, k, tseries_length, p0, &stage);
	/* the sky is refused after the powers are set */
	const int refused = sky->polar || L < Pmax;
	if(!rc && !refused)
		rc = grow(&p0->d_out, &p0->cap_out, 2 * nsky * nchunk);
	for(int c = 0; c < nchunk && !rc && !refused; c++) {
		const cplx<double> *pw[SPHR_MAX_BASELINES], *bk[SPHR_MAX_BASELINES];
		int Lb[SPHR_MAX_BASELINES], pol[SPHR_MAX_BASELINES], m = 0;
		for(k = c * SPHR_MAX_BASELINES; k < nb && m < SPHR_MAX_BASELINES; k++, m++) {
			const struct td_plan *p = (const struct td_plan *) plan->plans[k];
			pw[m] = (const cplx<double> *) call[k].pow;
			bk[m] = (const cplx<double> *) p->d_rows;
			Lb[m] = p->P;
			pol[m] = 1;
		}
		rc = launch_rotsum(m, pw, Lb, pol, bk, L, 1.0 / nb, (cplx<double> *) p0->d_out + nsky * c, sphr_rt_stream());
		if(rc)
			sphr_set_error("rotation launch failed");
	}
	if(!rc)
		rc = td_fetch(plan, p0, buf, npow, (double *) sky->coeff, refused ? 0 : 2 * nsky);
	if(!rc && refused)
		rc = -1;
	for(int c = 1; c < nchunk && !rc; c++) {
		rc = sphr_memcpy_dtoh(part, p0->d_out + 2 * nsky * c, 2 * nsky * sizeof(double));
		for(size_t i = 0; !rc && i < 2 * nsky; i++)
			((double *) sky->coeff)[i] += part[i];
	}
	if(rc)
		(void) hipStreamSynchronize(sphr_rt_stream());
	pthread_mutex_unlock(&sphr_dropin_lock);
	free(buf);
	free(off);
	free(call);
	free(part);
	if(rc) {
		sh_series_zero(sky);
		return NULL;
	}
	return sky;
}
