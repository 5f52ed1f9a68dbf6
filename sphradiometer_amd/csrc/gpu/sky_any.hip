/*
 * Sky stage of the batched path in one kernel for any order: K-split
 * partial sums -> a_lm (rotation rows, baseline average, rotate_z) ->
 * Legendre ring sums in LDS -> phi DFT on MFMA -> mesh, for the real skies
 * of real time series (F[r][-m] = conj F[r][m]: only m >= 0 is formed, the
 * meshes are written with a zero imaginary part).  sky_fused.hip is the same
 * stage with the order known to the compiler, for the two orders whose
 * throughput it is tuned for; this one takes its sizes at run time and can
 * split a segment's rings over several workgroups.
 *
 * Workgroup = one segment x a range of ring groups (8 northern rings and
 * their mirrors), 512 threads.  Every part of a segment forms the a_lm it
 * needs (m >= 0; the first part all, which it writes).  Legendre items are
 * (two rings, a): the orders a and L - a, L + 2 recurrence steps each, both
 * mirror rings from the parities of l - m.  The ring sums are the A operand
 * of the phi DFT, row = (north / south, ring of 8), columns (Re, Im) of the
 * even orders, then of the odd ones: with Ev and Od the sums over each,
 * map[k] = Ev + Od and map[k + n / 2] = Ev - Od.  Columns past an order's
 * end are zero in both operands; rows past the last ring and points past the
 * half turn are not stored.
 *
 * What bounds it: latency of its five phases, not bytes or arithmetic.  It
 * replaces two kernels with the full complex ring sums in HBM between them
 * (one lane per ring and order, then a GEMM over 2 (2 L + 1) columns):
 * 333 segments of order 41 in float32 34 + 40 -> 29 us.  512 threads and
 * two workgroups per CU's worth of parts: 256 threads or twice the parts
 * measured 2 % faster to 50 % slower.  The second set of coefficients that
 * SYM forms costs 0-5 % (float64, order 54: 64 segments 36.8 -> 38.6 us, 1000
 * 180.6 -> 179.0) and keeps the meshes at the two kernels' distance from
 * 64-bit sums with exact rows (order 54 2.9e-13; m >= 0 rows alone 3.5e-13).
 */
#include <hip/hip_runtime.h>
#include <string.h>
#include "kernels.h"
#include "runtime.h"

namespace {

#define SA_NT 512
#define SA_US 4			/* recurrence steps per batch of LDS reads */

template <typename T> struct sa_ops;
template <> struct sa_ops<float> {
	typedef float v4 __attribute__((ext_vector_type(4)));
	typedef float2 pair;
	static __device__ inline v4 mma(float a, float b, v4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
	static __device__ inline int row(int q, int e) { return 4 * q + e; }
	static __device__ inline const cplx<float> *rc(const struct synth_tables &tb) { return tb.rc32; }
};
template <> struct sa_ops<double> {
	typedef double v4 __attribute__((ext_vector_type(4)));
	typedef double2 pair;
	static __device__ inline v4 mma(double a, double b, v4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
	static __device__ inline int row(int q, int e) { return q + 4 * e; }
	static __device__ inline const cplx<double> *rc(const struct synth_tables &tb) { return tb.rc64; }
};

struct sa_geom {
	int L, B, n, nal, ncoef;
	int ge, go;		/* groups of eight columns, even and odd orders */
	int ld;			/* LDS row stride of the ring sums */
	int nct, tiles, tpp, parts;
};

/* the phi DFT in the operand's lane order, [column tile][group][lane][2]:
 * lane i + 16 q holds point i at columns 2 q, 2 q + 1 of the group */
template <typename T>
__global__ void k_sky_any_table(struct sa_geom g, const double *__restrict__ twp, T *__restrict__ W)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if(i >= g.nct * (g.ge + g.go) * 128)
		return;
	const int ct = i / ((g.ge + g.go) * 128), r = i - ct * (g.ge + g.go) * 128;
	const int grp = r >> 7, lane = (r >> 1) & 63, k = 16 * ct + (lane & 15);
	const int par = grp >= g.ge, col = 8 * (grp - (par ? g.ge : 0)) + 2 * (lane >> 4) + (r & 1);
	const int m = par + (col & ~1);
	double w = 0.;
	if(m <= g.L && k < g.B) {
		const int t = (int) (((long) m * k) % g.n);
		w = (m ? 2. : 1.) * (col & 1 ? -twp[2 * t + 1] : twp[2 * t]);
	}
	W[i] = (T) w;
}

template <typename T, bool SYM>
__global__ void __launch_bounds__(SA_NT) k_sky_any(const T *__restrict__ partial, int nsplit, int S, struct xproj_geom xg, const cplx<T> *__restrict__ R, const cplx<T> *__restrict__ Rs, const int2 *__restrict__ lm, const double *__restrict__ gmst, struct synth_tables tb, const T *__restrict__ W, struct sa_geom g, cplx<T> *__restrict__ alm, cplx<T> *__restrict__ map)
{
	typedef sa_ops<T> ops;
	typedef typename ops::v4 v4;
	typedef typename ops::pair pair;
	extern __shared__ __align__(16) unsigned char sa_sm[];
	T *F = reinterpret_cast<T *>(sa_sm);					/* [tpp][16][ld] */
	cplx<T> *sa = reinterpret_cast<cplx<T> *>(F + (map ? g.tpp * 16 * g.ld : 0));	/* [nal] */
	cplx<T> *cf = sa + g.nal;						/* [nal + 2] */
	cplx<T> *rot = cf + g.nal + 2;						/* [L + 1] */
	T *pw = reinterpret_cast<T *>(rot + g.L + 1);				/* [CT] */
	const int s = blockIdx.x / g.parts, part = blockIdx.x - s * g.parts;
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lq = lane >> 4;
	const int L = g.L;

	for(int c = tid; c < xg.CT; c += SA_NT) {
		const T *p = partial + (size_t) s * xg.CT + c;
		const size_t st = (size_t) S * xg.CT;
		T v[8];
#pragma unroll
		for(int u = 0; u < 8; u++)
			v[u] = 0;
		int sp = 0;
		for(; sp + 8 <= nsplit; sp += 8)
#pragma unroll
			for(int u = 0; u < 8; u++)
				v[u] += p[(sp + u) * st];
#pragma unroll
		for(int u = 0; u < 8; u++)
			if(sp + u < nsplit)
				v[u] += p[(sp + u) * st];
		pw[c] = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
	}
	for(int m = tid; m <= L; m += SA_NT) {
		double sn = 0.0, cs = 1.0;
		if(gmst && m)
			sincos(-(double) m * gmst[s], &sn, &cs);
		rot[m] = mk((T) cs, (T) sn);
	}
	if(map) {
		const cplx<T> *rc = ops::rc(tb);
		for(int t = tid; t < g.nal + 2; t += SA_NT)
			cf[t] = rc[t];
		for(int t = tid; t < g.tpp * 16 * g.ld; t += SA_NT)
			F[t] = (T) 0;
	}
	__syncthreads();

	/* a_lm: rotation row x the baseline's projected column, summed over the
	 * baselines in float64 whatever T, then rotate_z; the m >= 0 block
	 * comes first in the coefficient order.  With SYM the mesh's
	 * coefficients are those of the rows Rs (the real part of a mesh is the
	 * sum over the rows' symmetric part): the first part, which writes the
	 * a_lm, forms both */
	{
		const int nc = part ? g.nal : g.ncoef, ld = SYM && part ? g.nal : g.ncoef;
		const cplx<T> *rows = SYM && part ? Rs : R;
		cplx<T> *out = alm + (size_t) s * g.ncoef;
#pragma unroll 2
		for(int idx = tid; idx < nc; idx += SA_NT) {
			const int2 q = lm[idx];
			const bool two = SYM && !part && idx < g.nal;
			cplx<double> acc = mk(0.0, 0.0), accs = mk(0.0, 0.0);
			for(int b0 = 0; b0 < xg.nb; b0 += 4) {
				cplx<T> r[4], rs[4];
#pragma unroll
				for(int u = 0; u < 4; u++)
					if(b0 + u < xg.nb) {
						r[u] = rows[(size_t) (b0 + u) * ld + idx];
						if(two)
							rs[u] = Rs[(size_t) (b0 + u) * g.nal + idx];
					}
#pragma unroll
				for(int u = 0; u < 4; u++)
					if(b0 + u < xg.nb && q.x <= xg.Lb[b0 + u]) {
						const T *p = pw + xg.col_start[b0 + u] + 2 * q.x;
						const cplx<double> v = mk((double) p[0], (double) p[1]);
						cfma(acc, mk((double) r[u].re, (double) r[u].im), v);
						if(two)
							cfma(accs, mk((double) rs[u].re, (double) rs[u].im), v);
					}
			}
			cplx<T> a = mk((T) acc.re, (T) acc.im), as = two ? mk((T) accs.re, (T) accs.im) : a;
			if(gmst && q.y) {
				const cplx<T> z = q.y > 0 ? rot[q.y] : conjg(rot[-q.y]);
				a = a * z;
				if(SYM)
					as = as * z;
			}
			if(idx < g.nal)
				sa[idx] = SYM ? as : a;
			if(!part)
				out[idx] = a;
		}
	}
	if(!map)
		return;
	__syncthreads();

	/* ring sums */
	const int j0 = 8 * g.tpp * part, j1 = j0 + 8 * g.tpp < g.B ? j0 + 8 * g.tpp : g.B;
	{
		const int NG = (j1 - j0 + 1) / 2, NA = L / 2 + 1;
		for(int it = tid; it < NG * NA; it += SA_NT) {
			const int tg = it % NG, a = it / NG;
			const int j = j0 + 2 * tg, jb = j + 1 < j1 ? j + 1 : j;
			const T x[2] = { (T) tb.x[j], (T) tb.x[jb] };
#pragma unroll
			for(int h = 0; h < 2; h++) {
				const int am = h ? L - a : a;
				if(h && am == a)
					break;
				const int cbase = lm_offset(L, am, am);
				const cplx<T> *sp = sa + cbase, *cc = cf + cbase;
				const int cnt = L - am;
				T p2[2], p1[2];
				cplx<T> Ep[2], Op[2];
				p2[0] = (T) tb.smm[(size_t) j * (L + 1) + am];
				p2[1] = (T) tb.smm[(size_t) jb * (L + 1) + am];
				const cplx<T> a0 = sp[0], a1 = cnt >= 1 ? sp[1] : mk((T) 0, (T) 0);
				const T c1 = cnt >= 1 ? cc[1].re : (T) 0;
#pragma unroll
				for(int r = 0; r < 2; r++) {
					Ep[r] = a0 * p2[r];
					p1[r] = c1 * x[r] * p2[r];
					Op[r] = a1 * p1[r];
				}
				int i = 2;
				for(; i + SA_US - 1 <= cnt; i += SA_US) {
					cplx<T> c[SA_US], av[SA_US];
#pragma unroll
					for(int u = 0; u < SA_US; u++) {
						c[u] = cc[i + u];
						av[u] = sp[i + u];
					}
#pragma unroll
					for(int r = 0; r < 2; r++)
#pragma unroll
						for(int u = 0; u < SA_US; u += 2) {
							const T pe = c[u].re * x[r] * p1[r] - c[u].im * p2[r];
							const T po = c[u + 1].re * x[r] * pe - c[u + 1].im * p1[r];
							cfma(Ep[r], av[u], pe);
							cfma(Op[r], av[u + 1], po);
							p2[r] = pe;
							p1[r] = po;
						}
				}
				for(; i <= cnt; i += 2) {
					const cplx<T> c0 = cc[i], cn = cc[i + 1], b0 = sp[i];
					const cplx<T> b1 = i + 1 <= cnt ? sp[i + 1] : mk((T) 0, (T) 0);
#pragma unroll
					for(int r = 0; r < 2; r++) {
						const T pe = c0.re * x[r] * p1[r] - c0.im * p2[r];
						const T po = i + 1 <= cnt ? cn.re * x[r] * pe - cn.im * p1[r] : (T) 0;
						cfma(Ep[r], b0, pe);
						cfma(Op[r], b1, po);
						p2[r] = pe;
						p1[r] = po;
					}
				}
				const int col = (am & 1 ? 8 * g.ge : 0) + (am & ~1);
#pragma unroll
				for(int r = 0; r < 2; r++) {
					const int jj = 2 * tg + r;
					if(j0 + jj >= j1)
						continue;
					T *o = F + ((jj >> 3) * 16 + (jj & 7)) * g.ld + col;
					o[0] = Ep[r].re + Op[r].re;
					o[1] = Ep[r].im + Op[r].im;
					o[8 * g.ld] = Ep[r].re - Op[r].re;
					o[8 * g.ld + 1] = Ep[r].im - Op[r].im;
				}
			}
		}
	}
	__syncthreads();

	/* phi DFT: a wave's units are (ring group, column tile) */
	cplx<T> *mr = map + (size_t) s * g.n * g.n;
	const int nt = (j1 - j0 + 7) / 8, G = g.ge + g.go;
	for(int u = wave; u < nt * g.nct; u += SA_NT / 64) {
		const int t = u % nt, ct = u / nt;
		const T *A = F + (t * 16 + li) * g.ld + 2 * lq;
		const pair *w = reinterpret_cast<const pair *>(W) + (size_t) ct * G * 64 + lane;
		v4 ev = (v4) 0, od = (v4) 0;
		for(int k = 0; k < g.ge; k++) {
			const pair a = *reinterpret_cast<const pair *>(A + 8 * k), b = w[(size_t) k * 64];
			ev = ops::mma(a.x, b.x, ev);
			ev = ops::mma(a.y, b.y, ev);
		}
		for(int k = g.ge; k < G; k++) {
			const pair a = *reinterpret_cast<const pair *>(A + 8 * k), b = w[(size_t) k * 64];
			od = ops::mma(a.x, b.x, od);
			od = ops::mma(a.y, b.y, od);
		}
		const int k = 16 * ct + li;
		if(k < g.B)
#pragma unroll
			for(int e = 0; e < 4; e++) {
				const int row = ops::row(lq, e), j = j0 + 8 * t + (row & 7);
				if(j >= g.B)
					continue;
				const size_t o = (size_t) (row < 8 ? j : g.n - 1 - j) * g.n + k;
				mr[o] = mk(ev[e] + od[e], (T) 0);
				mr[o + g.B] = mk(ev[e] - od[e], (T) 0);
			}
	}
}

struct sa_geom sa_geom_of(int L, int f32)
{
	struct sa_geom g;
	memset(&g, 0, sizeof(g));
	g.L = L;
	g.B = L + 1;
	g.n = 2 * g.B;
	g.nal = (L + 1) * (L + 2) / 2;
	g.ncoef = (L + 1) * (L + 1);
	g.ge = (2 * (L / 2 + 1) + 7) / 8;
	g.go = (2 * ((L + 1) / 2) + 7) / 8;
	/* 16 rows start on distinct banks */
	g.ld = 8 * (g.ge + g.go) + (f32 ? 4 : 2);
	g.nct = (g.B + 15) / 16;
	g.tiles = (g.B + 7) / 8;
	return g;
}

}	/* namespace */

template <typename T>
size_t sky_any_table_bytes(int L)
{
	const struct sa_geom g = sa_geom_of(L, sizeof(T) == 4);
	return (size_t) g.nct * (g.ge + g.go) * 128 * sizeof(T);
}

template <typename T>
int sky_any_table(int L, const double *twp, T *W, hipStream_t st)
{
	const struct sa_geom g = sa_geom_of(L, sizeof(T) == 4);
	const int n = g.nct * (g.ge + g.go) * 128;
	hipLaunchKernelGGL((k_sky_any_table<T>), dim3((n + 255) / 256), dim3(256), 0, st, g, twp, W);
	return hipGetLastError() == hipSuccess ? 0 : -1;
}

/* LDS of a workgroup besides the ring sums, and of one group's ring sums */
static size_t sky_any_lds(const struct sa_geom *g, int CT, size_t esz, size_t *tile)
{
	*tile = (size_t) 16 * g->ld * esz;
	return ((size_t) 2 * g->nal + 2 + g->L + 1) * 2 * esz + (size_t) CT * esz;
}

#define SA_LDS ((size_t) 158 * 1024)

template <typename T>
int sky_any_fits(int L, int CT)
{
	const struct sa_geom g = sa_geom_of(L, sizeof(T) == 4);
	size_t tile;
	const size_t fixed = sky_any_lds(&g, CT, sizeof(T), &tile);
	return fixed + tile <= SA_LDS;
}

/* parts per segment: enough workgroups for two per CU, more where the ring
 * sums of a part would not fit in LDS; -1 where one ring group does not */
template <typename T>
int launch_sky_any(const T *partial, int nsplit, int S, const struct xproj_geom *xg, const cplx<T> *R, const cplx<T> *Rs, const int2 *lm, const double *gmst, int L, const struct synth_tables *tb, const T *W, cplx<T> *alm, cplx<T> *map, hipStream_t st)
{
	struct sa_geom g = sa_geom_of(L, sizeof(T) == 4);
	size_t tile;
	const size_t fixed = sky_any_lds(&g, xg->CT, sizeof(T), &tile);
	if(S <= 0)
		return 0;
	int parts = 1;
	if(map) {
		if(fixed + tile > SA_LDS)
			return -1;
		parts = 2 * sphr_rt_cus() / S;
		parts = parts < 1 ? 1 : parts > g.tiles ? g.tiles : parts;
		while(parts < g.tiles && fixed + (g.tiles + parts - 1) / parts * tile > SA_LDS)
			parts++;
	} else if(fixed > SA_LDS)
		return -1;
	g.tpp = (g.tiles + parts - 1) / parts;
	g.parts = (g.tiles + g.tpp - 1) / g.tpp;
	if(Rs)
		hipLaunchKernelGGL((k_sky_any<T, true>), dim3(S * g.parts), dim3(SA_NT), fixed + (map ? g.tpp * tile : 0), st, partial, nsplit, S, *xg, R, Rs, lm, gmst, *tb, W, g, alm, map);
	else
		hipLaunchKernelGGL((k_sky_any<T, false>), dim3(S * g.parts), dim3(SA_NT), fixed + (map ? g.tpp * tile : 0), st, partial, nsplit, S, *xg, R, Rs, lm, gmst, *tb, W, g, alm, map);
	return hipGetLastError() == hipSuccess ? 0 : -1;
}

template int sky_any_fits<float>(int, int);
template int sky_any_fits<double>(int, int);
template size_t sky_any_table_bytes<float>(int);
template size_t sky_any_table_bytes<double>(int);
template int sky_any_table<float>(int, const double *, float *, hipStream_t);
template int sky_any_table<double>(int, const double *, double *, hipStream_t);
template int launch_sky_any<float>(const float *, int, int, const struct xproj_geom *, const cplx<float> *, const cplx<float> *, const int2 *, const double *, int, const struct synth_tables *, const float *, cplx<float> *, cplx<float> *, hipStream_t);
template int launch_sky_any<double>(const double *, int, int, const struct xproj_geom *, const cplx<double> *, const cplx<double> *, const int2 *, const double *, int, const struct synth_tables *, const double *, cplx<double> *, cplx<double> *, hipStream_t);
