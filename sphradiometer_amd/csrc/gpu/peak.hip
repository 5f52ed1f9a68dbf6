/*
 * Extremum of a real function on the sphere given by its SH series
 * (sh_series_real_minimum, sh_series_extremize.c:273-360), batched: half
 * a wavefront per series.
 *
 * Seed: either the reference's (sh_series_extremize.c:168-241): the
 * series low-passed to l = l_seed, sampled on its 2(l_seed+1)-ring
 * Gauss-Legendre mesh, the extreme pixel; or the extreme pixel of a mesh
 * the caller already synthesised at full order.
 *
 * Refinement: Newton steps in the tangent plane at the current point p,
 * basis (theta-hat, phi-hat), a step length capped at 0.05 rad, and a
 * gradient step when the Hessian is not definite in the wanted direction.
 * The reference refines with GSL's BFGS2; the fixed point is the same
 * stationary point, the iterates are not.
 *
 * The gradient and Hessian are exact, from one pass over the coefficients.
 * With w = x + i y and Pi_lm(z) = Pbar_lm / sin^m theta (a polynomial),
 *   Re f = Re sum_m c_m(z) w^m,  c_m = sum_l b_lm Pi_lm(z),
 *   b_lm = a_lm + (-1)^m conj(a_l,-m) (m > 0), b_l0 = Re a_l0,
 * a smooth function of (x, y, z) also at the poles; its derivatives there
 * (c', c'' by the differentiated recurrence) give, with the normal n = p,
 * the tangent gradient E^T grad and Hessian E^T (grad grad) E - (n . grad) I.
 * The recurrences carry the factor sin^(m - k), k = min(m, 2), so that
 * values stay bounded at any order.
 *
 * 32 lanes per series, two series per wavefront; lane a takes the orders
 * a and L - a (L + 2 terms together), the b_lm staged in LDS once.  What
 * bounds it is the latency of those terms and of the step between passes
 * (the LDS of the coefficients leaves six wavefronts on a CU; float64 issue
 * is a third of the time): one pass per step in place of thirteen (central
 * differences: twelve around the point and one at the trial) with a division
 * per term, 8192 skies of order 32 in 0.21 ms against 4.53 (with the mesh
 * seeds, 0.26 against 4.64).  Sums over the lanes through DPP instead of
 * shuffles 0.40 -> 0.38 ms; steps within rounding of the maximum accepted
 * instead of halved eight times 0.38 -> 0.21.
 */
#include <hip/hip_runtime.h>
#include <math.h>
#include "kernels.h"

struct peak_tables {
	const double *cm;	/* L+1: Pbar_mm = cm[m] sin^m theta */
	const double *alpha;	/* packed alpha_lm of the l recurrence (order L) */
	const double *seed_x;	/* seed mesh rings, cos theta descending */
	int n_seed;		/* seed mesh size (rings = columns) */
};

/* v of the lane that a data-parallel-primitive pattern names (within rows of
 * 16 lanes: no LDS round trip, as a shuffle makes) */
template <int CTRL>
__device__ inline double lane_of(double v)
{
	union {
		double d;
		int i[2];
	} u;
	u.d = v;
	u.i[0] = __builtin_amdgcn_update_dpp(0, u.i[0], CTRL, 0xf, 0xf, false);
	u.i[1] = __builtin_amdgcn_update_dpp(0, u.i[1], CTRL, 0xf, 0xf, false);
	return u.d;
}

/* sum over the 32 lanes of a series; every lane returns the same total */
__device__ inline double half_sum(double v)
{
	v += lane_of<0xb1>(v);	/* quad_perm 1,0,3,2 */
	v += lane_of<0x4e>(v);	/* quad_perm 2,3,0,1 */
	v += lane_of<0x141>(v);	/* mirrored in 8 */
	v += lane_of<0x140>(v);	/* mirrored in 16 */
	return v + __shfl_xor(v, 16);
}

/* value and derivatives at a point, as a function of (x, y, z); F_yy = -F_xx */
struct peak_eval {
	double f, x, y, z, xx, xy, xz, yz, zz;
};

struct peak_point {
	double x, y, z;
};

/* Re f and its derivatives at p, the lanes over m, summed over the lanes of
 * the series.  The b_lm and recurrence pairs (alpha_l, alpha_l /
 * alpha_{l-1}) are in LDS (bc, rc, at the (l, m >= 0) slots) or, for orders
 * that do not fit, formed from global memory */
template <typename TI, bool LDS>
__device__ struct peak_eval eval_half(const cplx<TI> *a, int L, const struct peak_point p, const struct peak_tables &t, const cplx<double> *bc, const cplx<double> *rc)
{
	const int lane = threadIdx.x & 31;
	const double s = sqrt(p.x * p.x + p.y * p.y), z = p.z;
	const double ex = s > 0. ? p.x / s : 1., ey = s > 0. ? p.y / s : 0.;
	struct peak_eval r = { 0., 0., 0., 0., 0., 0., 0., 0., 0. };
	for(int i = lane; i <= L / 2; i += 32)
		for(int h = 0; h < 2; h++) {
			const int m = h ? L - i : i;
			if(h && m == i)
				continue;
			const int k = m < 2 ? m : 2;
			/* sin^(m-k) theta and exp(i (m-k) phi) by squaring */
			double q = t.cm[m], sp = s, ur = 1., ui = 0., vr = ex, vi = ey;
			for(int e = m - k; e; e >>= 1) {
				if(e & 1) {
					q *= sp;
					const double n = ur * vr - ui * vi;
					ui = ur * vi + ui * vr;
					ur = n;
				}
				sp *= sp;
				const double n = vr * vr - vi * vi;
				vi = 2. * vr * vi;
				vr = n;
			}
			/* the sums over l of b, times p, p', p'' */
			const int o = lm_offset(L, m, m), on = lm_offset(L, m, -m);
			const double sg = (m & 1) ? -1. : 1.;
			double p0 = 0., d0 = 0., e0 = 0., p1 = q, d1 = 0., e1 = 0., am = 1.;
			double cr = 0., ci = 0., dr = 0., di = 0., er = 0., ei = 0.;
#pragma unroll 4
			for(int l = 0; l <= L - m; l++) {
				cplx<double> b;
				if(LDS)
					b = bc[o + l];
				else {
					const cplx<TI> c = a[o + l];
					b = mk((double) c.re, m ? (double) c.im : 0.);
					if(m) {
						const cplx<TI> n = a[on + l];
						b.re += sg * (double) n.re;
						b.im -= sg * (double) n.im;
					}
				}
				if(l) {
					double al, ra;
					if(LDS) {
						al = rc[o + l].re;
						ra = rc[o + l].im;
					} else {
						al = t.alpha[o + l];
						ra = l > 1 ? al / am : 0.;
						am = al;
					}
					const double az = al * z;
					const double pn = fma(az, p1, -ra * p0);
					const double dn = fma(az, d1, fma(al, p1, -ra * d0));
					const double en = fma(az, e1, fma(2. * al, d1, -ra * e0));
					p0 = p1;
					d0 = d1;
					e0 = e1;
					p1 = pn;
					d1 = dn;
					e1 = en;
				}
				cr = fma(b.re, p1, cr);
				ci = fma(b.im, p1, ci);
				dr = fma(b.re, d1, dr);
				di = fma(b.im, d1, di);
				er = fma(b.re, e1, er);
				ei = fma(b.im, e1, ei);
			}
			/* u = w^(m-k) / sin^(m-k): times w^k, k w^(k-1), .. with the
			 * factors of the derivatives of w^m */
			const double u1r = ur * p.x - ui * p.y, u1i = ur * p.y + ui * p.x;		/* u w */
			const double u2r = u1r * p.x - u1i * p.y, u2i = u1r * p.y + u1i * p.x;		/* u w^2 */
			double fr = ur, fi = ui, gr = 0., gi = 0., hr = 0., hi = 0.;
			if(k == 1) {
				fr = u1r;
				fi = u1i;
				gr = ur;
				gi = ui;
			} else if(k == 2) {
				fr = u2r;
				fi = u2i;
				gr = m * u1r;
				gi = m * u1i;
				hr = (double) m * (m - 1) * ur;
				hi = (double) m * (m - 1) * ui;
			}
			r.f += cr * fr - ci * fi;
			r.z += dr * fr - di * fi;
			r.zz += er * fr - ei * fi;
			r.x += cr * gr - ci * gi;
			r.y -= cr * gi + ci * gr;
			r.xz += dr * gr - di * gi;
			r.yz -= dr * gi + di * gr;
			r.xx += cr * hr - ci * hi;
			r.xy -= cr * hi + ci * hr;
		}
	r.f = half_sum(r.f);
	r.x = half_sum(r.x);
	r.y = half_sum(r.y);
	r.z = half_sum(r.z);
	r.xx = half_sum(r.xx);
	r.xy = half_sum(r.xy);
	r.xz = half_sum(r.xz);
	r.yz = half_sum(r.yz);
	r.zz = half_sum(r.zz);
	return r;
}

__device__ inline void condition(double *theta, double *phi)
{
	/* theta into [0, pi] (flipping phi), phi into [0, 2 pi):
	 * sh_series_extremize.c:63-87 */
	double t = fmod(*theta, 2 * M_PI);
	if(t < 0)
		t += 2 * M_PI;
	double p = *phi;
	if(t > M_PI) {
		t = 2 * M_PI - t;
		p += M_PI;
	}
	p = fmod(p, 2 * M_PI);
	if(p < 0)
		p += 2 * M_PI;
	*theta = t;
	*phi = p;
}

/* the (theta-hat, phi-hat) basis at p */
__device__ inline void basis(const struct peak_point &p, double th[3], double ph[2])
{
	const double s = sqrt(p.x * p.x + p.y * p.y);
	const double ex = s > 0. ? p.x / s : 1., ey = s > 0. ? p.y / s : 0.;
	th[0] = p.z * ex;
	th[1] = p.z * ey;
	th[2] = -s;
	ph[0] = -ey;
	ph[1] = ex;
}

/* the seed's index in row-major order over the lanes of a series: the lowest value, the first on ties */
template <int LANES>
__device__ inline int first_lowest(double best, int bi)
{
	for(int off = LANES / 2; off > 0; off >>= 1) {
		const double ob = __shfl_xor(best, off);
		const int oi = __shfl_xor(bi, off);
		if(ob < best || (ob == best && oi < bi)) {
			best = ob;
			bi = oi;
		}
	}
	/* no value compares below infinity (all NaN): the first pixel */
	return bi == 0x7fffffff ? 0 : bi;
}

/* seeds from meshes of the full order: the direction of each mesh's extreme
 * pixel of sign * Re f, first in row-major order on ties, into theta and
 * phi.  One wavefront per mesh; reading the mesh bounds it (285 MB for 8192
 * meshes of order 32 in 50 us), so it runs at full occupancy ahead of the
 * refinement, whose LDS leaves six wavefronts on a CU. */
template <typename TI>
__global__ void __launch_bounds__(256) k_map_seed(const cplx<TI> *__restrict__ map, int S, int n, const double *__restrict__ map_x, int sign, double *__restrict__ theta, double *__restrict__ phi)
{
	const int s = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
	if(s >= S)
		return;
	const int nn = n * n;
	const cplx<TI> *mp = map + (size_t) s * nn;
	double best = INFINITY;
	int bi = 0x7fffffff, i = lane;
	for(; i + 7 * 64 < nn; i += 8 * 64) {
		TI v[8];
#pragma unroll
		for(int u = 0; u < 8; u++)
			v[u] = mp[i + 64 * u].re;
#pragma unroll
		for(int u = 0; u < 8; u++)
			if(sign * (double) v[u] < best) {
				best = sign * (double) v[u];
				bi = i + 64 * u;
			}
	}
	for(; i < nn; i += 64) {
		const double v = sign * (double) mp[i].re;
		if(v < best) {
			best = v;
			bi = i;
		}
	}
	bi = first_lowest<64>(best, bi);
	if(lane == 0) {
		const int j = bi / n, k = bi - j * n, B = n / 2;
		theta[s] = acos(j < B ? map_x[j] : -map_x[2 * B - 1 - j]);
		phi[s] = 2.0 * M_PI * k / n;
	}
}

template <typename TI, bool LDS>
__global__ void __launch_bounds__(128) k_extremize(const cplx<TI> *__restrict__ alm, int S, int alm_div, int L, int sign, int l_seed, const double *seed_theta, const double *seed_phi, int seed_ld, struct peak_tables t, int max_iter, double *theta_out, double *phi_out, double *__restrict__ value_out)
{
	extern __shared__ __align__(16) unsigned char peak_sm[];
	const int lane = threadIdx.x & 31, slot = threadIdx.x >> 5, ns = blockDim.x >> 5;
	/* the lanes past the last series repeat it and write nothing */
	const int s_own = blockIdx.x * ns + slot, s = s_own < S ? s_own : S - 1;
	const int ncoef = (L + 1) * (L + 1), nal = (L + 1) * (L + 2) / 2;
	const cplx<TI> *a = alm + (size_t) (s / alm_div) * ncoef;
	cplx<double> *rc = reinterpret_cast<cplx<double> *>(peak_sm);	/* [nal] */
	cplx<double> *bc = rc + nal * (1 + slot);			/* [nal] of this series */
	if(LDS) {
		for(int i = threadIdx.x; i < nal; i += blockDim.x) {
			const double al = t.alpha[i], ap = i ? t.alpha[i - 1] : 1.;
			/* the first term of an order has no predecessor: its ratio is
			 * not used with a value other than zero */
			rc[i] = mk(al, ap != 0. ? al / ap : 0.);
		}
#pragma unroll 4
		for(int i = lane; i < nal; i += 32) {
			const int m = lm_order(L, i);
			const cplx<TI> c = a[i], n = a[m ? i - lm_offset(L, m, m) + lm_offset(L, m, -m) : i];
			const double sg = !m ? 0. : (m & 1) ? -1. : 1.;
			bc[i] = mk((double) c.re + sg * (double) n.re, (m ? (double) c.im : 0.) - sg * (double) n.im);
		}
		__syncthreads();
	}
	double th, ph;
	if(seed_theta) {
		/* may be theta_out and phi_out themselves */
		th = seed_theta[(size_t) seed_ld * s];
		ph = seed_phi[(size_t) seed_ld * s];
	} else {
	/* seed: the extreme of sign * Re f over the low-pass mesh, first in
	 * row-major order on ties (sh_series_extremize.c:214-230) */
	double best = INFINITY;
	int bi = 0x7fffffff;
	const int lc = l_seed < L ? l_seed : L;
	const int n = t.n_seed;
	for(int i = lane; i < n * n; i += 32) {
		/* per-lane scalar evaluation of the low-passed series */
		const int j = i / n, k = i - j * n;
		const double x = t.seed_x[j], st = sqrt((1.0 - x) * (1.0 + x)), ph = 2.0 * M_PI * k / n;
		double f = 0.0;
		for(int m = 0; m <= lc; m++) {
			double pprev = 0.0, pcur = t.cm[m] * (m ? pow(st, (double) m) : 1.0), aprev = 1.0;
			double spr = 0, spi = 0, smr = 0, smi = 0;
			for(int l = m; l <= lc; l++) {
				if(l > m) {
					const double al = t.alpha[lm_offset(L, l, m)];
					const double pn = (l == m + 1) ? al * x * pcur : al * (x * pcur - pprev / aprev);
					pprev = pcur;
					pcur = pn;
					aprev = al;
				}
				const cplx<TI> cp = a[lm_offset(L, l, m)];
				spr += (double) cp.re * pcur;
				spi += (double) cp.im * pcur;
				if(m) {
					const cplx<TI> cn = a[lm_offset(L, l, -m)];
					smr += (double) cn.re * pcur;
					smi += (double) cn.im * pcur;
				}
			}
			double sn, cs;
			sincos((double) m * ph, &sn, &cs);
			f += cs * spr - sn * spi;
			if(m)
				f += ((m & 1) ? -1.0 : 1.0) * (cs * smr + sn * smi);
		}
		const double v = sign * f;
		if(v < best) {
			best = v;
			bi = i;
		}
	}
	bi = first_lowest<32>(best, bi);
	th = acos(t.seed_x[bi / n]);
	ph = 2.0 * M_PI * (bi % n) / n;
	}
	/* Newton in the tangent plane on g(p) = sign * Re f(p): each pass
	 * evaluates a trial point; a trial that does not increase g (beyond
	 * rounding) becomes the point and the next step is formed there, else the step is
	 * halved, eight times at most.  The two series of a wavefront run
	 * until both are done. */
	struct peak_point p, q;
	{
		double sn, cs;
		sincos(ph, &sn, &cs);
		const double st = sin(th);
		q = { st * cs, st * sn, cos(th) };
	}
	p = q;
	double f0 = 0., d1 = 0., d2 = 0., dn = 0., scale = 1., noise = 0.;
	double bth[3], bph[2];
	int it = -1, bt = 0;
	bool done = false;
	for(;;) {
		const struct peak_eval r = eval_half<TI, LDS>(a, L, q, t, bc, rc);
		if(!done) {
			const double nf = sign * r.f;
			if(it < 0 || nf <= f0 + noise) {
				p = q;
				f0 = nf;
				if(it >= 0 && scale * dn < 1e-11)
					done = true;
				if(++it >= max_iter)
					done = true;
				basis(p, bth, bph);
				const double g1 = sign * (bth[0] * r.x + bth[1] * r.y + bth[2] * r.z), g2 = sign * (bph[0] * r.x + bph[1] * r.y);
				const double gn_ = sign * (p.x * r.x + p.y * r.y + p.z * r.z);
				const double vx = bth[0] * r.xx + bth[1] * r.xy + bth[2] * r.xz, vy = bth[0] * r.xy - bth[1] * r.xx + bth[2] * r.yz;
				const double vz = bth[0] * r.xz + bth[1] * r.yz + bth[2] * r.zz;
				const double h11 = sign * (bth[0] * vx + bth[1] * vy + bth[2] * vz) - gn_, h12 = sign * (bph[0] * vx + bph[1] * vy);
				const double h22 = sign * (bph[0] * (bph[0] * r.xx + bph[1] * r.xy) + bph[1] * (bph[0] * r.xy - bph[1] * r.xx)) - gn_;
				/* eigenvalues of the Hessian; the step solves (H + mu I) d = -g
				 * with mu lifting the smallest eigenvalue to 1e-6 of the largest,
				 * so flat directions (a ring of minima of an axisymmetric
				 * function) take no large steps and negative curvature is
				 * followed downhill */
				const double tr2 = 0.5 * (h11 + h22), dh = 0.5 * (h11 - h22);
				const double disc = sqrt(dh * dh + h12 * h12);
				const double lmin = tr2 - disc, lmax = tr2 + disc;
				const double gn = sqrt(g1 * g1 + g2 * g2);
				if(it > 0 && gn <= 1e-10 * (fabs(f0) + fabs(lmax)))
					done = true;
				/* a few roundings of the sum: the last steps change g by
				 * less, and halving them would only repeat the point */
				noise = 1.8e-15 * (fabs(f0) + fabs(lmax));
				if(lmax > 0) {
					const double floor_ = 1e-6 * lmax;
					const double mu = lmin < floor_ ? floor_ - lmin : 0.0;
					const double a11 = h11 + mu, a22 = h22 + mu;
					const double det = a11 * a22 - h12 * h12;
					d1 = -(a22 * g1 - h12 * g2) / det;
					d2 = -(-h12 * g1 + a11 * g2) / det;
				} else {
					/* concave both ways: steepest descent */
					d1 = -0.02 * g1 / (gn + 1e-300);
					d2 = -0.02 * g2 / (gn + 1e-300);
				}
				dn = sqrt(d1 * d1 + d2 * d2);
				if(dn > 0.05) {
					d1 *= 0.05 / dn;
					d2 *= 0.05 / dn;
				}
				scale = 1.;
				bt = 0;
			} else {
				scale *= 0.5;
				if(++bt == 8)
					done = true;
			}
			/* the tangent offset, back onto the sphere */
			const double s1 = scale * d1, s2 = scale * d2;
			q = { p.x + s1 * bth[0] + s2 * bph[0], p.y + s1 * bth[1] + s2 * bph[1], p.z + s1 * bth[2] };
			const double w = 1. / sqrt(q.x * q.x + q.y * q.y + q.z * q.z);
			q = { q.x * w, q.y * w, q.z * w };
		}
		if(__all(done))
			break;
	}
	if(lane == 0 && s_own < S) {
		/* a series with values that are not numbers has no extremum */
		double to = f0 == f0 ? atan2(sqrt(p.x * p.x + p.y * p.y), p.z) : f0, po = f0 == f0 ? atan2(p.y, p.x) : f0;
		condition(&to, &po);
		theta_out[s] = to;
		phi_out[s] = po;
		value_out[s] = sign * f0;
	}
}

/* four series per workgroup while their b_lm and the recurrence pairs leave
 * room for several workgroups on a CU, two, or the coefficients from global
 * memory at the orders whose two series do not fit */
template <typename TI>
static int launch_k(const cplx<TI> *alm, int S, int alm_div, int L, int sign, int l_seed, const double *seed_theta, const double *seed_phi, int seed_ld, const struct peak_tables &t, int max_iter, double *theta, double *phi, double *value, hipStream_t st)
{
	const size_t one = (size_t) (L + 1) * (L + 2) / 2 * sizeof(cplx<double>);
	if(3 * one <= 150 * 1024) {
		const int ns = 5 * one <= 53 * 1024 ? 4 : 2;
		hipLaunchKernelGGL((k_extremize<TI, true>), dim3((S + ns - 1) / ns), dim3(32 * ns), (1 + ns) * one, st, alm, S, alm_div, L, sign, l_seed, seed_theta, seed_phi, seed_ld, t, max_iter, theta, phi, value);
	} else
		hipLaunchKernelGGL((k_extremize<TI, false>), dim3((S + 3) / 4), dim3(128), 0, st, alm, S, alm_div, L, sign, l_seed, seed_theta, seed_phi, seed_ld, t, max_iter, theta, phi, value);
	return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <typename TI>
int launch_extremize(const cplx<TI> *alm, int S, int L, int find_max, int l_seed, const cplx<TI> *seed_map, const double *map_x, const double *cm, const double *alpha, const double *seed_x, int n_seed, int max_iter, double *theta, double *phi, double *value, hipStream_t st)
{
	const struct peak_tables t = { cm, alpha, seed_x, n_seed };
	const int sign = find_max ? -1 : 1;
	if(!seed_map)
		return launch_k<TI>(alm, S, 1, L, sign, l_seed, NULL, NULL, 0, t, max_iter, theta, phi, value, st);
	hipLaunchKernelGGL((k_map_seed<TI>), dim3((S + 3) / 4), dim3(256), 0, st, seed_map, S, 2 * (L + 1), map_x, sign, theta, phi);
	return launch_k<TI>(alm, S, 1, L, sign, l_seed, theta, phi, 1, t, max_iter, theta, phi, value, st);
}

template <typename TI>
int launch_extremize_seeded(const cplx<TI> *alm, int S, int alm_div, int L, int find_max, const double *seeds, const double *cm, const double *alpha, int max_iter, double *theta, double *phi, double *value, hipStream_t st)
{
	const struct peak_tables t = { cm, alpha, NULL, 0 };
	return launch_k<TI>(alm, S, alm_div, L, find_max ? -1 : 1, 0, seeds, seeds + 1, 2, t, max_iter, theta, phi, value, st);
}

template int launch_extremize<double>(const cplx<double> *, int, int, int, int, const cplx<double> *, const double *, const double *, const double *, const double *, int, int, double *, double *, double *, hipStream_t);
template int launch_extremize<float>(const cplx<float> *, int, int, int, int, const cplx<float> *, const double *, const double *, const double *, const double *, int, int, double *, double *, double *, hipStream_t);
template int launch_extremize_seeded<double>(const cplx<double> *, int, int, int, int, const double *, const double *, const double *, int, double *, double *, double *, hipStream_t);
template int launch_extremize_seeded<float>(const cplx<float> *, int, int, int, int, const double *, const double *, const double *, int, double *, double *, double *, hipStream_t);
