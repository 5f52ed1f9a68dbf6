/*
 * HEALPix output on the GPU (sh_series_healpix.cc, healpix.py,
 * RapidLocalization.py:498-530 of the reference).
 *
 * The reference writes the real part of a series (sh_series_real) through
 * healpix_cxx alm2map into a RING-ordered map at the centres of the
 * pixels; for the real part's coefficients that is Re f at the centres,
 * f the series itself, which is what is computed here, for many series at
 * once.  Pixel centres (Gorski et al. 2005, ApJ 622, 759): 4 nside - 1
 * rings of constant z; ring i (1-based from the north pole) has
 *   north cap,  i < nside:        z = 1 - i^2 / (3 nside^2), 4 i pixels,
 *                                 phi_j = (j + 1/2) 2 pi / (4 i);
 *   equator, nside <= i <= 3 nside: z = 4/3 - 2 i / (3 nside), 4 nside
 *                                 pixels, phi_j = (j + o) 2 pi / (4 nside),
 *                                 o = 0 when i + nside is odd, else 1/2;
 *   south cap: the mirror of the north cap,
 * pixels numbered ring by ring from the north pole, phi ascending.
 *
 * With b_lm = a_lm + (-1)^m conj(a_l,-m) (m > 0), b_l0 = Re a_l0 and
 * F_m(z) = sum_l b_lm Pbar_lm(z), a ring's values are
 *   f(phi) = sum_m A_m cos(m phi) - B_m sin(m phi),  A_m + i B_m = F_m,
 * so a map is two contractions with tables that all series share: the
 * Legendre values of the rings and the cosines of the pixels.  k_healpix_mm
 * runs both on MFMA, eight series per workgroup (see there); a few series,
 * and orders and resolutions whose tables would be too large, run
 * k_healpix_ring, which forms them by recurrence.
 */
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <sphradiometer/sh_series.h>
#include <sphradiometer/sphradiometer_batch.h>
#include <sphradiometer/sphradiometer_gpu.h>
#include "../sphr_internal.h"
#include "kernels.h"
#include "runtime.h"

#define HP_NT 256
#define HP_NSIDE_MAX 4096	/* the per-ring form keeps nside twiddles in LDS */

struct sphr_healpix {
	int L, nside, precision;
	double *d_cf;	/* [nal][2]: alpha_lm, alpha_lm / alpha_{l-1,m} at the (l, m >= 0) slots */
	double *d_cm;	/* [L + 1]: Pbar_mm(cos theta) = cm[m] sin^m theta */
	/* the tables of k_healpix_mm, NULL (and rc 0) where k_healpix_ring always runs */
	double *P;	/* Legendre values */
	void *W;	/* cosines and sines of the pixels */
	int *off;	/* [L + 1] first step of an order, then [2 nside + 1] first tile of a ring */
	int k0, k2, k1, steps, rc;
};

/* ring geometry: z, sin theta (without cancellation near the poles), the
 * pixel count, the index of its first pixel and the phase offset phi_0 */
__device__ inline void hp_ring(int nside, int i, double *z, double *st, int *nphi, long *start, double *phi0)
{
	const long N = nside, npix = 12 * N * N, ncap = 2 * N * (N - 1);
	if(i < nside) {
		const double u = (double) i * i / (3. * N * N);	/* 1 - z */
		*z = 1. - u;
		*st = sqrt(u * (2. - u));
		*nphi = 4 * i;
		*start = 2L * i * (i - 1);
		*phi0 = M_PI / (4. * i);
	} else if(i <= 3 * nside) {
		*z = (4. / 3.) - 2. * i / (3. * N);
		*st = sqrt((1. - *z) * (1. + *z));
		*nphi = 4 * nside;
		*start = ncap + (long) (i - nside) * 4 * N;
		*phi0 = ((i + nside) & 1) ? 0. : M_PI / (4. * N);
	} else {
		const int k = 4 * nside - i;
		const double u = (double) k * k / (3. * N * N);
		*z = u - 1.;
		*st = sqrt(u * (2. - u));
		*nphi = 4 * k;
		*start = npix - 2L * k * (k + 1);
		*phi0 = M_PI / (4. * k);
	}
}

#define HP_SPW 4		/* series per workgroup of the per-ring form */

/*
 * The maps of eight series on 2 RC rings per workgroup (RC northern rings
 * and their mirrors), sixteen waves.
 *
 *  A. Legendre sums, in float64 whatever the maps' type: per order m the
 *     product [16 rings] x [l] x [8 series x (re, im)] on
 *     v_mfma_f64_16x16x4f64, the l of each parity apart: Pbar_lm(-z) =
 *     (-1)^(l+m) Pbar_lm(z), so the even and odd sums E and O give the ring
 *     (E + O) and its mirror (E - O).  The Legendre table is laid out in the
 *     operand's lane order; the coefficients come straight from the a_lm.
 *     The orders are dealt to the waves, results go to LDS as the next
 *     product's left operand [ring][north / south, series][m, (A, B)].
 *  B. Pixel sums: nphi is a multiple of 4 and the pixels j + q nphi / 4
 *     (q = 0..3) sit at phi + q pi / 2.  With C_m = A_m cos m phi -
 *     B_m sin m phi, D_m = A_m sin m phi + B_m cos m phi and
 *       S0, S2 = sums of C_m over m = 0, 2 mod 4,
 *       U = sum of C_m over odd m, V = sum of +-D_m over m = 1, 3 mod 4,
 *     the four pixels are S0 + S2 + U, S0 - S2 - V, S0 + S2 - U,
 *     S0 - S2 + V: four products over a quarter of the ring, rows =
 *     (north / south) x 8 series, columns = 16 pixels, on MFMA in the maps'
 *     type; the phase of the first pixel is in the table.  LDS columns are
 *     ordered by m mod 4 for it: m = 0 | m = 2 | odd.
 *
 * RC is 16, or fewer where the LDS operand would not fit (the Legendre
 * product then computes 16 rows and drops the rest).  What bounds it: at
 * l_max 50, nside 32 and 16384 series the products are 5.6 GFLOP in
 * float64 (77 us at the matrix peak) and 18 in float32 (113 us), the maps
 * 805 MB (165 us at the rate of a large copy); the phases of the one
 * workgroup that fits a CU do not overlap (A takes 0.43 of 0.9 ms).  It
 * replaces a recurrence per (series, m, ring) and a pass over m per pixel:
 * 2.99 -> 0.93 ms (0.98-0.99 under a kernel trace; float64 coefficients fetched one value per lane, 31 cache
 * accesses per load: 1.1; eight waves instead of sixteen, 1.2), nine events
 * of l_max 120 at nside 64 in float64 0.43 -> 0.09 ms.
 */
#define HM_W 16
#define HM_NT (64 * HM_W)
#define HM_R 4
#define HM_S 8			/* series per workgroup */
#define HM_STAGE (HM_W * 2 * 64 * 16)	/* bytes of the waves' fetches */

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

template <typename T> struct hm_ops;
template <> struct hm_ops<float> {
	typedef f4 acc;
	typedef float2 pair;
	/* two complex values, and the steps of a parity that 8 x 8 of them hold */
	typedef float piece __attribute__((ext_vector_type(4), aligned(8)));
	enum { STEPS = 2 };
	static __device__ inline acc mma(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
	static __device__ inline int row(int lq, int e) { return 4 * lq + e; }
};
template <> struct hm_ops<double> {
	typedef d4 acc;
	typedef double2 pair;
	typedef double piece __attribute__((ext_vector_type(2), aligned(8)));
	enum { STEPS = 1 };
	static __device__ inline acc mma(double a, double b, acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
	static __device__ inline int row(int lq, int e) { return lq + 4 * e; }
};

struct hm_geom {
	int L, nside, n, rc;
	int k0, k2, k1;		/* padded columns of the three classes of m */
	int ld, rs;		/* LDS strides: row, ring */
	int steps, chunks, groups;
	const double *P;
	const int *off;
};

/* the LDS column of order m's A (B follows) */
__device__ inline int hm_col(const struct hm_geom &g, int m)
{
	return m & 1 ? g.k0 + g.k2 + (m - 1) : m & 2 ? g.k0 + (m - 2) / 2 : m / 2;
}

template <typename T>
__global__ void __launch_bounds__(HM_NT) k_healpix_mm(const cplx<T> *__restrict__ alm, struct hm_geom g, const T *__restrict__ W, T *__restrict__ map)
{
	typedef hm_ops<T> ops;
	typedef T vec4 __attribute__((ext_vector_type(4)));
	extern __shared__ __align__(16) unsigned char hm_sm[];
	T *AB = reinterpret_cast<T *>(hm_sm);	/* [rc][16][ld], then the waves' fetches */
	/* workgroups go to the eight XCDs in turn: contiguous ranges of (group
	 * of series, chunk) per XCD, so that a group's chunks share one L2 and
	 * a single group still fills the chip (each group on one XCD left the
	 * others idle below eight groups: eight float64 series of order 160 at
	 * nside 128 638 -> 178 us, order 200 at nside 256 2597 -> 417) */
	const int all = gridDim.x & ~7, id = (int) blockIdx.x < all ? (blockIdx.x & 7) * (all >> 3) + (blockIdx.x >> 3) : blockIdx.x;
	const int grp = id / g.chunks, chunk = id - grp * g.chunks;
	const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, lq = lane >> 4;
	const int L = g.L, L1 = L + 1, s0 = grp * HM_S, r0 = chunk * g.rc, N2 = 2 * g.nside;
	/* the columns past the orders multiply zeros of the table: finite */
	for(int i = threadIdx.x; i < g.rc * g.rs / 4; i += HM_NT)
		reinterpret_cast<vec4 *>(AB)[i] = (vec4) 0;
	__syncthreads();
	{
		constexpr int ST = ops::STEPS, CP = 8 * ST;	/* coefficients of a series per fetch */
		typedef typename ops::piece piece;
		/* this wave's fetches of a+ and a-: [2][8 series][8 pieces, piece q
		 * at q ^ series: the series' reads fall on distinct banks] */
		piece *stage = reinterpret_cast<piece *>(AB + (size_t) g.rc * g.rs) + wave * 128;
		auto staged = [&](int h, int k) -> T {
			return reinterpret_cast<const T *>(stage + 64 * h + (li >> 1) * 8 + ((k / ST) ^ (li >> 1)))[2 * (k % ST) + (li & 1)];
		};
		const int ring = r0 + li < N2 ? r0 + li : N2 - 1;	/* 0-based northern ring of operand row li */
		const double *P = g.P + ((size_t) (ring >> 4) * g.steps * 64 + lq * 16 + (ring & 15));
		const int comp = li & 1;
		/* lane (series, piece): eight lanes read 128 consecutive bytes of
		 * a series; fetches past an order's last l run into the next
		 * order, past the series' last order they stay inside the array,
		 * and their values are not used */
		const long last = (long) g.n * L1 * L1 - ST;
		const int fs = s0 + (lane >> 3) < g.n ? s0 + (lane >> 3) : g.n - 1;
		const long fo = (long) fs * L1 * L1 + (lane & 7) * ST;
		const T *a0 = reinterpret_cast<const T *>(alm), *af = a0 + 2 * fo;
		struct fetch {
			piece p, n;
			double pe[ST], po[ST];
		};
		auto order = [&](int i) -> int { return HM_W * i + (i & 1 ? HM_W - 1 - wave : wave); };
		auto piece_at = [&](int o) -> piece {
			if(o + CP <= L1 * L1)
				return *reinterpret_cast<const piece *>(af + 2 * o);
			const long c = fo + o < last ? fo + o : last;
			piece v = *reinterpret_cast<const piece *>(a0 + 2 * c);
			if(ST == 2 && fo + o > last) {
				/* the array's last coefficient alone */
				v[0] = v[2 * (ST - 1)];
				v[1] = v[2 * (ST - 1) + 1];
			}
			return v;
		};
		auto get = [&](int m, int tb) -> struct fetch {
			struct fetch f;
			f.p = piece_at(lm_offset(L, m, m) + tb * CP);
			f.n = piece_at(lm_offset(L, m, -m) + tb * CP);
			const int n = L - m, ke = (n / 2 + 4) / 4, ko = ((n + 1) / 2 + 3) / 4;
			const double *Pe = P + (size_t) g.off[m] * 64, *Po = ko ? Pe + (size_t) ke * 64 : Pe;
#pragma unroll
			for(int u = 0; u < ST; u++) {
				const int t = ST * tb + u;
				f.pe[u] = Pe[(size_t) (t < ke ? t : ke - 1) * 64];
				f.po[u] = Po[(size_t) (t < ko ? t : ko ? ko - 1 : 0) * 64];
			}
			return f;
		};
		int i = 0, tb = 0, m = order(0);
		struct fetch f;
		if(m <= L)
			f = get(m, 0);
		d4 E = (d4) 0, O = (d4) 0;
		while(m <= L) {
			stage[lane ^ (lane >> 3)] = f.p;
			stage[64 + (lane ^ (lane >> 3))] = f.n;
			double pe[ST], po[ST];
#pragma unroll
			for(int u = 0; u < ST; u++) {
				pe[u] = f.pe[u];
				po[u] = f.po[u];
			}
			/* the next fetch, in flight during this one's products */
			const int mc = m, n = L - m, d0 = CP * tb;
			const bool end = d0 + CP > n;
			if(end) {
				tb = 0;
				m = order(++i);
			} else
				tb++;
			if(m <= L)
				f = get(m, tb);
			__builtin_amdgcn_wave_barrier();
			/* b = a+ + (-1)^m conj a-: re +-, im -+; m = 0: Re a */
			const double sg = (mc & 1) != comp ? -1. : 1.;
#pragma unroll
			for(int u = 0; u < ST; u++) {
				const int k = 2 * (4 * u + lq);
				double be = (double) staged(0, k), bo = (double) staged(0, k + 1);
				if(mc) {
					be = fma(sg, (double) staged(1, k), be);
					bo = fma(sg, (double) staged(1, k + 1), bo);
				} else if(comp)
					be = bo = 0.;
				if(end) {
					be = d0 + k <= n ? be : 0.;
					bo = d0 + k < n ? bo : 0.;
				}
				E = hm_ops<double>::mma(pe[u], be, E);
				O = hm_ops<double>::mma(po[u], bo, O);
			}
			__builtin_amdgcn_wave_barrier();
			if(end) {
				const int col = hm_col(g, mc) + comp;
#pragma unroll
				for(int e = 0; e < 4; e++) {
					const int rr = lq + 4 * e;
					if(rr < g.rc) {
						T *o = AB + rr * g.rs + (li >> 1) * g.ld + col;
						o[0] = (T) (E[e] + O[e]);
						o[8 * g.ld] = (T) (E[e] - O[e]);
					}
				}
				E = (d4) 0;
				O = (d4) 0;
			}
		}
	}
	__syncthreads();
	const long npix = 12L * g.nside * g.nside;
	const int g0 = g.k0 / 8, g2 = g.k2 / 8, g1 = g.k1 / 8;
	const size_t tile = (size_t) 64 * (g0 + g2 + 2 * g1);	/* pairs of one tile's table */
	for(int rr = wave; rr < g.rc && r0 + rr < N2; rr += HM_W) {
		const int ring = r0 + rr + 1, n4 = ring < g.nside ? ring : g.nside, nt = (n4 + 15) / 16;
		const T *A = AB + rr * g.rs + li * g.ld + 2 * lq;
		const typename ops::pair *Wr = reinterpret_cast<const typename ops::pair *>(W) + (size_t) g.off[L1 + ring] * tile + lane;
		/* first pixels of the ring and of its mirror */
		const long sn = ring < g.nside ? 2L * ring * (ring - 1) : 2L * g.nside * (g.nside - 1) + 4L * g.nside * (ring - g.nside);
		const long ss = npix - sn - 4L * n4;
		for(int t0 = 0; t0 < nt; t0 += 2) {
			const typename ops::pair *w0 = Wr + (size_t) t0 * tile, *w1 = t0 + 1 < nt ? w0 + tile : w0;
			typename ops::acc acc[2][4];
#pragma unroll
			for(int u = 0; u < 2; u++)
#pragma unroll
				for(int c = 0; c < 4; c++)
					acc[u][c] = (typename ops::acc) 0;
			/* groups in runs of HM_R, the run's table loads ahead of its
			 * products; group k of all: S0, S2, then U and V in turn */
			auto run = [&](int k0, int cnt, int col0, int c, int cs, int div) {
				for(int k = 0; k < cnt; k += HM_R) {
					typename ops::pair b0[HM_R], b1[HM_R], av[HM_R];
#pragma unroll
					for(int q = 0; q < HM_R; q++) {
						const int kq = k + q < cnt ? k + q : cnt - 1;
						b0[q] = w0[(size_t) (k0 + kq) * 64];
						b1[q] = w1[(size_t) (k0 + kq) * 64];
						av[q] = *reinterpret_cast<const typename ops::pair *>(A + col0 + 8 * (kq / div));
					}
#pragma unroll
					for(int q = 0; q < HM_R; q++)
						if(k + q < cnt) {
							const int cc = c + (cs ? (q & 1) : 0);
							acc[0][cc] = ops::mma(av[q].x, b0[q].x, acc[0][cc]);
							acc[1][cc] = ops::mma(av[q].x, b1[q].x, acc[1][cc]);
							acc[0][cc] = ops::mma(av[q].y, b0[q].y, acc[0][cc]);
							acc[1][cc] = ops::mma(av[q].y, b1[q].y, acc[1][cc]);
						}
				}
			};
			run(0, g0, 0, 0, 0, 1);
			run(g0, g2, g.k0, 1, 0, 1);
			run(g0 + g2, 2 * g1, g.k0 + g.k2, 2, 1, 2);
#pragma unroll
			for(int u = 0; u < 2; u++) {
				const int j = 16 * (t0 + u) + li;
				if(j >= n4)
					continue;
#pragma unroll
				for(int e = 0; e < 4; e++) {
					const int row = ops::row(lq, e), ser = s0 + (row & 7);
					const bool south = row >= 8;
					if(ser >= g.n || (south && ring == N2))
						continue;
					T *o = map + (size_t) ser * npix + (south ? ss : sn) + j;
					const T s = acc[u][0][e] + acc[u][1][e], d = acc[u][0][e] - acc[u][1][e], U = acc[u][2][e], V = acc[u][3][e];
					o[0] = s + U;
					o[n4] = d - V;
					o[2 * n4] = s - U;
					o[3 * n4] = d + V;
				}
			}
		}
	}
}

/* the Legendre table: [16 rings][step][lane], the steps of an order those of
 * its even l - m and then of its odd ones, lane i + 16 q of step t holding
 * ring i at l - m = 2 (4 t + q) (+ 1); zeros past the last l and ring */
__global__ void k_hm_legendre(int L, int nside, int steps, const int *__restrict__ off, const double *__restrict__ cf, const double *__restrict__ cm, double *__restrict__ P)
{
	const int ring = blockIdx.x * 16 + (threadIdx.x & 15), m = blockIdx.y * (blockDim.x / 16) + threadIdx.x / 16;
	if(m > L)
		return;
	double z = 0., st = 0., phi0;
	int nphi;
	long start;
	const bool in = ring < 2 * nside;
	if(in)
		hp_ring(nside, ring + 1, &z, &st, &nphi, &start, &phi0);
	double p2 = in ? cm[m] : 0., b = st, p1 = 0.;
	for(int e = m; e; e >>= 1) {
		if(e & 1)
			p2 *= b;
		b *= b;
	}
	const int ke = ((L - m) / 2 + 4) / 4, ko = ((L - m + 1) / 2 + 3) / 4;
	double *o = P + ((size_t) blockIdx.x * steps + off[m]) * 64 + (threadIdx.x & 15);
	const double *c = cf + 2 * lm_offset(L, m, m);
	for(int d = 0; d < 8 * ke || d < 8 * ko; d++) {
		double v = 0.;
		if(d == 0)
			v = p2;
		else if(d <= L - m) {
			v = d == 1 ? c[2] * z * p2 : c[2 * d] * z * p1 - c[2 * d + 1] * p2;
			if(d > 1)
				p2 = p1;
			p1 = v;
		}
		const int k = d >> 1, t = k >> 2;
		if(d & 1) {
			if(t < ko)
				o[(size_t) (ke + t) * 64 + (k & 3) * 16] = v;
		} else if(t < ke)
			o[(size_t) t * 64 + (k & 3) * 16] = v;
	}
}

/* the pixel table: per tile of 16 pixels of a quarter ring the groups of
 * eight columns of S0, S2, then U and V in turn, [group][lane][2]: lane
 * i + 16 q holds pixel i at columns 2 q, 2 q + 1 */
template <typename T>
__global__ void k_hm_pixels(struct hm_geom g, T *__restrict__ W)
{
	const int ring = blockIdx.x + 1, L1 = g.L + 1;
	/* the rings past nside alternate between two tables: those of rings
	 * nside and nside + 1 */
	if(ring > g.nside + 1)
		return;
	const int n4 = ring < g.nside ? ring : g.nside, nt = (n4 + 15) / 16;
	const int g0 = g.k0 / 8, g2 = g.k2 / 8, g1 = g.k1 / 8;
	const long tile = 128L * (g0 + g2 + 2 * g1);
	T *o = W + (size_t) g.off[L1 + ring] * tile;
	const int half = ring < g.nside || !((ring + g.nside) & 1);	/* first pixel half a step in */
	for(long i = blockIdx.y * blockDim.x + threadIdx.x; i < nt * tile; i += blockDim.x * gridDim.y) {
		const int t = (int) (i / tile), r = (int) (i - t * tile);
		const int grp = r / 128, lane = (r >> 1) & 63, j = 16 * t + (lane & 15);
		const int col = 2 * (lane >> 4) + (r & 1), comp = col & 1;
		int m, v = 0;
		if(grp < g0)
			m = 2 * (8 * grp + col - comp);
		else if(grp < g0 + g2)
			m = 2 + 2 * (8 * (grp - g0) + col - comp);
		else {
			v = (grp - g0 - g2) & 1;
			m = 1 + 8 * ((grp - g0 - g2) >> 1) + col - comp;
		}
		T w = 0;
		if(m <= g.L && j < n4) {
			/* m phi = pi m (2 j + half) / (4 n4), the fraction reduced
			 * exactly */
			double sn, cs;
			sincospi((double) ((long) m * (2 * j + half) % (8L * n4)) / (4. * n4), &sn, &cs);
			if(!v)
				w = (T) (comp ? -sn : cs);
			else
				w = (T) ((m & 2) ? -(comp ? cs : sn) : (comp ? cs : sn));
		}
		o[i] = w;
	}
}

/*
 * Without the tables: workgroup = one ring x HP_SPW series, the coefficients
 * read from global memory.  The quarter turn shares the pixels' phases as in
 * k_healpix_mm: with m j = q nphi / 4 + r, exp(2 pi i m j / nphi) is i^q
 * exp(2 pi i r / nphi), so LDS holds a quarter of the ring's twiddles, at
 * exact integer indices, and a thread sums the pixels j + k nphi / 4
 * (k = 0..3) of a series from one read of each m's twiddle and (A, B).
 * nside twiddles fit beside the (A, B) of any order up to 1500 at nside 4096
 * (a whole ring's did not in float64).  Bound by the recurrences, which every
 * ring repeats: one float64 series of order 120 at nside 512 260 us with
 * whole rings, 205 so; of order 50 at nside 1024 417, 165.
 */
template <typename T>
__global__ void __launch_bounds__(HP_NT) k_healpix_ring(const cplx<T> *__restrict__ alm, int n, int L, int nside, const double *__restrict__ cf, const double *__restrict__ cm, T *__restrict__ map)
{
	extern __shared__ __align__(16) unsigned char hp_sm[];
	const int ring = blockIdx.x + 1, s0 = (blockIdx.z * gridDim.y + blockIdx.y) * HP_SPW, ns = n - s0 < HP_SPW ? n - s0 : HP_SPW;
	if(ns <= 0)
		return;
	double z, st, phi0;
	int nphi;
	long start;
	hp_ring(nside, ring, &z, &st, &nphi, &start, &phi0);
	const long npix = 12L * nside * nside;
	const int ncoef = (L + 1) * (L + 1), n4 = nphi / 4;
	cplx<T> *AB = reinterpret_cast<cplx<T> *>(hp_sm);		/* [HP_SPW][L + 1]: (A, B) */
	cplx<T> *tw = AB + HP_SPW * (L + 1);				/* [n4]: cos, sin */
	for(int k = threadIdx.x; k < n4; k += HP_NT) {
		double sn, cs;
		sincospi(2. * k / nphi, &sn, &cs);
		tw[k] = mk((T) cs, (T) sn);
	}
	/* Legendre sums: thread (series, |m|) */
	for(int t = threadIdx.x; t < ns * (L + 1); t += HP_NT) {
		const int sl = t / (L + 1), m = t - sl * (L + 1);
		const cplx<T> *a = alm + (size_t) (s0 + sl) * ncoef;
		/* Pbar_mm = cm[m] sin^m theta by repeated products */
		double p2 = cm[m];
		for(int k = 0; k < m; k++)
			p2 *= st;
		const cplx<T> *ap = a + lm_offset(L, m, m);
		const cplx<T> *an = m ? a + lm_offset(L, m, -m) : ap;
		double fpr = (double) ap[0].re * p2, fpi = (double) ap[0].im * p2;
		double fnr = (double) an[0].re * p2, fni = (double) an[0].im * p2;
		const double *c = cf + 2 * lm_offset(L, m, m);
		double p1 = 0.;
		if(m < L) {
			p1 = c[2] * z * p2;
			fpr = fma((double) ap[1].re, p1, fpr);
			fpi = fma((double) ap[1].im, p1, fpi);
			fnr = fma((double) an[1].re, p1, fnr);
			fni = fma((double) an[1].im, p1, fni);
		}
		for(int l = m + 2; l <= L; l++) {
			const int d = l - m;
			const double p = c[2 * d] * z * p1 - c[2 * d + 1] * p2;
			fpr = fma((double) ap[d].re, p, fpr);
			fpi = fma((double) ap[d].im, p, fpi);
			fnr = fma((double) an[d].re, p, fnr);
			fni = fma((double) an[d].im, p, fni);
			p2 = p1;
			p1 = p;
		}
		/* Pbar_l,-m = (-1)^m Pbar_lm; G_+-m = F_+-m exp(+-i m phi_0) */
		if(m & 1) {
			fnr = -fnr;
			fni = -fni;
		}
		double sn, cs;
		sincos(m * phi0, &sn, &cs);
		const double gpr = fpr * cs - fpi * sn, gpi = fpr * sn + fpi * cs;
		const double gnr = fnr * cs + fni * sn, gni = -fnr * sn + fni * cs;
		AB[t] = m ? mk((T) (gpr + gnr), (T) (gpi - gni)) : mk((T) gpr, (T) 0);
	}
	__syncthreads();
	/* pixels: thread (series, j).  C_m = A_m cos m phi - B_m sin m phi and
	 * D_m = A_m sin m phi + B_m cos m phi; S_k, T_k their sums over m = k
	 * mod 4 */
	for(int t = threadIdx.x; t < ns * n4; t += HP_NT) {
		const int sl = t / n4, j = t - sl * n4;
		const cplx<T> *ab = AB + sl * (L + 1);
		T S0 = ab[0].re, S1 = 0, S2 = 0, S3 = 0, T1 = 0, T3 = 0;
		int r = j, q = 0;	/* m j = q n4 + r, q mod 4 */
		auto term = [&](int m, int k) {
			const cplx<T> e = tw[r], c = ab[m];
			const T x = q & 1 ? e.im : e.re, y = q & 1 ? e.re : e.im;
			const T cs = q == 1 || q == 2 ? -x : x, sn = q & 2 ? -y : y;
			if(k == 0)
				S0 = fma(c.re, cs, fma(-c.im, sn, S0));
			else if(k == 2)
				S2 = fma(c.re, cs, fma(-c.im, sn, S2));
			else if(k == 1) {
				S1 = fma(c.re, cs, fma(-c.im, sn, S1));
				T1 = fma(c.re, sn, fma(c.im, cs, T1));
			} else {
				S3 = fma(c.re, cs, fma(-c.im, sn, S3));
				T3 = fma(c.re, sn, fma(c.im, cs, T3));
			}
			r += j;
			if(r >= n4) {
				r -= n4;
				q = (q + 1) & 3;
			}
		};
		int m = 1;
		for(; m + 3 <= L; m += 4) {
			term(m, 1);
			term(m + 1, 2);
			term(m + 2, 3);
			term(m + 3, 0);
		}
		for(; m <= L; m++)
			term(m, m & 3);
		T *o = map + (size_t) (s0 + sl) * npix + start + j;
		o[0] = (S0 + S2) + (S1 + S3);
		o[n4] = (S0 - S2) - (T1 - T3);
		o[2 * n4] = (S0 + S2) - (S1 + S3);
		o[3 * n4] = (S0 - S2) + (T1 - T3);
	}
}

/*
 * The posterior of the two beta skies of each event (RapidLocalization.py:
 * 498-530): prob = (e_p / sum e_p + e_n / sum e_n) / 2, e = exp(map -
 * max map); maps [2][E][npix], one workgroup of NT threads per event.  Two
 * reads of the maps: the first keeps a running maximum and the sum relative
 * to it per thread (rescaled when the maximum grows), the second forms the
 * probabilities; the maps of the events in flight fit the last-level cache,
 * so the second read is not one of HBM: 8192 events at nside 32 in float32
 * 0.46 -> 0.30 ms (1.2 GB), nine at nside 64 in float64 with 1024 threads
 * each 0.14 -> 0.065 ms.
 *
 * VW values per load: 16 bytes where the arrays are aligned for it (npix is
 * a multiple of 12, so every event's row then is).
 */
template <typename T, int VW, int NT>
__global__ void __launch_bounds__(NT) k_healpix_posterior(const T *__restrict__ maps, int E, long npix, T *__restrict__ prob)
{
	typedef T vec __attribute__((ext_vector_type(VW)));
	/* exp(x - max) in the maps' precision (float32 maps: float32
	 * exponentials, float64 sums) */
	auto ex = [](T x, double m) -> double { return sizeof(T) == sizeof(float) ? (double) expf((float) ((double) x - m)) : exp((double) x - m); };
	__shared__ double red[4][NT / 64];
	const int e = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const vec *mp = reinterpret_cast<const vec *>(maps + (size_t) e * npix), *mn = reinterpret_cast<const vec *>(maps + ((size_t) E + e) * npix);
	const long nv = npix / VW;
	double x[2] = { -INFINITY, -INFINITY }, s[2] = { 0., 0. };
	auto take = [&](vec v, int k) {
		T m = v[0];
#pragma unroll
		for(int i = 1; i < VW; i++)
			m = v[i] > m ? v[i] : m;
		if((double) m > x[k]) {
			/* the first values come with s = 0; NaN stays */
			s[k] = s[k] > 0. ? s[k] * exp(x[k] - (double) m) : s[k];
			x[k] = m;
		}
		/* values of minus infinity ahead of the first finite one add
		 * nothing, NaN does */
#pragma unroll
		for(int i = 0; i < VW; i++)
			s[k] += x[k] > -INFINITY || v[i] != v[i] ? ex(v[i], x[k]) : 0.;
	};
	constexpr int U = 4;	/* loads of each map in flight */
	long p = threadIdx.x;
	for(; p + (U - 1) * NT < nv; p += U * NT) {
		vec a[U], b[U];
#pragma unroll
		for(int u = 0; u < U; u++) {
			a[u] = mp[p + u * NT];
			b[u] = mn[p + u * NT];
		}
#pragma unroll
		for(int u = 0; u < U; u++) {
			take(a[u], 0);
			take(b[u], 1);
		}
	}
	for(; p < nv; p += NT) {
		take(mp[p], 0);
		take(mn[p], 1);
	}
	double xm[2], ip[2];
#pragma unroll
	for(int k = 0; k < 2; k++) {
		double m = x[k];
		for(int o = 32; o; o >>= 1)
			m = fmax(m, __shfl_xor(m, o));
		if(!lane)
			red[k][wave] = m;
	}
	__syncthreads();
#pragma unroll
	for(int k = 0; k < 2; k++) {
		xm[k] = red[k][0];
		for(int w = 1; w < NT / 64; w++)
			xm[k] = fmax(xm[k], red[k][w]);
		/* a thread without pixels has nothing to add */
		double t = s[k] > 0. ? s[k] * exp(x[k] - xm[k]) : s[k];
		for(int o = 32; o; o >>= 1)
			t += __shfl_xor(t, o);
		if(!lane)
			red[2 + k][wave] = t;
	}
	__syncthreads();
#pragma unroll
	for(int k = 0; k < 2; k++) {
		double t = 0.;
		for(int w = 0; w < NT / 64; w++)
			t += red[2 + k][w];
		ip[k] = 0.5 / t;
	}
	vec *pr = reinterpret_cast<vec *>(prob + (size_t) e * npix);
	auto put = [&](long q, vec a, vec b) {
		vec o;
#pragma unroll
		for(int i = 0; i < VW; i++)
			o[i] = (T) (ex(a[i], xm[0]) * ip[0] + ex(b[i], xm[1]) * ip[1]);
		pr[q] = o;
	};
	for(p = threadIdx.x; p + (U - 1) * NT < nv; p += U * NT) {
		vec a[U], b[U];
#pragma unroll
		for(int u = 0; u < U; u++) {
			a[u] = mp[p + u * NT];
			b[u] = mn[p + u * NT];
		}
#pragma unroll
		for(int u = 0; u < U; u++)
			put(p + u * NT, a[u], b[u]);
	}
	for(; p < nv; p += NT)
		put(p, mp[p], mn[p]);
}

/* ---------------------------------------------------------------- C ABI */

extern "C" int sphr_healpix_nside(unsigned l_max)
{
	/* lmax2nside, sh_series_healpix.cc:196-238 */
	const double x = ceil(l_max / 2. + 0.75);
	for(int i = 1; i > 0; i <<= 1)
		if(i >= x)
			return i;
	return -1;
}

static struct hm_geom hm_geom_of(const struct sphr_healpix *h, int n)
{
	struct hm_geom g;
	memset(&g, 0, sizeof(g));
	g.L = h->L;
	g.nside = h->nside;
	g.n = n;
	g.rc = h->rc;
	g.k0 = h->k0;
	g.k2 = h->k2;
	g.k1 = h->k1;
	/* row strides whose 16 rows start on distinct banks */
	const int f = h->precision == SPHR_MIXED;
	g.ld = h->k0 + h->k2 + h->k1 + (f ? 4 : 2);
	g.rs = 16 * g.ld + (f ? 16 : 8);
	g.steps = h->steps;
	g.chunks = h->rc ? (2 * h->nside + h->rc - 1) / h->rc : 0;
	g.groups = (n + HM_S - 1) / HM_S;
	g.P = h->P;
	g.off = h->off;
	return g;
}

static void drop_mm(struct sphr_healpix *h)
{
	void *p[] = { h->P, h->W, h->off };
	for(unsigned i = 0; i < sizeof(p) / sizeof(p[0]); i++)
		if(p[i])
			(void) hipFree(p[i]);
	h->P = NULL;
	h->W = NULL;
	h->off = NULL;
	h->rc = 0;
}

/* the tables of k_healpix_mm; left out, for the recurrences of
 * k_healpix_ring, where they would pass 512 MB, one ring's operand does not
 * fit in LDS, or there is no memory for them */
template <typename T>
static int build_mm(struct sphr_healpix *h)
{
	const int L = h->L, ns = h->nside, n0 = L / 4 + 1, n2 = L >= 2 ? (L - 2) / 4 + 1 : 0, n1 = (L + 1) / 2;
	h->k0 = (2 * n0 + 7) / 8 * 8;
	h->k2 = (2 * n2 + 7) / 8 * 8;
	h->k1 = (2 * n1 + 7) / 8 * 8;
	struct hm_geom g = hm_geom_of(h, 1);
	int rc = 16;
	while(rc && (size_t) rc * g.rs * sizeof(T) + HM_STAGE > 160 * 1024)
		rc >>= 1;
	int *off = (int *) malloc((L + 1 + 2 * (size_t) ns + 1) * sizeof(int));
	if(!off) {
		sphr_set_error("sphr_healpix_new: out of memory");
		return -1;
	}
	long steps = 0, tiles = 0;
	for(int m = 0; m <= L; m++) {
		off[m] = (int) steps;
		steps += ((L - m) / 2 + 4) / 4 + ((L - m + 1) / 2 + 3) / 4;
	}
	off[L + 1] = 0;
	for(int r = 1; r <= 2 * ns; r++) {
		off[L + 1 + r] = r > ns + 1 ? off[L + 1 + r - 2] : (int) tiles;
		if(r <= ns + 1)
			tiles += ((r < ns ? r : ns) + 15) / 16;
	}
	const size_t bP = (size_t) ((2 * ns + 15) / 16) * steps * 64 * sizeof(double);
	const size_t bW = (size_t) tiles * 16 * (h->k0 + h->k2 + 2 * h->k1) * sizeof(T);
	/* order 0 has no second coefficient to fetch */
	if(!rc || L == 0 || bP + bW > (size_t) 512 << 20) {
		free(off);
		return 0;
	}
	h->rc = rc;
	h->steps = (int) steps;
	hipStream_t st = sphr_rt_stream();
	int none = sphr_rt_check(hipMalloc(&h->P, bP), "hipMalloc") || sphr_rt_check(hipMalloc(&h->W, bW), "hipMalloc")
		   || sphr_rt_check(hipMalloc(&h->off, (L + 1 + 2 * (size_t) ns + 1) * sizeof(int)), "hipMalloc");
	if(none) {
		/* the maps need no tables */
		drop_mm(h);
		free(off);
		return 0;
	}
	const int bad = sphr_rt_check(hipMemcpy(h->off, off, (L + 1 + 2 * (size_t) ns + 1) * sizeof(int), hipMemcpyHostToDevice), "hipMemcpy");
	free(off);
	if(bad)
		return -1;
	hipLaunchKernelGGL(k_hm_legendre, dim3((2 * ns + 15) / 16, (L + 16) / 16), dim3(256), 0, st, L, ns, (int) steps, h->off, h->d_cf, h->d_cm, h->P);
	g = hm_geom_of(h, 1);
	/* a ring's table is long and the rings are few: sixteen workgroups each */
	hipLaunchKernelGGL((k_hm_pixels<T>), dim3(ns + 1, 16), dim3(256), 0, st, g, (T *) h->W);
	return sphr_rt_check(hipGetLastError(), "healpix tables") || sphr_rt_check(hipStreamSynchronize(st), "healpix tables") ? -1 : 0;
}

/* with tables, or for few series without */
static struct sphr_healpix *healpix_new(unsigned l_max, int nside, int precision, bool tables)
{
	if(sphr_gpu_ensure())
		return NULL;
	if(nside < 1 || nside > HP_NSIDE_MAX || (precision != SPHR_FP64 && precision != SPHR_MIXED) || l_max > 4096) {
		sphr_set_error("sphr_healpix_new: bad arguments (l_max %u, nside %d, precision %d)", l_max, nside, precision);
		return NULL;
	}
	const int L = (int) l_max, nal = (L + 1) * (L + 2) / 2;
	struct sphr_healpix *h = (struct sphr_healpix *) calloc(1, sizeof(*h));
	double *hc = (double *) calloc(2 * (size_t) nal + L + 1, sizeof(double));
	if(!h || !hc) {
		free(h);
		free(hc);
		sphr_set_error("sphr_healpix_new: out of memory");
		return NULL;
	}
	h->L = L;
	h->nside = nside;
	h->precision = precision;
	/* alpha_lm = sqrt((4 l^2 - 1) / (l^2 - m^2)) and its ratio to
	 * alpha_{l-1,m} at the (l, m) slot; Pbar_mm at the equator */
	for(int m = 0; m <= L; m++) {
		double prev = 1.;
		for(int l = m + 1; l <= L; l++) {
			const double a = sqrt((4. * l * l - 1.) / ((double) (l - m) * (l + m)));
			const int o = lm_offset(L, l, m);
			hc[2 * o] = a;
			hc[2 * o + 1] = l > m + 1 ? a / prev : 0.;
			prev = a;
		}
		double one;
		sphr_plm(m, m, 0.0, &one);
		hc[2 * (size_t) nal + m] = one;
	}
	if(sphr_rt_check(hipMalloc(&h->d_cf, (2 * (size_t) nal + L + 1) * sizeof(double)), "hipMalloc")
	   || sphr_rt_check(hipMemcpy(h->d_cf, hc, (2 * (size_t) nal + L + 1) * sizeof(double), hipMemcpyHostToDevice), "hipMemcpy")) {
		free(hc);
		sphr_healpix_free(h);
		return NULL;
	}
	h->d_cm = h->d_cf + 2 * (size_t) nal;
	free(hc);
	if(tables && (precision == SPHR_MIXED ? build_mm<float>(h) : build_mm<double>(h))) {
		sphr_healpix_free(h);
		return NULL;
	}
	return h;
}

extern "C" struct sphr_healpix *sphr_healpix_new(unsigned l_max, int nside, int precision)
{
	return healpix_new(l_max, nside, precision, true);
}

extern "C" struct sphr_healpix *sphr_healpix_new_few(unsigned l_max, int nside, int precision)
{
	return healpix_new(l_max, nside, precision, false);
}

extern "C" void sphr_healpix_free(struct sphr_healpix *h)
{
	if(!h)
		return;
	drop_mm(h);
	if(h->d_cf)
		hipFree(h->d_cf);
	free(h);
}

extern "C" long sphr_healpix_npix(const struct sphr_healpix *h)
{
	return h ? 12L * h->nside * h->nside : -1;
}

/* which kernel for n series: both times in us from their sizes, fitted to 446
 * measured shapes (orders 1-400, nside 1-512, 1-1024 series; the faster one
 * is taken, or one within 15 % of it, at all but two).  k_healpix_mm makes
 * eight series and sixteen rings at a time whatever it is asked for;
 * k_healpix_ring's workgroups are independent, but each repeats the
 * recurrences: one float64 series of order 120 at nside 64 takes 36 us there
 * and 90 with the tables, nine 194 and 93. */
static bool use_mm(const struct sphr_healpix *h, const struct hm_geom &g)
{
	if(!h->rc)
		return false;
	const double terms = (double) (h->L + 1) * (h->L + 1), rings = (double) g.n * h->nside;
	const double rounds = ceil((double) g.groups * g.chunks / sphr_rt_cus());
	const double groups = (h->k0 + h->k2 + 2 * h->k1) / 8, pixels = (h->precision == SPHR_MIXED ? 0.010 : 0.014) * (h->rc == 16 ? 2. : 1.);
	return rounds * (5.5 + 0.0024 * terms + pixels * h->nside * groups) < 4.4 + rings * (2.2e-5 * terms + 6e-4);
}

extern "C" int sphr_healpix_form(const struct sphr_healpix *h, int n)
{
	return h && n > 0 ? use_mm(h, hm_geom_of(h, n)) : -1;
}

extern "C" int sphr_healpix_maps(const struct sphr_healpix *h, const void *alm, int n, void *map, void *stream)
{
	if(!h || !alm || !map || n < 0) {
		sphr_set_error("sphr_healpix_maps: bad arguments");
		return -1;
	}
	if(!n)
		return 0;
	hipStream_t st = stream ? (hipStream_t) stream : sphr_rt_stream();
	const size_t esz = h->precision == SPHR_MIXED ? sizeof(float) : sizeof(double);
	const struct hm_geom g = hm_geom_of(h, n);
	if(use_mm(h, g)) {
		const unsigned grid = (unsigned) g.groups * g.chunks;
		const size_t lds = (size_t) g.rc * g.rs * esz + HM_STAGE;
		if(h->precision == SPHR_MIXED)
			hipLaunchKernelGGL(k_healpix_mm<float>, dim3(grid), dim3(HM_NT), lds, st, (const cplx<float> *) alm, g, (const float *) h->W, (float *) map);
		else
			hipLaunchKernelGGL(k_healpix_mm<double>, dim3(grid), dim3(HM_NT), lds, st, (const cplx<double> *) alm, g, (const double *) h->W, (double *) map);
	} else {
		/* one workgroup per (ring, HP_SPW series) */
		const size_t lr = 2 * (HP_SPW * (size_t) (h->L + 1) + (size_t) h->nside) * esz;
		if(lr > 160 * 1024) {
			sphr_set_error("sphr_healpix_maps: l_max %d with nside %d needs %zu bytes of LDS", h->L, h->nside, lr);
			return -1;
		}
		/* where a workgroup's series pass an XCD's L2 (4 MB) and all of
		 * them together the caches' share of it, LDS keeps the workgroups
		 * per CU few, which then read less past it (64 float64 series of
		 * order 400 at nside 256 99 -> 71 ms; with few series more
		 * workgroups are faster, one of order 300 631 against 724 us) */
		const size_t one = (size_t) (h->L + 1) * (h->L + 1) * 2 * esz;
		const size_t lds = HP_SPW * one > (size_t) 4 << 20 && n * one > (size_t) 64 << 20 && lr < 42 * 1024 ? 42 * 1024 : lr;
		/* (rings, groups of series in y and z: y ends at 65535) */
		const unsigned ng = (unsigned) (((long) n + HP_SPW - 1) / HP_SPW), ny = ng < 32768 ? ng : 32768;
		const dim3 grid(4 * h->nside - 1, ny, (ng + ny - 1) / ny);
		if(h->precision == SPHR_MIXED)
			hipLaunchKernelGGL(k_healpix_ring<float>, grid, dim3(HP_NT), lds, st, (const cplx<float> *) alm, n, h->L, h->nside, h->d_cf, h->d_cm, (float *) map);
		else
			hipLaunchKernelGGL(k_healpix_ring<double>, grid, dim3(HP_NT), lds, st, (const cplx<double> *) alm, n, h->L, h->nside, h->d_cf, h->d_cm, (double *) map);
	}
	return sphr_rt_check(hipGetLastError(), "k_healpix") ? -1 : 0;
}

/* 1024 threads per event where the events are too few to fill the chip with
 * smaller workgroups (one per CU) and their maps long enough for them; one
 * wave per event for many maps of at most 1024 pixels (5000 of 12 pixels
 * 16.4 us with four waves, 9.0 so; 3000 of 768 21.9 and 20.1; one of 768 8.2
 * with one wave, 5.2 with four) */
template <typename T>
static void launch_posterior(const T *maps, int E, long npix, T *prob, hipStream_t st)
{
	constexpr int V = 16 / sizeof(T);
	const bool al = ((uintptr_t) maps | (uintptr_t) prob) % 16 == 0;
	const bool small = npix <= 1024, few = E <= 2 * sphr_rt_cus();
	if(small && !few && al)
		hipLaunchKernelGGL((k_healpix_posterior<T, V, 64>), dim3(E), dim3(64), 0, st, maps, E, npix, prob);
	else if(small && !few)
		hipLaunchKernelGGL((k_healpix_posterior<T, 1, 64>), dim3(E), dim3(64), 0, st, maps, E, npix, prob);
	else if(!small && few && al)
		hipLaunchKernelGGL((k_healpix_posterior<T, V, 1024>), dim3(E), dim3(1024), 0, st, maps, E, npix, prob);
	else if(!small && few)
		hipLaunchKernelGGL((k_healpix_posterior<T, 1, 1024>), dim3(E), dim3(1024), 0, st, maps, E, npix, prob);
	else if(al)
		hipLaunchKernelGGL((k_healpix_posterior<T, V, 256>), dim3(E), dim3(256), 0, st, maps, E, npix, prob);
	else
		hipLaunchKernelGGL((k_healpix_posterior<T, 1, 256>), dim3(E), dim3(256), 0, st, maps, E, npix, prob);
}

extern "C" int sphr_healpix_posterior(const struct sphr_healpix *h, const void *maps, int n_events, void *prob, void *stream)
{
	if(!h || !maps || !prob || n_events < 0) {
		sphr_set_error("sphr_healpix_posterior: bad arguments");
		return -1;
	}
	if(!n_events)
		return 0;
	hipStream_t st = stream ? (hipStream_t) stream : sphr_rt_stream();
	const long npix = 12L * h->nside * h->nside;
	if(h->precision == SPHR_MIXED)
		launch_posterior<float>((const float *) maps, n_events, npix, (float *) prob, st);
	else
		launch_posterior<double>((const double *) maps, n_events, npix, (double *) prob, st);
	return sphr_rt_check(hipGetLastError(), "k_healpix_posterior") ? -1 : 0;
}

/* sh_series_write_healpix_map (sh_series_healpix.cc:247-286): the map of
 * Re f at nside = lmax2nside(l_max), RING order, to a FITS file */
extern "C" int sh_series_write_healpix_map(const struct sh_series *series, const char *filename)
{
	if(!series || !filename) {
		sphr_set_error("sh_series_write_healpix_map: bad arguments");
		return -1;
	}
	const int L = (int) series->l_max, nside = sphr_healpix_nside(series->l_max);
	if(nside < 1)
		return -1;
	const size_t ncoef = (size_t) (L + 1) * (L + 1);
	const long npix = 12L * nside * nside;
	double _Complex *full = (double _Complex *) calloc(ncoef, sizeof(*full));
	double *hmap = (double *) malloc(npix * sizeof(double));
	struct sphr_healpix *h = NULL;
	void *d_alm = NULL, *d_map = NULL;
	int rc = -1;
	if(!full || !hmap) {
		sphr_set_error("sh_series_write_healpix_map: out of memory");
		goto done;
	}
	/* the full coefficient layout (a polar series has m = 0 only) */
	for(int l = 0; l <= L; l++)
		for(int m = series->polar ? 0 : -l; m <= (series->polar ? 0 : l); m++)
			full[lm_offset(L, l, m)] = sh_series_get(series, l, m);
	h = healpix_new(series->l_max, nside, SPHR_FP64, false);
	if(!h || sphr_rt_check(hipMalloc(&d_alm, ncoef * sizeof(*full)), "hipMalloc") || sphr_rt_check(hipMalloc(&d_map, npix * sizeof(double)), "hipMalloc")
	   || sphr_memcpy_htod(d_alm, full, ncoef * sizeof(*full)) || sphr_healpix_maps(h, d_alm, 1, d_map, NULL)
	   || sphr_memcpy_dtoh(hmap, d_map, npix * sizeof(double)))
		goto done;
	rc = sphr_fits_write_healpix_map(filename, hmap, nside);
done:
	if(d_alm)
		hipFree(d_alm);
	if(d_map)
		hipFree(d_map);
	sphr_healpix_free(h);
	free(full);
	free(hmap);
	return rc;
}
