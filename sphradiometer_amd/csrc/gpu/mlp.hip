/*
 * The learned peak proposal: a multilayer perceptron from the real-form SH
 * coefficients of a sky to K candidate peak directions, trained and run
 * with the kernels of this file.
 *
 *   h_0 = x (n_in), z_i = h_{i-1} W_i + b_i, h_i = GELU(z_i) (i = 1..depth),
 *   y = h_depth W_out + b_out (3 K outputs), candidate k = y[3k..3k+2] / |.|
 *
 * Weights are kept in float32 (master copy, Adam state).  The products run
 * on bfloat16 operands with float32 accumulation (mlp_bf16.hip) or, to
 * check gradients, on float32 operands (MFMA 16x16x4 f32, this file).
 *
 * Loss per sample, with t the unit target and d_k = 1 - c_k . t:
 *   min_k d_k + (lambda / K) sum_k d_k,
 * so the best candidate is pulled onto the target and the others stay
 * trained.
 */
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <sphradiometer/sphradiometer_batch.h>
#include "../sphr_internal.h"
#include "kernels.h"
#include "runtime.h"
#include "mlp_bf16.h"

extern "C" int sphr_mlp_set_params(struct sphr_mlp *, const float *);

/* ------------------------------------------------------------------ */
/* GEMM C[M][N] = op(A)[M][K] op(B)[K][N], float32                     */
/* ------------------------------------------------------------------ */

#define MG_BM 64
#define MG_BN 64
#define MG_KC 32
#define MG_PAD 4

typedef float f4v __attribute__((ext_vector_type(4)));

template <int TA, int TB>
__global__ void __launch_bounds__(256) k_mlp_gemm(int M, int N, int K, const float *__restrict__ A, int lda, const float *__restrict__ B, int ldb, float *__restrict__ C, int ldc)
{
	__shared__ __align__(16) float sA[MG_BM][MG_KC + MG_PAD];	/* [row][k] */
	__shared__ __align__(16) float sB[MG_BN][MG_KC + MG_PAD];	/* [col][k] */
	const int m0 = blockIdx.y * MG_BM, n0 = blockIdx.x * MG_BN;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
	const int li = lane & 15, lq = lane >> 4;
	f4v acc[2][2];
	for(int a = 0; a < 2; a++)
		for(int b = 0; b < 2; b++)
			acc[a][b] = (f4v) 0;
	for(int k0 = 0; k0 < K; k0 += MG_KC) {
		for(int idx = threadIdx.x; idx < MG_BM * MG_KC; idx += 256) {
			int i, k;
			if(TA) {
				k = idx / MG_BM;
				i = idx - k * MG_BM;
			} else {
				i = idx / MG_KC;
				k = idx - i * MG_KC;
			}
			const int gi = m0 + i, gk = k0 + k;
			float v = 0.f;
			if(gi < M && gk < K)
				v = TA ? A[(size_t) gk * lda + gi] : A[(size_t) gi * lda + gk];
			sA[i][k] = v;
		}
		for(int idx = threadIdx.x; idx < MG_BN * MG_KC; idx += 256) {
			int j, k;
			if(TB) {
				j = idx / MG_KC;
				k = idx - j * MG_KC;
			} else {
				k = idx / MG_BN;
				j = idx - k * MG_BN;
			}
			const int gj = n0 + j, gk = k0 + k;
			float v = 0.f;
			if(gj < N && gk < K)
				v = TB ? B[(size_t) gj * ldb + gk] : B[(size_t) gk * ldb + gj];
			sB[j][k] = v;
		}
		__syncthreads();
		for(int ks = 0; ks < MG_KC; ks += 4)
			for(int a = 0; a < 2; a++)
				for(int b = 0; b < 2; b++)
					acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(sA[wm + 16 * a + li][ks + lq], sB[wn + 16 * b + li][ks + lq], acc[a][b], 0, 0, 0);
		__syncthreads();
	}
	for(int a = 0; a < 2; a++)
		for(int b = 0; b < 2; b++) {
			const int gj = n0 + wn + 16 * b + li;
			if(gj >= N)
				continue;
			for(int e = 0; e < 4; e++) {
				const int gi = m0 + wm + 16 * a + 4 * lq + e;
				if(gi < M)
					C[(size_t) gi * ldc + gj] = acc[a][b][e];
			}
		}
}

static int mlp_gemm(int ta, int tb, int M, int N, int K, const float *A, int lda, const float *B, int ldb, float *C, int ldc, hipStream_t st)
{
	dim3 grid((N + MG_BN - 1) / MG_BN, (M + MG_BM - 1) / MG_BM);
	if(!ta && !tb)
		hipLaunchKernelGGL((k_mlp_gemm<0, 0>), grid, dim3(256), 0, st, M, N, K, A, lda, B, ldb, C, ldc);
	else if(ta && !tb)
		hipLaunchKernelGGL((k_mlp_gemm<1, 0>), grid, dim3(256), 0, st, M, N, K, A, lda, B, ldb, C, ldc);
	else if(!ta && tb)
		hipLaunchKernelGGL((k_mlp_gemm<0, 1>), grid, dim3(256), 0, st, M, N, K, A, lda, B, ldb, C, ldc);
	else
		return -1;
	return hipGetLastError() == hipSuccess ? 0 : -1;
}

/* ------------------------------------------------------------------ */
/* elementwise and reductions                                          */
/* ------------------------------------------------------------------ */

__device__ inline float gelu(float z)
{
	return 0.5f * z * (1.f + erff(z * 0.70710678118654752f));
}

__device__ inline float gelu_d(float z)
{
	return 0.5f * (1.f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

/* z += b; h = GELU(z) (hidden layers) */
__global__ void k_bias_gelu(float *__restrict__ Z, const float *__restrict__ b, int rows, int n, float *__restrict__ H)
{
	const long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
	if(i >= (long) rows * n)
		return;
	const float z = Z[i] + b[i % n];
	Z[i] = z;
	H[i] = gelu(z);
}

__global__ void k_bias(float *__restrict__ Z, const float *__restrict__ b, int rows, int n)
{
	const long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
	if(i >= (long) rows * n)
		return;
	Z[i] += b[i % n];
}

/* dZ = dH * GELU'(Z) */
__global__ void k_gelu_back(const float *__restrict__ dH, const float *__restrict__ Z, long count, float *__restrict__ dZ)
{
	const long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
	if(i >= count)
		return;
	dZ[i] = dH[i] * gelu_d(Z[i]);
}

/* db[j] = sum_r dZ[r][j]: 64 columns per workgroup, the rows over its four
 * waves */
__global__ void __launch_bounds__(256) k_colsum(const float *__restrict__ dZ, int rows, int n, float *__restrict__ db)
{
	__shared__ float part[4][64];
	const int c = threadIdx.x & 63, w = threadIdx.x >> 6, j = blockIdx.x * 64 + c;
	float s = 0.f;
	if(j < n)
		for(int r = w; r < rows; r += 4)
			s += dZ[(size_t) r * n + j];
	part[w][c] = s;
	__syncthreads();
	if(w == 0 && j < n)
		db[j] = (part[0][c] + part[1][c]) + (part[2][c] + part[3][c]);
}

/* candidate loss and its gradient; one thread per sample */
__global__ void k_loss(const float *__restrict__ Y, const float *__restrict__ T, int rows, int K, float lambda, float *__restrict__ loss, float *__restrict__ dY)
{
	const int r = blockIdx.x * blockDim.x + threadIdx.x;
	if(r >= rows)
		return;
	const float *y = Y + (size_t) r * 3 * K;
	const float t0 = T[3 * r], t1 = T[3 * r + 1], t2 = T[3 * r + 2];
	float d[16], nrm[16], dot[16];
	int best = 0;
	for(int k = 0; k < K; k++) {
		const float n = sqrtf(y[3 * k] * y[3 * k] + y[3 * k + 1] * y[3 * k + 1] + y[3 * k + 2] * y[3 * k + 2]) + 1e-12f;
		const float c = (y[3 * k] * t0 + y[3 * k + 1] * t1 + y[3 * k + 2] * t2) / n;
		nrm[k] = n;
		dot[k] = c;
		d[k] = 1.f - c;
		if(d[k] < d[best])
			best = k;
	}
	float l = d[best], sum = 0.f;
	for(int k = 0; k < K; k++)
		sum += d[k];
	l += lambda / K * sum;
	if(loss)
		loss[r] = l;
	if(dY) {
		const float inv_rows = 1.f / rows;
		for(int k = 0; k < K; k++) {
			const float w = ((k == best) ? 1.f : 0.f) + lambda / K;
			const float n = nrm[k];
			const float c0 = y[3 * k] / n, c1 = y[3 * k + 1] / n, c2 = y[3 * k + 2] / n;
			/* d(1 - c.t)/dy = -(t - (c.t) c) / |y| */
			float *g = dY + (size_t) r * 3 * K + 3 * k;
			g[0] = -w * (t0 - dot[k] * c0) / n * inv_rows;
			g[1] = -w * (t1 - dot[k] * c1) / n * inv_rows;
			g[2] = -w * (t2 - dot[k] * c2) / n * inv_rows;
		}
	}
}

__global__ void k_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m, float *__restrict__ v, long n, float lr, float b1, float b2, float eps, float c1, float c2)
{
	const long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
	if(i >= n)
		return;
	const float gi = g[i];
	const float mi = b1 * m[i] + (1.f - b1) * gi;
	const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
	m[i] = mi;
	v[i] = vi;
	p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

/* real-form SH coefficients of a real sky, scaled to unit RMS:
 * Re a_l0 (l = 0..L), then for m = 1..L, l = m..L: Re a_lm, Im a_lm */
template <typename TA>
__global__ void __launch_bounds__(256) k_features(const cplx<TA> *__restrict__ alm, int L, float *__restrict__ out)
{
	const int s = blockIdx.x;
	const int ncoef = (L + 1) * (L + 1);
	const cplx<TA> *a = alm + (size_t) s * ncoef;
	float *o = out + (size_t) s * ncoef;
	__shared__ float red[256];
	float ss = 0.f;
	for(int i = threadIdx.x; i < ncoef; i += 256) {
		float v;
		if(i <= L)
			v = (float) a[i].re;
		else {
			const int c = (L + 1) + (i - (L + 1)) / 2;	/* the m > 0 coefficient */
			v = ((i - (L + 1)) & 1) ? (float) a[c].im : (float) a[c].re;
		}
		o[i] = v;
		ss += v * v;
	}
	red[threadIdx.x] = ss;
	__syncthreads();
	for(int w = 128; w > 0; w >>= 1) {
		if(threadIdx.x < w)
			red[threadIdx.x] += red[threadIdx.x + w];
		__syncthreads();
	}
	const float scale = red[0] > 0.f ? rsqrtf(red[0] / ncoef) : 0.f;
	for(int i = threadIdx.x; i < ncoef; i += 256)
		o[i] *= scale;
}

/* candidate directions as (theta, phi) seeds, [rows][K][2] */
__global__ void k_seeds(const float *__restrict__ Y, int rows, int K, double *__restrict__ seeds)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if(i >= rows * K)
		return;
	const float *y = Y + 3 * (size_t) i;
	const double x = y[0], yy = y[1], z = y[2];
	double ph = atan2(yy, x);
	if(ph < 0)
		ph += 2 * M_PI;
	seeds[2 * (size_t) i] = atan2(sqrt(x * x + yy * yy), z);
	seeds[2 * (size_t) i + 1] = ph;
}

/* ------------------------------------------------------------------ */
/* the network object                                                  */
/* ------------------------------------------------------------------ */

struct sphr_mlp {
	int n_in, width, depth, K, max_batch, bf16;
	int nl;				/* layers = depth + 1 */
	int din[MLP_MAX_LAYERS], dout[MLP_MAX_LAYERS];
	size_t ow[MLP_MAX_LAYERS], ob[MLP_MAX_LAYERS];
	size_t nparam;
	float *p, *g, *m, *v;		/* params, grads, Adam moments */
	struct mlp_bf bf;		/* the bfloat16 form's buffers */
	/* the float32 form's */
	float *Z[MLP_MAX_LAYERS];	/* pre-activations [max_batch][dout] */
	float *H[MLP_MAX_LAYERS];	/* activations */
	float *dA, *dZ;			/* [max_batch][max width] */
	float *loss;			/* [max_batch] */
	/* [max_batch][3 K] outputs of the last forward */
	const float *y;
};

extern "C" void sphr_mlp_free(struct sphr_mlp *m)
{
	if(!m)
		return;
	void *ptrs[] = { m->p, m->g, m->m, m->v, m->dA, m->dZ, m->loss };
	for(unsigned i = 0; i < sizeof(ptrs) / sizeof(ptrs[0]); i++)
		if(ptrs[i])
			hipFree(ptrs[i]);
	for(int l = 0; l < m->nl; l++) {
		if(m->Z[l])
			hipFree(m->Z[l]);
		if(m->H[l])
			hipFree(m->H[l]);
	}
	mlp_bf_free(&m->bf);
	free(m);
}

extern "C" struct sphr_mlp *sphr_mlp_new(int n_in, int width, int depth, int n_candidates, int max_batch, int bf16, unsigned long long seed)
{
	if(sphr_gpu_ensure())
		return NULL;
	if(n_in < 1 || width < 1 || depth < 1 || depth + 1 > MLP_MAX_LAYERS || n_candidates < 1 || n_candidates > 16 || max_batch < 1) {
		sphr_set_error("sphr_mlp_new: bad shape");
		return NULL;
	}
	struct sphr_mlp *m = (struct sphr_mlp *) calloc(1, sizeof(*m));
	if(!m)
		return NULL;
	m->n_in = n_in;
	m->width = width;
	m->depth = depth;
	m->K = n_candidates;
	m->max_batch = max_batch;
	m->bf16 = bf16 ? 1 : 0;
	m->nl = depth + 1;
	size_t off = 0;
	for(int l = 0; l < m->nl; l++) {
		m->din[l] = l ? width : n_in;
		m->dout[l] = l < depth ? width : 3 * n_candidates;
		m->ow[l] = off;
		off += (size_t) m->din[l] * m->dout[l];
		m->ob[l] = off;
		off += m->dout[l];
	}
	m->nparam = off;
	const size_t wmax = width > 3 * n_candidates ? width : 3 * n_candidates;
	const size_t B = max_batch;
	int bad = sphr_rt_check(hipMalloc(&m->p, off * 4), "hipMalloc") || sphr_rt_check(hipMalloc(&m->g, off * 4), "hipMalloc")
		  || sphr_rt_check(hipMalloc(&m->m, off * 4), "hipMalloc") || sphr_rt_check(hipMalloc(&m->v, off * 4), "hipMalloc");
	if(m->bf16) {
		bad = bad || mlp_bf_alloc(&m->bf, m->nl, m->din, m->dout, m->ow, m->ob, m->K, max_batch);
		m->y = m->bf.Z[m->nl - 1];
	} else {
		bad = bad || sphr_rt_check(hipMalloc(&m->dA, B * wmax * 4), "hipMalloc") || sphr_rt_check(hipMalloc(&m->dZ, B * wmax * 4), "hipMalloc")
		      || sphr_rt_check(hipMalloc(&m->loss, B * 4), "hipMalloc");
		for(int l = 0; l < m->nl && !bad; l++)
			bad = sphr_rt_check(hipMalloc(&m->Z[l], B * m->dout[l] * 4), "hipMalloc") || sphr_rt_check(hipMalloc(&m->H[l], B * m->dout[l] * 4), "hipMalloc");
		m->y = m->Z[m->nl - 1];
	}
	if(bad) {
		sphr_mlp_free(m);
		return NULL;
	}
	/* He-style initialisation from a seeded splitmix64 stream */
	float *h = (float *) malloc(off * sizeof(float));
	if(!h) {
		sphr_mlp_free(m);
		return NULL;
	}
	uint64_t st = seed * 0x9e3779b97f4a7c15ull + 1;
	for(int l = 0; l < m->nl; l++) {
		const double sc = sqrt(2.0 / m->din[l]) * (l == m->nl - 1 ? 0.5 : 1.0);
		for(size_t i = 0; i < (size_t) m->din[l] * m->dout[l]; i++) {
			double u[2];
			for(int q = 0; q < 2; q++) {
				uint64_t z = (st += 0x9e3779b97f4a7c15ull);
				z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
				z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
				z ^= z >> 31;
				u[q] = ((z >> 11) + 0.5) * (1.0 / 9007199254740992.0);
			}
			h[m->ow[l] + i] = (float) (sc * sqrt(-2.0 * log(u[0])) * cos(2 * M_PI * u[1]));
		}
		for(int j = 0; j < m->dout[l]; j++)
			h[m->ob[l] + j] = 0.f;
	}
	const int rc = sphr_mlp_set_params(m, h);
	free(h);
	if(rc || sphr_rt_check(hipMemset(m->m, 0, off * 4), "hipMemset") || sphr_rt_check(hipMemset(m->v, 0, off * 4), "hipMemset")) {
		sphr_mlp_free(m);
		return NULL;
	}
	return m;
}

extern "C" int sphr_mlp_set_params(struct sphr_mlp *m, const float *host)
{
	hipStream_t st = sphr_rt_stream();
	if(sphr_rt_check(hipMemcpyAsync(m->p, host, m->nparam * 4, hipMemcpyHostToDevice, st), "hipMemcpy") || (m->bf16 && mlp_bf_refresh(&m->bf, m->p, st)))
		return -1;
	return sphr_rt_check(hipStreamSynchronize(st), "synchronize");
}

extern "C" int sphr_mlp_get_params(const struct sphr_mlp *m, float *host)
{
	return sphr_rt_check(hipMemcpy(host, m->p, m->nparam * 4, hipMemcpyDeviceToHost), "hipMemcpy");
}

extern "C" int sphr_mlp_get_grads(const struct sphr_mlp *m, float *host)
{
	return sphr_rt_check(hipMemcpy(host, m->g, m->nparam * 4, hipMemcpyDeviceToHost), "hipMemcpy");
}

extern "C" long sphr_mlp_n_params(const struct sphr_mlp *m)
{
	return (long) m->nparam;
}

static int forward_f32(struct sphr_mlp *m, const float *x, int B, hipStream_t st)
{
	const float *in = x;
	for(int l = 0; l < m->nl; l++) {
		if(mlp_gemm(0, 0, B, m->dout[l], m->din[l], in, m->din[l], m->p + m->ow[l], m->dout[l], m->Z[l], m->dout[l], st))
			return -1;
		const long n = (long) B * m->dout[l];
		if(l < m->depth)
			hipLaunchKernelGGL(k_bias_gelu, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, st, m->Z[l], m->p + m->ob[l], B, m->dout[l], m->H[l]);
		else
			hipLaunchKernelGGL(k_bias, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, st, m->Z[l], m->p + m->ob[l], B, m->dout[l]);
		in = m->H[l];
	}
	return hipGetLastError() == hipSuccess ? 0 : -1;
}

static int backward_f32(struct sphr_mlp *m, const float *x, int B, hipStream_t st)
{
	/* dY is in dZ on entry */
	for(int l = m->nl - 1; l >= 0; l--) {
		const int di = m->din[l], dn = m->dout[l];
		const float *in = l ? m->H[l - 1] : x;
		/* dW = in^T dZ, db = colsum dZ */
		if(mlp_gemm(1, 0, di, dn, B, in, di, m->dZ, dn, m->g + m->ow[l], dn, st))
			return -1;
		hipLaunchKernelGGL(k_colsum, dim3((dn + 63) / 64), dim3(256), 0, st, m->dZ, B, dn, m->g + m->ob[l]);
		if(l == 0)
			break;
		/* dA = dZ W^T, then through GELU of layer l-1 */
		if(mlp_gemm(0, 1, B, di, dn, m->dZ, dn, m->p + m->ow[l], dn, m->dA, di, st))
			return -1;
		const long n = (long) B * di;
		hipLaunchKernelGGL(k_gelu_back, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, st, m->dA, m->Z[l - 1], n, m->dZ);
	}
	return hipGetLastError() == hipSuccess ? 0 : -1;
}

static hipStream_t pick(void *stream)
{
	return stream ? (hipStream_t) stream : sphr_rt_stream();
}

extern "C" int sphr_mlp_forward(struct sphr_mlp *m, const float *x, int B, float *y, void *stream)
{
	if(!m || !x || B < 1 || B > m->max_batch)
		return -1;
	hipStream_t st = pick(stream);
	if(m->bf16 ? mlp_bf_forward(&m->bf, m->p, x, B, st) : forward_f32(m, x, B, st))
		return -1;
	if(y)
		return sphr_rt_check(hipMemcpyAsync(y, m->y, (size_t) B * 3 * m->K * 4, hipMemcpyDeviceToDevice, st), "hipMemcpy");
	return 0;
}

/* forward, loss and gradients (into the grad buffer) for a batch; per
 * sample losses to loss (device, may be NULL) */
extern "C" int sphr_mlp_loss_grad(struct sphr_mlp *m, const float *x, const float *target, int B, float lambda, float *loss, void *stream)
{
	if(!m || !x || !target || B < 1 || B > m->max_batch)
		return -1;
	hipStream_t st = pick(stream);
	if(m->bf16)
		return mlp_bf_loss_grad(&m->bf, m->p, m->g, x, target, B, lambda, loss, NULL, NULL, NULL, st);
	if(forward_f32(m, x, B, st))
		return -1;
	hipLaunchKernelGGL(k_loss, dim3((B + 255) / 256), dim3(256), 0, st, m->Z[m->nl - 1], target, B, m->K, lambda, loss ? loss : m->loss, m->dZ);
	if(hipGetLastError() != hipSuccess)
		return -1;
	return backward_f32(m, x, B, st);
}

static struct mlp_adam adam_args(float lr, float beta1, float beta2, float eps, int step)
{
	struct mlp_adam a = { lr, beta1, beta2, eps, 1.f - powf(beta1, (float) step), 1.f - powf(beta2, (float) step) };
	return a;
}

extern "C" int sphr_mlp_adam(struct sphr_mlp *m, float lr, float beta1, float beta2, float eps, int step, void *stream)
{
	hipStream_t st = pick(stream);
	const struct mlp_adam a = adam_args(lr, beta1, beta2, eps, step);
	if(m->bf16)
		return mlp_bf_adam(&m->bf, m->p, m->g, m->m, m->v, &a, st);
	const long n = (long) m->nparam;
	hipLaunchKernelGGL(k_adam, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, st, m->p, m->g, m->m, m->v, n, a.lr, a.b1, a.b2, a.eps, a.c1, a.c2);
	return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int sphr_mlp_train_step(struct sphr_mlp *m, const float *x, const float *target, int B, float lambda, float lr, int step, float *loss, void *stream)
{
	if(m && m->bf16 && x && target && B >= 1 && B <= m->max_batch) {
		const struct mlp_adam a = adam_args(lr, 0.9f, 0.999f, 1e-8f, step);
		return mlp_bf_loss_grad(&m->bf, m->p, m->g, x, target, B, lambda, loss, &a, m->m, m->v, pick(stream));
	}
	if(sphr_mlp_loss_grad(m, x, target, B, lambda, loss, stream))
		return -1;
	return sphr_mlp_adam(m, lr, 0.9f, 0.999f, 1e-8f, step, stream);
}

/* candidate seeds (theta, phi) for rows x K from the last forward */
extern "C" int sphr_mlp_seeds(struct sphr_mlp *m, int B, double *seeds, void *stream)
{
	hipStream_t st = pick(stream);
	const int n = B * m->K;
	hipLaunchKernelGGL(k_seeds, dim3((n + 255) / 256), dim3(256), 0, st, m->y, B, m->K, seeds);
	return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int sphr_features(const void *alm, int alm_f32, int S, int L, float *out, void *stream)
{
	hipStream_t st = pick(stream);
	if(alm_f32)
		hipLaunchKernelGGL((k_features<float>), dim3(S), dim3(256), 0, st, (const cplx<float> *) alm, L, out);
	else
		hipLaunchKernelGGL((k_features<double>), dim3(S), dim3(256), 0, st, (const cplx<double> *) alm, L, out);
	return hipGetLastError() == hipSuccess ? 0 : -1;
}

/* test hook: one GEMM of the network's operand type on device float
 * inputs, C = op(A) op(B) */
extern "C" int sphr_mlp_gemm_check(int bf16, int ta, int tb, int M, int N, int K, const float *A, const float *B, float *C)
{
	hipStream_t st = sphr_rt_stream();
	if(bf16)
		return ta && tb ? -1 : mlp_bf_gemm(ta, tb, M, N, K, A, B, C, st);
	if(mlp_gemm(ta, tb, M, N, K, A, ta ? M : K, B, tb ? K : N, C, N, st))
		return -1;
	return sphr_rt_check(hipStreamSynchronize(st), "synchronize");
}
