/*
 * The proposal network with bfloat16 operands and float32 accumulation
 * (v_mfma_f32_16x16x32_bf16): forward, loss, backward and Adam.
 *
 * Every product runs as C[m][n] = sum_k A[m][k] B[n][k] with both operands
 * K-contiguous, so that each lane's eight values are one 16-byte read.
 * That needs the activations and the output gradients in both
 * orientations (rows are K in the next layer, columns are K in the weight
 * gradients) and the weights too; the launch that makes an array writes
 * both.  Dimensions are padded to multiples of 128 with zeros, so the
 * products test no bounds.
 *
 * One training step is depth + 4 + (depth - 1) launches:
 *   k_in      x to bfloat16, both orientations
 *   k_nt      per hidden layer: z = A W + b, GELU, both orientations
 *   k_head    output layer, loss, its gradient and the last hidden layer's
 *   k_nt      per remaining hidden layer: dZ = (dZ W^T) GELU'(z)
 *   k_dw      all layers' weight gradients, K = the batch split
 *   k_update  sums the splits, and in a training step applies Adam and
 *             writes the operand weights
 * What bounds it: at 2048 rows of 1089 -> 3 x 512 -> 12 the step is 11
 * GFLOP (10 us at the 1.1 PFLOP/s a large product reaches) in nine
 * launches of 9-18 us each, most of them one round of workgroups that
 * wait for their first loads and write both orientations.  The step took
 * 3.1 ms as one-value-per-load products without batch splits and column
 * sums of one thread per column (k_colsum alone 1.6 ms), 0.10 ms as here;
 * sixteen steps and the weights' copy to the host 49.6 -> 2.05 ms.  Eight
 * waves of 16 x 32 and K chunks of 128 against four of 32 x 32 or chunks
 * of 64: 2.05 ms against 2.26 and 2.17 (both 2.36).
 */
#include <hip/hip_runtime.h>
#include <string.h>
#include "kernels.h"
#include "runtime.h"
#include "mlp_bf16.h"

namespace {

typedef bf16_t b8 __attribute__((ext_vector_type(8)));
typedef bf16_t b4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

#define NT_T 64			/* rows and columns of a tile */
#define NT_KC 128		/* K per staged chunk */
#define NT_W 8			/* waves of a workgroup */
#define NT_LD (NT_KC + 8)	/* LDS row stride: 16 rows' 16-byte reads on distinct banks */
#define NT_MB (8 / NT_W)	/* 16-row blocks of a wave */
#define NT_VT (NT_KC / 8)	/* threads per staged row */
#define NT_VR (64 * NT_W / NT_VT)	/* rows per staging step */
#define NT_VS (NT_T / NT_VR)

__device__ inline float gelu(float z)
{
	return 0.5f * z * (1.f + erff(z * 0.70710678118654752f));
}

__device__ inline float gelu_d(float z)
{
	return 0.5f * (1.f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

__device__ inline f4 mma(b8 a, b8 b, f4 c)
{
	return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

/* a 64 x 64 tile of A B^T over the chunks [c0, c1) of NT_KC: eight waves of
 * 16 x 32, the next chunk's global loads in flight during this chunk's
 * products, two LDS buffers and one barrier per chunk.  Accumulator
 * element e of lane i + 16 q holds row 4 q + e, column i of a 16 x 16
 * block. */
struct nt_lds {
	bf16_t a[2][NT_T][NT_LD], b[2][NT_T][NT_LD];
};

__device__ inline void nt_tile(struct nt_lds &s, const bf16_t *__restrict__ A, size_t lda, const bf16_t *__restrict__ B, size_t ldb, int c0, int c1, f4 (&acc)[NT_MB][2])
{
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int wm = wave % (NT_W / 2) * (16 * NT_MB), wn = wave / (NT_W / 2) * 32;
	const int li = lane & 15, lq = lane >> 4;
	const int vr = threadIdx.x / NT_VT, vc = threadIdx.x % NT_VT * 8;
	b8 ra[NT_VS], rb[NT_VS];
	auto load = [&](int c) {
#pragma unroll
		for(int u = 0; u < NT_VS; u++) {
			ra[u] = *reinterpret_cast<const b8 *>(A + (vr + NT_VR * u) * lda + (size_t) c * NT_KC + vc);
			rb[u] = *reinterpret_cast<const b8 *>(B + (vr + NT_VR * u) * ldb + (size_t) c * NT_KC + vc);
		}
	};
#pragma unroll
	for(int i = 0; i < NT_MB; i++)
#pragma unroll
		for(int j = 0; j < 2; j++)
			acc[i][j] = (f4) 0;
	if(c0 < c1)
		load(c0);
	for(int c = c0; c < c1; c++) {
		const int p = (c - c0) & 1;
#pragma unroll
		for(int u = 0; u < NT_VS; u++) {
			*reinterpret_cast<b8 *>(&s.a[p][vr + NT_VR * u][vc]) = ra[u];
			*reinterpret_cast<b8 *>(&s.b[p][vr + NT_VR * u][vc]) = rb[u];
		}
		__syncthreads();
		if(c + 1 < c1)
			load(c + 1);
#pragma unroll
		for(int ks = 0; ks < NT_KC; ks += 32) {
			b8 af[NT_MB], bf[2];
#pragma unroll
			for(int i = 0; i < NT_MB; i++)
				af[i] = *reinterpret_cast<const b8 *>(&s.a[p][wm + 16 * i + li][ks + 8 * lq]);
#pragma unroll
			for(int i = 0; i < 2; i++)
				bf[i] = *reinterpret_cast<const b8 *>(&s.b[p][wn + 16 * i + li][ks + 8 * lq]);
#pragma unroll
			for(int i = 0; i < NT_MB; i++)
#pragma unroll
				for(int j = 0; j < 2; j++)
					acc[i][j] = mma(af[i], bf[j], acc[i][j]);
		}
	}
}

/* the layer products and their epilogues */
struct nt_args {
	const bf16_t *A, *B;
	int lda, ldb, chunks;
	int rows, cols, ld, bp;		/* valid rows and columns; row stride of the outputs; stride of the transposed ones */
	const float *bias;
	float *Z;
	bf16_t *out, *outT;
	float *db;
	float *C;
};

enum { EPI_FWD, EPI_FWD_TRAIN, EPI_BWD, EPI_PLAIN };

template <int EPI>
__global__ void __launch_bounds__(64 * NT_W) k_nt(struct nt_args g)
{
	__shared__ __align__(16) struct nt_lds s;
	__shared__ float cs[NT_W / 2][NT_T];
	const int m0 = blockIdx.x * NT_T, n0 = blockIdx.y * NT_T;
	f4 acc[NT_MB][2];
	nt_tile(s, g.A + (size_t) m0 * g.lda, g.lda, g.B + (size_t) n0 * g.ldb, g.ldb, 0, g.chunks, acc);
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int wm = wave % (NT_W / 2) * (16 * NT_MB), wn = wave / (NT_W / 2) * 32;
	const int li = lane & 15, lq = lane >> 4;
#pragma unroll
	for(int j = 0; j < 2; j++) {
		const int col = n0 + wn + 16 * j + li;
		float sum = 0.f;
		const float b = (EPI == EPI_FWD || EPI == EPI_FWD_TRAIN) && col < g.cols ? g.bias[col] : 0.f;
#pragma unroll
		for(int i = 0; i < NT_MB; i++) {
			const int row0 = m0 + wm + 16 * i + 4 * lq;
			b4 t;
#pragma unroll
			for(int e = 0; e < 4; e++) {
				const int row = row0 + e;
				const bool in = row < g.rows && col < g.cols;
				if(EPI == EPI_PLAIN) {
					if(in)
						g.C[(size_t) row * g.ld + col] = acc[i][j][e];
					continue;
				}
				const size_t at = (size_t) row * g.ld + col;
				float v;
				if(EPI == EPI_BWD) {
					v = in ? acc[i][j][e] * gelu_d(g.Z[at]) : 0.f;
					sum += v;
				} else {
					const float z = acc[i][j][e] + b;
					if(EPI == EPI_FWD_TRAIN)
						g.Z[at] = z;
					v = in ? gelu(z) : 0.f;
				}
				t[e] = (bf16_t) v;
				g.out[at] = t[e];
			}
			if(EPI == EPI_FWD_TRAIN || EPI == EPI_BWD)
				*reinterpret_cast<b4 *>(g.outT + (size_t) col * g.bp + row0) = t;
		}
		if(EPI == EPI_BWD) {
			/* the bias gradient: column sums of the tile, in float32 */
			sum += __shfl_xor(sum, 16);
			sum += __shfl_xor(sum, 32);
			if(lq == 0)
				cs[wave % (NT_W / 2)][wn + 16 * j + li] = sum;
		}
	}
	if(EPI == EPI_BWD) {
		__syncthreads();
		if(threadIdx.x < NT_T) {
			float v = 0.f;
#pragma unroll
			for(int w = 0; w < NT_W / 2; w++)
				v += cs[w][threadIdx.x];
			g.db[(size_t) blockIdx.x * g.ld + n0 + threadIdx.x] = v;
		}
	}
}

/* x [B][n] to bfloat16, rows padded to [bp][np] and (train) transposed */
__global__ void __launch_bounds__(256) k_in(const float *__restrict__ x, int B, int n, int np, int bp, bf16_t *__restrict__ o, bf16_t *__restrict__ oT)
{
	__shared__ bf16_t t[64][66];
	const int r0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
	const int c = threadIdx.x & 63, rr = threadIdx.x >> 6;
#pragma unroll
	for(int k = 0; k < 16; k++) {
		const int r = rr + 4 * k;
		const bf16_t v = (bf16_t) (r0 + r < B && c0 + c < n ? x[(size_t) (r0 + r) * n + c0 + c] : 0.f);
		o[(size_t) (r0 + r) * np + c0 + c] = v;
		t[r][c] = v;
	}
	if(!oT)
		return;
	__syncthreads();
#pragma unroll
	for(int k = 0; k < 16; k++)
		oT[(size_t) (c0 + rr + 4 * k) * bp + r0 + c] = t[c][rr + 4 * k];
}

/*
 * The output layer, 16 rows per workgroup: y = H W + b (the waves split K,
 * partial sums added in LDS), then in training the loss of each row, its
 * gradient dY, the output layer's bias sums, and the last hidden layer's
 * dZ = (dY W^T) GELU'(z) with its bias sums.
 */
struct head_args {
	const bf16_t *H, *Wt, *W;	/* H [bp][wp], Wt [op][wp], W [wp][op] */
	const float *bias, *Zh, *target;
	float *Y, *loss;
	bf16_t *dYT, *dZ, *dZT;
	float *dbo, *dbh;
	int B, bp, w, wp, op, K;
	float lambda;
};

#define HD_T 3	/* column tiles: 3 K <= 48 outputs */
#define HD_C 4	/* column tiles of dZ in flight per wave */

template <bool TRAIN>
__global__ void __launch_bounds__(512) k_head(struct head_args g)
{
	__shared__ float red[8][16][16 * HD_T + 1];
	__shared__ float y[16][16 * HD_T + 1];
	__shared__ __align__(16) bf16_t dy[16][72];
	const int r0 = blockIdx.x * 16, n3 = 3 * g.K;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int li = lane & 15, lq = lane >> 4;
	f4 acc[HD_T];
#pragma unroll
	for(int t = 0; t < HD_T; t++)
		acc[t] = (f4) 0;
	for(int k = 32 * wave; k < g.wp; k += 256) {
		const b8 a = *reinterpret_cast<const b8 *>(g.H + (size_t) (r0 + li) * g.wp + k + 8 * lq);
#pragma unroll
		for(int t = 0; t < HD_T; t++)
			if(16 * t < n3)
				acc[t] = mma(a, *reinterpret_cast<const b8 *>(g.Wt + (size_t) (16 * t + li) * g.wp + k + 8 * lq), acc[t]);
	}
#pragma unroll
	for(int t = 0; t < HD_T; t++)
#pragma unroll
		for(int e = 0; e < 4; e++)
			red[wave][4 * lq + e][16 * t + li] = acc[t][e];
	__syncthreads();
	for(int i = threadIdx.x; i < 16 * n3; i += 512) {
		const int r = i / n3, j = i - r * n3;
		const float v = ((red[0][r][j] + red[1][r][j]) + (red[2][r][j] + red[3][r][j])) + ((red[4][r][j] + red[5][r][j]) + (red[6][r][j] + red[7][r][j])) + g.bias[j];
		y[r][j] = v;
		if(r0 + r < g.B)
			g.Y[(size_t) (r0 + r) * n3 + j] = v;
	}
	if(!TRAIN)
		return;
	/* a wave's next HD_C column tiles of W and z, the first ones in flight
	 * during the loss */
	b8 w0[HD_C], w1[HD_C];
	float zh[HD_C][4];
	auto fetch = [&](int ct0) {
#pragma unroll
		for(int u = 0; u < HD_C; u++) {
			const int ct = ct0 + 8 * u;
			if(ct >= g.wp / 16)
				continue;
			const bf16_t *wr = g.W + (size_t) (16 * ct + li) * g.op + 8 * lq;
			w0[u] = *reinterpret_cast<const b8 *>(wr);
			w1[u] = *reinterpret_cast<const b8 *>(wr + 32);
#pragma unroll
			for(int e = 0; e < 4; e++)
				zh[u][e] = g.Zh[(size_t) (r0 + 4 * lq + e) * g.wp + 16 * ct + li];
		}
	};
	fetch(wave);
	for(int i = threadIdx.x; i < 16 * 72; i += 512)
		dy[i / 72][i % 72] = (bf16_t) 0.f;
	__syncthreads();
	if(threadIdx.x < 16) {
		/* the candidate loss of one row and its gradient (in place of y) */
		const int r = threadIdx.x, row = r0 + r, K = g.K;
		float *yr = y[r];
		if(row < g.B) {
			const float t0 = g.target[3 * (size_t) row], t1 = g.target[3 * (size_t) row + 1], t2 = g.target[3 * (size_t) row + 2];
			int best = 0;
			float dbest = 0.f, sum = 0.f;
			for(int k = 0; k < K; k++) {
				const float n = sqrtf(yr[3 * k] * yr[3 * k] + yr[3 * k + 1] * yr[3 * k + 1] + yr[3 * k + 2] * yr[3 * k + 2]) + 1e-12f;
				const float d = 1.f - (yr[3 * k] * t0 + yr[3 * k + 1] * t1 + yr[3 * k + 2] * t2) / n;
				if(k == 0 || d < dbest) {
					best = k;
					dbest = d;
				}
				sum += d;
			}
			g.loss[row] = dbest + g.lambda / K * sum;
			const float inv_rows = 1.f / g.B;
			for(int k = 0; k < K; k++) {
				const float w = ((k == best) ? 1.f : 0.f) + g.lambda / K;
				const float n = sqrtf(yr[3 * k] * yr[3 * k] + yr[3 * k + 1] * yr[3 * k + 1] + yr[3 * k + 2] * yr[3 * k + 2]) + 1e-12f;
				const float dot = (yr[3 * k] * t0 + yr[3 * k + 1] * t1 + yr[3 * k + 2] * t2) / n;
				const float c0 = yr[3 * k] / n, c1 = yr[3 * k + 1] / n, c2 = yr[3 * k + 2] / n;
				/* d(1 - c.t)/dy = -(t - (c.t) c) / |y| */
				yr[3 * k] = -w * (t0 - dot * c0) / n * inv_rows;
				yr[3 * k + 1] = -w * (t1 - dot * c1) / n * inv_rows;
				yr[3 * k + 2] = -w * (t2 - dot * c2) / n * inv_rows;
			}
		} else
			for(int j = 0; j < n3; j++)
				yr[j] = 0.f;
		for(int j = 0; j < n3; j++)
			dy[r][j] = (bf16_t) yr[j];
	}
	__syncthreads();
	if(threadIdx.x < n3) {
		float s = 0.f;
		for(int r = 0; r < 16; r++)
			s += y[r][threadIdx.x];
		g.dbo[(size_t) blockIdx.x * g.op + threadIdx.x] = s;
	}
	for(int i = threadIdx.x; i < 16 * n3; i += 512)
		g.dYT[(size_t) (i / 16) * g.bp + r0 + i % 16] = dy[i % 16][i / 16];
	/* K = 3 K outputs, zero-padded to 32 or 64 */
	const b8 a0 = *reinterpret_cast<const b8 *>(&dy[li][8 * lq]), a1 = *reinterpret_cast<const b8 *>(&dy[li][32 + 8 * lq]);
	for(int ct0 = wave; ct0 < g.wp / 16; ct0 += 8 * HD_C) {
		if(ct0 != wave)
			fetch(ct0);
#pragma unroll
		for(int u = 0; u < HD_C; u++) {
			const int ct = ct0 + 8 * u, col = 16 * ct + li;
			if(ct >= g.wp / 16)
				continue;
			f4 c = mma(a0, w0[u], (f4) 0);
			if(n3 > 32)
				c = mma(a1, w1[u], c);
			float s = 0.f;
			b4 t;
#pragma unroll
			for(int e = 0; e < 4; e++) {
				const int row = r0 + 4 * lq + e;
				const float v = row < g.B && col < g.w ? c[e] * gelu_d(zh[u][e]) : 0.f;
				s += v;
				t[e] = (bf16_t) v;
				g.dZ[(size_t) row * g.wp + col] = t[e];
			}
			*reinterpret_cast<b4 *>(g.dZT + (size_t) col * g.bp + r0 + 4 * lq) = t;
			s += __shfl_xor(s, 16);
			s += __shfl_xor(s, 32);
			if(lq == 0)
				g.dbh[(size_t) blockIdx.x * g.wp + col] = s;
		}
	}
}

/* all layers' weight gradients: workgroup = a 64 x 64 tile of one layer x
 * one split of the batch */
struct dw_layer {
	const bf16_t *inT, *dZT;
	int tn, first, doutp;		/* column tiles, first tile, row stride of the output */
	size_t o;
};

struct dw_args {
	struct dw_layer l[MLP_MAX_LAYERS];
	int nl, tiles, bp, chunks, per_split;
	size_t padded;
	float *part;
};

__global__ void __launch_bounds__(64 * NT_W) k_dw(struct dw_args g)
{
	__shared__ __align__(16) struct nt_lds s;
	const int split = blockIdx.x / g.tiles, t = blockIdx.x - split * g.tiles;
	int k = 0;
	while(k + 1 < g.nl && t >= g.l[k + 1].first)
		k++;
	const struct dw_layer &L = g.l[k];
	const int m0 = (t - L.first) / L.tn * NT_T, n0 = (t - L.first) % L.tn * NT_T;
	const int c0 = split * g.per_split, c1 = c0 + g.per_split < g.chunks ? c0 + g.per_split : g.chunks;
	f4 acc[NT_MB][2];
	nt_tile(s, L.inT + (size_t) m0 * g.bp, g.bp, L.dZT + (size_t) n0 * g.bp, g.bp, c0, c1, acc);
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int wm = wave % (NT_W / 2) * (16 * NT_MB), wn = wave / (NT_W / 2) * 32;
	const int li = lane & 15, lq = lane >> 4;
	float *o = g.part + split * g.padded + L.o;
#pragma unroll
	for(int i = 0; i < NT_MB; i++)
#pragma unroll
		for(int j = 0; j < 2; j++)
#pragma unroll
			for(int e = 0; e < 4; e++)
				o[(size_t) (m0 + wm + 16 * i + 4 * lq + e) * L.doutp + n0 + wn + 16 * j + li] = acc[i][j][e];
}

#define UP_R 32	/* rows of an update tile */

/* per 32 x 64 tile of a layer: SUM, the splits' sum into g; ADAM, the
 * update of p; then the operand weights in both orientations (not after a
 * sum alone).  The first row of tiles takes the bias too. */
struct up_layer {
	int din, dout, dinp, doutp, tn, first, db_rows;
	size_t ow, ob, o;
	const float *db;
};

struct up_args {
	struct up_layer l[MLP_MAX_LAYERS];
	int nl, splits;
	size_t padded;
	const float *part;
	float *p, *g, *m, *v;
	bf16_t *W, *Wt;
	struct mlp_adam a;
};

__device__ inline float adam_step(const struct mlp_adam &a, float g, float *m, float *v, float p)
{
	const float mi = a.b1 * *m + (1.f - a.b1) * g;
	const float vi = a.b2 * *v + (1.f - a.b2) * g * g;
	*m = mi;
	*v = vi;
	return p - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
}

template <bool SUM, bool ADAM>
__global__ void __launch_bounds__(256) k_update(struct up_args g)
{
	__shared__ bf16_t t[UP_R][66];
	__shared__ float bs[4][64];
	int k = 0;
	while(k + 1 < g.nl && (int) blockIdx.x >= g.l[k + 1].first)
		k++;
	const struct up_layer &L = g.l[k];
	const int r0 = ((int) blockIdx.x - L.first) / L.tn * UP_R, c0 = ((int) blockIdx.x - L.first) % L.tn * 64;
	const int c = threadIdx.x & 63, rr = threadIdx.x >> 6;
	const bool colin = c0 + c < L.dout;
	/* all of a thread's values in flight at once */
	float gr[UP_R / 4], pw[UP_R / 4], mw[UP_R / 4], vw[UP_R / 4];
#pragma unroll
	for(int u = 0; u < UP_R / 4; u++) {
		const int r = rr + 4 * u;
		const bool in = colin && r0 + r < L.din;
		const size_t at = L.ow + (size_t) (r0 + r) * L.dout + c0 + c;
		gr[u] = !in ? 0.f : SUM ? g.part[L.o + (size_t) (r0 + r) * L.doutp + c0 + c] : ADAM ? g.g[at] : 0.f;
		pw[u] = in && (ADAM || !SUM) ? g.p[at] : 0.f;
		mw[u] = in && ADAM ? g.m[at] : 0.f;
		vw[u] = in && ADAM ? g.v[at] : 0.f;
	}
	if(SUM)
		for(int s = 1; s < g.splits; s++)
#pragma unroll
			for(int u = 0; u < UP_R / 4; u++)
				if(colin && r0 + rr + 4 * u < L.din)
					gr[u] += g.part[s * g.padded + L.o + (size_t) (r0 + rr + 4 * u) * L.doutp + c0 + c];
	if(r0 == 0) {
		/* bias: the four waves split the partial column sums */
		const size_t at = L.ob + c0 + c;
		float s = 0.f;
		if(SUM) {
			if(colin)
#pragma unroll 8
				for(int r = rr; r < L.db_rows; r += 4)
					s += L.db[(size_t) r * L.doutp + c0 + c];
			bs[rr][c] = s;
			__syncthreads();
			s = (bs[0][c] + bs[1][c]) + (bs[2][c] + bs[3][c]);
		}
		if(rr == 0 && colin) {
			if(SUM)
				g.g[at] = s;
			if(ADAM)
				g.p[at] = adam_step(g.a, SUM ? s : g.g[at], g.m + at, g.v + at, g.p[at]);
		}
	}
#pragma unroll
	for(int u = 0; u < UP_R / 4; u++) {
		const int r = rr + 4 * u;
		float w = pw[u];
		if(colin && r0 + r < L.din) {
			const size_t at = L.ow + (size_t) (r0 + r) * L.dout + c0 + c;
			if(SUM)
				g.g[at] = gr[u];
			if(ADAM) {
				w = adam_step(g.a, gr[u], &mw[u], &vw[u], w);
				g.m[at] = mw[u];
				g.v[at] = vw[u];
				g.p[at] = w;
			}
		}
		if(ADAM || !SUM) {
			const bf16_t b = (bf16_t) w;
			g.W[L.o + (size_t) (r0 + r) * L.doutp + c0 + c] = b;
			t[r][c] = b;
		}
	}
	if(SUM && !ADAM)
		return;
	__syncthreads();
#pragma unroll
	for(int i = threadIdx.x; i < 64 * UP_R; i += 256)
		g.Wt[L.o + (size_t) (c0 + i / UP_R) * L.dinp + r0 + i % UP_R] = t[i % UP_R][i / UP_R];
}

/* dst [rows padded][kp] bfloat16 of src (rows x k, or its transpose) */
__global__ void k_pad(const float *__restrict__ src, int trans, int rows, int k, int kp, bf16_t *__restrict__ dst, long n)
{
	const long i = (long) blockIdx.x * blockDim.x + threadIdx.x;
	if(i >= n)
		return;
	const int r = (int) (i / kp), c = (int) (i - (long) r * kp);
	dst[i] = (bf16_t) (r < rows && c < k ? src[trans ? (size_t) c * rows + r : (size_t) r * k + c] : 0.f);
}

int pad128(int n)
{
	return (n + 127) / 128 * 128;
}

int ok(void)
{
	return hipGetLastError() == hipSuccess ? 0 : -1;
}

/* splits of the weight gradients' K: about three workgroups per CU over all
 * layers' tiles (two fit at once: 70 KB of LDS each), each split a whole
 * number of chunks */
int dw_splits(int tiles, int chunks, int *per_split)
{
	int s = (3 * sphr_rt_cus() + tiles - 1) / tiles;
	s = s < 1 ? 1 : s > 8 ? 8 : s;
	*per_split = (chunks + s - 1) / s;
	return (chunks + *per_split - 1) / *per_split;
}

int launch_update(struct mlp_bf *m, bool sum, bool adam, int splits, int db_rows_head, int db_rows, float *p, float *g, float *pm, float *pv, const struct mlp_adam *a, hipStream_t st)
{
	struct up_args u;
	memset(&u, 0, sizeof(u));
	int first = 0;
	for(int k = 0; k < m->nl; k++) {
		const struct mlp_bf_layer &L = m->l[k];
		struct up_layer &q = u.l[k];
		q.din = L.din;
		q.dout = L.dout;
		q.dinp = L.dinp;
		q.doutp = L.doutp;
		q.tn = (L.dout + 63) / 64;
		q.first = first;
		/* the head's launch sums 16 rows each, for the output layer and
		 * the last hidden one; the others' 64 */
		q.db_rows = k >= m->nl - 2 ? db_rows_head : db_rows;
		q.ow = L.ow;
		q.ob = L.ob;
		q.o = L.o;
		q.db = m->db[k];
		first += q.tn * ((L.din + UP_R - 1) / UP_R);
	}
	u.nl = m->nl;
	u.splits = splits;
	u.padded = m->padded;
	u.part = m->part;
	u.p = p;
	u.g = g;
	u.m = pm;
	u.v = pv;
	u.W = m->W;
	u.Wt = m->Wt;
	if(a)
		u.a = *a;
	if(sum && adam)
		hipLaunchKernelGGL((k_update<true, true>), dim3(first), dim3(256), 0, st, u);
	else if(sum)
		hipLaunchKernelGGL((k_update<true, false>), dim3(first), dim3(256), 0, st, u);
	else if(adam)
		hipLaunchKernelGGL((k_update<false, true>), dim3(first), dim3(256), 0, st, u);
	else
		hipLaunchKernelGGL((k_update<false, false>), dim3(first), dim3(256), 0, st, u);
	return ok();
}

struct head_args head(struct mlp_bf *m, const float *p, int B, int bp)
{
	struct head_args h;
	memset(&h, 0, sizeof(h));
	const int o = m->nl - 1;
	const struct mlp_bf_layer &L = m->l[o];
	h.H = m->H[o - 1];
	h.Wt = m->Wt + L.o;
	h.W = m->W + L.o;
	h.bias = p + L.ob;
	h.Y = m->Z[o];
	h.B = B;
	h.bp = bp;
	h.w = L.din;
	h.wp = L.dinp;
	h.op = L.doutp;
	h.K = m->K;
	return h;
}

/* the hidden layers; with train, what the backward pass needs is kept */
int hidden(struct mlp_bf *m, const float *p, const float *x, int B, bool train, hipStream_t st)
{
	const int bp = pad128(B);
	hipLaunchKernelGGL(k_in, dim3(bp / 64, m->l[0].dinp / 64), dim3(256), 0, st, x, B, m->l[0].din, m->l[0].dinp, bp, m->x, train ? m->xT : (bf16_t *) NULL);
	for(int k = 0; k + 1 < m->nl; k++) {
		const struct mlp_bf_layer &L = m->l[k];
		struct nt_args g;
		memset(&g, 0, sizeof(g));
		g.A = k ? m->H[k - 1] : m->x;
		g.B = m->Wt + L.o;
		g.lda = g.ldb = L.dinp;
		g.chunks = L.dinp / NT_KC;
		g.rows = B;
		g.cols = L.dout;
		g.ld = L.doutp;
		g.bp = bp;
		g.bias = p + L.ob;
		g.Z = m->Z[k];
		g.out = m->H[k];
		g.outT = m->HT[k];
		if(train)
			hipLaunchKernelGGL((k_nt<EPI_FWD_TRAIN>), dim3(bp / NT_T, L.doutp / NT_T), dim3(64 * NT_W), 0, st, g);
		else
			hipLaunchKernelGGL((k_nt<EPI_FWD>), dim3(bp / NT_T, L.doutp / NT_T), dim3(64 * NT_W), 0, st, g);
	}
	return ok();
}

}	/* namespace */

void mlp_bf_free(struct mlp_bf *m)
{
	void *ptrs[] = { m->W, m->Wt, m->x, m->xT, m->part, m->loss };
	for(unsigned i = 0; i < sizeof(ptrs) / sizeof(ptrs[0]); i++)
		if(ptrs[i])
			hipFree(ptrs[i]);
	for(int k = 0; k < MLP_MAX_LAYERS; k++) {
		void *q[] = { m->H[k], m->HT[k], m->Z[k], m->dZ[k], m->dZT[k], m->db[k] };
		for(unsigned i = 0; i < sizeof(q) / sizeof(q[0]); i++)
			if(q[i])
				hipFree(q[i]);
	}
	memset(m, 0, sizeof(*m));
}

int mlp_bf_alloc(struct mlp_bf *m, int nl, const int *din, const int *dout, const size_t *ow, const size_t *ob, int K, int max_batch)
{
	memset(m, 0, sizeof(*m));
	m->nl = nl;
	m->K = K;
	m->max_bp = pad128(max_batch);
	for(int k = 0; k < nl; k++) {
		struct mlp_bf_layer &L = m->l[k];
		L.din = din[k];
		L.dout = dout[k];
		L.dinp = pad128(din[k]);
		L.doutp = pad128(dout[k]);
		L.ow = ow[k];
		L.ob = ob[k];
		L.o = m->padded;
		m->padded += (size_t) L.dinp * L.doutp;
		m->tiles += ((din[k] + 63) / 64) * ((dout[k] + 63) / 64);
	}
	int per;
	/* the most splits of any batch: at 64 chunks each split has several */
	m->max_splits = dw_splits(m->tiles, 64, &per);
	const size_t bp = m->max_bp;
	auto get = [](void *pp, size_t bytes) -> int {
		/* zeroed: the padding of the weights is never written */
		void **q = (void **) pp;
		return sphr_rt_check(hipMalloc(q, bytes), "hipMalloc") || sphr_rt_check(hipMemset(*q, 0, bytes), "hipMemset");
	};
	int bad = get(&m->W, m->padded * 2) || get(&m->Wt, m->padded * 2) || get(&m->x, bp * m->l[0].dinp * 2) || get(&m->xT, bp * m->l[0].dinp * 2)
		  || get(&m->part, m->max_splits * m->padded * 4) || get(&m->loss, bp * 4);
	for(int k = 0; k < nl && !bad; k++) {
		const size_t n = bp * m->l[k].doutp;
		bad = get(&m->Z[k], n * 4) || get(&m->dZT[k], n * 2) || get(&m->db[k], n / 16 * 4);
		if(!bad && k + 1 < nl)
			bad = get(&m->H[k], n * 2) || get(&m->HT[k], n * 2) || get(&m->dZ[k], n * 2);
	}
	bad = bad || sphr_rt_check(hipDeviceSynchronize(), "synchronize");
	if(bad)
		mlp_bf_free(m);
	return bad ? -1 : 0;
}

int mlp_bf_refresh(struct mlp_bf *m, float *p, hipStream_t st)
{
	return launch_update(m, false, false, 0, 0, 0, p, NULL, NULL, NULL, NULL, st);
}

int mlp_bf_adam(struct mlp_bf *m, float *p, float *g, float *pm, float *pv, const struct mlp_adam *adam, hipStream_t st)
{
	return launch_update(m, false, true, 0, 0, 0, p, g, pm, pv, adam, st);
}

int mlp_bf_forward(struct mlp_bf *m, const float *p, const float *x, int B, hipStream_t st)
{
	const int bp = pad128(B);
	if(hidden(m, p, x, B, false, st))
		return -1;
	hipLaunchKernelGGL((k_head<false>), dim3(bp / 16), dim3(512), 0, st, head(m, p, B, bp));
	return ok();
}

int mlp_bf_loss_grad(struct mlp_bf *m, float *p, float *g, const float *x, const float *target, int B, float lambda, float *loss, const struct mlp_adam *adam, float *pm, float *pv, hipStream_t st)
{
	const int bp = pad128(B), o = m->nl - 1;
	if(hidden(m, p, x, B, true, st))
		return -1;
	struct head_args h = head(m, p, B, bp);
	h.Zh = m->Z[o - 1];
	h.target = target;
	h.loss = loss ? loss : m->loss;
	h.dYT = m->dZT[o];
	h.dZ = m->dZ[o - 1];
	h.dZT = m->dZT[o - 1];
	h.dbo = m->db[o];
	h.dbh = m->db[o - 1];
	h.lambda = lambda;
	hipLaunchKernelGGL((k_head<true>), dim3(bp / 16), dim3(512), 0, st, h);
	for(int k = o - 1; k > 0; k--) {
		/* dZ of layer k - 1 from layer k's */
		const struct mlp_bf_layer &L = m->l[k];
		struct nt_args a;
		memset(&a, 0, sizeof(a));
		a.A = m->dZ[k];
		a.B = m->W + L.o;
		a.lda = a.ldb = L.doutp;
		a.chunks = L.doutp / NT_KC;
		a.rows = B;
		a.cols = L.din;
		a.ld = L.dinp;
		a.bp = bp;
		a.Z = m->Z[k - 1];
		a.out = m->dZ[k - 1];
		a.outT = m->dZT[k - 1];
		a.db = m->db[k - 1];
		hipLaunchKernelGGL((k_nt<EPI_BWD>), dim3(bp / NT_T, L.dinp / NT_T), dim3(64 * NT_W), 0, st, a);
	}
	struct dw_args d;
	memset(&d, 0, sizeof(d));
	int first = 0;
	for(int k = 0; k < m->nl; k++) {
		const struct mlp_bf_layer &L = m->l[k];
		d.l[k].inT = k ? m->HT[k - 1] : m->xT;
		d.l[k].dZT = m->dZT[k];
		d.l[k].tn = (L.dout + 63) / 64;
		d.l[k].first = first;
		d.l[k].doutp = L.doutp;
		d.l[k].o = L.o;
		first += d.l[k].tn * ((L.din + 63) / 64);
	}
	d.nl = m->nl;
	d.tiles = m->tiles;
	d.bp = bp;
	d.chunks = bp / NT_KC;
	d.padded = m->padded;
	d.part = m->part;
	const int splits = dw_splits(m->tiles, d.chunks, &d.per_split);
	hipLaunchKernelGGL(k_dw, dim3(splits * m->tiles), dim3(64 * NT_W), 0, st, d);
	if(ok())
		return -1;
	return launch_update(m, true, adam != NULL, splits, bp / 16, bp / NT_T, p, g, pm, pv, adam, st);
}

int mlp_bf_gemm(int ta, int tb, int M, int N, int K, const float *A, const float *B, float *C, hipStream_t st)
{
	const int mp = pad128(M), np = pad128(N), kp = pad128(K);
	bf16_t *a = NULL, *b = NULL;
	int rc = -1;
	if(!sphr_rt_check(hipMalloc(&a, (size_t) mp * kp * 2), "hipMalloc") && !sphr_rt_check(hipMalloc(&b, (size_t) np * kp * 2), "hipMalloc")) {
		const long na = (long) mp * kp, nb = (long) np * kp;
		struct nt_args g;
		memset(&g, 0, sizeof(g));
		hipLaunchKernelGGL(k_pad, dim3((unsigned) ((na + 255) / 256)), dim3(256), 0, st, A, ta, M, K, kp, a, na);
		hipLaunchKernelGGL(k_pad, dim3((unsigned) ((nb + 255) / 256)), dim3(256), 0, st, B, !tb, N, K, kp, b, nb);
		g.A = a;
		g.B = b;
		g.lda = g.ldb = kp;
		g.chunks = kp / NT_KC;
		g.rows = M;
		g.cols = N;
		g.ld = N;
		g.C = C;
		hipLaunchKernelGGL((k_nt<EPI_PLAIN>), dim3(mp / NT_T, np / NT_T), dim3(64 * NT_W), 0, st, g);
		rc = ok() || sphr_rt_check(hipStreamSynchronize(st), "synchronize") ? -1 : 0;
	}
	hipFree(a);
	hipFree(b);
	return rc;
}
