/*
 * The bfloat16 form of the proposal network (mlp_bf16.hip): its padded
 * operand buffers and the launches of forward, backward and the update.
 * The float32 master copies (p, g, Adam moments) stay with the caller in
 * the flat layout W_1 [in][out], b_1, ...
 */
#ifndef SPHR_MLP_BF16_H
#define SPHR_MLP_BF16_H

#include <hip/hip_runtime.h>

#define MLP_MAX_LAYERS 8

typedef __bf16 bf16_t;

/* one layer: sizes, padded sizes (multiples of 128), offsets in the flat
 * parameters (ow, ob) and in the padded operand weights and partial
 * gradients (o) */
struct mlp_bf_layer {
	int din, dout, dinp, doutp;
	size_t ow, ob, o;
};

struct mlp_bf {
	int nl, K, max_bp;		/* layers, candidates, largest padded batch */
	struct mlp_bf_layer l[MLP_MAX_LAYERS];
	size_t padded;			/* sum of dinp doutp */
	int tiles;			/* 64 x 64 weight tiles of all layers */
	int max_splits;
	bf16_t *W, *Wt;			/* [dinp][doutp] and [doutp][dinp] per layer */
	bf16_t *x, *xT;			/* [Bp][n_inp], [n_inp][Bp] */
	bf16_t *H[MLP_MAX_LAYERS], *HT[MLP_MAX_LAYERS];	/* activations of the hidden layers */
	float *Z[MLP_MAX_LAYERS];	/* pre-activations [Bp][doutp]; the last layer's [B][3 K] */
	bf16_t *dZ[MLP_MAX_LAYERS], *dZT[MLP_MAX_LAYERS];
	float *db[MLP_MAX_LAYERS];	/* [Bp / 16][doutp] partial column sums of dZ */
	float *part;			/* [splits][padded] partial weight gradients */
	float *loss;			/* [Bp] */
};

struct mlp_adam {
	float lr, b1, b2, eps, c1, c2;
};

int mlp_bf_alloc(struct mlp_bf *m, int nl, const int *din, const int *dout, const size_t *ow, const size_t *ob, int K, int max_batch);
void mlp_bf_free(struct mlp_bf *m);
/* operand weights from the master copy */
int mlp_bf_refresh(struct mlp_bf *m, float *p, hipStream_t st);
int mlp_bf_forward(struct mlp_bf *m, const float *p, const float *x, int B, hipStream_t st);
/* forward, loss, backward; g receives the gradients.  With adam, the
 * update runs in the launch that sums the gradients (pm, pv its moments) */
int mlp_bf_loss_grad(struct mlp_bf *m, float *p, float *g, const float *x, const float *target, int B, float lambda, float *loss, const struct mlp_adam *adam, float *pm, float *pv, hipStream_t st);
/* Adam from g */
int mlp_bf_adam(struct mlp_bf *m, float *p, float *g, float *pm, float *pv, const struct mlp_adam *adam, hipStream_t st);
/* C [M][N] = op(A) op(B) on the network's product kernel (device float32
 * in and out, operands rounded to bfloat16) */
int mlp_bf_gemm(int ta, int tb, int M, int N, int K, const float *A, const float *B, float *C, hipStream_t st);

#endif
