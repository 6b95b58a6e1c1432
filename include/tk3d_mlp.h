/*
 * tk3d_mlp.h - C ABI of the shared-MLP kernels (torkit3d_amd/csrc/mlp*.hip): the pieces of
 * "1x1 convolution, batch norm, ReLU" chains on [B, C, P] fp32 tensors, forward and backward,
 * that the reference runs as stock torch modules (torkit3d/nn/modules/mlp.py,
 * torkit3d/nn/modules/conv.py) on the tensors its ops produce (torkit3d/layers/pointnet2.py,
 * torkit3d/ops/edge_conv.py). Conventions of tk3d.h: device pointers, dense tensors, outputs
 * allocated by the caller and fully overwritten, nothing allocated or synchronised, 0 or an
 * error code returned.
 *
 * A layer computes y = W x, then z = relu((y - mean) / sqrt(var + eps) * gamma + beta). The
 * entry points hand y from layer to layer: the norm and the ReLU are applied where y is read.
 * Backward, with g the gradient of z, e = g where z > 0 (or NaN) else 0:
 *     dbeta = sum e,   dgamma = sum e (y - mean) / sqrt(var + eps),
 *     dy = a e + b y + d = a e + b (y - mean) + d0  with (a, b, d, d0) per channel
 * (tk3d_mlp_grad_coefficients_f32).
 *
 * Pooled layers. Where only the maximum of z over groups of `group` consecutive positions is
 * wanted, the place of the maximum and the y there are all of the layer that is kept. In the
 * backward e has one nonzero per group and channel, and with y = W x
 *     W^T dy = W^T (a e) + (W^T diag(b) W) x' + W^T d'
 *     dW     = (a e) x'^T + diag(b) W (x' x'^T) + d' (sum x')^T
 * so the dense part needs only the input x. In it x' = x - m and d' = d + b (W m) for any m (a
 * channel's dy add up to zero over the batch, so that sum dy m^T is nothing). Here m = relu(beta) of
 * the norm in front, of which the mean of x is never further than |gamma| / 2: with m = 0 the terms
 * of dW cancel where activations sit far from zero (mean / deviation of 8: 2.1 times the error of
 * the sum over positions).
 */
#ifndef TK3D_MLP_H
#define TK3D_MLP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct {
    const float *mean, *var, *gamma, *beta; /* [C] each */
    float eps; /* negative: var holds 1 / sqrt(variance + eps) itself */
} tk3d_mlp_norm;

typedef struct {
    const float *x;        /* [B, K, P]; batch_stride elements from one batch element to the next */
    const float *y;        /* same shape, for the gradient inputs */
    const float *coef;     /* [K][4]: (a, b, d, d0), for the gradient inputs */
    const float *w;        /* weight of input channel k and output channel c: w[k * wk + c * wc] */
    int64_t batch_stride;
    int32_t K, wk, wc;
} tk3d_mlp_source;

/* What a product reads (in) and what it does with its result (out). */
enum {
    TK3D_MLP_IN_RAW = 0,      /* x */
    TK3D_MLP_IN_RAW2 = 1,     /* the channels of src[0].x, then those of src[1].x */
    TK3D_MLP_IN_ACT = 2,      /* relu(in_norm(x)) */
    TK3D_MLP_IN_GRAD = 3,     /* a x + b y + d */
    TK3D_MLP_IN_GRAD_OUT = 4, /* the same with x masked by relu(in_norm(y)) first */
    TK3D_MLP_IN_CENTRED = 5,  /* relu(in_norm(x)) - relu(beta of in_norm) */
    TK3D_MLP_IN_SHIFTED = 7,  /* x - beta of in_norm; to OUT_PLAIN, + add, alone; slots 0: not for this size */
    TK3D_MLP_OUT_PLAIN = 1,     /* out + bias, channels from C0 on in out2; either may be NULL */
    TK3D_MLP_OUT_POINTS = 2,    /* out as [B, P, C] */
    TK3D_MLP_OUT_EVAL = 3,      /* relu(out_norm(out)) */
    TK3D_MLP_OUT_POOL_EVAL = 5, /* relu(out_norm(extreme over groups)) */
    TK3D_MLP_OUT_MASK = 6       /* e = (out + bias, IN_CENTRED: + add) where relu(out_norm(yprev)) passes, and partial
                                   sums of e and e (yprev - mean) */
};

typedef struct {
    tk3d_mlp_source src[2];
    tk3d_mlp_norm in_norm, out_norm;
    float *out, *out2;
    const float *yprev; /* [B, C, P] */
    const float *bias;  /* [C] or NULL */
    const float *add;   /* [B, C, P], may be out itself; IN_CENTRED (P % 4 == 0) and IN_SHIFTED alone */
    void *partial;      /* OUT_MASK: doubles [C][slots][2]; tk3d_mlp_product_slots gives slots */
    int32_t B, C, C0, P;
    int32_t group, M;   /* pooled forms: P == group * M, group 32 or 64 */
} tk3d_mlp_product;

/* One product. `slots` as tk3d_mlp_product_slots returns it for the same arguments. */
int tk3d_mlp_product_slots(int in, int out, const tk3d_mlp_product *p);
int tk3d_mlp_product_f32(int in, int out, const tk3d_mlp_product *p, void *stream);

/* Weight gradient: out[r][c] = sum over (b, p) of row(r, p) * colv(c, p), r < R, c < C, in
 * `splits` partial sums [splits][R][C]. Rows: raw x, gradient (a x + b y + d, masked or not),
 * or activations less relu(beta); columns: raw x, activations, or these less relu(beta). rowsum (NULL or [splits][R]) gets the
 * sums of the rows themselves. Activations less a centre come as rows and columns of one tensor: the result is
 * symmetric, and below the diagonal of more than 64 rows nothing need be written. */
enum {
    TK3D_MLP_ROW_RAW = 0,
    TK3D_MLP_ROW_GRAD = 1,
    TK3D_MLP_ROW_GRAD_OUT = 2,
    TK3D_MLP_ROW_CENTRED = 4,
    TK3D_MLP_ROW_SHIFTED = 5, /* x - beta of row_norm, with COL_SHIFTED; more than 64 rows */
    TK3D_MLP_COL_RAW = 0,
    TK3D_MLP_COL_ACT = 1,
    TK3D_MLP_COL_CENTRED = 2,
    TK3D_MLP_COL_SHIFTED = 3
};
typedef struct {
    tk3d_mlp_source row, col; /* K = R and C; weights unused */
    tk3d_mlp_norm row_norm, col_norm;
    float *partial, *rowsum;
    int32_t B, P;
} tk3d_mlp_outer;
int tk3d_mlp_outer_splits(const tk3d_mlp_outer *p);
int tk3d_mlp_outer_f32(int row, int col, const tk3d_mlp_outer *p, void *stream);

/* Both of a layer in one launch, where they read the same: the product IN_GRAD, IN_GRAD_OUT (weights
 * K = R output channels to C input channels) or IN_CENTRED (K = R = C) to OUT_MASK, and the weight gradient
 * with rows of the same kind and the product's yprev as COL_ACT (COL_CENTRED behind IN_CENTRED); or one to
 * OUT_PLAIN (C0 = C), columns COL_RAW. tk3d_mlp_pair_slots: slots and splits of the partial sums, 0 where the two
 * have to be called apart (more than 128 channels, 128 from 32, rows that are not 16-byte aligned, channels by
 * positions beyond 32-bit byte offsets). */
int tk3d_mlp_pair_slots(const tk3d_mlp_product *p, const tk3d_mlp_outer *o);
int tk3d_mlp_pair_f32(int in, int out, const tk3d_mlp_product *p, const tk3d_mlp_outer *o, void *stream);

/* out[r * ld + c] = sum over the splits of partial[r][c], rows of C, `stride` elements from one split
 * to the next; n of them in one launch. */
typedef struct {
    const float *partial;
    float *out;
    int64_t stride;
    int32_t splits, R, C, ld;
} tk3d_mlp_sum;
int tk3d_mlp_sum_f32(const tk3d_mlp_sum *sums, int n, void *stream);

/* A batch norm of a training step, statistics in the library's order (csrc/batch_norm.hip): first the
 * sums, then a pass that normalises with them and leaves mean, 1 / sqrt(variance + eps) and the updated
 * running statistics. y [B, C, P], 16-byte aligned. */
typedef struct {
    void *partial; /* tk3d_mlp_batch_norm_partial_bytes(C), as tk3d_mlp_batch_sums_f32 left it */
    const float *gamma, *beta;
    float *running_mean, *running_var, *mean, *inv_std;
    double eps;
    float momentum;
    int32_t B, C, P;
} tk3d_mlp_batch_norm;
int tk3d_mlp_batch_norm_supported(int64_t B, int64_t C, int64_t P);
int64_t tk3d_mlp_batch_norm_partial_bytes(int64_t C);
int tk3d_mlp_batch_sums_f32(const float *y, int B, int C, int P, void *partial, void *stream);
/* z = relu(norm(y)) */
int tk3d_mlp_batch_relu_f32(const float *y, const tk3d_mlp_batch_norm *norm, float *z, void *stream);
/* out = relu(max norm(y)) over groups of `size` <= 255 consecutive values, arg the place of the maximum
 * and extreme the y at that place, [B, C, P / size] each */
int tk3d_mlp_batch_pool_f32(const float *y, const tk3d_mlp_batch_norm *norm, int size, float *out,
                            float *extreme, unsigned char *arg, void *stream);

/* out = relu(max norm(y)) over whole rows, [B, C]; arg the place of the maximum, extreme the y there and index the
 * place of the maximum of relu(norm(y)), the first of equal ones. z: norm(y) where it is there, else norm is
 * as above. */
int tk3d_mlp_batch_rows_f32(const float *y, const float *z, const tk3d_mlp_batch_norm *norm, int B, int C, int P,
                            float *out, float *extreme, int32_t *arg, int64_t *index, void *stream);

/* The three with one added to *count, the norm's count of batches (NULL: none). */
int tk3d_mlp_batch_relu_counted_f32(const float *y, const tk3d_mlp_batch_norm *norm, int64_t *count, float *z,
                                    void *stream);
int tk3d_mlp_batch_pool_counted_f32(const float *y, const tk3d_mlp_batch_norm *norm, int64_t *count, int size,
                                    float *out, float *extreme, unsigned char *arg, void *stream);
int tk3d_mlp_batch_rows_counted_f32(const float *y, const float *z, const tk3d_mlp_batch_norm *norm, int64_t *count,
                                    int B, int C, int P, float *out, float *extreme, int32_t *arg, int64_t *index,
                                    void *stream);

/* A normalised layer's ReLU and maximum over groups of `size` <= 255 consecutive values: out =
 * relu(max z), arg the place of the maximum and extreme the y at that place, [groups] each. */
int tk3d_mlp_pool_max_f32(const float *z, const float *y, int64_t groups, int size, float *out,
                          float *extreme, unsigned char *arg, void *stream);

/* (a, b, d, d0) per channel from the partial sums of (e, e (y - mean)), and dgamma, dbeta.
 */
int tk3d_mlp_grad_coefficients_f32(const void *partial, int slots, int64_t n, int C,
                                   const tk3d_mlp_norm *norm, float *coef, float *dgamma,
                                   float *dbeta, void *stream);

/* Partial sums of (e, e (y - mean)) with e = g masked by relu(norm(y)); g, y [B, C, P].
 * slots of tk3d_mlp_mask_slots. */
int tk3d_mlp_mask_slots(int B, int C, int P);
int tk3d_mlp_mask_sums_f32(const float *g, const float *y, int B, int C, int P,
                           const tk3d_mlp_norm *norm, void *partial, void *stream);

/* z = relu(norm(y)), n rows of P values, channel = row modulo C. */
int tk3d_mlp_activate_f32(const float *y, int64_t rows, int C, int P, const tk3d_mlp_norm *norm,
                          float *z, void *stream);
/* dy = a e + b y + d over e itself, and dy rel^T, rel [B, 3, P], in partial sums [splits][C][3] (at most 2^31 - 1
 * rows B C). */
int tk3d_mlp_grad_apply_splits(int B, int P);
int tk3d_mlp_grad_apply_f32(float *e, const float *y, const float *coef, const float *rel, int B, int C, int P,
                            float *partial, void *stream);

/* Backward of a pooled layer, before the products: from g [B,C,M], the extremes and their places
 * the coefficients (a, b, d'), dgamma, dbeta and sel, [B, C, M] of (float a e, int32 place in the
 * group); positions = B * group * M, w [C][I], inner the norm in front of the layer, whose activations
 * are counted from relu(beta) (shifted != 0: the layer's input itself from beta); partial: doubles [C][slots][2]
 * of scratch memory, slots of tk3d_mlp_pool_grad_slots. The places come as bytes or, with arg NULL, in arg32. */
int tk3d_mlp_pool_grad_slots(int B, int C, int M);
int tk3d_mlp_pool_grad_f32(const float *g, const float *extreme, const unsigned char *arg,
                           const int32_t *arg32, int B, int C, int M, int64_t positions, const tk3d_mlp_norm *norm, const float *w,
                           int I, const tk3d_mlp_norm *inner, int shifted, void *partial, void *sel,
                           float *coef, float *dgamma, float *dbeta, void *stream);
/* The sparse half of W^T dy, [B, I, M * group] (groups of 32 or 64; W [O][I]), and that of dW in
 * partial sums [splits][O][I] (y [B, I, M * group], norm of y). */
int tk3d_mlp_pool_scatter_f32(const void *sel, const float *w, int B, int O, int I, int M, int group,
                              float *out, void *stream);
int tk3d_mlp_pool_outer_splits(int B, int O, int I, int M);
int tk3d_mlp_pool_outer_f32(const void *sel, const float *y, const tk3d_mlp_norm *norm, int B, int O,
                            int I, int M, int group, float *partial, void *stream);
/* The same where a group is a whole row of P values (M == 1, P % 4 == 0): the sparse half of W^T dy [B, I, P], and
 * that of dW [O][I] itself, from the activations of x [B, I, P] (or, shifted != 0, x - beta of norm). */
int tk3d_mlp_rows_scatter_f32(const void *sel, const float *w, int B, int O, int I, int P, float *out,
                              void *stream);
int tk3d_mlp_rows_outer_f32(const void *sel, const float *x, int shifted, const tk3d_mlp_norm *norm, int B, int O,
                            int I, int P, float *dw, void *stream);
/* mean[c] of x [B, C, P] */
int tk3d_mlp_channel_means_f32(const float *x, int B, int C, int P, float *mean, void *stream);
/* gram[k][c] = sum_o W[o][k] b[o] W[o][c] and bias[c] = sum_o W[o][c] d'[o]; W [O][I]. */
int tk3d_mlp_pool_gram_f32(const float *w, const float *coef, int O, int I, float *gram, float *bias,
                           void *stream);
/* dW[o][i] = sparse[o][i] + b[o] (W xx)[o][i] + d'[o] xsum[i]; sparse, xx, xsum as partial sums, of xx what is on
 * and above the diagonal. */
int tk3d_mlp_pool_weight_grad_f32(const float *sparse, int sparse_splits, const float *xx,
                                  const float *xsum, int xx_splits, const float *w,
                                  const float *coef, int O, int I, float *scratch, float *dw,
                                  void *stream);

/* First layer behind a grouping: y[b,c,m,s] = u[b,j,c] + sum_a wx[c][a] (xyz[b,a,j] -
 * centre[b,a,m]), j = index[b,m,s] (an index outside [0,N) reads as zeros). u [B,N,C] (the product
 * of the features with their weights, or NULL), wx rows ldw apart. */
int tk3d_mlp_group_f32(const float *u, const float *xyz, const float *centre, const int64_t *index,
                       const float *wx, int ldw, int B, int C, int N, int M, int S, float *y,
                       void *stream);

/* Evaluation of three layers behind a grouping, pooled over the S neighbours: y of tk3d_mlp_group_f32 with C[0]
 * channels, ReLU of its norm[0]; w2 [C[1]][C[0]] and norm[1], w3 [C[2]][C[1]] and norm[2] on top; out [B,C[2],M]
 * is the maximum over each group. `supported`: C multiples of 32 whose activations of 64 positions fit in LDS
 * (C[0] + C[1] up to 512 or so), S 32 or 64, u (or NULL), w2 and w3 16-byte aligned, and widths and sizes for which it is
 * the faster way; others are refused. */
typedef struct tk3d_mlp_grouped_pool {
    const float *u, *xyz, *centre;
    const int64_t *index;
    const float *wx, *w2, *w3;
    tk3d_mlp_norm norm[3];
    float *out;
    int32_t ldw, B, N, M, S;
    int32_t C[3];
} tk3d_mlp_grouped_pool;
int tk3d_mlp_grouped_pool_supported(const tk3d_mlp_grouped_pool *p);
int tk3d_mlp_grouped_pool_f32(const tk3d_mlp_grouped_pool *p, void *stream);

/* EdgeConv (torkit3d/ops/edge_conv.py) with one layer, on a graph of a cloud with itself, pooled
 * over the K neighbours: y(i, k) = W1 (x_j - x_i) + W2 x_i, j = index[b, i, k] (x_j = 0 for an index
 * outside [0,N)), where w [O][2 C] = [W1 W2] and x [B, C, N].
 * tk3d_mlp_edge_forward_f32: the extreme of y [B, O, N]; tk3d_mlp_edge_features_f32: the edge
 * features themselves, [B, 2 C, N, K]. Backward: lists is the inverse of the graph (int32
 * [B][N + 1 + N K], tk3d_mlp_edge_lists), extreme and arg [B, O, N] the y at the maxima and their
 * places, coef as tk3d_mlp_grad_coefficients_f32 leaves it; dx [B, C, N] may be NULL, dw is like w.
 * Workspaces, aligned to 8 bytes, have the sizes that the _bytes functions return.
 * tk3d_mlp_edge_supported: the sizes these take (N <= 32768, K <= 255). */
int tk3d_mlp_edge_supported(int64_t B, int64_t N, int64_t K, int64_t O);
int tk3d_mlp_edge_features_f32(const float *x, const int64_t *index, int B, int C, int N, int K,
                               float *out, void *stream);
int64_t tk3d_mlp_edge_forward_bytes(int B, int N, int C, int O);
int tk3d_mlp_edge_forward_f32(const float *x, const int64_t *index, const float *w, const float *gamma,
                              int B, int N, int K, int C, int O, void *workspace, float *extreme,
                              void *stream);
int tk3d_mlp_edge_lists(const int64_t *index, int B, int N, int K, int32_t *lists, void *stream);
int64_t tk3d_mlp_edge_backward_bytes(int B, int N, int O, int C);
int tk3d_mlp_edge_backward_f32(const float *g, const float *extreme, const unsigned char *arg,
                               const float *x, const int64_t *index, const int32_t *lists, const float *w,
                               int B, int N, int K, int C, int O, const tk3d_mlp_norm *norm,
                               const float *coef, void *workspace, float *dx, float *dw, void *stream);

#ifdef __cplusplus
}
#endif
#endif /* TK3D_MLP_H */
