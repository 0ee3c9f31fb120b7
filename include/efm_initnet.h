/*
 * efm_initnet.h — C ABI of the learned moment-tensor / location initializer
 * kernels in libefm.so (gfx950).  No counterpart in the reference: its
 * inversions start from a fixed moment tensor (mainPropElastic3D_MT.py
 * M:2777, Mmod = StressTensor(0.5, 0, 0.5, 0, 0.5, 0)) at the catalogue
 * location; this network proposes both from the recorded gathers.
 *
 * Building blocks of a 1-D convolutional network trained and run on the GPU:
 * a BF16 MFMA GEMM with FP32 accumulation and fused bias/ReLU epilogue,
 * im2col / col2im for strided 1-D convolutions, ReLU and bias backward, MSE
 * loss, Adam, and the packing of propagator gathers into network inputs.
 *
 * BF16 values are stored as uint16 (the upper half of an IEEE float32, rounded
 * to nearest even).  Activations are laid out (C, B, L): channel-major, then
 * example, then sample, so a convolution's GEMM output (Cout, B*Lout) is the
 * next layer's input without a transpose.  All pointers are device pointers;
 * every call is asynchronous on `stream` and returns 0 or a negative EFM_E_*.
 */
#ifndef EFM_INITNET_H
#define EFM_INITNET_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* y[i] = bf16(x[i]). */
int efm_net_cast_bf16(const float *x, uint16_t *y, long long n, void *stream);

/* C[m, n] = sum_k A[m, k] * B[k, n] for m < M, n < N, k < K, where
 * A[m, k] = A[m*sam + k*sak] and B[k, n] = B[k*sbk + n*sbn] (BF16), FP32
 * accumulation, C[m*ldc + n] FP32.  epilogue 0: C = AB; 1: C = max(AB + bias[m], 0);
 * 2: C = AB + bias[m].  Cb (nullable) receives bf16(C) at the same offsets. */
int efm_net_gemm(int M, int N, int K, const uint16_t *A, long long sam, long long sak,
                 const uint16_t *B, long long sbk, long long sbn, float *C, long long ldc,
                 const float *bias, uint16_t *Cb, int epilogue, void *stream);

/* Lout = (L + 2*pad - ks)/stride + 1.
 * col[(c*ks + k), b*Lout + l] = x[c, b, l*stride + k - pad] (0 outside [0, L)). */
int efm_net_im2col(const uint16_t *x, uint16_t *col, int C, int B, int L, int ks, int stride,
                   int pad, void *stream);
/* Transpose of im2col: dx[c, b, j] = sum over (k, l) with l*stride + k - pad = j
 * of dcol[(c*ks + k), b*Lout + l]. */
int efm_net_col2im(const float *dcol, float *dx, int C, int B, int L, int ks, int stride,
                   int pad, void *stream);

/* dpre = dy * (y > 0); dpre_b (nullable) = bf16(dpre). */
int efm_net_relu_backward(const float *dy, const float *y, float *dpre, uint16_t *dpre_b,
                          long long n, void *stream);
/* db[m] = sum_n dpre[m*N + n]. */
int efm_net_bias_grad(const float *dpre, float *db, int M, long long N, void *stream);

/* A convolution with bias and ReLU, its backward products, and the ReLU and bias
 * backward of a layer, without the im2col matrix in memory.  Kernel sizes 1 to 9 over
 * rows of at least 8 samples (else EFM_E_ARG).
 * x (C, B, L) BF16, W (M, C·ks) BF16; y[m, b*Lout + l] = max(sum_(c,k) W[m, c*ks + k] *
 * x[c, b, l*stride + k - pad] + bias[m], 0) (the sums of efm_net_im2col and
 * efm_net_gemm, bit for bit), yb = bf16(y) at the same offsets or, with flat,
 * flattened as efm_net_flatten. */
int efm_net_conv1d(const uint16_t *x, const uint16_t *W, const float *bias, float *y, uint16_t *yb,
                   int C, int B, int L, int M, int ks, int stride, int pad, int flat, void *stream);
/* 1 if efm_net_conv1d and efm_net_conv1d_back take this convolution, else 0. */
int efm_net_conv1d_fits(int C, int B, int L, int M, int ks, int stride, int pad);
/* ldp below: the distance of dp's (dpb's) rows.  dW (M, C·ks) of dp (M, B·Lout) BF16 against x, and dcol = W^T·dp (C·ks, B·Lout) beside
 * it unless null: the sums of efm_net_gemm over efm_net_im2col's matrix, bit for bit. */
int efm_net_conv1d_back(const uint16_t *dp, const uint16_t *x, const uint16_t *W, float *dW, float *dcol,
                        int C, int B, int L, int M, int ks, int stride, int pad, int ldp, void *stream);
/* dpb = bf16(dy * (y > 0)) and db[m] = sum_n dy * (y > 0) for rows m < M of N values (the
 * sum of efm_net_bias_grad, bit for bit); dy row-major, or with L > 0 flattened as
 * efm_net_flatten (N = B·L).  With chains (256·M floats, see efm_net_bias_split) the sums'
 * chains are left there for efm_net_bias_sums and db is not written. */
int efm_net_relu_bias_backward(const float *dy, const float *y, uint16_t *dpb, float *db, float *chains,
                               int M, int N, int B, int L, int ldp, void *stream);
/* The same for dy = efm_net_col2im(dcol), y (C, B, L). */
int efm_net_col2im_relu_bias(const float *dcol, const float *y, uint16_t *dpb, float *db, float *chains,
                             int C, int B, int L, int ks, int stride, int pad, int ldp,
                             void *stream);
/* Whether M rows of N values are faster through chains. */
int efm_net_bias_split(int M, int N);
/* db[m] from chains[256·m ..] for rows m < M of each of n biases, EFM_NET_BIASES to a launch. */
#define EFM_NET_BIASES 16
typedef struct {
    const float *chains;
    float *db;
    int M;
} EfmNetBias;
int efm_net_bias_sums(const EfmNetBias *biases, int n, void *stream);

/* The dense head.  1 if efm_net_head_forward takes these sizes, 3 if efm_net_head_backward
 * does too (at most 128 examples and 16 outputs), else 0. */
int efm_net_head_fits(int B, int flat, int hidden, int nout);
/* z = max(F1·X + c1, 0), zb = bf16(z), out = F2·zb + c2: X (flat, B), F1 (hidden, flat),
 * F2 (nout, hidden) BF16; the sums of efm_net_gemm, bit for bit. */
int efm_net_head_forward(const uint16_t *X, const uint16_t *F1, const float *c1, const uint16_t *F2,
                         const float *c2, float *z, uint16_t *zb, float *out, int B, int flat,
                         int hidden, int nout, void *stream);
/* loss = inv_n·sum (out - target)^2 (set, not added), and with dout = 2·inv_n·(out - target):
 * dF2 = bf16(dout)·zb^T, dc2 = row sums of dout, dzpb = bf16(dz·(z > 0)) and dc1 = row sums
 * of dz·(z > 0) for dz = F2^T·bf16(dout). */
int efm_net_head_backward(const float *out, const float *target, const float *z, const uint16_t *zb,
                          const uint16_t *F2, float *dF2, float *dc2, float *dc1, uint16_t *dzpb,
                          double *loss, int B, int hidden, int nout, float inv_n, void *stream);
/* Mean-squared error over n values: *loss += sum (out - t)^2 * inv_n (a device
 * double the caller zeroes); dout = 2 (out - t) inv_n; dout_b (nullable) = bf16(dout). */
int efm_net_mse(const float *out, const float *target, float *dout, uint16_t *dout_b,
                double *loss, long long n, float inv_n, void *stream);

/* Adam step on n parameters: m = b1 m + (1-b1) g; v = b2 v + (1-b2) g^2;
 * w -= lr * (m*c1) / (sqrt(v*c2) + eps) with c1 = 1/(1-b1^t), c2 = 1/(1-b2^t);
 * wb (nullable) = bf16(w). */
int efm_net_adam(float *w, const float *g, float *m, float *v, uint16_t *wb, long long n,
                 float lr, float b1, float b2, float eps, float c1, float c2, void *stream);

/* X[(c*L + l), b] = act[c, b, l] (flatten for the dense head) and its transpose
 * dact[c, b, l] = dX[(c*L + l), b]. */
int efm_net_flatten(const uint16_t *act, uint16_t *X, int C, int B, int L, void *stream);
int efm_net_unflatten(const float *dX, float *dact, int C, int B, int L, void *stream);

/* Network inputs from propagator gathers (S, ncomp, ntmax, nrec) FP32:
 * data[s0 + s, comp*nrec + r, l] = bf16(g[s, comp, l, r] / max|g[s]|) for
 * l < L (L <= ntmax), written into a (Ntotal, ncomp*nrec, L) dataset. */
int efm_net_pack_gathers(const float *g, int S, int ncomp, int ntmax, int nrec, int L,
                         uint16_t *data, long long s0, void *stream);
/* Mini-batch assembly from a dataset of ntotal examples: x[c, b, l] =
 * data[idx[b], c, l] (C channels, L samples) and t[j, b] = targets[idx[b]*nout + j];
 * an idx[b] outside [0, ntotal) yields zeros for that example. */
int efm_net_gather_batch(const uint16_t *data, const float *targets, long long ntotal,
                         const int *idx, int B, int C, int L, int nout, uint16_t *x, float *t,
                         void *stream);

#ifdef __cplusplus
}
#endif
#endif
