/*
 * pmmlp.h -- kernels of the spectral surrogate: a small MLP (dense layers,
 * GELU) trained and evaluated on the matrix cores in BF16 with FP32
 * accumulation and FP32 master weights.
 *
 * The reference has no learned model; its design loop is the parameter
 * sweep of src/prismo/optimization/sweep.py:119-167 (every candidate a full
 * FDTD run).  These entry points let a caller screen candidates with a
 * network trained on spectra from the batched FDTD (pmbatch.h) and send
 * only the promising or uncertain ones back to FDTD.
 *
 * All pointers are device memory (FP32, row-major with the given strides),
 * work is enqueued on `stream` (hipStream_t); status codes as pmfdtd.h.
 */
#ifndef PMMLP_H
#define PMMLP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

enum pm_mlp_mode {
  PM_MLP_LINEAR = 0,  /* C = A B (+ bias[n])                                 */
  PM_MLP_GELU = 1,    /* Z = A B + bias[n] stored to Z;  C = gelu(Z)         */
  PM_MLP_DGELU = 2,   /* C = (A B) * gelu'(Z)   (Z read: the layer's input)  */
  PM_MLP_PLAIN = 3    /* C = A B                                            */
};

/* C[m][n] (m < M, n < N, row stride ldc) from A[m][k] = A[m*lda_m + k*lda_k]
 * and B[k][n] = B[k*ldb_k + n*ldb_n], k < K.  Operands are rounded to BF16
 * (round to nearest even) for the MFMA products, sums are FP32.
 * gelu(z) = z (1 + erf(z / sqrt 2)) / 2. */
int pm_mlp_gemm(void* stream, int mode, int32_t M, int32_t N, int32_t K, const float* A,
                int64_t lda_m, int64_t lda_k, const float* B, int64_t ldb_k, int64_t ldb_n,
                float* C, int64_t ldc, const float* bias, float* Z);

/* out[n] = sum_m A[m*lda + n], n < N (bias gradients). */
int pm_mlp_colsum(void* stream, int32_t M, int32_t N, const float* A, int64_t lda, float* out);

/* Mean squared error over M x N with a per-column weight w[n] (NULL = 1):
 * loss[0] = sum w (Y-T)^2 / (M N) (accumulated with atomics into loss, which
 * the caller zeroes), dY = 2 w (Y - T) / (M N). */
int pm_mlp_mse(void* stream, int32_t M, int32_t N, const float* Y, const float* T,
               const float* w, float* dY, float* loss);

/* Batched forms: `batch` independent problems of the same shape (1 <=
 * batch <= 65535), problem q reading and writing its operands at q times
 * the given stride (in elements) from the base pointers; each problem's
 * result is the one the single call gives.  Loss of problem q in loss[q].
 * No counterpart in the reference: the surrogate trains its ensemble
 * members in lockstep, one launch for all members. */
int pm_mlp_gemm_batched(void* stream, int mode, int32_t batch, int32_t M, int32_t N, int32_t K,
                        const float* A, int64_t lda_m, int64_t lda_k, int64_t stride_a,
                        const float* B, int64_t ldb_k, int64_t ldb_n, int64_t stride_b,
                        float* C, int64_t ldc, int64_t stride_c, const float* bias,
                        int64_t stride_bias, float* Z, int64_t stride_z);
int pm_mlp_colsum_batched(void* stream, int32_t batch, int32_t M, int32_t N, const float* A,
                          int64_t lda, int64_t stride_a, float* out, int64_t stride_out);
int pm_mlp_mse_batched(void* stream, int32_t batch, int32_t M, int32_t N, const float* Y,
                       const float* T, int64_t stride, const float* w, float* dY, float* loss);

/* Adam with decoupled weight decay on n FP32 parameters, step t >= 1. */
int pm_mlp_adam(void* stream, int64_t n, float* p, const float* g, float* m, float* v,
                float lr, float beta1, float beta2, float eps, float weight_decay, int32_t t);

/* Whole networks: layers 1 <= L <= 12 of widths sizes[0] (input) ..
 * sizes[L] (output), each 1 .. 512; GELU after every layer but the last.  A
 * member's parameters are flat: all weights ([out][in] row-major, layer by
 * layer), then all biases.  Members (1 <= batch <= 65535) lie at multiples of
 * the given strides (elements).  The sums of every product are those of
 * pm_mlp_gemm.
 *
 * The kernels read the weights as BF16 in their operand order: `packed`, a
 * zero-filled buffer of pm_mlp_net_packed elements per member (with train != 0
 * also the transposes the backward pass reads; 0: the network is not taken),
 * 16-byte aligned with a stride that is a multiple of 8. */
int64_t pm_mlp_net_packed(int32_t layers, const int32_t* sizes, int32_t train);
int pm_mlp_net_pack(void* stream, int32_t batch, int32_t layers, const int32_t* sizes,
                    const float* P, int64_t stride_p, uint16_t* packed, int64_t stride_packed,
                    int32_t train);

/* Y[m][:] of every member for rows X[m][:] (stride_x 0: the members share X).
 * acts / zs (both or neither): activations and pre-activations of the hidden
 * layers, layer k as (M, sizes[k+1]) after the layers before it. */
int pm_mlp_net_forward(void* stream, int32_t batch, int32_t M, int32_t layers,
                       const int32_t* sizes, const float* P, int64_t stride_p,
                       const uint16_t* packed, int64_t stride_packed, const float* X,
                       int64_t stride_x, float* Y, int64_t stride_y, float* acts, float* zs,
                       int64_t stride_a);

/* One pass over `rows` training rows in minibatches of batch_rows (the last
 * one shorter): per minibatch s the mean squared error's gradient (weights w
 * per output column, NULL = 1) in G and one Adam step t0 + s + 1 with rate
 * lr[s] (a host array) and decay weight_decay on the weights.  Row r of member
 * q is row idx[q * stride_idx + r] of X and T (shared by the members).  packed
 * (train != 0) holds P's weights and is kept up to date; work:
 * batch * pm_mlp_net_work(.., batch_rows) elements, 16-byte aligned (else
 * PM_EINVAL); loss[s * batch + q], zeroed by the caller. */
int64_t pm_mlp_net_work(int32_t layers, const int32_t* sizes, int32_t rows);
int pm_mlp_net_train(void* stream, int32_t batch, int32_t layers, const int32_t* sizes, float* P,
                     float* G, float* m, float* v, int64_t stride_p, uint16_t* packed,
                     int64_t stride_packed, const float* X, const float* T, const int64_t* idx,
                     int64_t stride_idx, const float* w, int32_t rows, int32_t batch_rows,
                     float* work, const float* lr, float beta1, float beta2, float eps,
                     float weight_decay, int32_t t0, float* loss);

/* Mean and standard deviation (divisor members - 1) over the members of n
 * values at S[q * stride]. */
int pm_mlp_net_stats(void* stream, int32_t members, int64_t n, const float* S, int64_t stride,
                     float* mean, float* std);

#ifdef __cplusplus
}
#endif
#endif /* PMMLP_H */
