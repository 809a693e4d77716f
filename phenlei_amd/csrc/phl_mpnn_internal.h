// phl_mpnn_internal.h -- launchers of the warm-start network kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace phl {
namespace nn {

constexpr int kIn = 8;        // cell features
constexpr int kHidden = 128;  // hidden width
constexpr int kOut = 5;       // predicted state

// out[N,128] = relu(X W0 + b0), before the relu also to Z (may be null).
void input_layer(const float *X, const float *W0, const float *b0, int N, float *Z, float *out, hipStream_t s);
// The hidden layers' A_l, B_l as BF16 pieces [L][2][pieces][128][128]: 3, whose
// sum is the FP32 value, or 1, the value rounded to BF16; as they are for the
// forward products, transposed for the backward ones.  bad [L][2][kBadFlags]:
// whether part of a matrix does not split into pieces.
constexpr int kBadFlags = 64;
void split_weights(const float *A, const float *B, int L, int pieces, bool transpose, __bf16 *out, int *bad,
                   hipStream_t s);
// The operands of one product: rows A [N][128], the weights' pieces and flags
// from split_weights, and the FP32 weights they were made of ([k][column], or
// [column][k] when transposed).
struct Product {
    const float *A;
    const __bf16 *W;
    const int *bad;
    const float *W32;
};
// out[N,128] = p1 (+ p2, if its A is not null) + bias, epilogue by mode (see
// the kernel): FP32 products (3 pieces) or BF16 ones (1), FP32 accumulation.
void dense(const Product &p1, const Product &p2, bool transpose, const float *bias, int N, int mode,
           const float *Hres, float *Z, float *out, int pieces, hipStream_t s);
// Weight gradients; part: grad_floats(N) floats of workspace.
size_t grad_floats(int N);
// gA = A^T D, gB = B^T D [128,128] and gc = the column sums of D, all [N,128].
void wgrad(const float *A, const float *B, const float *D, int N, float *part, float *gA, float *gB, float *gc,
           hipStream_t s);
// gW0[8,128] = X^T D, gb0 = the column sums of D.
void input_grad(const float *X, const float *D, int N, float *part, float *gW0, float *gb0, hipStream_t s);
// gWo[128,5] = h^T dy, gbo = the column sums of dy.
void output_grad(const float *h, const float *dy, int N, float *part, float *gWo, float *gbo, hipStream_t s);
void neighbour_mean(const int *nbr, int W, int N, const float *invDeg, const float *h, float *m, hipStream_t s);
void neighbour_mean_transpose_add(const int *nbr, int W, int N, const float *invDeg, const float *dm, float *dh,
                                  hipStream_t s);
void relu_back(const float *dh, const float *z, size_t n, float *dz, hipStream_t s);
void add(float *a, const float *b, size_t n, hipStream_t s);
void out_layer(const float *h, const float *Wo, const float *bo, int N, float *y, hipStream_t s);
void out_layer_back(const float *dy, const float *Wo, int N, float *dh, hipStream_t s);
int loss_parts(int n);
void loss(const float *y, const float *t, int n, float *dy, double *part, double *out, hipStream_t s);
void adam(float *p, const float *g, float *m, float *v, int n, float lr, int step, hipStream_t s);

}  // namespace nn
}  // namespace phl
