// phl_mpnn.hip -- the warm-start message-passing network on gfx950: forward,
// backward and Adam, hand-written, FP32 with the dense layers on MFMA
// (v_mfma_f32_32x32x16_bf16 on exact three-way splits of the FP32 operands).
// The network (no reference counterpart):
//
//     h0 = relu(X W0 + b0)                     X [N, 8] cell features
//     l = 1..L:  m = mean_{j in N(i)} h_j       (face neighbours)
//                z = h A_l + m B_l + c_l ;  h = h + relu(z)
//     y  = h Wo + bo                           y [N, 5]
//
// Rows are cells, columns features, all row-major.  The hidden width is 128.
// Every reduction (weight gradients, bias gradients, loss) is a sum in a
// fixed order (no atomics), so training is deterministic.
#include "phl_mpnn_internal.h"

#include <hip/hip_runtime.h>

namespace phl {
namespace nn {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int H = kHidden;    // 128
constexpr int TR = 128;       // rows per workgroup tile
constexpr int kThreads = 256; // 4 waves
constexpr int kRowChunk = 2048;  // rows per partial of a weight gradient
constexpr int kMaxDeg = 8;       // neighbour lists up to this width take the batched-load path

// Logical block of hardware block b of nblk: workgroups go to the 8 XCDs
// round-robin, so this gives each XCD a contiguous range, whose cells'
// neighbours are rows that the same L2 holds (neighbour mean of 621,818 rows:
// 268 us in launch order, 215 so; of 123,240 rows 50 and 41).
__device__ __forceinline__ int xcd_block(int b, int nblk)
{
    const int q = nblk >> 3, r = nblk & 7, x = b & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// The 32x32 accumulator tiles of MFMA: register r of lane l holds
// D[(r % 4) + 4 * (l / 32) + 8 * (r / 4)][l % 32].
__device__ __forceinline__ int acc_row(int r, int lane) { return (r & 3) + 4 * (lane >> 5) + 8 * (r >> 2); }

// Input layer: z = X W0 + b0, out = relu(z); Z may be null.  Eight products
// per output, so the 512-byte rows written bound it: a thread keeps its four
// columns of W0 and walks kInRows rows.
constexpr int kInRows = 16;
__global__ void __launch_bounds__(kThreads) k_input(const float *__restrict__ X, const float *__restrict__ W0,
                                                    const float *__restrict__ b0, int N, float *__restrict__ Z,
                                                    float *__restrict__ out)
{
    static_assert(kIn == 8 && H == 128, "k_input's thread layout");
    const int c = 4 * ((int)threadIdx.x & 31);
    float4 w[kIn];
#pragma unroll
    for (int k = 0; k < kIn; ++k) w[k] = *(const float4 *)(W0 + k * H + c);
    const float4 b = *(const float4 *)(b0 + c);
    const int r0 = blockIdx.x * (8 * kInRows) + ((int)threadIdx.x >> 5);
#pragma unroll 4
    for (int i = 0; i < kInRows; ++i) {
        const int row = r0 + 8 * i;
        if (row >= N) return;
        const float4 x0 = *(const float4 *)(X + (size_t)row * kIn), x1 = *(const float4 *)(X + (size_t)row * kIn + 4);
        const float x[kIn] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int k = 0; k < kIn; ++k) {
            z.x = fmaf(x[k], w[k].x, z.x);
            z.y = fmaf(x[k], w[k].y, z.y);
            z.z = fmaf(x[k], w[k].z, z.z);
            z.w = fmaf(x[k], w[k].w, z.w);
        }
        z.x += b.x;
        z.y += b.y;
        z.z += b.z;
        z.w += b.w;
        const size_t o = (size_t)row * H + c;
        if (Z) *(float4 *)(Z + o) = z;
        *(float4 *)(out + o) = make_float4(z.x > 0.f ? z.x : 0.f, z.y > 0.f ? z.y : 0.f, z.z > 0.f ? z.z : 0.f,
                                           z.w > 0.f ? z.w : 0.f);
    }
}

// ---- products on BF16 matrix cores ----
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// x as NP BF16 pieces.  NP 1: x rounded to nearest even.  NP 3: three pieces
// (8 significant bits each, 24 in all): piece 0 is x rounded, piece 1 the
// remainder rounded, piece 2 what is left, and x is their exact sum.  It is not
// where x rounds to infinity (from 0x7f7f8000 on, infinities and NaN among
// them) or has bits below BF16's smallest subnormal, 2^-133 (from 2^-110 down).
// Returns what the pieces leave of x as bits without the sign: 0 if x splits.
template <int NP>
__device__ __forceinline__ unsigned split(float x, __bf16 *p)
{
    p[0] = (__bf16)x;
    if constexpr (NP == 3) {
        const float r = x - (float)p[0];
        p[1] = (__bf16)r;
        const float s = r - (float)p[1];
        p[2] = (__bf16)s;
        return __float_as_uint(s - (float)p[2]) & 0x7fffffffu;
    }
    return 0;
}

// The products of two three-piece operands that are kept beside the leading
// one: piece kTermA against piece kTermB.  Pieces 1 and 2 are at most 2^-8 and
// 2^-17 of a value in [1, 2), so the three left out are at most 2^-25, 2^-25 and
// 2^-34 of a product: with the rounding of the sum a single product is within
// 2^-23 of itself (1.78 x 2^-24 measured where every piece is as large as it can
// be), an FP32 product within 2^-24.  The sums do not feel it: over 25 seeds each of
// 39,600 and 123,240 rows the median error of the worst gradient tensor against
// 64 bits was 1.2e-6 and 1.3e-6 with FP32 products, 3.0e-7 and 8.5e-7 with these
// six terms, 3.1e-7 and 9.9e-7 with the two of 2^-25 as well, which took 5% more
// time for a whole pass.
constexpr int kTerms = 5, kTermA[kTerms] = {2, 0, 1, 1, 0}, kTermB[kTerms] = {0, 2, 1, 0, 1};

// Nonzero if a sum of a tile is infinite or NaN.  The leading pieces are
// rounded, so their product may overflow where that of the values does not.
__device__ __forceinline__ unsigned not_finite(const f32x16 (&acc)[2][2])
{
    unsigned top = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) top = max(top, __float_as_uint(acc[i][j][r]) & 0x7fffffffu);
    return top >= 0x7f800000u;
}

// out[N, 128] = A1[N, 128] W1 (+ A2[N, 128] W2) + bias, W1 and W2 as NP
// pieces from k_split_weights; A split while it is staged.  Epilogue: z =
// product + bias stored to Z (if non-null); out = z (mode 0), Hres + relu(z)
// (mode 2) or Hres + z (mode 3).
//
// A workgroup makes 128 rows x 128 columns, each of its four waves 64 x 64 in
// 2 x 2 accumulator tiles.  A runs through two LDS buffers of KB columns,
// the loads one chunk ahead of the stores and the stores one ahead of the
// products.  Lane l supplies A[l % 32][8 (l / 32) .. + 7] and
// B[8 (l / 32) .. + 7][l % 32] of a K = 16 step: A in one 16-byte LDS read per
// piece; the weights lie in memory as such operands, 1 KB per wave and piece,
// and come from the L2 caches straight into registers, a step ahead.
//
// NP 3 replaces v_mfma_f32_32x32x2_f32 (157 TFLOP/s): six BF16 products of
// 16 k take 192 cycles against 512.  Its error against 64 bits is no larger:
// network output 2.5e-7 against 2.9e-7 (200,704 rows), gradients (with
// k_wgrad_part) 4.7e-8 against 2.4e-7 at 315 rows and as under kTerms at
// 123,240.  A hidden layer of 200,704 rows takes 134 us instead of 262 (66 us
// are the bytes alone), bound by the latency of a workgroup's eight chunks at
// two workgroups per CU.  NP 1 (inference) is bound by its 1,536 bytes of
// activations per row: 621,818 rows in 224 us instead of 351, 4.3 TB/s.
//
// A value that does not split (see split), in the rows or in the weights
// (`bad`, one int per workgroup of k_split_weights), or a sum that is not
// finite, makes the tile be summed again value by value in FP32.
constexpr int KB = 32;       // K chunk staged in LDS
constexpr int KBP = KB + 8;  // LDS row length: 80-byte rows keep every 16-byte read aligned and conflict-free
constexpr int kVec = TR * KB / 4 / kThreads;  // float4 of A per thread and chunk (4)
constexpr int kSteps = KB / 16;               // K steps per chunk
static_assert(kVec * 4 * kThreads == TR * KB && H == TR, "chunk shares");
static_assert(kBadFlags == H * H / kThreads && kBadFlags == 64, "one flag per workgroup and per lane");

// Element (k, column) of a piece of a weight matrix in operand order:
// [K step of 16][32 columns][lane][8].
__device__ __forceinline__ int weight_at(int k, int col)
{
    return (((k >> 4) * (H / 32) + (col >> 5)) * 64 + ((k >> 3) & 1) * 32 + (col & 31)) * 8 + (k & 7);
}

__device__ __forceinline__ void load_rows(float4 (&st)[kVec], const float *__restrict__ A, int N, int row0, int k0)
{
#pragma unroll
    for (int i = 0; i < kVec; ++i) {  // A [TR][KB]: row q/8, k 4(q%8)..+3; rows past N repeat the last
        const int q = threadIdx.x + i * kThreads;
        st[i] = *(const float4 *)(A + (size_t)min(row0 + (q >> 3), N - 1) * H + k0 + 4 * (q & 7));
    }
}

// Returns nonzero if a value stored does not split.
template <int NP>
__device__ __forceinline__ unsigned store_rows(const float4 (&st)[kVec], __bf16 (*Al)[TR][KBP])
{
    unsigned left = 0;
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
        const int q = threadIdx.x + i * kThreads;
        const float x[4] = {st[i].x, st[i].y, st[i].z, st[i].w};
        bf16x4 v[NP];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            __bf16 pc[NP];
            left |= split<NP>(x[e], pc);
#pragma unroll
            for (int p = 0; p < NP; ++p) v[p][e] = pc[p];
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) *(bf16x4 *)&Al[p][q >> 3][4 * (q & 7)] = v[p];
    }
    return left;
}

// The wave's weight operands of K step `step`.
template <int NP>
__device__ __forceinline__ void load_weights(bf16x8 (&w)[NP][2], const __bf16 *__restrict__ W, int step, int wc,
                                             int lane)
{
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int j = 0; j < 2; ++j)
            w[p][j] = *(const bf16x8 *)(W + (size_t)p * H * H + ((step * (H / 32) + (wc >> 5) + j) * 64 + lane) * 8);
}

// One value of A W summed in FP32.
__device__ float dot_fp32(const Product &p, bool transpose, int row, int col, float s)
{
    for (int k = 0; k < H; ++k)
        s = fmaf(p.A[(size_t)row * H + k], p.W32[transpose ? col * H + k : k * H + col], s);
    return s;
}

template <int NP>
__global__ void __launch_bounds__(kThreads, 2) k_dense(Product P1, Product P2, bool transpose,
                                                       const float *__restrict__ bias, int N, int mode,
                                                       const float *__restrict__ Hres, float *__restrict__ Z,
                                                       float *__restrict__ out)
{
    const float *__restrict__ A1 = P1.A, *__restrict__ A2 = P2.A;
    const __bf16 *__restrict__ W1 = P1.W, *__restrict__ W2 = P2.W;
    __shared__ __attribute__((aligned(16))) __bf16 Al[2][NP][TR][KBP];
    const int row0 = blockIdx.x * TR;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wr = 64 * (wave >> 1), wc = 64 * (wave & 1);  // the wave's rows and columns
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    constexpr int half = H / KB;  // chunks of one operand
    const int chunks = A2 ? 2 * half : half;
    unsigned odd = 0;  // nonzero: the tile takes the FP32 sums
    if constexpr (NP == 3) odd = P1.bad[lane] | (A2 ? P2.bad[lane] : 0);
    float4 st[kVec];
    bf16x8 w[kSteps][NP][2];
    load_rows(st, A1, N, row0, 0);
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks) load_weights<NP>(w[ks], W1, ks, wc, lane);
    odd |= store_rows<NP>(st, Al[0]);
    load_rows(st, A1, N, row0, KB);
    __syncthreads();
    for (int ch = 0; ch < chunks; ++ch) {
        const int nc = ch + 1;
        const __bf16 *Wn = nc >= half ? W2 : W1;
#pragma unroll
        for (int ks = 0; ks < kSteps; ++ks) {
            const int k = 16 * ks + 8 * (lane >> 5), l = lane & 31;
            bf16x8 a[NP][2];
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int i = 0; i < 2; ++i) a[p][i] = *(const bf16x8 *)&Al[ch & 1][p][wr + 32 * i + l][k];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if constexpr (NP == 3) {
                        // the five small terms on their own, so that the sum takes one rounding for them
                        f32x16 t;
#pragma unroll
                        for (int r = 0; r < 16; ++r) t[r] = 0.f;
#pragma unroll
                        for (int q = 0; q < kTerms; ++q)
                            t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kTermA[q]][i], w[ks][kTermB[q]][j], t, 0, 0,
                                                                        0);
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][i], w[ks][0][j], acc[i][j], 0, 0, 0);
                        acc[i][j] += t;
                    } else {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][i], w[ks][0][j], acc[i][j], 0, 0, 0);
                    }
                }
            // this step's weights of the next chunk
            if (nc < chunks) load_weights<NP>(w[ks], Wn, (nc % half) * kSteps + ks, wc, lane);
        }
        if (nc < chunks) odd |= store_rows<NP>(st, Al[nc & 1]);
        if (ch + 2 < chunks) load_rows(st, ch + 2 >= half ? A2 : A1, N, row0, ((ch + 2) % half) * KB);
        __syncthreads();
    }
    if constexpr (NP == 3) odd |= not_finite(acc);
    if (NP == 3 && __syncthreads_or(odd != 0)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = row0 + wr + 32 * i + acc_row(r, lane), col = wc + 32 * j + (lane & 31);
                    if (row >= N) continue;
                    float v = dot_fp32(P1, transpose, row, col, 0.f);
                    if (A2) v = dot_fp32(P2, transpose, row, col, v);
                    acc[i][j][r] = v;
                }
    }
    // one 32 x 32 tile at a time, its 16 residual loads in flight together
    // (behind a branch per row each would wait for the one before it); rows
    // past N are clamped for the loads and left out of the stores
    const bool full = row0 + TR <= N;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int col = wc + 32 * j + (lane & 31);
            const float bc = bias ? bias[col] : 0.f;
            float h[16];
            if (mode != 0) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    h[r] = Hres[(size_t)min(row0 + wr + 32 * i + acc_row(r, lane), N - 1) * H + col];
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) h[r] = 0.f;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = row0 + wr + 32 * i + acc_row(r, lane);
                const size_t o = (size_t)row * H + col;
                const float z = acc[i][j][r] + bc;
                const float v = mode == 0 ? z : (mode == 2 ? h[r] + (z > 0.f ? z : 0.f) : h[r] + z);
                if (full || row < N) {
                    if (Z) Z[o] = z;
                    out[o] = v;
                }
            }
        }
}

// The hidden layers' A_l and B_l [L][128][128] FP32 as NP BF16 pieces in
// operand order, out [L][2][NP][128 * 128] (A_l, then B_l): as they are for the
// forward products h A, m B (k the row), or transposed for the backward
// products dz A^T, dz B^T (k the column).
template <int NP>
__global__ void __launch_bounds__(kThreads) k_split_weights(const float *__restrict__ A, const float *__restrict__ B,
                                                            int L, bool transpose, __bf16 *__restrict__ out,
                                                            int *__restrict__ bad)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t HH = (size_t)H * H;
    static_assert(H * H % kThreads == 0, "the grid covers whole matrices");
    const size_t lw = i / HH, r = i % HH;
    const int u = (int)(r / H), v = (int)(r % H);  // W[u][v] of the layer's matrix
    const float w = (((lw & 1) ? B : A) + (lw >> 1) * HH)[r];
    __bf16 p[NP];
    const unsigned left = split<NP>(w, p);
#pragma unroll
    for (int q = 0; q < NP; ++q) out[(lw * NP + q) * HH + (transpose ? weight_at(v, u) : weight_at(u, v))] = p[q];
    const int any = __syncthreads_or(left != 0);
    if (threadIdx.x == 0) bad[blockIdx.x] = any;
}

// ---- weight gradients ----
// Sums over all rows, in two steps of fixed order: partials over chunks of
// rows, then the partials (k_sum_parts).  A chunk is what gives about one
// workgroup per CU, at most kRowChunk rows (the FP32 chain of a partial): with
// 2,048 rows whatever N, 123,240 rows kept 61 of 256 CUs busy.
constexpr int kSlab = 32;           // rows staged at a time
constexpr int kSlabP = kSlab + 8;   // LDS row length, as KBP
constexpr int kGradThreads = 512;   // waves 0-3: A^T D, waves 4-7: B^T D
inline __host__ __device__ int grad_rows(int N)
{
    const int r = ((N + 255) / 256 + kSlab - 1) / kSlab * kSlab;
    return r < kRowChunk ? r : kRowChunk;
}
constexpr int kGradOut = 2 * H * H + H;  // A^T D, B^T D and the column sums of D

// Partials of A^T D, B^T D [128, 128] and of the column sums of D over rows
// r0 .. r0 + rows of A, B, D [N, 128], FP32 operands in three BF16 pieces as in
// k_dense.  The products run along the rows, so a slab is staged transposed
// ([feature][row], eight rows of a feature per 16-byte store) and a row of D
// is read once for both products and the bias.  123,240 rows: 78 us, and 17
// for the sum, for what took 420 (two products, FP32 MFMA) and 71 (the bias).
__global__ void __launch_bounds__(kGradThreads, 2) k_wgrad_part(const float *__restrict__ A,
                                                                const float *__restrict__ B,
                                                                const float *__restrict__ D, int N, int rows,
                                                                float *__restrict__ part)
{
    __shared__ __attribute__((aligned(16))) __bf16 T[3][3][H][kSlabP];  // operand, piece, feature, row
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int op = wave >> 2, wr = 64 * ((wave >> 1) & 1), wc = 64 * (wave & 1);
    const int r0 = blockIdx.x * rows, r1 = min(r0 + rows, N);
    const int f = threadIdx.x & (H - 1), g = threadIdx.x >> 7;  // staging: feature, rows 8g .. 8g + 7
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    float st[3][8], colSum = 0.f;
    unsigned odd = 0;
    auto load = [&](int s) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int row = s + 8 * g + i;
            const size_t o = (size_t)min(row, N - 1) * H + f;
            const float a = A[o], b = B[o], d = D[o];
            st[0][i] = row < r1 ? a : 0.f;
            st[1][i] = row < r1 ? b : 0.f;
            st[2][i] = row < r1 ? d : 0.f;
        }
    };
    load(r0);
    for (int s = r0; s < r1; s += kSlab) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            bf16x8 v[3];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                __bf16 p[3];
                odd |= split<3>(st[q][i], p);
                v[0][i] = p[0];
                v[1][i] = p[1];
                v[2][i] = p[2];
            }
#pragma unroll
            for (int p = 0; p < 3; ++p) *(bf16x8 *)&T[q][p][f][8 * g] = v[p];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) colSum += st[2][i];
        __syncthreads();
        if (s + kSlab < r1) load(s + kSlab);
#pragma unroll
        for (int ks = 0; ks < kSlab; ks += 16) {
            const int k = ks + 8 * (lane >> 5), l = lane & 31;
            bf16x8 a[3][2], d[3][2];
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    a[p][i] = *(const bf16x8 *)&T[op][p][wr + 32 * i + l][k];
                    d[p][i] = *(const bf16x8 *)&T[2][p][wc + 32 * i + l][k];
                }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    f32x16 t;
#pragma unroll
                    for (int r = 0; r < 16; ++r) t[r] = 0.f;
#pragma unroll
                    for (int q = 0; q < kTerms; ++q)
                        t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kTermA[q]][i], d[kTermB[q]][j], t, 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][i], d[0][j], acc[i][j], 0, 0, 0);
                    acc[i][j] += t;
                }
        }
    }
    odd |= not_finite(acc);
    if (__syncthreads_or(odd != 0)) {  // as in k_dense
        const float *S = op ? B : A;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = wr + 32 * i + acc_row(r, lane), col = wc + 32 * j + (lane & 31);
                    float v = 0.f;
                    for (int n = r0; n < r1; ++n) v = fmaf(S[(size_t)n * H + row], D[(size_t)n * H + col], v);
                    acc[i][j][r] = v;
                }
    }
    float *p = part + (size_t)blockIdx.x * kGradOut;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                p[op * H * H + (wr + 32 * i + acc_row(r, lane)) * H + wc + 32 * j + (lane & 31)] = acc[i][j][r];
    float *red = reinterpret_cast<float *>(T);  // [4][H]; every read of T is behind the barrier above
    red[g * H + f] = colSum;
    __syncthreads();
    if (g == 0) p[2 * H * H + f] = (red[f] + red[H + f]) + (red[2 * H + f] + red[3 * H + f]);
}

// The gradients of the input and the output layer: partials over `rows` rows
// of V^T M [KS, 128] for M [N, 128] and V [N, KS], thread = a column of M and
// every other row (a row of V is the same for a whole wave).
// Input layer (SUMS 0): G[k][c] as it is, then the column sums of M.
// Output layer (SUMS 1): G as [c][k], then the column sums of V.
template <int KS, int SUMS>
__global__ void __launch_bounds__(kThreads) k_edge_grad_part(const float *__restrict__ M, const float *__restrict__ V,
                                                             int N, int rows, float *__restrict__ part)
{
    constexpr int nOut = KS * H + (SUMS ? KS : H);
    __shared__ float red[nOut];
    const int c = threadIdx.x & (H - 1), half = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 7);
    const int r0 = blockIdx.x * rows, r1 = min(r0 + rows, N);
    float s[KS], sv[KS], sm = 0.f;
#pragma unroll
    for (int k = 0; k < KS; ++k) s[k] = sv[k] = 0.f;
#pragma unroll 8
    for (int r = r0 + half; r < r1; r += 2) {
        const float x = M[(size_t)r * H + c];
        sm += x;
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const float v = V[(size_t)r * KS + k];
            s[k] = fmaf(v, x, s[k]);
            if (SUMS) sv[k] += v;
        }
    }
    if (half) {
#pragma unroll
        for (int k = 0; k < KS; ++k) red[SUMS ? c * KS + k : k * H + c] = s[k];
        if (!SUMS) red[KS * H + c] = sm;
        else if (c == 0)
#pragma unroll
            for (int k = 0; k < KS; ++k) red[KS * H + k] = sv[k];
    }
    __syncthreads();
    if (half) return;
    float *p = part + (size_t)blockIdx.x * nOut;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        const int e = SUMS ? c * KS + k : k * H + c;
        p[e] = s[k] + red[e];
    }
    if (!SUMS) p[KS * H + c] = sm + red[KS * H + c];
    else if (c == 0)
#pragma unroll
        for (int k = 0; k < KS; ++k) p[KS * H + k] = sv[k] + red[KS * H + k];
}
inline __host__ __device__ int edge_rows(int N)
{
    const int r = (N + 1023) / 1024;
    return r < 64 ? 64 : (r < kRowChunk ? r : kRowChunk);
}

// Sums of nPart partials of n values, written in up to three runs (the first
// n0 values to o0, the next n1 to o1, the rest to o2).  A workgroup owns 64
// consecutive values (lane = value); wave w adds partials w, w + 4, w + 8, ..
// in order and the four wave sums are added in wave order: a fixed order, so
// the result is deterministic.  The partials are many and their sum long, so
// it is kept in FP64 (free: the kernel is bound by reading them).
constexpr int kSumWaves = kThreads / 64;
__global__ void __launch_bounds__(kThreads) k_sum_parts(const float *__restrict__ part, int nPart, int n, int n0,
                                                        int n1, float *__restrict__ o0, float *__restrict__ o1,
                                                        float *__restrict__ o2)
{
    __shared__ double red[kSumWaves][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int e = blockIdx.x * 64 + lane;
    double s = 0.0;
    if (e < n)
#pragma unroll 8
        for (int i = wave; i < nPart; i += kSumWaves) s += double(part[(size_t)i * n + e]);
    red[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && e < n) {
        double d = red[0][lane];
        for (int w = 1; w < kSumWaves; ++w) d += red[w][lane];
        const float t = float(d);
        if (e < n0) o0[e] = t;
        else if (e < n0 + n1) o1[e - n0] = t;
        else o2[e - n0 - n1] = t;
    }
}

// m_i = mean of h_j over the neighbours of i (scale = 1/deg_i), or, for the
// transpose in the backward pass, out_j += sum over neighbours i of
// w_i * h_i with w_i = 1/deg_i (TRANSPOSE).
// One thread per (cell, 4 columns), float4 rows; each column is summed in
// list order, as a scalar loop over the neighbours would sum it.
template <bool TRANSPOSE>
__device__ __forceinline__ void add_row(float4 &s, const float4 x, const float *__restrict__ invDeg, int j)
{
    if (TRANSPOSE) {
        const float w = invDeg[j];
        s.x += x.x * w;
        s.y += x.y * w;
        s.z += x.z * w;
        s.w += x.w * w;
    } else {
        s.x += x.x;
        s.y += x.y;
        s.z += x.z;
        s.w += x.w;
    }
}

template <bool TRANSPOSE>
__global__ void __launch_bounds__(kThreads) k_neighbour(const int *__restrict__ nbr, int W, int N,
                                                        const float *__restrict__ invDeg,
                                                        const float *__restrict__ h, float *__restrict__ out)
{
    constexpr int Q = H / 4;
    const size_t e = (size_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (e >= (size_t)N * Q) return;
    const int i = (int)(e / Q), c = 4 * (int)(e % Q);
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    if (W <= kMaxDeg) {
        // every index, then every row, in flight together; the lists are
        // compacted (valid entries first), so the sum order is k = 0, 1, ..
        int j[kMaxDeg];
        float4 x[kMaxDeg];
#pragma unroll
        for (int k = 0; k < kMaxDeg; ++k) j[k] = k < W ? nbr[(size_t)k * N + i] : -1;
#pragma unroll
        for (int k = 0; k < kMaxDeg; ++k) {
            x[k] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (j[k] >= 0) x[k] = *(const float4 *)(h + (size_t)j[k] * H + c);
        }
#pragma unroll
        for (int k = 0; k < kMaxDeg; ++k) {
            if (j[k] < 0) break;
            add_row<TRANSPOSE>(s, x[k], invDeg, j[k]);
        }
    } else {
        for (int k = 0; k < W; ++k) {
            const int jk = nbr[(size_t)k * N + i];
            if (jk < 0) break;
            add_row<TRANSPOSE>(s, *(const float4 *)(h + (size_t)jk * H + c), invDeg, jk);
        }
    }
    float4 *o = (float4 *)(out + (size_t)i * H + c);
    if (TRANSPOSE) {
        float4 v = *o;
        v.x += s.x;
        v.y += s.y;
        v.z += s.z;
        v.w += s.w;
        *o = v;
    } else {
        const float w = invDeg[i];
        *o = make_float4(s.x * w, s.y * w, s.z * w, s.w * w);
    }
}

// dz = dh * (z > 0): thread t does elements 4t..4t+3 (float4 when all four
// are in range; the arrays are rows of 128 floats, so only a tail past n
// would not be), scalar for a tail.
__global__ void __launch_bounds__(kThreads) k_relu_back(const float *__restrict__ dh, const float *__restrict__ z,
                                                        size_t n, float *__restrict__ dz)
{
    const size_t e = 4 * ((size_t)blockIdx.x * blockDim.x + threadIdx.x);
    if (e + 4 <= n) {
        const float4 zv = *(const float4 *)(z + e), hv = *(const float4 *)(dh + e);
        *(float4 *)(dz + e) = make_float4(zv.x > 0.f ? hv.x : 0.f, zv.y > 0.f ? hv.y : 0.f,
                                          zv.z > 0.f ? hv.z : 0.f, zv.w > 0.f ? hv.w : 0.f);
    } else {
        for (size_t k = e; k < n; ++k) dz[k] = z[k] > 0.f ? dh[k] : 0.f;
    }
}

__global__ void __launch_bounds__(kThreads) k_add(float *__restrict__ a, const float *__restrict__ b, size_t n)
{
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n) a[e] += b[e];
}

// Output layer: y = h Wo + bo, one thread per row (float4 reads of h), each
// output summed over k = 0..127 in order.
__global__ void __launch_bounds__(kThreads) k_out(const float *__restrict__ h, const float *__restrict__ Wo,
                                                  const float *__restrict__ bo, int N, float *__restrict__ y)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    float s[kOut];
#pragma unroll
    for (int o = 0; o < kOut; ++o) s[o] = bo[o];
    const float4 *hr = (const float4 *)(h + (size_t)i * H);
    for (int q = 0; q < H / 4; ++q) {
        const float4 x = hr[q];
        const float *w = Wo + 4 * q * kOut;
#pragma unroll
        for (int o = 0; o < kOut; ++o) s[o] += x.x * w[o];
#pragma unroll
        for (int o = 0; o < kOut; ++o) s[o] += x.y * w[kOut + o];
#pragma unroll
        for (int o = 0; o < kOut; ++o) s[o] += x.z * w[2 * kOut + o];
#pragma unroll
        for (int o = 0; o < kOut; ++o) s[o] += x.w * w[3 * kOut + o];
    }
#pragma unroll
    for (int o = 0; o < kOut; ++o) y[(size_t)i * kOut + o] = s[o];
}

// dh = dy Wo^T, one thread per (row, hidden column).
__global__ void __launch_bounds__(kThreads) k_out_back(const float *__restrict__ dy, const float *__restrict__ Wo,
                                                       int N, float *__restrict__ dh)
{
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)N * H) return;
    const int i = (int)(e / H), k = (int)(e % H);
    float s = 0.f;
#pragma unroll
    for (int o = 0; o < kOut; ++o) s += dy[(size_t)i * kOut + o] * Wo[k * kOut + o];
    dh[e] = s;
}

// dy = 2 (y - t) / (N * 5) and per-block partial sums of (y - t)^2.
__global__ void __launch_bounds__(kThreads) k_loss(const float *__restrict__ y, const float *__restrict__ t, int n,
                                                   float scale, float *__restrict__ dy, double *__restrict__ part)
{
    __shared__ double red[kThreads];
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    double s = 0.0;
    if (e < n) {
        const float d = y[e] - t[e];
        dy[e] = 2.f * d * scale;
        s = (double)d * (double)d;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void k_loss_final(const double *__restrict__ part, int nPart, double scale, double *__restrict__ out)
{
    __shared__ double red[kThreads];
    double s = 0.0;
    for (int i = threadIdx.x; i < nPart; i += blockDim.x) s += part[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0] * scale;
}

// Adam with bias correction (Kingma & Ba 2015, Algorithm 1).
__global__ void __launch_bounds__(kThreads) k_adam(float *__restrict__ p, const float *__restrict__ g,
                                                   float *__restrict__ m, float *__restrict__ v, int n, float lr,
                                                   float b1, float b2, float c1, float c2, float eps)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const float gi = g[e];
    const float mi = b1 * m[e] + (1.f - b1) * gi;
    const float vi = b2 * v[e] + (1.f - b2) * gi * gi;
    m[e] = mi;
    v[e] = vi;
    p[e] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

inline int nb(size_t n, int b) { return (int)((n + b - 1) / b); }

}  // namespace

// ---------------------------------------------------------------- launchers
void input_layer(const float *X, const float *W0, const float *b0, int N, float *Z, float *out, hipStream_t s)
{
    hipLaunchKernelGGL(k_input, dim3(nb(N, 8 * kInRows)), dim3(kThreads), 0, s, X, W0, b0, N, Z, out);
}

void split_weights(const float *A, const float *B, int L, int pieces, bool transpose, __bf16 *out, int *bad,
                   hipStream_t s)
{
    const dim3 g((unsigned)nb((size_t)L * 2 * H * H, kThreads));
    if (pieces == 3) hipLaunchKernelGGL(k_split_weights<3>, g, dim3(kThreads), 0, s, A, B, L, transpose, out, bad);
    else hipLaunchKernelGGL(k_split_weights<1>, g, dim3(kThreads), 0, s, A, B, L, transpose, out, bad);
}

void dense(const Product &p1, const Product &p2, bool transpose, const float *bias, int N, int mode,
           const float *Hres, float *Z, float *out, int pieces, hipStream_t s)
{
    const dim3 g(nb(N, TR)), b(kThreads);
    if (pieces == 3) hipLaunchKernelGGL(k_dense<3>, g, b, 0, s, p1, p2, transpose, bias, N, mode, Hres, Z, out);
    else hipLaunchKernelGGL(k_dense<1>, g, b, 0, s, p1, p2, transpose, bias, N, mode, Hres, Z, out);
}

size_t grad_floats(int N)
{
    const size_t w = (size_t)nb(N, grad_rows(N)) * kGradOut, e = (size_t)nb(N, edge_rows(N)) * ((kIn + 1) * H);
    static_assert(kOut * H + kOut <= (kIn + 1) * H, "the input layer's partials are the larger");
    return w > e ? w : e;
}

void wgrad(const float *A, const float *B, const float *D, int N, float *part, float *gA, float *gB, float *gc,
           hipStream_t s)
{
    const int rows = grad_rows(N), np = nb(N, rows);
    hipLaunchKernelGGL(k_wgrad_part, dim3(np), dim3(kGradThreads), 0, s, A, B, D, N, rows, part);
    hipLaunchKernelGGL(k_sum_parts, dim3(nb(kGradOut, 64)), dim3(kThreads), 0, s, part, np, kGradOut, H * H, H * H, gA,
                       gB, gc);
}

void input_grad(const float *X, const float *D, int N, float *part, float *gW0, float *gb0, hipStream_t s)
{
    const int rows = edge_rows(N), np = nb(N, rows), n = (kIn + 1) * H;
    hipLaunchKernelGGL((k_edge_grad_part<kIn, 0>), dim3(np), dim3(kThreads), 0, s, D, X, N, rows, part);
    hipLaunchKernelGGL(k_sum_parts, dim3(nb(n, 64)), dim3(kThreads), 0, s, part, np, n, kIn * H, H, gW0, gb0, gb0);
}

void output_grad(const float *h, const float *dy, int N, float *part, float *gWo, float *gbo, hipStream_t s)
{
    const int rows = edge_rows(N), np = nb(N, rows), n = kOut * H + kOut;
    hipLaunchKernelGGL((k_edge_grad_part<kOut, 1>), dim3(np), dim3(kThreads), 0, s, h, dy, N, rows, part);
    hipLaunchKernelGGL(k_sum_parts, dim3(nb(n, 64)), dim3(kThreads), 0, s, part, np, n, kOut * H, kOut, gWo, gbo, gbo);
}

void neighbour_mean(const int *nbr, int W, int N, const float *invDeg, const float *h, float *m, hipStream_t s)
{
    hipLaunchKernelGGL(k_neighbour<false>, dim3(nb((size_t)N * (H / 4), kThreads)), dim3(kThreads), 0, s, nbr, W, N,
                       invDeg, h, m);
}

void neighbour_mean_transpose_add(const int *nbr, int W, int N, const float *invDeg, const float *dm, float *dh,
                                  hipStream_t s)
{
    hipLaunchKernelGGL(k_neighbour<true>, dim3(nb((size_t)N * (H / 4), kThreads)), dim3(kThreads), 0, s, nbr, W, N,
                       invDeg, dm, dh);
}

void relu_back(const float *dh, const float *z, size_t n, float *dz, hipStream_t s)
{
    hipLaunchKernelGGL(k_relu_back, dim3(nb((n + 3) / 4, kThreads)), dim3(kThreads), 0, s, dh, z, n, dz);
}

void add(float *a, const float *b, size_t n, hipStream_t s)
{
    hipLaunchKernelGGL(k_add, dim3(nb(n, kThreads)), dim3(kThreads), 0, s, a, b, n);
}

void out_layer(const float *h, const float *Wo, const float *bo, int N, float *y, hipStream_t s)
{
    hipLaunchKernelGGL(k_out, dim3(nb((size_t)N, kThreads)), dim3(kThreads), 0, s, h, Wo, bo, N, y);
}

void out_layer_back(const float *dy, const float *Wo, int N, float *dh, hipStream_t s)
{
    hipLaunchKernelGGL(k_out_back, dim3(nb((size_t)N * H, kThreads)), dim3(kThreads), 0, s, dy, Wo, N, dh);
}

int loss_parts(int n) { return nb(n, kThreads); }

void loss(const float *y, const float *t, int n, float *dy, double *part, double *out, hipStream_t s)
{
    const int np = loss_parts(n);
    hipLaunchKernelGGL(k_loss, dim3(np), dim3(kThreads), 0, s, y, t, n, 1.f / (float)n, dy, part);
    hipLaunchKernelGGL(k_loss_final, dim3(1), dim3(kThreads), 0, s, part, np, 1.0 / (double)n, out);
}

void adam(float *p, const float *g, float *m, float *v, int n, float lr, int step, hipStream_t s)
{
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3(nb(n, kThreads)), dim3(kThreads), 0, s, p, g, m, v, n, lr, b1, b2, c1, c2, 1e-8f);
}

}  // namespace nn
}  // namespace phl
