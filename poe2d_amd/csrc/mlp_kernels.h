// Launchers of the surrogate network's kernels (mlp_kernels.hip) and the bf16 helpers they share
// with the host code.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>

namespace poe2d {
namespace mlp {

// bf16 bits of x, round to nearest even (NaN stays NaN).
__host__ __device__ inline uint16_t bf16_rne(float x)
{
    uint32_t u;
    __builtin_memcpy(&u, &x, 4);
    if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu)) return (uint16_t)((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__host__ __device__ inline float bf16_to_f32(uint16_t h)
{
    const uint32_t u = (uint32_t)h << 16;
    float f;
    __builtin_memcpy(&f, &u, 4);
    return f;
}

// EPI_MSE: instead of the output, the mean-squared-error gradient of output (product + bias)
// against a target, bf16, row-major and transposed, with per-block sums of squared errors.
// EPI_ADAM: the product is a weight gradient; the epilogue takes the Adam step of those master
// weights and writes their bf16 copy and its transpose.
enum { EPI_LINEAR = 0, EPI_GELU = 1, EPI_PARTIAL = 2, EPI_MSE = 3, EPI_ADAM = 4 };

// Where a GEMM's results go: bias added first (when given); `pre` receives the value before the
// activation; f32 / b16 the value after it.  Any pointer may be null.
struct GemmOut {
    float *f32 = nullptr;
    int ldf = 0;
    uint16_t *b16 = nullptr;
    int ldb = 0;
    float *pre = nullptr;
    int ldp = 0;
    const float *bias = nullptr;
    // EPI_MSE: g[m][n] = bf16(scale (out - tgt)), gt[n][m] its transpose, partial[block] = the
    // block's sum of (out - tgt)^2, dbp[tile row][n] = the sum of g over the tile's rows (lddb
    // apart; output_bias_step adds them up).  Target row m is tgt row m, or row
    // tgt_rows[m] when tgt_rows is given (a batch read in place from a dataset).
    const float *tgt = nullptr;
    int ldt = 0;
    const int *tgt_rows = nullptr;
    float scale = 0.f;
    uint16_t *g = nullptr, *gt = nullptr;
    int ldg = 0, ldgt = 0;
    float *partial = nullptr;
    float *dbp = nullptr;
    int lddb = 0;
    // EPI_ADAM: master weights w (leading dimension ldw; the product's [m][n] is weight [m][n]), Adam
    // moments, the step's constants, the bf16 copy w16 (ldw) and its transpose w16t (ld16t)
    float *w = nullptr, *mom = nullptr, *vel = nullptr;
    int ldw = 0;
    float lr = 0.f, b1 = 0.f, b2 = 0.f, eps = 0.f, c1 = 1.f, c2 = 1.f;
    uint16_t *w16 = nullptr, *w16t = nullptr;
    int ld16t = 0;
};

// C = A B^T (M x N, reduction over K), A [M][lda] and B [N][ldb] bf16 with K contiguous; K and the
// leading dimensions multiples of 32 / 8.  epi: EPI_LINEAR, EPI_GELU, EPI_MSE (partial holds one
// entry per 128 x 128 tile) or EPI_ADAM.  ksplit > 1 splits K over blocks into `work` (ksplit * M *
// N floats) and reduces (EPI_LINEAR and EPI_GELU only).
hipError_t gemm_bf16(const uint16_t *A, int lda, const uint16_t *B, int ldb, int M, int N, int K, int epi,
                     const GemmOut &out, float *work, size_t work_floats, int ksplit, hipStream_t stream);

// A hidden layer gelu(A B^T + bias) into b16 (and before the activation into pre when given): of one
// member (B, bias), or of several at once, member z's A + z stride_a (0: shared), bs[z] and biases[z] into
// b16 + z stride_b16.  Values equal gemm_bf16's with EPI_GELU and the same ksplit > 1.  K a multiple of 64.
hipError_t hidden_layer(const uint16_t *A, int lda, size_t stride_a, const uint16_t *B, const uint16_t *const *bs, int ldb,
                        const float *bias, const float *const *biases, int members, int M, int N, int K, int ksplit, float *pre,
                        int ldp, uint16_t *b16, int ldb16, size_t stride_b16, hipStream_t stream);
// Whether that is the faster way (gemm_bf16 the other).
bool hidden_in_registers(int members, int M, int N, int K);

// The members' output layer (A + z stride_a times bs[z]^T + biases[z]) and its statistics: mean over
// members times scale (either may be null) into mean [M][ldm], and spread[m] = ||standard deviation over
// members|| / ||unscaled mean|| over the row (null: not formed; part holds ensemble_part_doubles).
size_t ensemble_part_doubles(int M, int N);
hipError_t ensemble_output(const uint16_t *A, int lda, size_t stride_a, const uint16_t *const *bs, int ldb,
                           const float *const *biases, int members, int M, int N, int K, float *mean, size_t ldm,
                           const float *scale, double *part, float *spread, hipStream_t stream);

// The partial products of a GEMM split over ksplit ranges of K, part [ksplit][M][N] floats, not summed.
hipError_t gemm_partials(const uint16_t *A, int lda, const uint16_t *B, int ldb, int M, int N, int K, float *part,
                         size_t part_floats, int ksplit, hipStream_t stream);

// out[c][r] = in[r][c], R x C, for n matrices (kTransposes to a launch).
struct Transpose {
    const uint16_t *in;
    uint16_t *out;
    int ldi, ldo, R, C;
};
constexpr int kTransposes = 8;
struct TransposeList {
    Transpose m[kTransposes];
};
hipError_t transpose_bf16(const Transpose *m, int n, hipStream_t stream);

// An activation's gradient g = dh * gelu'(pre) (bf16, M x N, leading dimension ldg; pre: ld) and its
// transpose gt [N][ldgt], dh the sum of gemm_partials' nsplit partials.
hipError_t hidden_gradients(const float *part, int nsplit, const float *pre, int ld, int M, int N, uint16_t *g, int ldg,
                            uint16_t *gt, int ldgt, hipStream_t stream);

// Mean squared error over M x N: gradient 2 (y - t) / (M N) as bf16 into g and its transpose gt
// ([N][ldgt]), its column sums (the bias gradient) into db[N], and per-block sums of squares into
// partial[mse_blocks(N)].
int mse_blocks(int N);
// Entries of `partial` the EPI_MSE product writes for an M x N output.
inline int gemm_tiles(int M, int N) { return ((M + 127) / 128) * ((N + 127) / 128); }
hipError_t mse(const float *y, int ldy, const float *t, int ldt, int M, int N, uint16_t *g, int ldg, uint16_t *gt,
               int ldgt, float *db, float *partial, hipStream_t stream);

// Adam step t (1-based) of the output bias b[N], its gradient the sum over r < rows of part[r * ld + n]
// (EPI_MSE's dbp).
hipError_t output_bias_step(const float *part, int rows, int ld, int N, float *b, float *mom, float *vel, float lr, float b1,
                            float b2, float eps, long long t, hipStream_t stream);

// db[r] = sum_k gt[r][k] over the K = batch entries of the transposed gradient gt [R][ldgt].
hipError_t bias_gradient(const uint16_t *gt, int ldgt, int R, int K, float *db, hipStream_t stream);

// Adam step t of a layer: its R x C weights (R a multiple of 32, C of 64) from the sum of gemm_partials'
// nsplit partials, refreshing their bf16 copy w16 and the transposed copy w16t [C][R], and its bias from
// the sums over the K = batch entries of the transposed gradient gt [R][ldgt].
hipError_t adam_layer_step(float *w, float *m, float *v, const float *part, int nsplit, int R, int C, float lr, float b1,
                           float b2, float eps, long long t, uint16_t *w16, uint16_t *w16t, const uint16_t *gt, int ldgt, int K,
                           float *b, float *bm, float *bv, hipStream_t stream);

hipError_t convert_bf16(const float *in, uint16_t *out, size_t n, hipStream_t stream);

}  // namespace mlp
}  // namespace poe2d
