// Kernels of the surrogate network: a BF16 GEMM on the matrix cores (FP32 accumulation) with a
// fused bias / GELU epilogue and split-K, transposes, GELU backward, bias gradients, the MSE
// gradient and the Adam update.
//
// GEMM layout ("NT"): C[m][n] = sum_k A[m][k] B[n][k], both operands K-contiguous bf16 rows.  A
// block of 256 threads (4 waves, 2 x 2) owns a 128 x 128 tile of C; each wave computes 64 x 64
// with 2 x 2 v_mfma_f32_32x32x16_bf16.  Operand tiles of 128 rows x 32 k go through LDS, double
// buffered, one barrier per k tile; loads run two to four k tiles ahead of the MFMAs, through
// register sets sized so that every variant runs three waves per SIMD without spilling.  MFMA lane
// layout (gfx950, 32x32x16 bf16): lane l supplies
// row l % 32 of A and column l % 32 of B with 8 k values (the same 8 for both; here k = (l / 32) * 8
// + j of the 16-wide k step), and element i of its 16 results is C[(i / 4) * 8 + (l / 32) * 4 + i % 4]
// [l % 32].
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "mlp_kernels.h"
#include "mlp_plan.h"

namespace poe2d {
namespace mlp {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

constexpr int BM = 128, BN = 128, BK = 32;
constexpr int LDS_ROW = BK + 8;  // bf16 per LDS row (16-byte pad against bank conflicts)
// The shape of ensemble_output's tiles: the one with the least work per CU, tiles per block slot (counted
// two a CU of the 64 x 64 and 128 x 128, one of the 256 x 128; less than one slot each costs a whole
// tile) times a tile's cost relative to 64 x 64.  Larger tiles read their operands less often, but pad
// more rows and fill the chip later.  Measured, us per pass, five members of 512 hidden, rows x outputs:
//                 64 x 64   128 x 128   256 x 128
//   37 x 6300         100         121
//   130 x 20000       140         157         153
//   300 x 20000       193         174         219
//   130 x 75750       286         292         276
//   300 x 151500      949 *       636         743
//   1024 x 6300       267         252         245
//   2048 x 151500    4960 *      3000        2614      (* operands carried through registers)
constexpr int kCus = 256;
constexpr float kCostSquare = 3.0f, kCostTall = 2.7f;

// Hidden layers with at most this many inputs per member form their sums one after the other in a block;
// with more, the chain costs more than partials in memory unless the tiles fill the chip.  us per
// prediction, in registers / split (member by member): one member, 37 rows of 2000 inputs 92 / 103, 4000
// 110 / 112, 16000 214 / 193, 256 rows of 4000 245 / 258, 16000 619 / 600; five members, 37 rows of 4000
// 121 / 181, 16000 224 / 283.
constexpr int kHiddenChain = 4096;

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

__device__ __forceinline__ float gelu_grad(float x)
{
    const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}

// One Adam update of weight i (bias-corrected: c1 = 1 - b1^t, c2 = 1 - b2^t) from its gradient g.
__device__ __forceinline__ float adam_value(float w, float &m, float &v, float g, float lr, float b1, float b2,
                                            float eps, float c1, float c2)
{
    m = b1 * m + (1.f - b1) * g;
    v = b2 * v + (1.f - b2) * g * g;
    return w - lr * (m / c1) / (sqrtf(v / c2) + eps);
}

__device__ __forceinline__ float adam_update(float *w, float *mom, float *vel, float g, size_t i, float lr, float b1,
                                             float b2, float eps, float c1, float c2)
{
    float m = mom[i], v = vel[i];
    const float x = adam_value(w[i], m, v, g, lr, b1, b2, eps, c1, c2);
    mom[i] = m;
    vel[i] = v;
    w[i] = x;
    return x;
}

// C (+)= A B^T over k in [k0, k1) for the 128 x 128 tile (tm, tn); k0, k1 multiples of BK.
template <int EPI>
__global__ void __launch_bounds__(256, 3) gemm_nt(const uint16_t *__restrict__ A, int lda, const uint16_t *__restrict__ B,
                                               int ldb, int M, int N, int K, int ksplit, GemmOut out)
{
    // operand tiles (la, lb: two k tiles each), reused by the EPI_MSE / EPI_ADAM epilogues for the
    // transposed bf16 tile and the EPI_MSE sums (40 KiB)
    __shared__ uint16_t lds[2 * BM * LDS_ROW + 2 * BN * LDS_ROW];
    uint16_t(*la)[BM * LDS_ROW] = (uint16_t(*)[BM * LDS_ROW])lds;
    uint16_t(*lb)[BN * LDS_ROW] = (uint16_t(*)[BN * LDS_ROW])(lds + 2 * BM * LDS_ROW);
    // Tile order.  Row-major outputs: block b takes tile b, n fastest, so the blocks in flight write
    // long runs of the same rows.  EPI_MSE and split-K: blocks go to the 8 XCDs round-robin (block
    // b, counted x fastest, to XCD b % 8), and XCD x takes the x-th run of consecutive items
    // instead.  EPI_MSE walks m fastest, so the m tiles of one n tile follow each other on one XCD:
    // they share its operand tile in that XCD's L2 and finish the rows of the transposed gradient
    // together (225 -> 200 us on the 256 x 151552 x 512 output layer; the same order slowed the
    // plain epilogue from 89 to 104 us).  Split-K walks the tiles of one k range first, so every
    // tile of a k range runs on one XCD and each operand slice is read from HBM once.
    const int tiles_n = (N + BN - 1) / BN;
    int tm, tn, split = 0;
    if constexpr (EPI == EPI_MSE || EPI == EPI_PARTIAL) {
        const int nb = (int)(gridDim.x * gridDim.y), q8 = nb >> 3, r8 = nb & 7;
        const int b = (int)(blockIdx.y * gridDim.x + blockIdx.x);
        const int xcd = b & 7, slot = b >> 3;
        const int item = xcd < r8 ? xcd * (q8 + 1) + slot : r8 * (q8 + 1) + (xcd - r8) * q8 + slot;
        const int tile = item % (int)gridDim.x;
        if (EPI == EPI_PARTIAL) split = item / (int)gridDim.x;
        const int tiles_m = (M + BM - 1) / BM;
        tm = EPI == EPI_MSE ? tile % tiles_m : tile / tiles_n;
        tn = EPI == EPI_MSE ? tile / tiles_m : tile % tiles_n;
    } else {
        tm = (int)blockIdx.x / tiles_n;
        tn = (int)blockIdx.x % tiles_n;
    }
    const int kper = ((K / BK + ksplit - 1) / ksplit) * BK;
    const int k0 = split * kper, k1 = min(K, k0 + kper);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    // the bias of this lane's two result columns (wn * 64 + j * 32 + lane % 32)
    float bj[2];
    for (int j = 0; j < 2; ++j) {
        const int n = tn * BN + wn * 64 + j * 32 + (lane & 31);
        bj[j] = (EPI != EPI_PARTIAL && EPI != EPI_ADAM && out.bias && n < N) ? out.bias[n] : 0.f;
    }

    // each thread loads 2 x 16 bytes of each operand tile: rows r0 and r0 + 64, k chunk kc * 8
    const int r0 = t >> 2, kc = t & 3;
    // Loads are unconditional (rows past the edge read the last row, and are zeroed when stored to
    // LDS), so every path keeps the same number of loads in flight and the waits before the LDS
    // stores can leave the younger set's loads outstanding.
    bool a_ok[2], b_ok[2];
    for (int h = 0; h < 2; ++h) {
        a_ok[h] = tm * BM + r0 + h * 64 < M;
        b_ok[h] = tn * BN + r0 + h * 64 < N;
    }
    auto load_tile = [&](const uint16_t *P, int ld, int rows, int row0, int k, u16x8 *v) {
        for (int h = 0; h < 2; ++h) {
            const int r = min(row0 + r0 + h * 64, rows - 1);
            v[h] = *(const u16x8 *)(P + (size_t)r * ld + k + kc * 8);
        }
    };
    auto store_tile = [&](uint16_t *L, const u16x8 *v, const bool *ok) {
        for (int h = 0; h < 2; ++h)
            *(u16x8 *)(L + (r0 + h * 64) * LDS_ROW + kc * 8) = ok[h] ? v[h] : u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    };

    f32x16 acc[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j)
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    // PF register sets carry operand tiles from memory: tile i lives in set i % PF, loaded at the
    // start of k step i - PF and stored to LDS at the end of step i - 1, so each load has about PF - 1
    // steps of MFMA work to land.  As many sets as fit beside each epilogue at three waves per SIMD
    // (168 registers) without spilling.
    constexpr int PF = (EPI == EPI_ADAM || EPI == EPI_MSE) ? 2 : EPI == EPI_PARTIAL ? 4 : 3;
    u16x8 ra[PF][2], rb[PF][2];
    const int nk = k1 > k0 ? (k1 - k0) / BK : 0;
    auto compute = [&](const uint16_t *LA, const uint16_t *LB) {
#pragma unroll
        for (int kk = 0; kk < BK; kk += 16) {
            bf16x8 fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int ra = wm * 64 + i * 32 + (lane & 31);
                const int rb = wn * 64 + i * 32 + (lane & 31);
                fa[i] = *(const bf16x8 *)(LA + ra * LDS_ROW + kk + (lane >> 5) * 8);
                fb[i] = *(const bf16x8 *)(LB + rb * LDS_ROW + kk + (lane >> 5) * 8);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
    };
    const int last = k0 + (nk - 1) * BK;  // tiles past the end re-read the last one (never used)
    auto kof = [&](int i) { return min(k0 + i * BK, last); };
    if (nk > 0) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            load_tile(A, lda, M, tm * BM, kof(u), ra[u]);
            load_tile(B, ldb, N, tn * BN, kof(u), rb[u]);
        }
        store_tile(la[0], ra[0], a_ok);
        store_tile(lb[0], rb[0], b_ok);
    }
    __syncthreads();
    for (int it0 = 0; it0 < nk; it0 += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int it = it0 + u;
            if (it < nk) {
                // LDS buffer it & 1 holds tile it, so set u is free: refill it with tile it + PF
                load_tile(A, lda, M, tm * BM, kof(it + PF), ra[u]);
                load_tile(B, ldb, N, tn * BN, kof(it + PF), rb[u]);
                compute(la[it & 1], lb[it & 1]);
                if (it + 1 < nk) {
                    store_tile(la[(it + 1) & 1], ra[(u + 1) % PF], a_ok);
                    store_tile(lb[(it + 1) & 1], rb[(u + 1) % PF], b_ok);
                }
                __syncthreads();
            }
        }
    }

    if constexpr (EPI == EPI_MSE || EPI == EPI_ADAM) {
        // bf16 results of the tile go to memory row-major (g, or the updated weights' copy w16) and,
        // through a transposed tile in LDS, column-major (gt, or w16t) in 256-byte rows
        constexpr int TP = BM + 8;  // bf16 per transposed row
        uint16_t *tt = lds;
        float lsum = 0.f;
        __syncthreads();  // every wave is done with the operand tiles
        // Per 32 x 32 sub-tile: every operand load is issued before any store (the compiler cannot
        // tell the arrays apart and would otherwise hold each load behind the store before it).
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int nl = wn * 64 + j * 32 + (lane & 31), n = tn * BN + nl;
                auto row = [&](int e) { return wm * 64 + i * 32 + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3); };
                float va[16], vb[16], vc[16];
                if constexpr (EPI == EPI_MSE) {
                    // target rows: the batch's own, or looked up four at a time (the lane's rows come in
                    // runs of four, all below M or none: M % 4 == 0 with tgt_rows), lookups first
                    int tr[16];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int mg = tm * BM + row(4 * q);
                        if (out.tgt_rows) {
                            const int4 r4 = mg < M ? *(const int4 *)(out.tgt_rows + mg) : make_int4(0, 0, 0, 0);
                            tr[4 * q] = r4.x;
                            tr[4 * q + 1] = r4.y;
                            tr[4 * q + 2] = r4.z;
                            tr[4 * q + 3] = r4.w;
                        } else {
#pragma unroll
                            for (int u = 0; u < 4; ++u) tr[4 * q + u] = mg + u;
                        }
                    }
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        va[e] = (tm * BM + row(e) < M && n < N) ? out.tgt[(size_t)tr[e] * out.ldt + n] : 0.f;
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int m = tm * BM + row(e);
                    const bool ok = m < M && n < N;
                    if constexpr (EPI == EPI_ADAM) {
                        // the optimiser state streams through once per step: non-temporal
                        const size_t idx = (size_t)m * out.ldw + n;
                        va[e] = ok ? __builtin_nontemporal_load(out.w + idx) : 0.f;
                        vb[e] = ok ? __builtin_nontemporal_load(out.mom + idx) : 0.f;
                        vc[e] = ok ? __builtin_nontemporal_load(out.vel + idx) : 0.f;
                    }
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int ml = row(e), m = tm * BM + ml;
                    uint16_t h = 0;
                    if (m < M && n < N) {
                        if constexpr (EPI == EPI_MSE) {
                            // the output (product + bias) minus its target: loss and bf16 gradient
                            const float d = (acc[i][j][e] + bj[j]) - va[e];
                            lsum += d * d;
                            h = bf16_rne(out.scale * d);
                        } else {
                            // the product is this weight's gradient: Adam on the master weight
                            const size_t idx = (size_t)m * out.ldw + n;
                            float mo = vb[e], ve = vc[e];
                            const float x = adam_value(va[e], mo, ve, acc[i][j][e], out.lr, out.b1, out.b2, out.eps,
                                                       out.c1, out.c2);
                            __builtin_nontemporal_store(mo, out.mom + idx);
                            __builtin_nontemporal_store(ve, out.vel + idx);
                            __builtin_nontemporal_store(x, out.w + idx);
                            h = bf16_rne(x);
                        }
                    }
                    tt[nl * TP + ml] = h;
                }
            }
        __syncthreads();
        {
            const int nl = t >> 1, mh = (t & 1) * 64, n = tn * BN + nl;
            uint16_t *dst = EPI == EPI_MSE ? out.gt : out.w16t;
            const size_t ld = EPI == EPI_MSE ? (size_t)out.ldgt : (size_t)out.ld16t;
            if (n < N)
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const int m0 = tm * BM + mh + q * 8;
                    const uint16_t *src = tt + nl * TP + mh + q * 8;
                    if (m0 + 8 <= M) {
                        *(u16x8 *)(dst + (size_t)n * ld + m0) = *(const u16x8 *)src;
                    } else {
                        for (int r = 0; r < 8 && m0 + r < M; ++r) dst[(size_t)n * ld + m0 + r] = src[r];
                    }
                }
        }
        {
            // row-major from the same tile (g, or w16): thread t writes row t / 2, columns
            // (t & 1) * 64 .. + 63, in 16-byte pieces
            const int ml = t >> 1, nh = (t & 1) * 64, m = tm * BM + ml;
            uint16_t *dst = EPI == EPI_MSE ? out.g : out.w16;
            const size_t ld = EPI == EPI_MSE ? (size_t)out.ldg : (size_t)out.ldw;
            if (m < M)
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const int nl0 = nh + q * 8, n0 = tn * BN + nl0;
                    u16x8 v;
#pragma unroll
                    for (int r = 0; r < 8; ++r) v[r] = tt[(nl0 + r) * TP + ml];
                    if (n0 + 8 <= N) {
                        *(u16x8 *)(dst + (size_t)m * ld + n0) = v;
                    } else {
                        for (int r = 0; r < 8 && n0 + r < N; ++r) dst[(size_t)m * ld + n0 + r] = v[r];
                    }
                }
        }
        if constexpr (EPI == EPI_MSE) {
            // the bias gradient's partial sum over this tile's rows, per column, from the bf16
            // gradients in the transposed tile (fixed order: two halves of 64 rows, then the pair),
            // and the block's sum of squared errors (per wave by shuffles, then the four waves)
            const int nl = t >> 1, mh = (t & 1) * 64;
            float cs = 0.f;
            for (int q = 0; q < 64; ++q) cs += bf16_to_f32(tt[nl * TP + mh + q]);
            for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o);
            float *red = (float *)(lds + BN * TP);  // past the transposed tile
            red[t] = cs;
            if (lane == 0) red[256 + wave] = lsum;
            __syncthreads();
            const int n = tn * BN + nl;
            if ((t & 1) == 0 && n < N) out.dbp[(size_t)tm * out.lddb + n] = red[t] + red[t + 1];
            if (t == 0) out.partial[blockIdx.x] = (red[256] + red[257]) + (red[258] + red[259]);
        }
        return;
    }

    // epilogue: full tiles store without per-element bounds checks; the bias sits in registers
    // (loaded before the k loop), so no global load is pending here and the stores need no waits
    const bool full = (tm + 1) * BM <= M && (tn + 1) * BN <= N;
    auto emit = [&](int m, int n, float v, float b) {
        if (EPI == EPI_PARTIAL) {
            out.f32[(size_t)split * M * out.ldf + (size_t)m * out.ldf + n] = v;
            return;
        }
        v += b;
        if (out.pre) out.pre[(size_t)m * out.ldp + n] = v;
        if (EPI == EPI_GELU) v = gelu(v);
        if (out.f32) out.f32[(size_t)m * out.ldf + n] = v;
        if (out.b16) out.b16[(size_t)m * out.ldb + n] = bf16_rne(v);
    };
    if (full) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int n = tn * BN + wn * 64 + j * 32 + (lane & 31);
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    emit(tm * BM + wm * 64 + i * 32 + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3), n, acc[i][j][e], bj[j]);
            }
    } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int n = tn * BN + wn * 64 + j * 32 + (lane & 31);
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int m = tm * BM + wm * 64 + i * 32 + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3);
                    if (m < M && n < N) emit(m, n, acc[i][j][e], bj[j]);
                }
            }
    }
}

// Products over tiles of 64 k values.  A block of WM x WN waves, each with MI x NJ results of 32 x 32, owns
// the tile (tm, tn) of C = A B^T (M x N); its operand tiles reach LDS by direct loads, STAGES of them in
// the ring, so no register carries them and STAGES - 1 are in flight.  A wave's direct load writes 1 KiB
// of consecutive LDS, so rows are unpadded; the 16-byte chunks of a row are exchanged by its row bits
// instead, which spreads the sixteen rows that a phase of a fragment read touches over all 64 banks (by
// the low row bits alone, two rows met in each: 45 % of the LDS cycles, 3 % of the time of a large product).
//
// The ring (ring_elems long) is the kernel's only LDS array, what else the kernel keeps there behind it: of
// several arrays, or with its end out of the compiler's sight, the compiler holds every read until all
// direct loads in flight have landed.  The waits for the tile that is read are written out here.
//
// at(pa, pb) gives the addresses of A's and B's next k tile (the first 64 values of the block's first
// rows), next() moves on to the one after; they run STAGES - 1 tiles ahead, past the last step too (any
// readable tile does).  after(q) follows the matrix instructions of k values 16 q .. of a tile.
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void global_void;
// pointers in memory that no kernel writes: read by scalar loads, which no load in flight delays
typedef __attribute__((address_space(4))) const uint64_t const_u64;

constexpr int RING_K = 64;
constexpr int ring_elems(int tm, int tn, int stages) { return stages * (tm + tn) * RING_K; }

template <int WM, int WN, int MI, int NJ, int STAGES, class At, class Next, class After>
__device__ __forceinline__ void ring_product(uint16_t *ring, int M, int N, int lda, int ldb, int tm, int tn, int steps,
                                             f32x16 (&acc)[MI][NJ], const At &at, const Next &next, const After &after)
{
    static_assert(STAGES >= 2 && STAGES <= 4, "the loop over the steps");
    constexpr int TM = 32 * MI * WM, TN = 32 * NJ * WN, BKL = RING_K;
    constexpr int CH = BKL / 8;                         // 16-byte chunks of a row
    constexpr int RPL = 64 / CH;                        // rows one wave's load covers
    constexpr int LOADS = (TM + TN) / RPL / (WM * WN);  // loads per wave and tile
    constexpr int STAGE = (TM + TN) * BKL;              // bf16 per stage
    uint16_t *const s0 = ring, *const s1 = ring + STAGE, *const s2 = ring + (STAGES > 2 ? 2 : 0) * STAGE,
                   *const s3 = ring + (STAGES - 1) * STAGE;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave / WN, wn = wave % WN;
    // swizzle: chunk c of row r sits at chunk c ^ swz(r)
    auto swz = [](int r) -> int { return (r >> 1 & 3) << 1 | (r >> 3 & 1); };

    // the byte this lane loads, from the tile's first row: load l of the wave covers rows (wave * LOADS +
    // l) * RPL .. of the stage (A's rows, then B's)
    uint32_t off[LOADS];
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
        const int r = (wave * LOADS + l) * RPL + lane / CH, c = (lane % CH) ^ swz(r);
        off[l] = r < TM ? (uint32_t)(min(r, M - 1 - tm * TM) * lda + c * 8) * 2u
                        : (uint32_t)(min(r - TM, N - 1 - tn * TN) * ldb + c * 8) * 2u;
    }
    // the loads first <= l < last of a tile
    auto load = [&](uint16_t *stage, int first, int last) {
        uint64_t pa, pb;
        at(pa, pb);
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {
            if (l < first || l >= last) continue;
            const int r0 = (wave * LOADS + l) * RPL;  // (a load's rows are all A's or all B's)
            __builtin_amdgcn_global_load_lds(
                (global_void *)((__attribute__((address_space(1))) char *)(r0 < TM ? pa : pb) + off[l]),
                (lds_void *)(stage + r0 * BKL), 16, 0, 0);
        }
    };
    load(s0, 0, LOADS), next();
    if constexpr (STAGES > 2) load(s1, 0, LOADS), next();
    if constexpr (STAGES > 3) load(s2, 0, LOADS), next();

    // this lane's fragments: rows ar, ar + 32 of A and br, br + 32 of B, chunk (kk / 8 + lane / 32) ^ swz of
    // k step kk (32 rows on the swizzle is the same), as offsets into a stage
    const int ar = wm * 32 * MI + (lane & 31), br = TM + wn * 32 * NJ + (lane & 31);
    int ao[BKL / 16], bo[BKL / 16];
#pragma unroll
    for (int q = 0; q < BKL / 16; ++q) {
        ao[q] = ar * BKL + ((2 * q + (lane >> 5)) ^ swz(ar)) * 8;
        bo[q] = br * BKL + ((2 * q + (lane >> 5)) ^ swz(br)) * 8;
    }
    // one tile, in stage `from`; the next load goes to `to`, the stage of the tile before
    auto step = [&](const uint16_t *from, uint16_t *to) {
        // the tile has landed when no more than the STAGES - 2 tiles after it are in flight; past the
        // barrier that holds for every wave, and every wave is done with the tile before
        constexpr int PENDING = LOADS * (STAGES - 2);
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(PENDING) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        bf16x8 fa[2][MI], fb[2][NJ];  // the fragments of k step q and the next
        auto read = [&](int q) {
#pragma unroll
            for (int i = 0; i < MI; ++i) fa[q & 1][i] = *(const bf16x8 *)(from + ao[q] + i * 32 * BKL);
#pragma unroll
            for (int j = 0; j < NJ; ++j) fb[q & 1][j] = *(const bf16x8 *)(from + bo[q] + j * 32 * BKL);
        };
        read(0);
#pragma unroll
        for (int q = 0; q < BKL / 16; ++q) {
            if (q + 1 < BKL / 16) read(q + 1);
            load(to, q * LOADS / (BKL / 16), (q + 1) * LOADS / (BKL / 16));
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[q & 1][i], fb[q & 1][j], acc[i][j], 0, 0, 0);
            if (q + 1 == BKL / 16) next();
            after(q);
        }
        // (this wave's reads of the tile are done before it reaches the next barrier)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    // (left from the middle: an edge back from there would have the first step wait for all loads)
    for (int g = 0;;) {
        step(s0, s3);
        if (++g == steps) break;
        step(s1, s0);
        if (++g == steps) break;
        if constexpr (STAGES > 2) {
            step(s2, s1);
            if (++g == steps) break;
        }
        if constexpr (STAGES > 3) {
            step(s3, s2);
            if (++g == steps) break;
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the re-reads, before a stage is used again
    __syncthreads();
}

// Welford's update by member e's outputs.  The accumulators hold the outputs' differences from the
// running mean: they start at bias - mean (the first at the bias) instead of 0, which saves the sum
// and the difference, two operations of six; b is the next member's bias (per column).
template <int MI, int NJ>
__device__ __forceinline__ void welford_update(f32x16 (&acc)[MI][NJ], f32x16 (&mu)[MI][NJ], f32x16 (&m2)[MI][NJ], int e,
                                               const float (&b)[NJ])
{
    const float rcount = 1.0f / (float)(e + 1), weight = (float)e / (float)(e + 1);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const float d = acc[i][j][q];
                mu[i][j][q] = __builtin_fmaf(d, rcount, mu[i][j][q]);
                m2[i][j][q] = __builtin_fmaf(d * weight, d, m2[i][j][q]);
                acc[i][j][q] = b[j] - mu[i][j][q];
            }
}

// Stores a wave's means (scaled) and its row sums of the squared deviations and squared means into
// red[wn][row][0 / 1].  Lane l's 16 results of a 32 x 32 tile are rows (q / 4) * 8 + (l / 32) * 4 + q % 4
// of column l % 32.
template <int MI, int NJ, int ROWS>
__device__ __forceinline__ void ensemble_store(const f32x16 (&mu)[MI][NJ], const f32x16 (&m2)[MI][NJ], int m0, int n0, int wm,
                                               int wn, int M, int N, float *__restrict__ mean, size_t ldm,
                                               const float *__restrict__ scale, bool sums, double (*red)[ROWS][2])
{
    const int lane = threadIdx.x & 63;
    const bool full = m0 + ROWS <= M && n0 + 64 * NJ <= N;  // (the tile's columns: two waves of 32 NJ)
    bool ok_n[NJ];
    float sc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int n = n0 + wn * 32 * NJ + j * 32 + (lane & 31);
        ok_n[j] = n < N;
        sc[j] = scale && ok_n[j] ? scale[n] : 1.f;
    }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        double sv[16], sn[16];
        if (full) {
            float *const row = mean + (size_t)(m0 + wm * 32 * MI + i * 32 + (lane >> 5) * 4) * ldm + n0 + wn * 32 * NJ + (lane & 31);
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                sv[q] = sn[q] = 0.0;
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const float v = mu[i][j][q];
                    sv[q] += m2[i][j][q];
                    sn[q] += (double)v * v;
                    if (mean) row[((q >> 2) * 8 + (q & 3)) * ldm + j * 32] = v * sc[j];
                }
            }
        } else
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int m = m0 + wm * 32 * MI + i * 32 + (q >> 2) * 8 + (lane >> 5) * 4 + (q & 3);
            sv[q] = sn[q] = 0.0;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int n = n0 + wn * 32 * NJ + j * 32 + (lane & 31);
                if (ok_n[j]) {
                    const float v = mu[i][j][q];
                    sv[q] += m2[i][j][q];
                    sn[q] += (double)v * v;
                    if (mean && m < M) mean[(size_t)m * ldm + n] = v * sc[j];
                }
            }
        }
        if (!sums) continue;
        // sum over the 32 lanes of a half wave: at every step a lane keeps half of its rows, adding
        // its partner's sums of them; lane l ends with row q0, the bits 16, 8, 4 and 2 of l
        int q0 = 0;
        auto halve = [&](auto half) {
            constexpr int cnt = decltype(half)::value, h = 2 * cnt;
            const bool up = lane & h;
#pragma unroll
            for (int q = 0; q < cnt; ++q) {
                const double av = up ? sv[q] : sv[q + cnt], an = up ? sn[q] : sn[q + cnt];
                sv[q] = (up ? sv[q + cnt] : sv[q]) + __shfl_xor(av, h);
                sn[q] = (up ? sn[q + cnt] : sn[q]) + __shfl_xor(an, h);
            }
            if (up) q0 += cnt;
        };
        halve(std::integral_constant<int, 8>{});
        halve(std::integral_constant<int, 4>{});
        halve(std::integral_constant<int, 2>{});
        halve(std::integral_constant<int, 1>{});
        sv[0] += __shfl_xor(sv[0], 1);
        sn[0] += __shfl_xor(sn[0], 1);
        if (!(lane & 1)) {
            const int row = wm * 32 * MI + i * 32 + (q0 >> 2) * 8 + (lane >> 5) * 4 + (q0 & 3);
            red[wn][row][0] = sv[0];
            red[wn][row][1] = sn[0];
        }
    }
}

// The output layer of every ensemble member and their statistics in one pass: tile by tile, member
// e's product H_e W_e^T + b_e is formed in the accumulators and folded into the running mean and sum
// of squared deviations (Welford), both in registers.  Stores the mean (times scale[n] when given)
// and, per row and tile of BN columns, the sums over the tile's columns of the squared deviations and
// of the squared (unscaled) mean: part[(tn * 2 + 0 / 1) * M + m].
//
// What bounds it.  Members one at a time wrote each output array (620 MB of 1024 x 151 500) and read
// it back with mean and deviations: 0.33 ms of product and 0.51 ms of Welford per member, 0.8 ms of
// scaling and row sums, 5.3 ms for five members.  Here the mean is the only array that reaches HBM.
// Results of 64 x 64 a wave take 192 of its 256 registers.  Tile order as EPI_MSE's: m fastest within an
// XCD's run, so the m tiles of one n tile share its weights in that L2.
//
// On 1024 x 151500 x 512 and five members in 256 x 128 tiles 1.19 ms, 670 TFLOP/s (operands through
// registers, 128 x 128 tiles: 2.13): the matrix cores are busy a third of the cycles, the mean's 620 MB
// take 0.2 ms in which nothing else runs (one block per CU), the statistics 0.07, and each of the 8 k
// tiles of a member begins with a barrier and a round trip to LDS.
constexpr int kBiasMembers = 16;  // members whose biases are in LDS at a time

template <int WM, int WN, int MI, int NJ, int STAGES>
__global__ void __launch_bounds__(64 * WM * WN, 2)
    ensemble_tiles(const uint16_t *__restrict__ A, int lda, size_t stride_a, const uint16_t *const *__restrict__ bs, int ldb,
                  const float *const *__restrict__ biases, int M, int N, int K, int members, float *__restrict__ mean,
                  size_t ldm, const float *__restrict__ scale, double *__restrict__ part)
{
    constexpr int TM = 32 * MI * WM, TN = 32 * NJ * WN, THREADS = 64 * WM * WN;
    // behind the ring the biases (read from memory at a member's end, they would wait for every load in
    // flight)
    __shared__ __align__(1024) uint16_t ring[ring_elems(TM, TN, STAGES) + 2 * kBiasMembers * TN];
    float *const lbias = (float *)(ring + ring_elems(TM, TN, STAGES));
    const int tiles_m = (M + TM - 1) / TM;
    const int nb = (int)gridDim.x, q8 = nb >> 3, r8 = nb & 7;
    const int xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3;
    const int tile = xcd < r8 ? xcd * (q8 + 1) + slot : r8 * (q8 + 1) + (xcd - r8) * q8 + slot;
    const int tm = tile % tiles_m, tn = tile / tiles_m;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int nk = K / RING_K;
    const_u64 *const b_at = (const_u64 *)(uintptr_t)bs, *const bias_at = (const_u64 *)(uintptr_t)biases;
    auto fill_biases = [&](int e0) {
        for (int i = t; i < min(members - e0, kBiasMembers) * TN; i += THREADS) {
            const int n = tn * TN + i % TN;
            lbias[i] = n < N ? ((const __attribute__((address_space(1))) float *)bias_at[e0 + i / TN])[n] : 0.f;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    f32x16 acc[MI][NJ], mu[MI][NJ], m2[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) mu[i][j][e] = m2[i][j][e] = 0.f;
    fill_biases(0);
    __syncthreads();
    float b[NJ];
    auto bias_of = [&](int e) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) b[j] = lbias[(e % kBiasMembers) * TN + wn * 32 * NJ + j * 32 + (lane & 31)];
    };
    bias_of(0);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = b[j];

    int ge = 0, gk = 0;  // member and k tile of the next load
    int kt = 0, e = 0;   // k tiles done of member e
    ring_product<WM, WN, MI, NJ, STAGES>(
        ring, M, N, lda, ldb, tm, tn, nk * members, acc,
        [&](uint64_t &pa, uint64_t &pb) {
            pa = (uint64_t)(uintptr_t)(A + ge * stride_a + (size_t)tm * TM * lda + gk * RING_K);
            pb = b_at[ge] + ((size_t)tn * TN * ldb + gk * RING_K) * 2;
        },
        [&] {
            if (++gk == nk) {
                gk = 0;
                if (ge + 1 < members) ++ge;
            }
        },
        [&](int q) {
            if (q + 1 < RING_K / 16 || ++kt < nk) return;
            if ((e + 1) % kBiasMembers == 0 && e + 1 < members) {
                __builtin_amdgcn_s_barrier();  // every wave has read the biases it needs of these
                fill_biases(e + 1);
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            }
            bias_of(e + 1);  // (of no use after the last)
            welford_update<MI, NJ>(acc, mu, m2, e, b);
            kt = 0;
            ++e;
        });
    double(*const red)[TM][2] = (double(*)[TM][2])ring;
    ensemble_store<MI, NJ>(mu, m2, tm * TM, tn * TN, wm, wn, M, N, mean, ldm, scale, part != nullptr, red);
    if (!part) return;
    __syncthreads();
    for (int r = t; r < 2 * TM; r += THREADS) {
        const int row = r % TM, w = r / TM, m = tm * TM + row;
        if (m < M) part[((size_t)tn * 2 + w) * M + m] = red[0][row][w] + red[1][row][w];
    }
}

// A hidden layer of one or several members (blockIdx.y): gelu(A B^T + bias) as bf16 (b16), before the
// activation as FP32 (pre) when given.  The sums over ranges of kper k values are formed one after the
// other and added up in range order, so the values are those of the product split over K (EPI_PARTIAL and
// reduce_splits) without the partials' way through memory and the second launch.  Latency bounds it, the k
// tiles one after the other: five members of 512 x 512 take 8.1 us on 37 rows (10.4 split) and 15.0 us on
// 1024 (40; 19.1 with four stages and two blocks to a CU), one member on 256 rows of a training step 3 us
// less.
__global__ void __launch_bounds__(256, 2)
    hidden_product(const uint16_t *__restrict__ A, int lda, size_t stride_a, const uint16_t *B,
                   const uint16_t *const *__restrict__ bs, int ldb, const float *bias, const float *const *__restrict__ biases,
                   int M, int N, int K, int kper, float *__restrict__ pre, int ldp, uint16_t *__restrict__ b16, int ldb16,
                   size_t stride_b16)
{
    constexpr int T = 64;  // 2 x 2 waves of 32 x 32
    __shared__ __align__(1024) uint16_t ring[ring_elems(T, T, 3)];
    const int tiles_n = (N + T - 1) / T, tm = (int)blockIdx.x / tiles_n, tn = (int)blockIdx.x % tiles_n;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (bs) B = bs[blockIdx.y], bias = biases[blockIdx.y];
    const int n = tn * T + (wave & 1) * 32 + (lane & 31);
    const float b = n < N ? bias[n] : 0.f;
    const uint64_t a0 = (uint64_t)(uintptr_t)(A + blockIdx.y * stride_a + (size_t)tm * T * lda);
    const uint64_t b0 = (uint64_t)(uintptr_t)(B + (size_t)tn * T * ldb);
    f32x16 acc[1][1], sums;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[0][0][e] = sums[e] = 0.f;
    auto flush = [&] {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            sums[e] += acc[0][0][e];
            acc[0][0][e] = 0.f;
        }
    };
    int gk = 0, k = 0, end = kper;
    ring_product<2, 2, 1, 1, 3>(
        ring, M, N, lda, ldb, tm, tn, K / RING_K, acc,
        [&](uint64_t &pa, uint64_t &pb) { pa = a0 + gk * 2, pb = b0 + gk * 2; },
        [&] { gk = min(gk + RING_K, K - RING_K); },
        [&](int) {
            if ((k += 16) < end) return;
            flush();
            end += kper;
        });
    if (k > end - kper) flush();
    const int m0 = tm * T + (wave >> 1) * 32 + (lane >> 5) * 4;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int m = m0 + (e >> 2) * 8 + (e & 3);
        if (m >= M || n >= N) continue;
        const float v = sums[e] + b;
        if (pre) pre[(size_t)m * ldp + n] = v;
        b16[blockIdx.y * stride_b16 + (size_t)m * ldb16 + n] = bf16_rne(gelu(v));
    }
}

// spread[m] = ||standard deviation over members|| / ||mean|| from the sums of `tiles` tiles per row:
// kSpreadRows rows per block, 64 threads a row over the tiles, then over the threads in order.  Latency
// bounds it: 64 rows and 16 threads a row took 40 us on 1024 rows of 1184 tiles (16 blocks on 256 CUs),
// this 14 us.
constexpr int kSpreadRows = 16;

__global__ void __launch_bounds__(1024) ensemble_spread(const double *__restrict__ part, int tiles, int M, int members,
                                                        float *__restrict__ spread)
{
    __shared__ double red[2][64][kSpreadRows];
    const int r = threadIdx.x % kSpreadRows, g = threadIdx.x / kSpreadRows, m = blockIdx.x * kSpreadRows + r;
    double var = 0, nrm = 0;
    if (m < M)
#pragma unroll 4
        for (int t = g; t < tiles; t += 64) {
            var += part[((size_t)t * 2 + 0) * M + m];
            nrm += part[((size_t)t * 2 + 1) * M + m];
        }
    red[0][g][r] = var;
    red[1][g][r] = nrm;
    __syncthreads();
    if (g || m >= M) return;
    for (int k = 1; k < 64; ++k) {
        var += red[0][k][r];
        nrm += red[1][k][r];
    }
    spread[m] = (float)(sqrt(var / (members > 1 ? members - 1 : 1)) / fmax(sqrt(nrm), 1e-30));
}

// out[m][n] = sum over splits of part[s][m][n] (+ bias), then as the GEMM epilogue.
__global__ void reduce_splits(const float *__restrict__ part, int nsplit, int M, int N, int ldf, GemmOut out, int gelu_on)
{
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i >= (size_t)M * N) return;
    const int m = (int)(i / N), n = (int)(i % N);
    // eight partials in flight at a time, summed in split order
    const float *p = part + (size_t)m * ldf + n;
    const size_t stride = (size_t)M * ldf;
    float v = 0.f;
    int s = 0;
    for (; s + 8 <= nsplit; s += 8) {
        float q[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) q[u] = p[(size_t)(s + u) * stride];
#pragma unroll
        for (int u = 0; u < 8; ++u) v += q[u];
    }
    for (; s < nsplit; ++s) v += p[(size_t)s * stride];
    if (out.bias) v += out.bias[n];
    if (out.pre) out.pre[(size_t)m * out.ldp + n] = v;
    if (gelu_on) v = gelu(v);
    if (out.f32) out.f32[(size_t)m * out.ldf + n] = v;
    if (out.b16) out.b16[(size_t)m * out.ldb + n] = bf16_rne(v);
}

// out[c][r] = in[r][c] for the R x C bf16 matrices of a list (blockIdx.z), 32 x 32 tiles.
__global__ void transpose16(const TransposeList list)
{
    __shared__ uint16_t tile[32][33];
    const Transpose &t = list.m[blockIdx.z];
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    if (c0 >= t.C || r0 >= t.R) return;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 256 threads: 8 rows per pass
#pragma unroll
    for (int y = ty; y < 32; y += 8) {
        const int r = r0 + y, c = c0 + tx;
        tile[y][tx] = (r < t.R && c < t.C) ? t.in[(size_t)r * t.ldi + c] : 0;
    }
    __syncthreads();
#pragma unroll
    for (int y = ty; y < 32; y += 8) {
        const int c = c0 + y, r = r0 + tx;
        if (c < t.C && r < t.R) t.out[(size_t)c * t.ldo + r] = tile[tx][y];
    }
}

// The kernels below work on 64-column strips with 256 threads: thread (group q = t / 64, lane)
// owns column c0 + lane and rows q, q + 4, q + 8, ... of each 64-row chunk, so a wave reads 64
// consecutive elements of a row; 64 x 64 tiles pass through LDS where a transposed copy is written.

// MSE over the valid M x N outputs: g = bf16(2 (y - t) / (M N)) into g and its transpose gt
// ([N][ldgt]); db[c] = sum over the rows of the bf16 g (the bias gradient); partial[block] = the
// block's sum of (y - t)^2.
__global__ void __launch_bounds__(256) mse_grad(const float *__restrict__ y, int ldy, const float *__restrict__ tgt,
                                                int ldt, int M, int N, uint16_t *__restrict__ g, int ldg,
                                                uint16_t *__restrict__ gt, int ldgt, float *__restrict__ db,
                                                float *__restrict__ partial)
{
    __shared__ uint16_t tile[64][66];
    __shared__ float red[256];
    const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
    const int c0 = blockIdx.x * 64, c = c0 + lane;
    const float scale = 2.0f / ((float)M * (float)N);
    float loss = 0.f, col = 0.f;
    for (int r0 = 0; r0 < M; r0 += 64) {
        for (int k = 0; k < 16; ++k) {
            const int rr = q + 4 * k, r = r0 + rr;
            uint16_t v = 0;
            if (r < M && c < N) {
                const float d = y[(size_t)r * ldy + c] - tgt[(size_t)r * ldt + c];
                loss += d * d;
                v = bf16_rne(scale * d);
                g[(size_t)r * ldg + c] = v;
                col += bf16_to_f32(v);
            }
            tile[rr][lane] = v;
        }
        __syncthreads();
        for (int k = 0; k < 16; ++k) {
            const int cc = q + 4 * k, r = r0 + lane;
            if (c0 + cc < N && r < M) gt[(size_t)(c0 + cc) * ldgt + r] = tile[lane][cc];
        }
        __syncthreads();
    }
    red[threadIdx.x] = col;
    __syncthreads();
    if (q == 0 && c < N) db[c] = (red[lane] + red[lane + 64]) + (red[lane + 128] + red[lane + 192]);
    __syncthreads();
    red[threadIdx.x] = loss;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// db[r] = sum of row r (K entries) of the transposed bf16 gradient gt [R][ldgt]: one wave per row.
__global__ void __launch_bounds__(256) bias_grad(const uint16_t *__restrict__ gt, int ldgt, int R, int K,
                                                 float *__restrict__ db)
{
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= R) return;
    float s = 0.f;
    for (int k = lane; k < K; k += 64) s += bf16_to_f32(gt[(size_t)r * ldgt + k]);
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0) db[r] = s;
}

// v[k] = the sum of a split product's partials at offset at(k), in split order as reduce_splits (one
// partial: itself); the loads of U splits in flight together.
template <int U, int N, class At>
__device__ __forceinline__ void split_sums(const float *__restrict__ part, int nsplit, size_t stride, float (&v)[N], const At &at)
{
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = nsplit > 1 ? 0.f : -0.f;
    int s = 0;
    for (; s + U <= nsplit; s += U, part += U * stride) {
        float q[U][N];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < N; ++k) q[u][k] = part[u * stride + at(k)];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < N; ++k) v[k] += q[u][k];
    }
    for (; s < nsplit; ++s, part += stride)
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] += part[at(k)];
}

// The training step's small kernels are bound by launches and latency (3 to 5 us each, 13 of a 512 x 512
// Adam pass that loaded a row at a time): one per stage of a layer, loads first.

// An activation's gradient g = bf16(dh gelu'(pre)) and its transpose gt, dh from the product's nsplit
// partials (part [nsplit][M][ldp]); tiles of 32 x 32.
__global__ void __launch_bounds__(256) hidden_gradient(const float *__restrict__ part, int nsplit, int ldp,
                                                       const float *__restrict__ pre, int ld, int M, int N,
                                                       uint16_t *__restrict__ g, int ldg, uint16_t *__restrict__ gt, int ldgt)
{
    __shared__ uint16_t tile[32][33];
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int c = c0 + tx;
    float dh[4], z[4];
    auto row = [&](int k) { return (size_t)min(r0 + ty + 8 * k, M - 1); };
    const int cc = min(c, N - 1);
#pragma unroll
    for (int k = 0; k < 4; ++k) z[k] = pre[row(k) * ld + cc];
    split_sums<8>(part, nsplit, (size_t)M * ldp, dh, [&](int k) { return row(k) * ldp + cc; });
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int y = ty + 8 * k, r = r0 + y;
        const uint16_t v = bf16_rne(dh[k] * gelu_grad(z[k]));
        if (r < M && c < N) g[(size_t)r * ldg + c] = v;
        tile[y][tx] = v;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int y = ty + 8 * k;
        if (c0 + y < N && r0 + tx < M) gt[(size_t)(c0 + y) * ldgt + r0 + tx] = tile[tx][y];
    }
}

// A layer's Adam step: the weights [R][C] (gradient: the sum of nsplit partials [R][C]), their bf16 copy
// w16 and its transpose w16t [C][R], in tiles of 32 x 64; in the blocks after those, a wave per row of the
// transposed gradient gt [R][ldgt], the bias (gradient: the sum over the batch's K entries).
__global__ void __launch_bounds__(256) adam_layer(float *__restrict__ w, float *__restrict__ mom, float *__restrict__ vel,
                                                  const float *__restrict__ part, int nsplit, int R, int C, float lr,
                                                  float b1, float b2, float eps, float c1, float c2,
                                                  uint16_t *__restrict__ w16, uint16_t *__restrict__ w16t,
                                                  const uint16_t *__restrict__ gt, int ldgt, int K, float *__restrict__ b,
                                                  float *__restrict__ bmom, float *__restrict__ bvel)
{
    __shared__ uint16_t tile[32][66];
    const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
    const int tiles_c = C / 64, tiles = R / 32 * tiles_c;
    if ((int)blockIdx.x >= tiles) {
        const int r = ((int)blockIdx.x - tiles) * 4 + q;
        if (r >= R) return;
        float s = 0.f;
        for (int k = lane; k < K; k += 64) s += bf16_to_f32(gt[(size_t)r * ldgt + k]);
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (lane == 0) adam_update(b, bmom, bvel, s, r, lr, b1, b2, eps, c1, c2);
        return;
    }
    const int r0 = (int)blockIdx.x / tiles_c * 32, c0 = (int)blockIdx.x % tiles_c * 64;
    float x[8], m[8], v[8], g[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const size_t i = (size_t)(r0 + q + 4 * k) * C + c0 + lane;
        x[k] = w[i], m[k] = mom[i], v[k] = vel[i];
    }
    split_sums<4>(part, nsplit, (size_t)R * C, g, [&](int k) { return (size_t)(r0 + q + 4 * k) * C + c0 + lane; });
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int rr = q + 4 * k;
        const size_t i = (size_t)(r0 + rr) * C + c0 + lane;
        x[k] = adam_value(x[k], m[k], v[k], g[k], lr, b1, b2, eps, c1, c2);
        const uint16_t h = bf16_rne(x[k]);
        w[i] = x[k], mom[i] = m[k], vel[i] = v[k], w16[i] = h;
        tile[rr][lane] = h;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int cc = (threadIdx.x >> 5) + 8 * k, rr = threadIdx.x & 31;
        w16t[(size_t)(c0 + cc) * R + r0 + rr] = tile[rr][cc];
    }
}

// The output bias's Adam step from its gradient, the sum over r < rows of part[r][n] in order.
__global__ void adam_output_bias(const float *__restrict__ part, int rows, int ld, int N,
                                 float *__restrict__ b, float *__restrict__ mom, float *__restrict__ vel, float lr, float b1,
                                 float b2, float eps, float c1, float c2)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    float v = 0.f;
    for (int r = 0; r < rows; ++r) v += part[(size_t)r * ld + n];
    adam_update(b, mom, vel, v, n, lr, b1, b2, eps, c1, c2);
}

__global__ void to_bf16(const float *__restrict__ in, uint16_t *__restrict__ out, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        out[i] = bf16_rne(in[i]);
}

int grid_for(size_t n, int bs = 256) { return (int)std::min<size_t>((n + bs - 1) / bs, 65536); }

}  // namespace

hipError_t gemm_bf16(const uint16_t *A, int lda, const uint16_t *B, int ldb, int M, int N, int K, int epi,
                     const GemmOut &out, float *work, size_t work_floats, int ksplit, hipStream_t stream)
{
    if (M < 1 || N < 1 || K < BK || K % BK || lda % 8 || ldb % 8 || lda < K || ldb < K) return hipErrorInvalidValue;
    const int tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
    if (ksplit < 1) ksplit = 1;
    ksplit = std::min(ksplit, K / BK);
    if (epi == EPI_MSE || epi == EPI_ADAM) {
        // (no split: the epilogue needs the whole sum)
        if (out.ldg % 8 && epi == EPI_MSE) return hipErrorInvalidValue;
        const dim3 grid(tiles, 1);
        if (epi == EPI_MSE) {
            if (!out.tgt || !out.g || !out.gt || !out.partial || !out.dbp || out.ldgt % 8 || (uintptr_t)out.g % 16 ||
                (uintptr_t)out.gt % 16 || (out.tgt_rows && (M % 4 || (uintptr_t)out.tgt_rows % 16)))
                return hipErrorInvalidValue;
            gemm_nt<EPI_MSE><<<grid, 256, 0, stream>>>(A, lda, B, ldb, M, N, K, 1, out);
        } else {
            if (!out.w || !out.mom || !out.vel || !out.w16 || !out.w16t || out.ld16t % 8 || out.ldw % 8 ||
                (uintptr_t)out.w16 % 16 || (uintptr_t)out.w16t % 16)
                return hipErrorInvalidValue;
            gemm_nt<EPI_ADAM><<<grid, 256, 0, stream>>>(A, lda, B, ldb, M, N, K, 1, out);
        }
        return hipGetLastError();
    }
    if (ksplit == 1) {
        const dim3 grid(tiles, 1);
        if (epi == EPI_GELU) gemm_nt<EPI_GELU><<<grid, 256, 0, stream>>>(A, lda, B, ldb, M, N, K, 1, out);
        else gemm_nt<EPI_LINEAR><<<grid, 256, 0, stream>>>(A, lda, B, ldb, M, N, K, 1, out);
        return hipGetLastError();
    }
    if (!work || work_floats < (size_t)ksplit * M * N) return hipErrorInvalidValue;
    GemmOut part{};
    part.f32 = work;
    part.ldf = N;
    gemm_nt<EPI_PARTIAL><<<dim3(tiles, ksplit), 256, 0, stream>>>(A, lda, B, ldb, M, N, K, ksplit, part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    reduce_splits<<<grid_for((size_t)M * N), 256, 0, stream>>>(work, ksplit, M, N, N, out, epi == EPI_GELU);
    return hipGetLastError();
}

bool hidden_in_registers(int members, int M, int N, int K)
{
    return K % RING_K == 0 && K <= kRingRow && members <= 65535 &&
           (K <= (long long)kHiddenChain * members || (long long)members * ((M + 63) / 64) * ((N + 63) / 64) >= 2 * kCus);
}

hipError_t hidden_layer(const uint16_t *A, int lda, size_t stride_a, const uint16_t *B, const uint16_t *const *bs, int ldb,
                        const float *bias, const float *const *biases, int members, int M, int N, int K, int ksplit, float *pre,
                        int ldp, uint16_t *b16, int ldb16, size_t stride_b16, hipStream_t stream)
{
    if (M < 1 || N < 1 || K < RING_K || K % RING_K || lda % 8 || ldb % 8 || lda < K || ldb < K || lda > kRingRow ||
        ldb > kRingRow || members < 1 || members > 65535 || ksplit < 1 || ksplit > K / BK || (bs ? !biases : !B || !bias || members > 1))
        return hipErrorInvalidValue;
    const int kper = ((K / BK + ksplit - 1) / ksplit) * BK;
    hidden_product<<<dim3(((M + 63) / 64) * ((N + 63) / 64), members), 256, 0, stream>>>(
        A, lda, stride_a, B, bs, ldb, bias, biases, M, N, K, kper, pre, ldp, b16, ldb16, stride_b16);
    return hipGetLastError();
}

size_t ensemble_part_doubles(int M, int N) { return (size_t)2 * M * ((N + 63) / 64); }

hipError_t ensemble_output(const uint16_t *A, int lda, size_t stride_a, const uint16_t *const *bs, int ldb,
                           const float *const *biases, int members, int M, int N, int K, float *mean, size_t ldm,
                           const float *scale, double *part, float *spread, hipStream_t stream)
{
    if (M < 1 || N < 1 || K < 64 || K % 64 || lda % 8 || ldb % 8 || lda < K || ldb < K || lda > kRingRow || ldb > kRingRow ||
        members < 1 || (spread && !part))
        return hipErrorInvalidValue;
    if (!spread) part = nullptr;
    const auto tiles = [&](int tm, int tn) { return (long long)((M + tm - 1) / tm) * ((N + tn - 1) / tn); };
    const auto cost = [&](int tm, int tn, int slots, float tile) { return std::max(1.f, tiles(tm, tn) / (float)slots) * tile; };
    const float c64 = cost(64, 64, 2 * kCus, 1.f), c128 = cost(128, 128, 2 * kCus, kCostSquare);
    const bool tall = cost(256, 128, kCus, kCostTall) < std::min(c64, c128), square = !tall && c128 < c64;
    const int tiles_n = (N + (tall || square ? 127 : 63)) / (tall || square ? 128 : 64);
    const int blocks = (int)(tall ? tiles(256, 128) : square ? tiles(128, 128) : tiles(64, 64));
    auto launch = [&](auto kernel, int threads) {
        kernel<<<blocks, threads, 0, stream>>>(A, lda, stride_a, bs, ldb, biases, M, N, K, members, mean, ldm, scale, part);
    };
    if (tall) launch(ensemble_tiles<4, 2, 2, 2, 3>, 512);
    else if (square) launch(ensemble_tiles<2, 2, 2, 2, 2>, 256);
    // (three stages, three blocks to a CU: four stages leave room for two, 100 x 20000 116 us instead of 109,
    // 700 x 6300 158 instead of 150, 40 x 151500 261 instead of 254)
    else launch(ensemble_tiles<2, 2, 1, 1, 3>, 256);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !spread) return e;
    ensemble_spread<<<(M + kSpreadRows - 1) / kSpreadRows, 1024, 0, stream>>>(part, tiles_n, M, members, spread);
    return hipGetLastError();
}

hipError_t transpose_bf16(const Transpose *m, int n, hipStream_t stream)
{
    for (int i0 = 0; i0 < n; i0 += kTransposes) {
        TransposeList list{};
        const int k = std::min(n - i0, kTransposes);
        int rows = 0, cols = 0;
        for (int i = 0; i < k; ++i) {
            list.m[i] = m[i0 + i];
            rows = std::max(rows, list.m[i].R);
            cols = std::max(cols, list.m[i].C);
        }
        transpose16<<<dim3((cols + 31) / 32, (rows + 31) / 32, k), 256, 0, stream>>>(list);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

int mse_blocks(int N) { return (N + 63) / 64; }

hipError_t mse(const float *y, int ldy, const float *t, int ldt, int M, int N, uint16_t *g, int ldg, uint16_t *gt,
               int ldgt, float *db, float *partial, hipStream_t stream)
{
    mse_grad<<<mse_blocks(N), 256, 0, stream>>>(y, ldy, t, ldt, M, N, g, ldg, gt, ldgt, db, partial);
    return hipGetLastError();
}

hipError_t output_bias_step(const float *part, int rows, int ld, int N, float *b, float *mom, float *vel, float lr,
                            float b1, float b2, float eps, long long t, hipStream_t stream)
{
    const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
    adam_output_bias<<<(N + 255) / 256, 256, 0, stream>>>(part, rows, ld, N, b, mom, vel, lr, b1, b2, eps, c1, c2);
    return hipGetLastError();
}

hipError_t gemm_partials(const uint16_t *A, int lda, const uint16_t *B, int ldb, int M, int N, int K, float *work,
                         size_t work_floats, int ksplit, hipStream_t stream)
{
    if (M < 1 || N < 1 || K < BK || K % BK || lda % 8 || ldb % 8 || lda < K || ldb < K || ksplit < 1 || ksplit > K / BK ||
        work_floats < (size_t)ksplit * M * N)
        return hipErrorInvalidValue;
    GemmOut part{};
    part.f32 = work;
    part.ldf = N;
    gemm_nt<EPI_PARTIAL><<<dim3(((M + BM - 1) / BM) * ((N + BN - 1) / BN), ksplit), 256, 0, stream>>>(A, lda, B, ldb, M, N, K,
                                                                                                     ksplit, part);
    return hipGetLastError();
}

hipError_t hidden_gradients(const float *part, int nsplit, const float *pre, int ld, int M, int N, uint16_t *g, int ldg,
                            uint16_t *gt, int ldgt, hipStream_t stream)
{
    hidden_gradient<<<dim3((N + 31) / 32, (M + 31) / 32), 256, 0, stream>>>(part, nsplit, N, pre, ld, M, N, g, ldg, gt, ldgt);
    return hipGetLastError();
}

hipError_t bias_gradient(const uint16_t *gt, int ldgt, int R, int K, float *db, hipStream_t stream)
{
    bias_grad<<<(R + 3) / 4, 256, 0, stream>>>(gt, ldgt, R, K, db);
    return hipGetLastError();
}

hipError_t adam_layer_step(float *w, float *m, float *v, const float *part, int nsplit, int R, int C, float lr, float b1,
                           float b2, float eps, long long t, uint16_t *w16, uint16_t *w16t, const uint16_t *gt, int ldgt, int K,
                           float *b, float *bm, float *bv, hipStream_t stream)
{
    if (R % 32 || C % 64) return hipErrorInvalidValue;
    const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
    adam_layer<<<R / 32 * (C / 64) + (R + 3) / 4, 256, 0, stream>>>(w, m, v, part, nsplit, R, C, lr, b1, b2, eps, c1, c2, w16,
                                                                  w16t, gt, ldgt, K, b, bm, bv);
    return hipGetLastError();
}

hipError_t convert_bf16(const float *in, uint16_t *out, size_t n, hipStream_t stream)
{
    to_bf16<<<grid_for(n), 256, 0, stream>>>(in, out, n);
    return hipGetLastError();
}

}  // namespace mlp
}  // namespace poe2d
