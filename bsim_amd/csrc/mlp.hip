/*
 * mlp.hip -- the rate surrogate: a ReLU multilayer perceptron trained and run
 * on the GPU with bf16 MFMA (v_mfma_f32_16x16x32_bf16, fp32 accumulation).
 *
 * Model: in (padded to 64) -> L hidden layers of H units (ReLU) -> out
 * (padded to a multiple of 64, linear).  Weights are held twice: an fp32
 * master copy updated by Adam and the bf16 copy the GEMMs read.  Activations
 * and activation gradients are stored in bf16 (round to nearest even, done
 * here bit by bit), every product is accumulated in fp32.
 *
 * One training step (bsim_mlp_train):
 *   gather     minibatch rows of the resident data set -> X (bf16), Y (f32)
 *   forward    H_l = bf16(relu(H_{l-1} W_l^T + b_l)),  out = H_L W^T + b (f32)
 *   loss       dZ = bf16(2 (out - Y) / (B * out_dim)); loss and bias-gradient
 *              partials
 *   backward   dZ_{l-1} = bf16(dZ_l W_l) where H_{l-1} > 0, with its
 *              bias-gradient partials
 *   update     dW_l = dZ_l^T H_{l-1} in four sums over quarters of the batch,
 *              added in order; Adam (Kingma & Ba, 2015) on the fp32 master;
 *              the bf16 copies of W_l and its transpose
 * Launches per step: with layers of up to 512 units two, everything up to the
 * backward products (mlp_chain) and the update (mlp_update); with wider ones a
 * GEMM per layer forward and per activation gradient (mlp_gemm) before the
 * update.
 *
 * Operands that are read along a reduction index from memory lie in fragments
 * (frag_index): the bf16 copies of the weights and, for the weight gradients,
 * the transposed copies of the inputs, activations and activation gradients.  A
 * wavefront loads or stores a fragment as one contiguous KB, straight to and
 * from the registers that the MFMA reads and writes.  In rows, the same loads
 * fetched 64 bytes from each of 16 rows: mlp_chain's launch of 4,096 rows
 * through 4 x 512 units took 73 us that way and 28 in fragments (predict).
 * Every reduction has a fixed order, so results repeat bit for bit.
 *
 * There is no counterpart in the reference; the algorithm is the textbook
 * back-propagation of a fully connected ReLU network and Adam.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "../../include/bsim_mlp.h"
#include <omp.h>

#include "internal.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int WAVE = 64;
constexpr int BM = 64, BN = 64, BK = 64;   /* workgroup tile and k step */
constexpr int LDS_STRIDE = BK + 8;         /* bf16 per LDS tile row (144 B) */
constexpr int GEMM_THREADS = 256;          /* 2 x 2 wavefronts of 32 x 32 */
constexpr int KSPLIT = 4;                  /* batch split of the weight gradients */
constexpr int TRAIN_BATCH_ALIGN = KSPLIT * BK;   /* training batches: whole pairs of 32 rows per split */
constexpr int ROWS_PER_PART = 32;          /* bias-gradient partial: rows per partial */
constexpr int MAX_LAYERS = 10;             /* linear layers (hidden + 1) */

__host__ __device__ inline uint16_t f2bf(float x)
{
    uint32_t u;
    memcpy(&u, &x, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);   /* round to nearest even (finite x) */
    return (uint16_t)(u >> 16);
}

/* Two at once on the device, v_cvt_pk_bf16_f32: lo in the low half. */
__device__ inline uint32_t pack_bf(float lo, float hi)
{
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, bf16x2{(__bf16)lo, (__bf16)hi});
}

__host__ __device__ inline float bf2f(uint16_t h)
{
    const uint32_t u = (uint32_t)h << 16;
    float x;
    memcpy(&x, &u, 4);
    return x;
}

/* Where element (n, k) of a matrix [N][K] with reduction index k lies in
 * fragments: the 16 x 32 operand of one MFMA, as the wavefront's lanes hold it,
 * is 1 KB; those of 32 k for all n follow one another. */
__host__ __device__ inline int64_t frag_index(int32_t n, int32_t k, int32_t N)
{
    return ((int64_t)(k / 32) * (N / 16) + n / 16) * 512 + (k % 32 / 8 * 16 + n % 16) * 8 + k % 8;
}

enum Epi { EPI_RELU_BF16 = 0, EPI_LINEAR_F32 = 1, EPI_DRELU_BF16 = 2, EPI_LOSS = 3 };

/* C[m][n] = sum_k A[m * lda + k] B(n, k), B in fragments. */
struct GemmArgs {
    const uint16_t *A;
    const uint16_t *B;
    int64_t lda;
    int32_t M, N, K;
    int32_t pad;
    const float *bias;      /* EPI_RELU_BF16, EPI_LINEAR_F32: [N] */
    uint16_t *out_bf;       /* EPI_RELU_BF16, EPI_DRELU_BF16: [M][ldo] */
    float *out_f;           /* EPI_LINEAR_F32: [M][ny] */
    int64_t ldo;
    const uint16_t *mask;   /* EPI_DRELU_BF16: keep where mask[m * ldo + n] > 0 */
    float *bpart;           /* EPI_DRELU_BF16, EPI_LOSS: bias-gradient partials [M / 32][N] */
    uint16_t *out_t;        /* EPI_RELU_BF16, EPI_DRELU_BF16, EPI_LOSS: transposed copy [N][M] in fragments, or null */
    const int32_t *arow;    /* row m of A is row arow[m] of the array A (null: row m) */
    uint16_t *a_t;          /* with K == BK: workgroups of column tile 0 write A^T [K][M] in fragments */
    const float *y;         /* EPI_LOSS: targets, row m at y[(yrow ? yrow[m] : m) * ny] */
    const int32_t *yrow;
    int32_t ny;             /* EPI_LINEAR_F32, EPI_LOSS: valid output columns */
    float scale;            /* EPI_LOSS: dZ = bf16(scale * (C + bias - y)) */
    float *lpart;           /* EPI_LOSS: squared-error sums, of the quadrants of each 64 x 64 tile [M / 64][N / 64][4] */
};

/* One k step of a 64-row operand: thread tid holds rows tid / 8 and
 * tid / 8 + 32, k (tid % 8) * 8 .. + 7. */
struct Tile {
    uint4 v[2];
};

__device__ inline Tile load_tile(const uint16_t *P, int64_t ld, int32_t r0, int32_t k0, uint32_t tid,
                                 const int32_t *rowmap = nullptr)
{
    const uint32_t r = tid >> 3, kc = (tid & 7u) * 8u;
    const int64_t ra = rowmap ? (int64_t)rowmap[r0 + r] : (int64_t)(r0 + r);
    const int64_t rb = rowmap ? (int64_t)rowmap[r0 + r + 32] : (int64_t)(r0 + r + 32);
    Tile t;
    t.v[0] = *(const uint4 *)(P + ra * ld + k0 + kc);
    t.v[1] = *(const uint4 *)(P + rb * ld + k0 + kc);
    return t;
}

__device__ inline void store_tile(uint16_t *T, const Tile &t, uint32_t tid)
{
    const uint32_t r = tid >> 3, kc = (tid & 7u) * 8u;
    *(uint4 *)(T + r * LDS_STRIDE + kc) = t.v[0];
    *(uint4 *)(T + (r + 32) * LDS_STRIDE + kc) = t.v[1];
}

/* The same of an operand in fragments: of each 32 k, the tile's four are
 * contiguous, and a wavefront takes one. */
__device__ inline Tile load_frag_tile(const uint16_t *P, int32_t N, int32_t r0, int32_t k0, uint32_t tid)
{
    const uint16_t *p = P + ((int64_t)(k0 / 32) * (N / 16) + r0 / 16) * 512;
    Tile t;
    t.v[0] = *(const uint4 *)(p + tid * 8u);
    t.v[1] = *(const uint4 *)(p + (uint32_t)N * 32u + tid * 8u);
    return t;
}

__device__ inline void store_frag_tile(uint16_t *T, const Tile &t, uint32_t tid)
{
    const uint32_t r = tid / 64 * 16 + tid % 16, k = tid % 64 / 16 * 8;
    *(uint4 *)(T + r * LDS_STRIDE + k) = t.v[0];
    *(uint4 *)(T + r * LDS_STRIDE + k + 32) = t.v[1];
}

/* Output tile (bx, by): C[by * 64 .. + 63][bx * 64 .. + 63]. */
template <int EPI>
__device__ inline void gemm_tile(const GemmArgs &g, int32_t bx, int32_t by)
{
    __shared__ __attribute__((aligned(16))) uint16_t As[2][BM * LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[2][BN * LDS_STRIDE];
    __shared__ float bsum[2][BN];

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & (WAVE - 1), w = tid / WAVE;
    const uint32_t wm = w >> 1, wn = w & 1u;     /* wavefront's 32 x 32 quadrant */
    const int32_t n0 = bx * BN, m0 = by * BM;
    const int32_t nk = g.K / BK;

    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    /* k step s is multiplied from LDS buffer s & 1; at its start, step s+1
     * (loaded during step s-1) moves from registers to the other buffer and
     * the loads of step s+2 are issued, so that they are in flight during a
     * whole step */
    Tile ra, rb;
    {
        const Tile a0 = load_tile(g.A, g.lda, m0, 0, tid, g.arow);
        const Tile b0 = load_frag_tile(g.B, g.N, n0, 0, tid);
        if (nk > 1) {
            ra = load_tile(g.A, g.lda, m0, BK, tid, g.arow);
            rb = load_frag_tile(g.B, g.N, n0, BK, tid);
        }
        store_tile(As[0], a0, tid);
        store_frag_tile(Bs[0], b0, tid);
    }
    /* the epilogue's other operands for this lane's 16 outputs (rows m0 +
     * 32 wm + 16 i + 4 (lane / 16) + r, column n0 + 32 wn + 16 j + lane %
     * 16): the activation mask (EPI_DRELU_BF16) is loaded while the products
     * run; of the targets (EPI_LOSS) only the row indices are -- the target
     * loads themselves are issued after the products, since loads issued
     * before them hold up every wait of the k loop (the wait counter is in
     * order) and the gathered targets are a chain of two loads */
    uint16_t mk[2][2][4];
    float yv[2][2][4];
    int32_t yr[2][4];
    const uint32_t rq0 = (lane >> 4) * 4u, c16 = lane & 15u;
    if (EPI == EPI_DRELU_BF16) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int32_t row = m0 + (int32_t)(wm * 32 + i * 16 + rq0) + r;
                    const int32_t col = n0 + (int32_t)(wn * 32 + j * 16 + c16);
                    mk[i][j][r] = g.mask[(int64_t)row * g.ldo + col];
                }
    }
    if (EPI == EPI_LOSS) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int32_t row = m0 + (int32_t)(wm * 32 + i * 16 + rq0) + r;
                yr[i][r] = g.yrow ? g.yrow[row] : row;
            }
    }
    __syncthreads();
    /* the first layer of a training step: A's rows are gathered, and the
     * workgroups of column tile 0 also write them transposed (one k step) */
    if (g.a_t && bx == 0 && nk == 1) {
        for (uint32_t x = tid; x < (uint32_t)(BM * BK); x += GEMM_THREADS) {
            const uint32_t k = x / BM, r = x % BM;
            g.a_t[frag_index((int32_t)k, m0 + (int32_t)r, g.K)] = As[0][r * LDS_STRIDE + k];
        }
    }

    const uint32_t r16 = lane & 15u, kg = (lane >> 4) * 8u;
    for (int32_t s = 0; s < nk; s++) {
        const int cur = s & 1;
        if (s + 1 < nk) {
            store_tile(As[cur ^ 1], ra, tid);
            store_frag_tile(Bs[cur ^ 1], rb, tid);
            if (s + 2 < nk) {
                ra = load_tile(g.A, g.lda, m0, (s + 2) * BK, tid, g.arow);
                rb = load_frag_tile(g.B, g.N, n0, (s + 2) * BK, tid);
            }
        }
#pragma unroll
        for (int kk = 0; kk < BK; kk += 32) {
            bf16x8 a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; i++)
                a[i] = *(const bf16x8 *)(As[cur] + (wm * 32 + i * 16 + r16) * LDS_STRIDE + kk + kg);
#pragma unroll
            for (int j = 0; j < 2; j++)
                b[j] = *(const bf16x8 *)(Bs[cur] + (wn * 32 + j * 16 + r16) * LDS_STRIDE + kk + kg);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }

    if (EPI == EPI_LOSS) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int32_t col = n0 + (int32_t)(wn * 32 + j * 16 + c16);
                    yv[i][j][r] = col < g.ny ? g.y[(int64_t)yr[i][r] * g.ny + col] : 0.f;
                }
    }
    /* lane holds C[row0 + 4 * (lane / 16) + r][col0 + lane % 16], r = 0..3 */
    const uint32_t rq = (lane >> 4) * 4u;
    float csum[2] = {0.f, 0.f};
    float lsum = 0.f;
#pragma unroll
    for (int i = 0; i < 2; i++) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int32_t col = n0 + wn * 32 + j * 16 + r16;
            const int32_t row0 = m0 + wm * 32 + i * 16 + rq;
            uint16_t h[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int32_t row = row0 + r;
                const float v = acc[i][j][r];
                if (EPI == EPI_RELU_BF16) {
                    const float z = v + g.bias[col];
                    h[r] = f2bf(z > 0.f ? z : 0.f);
                    g.out_bf[(int64_t)row * g.ldo + col] = h[r];
                } else if (EPI == EPI_LINEAR_F32) {
                    if (col < g.ny) g.out_f[(int64_t)row * g.ny + col] = v + g.bias[col];
                } else if (EPI == EPI_DRELU_BF16) {
                    const uint16_t m = mk[i][j][r];
                    h[r] = (m != 0 && !(m & 0x8000u)) ? f2bf(v) : (uint16_t)0;
                    g.out_bf[(int64_t)row * g.ldo + col] = h[r];
                    csum[j] += bf2f(h[r]);
                } else if (EPI == EPI_LOSS) {
                    /* the output (as EPI_LINEAR_F32 rounds it), its error and dZ */
                    const float out = v + g.bias[col];
                    h[r] = 0;
                    if (col < g.ny) {
                        const float diff = out - yv[i][j][r];
                        lsum += diff * diff;
                        h[r] = f2bf(g.scale * diff);
                    }
                    g.out_bf[(int64_t)row * g.ldo + col] = h[r];
                    csum[j] += bf2f(h[r]);
                }
            }
            if ((EPI == EPI_RELU_BF16 || EPI == EPI_DRELU_BF16 || EPI == EPI_LOSS) && g.out_t) {
                /* 4 consecutive rows of one column: one 8-byte store */
                const uint2 q = {(uint32_t)h[0] | ((uint32_t)h[1] << 16),
                                 (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
                *(uint2 *)(g.out_t + frag_index(col, row0, g.N)) = q;
            }
        }
    }
    if (EPI == EPI_DRELU_BF16 || EPI == EPI_LOSS) {
        /* column sums over 32 rows each, in a fixed order */
#pragma unroll
        for (int j = 0; j < 2; j++) {
            float x = csum[j];
            x += __shfl_xor(x, 16);
            x += __shfl_xor(x, 32);
            if (lane < 16) bsum[wm][wn * 32 + j * 16 + lane] = x;
        }
        if (EPI == EPI_LOSS) {
            /* the quadrant's squared error, in a fixed order */
#pragma unroll
            for (int o = 1; o < WAVE; o <<= 1) lsum += __shfl_xor(lsum, o);
            if (lane == 0) g.lpart[((int64_t)by * (g.N / BN) + bx) * 4 + w] = lsum;
        }
        __syncthreads();
        if (tid < 2 * BN) g.bpart[(2 * (int64_t)by + tid / BN) * g.N + n0 + tid % BN] = bsum[tid / BN][tid % BN];
    }
}

/* Tile t of ny x nx: bands of `band` rows, in a band column by column.  The
 * workgroups that an XCD runs at a time so form a block of tiles that shares rows
 * and columns in its L2; row by row (a band of 1) they read one row of tiles and,
 * in wide layers, more columns than it holds.  Training steps of 4,096 rows, us,
 * products and weight gradients row by row / in bands: 3 x 1,024 units 185 / 179,
 * 3 x 1,536 317 / 290, 2 x 4,096 and 4,096 outputs 2,020 / 1,560. */
__device__ inline void band_tile(int32_t t, int32_t nx, int32_t ny, int32_t band, int32_t &bx, int32_t &by)
{
    if (band == 1) {
        by = t / nx;
        bx = t - by * nx;
        return;
    }
    const int32_t b = t / (band * nx) * band, h = min(band, ny - b), i = t - b * nx;
    bx = i / h;
    by = b + (i - bx * h);
}

template <int EPI>
__global__ __launch_bounds__(GEMM_THREADS) void mlp_gemm(GemmArgs g)
{
    /* an XCD takes consecutive tiles: it reads an eighth of A, and the rows that
     * it wrote itself in the layer before */
    const int32_t nt = (int32_t)gridDim.x, x = (int32_t)blockIdx.x % 8;
    int32_t bx, by;
    band_tile(x * (nt / 8) + min(x, nt % 8) + (int32_t)blockIdx.x / 8, g.N / BN, g.M / BM, 8, bx, by);
    gemm_tile<EPI>(g, bx, by);
}

/* ---- every layer in one launch ---------------------------------------------
 *
 * A row of the batch depends on no other row until the weight gradients, so a
 * workgroup can take CH_ROWS rows through all layers, forward and back, with
 * the activations in LDS.  A stage is one product with a weight matrix: the
 * forward layers in order, then (training) the activation gradients from the
 * last layer to the second.
 *
 * What bounds it: every workgroup reads every weight, 512 KB per stage of 512 x
 * 512 from its XCD's L2 at the 64 bytes per cycle that a compute unit takes in,
 * 3.4 us, against 1.7 of MFMA; measured 4.7 us per such stage (the rest is the
 * epilogue, between two barriers), and 8 to launch, load the input and start
 * the stream.  A launch per layer took 9 to 10 us for the same stage, of which
 * the kernel's start, a pass of loads that nothing hides and the end of the
 * grid were most.  The weights are loaded 128 rows of the reduction index ahead,
 * through the ends of the stages, as they depend on nothing; 16 rows per
 * workgroup would read the weights twice as often in the same time, 64 would
 * leave more compute units idle.  Sixteen wavefronts of 32 columns each against
 * eight of 64: 51 / 54 us.  Training step of 4,096 rows through 4 x 512 units,
 * 200 outputs: 83 us in nine launches, 51 chained; 256 rows through 2 x 192: 33
 * / 12; predict 4,096 rows: 47 / 25.
 *
 * Layers wider than CH_MAX run in a launch each: 1,024 units would take 14 us
 * per stage here whatever the rows, as many as 2,048 rows take in a launch of
 * their own, and two of them exceed a wavefront's registers.
 */
constexpr int CH_ROWS = 32;                /* rows of a workgroup: two MFMA tiles, one bias-gradient partial */
constexpr int CH_MAX = 512;                /* widest layer */
static_assert(CH_ROWS == ROWS_PER_PART, "a workgroup writes its rows' bias-gradient partial");

struct ChainArgs {
    int32_t nlin, ld;                      /* ld: LDS row stride, widest layer + 8 */
    int32_t kdim[MAX_LAYERS + 1];
    int32_t din;
    int64_t woff[MAX_LAYERS], boff[MAX_LAYERS];
    const uint16_t *w, *wt;                /* W_l and W_l^T at woff[l], in fragments (frag_index) */
    const float *p;                        /* biases at boff[l] */
    const uint16_t *xb;                    /* input rows, bf16 [.][kdim[0]], or null: */
    const float *xf;                       /* f32 [n][din] */
    const int32_t *rows;                   /* row m of the batch is row rows[m] of xb and y (null: row m) */
    int64_t n;                             /* rows of xf; the batch's others are 0 */
    float *out;                            /* predict: [batch][ny] */
    uint16_t *act_t[MAX_LAYERS], *dzt[MAX_LAYERS];   /* training: transposed, [unit][batch] in fragments */
    float *bpart[MAX_LAYERS], *lpart;
    const float *y;
    int32_t ny;
    float scale;
};

/* The product of a stage: W [N][K]. */
struct ChainStage {
    const uint16_t *w;
    int32_t K, N;
};

__device__ inline ChainStage chain_stage(const ChainArgs &a, int32_t s)
{
    if (s < a.nlin) return ChainStage{a.w + a.woff[s], a.kdim[s], a.kdim[s + 1]};
    const int32_t l = 2 * a.nlin - 1 - s;
    return ChainStage{a.wt + a.woff[l], a.kdim[l + 1], a.kdim[l]};
}

/* 0xFFFF in each half of x that is not 0; no half has its top bit set. */
__device__ inline uint32_t nonzero_halves(uint32_t x)
{
    const uint32_t t = (x + 0x7FFF7FFFu) & 0x80008000u;
    return (t - (t >> 15)) | t;
}

/* W wavefronts; wavefront w has the columns 32 w .. 32 w + 31 of every stage. */
template <int W, bool TRAIN>
__global__ __launch_bounds__(W * WAVE) void mlp_chain(ChainArgs a)
{
    constexpr int T = 2;                                        /* tiles of 16 columns */
    extern __shared__ __align__(16) uint16_t ch_lds[];
    const int32_t LD = a.ld, L = a.nlin;
    int32_t *rowid = reinterpret_cast<int32_t *>(ch_lds + 2 * CH_ROWS * LD);      /* [CH_ROWS] rows of y */
    const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1), w = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const uint32_t r16 = lane & 15u, kg = (lane >> 4) * 8u, rq = (lane >> 4) * 4u;
    /* an XCD takes consecutive row tiles: two of them share the lines of the transposed copies */
    const int32_t nt = (int32_t)gridDim.x, x = (int32_t)blockIdx.x % 8, q = (int32_t)blockIdx.x / 8;
    const int32_t mt = x * (nt / 8) + min(x, nt % 8) + q;
    const int32_t m0 = mt * CH_ROWS;
    const int32_t S = TRAIN ? 2 * L - 1 : L;
    /* rows rq .. rq + 3 of unit r16 in a fragment (rows 16 on: 256 further) */
    const uint32_t fl = (rq / 8 * 16 + r16) * 8 + rq % 8;

    /* the weights stream: two steps of 64 of the reduction index in registers,
     * through the stages' ends.  Stages with an odd number of steps take one more,
     * which is loaded (the last again) and not multiplied. */
    bf16x8 B[2][T][2];
    int32_t ls = 0, lc = 0, lnk = 0, lst = 0;
    const uint16_t *lp[T];
    auto enter = [&]() {
        const ChainStage g = chain_stage(a, ls);
        lnk = g.K / BK;
        lst = g.N * 32;
#pragma unroll
        for (int j = 0; j < T; j++) {
            /* columns past the stage's: any others of it */
            const int32_t c = (int32_t)w * 32, col = (c < g.N ? c : 0) + j * 16;
            lp[j] = g.w + col * 32;
        }
    };
    auto issue = [&](bf16x8 (&b)[T][2]) {
        const int32_t k = min(lc, lnk - 1) * 2 * lst;
#pragma unroll
        for (int j = 0; j < T; j++)
#pragma unroll
            for (int h = 0; h < 2; h++) b[j][h] = *(const bf16x8 *)(lp[j] + k + h * lst + lane * 8u);
        if (++lc >= ((lnk + 1) & ~1) && ls + 1 < S) {
            ls++;
            lc = 0;
            enter();
        }
    };
    enter();
    issue(B[0]);
    issue(B[1]);

    /* the input rows: thread tid has four columns of row tid / 16 */
    if (tid < CH_ROWS * 16) {
        const int32_t r = (int32_t)tid / 16, c = (int32_t)(tid % 16) * 4;
        uint2 v = {0u, 0u};
        const int64_t row = a.rows ? (int64_t)a.rows[m0 + r] : (int64_t)(m0 + r);
        if (a.xb) {
            v = *(const uint2 *)(a.xb + row * BK + c);
        } else if (row < a.n) {
            uint16_t h[4];
#pragma unroll
            for (int i = 0; i < 4; i++) h[i] = c + i < a.din ? f2bf(a.xf[row * a.din + c + i]) : (uint16_t)0;
            v = {(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
        }
        *(uint2 *)(ch_lds + r * LD + c) = v;
        if (c == 0) rowid[r] = (int32_t)row;
    }
    __syncthreads();
    if (TRAIN && tid < CH_ROWS * 16) {
        const int32_t k = (int32_t)tid / 8, r = (int32_t)(tid % 8) * 4;
        const uint16_t *c = ch_lds + r * LD + k;
        const uint2 v = {(uint32_t)c[0] | ((uint32_t)c[LD] << 16),
                         (uint32_t)c[2 * LD] | ((uint32_t)c[3 * LD] << 16)};
        *(uint2 *)(a.act_t[0] + frag_index(k, m0 + r, BK)) = v;
    }

    for (int32_t s = 0; s < S; s++) {
        const ChainStage g = chain_stage(a, s);
        const int32_t nk = g.K / BK;
        const uint16_t *in = ch_lds + (s & 1) * CH_ROWS * LD;
        uint16_t *nx = ch_lds + ((s + 1) & 1) * CH_ROWS * LD;
        const bool fwd = !TRAIN || s < L;
        float bias[T];
        int32_t col[T];
        int64_t fr[T];                                          /* this lane's rows of a transposed copy */
        const int32_t c0 = (int32_t)w * 32;
        const bool on = c0 < g.N;                               /* uniform */
#pragma unroll
        for (int j = 0; j < T; j++) {
            col[j] = (on ? c0 : 0) + j * 16 + (int32_t)r16;
            fr[j] = ((int64_t)mt * (g.N / 16) + (on ? c0 : 0) / 16 + j) * 512;
            bias[j] = fwd ? a.p[a.boff[s] + col[j]] : 0.f;
        }
        f32x4 acc[2][T];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < T; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto mul = [&](bf16x8 (&b)[T][2], int32_t k0) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                bf16x8 av[2];
#pragma unroll
                for (int i = 0; i < 2; i++) av[i] = *(const bf16x8 *)(in + (i * 16 + r16) * LD + k0 + h * 32 + kg);
#pragma unroll
                for (int j = 0; j < T; j++)
#pragma unroll
                    for (int i = 0; i < 2; i++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], b[j][h], acc[i][j], 0, 0, 0);
            }
        };
        /* dZ of layer l's output is what a stage from the loss on forms */
        const int32_t l = s < L ? s : 2 * L - 2 - s;
        uint16_t *tr = !TRAIN ? nullptr : s < L - 1 ? a.act_t[s + 1] : a.dzt[l];
        float yv[2][T][4];
        uint2 act[2][T];
        if (TRAIN && s == L - 1) {
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int64_t row = rowid[i * 16 + (int32_t)rq + r];
#pragma unroll
                    for (int j = 0; j < T; j++) yv[i][j][r] = a.y[row * a.ny + min(col[j], a.ny - 1)];
                }
        }
        if (TRAIN && s >= L) {
            /* this lane's own values, written in the forward stage */
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < T; j++)
                    act[i][j] = *(const uint2 *)(a.act_t[l + 1] + fr[j] + i * 256 + fl);
        }
        int32_t c = 0;
        do {
            mul(B[0], c * BK);
            issue(B[0]);
            if (c + 1 < nk) mul(B[1], (c + 1) * BK);
            issue(B[1]);
            c += 2;
        } while (c < nk);           /* at least once: the loads before it then have 16 after them */
        /* lane holds rows 16 i + rq + r, columns col[j] */
        if (!TRAIN && s == L - 1) {
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < T; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (on && col[j] < a.ny)
                            a.out[(int64_t)(m0 + i * 16 + (int32_t)rq + r) * a.ny + col[j]] = acc[i][j][r] + bias[j];
            break;
        }
        uint2 h[2][T];                                          /* the stage's bf16 values */
        if (s < L - 1) {
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < T; j++) {
                    float z[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        z[r] = acc[i][j][r] + bias[j];
                        z[r] = z[r] > 0.f ? z[r] : 0.f;
                    }
                    h[i][j] = uint2{pack_bf(z[0], z[1]), pack_bf(z[2], z[3])};
                }
        } else if (TRAIN && s == L - 1) {
            float lsum = 0.f;
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < T; j++) {
                    float z[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float diff = col[j] < a.ny ? acc[i][j][r] + bias[j] - yv[i][j][r] : 0.f;
                        lsum += diff * diff;
                        z[r] = a.scale * diff;
                    }
                    h[i][j] = uint2{pack_bf(z[0], z[1]), pack_bf(z[2], z[3])};
                }
#pragma unroll
            for (int o = 1; o < WAVE; o <<= 1) lsum += __shfl_xor(lsum, o);
            /* a quadrant of a tile of 64 x 64 */
            if (lane == 0 && on)
                a.lpart[((int64_t)(mt / 2) * (g.N / BN) + w / 2) * 4 + (mt & 1) * 2 + (w & 1)] = lsum;
        } else if (TRAIN) {
            /* where the activation is not 0 (it is never below) */
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < T; j++) {
                    h[i][j] = uint2{pack_bf(acc[i][j][0], acc[i][j][1]), pack_bf(acc[i][j][2], acc[i][j][3])};
                    h[i][j].x &= nonzero_halves(act[i][j].x);
                    h[i][j].y &= nonzero_halves(act[i][j].y);
                }
        }
#pragma unroll
        for (int j = 0; j < T; j++) {
            if (!on) continue;                                  /* uniform */
#pragma unroll
            for (int i = 0; i < 2; i++) {
                uint16_t *c = nx + (i * 16 + rq) * LD + col[j];
                c[0] = (uint16_t)h[i][j].x;
                c[LD] = (uint16_t)(h[i][j].x >> 16);
                c[2 * LD] = (uint16_t)h[i][j].y;
                c[3 * LD] = (uint16_t)(h[i][j].y >> 16);
                if (TRAIN) *(uint2 *)(tr + fr[j] + i * 256 + fl) = h[i][j];
            }
            if (TRAIN && s >= L - 1) {
                float v = 0.f;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    v += __uint_as_float(h[i][j].x << 16);
                    v += __uint_as_float(h[i][j].x & 0xFFFF0000u);
                    v += __uint_as_float(h[i][j].y << 16);
                    v += __uint_as_float(h[i][j].y & 0xFFFF0000u);
                }
                v += __shfl_xor(v, 16);
                v += __shfl_xor(v, 32);
                if (lane < 16) a.bpart[l][(int64_t)mt * g.N + col[j]] = v;
            }
        }
        __syncthreads();
    }
}

/* ---- weight gradients and Adam ---------------------------------------------- */

struct UpdateArgs {
    int32_t nlin, batch;
    int32_t n[MAX_LAYERS], k[MAX_LAYERS];   /* W_l is [n][k] */
    int32_t tfirst[MAX_LAYERS + 1];         /* first workgroup of W_l's tiles */
    int32_t wide[MAX_LAYERS];               /* tiles of 128 x 128, else 64 x 64 */
    int32_t bfirst[MAX_LAYERS + 1];         /* first bias workgroup of layer l; those before the tiles': */
    int32_t nbias;                          /*   a multiple of 8, the last ones idle */
    int32_t update;                         /* 0: only write the gradient */
    int64_t woff[MAX_LAYERS], boff[MAX_LAYERS];
    const uint16_t *dzt[MAX_LAYERS], *act_t[MAX_LAYERS];    /* [unit][batch], in fragments */
    const float *bpart[MAX_LAYERS];         /* bias-gradient partials [batch / 32][n] */
    float lr, b1, b2, eps, c1, c2;          /* c1 = 1 - b1^t, c2 = 1 - b2^t */
    float *p, *m, *v, *grad;
    uint16_t *w, *wt;                       /* bf16 W_l and W_l^T at woff[l], in fragments */
    const float4 *lpart;                    /* loss partials of the step */
    int32_t nlpart;
    float lscale;
    float *loss;
};

/* Adam (Kingma & Ba, 2015) for one parameter: its state before, gradient g;
 * the parameter after. */
__device__ inline float adam(const UpdateArgs &a, int64_t i, float g, float p, float m, float v)
{
    m = a.b1 * m + (1.f - a.b1) * g;
    v = a.b2 * v + (1.f - a.b2) * (g * g);
    a.m[i] = m;
    a.v[i] = v;
    const float mhat = m / a.c1, vhat = v / a.c2;
    p -= a.lr * (mhat / (sqrtf(vhat) + a.eps));
    a.p[i] = p;
    return p;
}

typedef uint16_t WTile[64][66];

/* A 64 x 64 tile (row r0, column c0) of W [N][K] to the bf16 copies of W and
 * its transpose: a lane's eight elements of a fragment at a time. */
__device__ inline void put_weights(const WTile &tile, uint16_t *w, uint16_t *wt, int32_t N, int32_t K, int32_t r0,
                                   int32_t c0)
{
    for (int32_t x = (int32_t)threadIdx.x; x < 512; x += (int32_t)blockDim.x) {
        const int32_t f = x / 64, l = x % 64;
        const int32_t n = f / 2 * 16 + l % 16, k = f % 2 * 32 + l / 16 * 8;
        uint32_t q[4], t[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            q[i] = (uint32_t)tile[n][k + 2 * i] | ((uint32_t)tile[n][k + 2 * i + 1] << 16);
            t[i] = (uint32_t)tile[k + 2 * i][n] | ((uint32_t)tile[k + 2 * i + 1][n] << 16);
        }
        *(uint4 *)(w + frag_index(r0 + n, c0 + k, N)) = uint4{q[0], q[1], q[2], q[3]};
        *(uint4 *)(wt + frag_index(c0 + n, r0 + k, K)) = uint4{t[0], t[1], t[2], t[3]};
    }
}

/* One workgroup per 64 x 64 tile of a weight matrix: dW_l = dZ_l^T H_l, a
 * quarter of the batch per wavefront, the quarters' sums added in order, then
 * Adam on the tile and its bf16 copies.
 *
 * What bounds it: a tile reads 1 MB of fragments at 4,096 rows, 6.8 us at the 64
 * bytes per cycle of a compute unit, of which a few are waits for what other
 * XCDs wrote; 8 us go to the launch, the exchange of the sums and Adam's divides
 * and square roots.  Without LDS for the operands: each wavefront multiplies 64 x
 * 64 outputs from registers (8 KB of loads per 16 MFMAs).  In two launches, with
 * the four sums written out and read back, this took 25 + 10 us where it takes
 * 22 now (950,000 parameters, 4,096 rows), and 27 + 10 / 22 (2,600,000, 2,048
 * rows).  Four steps in flight instead of two need the registers of a second
 * workgroup per compute unit: 28 us for the latter.
 *
 * Layers of 2,048 x 2,048 and more whose operands exceed 192 MB (a quarter less
 * than the 256 MB cache between the L2s and memory) go in tiles of 128 x 128, a
 * 64 x 64 quadrant per wavefront in the whole batch, quarter by quarter: the four
 * wavefronts walk one place of the batch instead of four, with half the bytes per
 * product.  Two layers of 4,096 x 4,096, 16,384 rows: 158 million lines missed the
 * L2s in tiles of 64, 2,900 us; the training step 6,950 us so, 5,850 in tiles of
 * 128.  Below the line tiles of 64 are as good (3,072 x 3,072, 8,192 rows: 2,475 /
 * 2,436; 2,048 x 2,048, 16,384 rows: 2,310 / 2,412), and with fewer than 256 tiles
 * of 128 compute units stay idle (512 x 512, 65,536 rows: 740 / 1,270).
 * Tiles of 64 of layers from 1,024 x 1,024 up are taken in bands of four (band_tile);
 * smaller ones row by row (9 x 512 units, 16,384 rows: 490 / 502).
 * The workgroups before them take 256 biases each, the first also the step's loss. */
constexpr int UP_THREADS = KSPLIT * WAVE;
constexpr int64_t UP_WIDE_BYTES = 192ll << 20;   /* operands of a layer that goes in tiles of 128 x 128, */
constexpr int UP_WIDE_TILES = 256;         /*   if it has as many */
constexpr int UP_BAND_AREA = 1024 * 1024;  /* parameters of a layer whose tiles of 64 go in bands */
constexpr int UP_DEPTH = 2;                /* steps of 32 rows in flight; a quarter of a batch has whole pairs */
constexpr int UP_JS = 80, UP_IR = 4 * UP_JS;     /* LDS strides (floats) of a sum's 16 columns and 4 x 16 */

/* Adam's operands of a thread: column lane of rows w, w + 4, ... of a tile of W
 * whose first is parameter i0. */
constexpr int UP_E = 64 / KSPLIT;
struct AdamState {
    float p[UP_E], m[UP_E], v[UP_E];
};

__device__ inline void load_adam(const UpdateArgs &a, int64_t i0, int32_t K, AdamState &st)
{
#pragma unroll
    for (int e = 0; e < UP_E; e++) {
        const int64_t i = i0 + (int64_t)e * KSPLIT * K;
        st.p[e] = a.p[i];
        st.m[e] = a.m[i];
        st.v[e] = a.v[i];
    }
}

typedef float TileSum[16 * UP_IR];

/* Where the sum of (row, column lane) of a tile lies. */
__device__ inline uint32_t sum_at(uint32_t row, uint32_t lane)
{
    return (row / 16 * 4 + row % 4) * UP_IR + lane / 16 * UP_JS + row % 16 / 4 * 16 + lane % 16;
}

/* The gradient of a tile (row r0, column c0) of W_l in g: written out, and with
 * update Adam's step and the bf16 copies, through LDS that nobody reads any more. */
__device__ inline void finish_tile(const UpdateArgs &a, int l, int32_t r0, int32_t c0, int64_t i0,
                                   const float (&g)[UP_E], const AdamState &st, TileSum &lds)
{
    const uint32_t lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
    const int32_t N = a.n[l], K = a.k[l];
    if (a.grad)
#pragma unroll
        for (int e = 0; e < UP_E; e++) a.grad[i0 + (int64_t)e * KSPLIT * K] = g[e];
    if (!a.update) return;                                      /* uniform */
    __syncthreads();                                            /* the sums are read */
    WTile &tile = *reinterpret_cast<WTile *>(&lds[0]);
#pragma unroll
    for (int e = 0; e < UP_E; e++)
        tile[w + e * KSPLIT][lane] = f2bf(adam(a, i0 + (int64_t)e * KSPLIT * K, g[e], st.p[e], st.m[e], st.v[e]));
    __syncthreads();
    put_weights(tile, a.w + a.woff[l], a.wt + a.woff[l], N, K, r0, c0);
}

/* WIDE: some layers in tiles of 128 x 128 (UpdateArgs::wide). */
template <bool WIDE>
__global__ __launch_bounds__(UP_THREADS, 2) void mlp_update(UpdateArgs a)
{
    __shared__ __align__(16) TileSum sums[KSPLIT];
    const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1), w = __builtin_amdgcn_readfirstlane(tid / WAVE);
    if ((int32_t)blockIdx.x < a.nbias) {
        if (blockIdx.x == 0 && w == 0 && a.loss) {
            /* lane l adds partials l, l + 64, ... in order, then a fixed
             * butterfly combines the lanes */
            float s = 0.f;
#pragma unroll 4
            for (int32_t k = (int32_t)lane; k < a.nlpart; k += WAVE) {
                const float4 q = a.lpart[k];
                s += ((q.x + q.y) + q.z) + q.w;
            }
#pragma unroll
            for (int o = 1; o < WAVE; o <<= 1) s += __shfl_xor(s, o);
            if (lane == 0) *a.loss = s * a.lscale;
        }
        const int32_t b = (int32_t)blockIdx.x;
        if (b >= a.bfirst[a.nlin]) return;
        int l = 0;
        while (l + 1 < a.nlin && b >= a.bfirst[l + 1]) l++;
        const int32_t n = a.n[l], j = (b - a.bfirst[l]) * UP_THREADS + (int32_t)tid;
        if (j >= n) return;
        /* the partials in order, the two of every 64 rows first */
        const float *parts = a.bpart[l] + j;
        float g = 0.f;
#pragma unroll 32
        for (int32_t k = 0; k < a.batch / ROWS_PER_PART; k += 2)
            g += parts[(int64_t)k * n] + parts[(int64_t)(k + 1) * n];
        const int64_t i = a.boff[l] + j;
        if (a.grad) a.grad[i] = g;
        if (a.update) (void)adam(a, i, g, a.p[i], a.m[i], a.v[i]);
        return;
    }
    /* an XCD takes consecutive tiles: they share rows of dZ and of the inputs */
    const int32_t nt = a.tfirst[a.nlin], b = (int32_t)blockIdx.x - a.nbias, x = b % 8;
    const int32_t t = x * (nt / 8) + min(x, nt % 8) + b / 8;
    int l = 0;
    while (l + 1 < a.nlin && t >= a.tfirst[l + 1]) l++;
    const bool wide = WIDE && a.wide[l] != 0;                   /* uniform */
    const int32_t N = a.n[l], K = a.k[l], ti = t - a.tfirst[l], ns = a.batch / 32 / KSPLIT;
    int32_t r0, c0;
    const int32_t side = wide ? 128 : 64;
    band_tile(ti, K / side, N / side, wide ? 8 : N * K >= UP_BAND_AREA ? 4 : 1, c0, r0);
    r0 *= side;
    c0 *= side;
    /* this wavefront's 64 x 64: the tile in its quarter of the batch, or its
     * quadrant of a wide tile in all of it */
    const int32_t wr = wide ? r0 + (int32_t)w / 2 * 64 : r0, wc = wide ? c0 + (int32_t)w % 2 * 64 : c0;
    const int32_t s0 = wide ? 0 : (int32_t)w * ns;
    const uint16_t *pa = a.dzt[l] + ((int64_t)s0 * N + wr) * 32;
    const uint16_t *pb = a.act_t[l] + ((int64_t)s0 * K + wc) * 32;
    constexpr int D = UP_DEPTH;
    bf16x8 fa[D][4], fb[D][4];
    f32x4 acc[4][4];
    auto issue = [&](int d, int32_t s) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            fa[d][i] = *(const bf16x8 *)(pa + (int64_t)s * N * 32 + i * 512 + lane * 8u);
            fb[d][i] = *(const bf16x8 *)(pb + (int64_t)s * K * 32 + i * 512 + lane * 8u);
        }
    };
    auto mul = [&](int d) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[d][i], fb[d][j], acc[i][j], 0, 0, 0);
    };
    const int64_t i0 = a.woff[l] + (int64_t)(r0 + (int32_t)w) * K + c0 + lane;
    AdamState st;
    if (!WIDE && a.update) load_adam(a, i0, K, st);             /* arrives during the products */
    const int32_t nq = wide ? KSPLIT : 1;
    for (int32_t q = 0; q < nq; q++) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < D; d++) issue(d, d);
        for (int32_t s = D; s < ns; s += D) {
#pragma unroll
            for (int d = 0; d < D; d++) {
                mul(d);
                issue(d, s + d);
            }
        }
#pragma unroll
        for (int d = 0; d < D; d++) mul(d);
        pa += (int64_t)ns * N * 32;
        pb += (int64_t)ns * K * 32;
        /* lane holds rows 16 i + 4 (lane / 16) + r, column 16 j + lane % 16 */
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float &x = sums[w][(i * 4 + r) * UP_IR + j * UP_JS + lane];
                    x = q == 0 ? acc[i][j][r] : x + acc[i][j][r];
                }
    }
    __syncthreads();
    for (int32_t z = 0; z < nq; z++) {
        const int32_t zr = z / 2 * 64, zc = z % 2 * 64;
        const int64_t zi = i0 + (int64_t)zr * K + zc;
        if (WIDE && a.update) load_adam(a, zi, K, st);
        float g[UP_E];
#pragma unroll
        for (int e = 0; e < UP_E; e++) {
            const uint32_t o = sum_at(w + e * KSPLIT, lane);
            g[e] = 0.f;
            if (wide)
                g[e] += sums[z][o];
            else
#pragma unroll
                for (int y = 0; y < KSPLIT; y++) g[e] += sums[y][o];
        }
        finish_tile(a, l, r0 + zr, c0 + zc, zi, g, st, sums[z]);
    }
}

/* Input conversion: f32 [rows][in_dim] -> bf16 [n][kin] (zero padded). */
__global__ __launch_bounds__(256) void mlp_convert_x(const float *x, uint16_t *xb, uint16_t *xb_t,
                                                     int64_t n, int64_t rows, int32_t in_dim, int32_t kin)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * kin) return;
    const int64_t r = i / kin;
    const int32_t c = (int32_t)(i % kin);
    const uint16_t v = c < in_dim && r < rows ? f2bf(x[r * in_dim + c]) : (uint16_t)0;
    xb[i] = v;
    if (xb_t) xb_t[frag_index(c, (int32_t)r, kin)] = v;
}

struct PackArgs {
    int64_t off[MAX_LAYERS];    /* weight matrix l at off[l] in all copies */
    int32_t n[MAX_LAYERS], k[MAX_LAYERS];
    int32_t first[MAX_LAYERS + 1];   /* first 64 x 64 tile of matrix l */
    int32_t nlin;
    const float *p;              /* W_l [n][k] */
    uint16_t *w, *wt;            /* bf16 W_l and W_l^T, in fragments */
};

/* The bf16 weights and their transpose from the master, one 64 x 64 tile per
 * workgroup. */
__global__ __launch_bounds__(256) void mlp_pack(PackArgs a)
{
    __shared__ WTile t;
    int l = 0;
    while (l + 1 < a.nlin && (int32_t)blockIdx.x >= a.first[l + 1]) l++;
    const int32_t tile = blockIdx.x - a.first[l];
    const int32_t tk = a.k[l] / 64;
    const int32_t r0 = (tile / tk) * 64, c0 = (tile % tk) * 64;
    const uint32_t x = threadIdx.x & 63u;
    for (uint32_t y = threadIdx.x >> 6; y < 64; y += 4)
        t[y][x] = f2bf(a.p[a.off[l] + (int64_t)(r0 + y) * a.k[l] + c0 + x]);
    __syncthreads();
    put_weights(t, a.w + a.off[l], a.wt + a.off[l], a.n[l], a.k[l], r0, c0);
}

template <int EPI>
hipError_t gemm(const GemmArgs &g, hipStream_t st)
{
    const dim3 grid((uint32_t)(g.N / BN) * (uint32_t)(g.M / BM));
    (void)hipGetLastError();   /* the check after the launch reports it alone */
    hipLaunchKernelGGL((mlp_gemm<EPI>), grid, dim3(GEMM_THREADS), 0, st, g);
    return hipGetLastError();
}

int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

}  // namespace

struct bsim_mlp {
    bsim_mlp_config cfg{};
    int32_t nlin = 0;                 /* linear layers */
    int32_t kdim[MAX_LAYERS + 1]{};   /* padded widths: kdim[0] input, kdim[nlin] output */
    int64_t woff[MAX_LAYERS]{}, boff[MAX_LAYERS]{};
    int64_t nparam = 0;
    int32_t step = 0;                 /* Adam steps taken */
    hipStream_t stream = nullptr;
    std::vector<void *> allocs;
    float *p = nullptr, *m = nullptr, *v = nullptr, *grad = nullptr;
    uint16_t *pbf = nullptr, *pbf_t = nullptr;   /* bf16 W_l and W_l^T at woff[l], in fragments */
    uint16_t *act[MAX_LAYERS + 1]{};  /* act[0] input, act[l] hidden l (bf16) */
    float *out = nullptr, *ybat = nullptr;
    uint16_t *dz[2]{};                /* activation gradients (ping-pong) */
    uint16_t *act_t[MAX_LAYERS]{};    /* act[l] transposed, [kdim[l]][batch] in fragments */
    float *bpart[MAX_LAYERS]{};
    float *lpart = nullptr;
    uint16_t *xall = nullptr;
    float *yall = nullptr;
    int64_t ndata = 0;
    float *xstage = nullptr;          /* predict and gradient inputs (f32) */
    int32_t *rows = nullptr;          /* row indices of training steps */
    float *losses = nullptr;          /* and their losses (host memory, written by the update) */
    char *pin[2]{};                   /* host memory that the copies go through, PIN_BYTES each */
    hipEvent_t pin_done[2]{};         /* the last copy from or to it */
    uint16_t *dzt[MAX_LAYERS]{};      /* dZ of layer l's output, transposed [kdim[l+1]][batch] in fragments */
};

namespace {

int mfail(int code, const std::string &msg)
{
    g_bsim_err = msg;
    return code;
}

int hip_check(hipError_t e, const char *what)
{
    if (e == hipSuccess) return BSIM_OK;
    return mfail(BSIM_E_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

template <typename T>
int dalloc(bsim_mlp *m, T **p, int64_t count)
{
    void *q = nullptr;
    const hipError_t e = hipMalloc(&q, (size_t)std::max<int64_t>(count, 1) * sizeof(T));
    if (e != hipSuccess) {
        (void)hipGetLastError();   /* the failure is reported here, not by a later launch check */
        return hip_check(e, "hipMalloc");
    }
    m->allocs.push_back(q);
    *p = (T *)q;
    return BSIM_OK;
}

/* Copies between the caller's memory and the GPU go through two pinned buffers:
 * one piece moves over the bus while the host copies another.  The runtime's
 * own copies of pageable memory, one after the other, and the first touch of
 * the caller's pages by one thread took most of these calls; us before and
 * after: gradients of 2.6 million parameters 960 / 620, predict of 100,003 rows
 * with 200 outputs (80 MB, of which the caller's pages are now most) 14,300 /
 * 4,300.  Short copies stay with the calling thread: to wake others costs
 * more (800 KB: 110 / 95 us).  A model's first calls cost more, by the host's
 * first touch of its two buffers, a page fault per 4 KB: get_params of 3.8 MB takes
 * 750 us the first time and 200 after. */
constexpr size_t PIN_BYTES = 4u << 20;
constexpr size_t OMP_COPY_BYTES = 1u << 20;
constexpr int COPY_THREADS = 4;            /* as good as 8 or 16: the page faults of a process take turns */

void copy_bytes(void *dst, const void *src, size_t n)
{
    if (n < OMP_COPY_BYTES) {
        memcpy(dst, src, n);
        return;
    }
    constexpr size_t piece = 64u << 10;
    const int64_t np = (int64_t)((n + piece - 1) / piece);
#pragma omp parallel for schedule(static) num_threads(std::min(COPY_THREADS, omp_get_max_threads()))
    for (int64_t i = 0; i < np; i++)
        memcpy((char *)dst + i * piece, (const char *)src + i * piece, std::min(piece, n - (size_t)i * piece));
}

/* Waits until buffer b is free. */
int pin_wait(bsim_mlp *m, int b) { return hip_check(hipEventSynchronize(m->pin_done[b]), "hipEventSynchronize"); }

int to_device(bsim_mlp *m, void *dev, const void *src, size_t n)
{
    int rc = BSIM_OK;
    for (size_t o = 0, b = 0; o < n && !rc; o += PIN_BYTES, b ^= 1) {
        const size_t k = std::min(PIN_BYTES, n - o);
        if ((rc = pin_wait(m, (int)b))) break;
        copy_bytes(m->pin[b], (const char *)src + o, k);
        rc = hip_check(hipMemcpyAsync((char *)dev + o, m->pin[b], k, hipMemcpyHostToDevice, m->stream),
                       "hipMemcpyAsync");
        if (!rc) rc = hip_check(hipEventRecord(m->pin_done[b], m->stream), "hipEventRecord");
    }
    return rc;
}

/* Returns with the bytes at dst, so with the stream's work so far done. */
int to_host(bsim_mlp *m, void *dst, const void *dev, size_t n)
{
    int rc = BSIM_OK;
    const size_t np = (n + PIN_BYTES - 1) / PIN_BYTES;
    for (size_t i = 0; i <= np && !rc; i++) {
        if (i < np) {
            rc = hip_check(hipMemcpyAsync(m->pin[i & 1], (const char *)dev + i * PIN_BYTES,
                                          std::min(PIN_BYTES, n - i * PIN_BYTES), hipMemcpyDeviceToHost, m->stream),
                           "hipMemcpyAsync");
            if (!rc) rc = hip_check(hipEventRecord(m->pin_done[i & 1], m->stream), "hipEventRecord");
        }
        if (i > 0 && !rc) {
            const size_t o = (i - 1) * PIN_BYTES;
            rc = pin_wait(m, (int)((i - 1) & 1));
            if (!rc) copy_bytes((char *)dst + o, m->pin[(i - 1) & 1], std::min(PIN_BYTES, n - o));
        }
    }
    return rc;
}

/* uniform in [-1, 1) from (seed, index) */
double hash_uniform(uint64_t seed, uint64_t i)
{
    uint64_t z = seed + 0x9E3779B97F4A7C15ull * (i + 1);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) * (2.0 / 9007199254740992.0) - 1.0;
}

bool chained(const bsim_mlp *m)
{
    return *std::max_element(m->kdim, m->kdim + m->nlin + 1) <= CH_MAX;
}

/* The chain's launch: predict (f32 input xf of n rows, output in out), or
 * training (as forward and the activation gradients of backward), from the
 * resident rows or, with rows null, from xf and y. */
int chain(bsim_mlp *m, int32_t batch, bool train, const int32_t *rows, const float *xf, const float *y, int64_t n,
          float *out)
{
    const int L = m->nlin;
    ChainArgs a{};
    a.nlin = L;
    int32_t wide = 0;
    for (int l = 0; l <= L; l++) {
        a.kdim[l] = m->kdim[l];
        wide = std::max(wide, m->kdim[l]);
    }
    a.ld = wide + 8;
    a.din = m->cfg.in_dim;
    for (int l = 0; l < L; l++) {
        a.woff[l] = m->woff[l];
        a.boff[l] = m->boff[l];
        a.act_t[l] = m->act_t[l];
        a.dzt[l] = m->dzt[l];
        a.bpart[l] = m->bpart[l];
    }
    a.w = m->pbf;
    a.wt = m->pbf_t;
    a.p = m->p;
    a.xb = rows ? m->xall : nullptr;
    a.xf = xf;
    a.rows = rows;
    a.n = n;
    a.out = out;
    a.lpart = m->lpart;
    a.y = rows ? m->yall : y;
    a.ny = m->cfg.out_dim;
    a.scale = 2.0f / ((float)batch * (float)m->cfg.out_dim);
    const dim3 grid((uint32_t)(batch / CH_ROWS));
    const size_t lds = (size_t)2 * CH_ROWS * a.ld * 2 + CH_ROWS * 4;
    (void)hipGetLastError();   /* the check after the launch reports it alone */
#define CHAIN(W, TRAIN) hipLaunchKernelGGL((mlp_chain<W, TRAIN>), grid, dim3((W) * WAVE), lds, m->stream, a)
    if (wide <= CH_MAX / 2) {
        if (train) CHAIN(8, true);
        else CHAIN(8, false);
    } else {
        if (train) CHAIN(16, true);
        else CHAIN(16, false);
    }
#undef CHAIN
    return hip_check(hipGetLastError(), "chain launch");
}

/* Forward pass of a batch.  predict (train false): from act[0], fp32 output
 * in m->out.  train: the hidden activations also written transposed, and the
 * output layer forms the loss partials, dZ of the output (row-major and
 * transposed) and its bias partials against the targets (EPI_LOSS); with
 * rows, layer 0 gathers its inputs from the resident set (writing them
 * transposed) and the targets are the resident ones, else act[0] / act_t[0]
 * and y hold them. */
int forward(bsim_mlp *m, int32_t batch, bool train, const int32_t *rows = nullptr, const float *y = nullptr)
{
    const int L = m->nlin;
    for (int l = 0; l < L; l++) {
        GemmArgs g{};
        g.A = (l == 0 && rows) ? m->xall : m->act[l];
        g.arow = l == 0 ? rows : nullptr;
        g.a_t = (l == 0 && rows) ? m->act_t[0] : nullptr;
        g.lda = m->kdim[l];
        g.B = m->pbf + m->woff[l];
        g.M = batch;
        g.N = m->kdim[l + 1];
        g.K = m->kdim[l];
        g.bias = m->p + m->boff[l];
        g.ldo = m->kdim[l + 1];
        hipError_t e;
        if (l + 1 < L) {
            g.out_bf = m->act[l + 1];
            g.out_t = train ? m->act_t[l + 1] : nullptr;
            e = gemm<EPI_RELU_BF16>(g, m->stream);
        } else if (!train) {
            g.out_f = m->out;
            g.ny = m->cfg.out_dim;
            e = gemm<EPI_LINEAR_F32>(g, m->stream);
        } else {
            g.out_bf = m->dz[0];
            g.out_t = m->dzt[L - 1];
            g.bpart = m->bpart[L - 1];
            g.lpart = m->lpart;
            g.y = rows ? m->yall : y;
            g.yrow = rows;
            g.ny = m->cfg.out_dim;
            g.scale = 2.0f / ((float)batch * (float)m->cfg.out_dim);
            e = gemm<EPI_LOSS>(g, m->stream);
        }
        if (e != hipSuccess) return hip_check(e, "forward launch");
    }
    return BSIM_OK;
}

/* The activation gradients after a training forward pass (which formed dZ of
 * the output), one GEMM each down the layers: transposed copies in dzt, bias
 * partials in bpart. */
int backward(bsim_mlp *m, int32_t batch)
{
    const int L = m->nlin;
    hipError_t e;
    int cur = 0;
    for (int l = L - 1; l >= 1; l--) {
        /* dZ_{l-1} [batch][kdim[l]] = (dZ W_l) where H > 0:
         * B(n = in unit, k = out unit) = W[k][n] = W^T[n][k] */
        GemmArgs gx{};
        gx.A = m->dz[cur];
        gx.lda = m->kdim[l + 1];
        gx.B = m->pbf_t + m->woff[l];
        gx.M = batch;
        gx.N = m->kdim[l];
        gx.K = m->kdim[l + 1];
        gx.out_bf = m->dz[cur ^ 1];
        gx.ldo = m->kdim[l];
        gx.mask = m->act[l];
        gx.bpart = m->bpart[l - 1];
        gx.out_t = m->dzt[l - 1];
        e = gemm<EPI_DRELU_BF16>(gx, m->stream);
        if (e != hipSuccess) return hip_check(e, "activation-gradient launch");
        cur ^= 1;
    }
    return BSIM_OK;
}

/* Weight and bias gradients of a batch, and with update Adam's step. */
int update(bsim_mlp *m, int32_t batch, bool upd, float lr, float *grad_out, float *loss_dev)
{
    const int L = m->nlin, t = m->step + 1;
    UpdateArgs a{};
    bool any_wide = false;
    a.nlin = L;
    a.batch = batch;
    for (int l = 0; l < L; l++) {
        a.n[l] = m->kdim[l + 1];
        a.k[l] = m->kdim[l];
        const int32_t nt = (a.n[l] / 64) * (a.k[l] / 64);
        a.wide[l] = a.n[l] % 128 == 0 && a.k[l] % 128 == 0 && nt / 4 >= UP_WIDE_TILES &&
                    (int64_t)(a.n[l] + a.k[l]) * batch * 2 >= UP_WIDE_BYTES;
        any_wide |= a.wide[l] != 0;
        a.tfirst[l + 1] = a.tfirst[l] + (a.wide[l] ? nt / 4 : nt);
        a.bfirst[l + 1] = a.bfirst[l] + (a.n[l] + UP_THREADS - 1) / UP_THREADS;
        a.woff[l] = m->woff[l];
        a.boff[l] = m->boff[l];
        a.dzt[l] = m->dzt[l];
        a.act_t[l] = m->act_t[l];
        a.bpart[l] = m->bpart[l];
    }
    a.nbias = (int32_t)round_up(a.bfirst[L], 8);
    a.update = upd ? 1 : 0;
    a.lr = lr;
    a.b1 = m->cfg.beta1;
    a.b2 = m->cfg.beta2;
    a.eps = m->cfg.eps;
    a.c1 = (float)(1.0 - std::pow((double)m->cfg.beta1, t));
    a.c2 = (float)(1.0 - std::pow((double)m->cfg.beta2, t));
    a.p = m->p;
    a.m = m->m;
    a.v = m->v;
    a.grad = grad_out;
    a.w = m->pbf;
    a.wt = m->pbf_t;
    a.lpart = (const float4 *)m->lpart;
    a.nlpart = batch / BM * (m->kdim[L] / BN);
    a.lscale = 1.0f / ((float)batch * (float)m->cfg.out_dim);
    a.loss = loss_dev;
    (void)hipGetLastError();   /* the check after the launch reports it alone */
    const dim3 grid((uint32_t)(a.nbias + a.tfirst[L]));
    if (any_wide) hipLaunchKernelGGL((mlp_update<true>), grid, dim3(UP_THREADS), 0, m->stream, a);
    else hipLaunchKernelGGL((mlp_update<false>), grid, dim3(UP_THREADS), 0, m->stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_check(e, "update launch");
    if (upd) m->step++;
    return BSIM_OK;
}

int pack_weights(bsim_mlp *m)
{
    PackArgs a{};
    a.nlin = m->nlin;
    a.first[0] = 0;
    for (int l = 0; l < m->nlin; l++) {
        a.off[l] = m->woff[l];
        a.n[l] = m->kdim[l + 1];
        a.k[l] = m->kdim[l];
        a.first[l + 1] = a.first[l] + (a.n[l] / 64) * (a.k[l] / 64);
    }
    a.p = m->p;
    a.w = m->pbf;
    a.wt = m->pbf_t;
    (void)hipGetLastError();   /* the check after the launch reports it alone */
    hipLaunchKernelGGL(mlp_pack, dim3(a.first[m->nlin]), dim3(256), 0, m->stream, a);
    return hip_check(hipGetLastError(), "pack launch");
}

/* Row indices of the steps that bsim_mlp_train hands over at a time. */
int64_t train_words(const bsim_mlp *m)
{
    return std::max<int64_t>(m->cfg.max_batch, (int64_t)(PIN_BYTES / sizeof(int32_t)));
}

int check_batch(const bsim_mlp *m, int32_t batch)
{
    if (batch <= 0 || batch % TRAIN_BATCH_ALIGN != 0 || batch > m->cfg.max_batch)
        return mfail(BSIM_E_ARG, "batch must be a positive multiple of " +
                                     std::to_string(TRAIN_BATCH_ALIGN) + " and at most max_batch (" +
                                     std::to_string(m->cfg.max_batch) + ")");
    return BSIM_OK;
}

}  // namespace

extern "C" {

bsim_mlp *bsim_mlp_create(const bsim_mlp_config *cfg)
{
    if (!cfg) {
        g_bsim_err = "null config";
        return nullptr;
    }
    const bsim_mlp_config c = *cfg;
    if (c.in_dim < 1 || c.in_dim > 64 || c.hidden < 64 || c.hidden % 64 != 0 || c.hidden > 4096 ||
        c.layers < 1 || c.layers > MAX_LAYERS - 1 || c.out_dim < 1 || c.out_dim > 4096 ||
        c.max_batch < TRAIN_BATCH_ALIGN || c.max_batch % TRAIN_BATCH_ALIGN != 0 ||
        c.max_batch > (1 << 20) || !(c.beta1 >= 0.f && c.beta1 < 1.f) ||
        !(c.beta2 >= 0.f && c.beta2 < 1.f) || !(c.eps > 0.f)) {
        g_bsim_err = "invalid MLP config: in_dim 1..64, hidden a multiple of 64 up to 4096, "
                     "layers 1..9, out_dim 1..4096, max_batch a multiple of 256 up to 2^20, "
                     "0 <= beta < 1, eps > 0";
        return nullptr;
    }
    bsim_mlp *m = new (std::nothrow) bsim_mlp();
    if (!m) {
        g_bsim_err = "out of host memory";
        return nullptr;
    }
    m->cfg = c;
    m->nlin = c.layers + 1;
    m->kdim[0] = 64;
    for (int l = 1; l < m->nlin; l++) m->kdim[l] = c.hidden;
    m->kdim[m->nlin] = (int32_t)round_up(c.out_dim, 64);
    int64_t off = 0;
    for (int l = 0; l < m->nlin; l++) {
        m->woff[l] = off;
        off += (int64_t)m->kdim[l + 1] * m->kdim[l];
        m->boff[l] = off;
        off += m->kdim[l + 1];
    }
    m->nparam = off;
    auto bad = [&](int) {
        bsim_mlp_destroy(m);
        return (bsim_mlp *)nullptr;
    };
    if (hip_check(hipSetDevice(c.device), "hipSetDevice") != BSIM_OK) return bad(0);
    if (hip_check(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking), "stream") != BSIM_OK)
        return bad(0);
    const int64_t B = c.max_batch;
    int rc = dalloc(m, &m->p, m->nparam);
    if (!rc) rc = dalloc(m, &m->m, m->nparam);
    if (!rc) rc = dalloc(m, &m->v, m->nparam);
    if (!rc) rc = dalloc(m, &m->grad, m->nparam);
    if (!rc) rc = dalloc(m, &m->pbf, m->nparam);
    if (!rc) rc = dalloc(m, &m->pbf_t, m->nparam);
    for (int l = 0; l < m->nlin && !rc && !chained(m); l++) rc = dalloc(m, &m->act[l], B * m->kdim[l]);
    if (!rc && !chained(m)) rc = dalloc(m, &m->out, B * c.out_dim);
    if (!rc) rc = dalloc(m, &m->ybat, B * c.out_dim);
    int32_t wmax = 0;
    for (int l = 0; l <= m->nlin; l++) wmax = std::max(wmax, m->kdim[l]);
    if (!rc && !chained(m)) rc = dalloc(m, &m->dz[0], B * wmax);
    if (!rc && !chained(m)) rc = dalloc(m, &m->dz[1], B * wmax);
    for (int l = 0; l < m->nlin && !rc; l++) rc = dalloc(m, &m->act_t[l], B * m->kdim[l]);
    for (int l = 0; l < m->nlin && !rc; l++) {
        rc = dalloc(m, &m->bpart[l], B / ROWS_PER_PART * m->kdim[l + 1]);
        if (!rc) rc = dalloc(m, &m->dzt[l], B * m->kdim[l + 1]);
    }
    if (!rc) rc = dalloc(m, &m->lpart, B / BM * (m->kdim[m->nlin] / BN) * 4);
    if (!rc) rc = dalloc(m, &m->xstage, B * c.in_dim);
    if (!rc) rc = dalloc(m, &m->rows, train_words(m));
    if (!rc) rc = hip_check(hipHostMalloc((void **)&m->losses, (size_t)(train_words(m) / TRAIN_BATCH_ALIGN) * 4,
                                          hipHostMallocDefault), "hipHostMalloc");
    for (int b = 0; b < 2 && !rc; b++) {
        rc = hip_check(hipHostMalloc((void **)&m->pin[b], PIN_BYTES, hipHostMallocDefault), "hipHostMalloc");
        if (!rc) rc = hip_check(hipEventCreateWithFlags(&m->pin_done[b], hipEventDisableTiming), "hipEventCreate");
    }
    if (rc != BSIM_OK) return bad(0);
    /* He-uniform weights (bound sqrt(6 / fan_in)), zero biases, from the seed */
    std::vector<float> init(m->nparam, 0.f);
    for (int l = 0; l < m->nlin; l++) {
        const int32_t fan_in = l == 0 ? c.in_dim : c.hidden;
        const int32_t nrow = l + 1 == m->nlin ? c.out_dim : c.hidden;
        const double bound = std::sqrt(6.0 / fan_in);
        for (int32_t r = 0; r < nrow; r++)
            for (int32_t k = 0; k < fan_in; k++) {
                const int64_t i = m->woff[l] + (int64_t)r * m->kdim[l] + k;
                init[i] = (float)(bound * hash_uniform(c.seed, (uint64_t)i));
            }
    }
    if (bsim_mlp_set_params(m, init.data()) != BSIM_OK) return bad(0);
    return m;
}

void bsim_mlp_destroy(bsim_mlp *m)
{
    if (!m) return;
    if (m->stream) hipStreamSynchronize(m->stream);
    for (void *q : m->allocs) hipFree(q);
    for (int b = 0; b < 2; b++) {
        if (m->pin_done[b]) hipEventDestroy(m->pin_done[b]);
        if (m->pin[b]) hipHostFree(m->pin[b]);
    }
    if (m->losses) hipHostFree(m->losses);
    if (m->stream) hipStreamDestroy(m->stream);
    delete m;
}

int64_t bsim_mlp_num_params(const bsim_mlp *m) { return m ? m->nparam : -1; }

int bsim_mlp_layout(const bsim_mlp *m, int32_t *dims, int32_t cap)
{
    if (!m || !dims) return mfail(BSIM_E_ARG, "null argument");
    if (cap < m->nlin + 1) return mfail(BSIM_E_ARG, "dims capacity too small");
    for (int l = 0; l <= m->nlin; l++) dims[l] = m->kdim[l];
    return m->nlin;
}

int bsim_mlp_get_params(bsim_mlp *m, float *out)
{
    if (!m || !out) return mfail(BSIM_E_ARG, "null argument");
    return to_host(m, out, m->p, (size_t)m->nparam * sizeof(float));
}

int bsim_mlp_set_params(bsim_mlp *m, const float *in)
{
    if (!m || !in) return mfail(BSIM_E_ARG, "null argument");
    if (int rc = hip_check(hipStreamSynchronize(m->stream), "sync")) return rc;
    std::vector<float> p(in, in + m->nparam);
    /* padded positions stay zero */
    for (int l = 0; l < m->nlin; l++) {
        const int32_t fan_in = l == 0 ? m->cfg.in_dim : m->cfg.hidden;
        const int32_t nrow = l + 1 == m->nlin ? m->cfg.out_dim : m->cfg.hidden;
        for (int32_t r = 0; r < m->kdim[l + 1]; r++) {
            for (int32_t k = 0; k < m->kdim[l]; k++)
                if (r >= nrow || k >= fan_in) p[m->woff[l] + (int64_t)r * m->kdim[l] + k] = 0.f;
            if (r >= nrow) p[m->boff[l] + r] = 0.f;
        }
    }
    int rc = hip_check(hipMemcpy(m->p, p.data(), m->nparam * 4, hipMemcpyHostToDevice), "hipMemcpy");
    if (!rc) rc = pack_weights(m);
    if (!rc) rc = hip_check(hipStreamSynchronize(m->stream), "sync");
    if (!rc) rc = hip_check(hipMemset(m->m, 0, m->nparam * 4), "hipMemset");
    if (!rc) rc = hip_check(hipMemset(m->v, 0, m->nparam * 4), "hipMemset");
    m->step = 0;
    return rc;
}

int bsim_mlp_set_data(bsim_mlp *m, const float *x, const float *y, int64_t n)
{
    if (!m || !x || !y || n <= 0) return mfail(BSIM_E_ARG, "null argument or empty data set");
    if (int rc = hip_check(hipStreamSynchronize(m->stream), "sync")) return rc;
    if (m->xall) {
        for (auto it = m->allocs.begin(); it != m->allocs.end();)
            if (*it == m->xall || *it == m->yall) {
                hipFree(*it);
                it = m->allocs.erase(it);
            } else {
                ++it;
            }
        m->xall = nullptr;
        m->yall = nullptr;
        m->ndata = 0;
    }
    const int32_t kin = m->kdim[0], din = m->cfg.in_dim, dout = m->cfg.out_dim;
    if (int rc = dalloc(m, &m->xall, n * kin)) return rc;
    if (int rc = dalloc(m, &m->yall, n * dout)) return rc;
    std::vector<uint16_t> xb((size_t)(n * kin), 0);
    for (int64_t r = 0; r < n; r++)
        for (int32_t c = 0; c < din; c++) xb[r * kin + c] = f2bf(x[r * din + c]);
    int rc = hip_check(hipMemcpy(m->xall, xb.data(), xb.size() * 2, hipMemcpyHostToDevice), "hipMemcpy");
    if (!rc) rc = hip_check(hipMemcpy(m->yall, y, (size_t)(n * dout) * 4, hipMemcpyHostToDevice), "hipMemcpy");
    if (!rc) m->ndata = n;
    return rc;
}

}  // extern "C"

namespace {

int check_train(bsim_mlp *m, const int32_t *rows, int32_t steps, int32_t batch)
{
    if (!m || !rows || steps < 0) return mfail(BSIM_E_ARG, "null argument");
    if (int rc = check_batch(m, batch)) return rc;
    if (m->ndata <= 0) return mfail(BSIM_E_ARG, "no data set (bsim_mlp_set_data)");
    uint32_t most = 0;                  /* a negative index is a large one */
    for (int64_t i = 0; i < (int64_t)steps * batch; i++) most = std::max(most, (uint32_t)rows[i]);
    if (steps > 0 && (int64_t)most >= m->ndata) return mfail(BSIM_E_ARG, "row index out of range");
    return BSIM_OK;
}

/* The training steps of bsim_mlp_train and bsim_mlp_train_noalloc: the
 * minibatch row indices are in rdev (device), step s's loss goes to ldev[s]
 * (device). */
int train_steps(bsim_mlp *m, const int32_t *rdev, float *ldev, int32_t steps, int32_t batch, float lr)
{
    int rc = BSIM_OK;
    for (int32_t s = 0; s < steps && !rc; s++) {
        /* the minibatch is gathered by the first layer's GEMM and the loss */
        const int32_t *rows = rdev + (int64_t)s * batch;
        rc = chained(m) ? chain(m, batch, true, rows, nullptr, nullptr, 0, nullptr) : forward(m, batch, true, rows);
        if (!rc && !chained(m)) rc = backward(m, batch);
        if (!rc) rc = update(m, batch, true, lr, nullptr, ldev + s);
    }
    return rc;
}

/* Scratch of bsim_mlp_train_noalloc: the per-step losses (from word 0), then
 * the minibatch row indices (from word round_up(steps, 64)).  A file-scope
 * device array, one copy per GPU, held until the process ends; its address
 * on each device is taken once, with that device current, by
 * hipGetSymbolAddress (the array's name is only a host-side stand-in). */
static __device__ __align__(256) uint32_t scratch[BSIM_MLP_NOALLOC_WORDS];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
uint32_t *g_scratch_ptr[kMaxDevices] = {};

int scratch_on(int device, uint32_t **out)
{
    if (device < 0 || device >= kMaxDevices) return mfail(BSIM_E_ARG, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_check(e, "hipGetSymbolAddress(scratch)");
        g_scratch_ptr[device] = static_cast<uint32_t *>(ptr);
    }
    *out = g_scratch_ptr[device];
    return BSIM_OK;
}

}  // namespace

extern "C" {

int bsim_mlp_train(bsim_mlp *m, const int32_t *rows, int32_t steps, int32_t batch, float lr,
                   float *loss)
{
    if (int rc = check_train(m, rows, steps, batch)) return rc;
    if (steps == 0) return BSIM_OK;
    int rc = BSIM_OK;
    const int32_t some = (int32_t)(train_words(m) / batch);
    for (int32_t s = 0; s < steps && !rc; s += some) {
        const int32_t n = std::min(some, steps - s);
        rc = to_device(m, m->rows, rows + (int64_t)s * batch, (size_t)n * batch * sizeof(int32_t));
        if (!rc) rc = train_steps(m, m->rows, m->losses, n, batch, lr);
        const int src = hip_check(hipStreamSynchronize(m->stream), "sync");
        if (!rc) rc = src;
        if (!rc && loss) memcpy(loss + s, m->losses, (size_t)n * sizeof(float));
    }
    return rc;
}

int bsim_mlp_train_noalloc(bsim_mlp *m, const int32_t *rows, int32_t steps, int32_t batch,
                           float lr, float *loss)
{
    if (int rc = check_train(m, rows, steps, batch)) return rc;
    const int64_t roff = round_up(steps, 64);
    if (roff + (int64_t)steps * batch > (int64_t)BSIM_MLP_NOALLOC_WORDS)
        return mfail(BSIM_E_ARG, "bsim_mlp_train_noalloc: round_up(steps, 64) + steps * batch exceeds "
                                 "the scratch of " + std::to_string(BSIM_MLP_NOALLOC_WORDS) + " words");
    if (steps == 0) return BSIM_OK;
    int rc = hip_check(hipSetDevice(m->cfg.device), "hipSetDevice");
    uint32_t *base = nullptr;
    if (!rc) rc = scratch_on(m->cfg.device, &base);
    if (rc) return rc;
    float *ldev = reinterpret_cast<float *>(base);
    int32_t *rdev = reinterpret_cast<int32_t *>(base + roff);
    /* every word the steps read is written here first; the losses are
     * stored, not accumulated: nothing needs clearing */
    rc = hip_check(hipMemcpyAsync(rdev, rows, (size_t)steps * batch * 4, hipMemcpyHostToDevice,
                                  m->stream), "hipMemcpyAsync");
    if (!rc) rc = train_steps(m, rdev, ldev, steps, batch, lr);
    if (!rc && loss)
        rc = hip_check(hipMemcpyAsync(loss, ldev, (size_t)steps * 4, hipMemcpyDeviceToHost, m->stream),
                       "hipMemcpyAsync");
    const int src = hip_check(hipStreamSynchronize(m->stream), "sync");
    return rc ? rc : src;
}

int bsim_mlp_gradients(bsim_mlp *m, const float *x, const float *y, int32_t batch, float *grad,
                       float *loss)
{
    if (!m || !x || !y || !grad || !loss) return mfail(BSIM_E_ARG, "null argument");
    if (int rc = check_batch(m, batch)) return rc;
    const int32_t din = m->cfg.in_dim, kin = m->kdim[0];
    /* What fits a pinned buffer is read or written there by the kernels, once,
     * without a copy's launch: 4,700 parameters 95 / 31 us, 56,000 115 / 45; from
     * a million on no difference. */
    const size_t xb = (size_t)batch * din * 4, yb = (size_t)batch * m->cfg.out_dim * 4, gb = (size_t)m->nparam * 4;
    const bool in_place = xb + yb <= PIN_BYTES, out_place = gb <= PIN_BYTES;
    const float *xs = m->xstage, *ys = m->ybat;
    int rc = BSIM_OK;
    for (int b = 0; b < 2 && !rc; b++) rc = pin_wait(m, b);
    if (rc) return rc;
    if (in_place) {
        copy_bytes(m->pin[0], x, xb);
        copy_bytes(m->pin[0] + xb, y, yb);
        xs = (const float *)m->pin[0];
        ys = (const float *)(m->pin[0] + xb);
    } else {
        rc = to_device(m, m->xstage, x, xb);
        if (!rc) rc = to_device(m, m->ybat, y, yb);
        if (rc) return rc;
    }
    if (chained(m)) {
        rc = chain(m, batch, true, nullptr, xs, ys, batch, nullptr);
    } else {
        const int64_t tot = (int64_t)batch * kin;
        (void)hipGetLastError();   /* the check after the launch reports it alone */
        hipLaunchKernelGGL(mlp_convert_x, dim3((uint32_t)((tot + 255) / 256)), dim3(256), 0, m->stream,
                           xs, m->act[0], m->act_t[0], (int64_t)batch, (int64_t)batch, din, kin);
        rc = hip_check(hipGetLastError(), "convert launch");
        if (!rc) rc = forward(m, batch, true, nullptr, ys);
        if (!rc) rc = backward(m, batch);
    }
    if (!rc) rc = update(m, batch, false, 0.f, out_place ? (float *)m->pin[1] : m->grad, m->losses);
    if (!rc && !out_place) rc = to_host(m, grad, m->grad, gb);
    const int src = hip_check(hipStreamSynchronize(m->stream), "sync");
    if (rc || src) return rc ? rc : src;
    if (out_place) copy_bytes(grad, m->pin[1], gb);
    *loss = m->losses[0];
    return BSIM_OK;
}

int bsim_mlp_predict(bsim_mlp *m, const float *x, int64_t n, float *y)
{
    if (!m || !x || !y || n < 0) return mfail(BSIM_E_ARG, "null argument");
    const int32_t din = m->cfg.in_dim, kin = m->kdim[0], dout = m->cfg.out_dim;
    /* Rows at a time: as a pinned buffer holds inputs and outputs of, where the
     * chain reads and writes them (each row's values once; the copies and their
     * launches took as long or longer at every size: us for 37 rows 55 / 37, 300
     * rows 65 / 47, 4,096 rows 245 / 225).  A launch per layer works on device
     * buffers of max_batch rows. */
    const int64_t fit = (int64_t)PIN_BYTES / (4 * (din + dout)) / BM * BM;
    const int64_t B = chained(m) ? fit : std::min<int64_t>(m->cfg.max_batch, fit), nc = (n + B - 1) / B;
    const size_t in_bytes = (size_t)B * din * 4;
    int rc = BSIM_OK;
    for (int64_t c = 0; c <= nc && !rc; c++) {
        if (c < nc) {
            const int64_t rows = std::min(B, n - c * B);
            float *in = (float *)m->pin[c & 1], *out = (float *)(m->pin[c & 1] + in_bytes);
            const size_t ib = (size_t)rows * din * 4, ob = (size_t)rows * dout * 4;
            if ((rc = pin_wait(m, (int)(c & 1)))) break;
            copy_bytes(in, x + c * B * din, ib);
            if (chained(m)) {
                rc = chain(m, (int32_t)round_up(rows, CH_ROWS), false, nullptr, in, nullptr, rows, out);
            } else {
                const int32_t batch = (int32_t)round_up(rows, BM);
                const int64_t tot = (int64_t)batch * kin;
                rc = hip_check(hipMemcpyAsync(m->xstage, in, ib, hipMemcpyHostToDevice, m->stream), "hipMemcpyAsync");
                (void)hipGetLastError();   /* the check after the launch reports it alone */
                if (!rc) {
                    hipLaunchKernelGGL(mlp_convert_x, dim3((uint32_t)((tot + 255) / 256)), dim3(256), 0, m->stream,
                                       m->xstage, m->act[0], (uint16_t *)nullptr, (int64_t)batch, rows, din, kin);
                    rc = hip_check(hipGetLastError(), "convert launch");
                }
                if (!rc) rc = forward(m, batch, false);
                if (!rc) rc = hip_check(hipMemcpyAsync(out, m->out, ob, hipMemcpyDeviceToHost, m->stream),
                                        "hipMemcpyAsync");
            }
            if (!rc) rc = hip_check(hipEventRecord(m->pin_done[c & 1], m->stream), "hipEventRecord");
        }
        if (c > 0 && !rc) {
            const int64_t r0 = (c - 1) * B;
            rc = pin_wait(m, (int)((c - 1) & 1));
            if (!rc)
                copy_bytes(y + r0 * dout, m->pin[(c - 1) & 1] + in_bytes, (size_t)std::min(B, n - r0) * dout * 4);
        }
    }
    const int src = hip_check(hipStreamSynchronize(m->stream), "sync");
    return rc ? rc : src;
}

}  // extern "C"
