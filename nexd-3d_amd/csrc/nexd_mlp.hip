// libnexd_gpu.so, the nexd_mlp_* part of include/nexd_gpu.h: a multilayer
// perceptron (GELU hidden layers, linear output) trained and evaluated by
// this file's kernels.  Weights are kept in FP32 (the Adam master copy) and
// in BF16 (the GEMM operand); every product runs on the matrix cores as
// v_mfma_f32_16x16x32_bf16 with FP32 accumulation.
//
// Layer l maps in_l -> out_l:  Z = A_prev W^T + b,  A = GELU(Z) (hidden),
// Y = Z (output).  Shapes on the device are padded to multiples of 64
// (rows of the batch, every feature dimension), with zero padding that
// stays zero through training (its inputs and gradients are zero).
//
// No counterpart in the reference: this is the learned source-to-
// seismogram surrogate that is trained on, and judged by, the solver.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/nexd_gpu.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t bf16_t;   // storage of one bfloat16

// round to nearest even (inputs are finite)
__host__ __device__ inline bf16_t to_bf16(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}

// GELU with the error function, and its derivative
__device__ inline float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ inline float gelu_grad(float x) {
    const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}

// ---------------------------------------------------------------------------
// Products  C[m][n] = sum_k A[m][k] B[n][k], both operands with k contiguous
// (every tensor that meets a product along both of its dimensions is written
// by its producer in both layouts), M, N and K multiples of 64.
//
// Block of 256 threads = 4 waves in 2 x 2, block tile T x T, each wave T/2 x
// T/2 in MFMA tiles of 16 x 16.  k-tiles of 64 go through LDS as [row][k]
// with a padded row (72 bf16: the 16-byte fragment reads of 16 rows fall in
// different banks), in two buffers with one barrier per k-tile; the loads of
// the next D k-tiles are in flight in registers, whole 128-byte lines each.
// The sum over k runs in ascending order in every shape.
// A batch is a few hundred rows, so most products have few outputs and are
// bound by the latency of their loads: D k-tiles deep, and 32 x 32 tiles where
// 64 x 64 ones would leave CUs idle.  (Fragments loaded straight into
// registers, without LDS: 16 rows x 64 bytes per load, 88 us for the
// 256 x 512 outputs of K = 24,576 at any depth and tile, against 57 here and
// 450 with one k-tile of 32 ahead in 32 blocks.)
// ---------------------------------------------------------------------------
constexpr int BK = 64, LROW = BK + 8;
constexpr unsigned kXcds = 8;   // accelerator complex dies, each with its own L2

template <int T>
constexpr int product_depth() { return T == 32 ? 8 : 4; }

template <int T>
__device__ __forceinline__ void block_product(const bf16_t *A, int lda, const bf16_t *B, int ldb, int K,
                                              f32x4 (&acc)[T / 32][T / 32], bf16_t *lds) {
    constexpr int TW = T / 32, D = product_depth<T>(), NL = T / 32;   // loads of 16 bytes per operand and thread
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int wm = (w >> 1) * (T / 2), wn = (w & 1) * (T / 2);
    // thread t: row t/8 (+ 32), k chunk (t%8)*8
    const bf16_t *pa = A + (size_t)(t >> 3) * lda + (t & 7) * 8, *pb = B + (size_t)(t >> 3) * ldb + (t & 7) * 8;
    const int so = (t >> 3) * LROW + (t & 7) * 8;
    const int fo = (lane & 15) * LROW + 8 * (lane >> 4);
    const int nk = K / BK;
    u32x4 ra[D][NL], rb[D][NL];
    auto load = [&](int d, int kt) {   // past the end: the last k-tile again, not used
        const size_t k = (size_t)(kt < nk ? kt : nk - 1) * BK;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            ra[d][i] = *reinterpret_cast<const u32x4 *>(pa + (size_t)(32 * i) * lda + k);
            rb[d][i] = *reinterpret_cast<const u32x4 *>(pb + (size_t)(32 * i) * ldb + k);
        }
    };
    auto stage = [&](int d, bf16_t *s) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            *reinterpret_cast<u32x4 *>(s + so + 32 * i * LROW) = ra[d][i];
            *reinterpret_cast<u32x4 *>(s + T * LROW + so + 32 * i * LROW) = rb[d][i];
        }
    };
    // fragments: lane l holds row l%16 and k 8*(l/16) .. +8 of its tile
    auto compute = [&](const bf16_t *s) {
#pragma unroll
        for (int h = 0; h < BK / 32; ++h) {
            bf16x8 a[TW], b[TW];
#pragma unroll
            for (int i = 0; i < TW; ++i) a[i] = *reinterpret_cast<const bf16x8 *>(s + (wm + 16 * i) * LROW + fo + 32 * h);
#pragma unroll
            for (int j = 0; j < TW; ++j)
                b[j] = *reinterpret_cast<const bf16x8 *>(s + T * LROW + (wn + 16 * j) * LROW + fo + 32 * h);
#pragma unroll
            for (int i = 0; i < TW; ++i)
#pragma unroll
                for (int j = 0; j < TW; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    };
    bf16_t *buf[2] = {lds, lds + 2 * T * LROW};
    static_assert(D % 2 == 0, "the LDS buffer of k-tile kt is kt % 2");
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, d);
    // The loop has no branch but its own: with one between a load and its use
    // the compiler waits for every load in flight.
    int kt = 0;
    for (; kt + D <= nk; kt += D)
#pragma unroll
        for (int d = 0; d < D; ++d) {
            stage(d, buf[d & 1]);
            load(d, kt + D + d);
            __syncthreads();
            compute(buf[d & 1]);
        }
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (kt + d < nk) {
            stage(d, buf[d & 1]);
            __syncthreads();
            compute(buf[d & 1]);
        }
}

template <int T>
constexpr int product_lds() { return 4 * T * LROW; }   // bf16 of two buffers

enum Epi {
    EPI_BIAS_GELU = 1,    // out_f32 = acc + b; out_bf16 = GELU    (hidden layer forward)
    EPI_BIAS = 2,         // out_f32 = acc + b                     (output layer forward)
    EPI_GELU_GRAD = 3,    // g = acc * GELU'(aux); out_f32 = g, out_bf16 = g   (backward)
    EPI_MSE = 4,          // d = acc + b - target; out_f32, out_bf16 = scale * d, the sum of d^2 (training forward)
};

struct GemmArgs {
    const bf16_t *A, *B;  // [M][lda], [N][ldb], k contiguous
    int M, N, K, lda, ldb;
    float *out_f32;       // [M][ldc]
    bf16_t *out_bf16;     // [M][ldc]
    bf16_t *out_bf16_t;   // [N][ldt], the same values with m contiguous, or null
    int ldc, ldt;
    const float *bias;    // [N]
    const float *aux;     // [M][ldc] pre-activations for EPI_GELU_GRAD
    const float *target;  // [rows][ldc] dataset targets and the batch's rows (EPI_MSE)
    const int *idx;
    float scale;          // 2 / (M * N)
    float *partial;       // [blocks * 4] sums of squares
};

// Blocks are dealt round-robin to the XCDs; the tile index gives each XCD one
// contiguous range with the rows (the batch) varying fastest, so a row of B is
// read by one L2 only.
template <int T, int EPI>
__global__ void __launch_bounds__(256) layer_kernel(GemmArgs g) {
    __shared__ __align__(16) bf16_t lds[product_lds<T>()];
    constexpr int TW = T / 32;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const unsigned nb = gridDim.x, xcd = blockIdx.x % kXcds, rank = blockIdx.x / kXcds;
    const unsigned per = nb / kXcds, extra = nb % kXcds;
    const int tile = (int)(xcd * per + (xcd < extra ? xcd : extra) + rank);
    const int mtiles = g.M / T, bm0 = tile % mtiles * T, bn0 = tile / mtiles * T;
    const int m0 = bm0 + (w >> 1) * (T / 2) + 4 * (lane >> 4), n0 = bn0 + (w & 1) * (T / 2) + (lane & 15);
    // what the epilogue reads is loaded ahead of the product: the targets of
    // the batch's rows, or the pre-activations
    float ep[TW][TW][4];
    if constexpr (EPI == EPI_MSE || EPI == EPI_GELU_GRAD) {
#pragma unroll
        for (int i = 0; i < TW; ++i) {
            int row[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) row[v] = EPI == EPI_MSE ? g.idx[m0 + 16 * i + v] : m0 + 16 * i + v;
#pragma unroll
            for (int j = 0; j < TW; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    ep[i][j][v] = (EPI == EPI_MSE ? g.target : g.aux)[(size_t)row[v] * g.ldc + n0 + 16 * j];
        }
    }
    f32x4 acc[TW][TW];
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
        for (int j = 0; j < TW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    block_product<T>(g.A + (size_t)bm0 * g.lda, g.lda, g.B + (size_t)bn0 * g.ldb, g.ldb, g.K, acc, lds);
    // accumulator element v of tile (i, j): row 4*(l/16)+v, column l%16
    float sq = 0.f;
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
        for (int j = 0; j < TW; ++j) {
            const int m = m0 + 16 * i, n = n0 + 16 * j;
            const float b = EPI == EPI_GELU_GRAD ? 0.f : g.bias[n];
            bf16_t h[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const size_t o = (size_t)(m + v) * g.ldc + n;
                float x = acc[i][j][v];
                if constexpr (EPI == EPI_BIAS_GELU) {
                    x += b;
                    g.out_f32[o] = x;
                    h[v] = to_bf16(gelu(x));
                } else if constexpr (EPI == EPI_BIAS) {
                    g.out_f32[o] = x + b;
                } else if constexpr (EPI == EPI_MSE) {
                    const float d = (x + b) - ep[i][j][v];
                    sq += d * d;
                    g.out_f32[o] = g.scale * d;
                    h[v] = to_bf16(g.scale * d);
                } else {
                    x *= gelu_grad(ep[i][j][v]);
                    g.out_f32[o] = x;
                    h[v] = to_bf16(x);
                }
                if constexpr (EPI != EPI_BIAS) g.out_bf16[o] = h[v];
            }
            if constexpr (EPI != EPI_BIAS) {
                if (g.out_bf16_t)
                    *reinterpret_cast<ushort4 *>(g.out_bf16_t + (size_t)n * g.ldt + m) = ushort4{h[0], h[1], h[2], h[3]};
            }
        }
    if constexpr (EPI == EPI_MSE) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) sq += __shfl_down(sq, off, 64);
        if (lane == 0) g.partial[tile * 4 + w] = sq;
    }
}

// ---------------------------------------------------------------------------
// Gradients of every layer and, in training, the Adam step on them, in one
// launch.  Weight blocks: the 64 x 64 block of gW = dz^T . act by four waves
// (32 x 32 each, K = the batch), whose epilogue applies Adam to the values in
// its registers, so the gradient of a training step reaches memory only where
// it is asked for (the last step of a call).  Bias blocks: 64 column sums of
// dz over the batch, row after row, staged through LDS so that the loads of
// 128 rows are in flight at once.  The last block sums the loss.
// The update moves 28 bytes per weight (w, m, v and the two BF16 copies) and
// that bounds the launch.  Measured on the network above (13.4e6 weights, 256
// rows): gradients, sums and Adam 500 us in 20 launches -> 101 us in one, 0.40 GB
// at 4.0 TB/s (a large copy reaches 4.7).
//
// Adam (Kingma and Ba, 2015) with bias correction folded into the step:
// m = b1 m + (1-b1) g, v = b2 v + (1-b2) g^2, w -= lr_t m / (sqrt(v) + eps_t);
// the BF16 copies of w follow.  Padding entries are not touched and stay zero.
// ---------------------------------------------------------------------------
constexpr int kMaxLayers = 16;

struct UpdateLayer {
    const bf16_t *dzt, *actt;    // [outp][ldt], [inp][ldt]
    const float *dz;             // [B][outp]
    float *W, *gW, *mW, *vW;     // [outp][inp]
    bf16_t *Wb, *Wbt;            // [outp][inp], [inp][outp]
    float *b, *gb, *mb, *vb;     // [outp]
    int in, out, inp, outp;
    int wblock0, bblock0;        // first weight and bias block
};

struct UpdateArgs {
    UpdateLayer l[kMaxLayers];
    int nl, wblocks, bblocks;    // layers, weight blocks and bias blocks of all of them
    int B, ldt;
    int train, store;            // apply Adam; write the weight gradients
    float lr_t, b1, b2, eps_t;
    const float *partial;        // [npartial] loss partials
    int npartial;
    float inv;                   // 1 / (B * outputs)
    float *loss;
};

__device__ __forceinline__ float adam_step(float w, float gi, float &m, float &v, float lr_t, float b1, float b2, float eps_t) {
    // the fused operations are written out: a last-bit change of a moment
    // turns BF16 roundings over and a training run takes another path
#pragma clang fp contract(off)
    const float mi = __builtin_fmaf(1.f - b1, gi, b1 * m);
    const float vi = __builtin_fmaf(gi, (1.f - b2) * gi, b2 * v);
    m = mi;
    v = vi;
    return w - lr_t * mi / (sqrtf(vi) + eps_t);
}

// The product is formed transposed (rows: inputs), so that a lane's four
// accumulator elements are consecutive weights: w, m and v move as 16 bytes
// per lane.
__device__ __forceinline__ void update_weights(const UpdateArgs &a, const UpdateLayer &L, int blk, bf16_t *lds) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int nbi = L.inp / 64;
    const int o0 = blk / nbi * 64, c0 = blk % nbi * 64;
    // element v of tile (i, j): input c + 16 i + v of output o + 16 j
    const int c = c0 + (w >> 1) * 32 + 4 * (lane >> 4), o = o0 + (w & 1) * 32 + (lane & 15);
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    block_product<64>(L.actt + (size_t)c0 * a.ldt, a.ldt, L.dzt + (size_t)o0 * a.ldt, a.ldt, a.B, acc, lds);
    if (a.store) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) *reinterpret_cast<f32x4 *>(L.gW + (size_t)(o + 16 * j) * L.inp + c + 16 * i) = acc[i][j];
    }
    if (!a.train) return;
    // after the product: its registers are free, and four blocks per CU cover
    // the round trip (loaded ahead of it, at two: 119 against 106 us)
    f32x4 wv[2][2], mv[2][2], vv[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const size_t at = (size_t)(o + 16 * j) * L.inp + c + 16 * i;
            wv[i][j] = *reinterpret_cast<const f32x4 *>(L.W + at);
            mv[i][j] = *reinterpret_cast<const f32x4 *>(L.mW + at);
            vv[i][j] = *reinterpret_cast<const f32x4 *>(L.vW + at);
        }
    // the [input][output] copy goes through LDS to whole 128-byte lines
    constexpr int TROW = 64 + 8;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const size_t at = (size_t)(o + 16 * j) * L.inp + c + 16 * i;
            f32x4 wn = wv[i][j], mn = mv[i][j], vn = vv[i][j];
            bf16_t h[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                // padding keeps its zeros
                float m = mn[v], s = vn[v];
                const float x = adam_step(wn[v], acc[i][j][v], m, s, a.lr_t, a.b1, a.b2, a.eps_t);
                const bool on = o + 16 * j < L.out && c + 16 * i + v < L.in;
                wn[v] = on ? x : 0.f;
                mn[v] = on ? m : 0.f;
                vn[v] = on ? s : 0.f;
                h[v] = to_bf16(wn[v]);
                lds[(c - c0 + 16 * i + v) * TROW + o - o0 + 16 * j] = h[v];
            }
            *reinterpret_cast<f32x4 *>(L.W + at) = wn;
            *reinterpret_cast<f32x4 *>(L.mW + at) = mn;
            *reinterpret_cast<f32x4 *>(L.vW + at) = vn;
            *reinterpret_cast<ushort4 *>(L.Wb + at) = ushort4{h[0], h[1], h[2], h[3]};
        }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int row = (t >> 3) + 32 * r, k = (t & 7) * 8;
        *reinterpret_cast<u32x4 *>(L.Wbt + (size_t)(c0 + row) * L.outp + o0 + k) =
            *reinterpret_cast<const u32x4 *>(lds + row * TROW + k);
    }
}

constexpr int kSumRows = 128;   // rows of a bias block in LDS

__device__ void update_bias(const UpdateArgs &a, const UpdateLayer &L, int blk, float (*rows)[64]) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, c = blk * 64 + lane;
    float s = 0.f;
    for (int r0 = 0; r0 < a.B; r0 += kSumRows) {
        float x[kSumRows / 4];
#pragma unroll
        for (int r = 0; r < kSumRows / 4; ++r) {
            const int row = r0 + 4 * r + w;
            x[r] = L.dz[(size_t)(row < a.B ? row : 0) * L.outp + c];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kSumRows / 4; ++r) rows[4 * r + w][lane] = x[r];
        __syncthreads();
        if (w == 0) {
            const int n = a.B - r0 < kSumRows ? a.B - r0 : kSumRows;   // a multiple of 64
            for (int r = 0; r < n; r += 16)
#pragma unroll
                for (int u = 0; u < 16; ++u) s += rows[r + u][lane];
        }
    }
    if (w != 0) return;
    L.gb[c] = s;
    if (!a.train || c >= L.out) return;
    float m = L.mb[c], v = L.vb[c];
    L.b[c] = adam_step(L.b[c], s, m, v, a.lr_t, a.b1, a.b2, a.eps_t);
    L.mb[c] = m;
    L.vb[c] = v;
}

__global__ void __launch_bounds__(256, 4) update_kernel(UpdateArgs a) {
    __shared__ __align__(16) char shared[product_lds<64>() * sizeof(bf16_t)];
    float(*rows)[64] = reinterpret_cast<float(*)[64]>(shared);
    static_assert(sizeof(shared) >= kSumRows * 64 * sizeof(float), "the rows of a bias block must fit");
    const int blk = blockIdx.x;
    if (blk < a.wblocks) {
        int l = 0;
        while (l + 1 < a.nl && blk >= a.l[l + 1].wblock0) ++l;
        update_weights(a, a.l[l], blk - a.l[l].wblock0, reinterpret_cast<bf16_t *>(shared));
    } else if (blk < a.wblocks + a.bblocks) {
        const int bb = blk - a.wblocks;
        int l = 0;
        while (l + 1 < a.nl && bb >= a.l[l + 1].bblock0) ++l;
        update_bias(a, a.l[l], bb - a.l[l].bblock0, rows);
    } else {
        // fixed-order sum of the loss partials
        float *red = &rows[0][0];
        float s = 0.f;
        for (int i = threadIdx.x; i < a.npartial; i += 256) s += a.partial[i];
        red[threadIdx.x] = s;
        __syncthreads();
        for (int k = 128; k > 0; k >>= 1) {
            if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
            __syncthreads();
        }
        if (threadIdx.x == 0) *a.loss = red[0] * a.inv;
    }
}

// ---------------------------------------------------------------------------
// element-wise and reduction kernels
// ---------------------------------------------------------------------------
// rows of an FP32 batch [rows][cols] (host layout) into a padded BF16 [rows][ldp]
__global__ void pack_rows_kernel(const float *src, int rows, int cols, bf16_t *dst, int ldp) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)rows * ldp) return;
    const int r = (int)(i / ldp), c = (int)(i % ldp);
    dst[i] = c < cols ? to_bf16(src[(size_t)r * cols + c]) : (bf16_t)0;
}

// gathers batch rows idx[0..B) of a dataset [n][cols] (device) into padded
// BF16, in both layouts
__global__ void gather_rows_kernel(const float *src, const int *idx, int B, int cols, bf16_t *dst, int ldp, bf16_t *dstt,
                                   int ldt) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)B * ldp) return;
    const int r = (int)(i / ldp), c = (int)(i % ldp);
    const bf16_t h = c < cols ? to_bf16(src[(size_t)idx[r] * cols + c]) : (bf16_t)0;
    dst[i] = h;
    dstt[(size_t)c * ldt + r] = h;
}

// the two BF16 copies of a weight matrix [rows][cols]
__global__ void to_bf16_kernel(const float *src, int rows, int cols, bf16_t *dst, bf16_t *dstt) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)rows * cols) return;
    const bf16_t h = to_bf16(src[i]);
    dst[i] = h;
    dstt[i % cols * rows + i / cols] = h;
}

int pad64(int x) { return (x + 63) / 64 * 64; }

}  // namespace

// ===========================================================================
// the network object
// ===========================================================================
struct nexd_mlp {
    int nl = 0;                       // layers
    std::vector<int> in, out;         // true widths
    std::vector<int> inp, outp;       // padded widths
    int max_batch = 0, device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    std::string err;
    std::vector<void *> allocs;
    // per layer
    std::vector<float *> W, b, gW, gb, mW, vW, mb, vb;
    std::vector<bf16_t *> Wb, Wbt;    // [outp][inp] and [inp][outp]
    // activations: act[0] = input (bf16), act[l+1] = GELU(Z_l) (bf16), Z[l] f32
    // (the last one: the outputs); actt with the batch contiguous, [inp_l][max_batch]
    std::vector<bf16_t *> act, actt;
    std::vector<float *> Z;
    std::vector<float *> dz;          // f32 gradient w.r.t. Z_l
    std::vector<bf16_t *> dzb, dzt;   // bf16 copies (GEMM operands), dzt [outp][max_batch]
    float *partial = nullptr;
    float *xin = nullptr;             // [max_batch][in_0] FP32 inputs of nexd_mlp_forward
    // dataset
    float *dx = nullptr, *dt = nullptr;
    int dn = 0;
    int *idx = nullptr;               // rows of the batches of one call
    size_t idx_cap = 0;
    float *losses = nullptr;          // loss of each step of one call
    size_t loss_cap = 0;
    int adam_t = 0;
    float last_ms = 0.f;
};

namespace {

int mfail(nexd_mlp *m, int code, const std::string &s) {
    m->err = s;
    return code;
}

#define MCHK(m, expr)                                                                         \
    do {                                                                                      \
        hipError_t _e = (expr);                                                               \
        if (_e != hipSuccess) return mfail(m, NEXD_E_HIP, std::string(#expr ": ") + hipGetErrorString(_e)); \
    } while (0)

template <typename T>
int malloc_zero(nexd_mlp *m, T **p, size_t n) {
    void *v = nullptr;
    MCHK(m, hipMalloc(&v, (n ? n : 1) * sizeof(T)));
    m->allocs.push_back(v);
    MCHK(m, hipMemset(v, 0, (n ? n : 1) * sizeof(T)));
    *p = static_cast<T *>(v);
    return 0;
}

unsigned nblk(size_t n, unsigned b = 256) { return (unsigned)((n + b - 1) / b); }

// 64 x 64 tiles where they give every CU a block, else 32 x 32.  256 x 24,576
// outputs of K = 512 with the loss: 37 us with 64 x 64 tiles (1,536 blocks), 57
// with 32 x 32; 256 x 512 outputs of K = 512: 9.5 with 64 x 64 (32 blocks, one
// k-tile ahead), 4.6 with 32 x 32.
constexpr int kFillBlocks = 256;

bool small_tiles(int M, int N) { return (M / 64) * (N / 64) < kFillBlocks; }
int product_blocks(int M, int N) { return (M / 64) * (N / 64) * (small_tiles(M, N) ? 4 : 1); }

template <int EPI>
void product(nexd_mlp *m, const GemmArgs &g) {
    const dim3 grid(product_blocks(g.M, g.N));
    if (small_tiles(g.M, g.N)) hipLaunchKernelGGL((layer_kernel<32, EPI>), grid, dim3(256), 0, m->stream, g);
    else hipLaunchKernelGGL((layer_kernel<64, EPI>), grid, dim3(256), 0, m->stream, g);
}

// Forward pass of a batch already in act[0] (B rows).  rows: the batch's
// dataset rows (device) in training, whose last layer goes on to the loss
// partials and dz; null: the outputs go to Z.
void forward(nexd_mlp *m, int B, const int *rows) {
    for (int l = 0; l < m->nl; ++l) {
        GemmArgs g{};
        g.A = m->act[l]; g.lda = m->inp[l];
        g.B = m->Wb[l]; g.ldb = m->inp[l];
        g.M = B; g.N = m->outp[l]; g.K = m->inp[l];
        g.ldc = m->outp[l]; g.ldt = m->max_batch; g.bias = m->b[l];
        if (l + 1 < m->nl) {
            g.out_f32 = m->Z[l];
            g.out_bf16 = m->act[l + 1];
            g.out_bf16_t = rows ? m->actt[l + 1] : nullptr;
            product<EPI_BIAS_GELU>(m, g);
        } else if (rows) {
            g.out_f32 = m->dz[l]; g.out_bf16 = m->dzb[l]; g.out_bf16_t = m->dzt[l];
            g.target = m->dt; g.idx = rows;
            g.scale = 2.0f / (float)((size_t)B * m->out[l]);
            g.partial = m->partial;
            product<EPI_MSE>(m, g);
        } else {
            g.out_f32 = m->Z[l];
            product<EPI_BIAS>(m, g);
        }
    }
}

// Backward pass from dz[nl-1]: dz of the hidden layers, then the gradients of
// every layer with, in training, their Adam step; loss: where the batch's
// loss goes.  The weights change only after every dz that reads them.
void backward(nexd_mlp *m, int B, UpdateArgs &u, bool store, float *loss) {
    for (int l = m->nl - 1; l > 0; --l) {
        // dz_{l-1} = (dz_l . W_l) * GELU'(Z_{l-1})
        GemmArgs h{};
        h.A = m->dzb[l]; h.lda = m->outp[l];
        h.B = m->Wbt[l]; h.ldb = m->outp[l];
        h.M = B; h.N = m->inp[l]; h.K = m->outp[l];
        h.out_f32 = m->dz[l - 1]; h.out_bf16 = m->dzb[l - 1]; h.out_bf16_t = m->dzt[l - 1];
        h.ldc = m->inp[l]; h.ldt = m->max_batch;
        h.aux = m->Z[l - 1];
        product<EPI_GELU_GRAD>(m, h);
    }
    u.nl = m->nl;
    u.wblocks = u.bblocks = 0;
    for (int l = 0; l < m->nl; ++l)
        u.l[l] = UpdateLayer{m->dzt[l], m->actt[l], m->dz[l], m->W[l], m->gW[l], m->mW[l], m->vW[l], m->Wb[l],
                             m->Wbt[l], m->b[l], m->gb[l], m->mb[l], m->vb[l], m->in[l], m->out[l], m->inp[l],
                             m->outp[l], 0, 0};
    for (int l = 0; l < m->nl; ++l) {
        u.l[l].wblock0 = u.wblocks;
        u.l[l].bblock0 = u.bblocks;
        u.wblocks += (m->outp[l] / 64) * (m->inp[l] / 64);
        u.bblocks += m->outp[l] / 64;
    }
    u.B = B; u.ldt = m->max_batch;
    u.store = store;
    const int L = m->nl - 1;
    u.partial = m->partial;
    u.npartial = 4 * product_blocks(B, m->outp[L]);
    u.inv = 1.0f / ((float)B * (float)m->out[L]);
    u.loss = loss;
    hipLaunchKernelGGL(update_kernel, dim3(u.wblocks + u.bblocks + 1), dim3(256), 0, m->stream, u);
}

// the Adam step's constants, counted
void adam(nexd_mlp *m, float lr, float b1, float b2, float eps, UpdateArgs &u) {
    m->adam_t += 1;
    const double c1 = 1.0 - std::pow((double)b1, m->adam_t), c2 = 1.0 - std::pow((double)b2, m->adam_t);
    u.train = 1;
    u.lr_t = (float)(lr * std::sqrt(c2) / c1);
    u.eps_t = (float)(eps * std::sqrt(c2));
    u.b1 = b1;
    u.b2 = b2;
}

int check_batch(nexd_mlp *m, int B) {
    if (B <= 0 || B % 64 != 0 || B > m->max_batch)
        return mfail(m, NEXD_E_ARG, "batch must be a positive multiple of 64, at most max_batch");
    return 0;
}

}  // namespace

static std::string g_mlp_create_error;

extern "C" {

int nexd_mlp_create(int nlayers, const int *widths, int max_batch, int device, nexd_mlp **out) {
    if (!out || !widths || nlayers < 1 || nlayers > 16) { g_mlp_create_error = "bad arguments"; return NEXD_E_ARG; }
    *out = nullptr;
    if (max_batch <= 0 || max_batch % 64) { g_mlp_create_error = "max_batch must be a positive multiple of 64"; return NEXD_E_ARG; }
    for (int i = 0; i <= nlayers; ++i)
        if (widths[i] <= 0) { g_mlp_create_error = "widths must be positive"; return NEXD_E_ARG; }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) {
        g_mlp_create_error = "no such HIP device";
        return NEXD_E_HIP;
    }
    nexd_mlp *m = new nexd_mlp();
    m->nl = nlayers;
    m->max_batch = max_batch;
    m->device = device;
    auto bail = [&](int rc) { g_mlp_create_error = m->err; nexd_mlp_destroy(m); return rc; };
    if (hipSetDevice(device) != hipSuccess || hipStreamCreate(&m->stream) != hipSuccess ||
        hipEventCreate(&m->ev0) != hipSuccess || hipEventCreate(&m->ev1) != hipSuccess)
        return bail(mfail(m, NEXD_E_HIP, "stream/event creation failed"));
    for (int l = 0; l < nlayers; ++l) {
        m->in.push_back(widths[l]);
        m->out.push_back(widths[l + 1]);
        m->inp.push_back(pad64(widths[l]));
        m->outp.push_back(pad64(widths[l + 1]));
    }
    const int L = nlayers;
    m->W.assign(L, nullptr); m->b.assign(L, nullptr); m->gW.assign(L, nullptr); m->gb.assign(L, nullptr);
    m->mW.assign(L, nullptr); m->vW.assign(L, nullptr); m->mb.assign(L, nullptr); m->vb.assign(L, nullptr);
    m->Wb.assign(L, nullptr); m->Wbt.assign(L, nullptr);
    m->act.assign(L + 1, nullptr); m->actt.assign(L, nullptr); m->Z.assign(L, nullptr);
    m->dz.assign(L, nullptr); m->dzb.assign(L, nullptr); m->dzt.assign(L, nullptr);
    int rc = 0;
    for (int l = 0; l < L && !rc; ++l) {
        const size_t nw = (size_t)m->outp[l] * m->inp[l], no = m->outp[l];
        (rc = malloc_zero(m, &m->W[l], nw)) || (rc = malloc_zero(m, &m->b[l], no)) ||
            (rc = malloc_zero(m, &m->gW[l], nw)) || (rc = malloc_zero(m, &m->gb[l], no)) ||
            (rc = malloc_zero(m, &m->mW[l], nw)) || (rc = malloc_zero(m, &m->vW[l], nw)) ||
            (rc = malloc_zero(m, &m->mb[l], no)) || (rc = malloc_zero(m, &m->vb[l], no)) ||
            (rc = malloc_zero(m, &m->Wb[l], nw)) || (rc = malloc_zero(m, &m->Wbt[l], nw)) ||
            (rc = malloc_zero(m, &m->Z[l], (size_t)max_batch * no)) ||
            (rc = malloc_zero(m, &m->dz[l], (size_t)max_batch * no)) ||
            (rc = malloc_zero(m, &m->dzb[l], (size_t)max_batch * no)) ||
            (rc = malloc_zero(m, &m->dzt[l], (size_t)max_batch * no)) ||
            (rc = malloc_zero(m, &m->act[l + 1], (size_t)max_batch * no)) ||
            (rc = malloc_zero(m, &m->actt[l], (size_t)max_batch * m->inp[l]));
    }
    if (!rc) rc = malloc_zero(m, &m->act[0], (size_t)max_batch * m->inp[0]);
    // a wave per 16 x 16 outputs at most (32 x 32 tiles)
    if (!rc) (rc = malloc_zero(m, &m->partial, (size_t)(max_batch / 16) * (m->outp[L - 1] / 16))) ||
             (rc = malloc_zero(m, &m->xin, (size_t)max_batch * m->in[0]));
    if (rc) return bail(rc);
    *out = m;
    return NEXD_OK;
}

int nexd_mlp_set_params(nexd_mlp *m, int layer, const float *W, const float *b) {
    if (!m || !W || !b || layer < 0 || layer >= m->nl) return m ? mfail(m, NEXD_E_ARG, "bad layer or null") : NEXD_E_ARG;
    MCHK(m, hipSetDevice(m->device));
    const int o = m->out[layer], i = m->in[layer], ip = m->inp[layer];
    std::vector<float> wp((size_t)m->outp[layer] * ip, 0.f), bp(m->outp[layer], 0.f);
    for (int r = 0; r < o; ++r) {
        for (int c = 0; c < i; ++c) wp[(size_t)r * ip + c] = W[(size_t)r * i + c];
        bp[r] = b[r];
    }
    MCHK(m, hipMemcpy(m->W[layer], wp.data(), wp.size() * 4, hipMemcpyHostToDevice));
    MCHK(m, hipMemcpy(m->b[layer], bp.data(), bp.size() * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(to_bf16_kernel, dim3(nblk(wp.size())), dim3(256), 0, m->stream, m->W[layer], m->outp[layer], ip,
                       m->Wb[layer], m->Wbt[layer]);
    // a new parameter set restarts the optimiser
    MCHK(m, hipMemsetAsync(m->mW[layer], 0, wp.size() * 4, m->stream));
    MCHK(m, hipMemsetAsync(m->vW[layer], 0, wp.size() * 4, m->stream));
    MCHK(m, hipMemsetAsync(m->mb[layer], 0, bp.size() * 4, m->stream));
    MCHK(m, hipMemsetAsync(m->vb[layer], 0, bp.size() * 4, m->stream));
    m->adam_t = 0;
    MCHK(m, hipStreamSynchronize(m->stream));
    return NEXD_OK;
}

// which: 0 the FP32 weights and biases, 1 their gradients of the last
// nexd_mlp_gradients / training step
// Rows of n of their stride values into the caller's array.  Without padding
// they are copied there directly: a vector between, zeroed and copied again, took
// a fifth of an inference of 256 x 24,576 outputs (3.7 -> 3.0 ms) and 4 of the 37 ms
// of 128 training steps and their weights' fetch.
static int fetch_rows(nexd_mlp *m, float *out, const float *dev, int rows, int n, int stride) {
    if (n == stride) {
        MCHK(m, hipMemcpy(out, dev, (size_t)rows * n * 4, hipMemcpyDeviceToHost));
        return NEXD_OK;
    }
    std::vector<float> h((size_t)rows * stride);
    MCHK(m, hipMemcpy(h.data(), dev, h.size() * 4, hipMemcpyDeviceToHost));
    for (int r = 0; r < rows; ++r) std::memcpy(out + (size_t)r * n, h.data() + (size_t)r * stride, (size_t)n * 4);
    return NEXD_OK;
}

int nexd_mlp_get_params(nexd_mlp *m, int layer, int which, float *W, float *b) {
    if (!m || layer < 0 || layer >= m->nl || (which != 0 && which != 1)) return m ? mfail(m, NEXD_E_ARG, "bad argument") : NEXD_E_ARG;
    MCHK(m, hipSetDevice(m->device));
    MCHK(m, hipStreamSynchronize(m->stream));
    const int o = m->out[layer], i = m->in[layer], ip = m->inp[layer];
    if (W) {
        int rc = fetch_rows(m, W, which ? m->gW[layer] : m->W[layer], o, i, ip);
        if (rc) return rc;
    }
    if (b) MCHK(m, hipMemcpy(b, which ? m->gb[layer] : m->b[layer], (size_t)o * 4, hipMemcpyDeviceToHost));
    return NEXD_OK;
}

int nexd_mlp_forward(nexd_mlp *m, const float *x, int B, float *y) {
    if (!m || !x || !y) return m ? mfail(m, NEXD_E_ARG, "null argument") : NEXD_E_ARG;
    int rc = check_batch(m, B);
    if (rc) return rc;
    MCHK(m, hipSetDevice(m->device));
    MCHK(m, hipMemcpyAsync(m->xin, x, (size_t)B * m->in[0] * 4, hipMemcpyHostToDevice, m->stream));
    hipLaunchKernelGGL(pack_rows_kernel, dim3(nblk((size_t)B * m->inp[0])), dim3(256), 0, m->stream, m->xin, B,
                       m->in[0], m->act[0], m->inp[0]);
    forward(m, B, nullptr);
    MCHK(m, hipStreamSynchronize(m->stream));
    MCHK(m, hipGetLastError());
    const int L = m->nl - 1, O = m->out[L], Op = m->outp[L];
    return fetch_rows(m, y, m->Z[L], B, O, Op);
}

// The training set [n][in] inputs and [n][out] targets, kept on the device.
int nexd_mlp_upload_dataset(nexd_mlp *m, const float *x, const float *t, int n) {
    if (!m || !x || !t || n <= 0) return m ? mfail(m, NEXD_E_ARG, "bad dataset") : NEXD_E_ARG;
    MCHK(m, hipSetDevice(m->device));
    if (m->dx) { (void)hipFree(m->dx); m->dx = nullptr; }
    if (m->dt) { (void)hipFree(m->dt); m->dt = nullptr; }
    const size_t ni = (size_t)n * m->in[0], no = (size_t)n * m->out[m->nl - 1];
    MCHK(m, hipMalloc(&m->dx, ni * 4));
    MCHK(m, hipMalloc(&m->dt, no * 4));
    MCHK(m, hipMemcpy(m->dx, x, ni * 4, hipMemcpyHostToDevice));
    MCHK(m, hipMemcpy(m->dt, t, no * 4, hipMemcpyHostToDevice));
    m->dn = n;
    return NEXD_OK;
}

// What a batch of dataset rows idx[0..B) has to fulfil.
static int check_rows(nexd_mlp *m, const int *idx, int B) {
    int rc = check_batch(m, B);
    if (rc) return rc;
    if (!m->dx) return mfail(m, NEXD_E_STATE, "upload a dataset first");
    for (int r = 0; r < B; ++r)
        if (idx[r] < 0 || idx[r] >= m->dn) return mfail(m, NEXD_E_ARG, "dataset row out of range");
    const int L = m->nl - 1;
    if (m->out[L] != m->outp[L]) return mfail(m, NEXD_E_UNSUPPORTED, "training needs an output width that is a multiple of 64");
    return 0;
}

// The rows of nsteps batches on the device, and room for their losses.
static int put_rows(nexd_mlp *m, const int *idx, int B, int nsteps) {
    const size_t n = (size_t)nsteps * B;
    if (n > m->idx_cap) {
        MCHK(m, hipStreamSynchronize(m->stream));
        if (m->idx) (void)hipFree(m->idx);
        m->idx = nullptr; m->idx_cap = 0;
        MCHK(m, hipMalloc(&m->idx, n * sizeof(int)));
        m->idx_cap = n;
    }
    if ((size_t)nsteps > m->loss_cap) {
        MCHK(m, hipStreamSynchronize(m->stream));
        if (m->losses) (void)hipFree(m->losses);
        m->losses = nullptr; m->loss_cap = 0;
        MCHK(m, hipMalloc(&m->losses, (size_t)nsteps * sizeof(float)));
        m->loss_cap = (size_t)nsteps;
    }
    MCHK(m, hipMemcpyAsync(m->idx, idx, n * sizeof(int), hipMemcpyHostToDevice, m->stream));
    return 0;
}

// Loss (to *loss, device) and gradients of the batch of dataset rows
// rows[0..B) (device); u says whether Adam follows.
static void batch_step(nexd_mlp *m, const int *rows, int B, UpdateArgs &u, bool store, float *loss) {
    hipLaunchKernelGGL(gather_rows_kernel, dim3(nblk((size_t)B * m->inp[0])), dim3(256), 0, m->stream, m->dx, rows, B,
                       m->in[0], m->act[0], m->inp[0], m->actt[0], m->max_batch);
    forward(m, B, rows);
    backward(m, B, u, store, loss);
}

// Loss and gradients of one batch (no update); loss = mean squared error
// over the batch's outputs.
int nexd_mlp_gradients(nexd_mlp *m, const int *idx, int B, float *loss) {
    if (!m || !idx) return m ? mfail(m, NEXD_E_ARG, "null argument") : NEXD_E_ARG;
    MCHK(m, hipSetDevice(m->device));
    int rc = check_rows(m, idx, B);
    if (rc || (rc = put_rows(m, idx, B, 1))) return rc;
    UpdateArgs u{};
    batch_step(m, m->idx, B, u, true, m->losses);
    if (loss) MCHK(m, hipMemcpyAsync(loss, m->losses, 4, hipMemcpyDeviceToHost, m->stream));
    MCHK(m, hipStreamSynchronize(m->stream));
    MCHK(m, hipGetLastError());
    return NEXD_OK;
}

// nsteps Adam steps over consecutive batches of idx (nsteps * B rows);
// losses[k] (optional) receives the loss of step k before its update.  A
// batch that cannot be taken ends the call after the steps before it.
int nexd_mlp_train(nexd_mlp *m, const int *idx, int B, int nsteps, float lr, float beta1, float beta2, float eps,
                   float *losses) {
    if (!m || !idx || nsteps <= 0) return m ? mfail(m, NEXD_E_ARG, "bad argument") : NEXD_E_ARG;
    MCHK(m, hipSetDevice(m->device));
    int bad = 0, good = 0;
    while (good < nsteps && !(bad = check_rows(m, idx + (size_t)good * B, B))) ++good;
    if (good) {
        const std::string why = m->err;
        int rc = put_rows(m, idx, B, good);
        if (rc) return rc;
        MCHK(m, hipEventRecord(m->ev0, m->stream));
        for (int s = 0; s < good; ++s) {
            UpdateArgs u{};
            adam(m, lr, beta1, beta2, eps, u);
            // the gradients that can be asked for afterwards are the last step's
            batch_step(m, m->idx + (size_t)s * B, B, u, s + 1 == good, m->losses + s);
        }
        MCHK(m, hipEventRecord(m->ev1, m->stream));
        if (losses) MCHK(m, hipMemcpyAsync(losses, m->losses, (size_t)good * 4, hipMemcpyDeviceToHost, m->stream));
        MCHK(m, hipStreamSynchronize(m->stream));
        MCHK(m, hipGetLastError());
        if (!bad) MCHK(m, hipEventElapsedTime(&m->last_ms, m->ev0, m->ev1));
        m->err = why;
    }
    return bad ? bad : NEXD_OK;
}

int nexd_mlp_last_run_ms(nexd_mlp *m, double *ms) {
    if (!m || !ms) return NEXD_E_ARG;
    *ms = m->last_ms;
    return NEXD_OK;
}

void nexd_mlp_destroy(nexd_mlp *m) {
    if (!m) return;
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    for (void *p : m->allocs) (void)hipFree(p);
    if (m->dx) (void)hipFree(m->dx);
    if (m->dt) (void)hipFree(m->dt);
    if (m->idx) (void)hipFree(m->idx);
    if (m->losses) (void)hipFree(m->losses);
    if (m->ev0) (void)hipEventDestroy(m->ev0);
    if (m->ev1) (void)hipEventDestroy(m->ev1);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
}

const char *nexd_mlp_last_error(const nexd_mlp *m) { return m ? m->err.c_str() : g_mlp_create_error.c_str(); }

}  // extern "C"
