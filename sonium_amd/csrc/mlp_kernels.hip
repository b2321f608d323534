// Learned warm start: a 4-layer MLP (64 features -> W -> W -> W -> 2) with
// BF16 weights and activations, FP32 accumulation on
// v_mfma_f32_32x32x16_bf16, trained with hand-written forward and backward
// kernels and Adam on FP32 master weights.
//
// GEMM.  One kernel computes C = A B^T for row-major BF16 A (M x K) and B
// (N x K): both operands are K-contiguous.  The products of a layer use it as
//   forward      H   = A_prev W^T          (A_prev: M x K_in,  W:  N_out x K_in)
//   input grad   dA  = dZ (W^T)^T          (dZ:     M x N_out, W^T: K_in x N_out)
//   weight grad  dW  = dZ^T (A_prev^T)^T   (dZ^T:   N_out x M, A_prev^T: K_in x M)
// and each product's elementwise work runs on its accumulators: bias, SiLU and
// its derivative (forward), the derivative's product and the bias gradient's
// partial sums (input gradient), the loss (output layer).  Activations and
// their gradients are written in both layouts, and the weight copy is kept as
// W and W^T.  Weight gradients reduce over the M samples with split K (FP32
// partials, summed in a fixed order by the parameter update).
//
// Features of a sample (c centroid, n normal, d incident direction, k):
//   c, n, d, k/12, d.n, d.c, then sin/cos(2^l pi q) for l = 0..5 and
//   q in {d.c, d.n, k/12, (k/12)(d.c)}: 12 + 48 = 60, zero padded to 64.
// Activation: SiLU.  Output: 2 values (Re, Im of the incident-phase-free
// density), padded to 64 rows in the last layer.

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <random>

#include "internal.hpp"

namespace sbh {
namespace {

#include "lowp_common.hpp"

constexpr int FEAT = 64;
constexpr int FEAT_USED = 60;
constexpr int OUT_PAD = 64;
constexpr int RAW = 10;  // c[3], n[3], d[3], k

__device__ __forceinline__ u16 to_bf16(float f) { return Half<1>::from_float(f); }
__device__ __forceinline__ float from_bf16(u16 v) { return Half<1>::to_float(v); }

__device__ __forceinline__ float silu(float x) { return x / (1.0f + expf(-x)); }

// What a product does with its accumulators (EPI_*), and the arrays it takes.
enum { EPI_PART, EPI_ACT, EPI_GRAD, EPI_OUT };
struct GemmArgs {
    const u16* A;
    const u16* B;
    int lda, ldb, M, N, K;
    int kslice;          // K range of a block (a multiple of 64), blockIdx.z the slice
    float* C;            // EPI_PART: partials, one M x N slab per slice
    const float* bias;   // EPI_ACT, EPI_OUT
    float* G;            // EPI_ACT: silu'(H), written; EPI_GRAD: the same, read (null: not kept)
    u16* Y;              // EPI_ACT: silu(H); EPI_GRAD, EPI_OUT: dZ.  M x N
    u16* YT;             // the same, N x M (null: not kept)
    float* colsum;       // EPI_GRAD, EPI_OUT: sums of dZ over each 64 or 32 rows (half a row tile), [half tile][N]
    const float* targets;
    const int64_t* idx;  // EPI_OUT: sample of each row (null: the row)
    float* out;          // EPI_OUT: M x 2
    double* loss;        // EPI_OUT: one partial per block
};

// C = A B^T on v_mfma_f32_32x32x16_bf16.  What bounds it at the training sizes
// (16384 x 512 x 512: 8.6 GFLOP against 17 MB in and, with the FP32 derivative,
// 67 MB out) is the epilogue: 84 MB at 3.2 TB/s, where a copy reaches 4.9, in
// stores of two bytes a lane and, for the transposed copy, of eight at a stride
// of M; the tile keeps the MFMAs from adding to it.  A block of four waves takes TM x TN outputs (2 x 2 waves), K in
// stages of 64 through two LDS buffers, the next stage's pieces in registers
// while one is multiplied.  LDS rows are 72 halves, so the 16-byte operand
// reads of 16 consecutive lanes fall in distinct banks.  Every output
// accumulates its products in order of k, 16 at a time, as the fused inference
// kernel does.  Lane l holds column l % 32 and, per accumulator group, four
// consecutive rows: the transposed copy is stored 8 bytes at a time.
// At 16384 x 512 x 512 the product with its epilogue takes 26 us forward and 29 us
// backward, where a product from global memory and separate elementwise passes
// took 42 + 46 and 42 + 52; a weight gradient takes 21 us instead of 42.
template <int TM, int TN, int EPI>
__global__ __launch_bounds__(BLOCK, 2) void mlp_gemm_kernel(GemmArgs g) {
    constexpr int LR = 64 + 8;
    constexpr int WM = TM / 2, WN = TN / 2, MT = WM / 32, NT = WN / 32;
    constexpr int AP = TM * 8 / BLOCK, BP = TN * 8 / BLOCK;  // 16-byte pieces per thread per stage
    __shared__ __attribute__((aligned(16))) u16 As[2][TM * LR];
    __shared__ __attribute__((aligned(16))) u16 Bs[2][TN * LR];
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wm = t >> 7, wn = (t >> 6) & 1;
    const int m0 = blockIdx.x * TM, n0 = blockIdx.y * TN;
    const int kb = blockIdx.z * g.kslice, ke = min(g.K, kb + g.kslice);
    const u16* ap = g.A + (int64_t)(m0 + (t >> 3)) * g.lda + (t & 7) * 8;
    const u16* bp = g.B + (int64_t)(n0 + (t >> 3)) * g.ldb + (t & 7) * 8;
    u32x4 ra[AP], rb[BP];
    auto load = [&](int k) {
#pragma unroll
        for (int i = 0; i < AP; ++i) ra[i] = *reinterpret_cast<const u32x4*>(ap + (int64_t)32 * i * g.lda + k);
#pragma unroll
        for (int i = 0; i < BP; ++i) rb[i] = *reinterpret_cast<const u32x4*>(bp + (int64_t)32 * i * g.ldb + k);
    };
    auto store = [&](int buf) {
        const int o = (t >> 3) * LR + (t & 7) * 8;
#pragma unroll
        for (int i = 0; i < AP; ++i) *reinterpret_cast<u32x4*>(&As[buf][o + 32 * i * LR]) = ra[i];
#pragma unroll
        for (int i = 0; i < BP; ++i) *reinterpret_cast<u32x4*>(&Bs[buf][o + 32 * i * LR]) = rb[i];
    };
    f32x16 acc[MT][NT];
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;
    load(kb);
    // the output layer's targets of this block's rows, gathered behind the product
    __shared__ float2 tg[EPI == EPI_OUT ? TM : 1];
    if (EPI == EPI_OUT && g.targets && t < TM) {
        const int64_t at = g.idx ? g.idx[m0 + t] : m0 + t;
        tg[t] = make_float2(g.targets[2 * at], g.targets[2 * at + 1]);
    }
    store(0);
    int buf = 0;
    for (int k = kb; k < ke; k += 64) {
        __syncthreads();  // this stage is in LDS, and every wave is done with the other buffer
        const bool more = k + 64 < ke;
        if (more) load(k + 64);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int ko = 16 * s + 8 * (lane >> 5);
            u32x4 av[MT], bv[NT];
#pragma unroll
            for (int a = 0; a < MT; ++a)
                av[a] = *reinterpret_cast<const u32x4*>(&As[buf][(wm * WM + 32 * a + (lane & 31)) * LR + ko]);
#pragma unroll
            for (int b = 0; b < NT; ++b)
                bv[b] = *reinterpret_cast<const u32x4*>(&Bs[buf][(wn * WN + 32 * b + (lane & 31)) * LR + ko]);
#pragma unroll
            for (int a = 0; a < MT; ++a)
#pragma unroll
                for (int b = 0; b < NT; ++b) acc[a][b] = mfma32<1>(av[a], bv[b], acc[a][b]);
        }
        buf ^= 1;
        if (more) store(buf);
    }
    // silu' of one 32 x 32 tile, loaded ahead of the stores of the tile before it
    float gv[2][16];
    auto load_grad = [&](int a, int b, float* v) {
        const float* __restrict__ p = g.G + (int64_t)(m0 + wm * WM + 32 * a + 4 * (lane >> 5)) * g.N + n0 + wn * WN +
                                      32 * b + (lane & 31);
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) v[4 * q + r] = p[(int64_t)(8 * q + r) * g.N];
    };
    if (EPI == EPI_GRAD) load_grad(0, 0, gv[0]);
    double loss = 0.0;
#pragma unroll
    for (int b = 0; b < NT; ++b) {
        const int col = n0 + wn * WN + 32 * b + (lane & 31);
        const float bias = EPI == EPI_ACT || (EPI == EPI_OUT && col < 2) ? g.bias[col] : 0.f;
        float sum = 0.f;
#pragma unroll
        for (int a = 0; a < MT; ++a) {
            const int tile = b * MT + a;
            if (EPI == EPI_GRAD && tile + 1 < MT * NT) load_grad((tile + 1) % MT, (tile + 1) / MT, gv[(tile + 1) & 1]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = m0 + wm * WM + 32 * a + 8 * q + 4 * (lane >> 5);
                u16 y[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float x = acc[a][b][4 * q + r];
                    const int64_t o = (int64_t)(row + r) * g.N + col;
                    if (EPI == EPI_PART) {
                        g.C[(int64_t)blockIdx.z * g.M * g.N + o] = x;
                    } else if (EPI == EPI_ACT) {
                        const float h = bias + x;
                        const float e = 1.0f + expf(-h);
                        y[r] = to_bf16(h / e);
                        g.Y[o] = y[r];
                        if (g.G) {
                            const float sg = 1.0f / e;
                            g.G[o] = sg * (1.0f + h * (1.0f - sg));
                        }
                    } else if (EPI == EPI_GRAD) {
                        y[r] = to_bf16(x * gv[tile & 1][4 * q + r]);
                        g.Y[o] = y[r];
                        sum += from_bf16(y[r]);
                    } else {
                        y[r] = 0;
                        if (col < 2) {
                            const float v = bias + x;
                            g.out[(int64_t)(row + r) * 2 + col] = v;
                            if (g.targets) {
                                const float2 w = tg[row + r - m0];
                                const float e = v - (col == 0 ? w.x : w.y);
                                loss += 0.5 * (double)e * (double)e;
                                y[r] = to_bf16(e / (float)g.M);
                            }
                        }
                        if (g.Y) g.Y[o] = y[r];
                        sum += from_bf16(y[r]);
                    }
                }
                if (EPI != EPI_PART && g.YT) {
                    const uint2 w = make_uint2((unsigned)y[0] | ((unsigned)y[1] << 16),
                                               (unsigned)y[2] | ((unsigned)y[3] << 16));
                    *reinterpret_cast<uint2*>(&g.YT[(int64_t)col * g.M + row]) = w;
                }
            }
        }
        if ((EPI == EPI_GRAD || EPI == EPI_OUT) && g.colsum) {
            sum += __shfl_xor(sum, 32, 64);
            if (lane < 32) g.colsum[(int64_t)(blockIdx.x * 2 + wm) * g.N + col] = sum;
        }
    }
    if (EPI == EPI_OUT && g.loss) {
        __shared__ double part[4];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
        if (lane == 0) part[t >> 6] = loss;
        __syncthreads();
        if (t == 0) g.loss[blockIdx.x] = (part[0] + part[1]) + (part[2] + part[3]);
    }
}

// Features 2j and 2j + 1 (j < 32) of one raw sample {c, n, d, k}: FEAT_USED
// used, zero padded.  The sums are explicit FMAs, so every kernel forms the
// same bits.
__device__ __forceinline__ float2 sample_feature_pair(const float* __restrict__ r, int j) {
    if (j >= FEAT_USED / 2) return make_float2(0.f, 0.f);
    const float kk = r[9] * (1.0f / 12.0f);
    const float dc = fmaf(r[8], r[2], fmaf(r[7], r[1], r[6] * r[0]));
    const float dn = fmaf(r[8], r[5], fmaf(r[7], r[4], r[6] * r[3]));
    if (j < 4) return make_float2(r[2 * j], r[2 * j + 1]);
    if (j == 4) return make_float2(r[8], kk);
    if (j == 5) return make_float2(dn, dc);
    const int a = (j - 6) / 6, l = (j - 6) % 6;
    const float q = a == 0 ? dc : a == 1 ? dn : a == 2 ? kk : kk * dc;
    const float x = (3.14159265358979f * (float)(1 << l)) * q;
    return make_float2(sinf(x), cosf(x));
}

__device__ __forceinline__ unsigned pack_bf16(float2 f) {
    return (unsigned)to_bf16(f.x) | ((unsigned)to_bf16(f.y) << 16);
}

// Sample of row s of step `seed`: hash(seed, s) mod count.
__device__ __forceinline__ int64_t sample_index(uint64_t seed, int s, int64_t count) {
    uint64_t z = seed + 0x9E3779B97F4A7C15ull * (uint64_t)(s + 1);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (int64_t)(z % (uint64_t)count);
}

// Features of M rows -> X (M x 64) and X^T (64 x M; not written when XT is null,
// as in inference).  With idx the rows are samples drawn by sample_index and
// left in idx; without it row s is sample s.  A thread takes one feature pair
// of a sample (32 threads a sample: one sine and cosine each), a block 64
// samples, whose transposed copy leaves through LDS.
constexpr int FEAT_ROWS = 64;
__global__ __launch_bounds__(BLOCK) void mlp_features_kernel(const float* __restrict__ raw, int64_t* __restrict__ idx,
                                                             uint64_t seed, int64_t count, int M,
                                                             u16* __restrict__ X, u16* __restrict__ XT) {
    __shared__ unsigned sh[FEAT_ROWS][33];
    const int s0 = blockIdx.x * FEAT_ROWS;
    const int j = threadIdx.x & 31;
#pragma unroll
    for (int i = 0; i < FEAT_ROWS * 32 / BLOCK; ++i) {
        const int r = (threadIdx.x >> 5) + i * (BLOCK / 32);
        const int s = s0 + r;
        if (s >= M) break;
        const int64_t at = idx ? sample_index(seed, s, count) : s;
        if (idx && j == 0) idx[s] = at;
        const unsigned w = pack_bf16(sample_feature_pair(raw + at * RAW, j));
        reinterpret_cast<unsigned*>(X)[(int64_t)s * (FEAT / 2) + j] = w;
        sh[r][j] = w;
    }
    if (!XT) return;
    __syncthreads();
    // 8 samples of one feature per thread and pass
#pragma unroll
    for (int i = 0; i < FEAT * (FEAT_ROWS / 8) / BLOCK; ++i) {
        const int e = threadIdx.x + i * BLOCK;
        const int f = e >> 3, r0 = (e & 7) * 8;
        if (s0 + r0 >= M) continue;  // M is a multiple of 8
        u32x4 w;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const unsigned lo = sh[r0 + 2 * v][f >> 1], hi = sh[r0 + 2 * v + 1][f >> 1];
            w[v] = (f & 1) ? (lo >> 16) | (hi & 0xffff0000u) : (lo & 0xffffu) | (hi << 16);
        }
        *reinterpret_cast<u32x4*>(&XT[(int64_t)f * M + s0 + r0]) = w;
    }
}

// One layer of the parameter update, for every layer in one launch
// (blockIdx.y): the gradient of each weight is the sum of its split-K partials
// in slice order, that of each bias the sum of its column partials.  ADAM steps
// the FP32 master parameters and refreshes the BF16 copies W and W^T; without it
// the gradients are written out.  A block takes a 32 x 32 weight tile (the
// transposed copy leaves through LDS) or, past the tiles, 32 biases.
constexpr int kSplitW = 16;  // at most so many K slices (samples) of the weight-gradient products
struct UpdateLayer {
    const float* part;    // nsplit slabs of prow x cols
    const float* colsum;  // nsum rows of prow
    int rows, cols, prow, nsum;
    int64_t w_off, b_off;
    u16* W;
    u16* WT;
};
struct UpdateArgs {
    UpdateLayer layer[4];
    int nsplit;
    float *p, *m1, *m2, *grads;
    float lr, b1, b2, eps, c1, c2;
};

__device__ __forceinline__ float adam_step(const UpdateArgs& u, int64_t t, float gr) {
    const float a = u.b1 * u.m1[t] + (1.f - u.b1) * gr;
    const float b = u.b2 * u.m2[t] + (1.f - u.b2) * gr * gr;
    u.m1[t] = a;
    u.m2[t] = b;
    const float p = u.p[t] - u.lr * (a / u.c1) / (sqrtf(b / u.c2) + u.eps);
    u.p[t] = p;
    return p;
}

template <bool ADAM>
__global__ __launch_bounds__(BLOCK) void mlp_update_kernel(UpdateArgs u) {
    const UpdateLayer& l = u.layer[blockIdx.y];
    const int tr = (l.rows + 31) / 32, tc = l.cols / 32;
    const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
    int b = blockIdx.x;
    if (b < tr * tc) {
        __shared__ u16 sh[32][34];
        const int r0 = (b / tc) * 32, c = (b % tc) * 32 + x;
        const int64_t slab = (int64_t)l.prow * l.cols;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = r0 + y + 8 * i;
            if (r < l.rows) {
                const int64_t o = (int64_t)r * l.cols + c;
                float v[kSplitW];
#pragma unroll
                for (int z = 0; z < kSplitW; ++z) v[z] = z < u.nsplit ? l.part[z * slab + o] : 0.f;
                float g = 0.f;
#pragma unroll
                for (int z = 0; z < kSplitW; ++z)
                    if (z < u.nsplit) g += v[z];
                if (ADAM) {
                    const u16 h = to_bf16(adam_step(u, l.w_off + o, g));
                    l.W[o] = h;
                    sh[y + 8 * i][x] = h;
                } else {
                    u.grads[l.w_off + o] = g;
                }
            }
        }
        if (ADAM) {
            __syncthreads();
            const int r = r0 + x;
            if (r < l.rows)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int cc = y + 8 * i;
                    l.WT[(int64_t)((b % tc) * 32 + cc) * l.prow + r] = sh[x][cc];
                }
        }
        return;
    }
    b -= tr * tc;
    if (b >= tr) return;
    __shared__ float bs[8][32];
    const int col = b * 32 + x;
    float s = 0.f;
    if (col < l.rows)
#pragma unroll 8
        for (int z = y; z < l.nsum; z += 8) s += l.colsum[(int64_t)z * l.prow + col];
    bs[y][x] = s;
    __syncthreads();
    if (y == 0 && col < l.rows) {
        float g = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) g += bs[i][x];
        if (ADAM)
            (void)adam_step(u, l.b_off + col, g);
        else
            u.grads[l.b_off + col] = g;
    }
}

// BF16 copies W (rows x cols, padded to prow rows) and W^T (cols x prow).
__global__ void mlp_cast_kernel(const float* __restrict__ w, int rows, int cols, int prow, u16* __restrict__ W,
                                u16* __restrict__ WT) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)prow * cols) return;
    const int r = (int)(t / cols), c = (int)(t % cols);
    const u16 h = r < rows ? to_bf16(w[(int64_t)r * cols + c]) : (u16)0;
    W[t] = h;
    WT[(int64_t)c * prow + r] = h;
}

inline unsigned nb(int64_t n) { return (unsigned)((n + BLOCK - 1) / BLOCK); }


// Inference through all layers: a workgroup carries INFER_ROWS samples, their
// activations held in LDS (two row-major buffers of ldr halves per row, rows
// padded by 8 halves); each wave computes 32-column tiles of a layer with
// the GEMM's operand layout and accumulation order (one MFMA per 16 inputs,
// in order), then bias + SiLU in registers, so the outputs equal the
// layer-by-layer forward pass bit for bit.  Weights stream from L2.
constexpr int INFER_ROWS = 32;
constexpr int INFER_MAX_TILES = 8;  // 32-column tiles per wave (TPW <= 8): width <= 4 * 8 * 32 = 1024
struct InferArgs {
    const u16* w[4];
    const float* b[4];
    int in[4];
    int out[4];
};

template <int TPW>
__global__ __launch_bounds__(BLOCK) void mlp_infer_kernel(const float* __restrict__ raw, InferArgs a, int ldr,
                                                          float* __restrict__ Y) {
    extern __shared__ __attribute__((aligned(16))) u16 act[];
    u16* src = act;
    u16* dst = act + INFER_ROWS * ldr;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int64_t s0 = (int64_t)blockIdx.x * INFER_ROWS;
#pragma unroll
    for (int i = 0; i < INFER_ROWS * 32 / BLOCK; ++i) {
        const int r = (threadIdx.x >> 5) + i * (BLOCK / 32), j = threadIdx.x & 31;
        *reinterpret_cast<unsigned*>(&src[r * ldr + 2 * j]) = pack_bf16(sample_feature_pair(raw + (s0 + r) * RAW, j));
    }
    __syncthreads();
    for (int l = 0; l < 4; ++l) {
        const int in = a.in[l];
        const int ntiles = (a.out[l] + 31) / 32;
        const u16* __restrict__ w = a.w[l];
        f32x16 acc[TPW];
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[t][v] = 0.f;
        const int kq = (lane >> 5) * 8;
        for (int k = 0; k < in; k += 16) {
            const u32x4 av = *reinterpret_cast<const u32x4*>(&src[(lane & 31) * ldr + k + kq]);
#pragma unroll
            for (int t = 0; t < TPW; ++t) {
                const int tile = wave + 4 * t;
                if (tile < ntiles) {
                    const u32x4 bv =
                        *reinterpret_cast<const u32x4*>(w + (int64_t)(32 * tile + (lane & 31)) * in + k + kq);
                    acc[t] = mfma32<1>(av, bv, acc[t]);
                }
            }
        }
        const float* __restrict__ bias = a.b[l];
        if (l < 3) {
#pragma unroll
            for (int t = 0; t < TPW; ++t) {
                const int tile = wave + 4 * t;
                if (tile < ntiles) {
                    const int col = 32 * tile + (lane & 31);
                    const float bc = bias[col];
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int row = 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                        dst[row * ldr + col] = to_bf16(silu(bc + acc[t][v]));
                    }
                }
            }
            __syncthreads();
            u16* tmp = src;
            src = dst;
            dst = tmp;
        } else if (wave == 0 && (lane & 31) < 2) {
            const int col = lane & 31;
            const float bc = bias[col];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                Y[(s0 + row) * 2 + col] = bc + acc[0][v];
            }
        }
    }
}

}  // namespace

// ---- host side ----

namespace mlp {

// Layer l: rows x cols weights (rows padded to prow for the last layer).
struct Layer {
    int rows, cols, prow;
    int64_t w_off, b_off;  // offsets in the FP32 parameter vector
};

}  // namespace mlp
}  // namespace sbh

struct sbh_mlp {
    sbh_context* ctx = nullptr;
    int width = 512;
    int layers = 4;
    std::vector<sbh::mlp::Layer> L;
    int64_t nparams = 0;
    sbh::DeviceArray<float> params, grads, m1, m2;
    sbh::DeviceArray<uint16_t> Wb, WTb;  // BF16 weight copies, per layer at wb_off
    std::vector<int64_t> wb_off;
    int64_t step = 0;
    // batch workspace (sized for max_batch samples)
    int max_batch = 0;
    int max_train = 0;  // and the training arrays
    sbh::WorkArray<uint16_t> X, XT;
    std::vector<sbh::WorkArray<float>> G;     // silu' of the pre-activations per hidden layer
    std::vector<sbh::WorkArray<uint16_t>> A, AT;  // activations per hidden layer
    sbh::WorkArray<uint16_t> dZ, dZT, dZ2, dZ2T;
    sbh::WorkArray<float> part, colsum, Y;  // per layer: weight-gradient and bias-gradient partials
    sbh::WorkArray<double> loss_part;
    sbh::WorkArray<int64_t> idx;
    sbh::WorkArray<float> raw_ws;  // raw inputs of device-side predictions
    // dataset
    sbh::WorkArray<float> data_in, data_out;
    int64_t data_count = 0;
};

namespace sbh {
inline sbh_context* ctx_of(const sbh_mlp* n) { return n ? n->ctx : nullptr; }
}  // namespace sbh

namespace sbh {
namespace {

constexpr int kLossSteps = 256;  // steps whose loss partials stay on the device between reads

// K slices of the weight-gradient products over M samples: whole stages of 64.
int weight_slice(int M) { return (M / 64 + kSplitW - 1) / kSplitW * 64; }
int weight_splits(int M) { return (M + weight_slice(M) - 1) / weight_slice(M); }

// The product's tile: 128 x 128, or 64 where a side is no multiple of 128 or the
// larger tiles make fewer than 192 blocks, leaving more than a quarter of the
// 256 CUs without one (batches below 6144 at width 512).
template <int EPI>
int gemm(sbh_context* ctx, const GemmArgs& g) {
    SBH_REQUIRE(g.M % 64 == 0 && g.N % 64 == 0 && g.K % 64 == 0 && g.kslice % 64 == 0,
                "MLP GEMM shape is not tile aligned");
    const int z = (g.K + g.kslice - 1) / g.kslice;
    const bool small = (int64_t)((g.M + 127) / 128) * ((g.N + 127) / 128) * z < 192;
    const bool m128 = g.M % 128 == 0 && !small, n128 = g.N % 128 == 0 && !small;
    const dim3 grid(g.M / (m128 ? 128 : 64), g.N / (n128 ? 128 : 64), z);
    if (m128 && n128)
        hipLaunchKernelGGL((mlp_gemm_kernel<128, 128, EPI>), grid, dim3(BLOCK), 0, ctx->stream, g);
    else if (m128)
        hipLaunchKernelGGL((mlp_gemm_kernel<128, 64, EPI>), grid, dim3(BLOCK), 0, ctx->stream, g);
    else if (n128)
        hipLaunchKernelGGL((mlp_gemm_kernel<64, 128, EPI>), grid, dim3(BLOCK), 0, ctx->stream, g);
    else
        hipLaunchKernelGGL((mlp_gemm_kernel<64, 64, EPI>), grid, dim3(BLOCK), 0, ctx->stream, g);
    SBH_HIP(hipGetLastError());
    return (int)grid.x;  // row tiles
}

GemmArgs gemm_args(const uint16_t* A, int lda, const uint16_t* B, int ldb, int M, int N, int K, int kslice) {
    GemmArgs g;
    std::memset(&g, 0, sizeof(g));
    g.A = reinterpret_cast<const u16*>(A);
    g.B = reinterpret_cast<const u16*>(B);
    g.lda = lda;
    g.ldb = ldb;
    g.M = M;
    g.N = N;
    g.K = K;
    g.kslice = kslice;
    return g;
}

void ensure_batch(sbh_mlp* net, int M, bool training) {
    const int W = net->width;
    if (M > net->max_batch) {
        net->max_batch = 0;  // a failed allocation below leaves no stale size
        net->max_train = 0;
        net->X.allocate((size_t)M * FEAT);
        net->A.clear();
        for (int l = 0; l < net->layers - 1; ++l) net->A.emplace_back((size_t)M * W);
        net->Y.allocate((size_t)M * 2);
        net->max_batch = M;
    }
    if (!training || M <= net->max_train) return;
    net->max_train = 0;
    net->XT.allocate((size_t)M * FEAT);
    net->G.clear();
    net->AT.clear();
    for (int l = 0; l < net->layers - 1; ++l) {
        net->G.emplace_back((size_t)M * W);
        net->AT.emplace_back((size_t)M * W);
    }
    net->dZ.allocate((size_t)M * W);
    net->dZT.allocate((size_t)M * W);
    net->dZ2.allocate((size_t)M * W);
    net->dZ2T.allocate((size_t)M * W);
    size_t weights = 0, biases = 0;
    for (const auto& ly : net->L) {
        weights += (size_t)ly.prow * ly.cols;
        biases += (size_t)ly.prow;
    }
    net->part.allocate((size_t)kSplitW * weights);
    net->colsum.allocate((size_t)(M / 32) * biases);
    net->loss_part.allocate((size_t)(M / 64) * kLossSteps);
    net->idx.allocate((size_t)M);
    net->max_train = M;
}

void refresh_weights(sbh_mlp* net) {
    for (int l = 0; l < net->layers; ++l) {
        const mlp::Layer& ly = net->L[l];
        hipLaunchKernelGGL(mlp_cast_kernel, dim3(nb((int64_t)ly.prow * ly.cols)), dim3(BLOCK), 0, net->ctx->stream,
                           net->params.ptr + ly.w_off, ly.rows, ly.cols, ly.prow,
                           reinterpret_cast<u16*>(net->Wb.ptr + net->wb_off[l]),
                           reinterpret_cast<u16*>(net->WTb.ptr + net->wb_off[l]));
        SBH_HIP(hipGetLastError());
    }
}

// Forward pass over M samples; with targets also the loss partials (one per
// row tile, at `loss`) and the backward pass, whose gradient partials are left
// for `update`.  With draw, row s takes dataset sample sample_index(seed, s,
// count).  Returns the number of loss partials (0 without targets).
int forward_backward(sbh_mlp* net, const float* raw, bool draw, uint64_t seed, int64_t count, int M,
                     const float* targets, double* loss, UpdateArgs* update) {
    sbh_context* ctx = net->ctx;
    const int W = net->width;
    const int last = net->layers - 1;
    auto u = [](uint16_t* p) { return reinterpret_cast<u16*>(p); };
    // the transposed activations, derivatives and output gradients only feed
    // the backward pass
    const bool keep = targets != nullptr;
    hipLaunchKernelGGL(mlp_features_kernel, dim3((M + FEAT_ROWS - 1) / FEAT_ROWS), dim3(BLOCK), 0, ctx->stream, raw,
                       draw ? net->idx.ptr : nullptr, seed, count, M, u(net->X.ptr), keep ? u(net->XT.ptr) : nullptr);
    SBH_HIP(hipGetLastError());
    const uint16_t* in = net->X.ptr;
    int in_dim = FEAT;
    for (int l = 0; l < last; ++l) {
        GemmArgs g = gemm_args(in, in_dim, net->Wb.ptr + net->wb_off[l], in_dim, M, W, in_dim, in_dim);
        g.bias = net->params.ptr + net->L[l].b_off;
        g.G = keep ? net->G[l].ptr : nullptr;
        g.Y = u(net->A[l].ptr);
        g.YT = keep ? u(net->AT[l].ptr) : nullptr;
        gemm<EPI_ACT>(ctx, g);
        in = net->A[l].ptr;
        in_dim = W;
    }
    GemmArgs out = gemm_args(in, W, net->Wb.ptr + net->wb_off[last], W, M, OUT_PAD, W, W);
    out.bias = net->params.ptr + net->L[last].b_off;
    out.out = net->Y.ptr;
    if (!keep) {
        gemm<EPI_OUT>(ctx, out);
        return 0;
    }
    SBH_REQUIRE(M % 256 == 0, "training batch must be a multiple of 256 samples");
    const int splits = weight_splits(M);
    std::memset(update, 0, sizeof(*update));
    update->nsplit = splits;
    float* part = net->part.ptr;
    float* colsum = net->colsum.ptr;
    for (int l = 0; l <= last; ++l) {
        const mlp::Layer& ly = net->L[l];
        UpdateLayer& ul = update->layer[l];
        ul.part = part;
        ul.colsum = colsum;
        ul.rows = ly.rows;
        ul.cols = ly.cols;
        ul.prow = ly.prow;
        ul.w_off = ly.w_off;
        ul.b_off = ly.b_off;
        ul.W = u(net->Wb.ptr + net->wb_off[l]);
        ul.WT = u(net->WTb.ptr + net->wb_off[l]);
        ul.nsum = 0;
        part += (size_t)kSplitW * ly.prow * ly.cols;
        colsum += (size_t)(M / 32) * ly.prow;
    }
    out.targets = targets;
    out.idx = draw ? net->idx.ptr : nullptr;
    out.Y = u(net->dZ.ptr);
    out.YT = u(net->dZT.ptr);
    out.colsum = const_cast<float*>(update->layer[last].colsum);
    out.loss = loss;
    const int blocks = gemm<EPI_OUT>(ctx, out);
    update->layer[last].nsum = 2 * blocks;
    // backward, last layer first; dz/dzt hold the current layer's gradient, width = its output size
    uint16_t* dz = net->dZ.ptr;
    uint16_t* dzt = net->dZT.ptr;
    uint16_t* dz_next = net->dZ2.ptr;
    uint16_t* dzt_next = net->dZ2T.ptr;
    for (int l = last; l >= 0; --l) {
        const mlp::Layer& ly = net->L[l];
        const int out_dim = ly.prow;
        const int kin = ly.cols;
        const uint16_t* prevT = l == 0 ? net->XT.ptr : net->AT[l - 1].ptr;
        // dW (out_dim x kin) = dZ^T prev ; rows >= ly.rows are padding, never read
        GemmArgs gw = gemm_args(dzt, M, prevT, M, out_dim, kin, M, weight_slice(M));
        gw.C = const_cast<float*>(update->layer[l].part);
        gemm<EPI_PART>(ctx, gw);
        if (l == 0) break;
        // dA_prev (M x kin) = dZ W  (W^T is kin x out_dim)
        GemmArgs ga = gemm_args(dz, out_dim, net->WTb.ptr + net->wb_off[l], out_dim, M, kin, out_dim, out_dim);
        ga.G = net->G[l - 1].ptr;
        ga.Y = u(dz_next);
        ga.YT = u(dzt_next);
        ga.colsum = const_cast<float*>(update->layer[l - 1].colsum);
        update->layer[l - 1].nsum = 2 * gemm<EPI_GRAD>(ctx, ga);
        std::swap(dz, dz_next);
        std::swap(dzt, dzt_next);
    }
    return blocks;
}

template <bool ADAM>
void apply_update(sbh_mlp* net, UpdateArgs& u) {
    u.p = net->params.ptr;
    u.m1 = net->m1.ptr;
    u.m2 = net->m2.ptr;
    u.grads = net->grads.ptr;
    const int W = net->width;
    const unsigned blocks = (unsigned)(W / 32 * (W / 32) + W / 32);  // the widest layer's tiles and biases
    hipLaunchKernelGGL(mlp_update_kernel<ADAM>, dim3(std::max(blocks, 64u), net->layers), dim3(BLOCK), 0,
                       net->ctx->stream, u);
    SBH_HIP(hipGetLastError());
}

// Predictions of Mp samples (a multiple of 256) into net->Y: the fused
// kernel when the width allows (every layer's tiles fit the waves' tile
// registers), else the layer-by-layer forward pass.  Same bits either way.
void infer(sbh_mlp* net, const float* raw, int Mp) {
    const int W = net->width;
    if (W > 4 * INFER_MAX_TILES * 32) {
        ensure_batch(net, Mp, false);
        forward_backward(net, raw, false, 0, 0, Mp, nullptr, nullptr, nullptr);
        return;
    }
    if ((int64_t)net->Y.count < (int64_t)Mp * 2) net->Y.allocate((size_t)Mp * 2);
    InferArgs a;
    for (int l = 0; l < 4; ++l) {
        const mlp::Layer& ly = net->L[l];
        a.w[l] = reinterpret_cast<const u16*>(net->Wb.ptr + net->wb_off[l]);
        a.b[l] = net->params.ptr + ly.b_off;
        a.in[l] = ly.cols;
        a.out[l] = ly.rows;
    }
    const int ldr = W + 8;
    const size_t lds = (size_t)2 * INFER_ROWS * ldr * sizeof(uint16_t);
    const int tiles = (W / 32 + 3) / 4;  // 32-column tiles per wave in the hidden layers
    auto launch = [&](auto kernel) {
        SBH_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)lds));
        hipLaunchKernelGGL(kernel, dim3((unsigned)(Mp / INFER_ROWS)), dim3(BLOCK), lds, net->ctx->stream, raw, a, ldr,
                           net->Y.ptr);
    };
    if (tiles <= 1)
        launch(mlp_infer_kernel<1>);
    else if (tiles <= 2)
        launch(mlp_infer_kernel<2>);
    else if (tiles <= 4)
        launch(mlp_infer_kernel<4>);
    else
        launch(mlp_infer_kernel<8>);
    SBH_HIP(hipGetLastError());
}

// Sums of `steps` steps' loss partials (blocks each, a step's at every `stride`), added in block order.
void read_losses(sbh_mlp* net, int steps, int stride, int blocks, double* out) {
    std::vector<double> h((size_t)(steps - 1) * stride + blocks);
    copy_on_stream(net->ctx, h.data(), net->loss_part.ptr, h.size() * sizeof(double), hipMemcpyDeviceToHost);
    for (int t = 0; t < steps; ++t) {
        double s = 0.0;
        for (int b = 0; b < blocks; ++b) s += h[(size_t)t * stride + b];
        out[t] = s;
    }
}

inline void use_device(sbh_context* ctx) { SBH_HIP(hipSetDevice(ctx->device)); }

}  // namespace
}  // namespace sbh

namespace sbh {

sbh_context* mlp_context(const sbh_mlp* net) { return net ? net->ctx : nullptr; }

float* mlp_raw_workspace(sbh_mlp* net, int64_t M) {
    SBH_REQUIRE(M > 0 && M <= (1 << 24), "sample count out of range");
    const int64_t Mp = (M + 255) / 256 * 256;
    if (net->raw_ws.count < (size_t)Mp * RAW) net->raw_ws.allocate((size_t)Mp * RAW);
    if (Mp > M)
        SBH_HIP(hipMemsetAsync(net->raw_ws.ptr + M * RAW, 0, (size_t)(Mp - M) * RAW * sizeof(float),
                               net->ctx->stream));
    return net->raw_ws.ptr;
}

const float* mlp_forward_device(sbh_mlp* net, const float* raw, int64_t M) {
    SBH_REQUIRE(M > 0 && M <= (1 << 24), "sample count out of range");
    const int Mp = (int)((M + 255) / 256 * 256);
    infer(net, raw, Mp);
    return net->Y.ptr;
}

}  // namespace sbh

using namespace sbh;

extern "C" {

sbh_status sbh_mlp_create(sbh_context* ctx, int32_t width, uint64_t seed, sbh_mlp** out) {
    return guard_on(ctx_of(ctx), [&] {
        SBH_REQUIRE(ctx && out, "ctx/out is null");
        SBH_REQUIRE(width >= 64 && width <= 4096 && width % 64 == 0, "width must be a multiple of 64 in 64..4096");
        use_device(ctx);
        std::unique_ptr<sbh_mlp> net(new sbh_mlp());
        net->ctx = ctx;
        net->width = width;
        const int dims[5] = {FEAT, width, width, width, 2};
        int64_t off = 0, woff = 0;
        for (int l = 0; l < 4; ++l) {
            mlp::Layer ly;
            ly.rows = dims[l + 1];
            ly.cols = dims[l];
            ly.prow = l == 3 ? OUT_PAD : dims[l + 1];
            ly.w_off = off;
            off += (int64_t)ly.rows * ly.cols;
            ly.b_off = off;
            off += ly.rows;
            net->L.push_back(ly);
            net->wb_off.push_back(woff);
            woff += (int64_t)ly.prow * ly.cols;
        }
        net->nparams = off;
        // He-uniform weights from a seeded generator, zero biases
        std::vector<float> p((size_t)off, 0.f);
        std::mt19937_64 gen(seed);
        for (const auto& ly : net->L) {
            const double bound = std::sqrt(6.0 / ly.cols) * (ly.rows == 2 ? 0.1 : 1.0);
            std::uniform_real_distribution<double> U(-bound, bound);
            for (int64_t i = 0; i < (int64_t)ly.rows * ly.cols; ++i) p[ly.w_off + i] = (float)U(gen);
        }
        net->params.allocate((size_t)off);
        net->grads.allocate((size_t)off);
        net->m1.allocate((size_t)off);
        net->m2.allocate((size_t)off);
        copy_on_stream(net->ctx, net->params.ptr, p.data(), p.size() * sizeof(float), hipMemcpyHostToDevice);
        zero_on_stream(net->ctx, net->grads.ptr, net->grads.bytes());
        zero_on_stream(net->ctx, net->m1.ptr, net->m1.bytes());
        zero_on_stream(net->ctx, net->m2.ptr, net->m2.bytes());
        net->Wb.allocate((size_t)woff);
        net->WTb.allocate((size_t)woff);
        refresh_weights(net.get());
        SBH_HIP(hipStreamSynchronize(ctx->stream));
        context_retain(ctx);
        *out = net.release();
    });
}

void sbh_mlp_destroy(sbh_mlp* net) {
    if (!net) return;
    sbh_context* ctx = net->ctx;
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    delete net;
    context_release(ctx);
}

int64_t sbh_mlp_num_params(const sbh_mlp* net) { return net ? net->nparams : 0; }

sbh_status sbh_mlp_get_params(sbh_mlp* net, float* out) {
    return guard_on(ctx_of(net), [&] {
        SBH_REQUIRE(net && out, "null argument");
        use_device(net->ctx);
        SBH_HIP(hipStreamSynchronize(net->ctx->stream));
        copy_on_stream(net->ctx, out, net->params.ptr, net->params.bytes(), hipMemcpyDeviceToHost);
    });
}

sbh_status sbh_mlp_set_params(sbh_mlp* net, const float* in) {
    return guard_on(ctx_of(net), [&] {
        SBH_REQUIRE(net && in, "null argument");
        use_device(net->ctx);
        SBH_HIP(hipStreamSynchronize(net->ctx->stream));
        copy_on_stream(net->ctx, net->params.ptr, in, net->params.bytes(), hipMemcpyHostToDevice);
        refresh_weights(net);
        SBH_HIP(hipStreamSynchronize(net->ctx->stream));
    });
}

sbh_status sbh_mlp_loss_and_gradients(sbh_mlp* net, const float* inputs, const float* targets, int64_t M,
                                      double* loss, float* grads) {
    return guard_on(ctx_of(net), [&] {
        SBH_REQUIRE(net && inputs && targets, "null argument");
        SBH_REQUIRE(M > 0 && M % 256 == 0 && M <= (1 << 24), "M must be a positive multiple of 256");
        use_device(net->ctx);
        ensure_batch(net, (int)M, true);
        WorkArray<float> din((size_t)M * RAW), dout((size_t)M * 2);
        copy_on_stream(net->ctx, din.ptr, inputs, din.bytes(), hipMemcpyHostToDevice);
        copy_on_stream(net->ctx, dout.ptr, targets, dout.bytes(), hipMemcpyHostToDevice);
        UpdateArgs u;
        const int blocks =
            forward_backward(net, din.ptr, false, 0, 0, (int)M, dout.ptr, net->loss_part.ptr, &u);
        apply_update<false>(net, u);
        double l = 0.0;
        read_losses(net, 1, blocks, blocks, &l);
        if (loss) *loss = l / (double)M;
        if (grads) copy_on_stream(net->ctx, grads, net->grads.ptr, net->grads.bytes(), hipMemcpyDeviceToHost);
    });
}

sbh_status sbh_mlp_set_dataset(sbh_mlp* net, const float* inputs, const float* targets, int64_t count) {
    return guard_on(ctx_of(net), [&] {
        SBH_REQUIRE(net && inputs && targets && count > 0, "null argument or empty dataset");
        use_device(net->ctx);
        SBH_HIP(hipStreamSynchronize(net->ctx->stream));
        net->data_in.allocate((size_t)count * RAW);
        net->data_out.allocate((size_t)count * 2);
        copy_on_stream(net->ctx, net->data_in.ptr, inputs, net->data_in.bytes(), hipMemcpyHostToDevice);
        copy_on_stream(net->ctx, net->data_out.ptr, targets, net->data_out.bytes(), hipMemcpyHostToDevice);
        net->data_count = count;
    });
}

sbh_status sbh_mlp_train(sbh_mlp* net, int64_t steps, int64_t batch, double lr_max, double lr_min, uint64_t seed,
                         double* losses) {
    return guard_on(ctx_of(net), [&] {
        SBH_REQUIRE(net, "net is null");
        SBH_REQUIRE(net->data_count > 0, "sbh_mlp_set_dataset has not been called");
        SBH_REQUIRE(batch > 0 && batch % 256 == 0 && batch <= (1 << 20), "batch must be a multiple of 256");
        SBH_REQUIRE(steps >= 0, "steps must be >= 0");
        use_device(net->ctx);
        sbh_context* ctx = net->ctx;
        ensure_batch(net, (int)batch, true);
        const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
        int pending = 0, blocks = 0;  // steps whose loss partials are still on the device
        for (int64_t s = 0; s < steps; ++s) {
            UpdateArgs u;
            blocks = forward_backward(net, net->data_in.ptr, true, seed * 0x100000001B3ull + (uint64_t)net->step,
                                      net->data_count, (int)batch, net->data_out.ptr,
                                      net->loss_part.ptr + (size_t)pending * (batch / 64), &u);
            net->step += 1;
            const double frac = steps > 1 ? (double)s / (double)(steps - 1) : 0.0;
            const double lr = lr_min + 0.5 * (lr_max - lr_min) * (1.0 + std::cos(M_PI * frac));
            u.lr = (float)lr;
            u.b1 = b1;
            u.b2 = b2;
            u.eps = eps;
            u.c1 = 1.f - std::pow(b1, (float)net->step);
            u.c2 = 1.f - std::pow(b2, (float)net->step);
            apply_update<true>(net, u);
            if (++pending == kLossSteps || s + 1 == steps) {
                // the host reads the losses of a run of steps together
                if (losses) {
                    std::vector<double> l((size_t)pending);
                    read_losses(net, pending, (int)(batch / 64), blocks, l.data());
                    for (int t = 0; t < pending; ++t) losses[s + 1 - pending + t] = l[t] / (double)batch;
                } else {
                    SBH_HIP(hipStreamSynchronize(ctx->stream));  // bounds the queue
                }
                pending = 0;
            }
        }
        SBH_HIP(hipStreamSynchronize(ctx->stream));
    });
}

sbh_status sbh_debug_mlp_predict_layered(sbh_mlp* net, const float* inputs, int64_t M, float* out) {
    return guard_on(ctx_of(net), [&] {
        SBH_REQUIRE(net && inputs && out, "null argument");
        SBH_REQUIRE(M > 0 && M <= (1 << 24), "M out of range");
        use_device(net->ctx);
        const int Mp = (int)((M + 255) / 256 * 256);
        ensure_batch(net, Mp, false);
        WorkArray<float> din((size_t)Mp * RAW);
        SBH_HIP(hipMemsetAsync(din.ptr, 0, din.bytes(), net->ctx->stream));
        SBH_HIP(hipMemcpyAsync(din.ptr, inputs, (size_t)M * RAW * sizeof(float), hipMemcpyHostToDevice,
                               net->ctx->stream));
        forward_backward(net, din.ptr, false, 0, 0, Mp, nullptr, nullptr, nullptr);
        SBH_HIP(hipMemcpyAsync(out, net->Y.ptr, (size_t)M * 2 * sizeof(float), hipMemcpyDeviceToHost,
                               net->ctx->stream));
        SBH_HIP(hipStreamSynchronize(net->ctx->stream));
    });
}

sbh_status sbh_mlp_predict(sbh_mlp* net, const float* inputs, int64_t M, float* out, int memory) {
    return guard_on(ctx_of(net), [&] {
        SBH_REQUIRE(net && inputs && out, "null argument");
        SBH_REQUIRE(M > 0 && M <= (1 << 24), "M out of range");
        use_device(net->ctx);
        const int Mp = (int)((M + 255) / 256 * 256);
        WorkArray<float> din((size_t)Mp * RAW);
        SBH_HIP(hipMemsetAsync(din.ptr, 0, din.bytes(), net->ctx->stream));
        SBH_HIP(hipMemcpyAsync(din.ptr, inputs, (size_t)M * RAW * sizeof(float),
                               memory == SBH_MEM_DEVICE ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice,
                               net->ctx->stream));
        infer(net, din.ptr, Mp);
        SBH_HIP(hipMemcpyAsync(out, net->Y.ptr, (size_t)M * 2 * sizeof(float),
                               memory == SBH_MEM_DEVICE ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost,
                               net->ctx->stream));
        SBH_HIP(hipStreamSynchronize(net->ctx->stream));
    });
}

}  // extern "C"
