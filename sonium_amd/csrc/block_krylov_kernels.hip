// Device kernels of the shared-basis block GMRES (block_krylov.cpp), which
// restates block_gmres_inner (crates/sonium-solvers/crates/
// sonium-solvers-iterative/src/block_gmres.rs:666-1120).
//
// Layout.  The block Krylov basis is column-major as in the reference:
// vector i of length n at V + i*n (complex FP64, interleaved).  The new
// Arnoldi block W (sj vectors) uses the same layout.  Right-hand sides and
// solutions are n x s row-major (one right-hand side per column).
//
// Block Gram G = V^H W (block_gram_into, :474-499) and the combinations
// W -= V G (block_project_into, :505-530) and X += V Y (apply_block_update,
// :545-565) run on v_mfma_f64_16x16x4_f64 in the real formulation:
//   Gram:     G~ (p x 2sj) = V~ (p x 2n) * Bt (2n x 2sj), V~ the interleaved
//             rows of V, and per complex entry w of W the 2x2 real block
//             [[Re w, Im w], [Im w, -Re w]] (columns Re g, Im g);
//   combine:  O~ (sj x 2n) = C~ (sj x 2p) * Bv (2p x 2n), C~ the rows
//             [Re c, Im c] of the coefficients, and per basis entry v the
//             block [[Re v, Im v], [-Im v, Re v]].
// MFMA operand/result layout of the 16x16x4 f64 form: A[m][k] from lane
// m + 16k, B[k][n] from lane n + 16k, result register v of lane l holds row
// 4v + l/16, column l%16.
//
// The in-block QR with rank-drop deflation (CGS2 per column, :992-1025) is a
// chain of small kernels over row chunks; the accept/deflate decision is taken
// on the device from reductions summed in a fixed order, so every workgroup
// takes the same decision and the host reads the outcome once per block step.

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstddef>
#include <type_traits>

#include "block_krylov.hpp"
#include "internal.hpp"

namespace sbh {

namespace {

constexpr int BK_THREADS = 256;
constexpr int BK_XCD = 8;          // XCDs of the MI355X; K slices are grouped per XCD
constexpr int BK_CK = 16;          // complex output entries per combine tile
constexpr int QR_CHUNK = 256;      // rows per workgroup in the in-block QR chain (one per thread)
constexpr int QR_MAXC = 64;        // block width limit
constexpr int QR_SLOTS = QR_MAXC + 1;  // dots + squared norm per chunk

typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cmulc(double2 a, double2 b) {  // conj(a) * b
    return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
}

// Barrier for what the workgroup exchanges through LDS.  __syncthreads() also
// waits for every global load and store in flight: 1 us a barrier where a loop
// loads ahead or stores as it goes.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// x plus the lane that a rotation by `CTRL & 15` within rows of 16 lanes brings
template <int CTRL>
__device__ __forceinline__ double add_row_rotated(double x) {
    const int lo = __double2loint(x), hi = __double2hiint(x);
    return x + __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false),
                                __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false));
}
// sum over each row of 16 lanes, in all of them
__device__ __forceinline__ double row_sum(double x) {
    x = add_row_rotated<0x128>(x);
    x = add_row_rotated<0x124>(x);
    x = add_row_rotated<0x122>(x);
    return add_row_rotated<0x121>(x);
}
// sum over the wave, in every lane
__device__ __forceinline__ double wave_sum(double x) {
    x = row_sum(x);
    // of two copies of x: even rows beside odd ones, then the lower half beside the upper
    const auto l16 = __builtin_amdgcn_permlane16_swap(__double2loint(x), __double2loint(x), false, false);
    const auto h16 = __builtin_amdgcn_permlane16_swap(__double2hiint(x), __double2hiint(x), false, false);
    x = __hiloint2double(h16[0], l16[0]) + __hiloint2double(h16[1], l16[1]);
    const auto l32 = __builtin_amdgcn_permlane32_swap(__double2loint(x), __double2loint(x), false, false);
    const auto h32 = __builtin_amdgcn_permlane32_swap(__double2hiint(x), __double2hiint(x), false, false);
    return __hiloint2double(h32[0], l32[0]) + __hiloint2double(h32[1], l32[1]);
}

// ---------------------------------------------------------------- Gram

// part[(slice * p + i) * 2sj + 2c + {0,1}] = sum over the slice's rows k of
// conj(V[i][k]) W[c][k] (re, im).  Blocks: (tile of 16 MB basis vectors, K
// slice); the K slices of one XCD (blockIdx % 8) are shared by consecutive
// basis tiles so the W slice stays in that XCD's L2.
//
// Each wave takes a quarter of the slice's rows for the whole tile and feeds
// the matrix cores straight from global memory: in the order k = (row, re/im)
// lane (m, g) needs entry (m, row g) of both operands and forms the real and
// the imaginary line of its 2x2 blocks from one 16-byte load, so neither
// operand passes through LDS and no barrier stands in the loop.  The next 8
// rows are loaded while the present ones are multiplied.  The work of a step
// (p 24 to 600, 24 columns, 5056 rows: 0.02 to 0.6 GFLOP) is far too small to
// hide a barrier per 16 rows behind: staged through LDS in slices of 316 rows,
// 16 to 160 workgroups, it took 40 us on average; this way 11.
template <int NT, int MB>
__global__ __launch_bounds__(BK_THREADS) void bk_gram_kernel(const double2* __restrict__ V, int64_t ldv, int p,
                                                             const double2* __restrict__ W, int64_t ldw, int sj,
                                                             int64_t n, int64_t kslice, int itiles,
                                                             double* __restrict__ part, const int* __restrict__ flag) {
    if (flag && *flag == 0) return;
    __shared__ double red[4][MB * NT * 4][64];
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int xcd = blockIdx.x % BK_XCD;
    const int local = blockIdx.x / BK_XCD;
    const int i0 = (local % itiles) * 16 * MB;
    const int slice = (local / itiles) * BK_XCD + xcd;
    const int64_t kbeg = (int64_t)slice * kslice + w * (kslice / 4);
    const int64_t kend = min(n, kbeg + kslice / 4);
    const int g = lane >> 4, m = lane & 15;
    // rows past the tile's end repeat the last one and are not stored
    const double2* va[MB];
    const double2* wa[NT];
#pragma unroll
    for (int a = 0; a < MB; ++a) va[a] = V + (int64_t)min(i0 + 16 * a + m, p - 1) * ldv;
#pragma unroll
    for (int b = 0; b < NT; ++b) wa[b] = W + (int64_t)min(8 * b + (m >> 1), sj - 1) * ldw;
    f64x4 acc[MB][NT];
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b) acc[a][b] = f64x4{0.0, 0.0, 0.0, 0.0};
    struct Rows {
        double2 v[2][MB], w[2][NT];
    };
    // 8 rows from k0, the first again for those past the end (cleared by mul)
    auto gload = [&](int64_t k0, Rows& r) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int64_t k = k0 + 4 * u + g < kend ? k0 + 4 * u + g : kbeg;
#pragma unroll
            for (int a = 0; a < MB; ++a) r.v[u][a] = va[a][k];
#pragma unroll
            for (int b = 0; b < NT; ++b) r.w[u][b] = wa[b][k];
        }
    };
    auto mul = [&](int64_t k0, Rows& r) {
        if (k0 + 8 > kend) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const bool in = k0 + 4 * u + g < kend;
#pragma unroll
                for (int a = 0; a < MB; ++a) r.v[u][a] = in ? r.v[u][a] : make_double2(0.0, 0.0);
#pragma unroll
                for (int b = 0; b < NT; ++b) r.w[u][b] = in ? r.w[u][b] : make_double2(0.0, 0.0);
            }
        }
        const bool im = m & 1;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int b = 0; b < NT; ++b) {
                const double2 x = r.w[u][b];
                const double line0 = im ? x.y : x.x;
                const double line1 = im ? -x.x : x.y;
#pragma unroll
                for (int a = 0; a < MB; ++a) {
                    acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(r.v[u][a].x, line0, acc[a][b], 0, 0, 0);
                    acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(r.v[u][a].y, line1, acc[a][b], 0, 0, 0);
                }
            }
        }
    };
    if (kbeg < kend) {
        Rows r0, r1;
        gload(kbeg, r0);
        for (int64_t k0 = kbeg; k0 < kend; k0 += 16) {
            if (k0 + 8 < kend) gload(k0 + 8, r1);
            mul(k0, r0);
            if (k0 + 8 >= kend) break;
            if (k0 + 16 < kend) gload(k0 + 16, r0);
            mul(k0 + 8, r1);
        }
    }
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[w][(a * NT + b) * 4 + v][lane] = acc[a][b][v];
    __syncthreads();
    // wave w adds the four waves' sums (in order) of result register w of every tile
    const int ncol = 2 * sj;
#pragma unroll
    for (int a = 0; a < MB; ++a) {
        const int i = i0 + 16 * a + 4 * w + g;
#pragma unroll
        for (int b = 0; b < NT; ++b) {
            const int q = (a * NT + b) * 4 + w;
            const double sum = ((red[0][q][lane] + red[1][q][lane]) + red[2][q][lane]) + red[3][q][lane];
            const int col = 16 * b + m;
            if (i < p && col < ncol) part[((int64_t)slice * p + i) * ncol + col] = sum;
        }
    }
}

// gram[i*sj + c] = sum of the slice partials in slice order; hmode 1 sets and
// hmode 2 adds the result into hacc (the Hessenberg block h[0:p, p_start:+sj]).
__global__ void bk_gram_reduce_kernel(const double* __restrict__ part, int nslices, int p, int sj,
                                      double2* __restrict__ gram, double2* __restrict__ hacc, int hmode,
                                      const int* __restrict__ flag) {
    if (flag && *flag == 0) return;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)p * sj) return;
    const int64_t i = e / sj;
    const int c = (int)(e % sj);
    const int ncol = 2 * sj;
    double re = 0.0, im = 0.0;
#pragma unroll 8
    for (int s = 0; s < nslices; ++s) {
        const double2 v = *reinterpret_cast<const double2*>(part + ((int64_t)s * p + i) * ncol + 2 * c);
        re += v.x;
        im += v.y;
    }
    const double2 g = make_double2(re, im);
    gram[e] = g;
    if (hmode == 1) {
        hacc[e] = g;
    } else if (hmode == 2) {
        const double2 h = hacc[e];
        hacc[e] = make_double2(h.x + g.x, h.y + g.y);
    }
}

// ---------------------------------------------------------------- combine

// O[c*osc + k*osk] = (add ? O : 0) + alpha * sum_{i<p} C[i*ldc + c] V[i*ldv + k]
// for c < sj, k < n.  A block owns 16 complex k (32 real output columns) and
// every c; its four waves take a quarter of the basis vectors each and their
// sums are added in order at the end.  As in the Gram kernel the operands go
// from global memory straight to the matrix cores, four basis vectors a step:
// lane (m, g) holds C[i + g][c = m] and V[i + g][k of column m], and forms the
// real and the imaginary line of both from one 16-byte load.  Staged through
// LDS in tiles of 64 k the 5056-row case ran on 79 of 256 CUs with two
// barriers per 16 basis vectors: 26 us on average, now 10.
template <int MT>
__global__ __launch_bounds__(BK_THREADS) void bk_combine_kernel(const double2* __restrict__ V, int64_t ldv, int p,
                                                                const double2* __restrict__ C, int ldc, int sj,
                                                                int64_t n, double2* __restrict__ O, int64_t osc,
                                                                int64_t osk, int add, double alpha,
                                                                const int* __restrict__ flag) {
    if (flag && *flag == 0) return;
    __shared__ double red[4][MT * 8][64];
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    const int g = lane >> 4, m = lane & 15;
    const int64_t k0 = (int64_t)blockIdx.x * BK_CK;
    const int quarter = (p + 15) / 16 * 4;
    const int ibeg = w * quarter, iend = min(p, ibeg + quarter);
    f64x4 acc[MT][2];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t][0] = acc[t][1] = f64x4{0.0, 0.0, 0.0, 0.0};
    // columns past the end repeat the last one and are not stored
    int64_t kc[2];
    int cc[MT];
#pragma unroll
    for (int q = 0; q < 2; ++q) kc[q] = min(k0 + 8 * q + (m >> 1), n - 1);
#pragma unroll
    for (int t = 0; t < MT; ++t) cc[t] = min(16 * t + m, sj - 1);
    struct Vectors {
        double2 v[2][2], c[2][MT];
    };
    // 8 basis vectors from i0, the first again for those past the end (cleared by mul)
    auto gload = [&](int i0, Vectors& r) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int i = i0 + 4 * u + g < iend ? i0 + 4 * u + g : ibeg;
#pragma unroll
            for (int q = 0; q < 2; ++q) r.v[u][q] = V[(int64_t)i * ldv + kc[q]];
#pragma unroll
            for (int t = 0; t < MT; ++t) r.c[u][t] = C[(int64_t)i * ldc + cc[t]];
        }
    };
    auto mul = [&](int i0, Vectors& r) {
        if (i0 + 8 > iend) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const bool in = i0 + 4 * u + g < iend;
#pragma unroll
                for (int q = 0; q < 2; ++q) r.v[u][q] = in ? r.v[u][q] : make_double2(0.0, 0.0);
#pragma unroll
                for (int t = 0; t < MT; ++t) r.c[u][t] = in ? r.c[u][t] : make_double2(0.0, 0.0);
            }
        }
        const bool im = m & 1;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const double2 x = r.v[u][q];
                const double line0 = im ? x.y : x.x;
                const double line1 = im ? x.x : -x.y;
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    acc[t][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(r.c[u][t].x, line0, acc[t][q], 0, 0, 0);
                    acc[t][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(r.c[u][t].y, line1, acc[t][q], 0, 0, 0);
                }
            }
    };
    if (ibeg < iend) {
        Vectors r0, r1;
        gload(ibeg, r0);
        for (int i0 = ibeg; i0 < iend; i0 += 16) {
            if (i0 + 8 < iend) gload(i0 + 8, r1);
            mul(i0, r0);
            if (i0 + 8 >= iend) break;
            if (i0 + 16 < iend) gload(i0 + 16, r0);
            mul(i0 + 8, r1);
        }
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[w][(t * 2 + q) * 4 + v][lane] = acc[t][q][v];
    __syncthreads();
    // wave w adds the four waves' sums (in order) of result register w of every tile
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int c = 16 * t + 4 * w + g;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int r = (t * 2 + q) * 4 + w;
            const double sum = ((red[0][r][lane] + red[1][r][lane]) + red[2][r][lane]) + red[3][r][lane];
            const int64_t k = k0 + 8 * q + (m >> 1);
            if (c < sj && k < n) {
                double* o = reinterpret_cast<double*>(O + c * osc + k * osk) + (m & 1);
                *o = (add ? *o : 0.0) + alpha * sum;
            }
        }
    }
}

// ---------------------------------------------------------------- Cholesky QR

// What one block QR by Cholesky leaves: R with W = Q R, ok = 0 when a pivot
// was not clearly positive (the CGS2 chain takes over).
struct CholState {
    int ok;
    int pad[3];
    double2 r[QR_MAXC * QR_MAXC];  // m x m row-major, upper
};

// One pass of Cholesky QR in one workgroup: G = R^H R (m x m, Hermitian,
// row-major), T = R^-1 for the combination Q = W T.  Pass 0 leaves R in st->r;
// pass 1 (only if pass 0 was ok) leaves R R0, the factor of both passes.  A pivot fails below floor^2 times its diagonal
// entry.  Sixteen lanes hold one column, four entries each, through the
// factorisation (one barrier per row) and the inversion (none: a column of T
// depends on that column alone).  The chain of m rows bounds it: 27 us for 24
// columns, where reading G to the host, factoring there and sending T back
// cost two synchronisations, about 50.
__global__ __launch_bounds__(1024) void bk_cholesky_kernel(const double2* __restrict__ G, int m, double floor, int pass,
                                                           CholState* st, double2* __restrict__ T) {
    if (pass == 1 && st->ok == 0) return;
    __shared__ double2 R[QR_MAXC * (QR_MAXC + 1) / 2];  // row i from i*m - i(i+1)/2, entry k >= i at + k
    __shared__ double2 line[2][QR_MAXC];
    __shared__ double diag[QR_MAXC], rinv[QR_MAXC];
    const int c = threadIdx.x >> 4, l = threadIdx.x & 15;
    double2 e[4];  // rows l, 16 + l, 32 + l, 48 + l of column c
    double2 first[4];  // the same of the first pass's R
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int i = 16 * q + l;
        e[q] = i < m && c < m ? G[i * m + c] : make_double2(0.0, 0.0);
        first[q] = pass == 1 && i <= c && c < m ? st->r[i * m + c] : make_double2(0.0, 0.0);
        if (i == c) diag[c] = e[q].x;
    }
    bool ok = true;
    for (int j = 0; j < m; ++j) {
        double2* lj = line[j & 1];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (16 * q + l == j) lj[c] = e[q];
        lds_barrier();
        const double d = lj[j].x;
        ok = diag[j] > 0.0 && d > floor * floor * diag[j] && isfinite(d);  // the same in every thread
        if (!ok) break;
        const double inv = rsqrt(d);
        const double2 rc = c == j ? make_double2(d * inv, 0.0) : make_double2(lj[c].x * inv, lj[c].y * inv);
        if (l == (j & 15) && c >= j && c < m) R[j * m - j * (j + 1) / 2 + c] = rc;
        if (threadIdx.x == 0) rinv[j] = inv;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = 16 * q + l;
            if (i > j && i < m) {
                const double2 x = cmulc(make_double2(lj[i].x * inv, lj[i].y * inv), rc);
                e[q] = make_double2(e[q].x - x.x, e[q].y - x.y);
            }
        }
    }
    if (threadIdx.x == 0) st->ok = ok ? 1 : 0;
    if (!ok) return;
    __syncthreads();
    double2 t[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) t[q] = make_double2(0.0, 0.0);
    for (int i = m - 1; i >= 0; --i) {
        const double2* ri = R + i * m - i * (i + 1) / 2;
        double2 acc = make_double2(0.0, 0.0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = 16 * q + l;
            if (k > i && k < m) {
                const double2 x = cmul(ri[k], t[q]);
                acc = make_double2(acc.x + x.x, acc.y + x.y);
            }
        }
        acc = make_double2(row_sum(acc.x), row_sum(acc.y));
        if (l == (i & 15) && i <= c) {
            const double inv = rinv[i];
            const double2 x = i == c ? make_double2(inv, 0.0) : make_double2(-acc.x * inv, -acc.y * inv);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                t[q].x = 16 * q + l == i ? x.x : t[q].x;
                t[q].y = 16 * q + l == i ? x.y : t[q].y;
            }
        }
    }
    double2 prod[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) prod[q] = make_double2(0.0, 0.0);
    if (pass == 1) {
#pragma unroll
        for (int kq = 0; kq < 4; ++kq)
            for (int kl = 0; kl < 16 && 16 * kq + kl < m; ++kl) {
                const int k = 16 * kq + kl;
                const double2 r0 = make_double2(__shfl(first[kq].x, kl, 16), __shfl(first[kq].y, kl, 16));
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int i = 16 * q + l;
                    if (i <= k && k <= c) {
                        const double2 x = cmul(R[i * m - i * (i + 1) / 2 + k], r0);
                        prod[q] = make_double2(prod[q].x + x.x, prod[q].y + x.y);
                    }
                }
            }
    }
    if (c < m) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = 16 * q + l;
            if (i < m) {
                T[i * m + c] = t[q];
                double2 x = make_double2(0.0, 0.0);
                if (i <= c) {
                    const double2 r = R[i * m - i * (i + 1) / 2 + c];
                    x.x = pass == 0 ? r.x : prod[q].x;
                    x.y = pass == 0 ? r.y : prod[q].y;
                }
                st->r[i * m + c] = x;
            }
        }
    }
}

// ---------------------------------------------------------------- layout and reductions

// out[k*cols + c] = in[c*ld + k] (column-major -> row-major), 16 x 64 tiles
__global__ void bk_to_rowmajor_kernel(const double2* __restrict__ in, int64_t ld, int cols, int64_t n,
                                      double2* __restrict__ out) {
    __shared__ double2 tile[16][65];
    const int64_t k0 = (int64_t)blockIdx.x * 64;
    const int c0 = blockIdx.y * 16;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    for (int r = ty; r < 16; r += 4) {
        const int c = c0 + r;
        tile[r][tx] = (c < cols && k0 + tx < n) ? in[(int64_t)c * ld + k0 + tx] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * 64; e += blockDim.x) {
        const int kk = e >> 4, cc = e & 15;
        if (c0 + cc < cols && k0 + kk < n) out[(k0 + kk) * cols + c0 + cc] = tile[cc][kk];
    }
}

// out[c*ld + k] = d[k] * in[k*cols + c] (row-major -> column-major; d may be null)
__global__ void bk_to_colmajor_kernel(const double2* __restrict__ in, int cols, int64_t n,
                                      const double2* __restrict__ d, double2* __restrict__ out, int64_t ld) {
    __shared__ double2 tile[16][65];
    const int64_t k0 = (int64_t)blockIdx.x * 64;
    const int c0 = blockIdx.y * 16;
    for (int e = threadIdx.x; e < 16 * 64; e += blockDim.x) {
        const int kk = e >> 4, cc = e & 15;
        double2 v = make_double2(0.0, 0.0);
        if (c0 + cc < cols && k0 + kk < n) {
            v = in[(k0 + kk) * cols + c0 + cc];
            if (d) v = cmul(d[k0 + kk], v);
        }
        tile[cc][kk] = v;
    }
    __syncthreads();
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    for (int r = ty; r < 16; r += 4) {
        const int c = c0 + r;
        if (c < cols && k0 + tx < n) out[(int64_t)c * ld + k0 + tx] = tile[r][tx];
    }
}

// R[c*n + k] = d[k] * (B[k*s + c] - AX[k*s + c]) (AX may be null: zero)
__global__ void bk_residual_cm_kernel(const double2* __restrict__ B, const double2* __restrict__ AX, int s,
                                      int64_t n, const double2* __restrict__ d, double2* __restrict__ R) {
    __shared__ double2 tile[16][65];
    const int64_t k0 = (int64_t)blockIdx.x * 64;
    const int c0 = blockIdx.y * 16;
    for (int e = threadIdx.x; e < 16 * 64; e += blockDim.x) {
        const int kk = e >> 4, cc = e & 15;
        double2 v = make_double2(0.0, 0.0);
        if (c0 + cc < s && k0 + kk < n) {
            const int64_t idx = (k0 + kk) * s + c0 + cc;
            v = B[idx];
            if (AX) {
                const double2 a = AX[idx];
                v = make_double2(v.x - a.x, v.y - a.y);
            }
            if (d) v = cmul(d[k0 + kk], v);
        }
        tile[cc][kk] = v;
    }
    __syncthreads();
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    for (int r = ty; r < 16; r += 4) {
        const int c = c0 + r;
        if (c < s && k0 + tx < n) R[(int64_t)c * n + k0 + tx] = tile[r][tx];
    }
}

// Squared norms of `cols` contiguous vectors of length n: part[chunk*cols + c]
// over rows [chunk*len, ...), each thread in row order, then a fixed tree.
__global__ __launch_bounds__(BK_THREADS) void bk_colnorm_partials_kernel(const double2* __restrict__ X, int64_t ld,
                                                                         int cols, int64_t n, int64_t len,
                                                                         double* __restrict__ part) {
    __shared__ double red[BK_THREADS];
    const int c = blockIdx.y;
    const int64_t b = (int64_t)blockIdx.x * len;
    const int64_t e = min(n, b + len);
    double s = 0.0;
    for (int64_t k = b + threadIdx.x; k < e; k += BK_THREADS) {
        const double2 v = X[(int64_t)c * ld + k];
        s += v.x * v.x + v.y * v.y;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int h = BK_THREADS / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[(int64_t)blockIdx.x * cols + c] = red[0];
}

// out[c] = sqrt(sum over chunks in chunk order of part[chunk*cols + c])
__global__ void bk_sum_sqrt_kernel(const double* __restrict__ part, int chunks, int cols, double* __restrict__ out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= cols) return;
    double s = 0.0;
    for (int q = 0; q < chunks; ++q) s += part[(int64_t)q * cols + c];
    out[c] = sqrt(s);
}

// DGKS trigger on the block Frobenius norm (block_gmres.rs:962-987):
// flag = ||W_after||_F < 0.707 ||W_before||_F, from squared-norm partials.
__global__ void bk_dgks_flag_kernel(const double* __restrict__ before, const double* __restrict__ after, int chunks,
                                    int* __restrict__ flag, double* __restrict__ frob) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    double b = 0.0, a = 0.0;
    for (int q = 0; q < chunks; ++q) b += before[q];
    for (int q = 0; q < chunks; ++q) a += after[q];
    const double fb = sqrt(b), fa = sqrt(a);
    frob[0] = fb;
    frob[1] = fa;
    *flag = (fa >= 0.707 * fb) ? 0 : 1;
}

// Per column of n x s row-major blocks: ||B - AX||^2, ||AX||^2, ||B||^2
// partials (block_true_metrics, block_gmres.rs:567-612) into part[chunk][3s].
__global__ __launch_bounds__(BK_THREADS) void bk_true_partials_kernel(const double2* __restrict__ B,
                                                                      const double2* __restrict__ AX, int s,
                                                                      int64_t n, int64_t len,
                                                                      double* __restrict__ part) {
    __shared__ double red[3][BK_THREADS];
    const int c = blockIdx.y;
    const int64_t b = (int64_t)blockIdx.x * len;
    const int64_t e = min(n, b + len);
    double r2 = 0.0, a2 = 0.0, b2 = 0.0;
    for (int64_t k = b + threadIdx.x; k < e; k += BK_THREADS) {
        const double2 bb = B[k * s + c], aa = AX[k * s + c];
        const double dr = bb.x - aa.x, di = bb.y - aa.y;
        r2 += dr * dr + di * di;
        a2 += aa.x * aa.x + aa.y * aa.y;
        b2 += bb.x * bb.x + bb.y * bb.y;
    }
    red[0][threadIdx.x] = r2;
    red[1][threadIdx.x] = a2;
    red[2][threadIdx.x] = b2;
    __syncthreads();
    for (int h = BK_THREADS / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h)
            for (int q = 0; q < 3; ++q) red[q][threadIdx.x] += red[q][threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int q = 0; q < 3; ++q) part[((int64_t)blockIdx.x * 3 + q) * s + c] = red[q][0];
}

// ---------------------------------------------------------------- in-block QR chain

// Device state of one block QR (initial block or a new Arnoldi block).
struct QrState {
    int snext[QR_MAXC + 1];   // accepted directions before column c (snext[0] = 0)
    int accepted[QR_MAXC];    // slot of column c, or -1 if deflated
    unsigned counter;         // finished workgroups of the running launch
    int pad[2];
    double orig[QR_MAXC];     // ||w_c|| before the passes
    double wnorm[QR_MAXC];    // ||w_c|| after the passes
    double2 r[QR_MAXC][QR_MAXC];  // h[p + a][p_start + c] += d1[a] + d2[a]  (a < snext[c])
    double2 coef[QR_MAXC];    // coefficients of the pass in progress
};

struct QrArgs {
    double2* W;       // sj column-major vectors of length n
    double2* Q;       // the block's accepted directions: slot a at Q + a*n
    int64_t n;
    int sj;
    int budget;       // accepted directions allowed in this block
    double defl_tol;  // sqrt(eps)
    QrState* st;
    double2* part;    // chunks x QR_SLOTS partial sums (dots in slots 0..63, ||w||^2 in slot 64)
};

// True in the workgroup that finishes last: each workgroup publishes its
// partials, then takes a ticket; the last one sums every chunk's partials
// (in chunk order) and clears the counter for the next launch.
__device__ bool qr_last_block(unsigned* counter) {
    __shared__ bool last;
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) last = atomicAdd(counter, 1u) == gridDim.x - 1;
    __syncthreads();
    if (last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    return last;
}

// out[v] = sum over chunks of part[chunk][v] for v < cnt and, with the norm,
// v = QR_MAXC: four strided quarter sums, added in order.
__device__ void qr_sum_chunks(const double2* __restrict__ part, int chunks, int cnt, bool with_norm, double2* out,
                              double2 (*quarter)[4]) {
    const int t = threadIdx.x;
    const int items = 4 * (cnt + (with_norm ? 1 : 0));
    for (int w = t; w < items; w += BK_THREADS) {
        const int idx = w >> 2, q = w & 3;
        const int v = idx < cnt ? idx : QR_MAXC;
        double re = 0.0, im = 0.0;
        for (int ch = q; ch < chunks; ch += 4) {
            const double2 x = part[(int64_t)ch * QR_SLOTS + v];
            re += x.x;
            im += x.y;
        }
        quarter[v][q] = make_double2(re, im);
    }
    __syncthreads();
    if (t < cnt || (with_norm && t == QR_MAXC)) {
        double re = quarter[t][0].x, im = quarter[t][0].y;
        for (int q = 1; q < 4; ++q) {
            re += quarter[t][q].x;
            im += quarter[t][q].y;
        }
        out[t] = make_double2(re, im);
    }
    __syncthreads();
}

// This chunk's partials of conj(q_a) . w (a < cnt; the LDS copy ql replaces
// slot cnt - 1 when given) and ||w||^2, w in LDS.  Thread (a = t % 64,
// segment = t / 64) sums a quarter of the chunk in row order; the quarters
// are added in order.
__device__ void qr_chunk_dots(const double2* __restrict__ Q, int64_t n, int64_t r0, int len, int cnt,
                              const double2* wl, const double2* ql, double2* __restrict__ part_out,
                              double2 (*seg)[4], double* red) {
    const int t = threadIdx.x;
    const int a = t & 63, sg = t >> 6;
    const int slen = (len + 3) / 4;
    const int b = sg * slen, e = min(len, b + slen);
    if (a < cnt) {
        double re = 0.0, im = 0.0;
        const bool from_lds = ql && a == cnt - 1;
        const double2* q = Q + (int64_t)a * n + r0;
#pragma unroll 8
        for (int k = b; k < e; ++k) {
            const double2 qa = from_lds ? ql[k] : q[k];
            const double2 d = cmulc(qa, wl[k]);
            re += d.x;
            im += d.y;
        }
        seg[a][sg] = make_double2(re, im);
    }
    double s2 = 0.0;
    for (int k = t; k < len; k += BK_THREADS) s2 += wl[k].x * wl[k].x + wl[k].y * wl[k].y;
    red[t] = s2;
    __syncthreads();
    for (int h = BK_THREADS / 2; h > 0; h >>= 1) {
        if (t < h) red[t] += red[t + h];
        __syncthreads();
    }
    if (t < cnt) {
        double re = seg[t][0].x, im = seg[t][0].y;
        for (int q = 1; q < 4; ++q) {
            re += seg[t][q].x;
            im += seg[t][q].y;
        }
        part_out[t] = make_double2(re, im);
    }
    if (t == 0) part_out[QR_MAXC] = make_double2(red[0], 0.0);
}

// Start of column c (c == sj: finish only): the previous column's direction
// q = w * (1/||w||) if it was accepted, then pass-1 partials of column c;
// the last workgroup turns them into d1 (the first h entries) and ||w_c||.
__global__ __launch_bounds__(BK_THREADS) void bk_qr_start_kernel(QrArgs a, int c) {
    __shared__ double2 wl[QR_CHUNK];
    __shared__ double2 ql[QR_CHUNK];
    __shared__ double2 seg[QR_MAXC][4];
    __shared__ double2 quarter[QR_SLOTS][4];
    __shared__ double2 sums[QR_SLOTS];
    __shared__ double red[BK_THREADS];
    const int t = threadIdx.x;
    const int64_t r0 = (int64_t)blockIdx.x * QR_CHUNK;
    const int len = (int)min((int64_t)QR_CHUNK, a.n - r0);
    bool fresh = false;
    if (c > 0) {
        const int slot = a.st->accepted[c - 1];
        if (slot >= 0) {
            const double inv = 1.0 / a.st->wnorm[c - 1];
            const double2* wp = a.W + (int64_t)(c - 1) * a.n + r0;
            double2* q = a.Q + (int64_t)slot * a.n + r0;
            for (int k = t; k < len; k += BK_THREADS) {
                const double2 v = wp[k];
                const double2 qv = make_double2(v.x * inv, v.y * inv);
                q[k] = qv;
                ql[k] = qv;
            }
            fresh = true;
        }
    }
    if (c >= a.sj) return;
    const int cnt = c == 0 ? 0 : a.st->snext[c];
    const double2* wc = a.W + (int64_t)c * a.n + r0;
    for (int k = t; k < len; k += BK_THREADS) wl[k] = wc[k];
    __syncthreads();
    qr_chunk_dots(a.Q, a.n, r0, len, cnt, wl, fresh ? ql : nullptr, a.part + (int64_t)blockIdx.x * QR_SLOTS, seg,
                  red);
    if (!qr_last_block(&a.st->counter)) return;
    qr_sum_chunks(a.part, gridDim.x, cnt, true, sums, quarter);
    if (t < cnt) {
        a.st->r[c][t] = sums[t];
        a.st->coef[t] = sums[t];
    }
    if (t == 0) {
        if (c == 0) a.st->snext[0] = 0;
        a.st->orig[c] = sqrt(sums[QR_MAXC].x);
        a.st->counter = 0;
    }
}

// w_c -= sum_a coef[a] q_a (the reference's axpy order), then (second) the
// pass-2 partials, whose sums become coef and are added into the h entries,
// or (third) the partial ||w_c||^2, whose square root decides acceptance:
// wn > defl_tol * max(orig, tiny) and room left in the block
// (block_gmres.rs:1014-1024).
__global__ __launch_bounds__(BK_THREADS) void bk_qr_project_kernel(QrArgs a, int c, int third) {
    __shared__ double2 wl[QR_CHUNK];
    __shared__ double2 d[QR_MAXC];
    __shared__ double2 seg[QR_MAXC][4];
    __shared__ double2 quarter[QR_SLOTS][4];
    __shared__ double2 sums[QR_SLOTS];
    __shared__ double red[BK_THREADS];
    const int t = threadIdx.x;
    const int cnt = a.st->snext[c];
    const int64_t r0 = (int64_t)blockIdx.x * QR_CHUNK;
    const int len = (int)min((int64_t)QR_CHUNK, a.n - r0);
    if (t < cnt) d[t] = a.st->coef[t];
    __syncthreads();
    double2* wc = a.W + (int64_t)c * a.n + r0;
    for (int k = t; k < len; k += BK_THREADS) {
        double2 v = wc[k];
        for (int q = 0; q < cnt; ++q) {
            const double2 nd = make_double2(-d[q].x, -d[q].y);
            const double2 t2 = cmul(nd, a.Q[(int64_t)q * a.n + r0 + k]);
            v = make_double2(v.x + t2.x, v.y + t2.y);
        }
        wc[k] = v;
        wl[k] = v;
    }
    __syncthreads();
    qr_chunk_dots(a.Q, a.n, r0, len, third ? 0 : cnt, wl, nullptr, a.part + (int64_t)blockIdx.x * QR_SLOTS, seg,
                  red);
    if (!qr_last_block(&a.st->counter)) return;
    qr_sum_chunks(a.part, gridDim.x, third ? 0 : cnt, third != 0, sums, quarter);
    if (!third) {
        if (t < cnt) {
            const double2 h = a.st->r[c][t];
            a.st->r[c][t] = make_double2(h.x + sums[t].x, h.y + sums[t].y);
            a.st->coef[t] = sums[t];
        }
    } else if (t == 0) {
        const double wn = sqrt(sums[QR_MAXC].x);
        const bool accept = wn > a.defl_tol * fmax(a.st->orig[c], 1e-30) && cnt < a.budget;
        a.st->wnorm[c] = wn;
        a.st->accepted[c] = accept ? cnt : -1;
        a.st->snext[c + 1] = cnt + (accept ? 1 : 0);
    }
    if (t == 0) a.st->counter = 0;
}

// ---------------------------------------------------------------- least squares

// Householder QR of the block Hessenberg matrix, kept across the block steps of
// a cycle: the least-squares problem that solve_block_ls (block_gmres.rs:
// 614-664) solves with Givens rotations.  Step q holds columns and rows
// [p_q, p_q + s_q); its columns reach s_{q+1} rows further, so its
// transformation acts on the window [p_q, p_q + s_q + s_{q+1}), at most 2 * 64
// rows: one or two (W) entries per lane of a wave.  Consecutive steps whose
// windows fit one of 64 W rows together make one group with one unitary factor,
// so the chain that a new column goes through is as long as the basis, not the
// steps: with a group to each step, 200 steps of one column on 2048 rows took
// 45.7 ms (40.0 with the rotations on the host), now 21.5; of 16 columns on 5120
// rows 123 (175), now 101.
//
// On the host the rotations of a 24-column step took 350 us (half of it the
// new block's own, in one thread), more than the device needs for the step,
// and every Hessenberg block and every coefficient crossed the bus.
struct LsState {
    int4* groups;       // of steps: first row, columns, rows of the last step's QR after them
    double2* refl;      // the last step's column c: 64 W window entries of v, H = I - v v^H
    double2* qh;        // group q: Q^H of its window, column by column, (64 W)^2 entries
    double2* R;         // packed columns of the triangle, column c from c(c+1)/2
    double2* window;    // the new columns' windows, 64 W entries each
    double2* g;         // transformed right-hand sides, column q from q * ldg
    int64_t ldg;
    BlockStep* host;    // pinned: the step's outcome
};

// The QR of a step: by Cholesky, or the chain's
struct LsQr {
    const CholState* chol;
    const QrState* chain;  // used if not null
    __device__ int next(int sj) const { return chain ? chain->snext[sj] : sj; }
    __device__ double2 entry(int sj, int c, int a) const {
        if (!chain) return a <= c ? chol->r[a * sj + c] : make_double2(0.0, 0.0);
        if (a < chain->snext[c]) return chain->r[c][a];
        return a == chain->accepted[c] ? make_double2(chain->wnorm[c], 0.0) : make_double2(0.0, 0.0);
    }
};

// x -= v (v^H x), one or two entries per lane
template <int W>
__device__ __forceinline__ void reflect(const double2 (&v)[W], double2 (&x)[W]) {
    double2 d = make_double2(0.0, 0.0);
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const double2 y = cmulc(v[w], x[w]);
        d = make_double2(d.x + y.x, d.y + y.y);
    }
    d = make_double2(wave_sum(d.x), wave_sum(d.y));
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const double2 y = cmul(v[w], d);
        x[w] = make_double2(x[w].x - y.x, x[w].y - y.y);
    }
}

// The `done` groups' transformations on one new Hessenberg column per
// workgroup: the finished entries go to R, the rest to its window.  Lane l of
// wave w forms row l of a quarter of the product Q_q^H x, so a group costs two
// barriers and a fourth of the window's multiplications in a row.  Reflector by
// reflector, each with its dot product across a wave, the 265 of an average
// step of a 24-column solve took 62 us; the products take 27, and Q^H 7 to form.
template <int W>
__global__ __launch_bounds__(256) void bk_ls_apply_kernel(LsState ls, LsQr qr, const double2* __restrict__ hacc, int sj,
                                                          int done, int p_start) {
    if (!qr.chain && qr.chol->ok == 0) return;
    constexpr int N = 64 * W;
    constexpr int AHEAD = 16 / W;  // rows of the next product loaded ahead, of 16 W to a wave
    __shared__ double2 x[N];
    __shared__ double2 sum[4][N];
    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int c = blockIdx.x;
    const int p = p_start + sj;
    const int s_next = qr.next(sj);
    auto entry = [&](int row) {
        if (row < p) return hacc[(int64_t)row * sj + c];
        return qr.entry(sj, c, row - p);
    };
    // the groups, read ahead as well; after the last the new step's own window
    auto group = [&](int q) { return q < done ? ls.groups[q] : make_int4(p_start, sj, s_next, 0); };
    int4 now = group(0), next = group(1), third = group(2);
    int base = 0;
    double2 qh[AHEAD][W];
    auto load = [&](int q, int rows) {
        const int quarter = (rows + 3) / 4;
        const double2* Qh = ls.qh + (int64_t)q * N * N + lane;
#pragma unroll
        for (int k = 0; k < AHEAD; ++k)
#pragma unroll
            for (int w = 0; w < W; ++w) qh[k][w] = Qh[(int64_t)min(wave * quarter + k, rows - 1) * N + 64 * w];
    };
    double2 fresh = make_double2(0.0, 0.0);  // the row that enters the window with the next step
    auto load_fresh = [&](int row0, int from, int count) {
        if (t < N && t >= from && t < from + count) fresh = entry(row0 + t);
    };
    if (done > 0) {
        load(0, now.y + now.z);
        load_fresh(now.y, now.z, next.y + next.z - now.z);
    }
    if (t < N) x[t] = t < now.y + now.z ? entry(t) : make_double2(0.0, 0.0);
    lds_barrier();
    const int64_t column = (int64_t)p_start + c;
    double2* Rc = ls.R + column * (column + 1) / 2;
    for (int q = 0; q < done; ++q) {
        const int4 fourth = q + 1 < done ? group(q + 3) : now;
        const int rows = now.y + now.z;
        const int quarter = (rows + 3) / 4;
        const int kbeg = wave * quarter, kend = min(rows, kbeg + quarter);
        double2 acc[W];
#pragma unroll
        for (int w = 0; w < W; ++w) acc[w] = make_double2(0.0, 0.0);
        auto add = [&](const double2* row, double2 xk) {
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const double2 y = cmul(row[w], xk);
                acc[w] = make_double2(acc[w].x + y.x, acc[w].y + y.y);
            }
        };
#pragma unroll
        for (int k = 0; k < AHEAD; ++k)
            if (kbeg + k < kend) add(qh[k], x[kbeg + k]);
        if constexpr (W > 1) {
            const double2* Qh = ls.qh + (int64_t)q * N * N + lane;
#pragma unroll 8
            for (int k = kbeg + AHEAD; k < kend; ++k) {
                double2 row[W];
#pragma unroll
                for (int w = 0; w < W; ++w) row[w] = Qh[(int64_t)k * N + 64 * w];
                add(row, x[k]);
            }
        }
#pragma unroll
        for (int w = 0; w < W; ++w) sum[wave][lane + 64 * w] = acc[w];
        const double2 enters = fresh;
        if (q + 1 < done) {
            load(q + 1, next.y + next.z);
            fresh = make_double2(0.0, 0.0);
            load_fresh(base + now.y + next.y, next.z, third.y + third.z - next.z);
        }
        lds_barrier();
        if (t < rows) {
            const double2 y = make_double2(((sum[0][t].x + sum[1][t].x) + sum[2][t].x) + sum[3][t].x,
                                           ((sum[0][t].y + sum[1][t].y) + sum[2][t].y) + sum[3][t].y);
            // the group's own rows are finished; the window moves on by them
            if (t < now.y)
                Rc[base + t] = y;
            else
                x[t - now.y] = y;
        }
        if (t < N && t >= now.z) x[t] = enters;
        lds_barrier();
        base += now.y;
        now = next;
        next = third;
        third = fourth;
    }
    if (t < N) ls.window[(int64_t)c * N + t] = x[t];
}

// Column k = blockIdx.x of Q^H of group `group` with the step just factored, whose
// rows start at `offset` in the group's window: the step's reflectors on the
// column that the group had, or on e_k for the rows that are new to it.
template <int W>
__global__ __launch_bounds__(64) void bk_ls_form_kernel(LsState ls, LsQr qr, int sj, int group, int offset) {
    if (!qr.chain && qr.chol->ok == 0) return;
    constexpr int N = 64 * W;
    const int lane = threadIdx.x;
    const int k = blockIdx.x;
    if (k >= offset + sj + qr.next(sj)) return;
    double2* column = ls.qh + ((int64_t)group * N + k) * N + lane;
    double2 x[W];
#pragma unroll
    for (int w = 0; w < W; ++w)
        x[w] = offset > 0 && k < offset + sj ? column[64 * w] : make_double2(lane + 64 * w == k ? 1.0 : 0.0, 0.0);
    for (int a = 0; a < sj; a += 8) {
        double2 v[8][W];
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const int i = lane + 64 * w - offset;
                const double2 y = ls.refl[(int64_t)min(a + u, sj - 1) * N + max(i, 0)];
                v[u][w] = a + u < sj && i >= 0 ? y : make_double2(0.0, 0.0);  // past the last: no reflection
            }
#pragma unroll
        for (int u = 0; u < 8; ++u) reflect<W>(v[u], x);
    }
#pragma unroll
    for (int w = 0; w < W; ++w) column[64 * w] = x[w];
}

// Householder QR of the new step's windows, its reflectors on the s
// right-hand sides, and their residual norms to the host.  One workgroup.
// Sixteen lanes hold one Hessenberg column and one right-hand side in
// registers (rows l, 16 + l, ...), so a dot product is summed within a row of
// lanes, for four columns at once; across a whole wave the sums alone were
// most of the instructions (24 columns: 43 us, now 28).  A column costs one
// barrier: the owner of the next one reflects it first and forms its reflector
// while the others still apply the present one.
template <int W>
__global__ __launch_bounds__(1024) void bk_ls_factor_kernel(LsState ls, LsQr qr, int sj, int s, int group,
                                                            int offset, int p_start) {
    if (!qr.chain && qr.chol->ok == 0) {
        if (threadIdx.x == 0) ls.host->ok = 0;
        return;
    }
    constexpr int N = 64 * W;
    constexpr int E = N / 16;  // entries of a column in one lane
    __shared__ double2 vbuf[2][N];
    constexpr double kTiny = 1e-30;  // columns below it are left as they are (TINY, gmres_common.rs)
    const int c = threadIdx.x >> 4, l = threadIdx.x & 15;
    const int s_next = qr.next(sj);
    const int rows = sj + s_next;
    double2 h[E], r[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = 16 * e + l;
        h[e] = c < sj && i < rows ? ls.window[(int64_t)c * N + i] : make_double2(0.0, 0.0);
        r[e] = c < s && i < sj ? ls.g[c * ls.ldg + p_start + i] : make_double2(0.0, 0.0);
    }
    // v = (x - beta e_a) / sqrt(norm (norm + |x_a|)), beta = -phase(x_a) norm, from column a
    auto form = [&](int a) {
        double below = 0.0, ax = 0.0, ay = 0.0;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = 16 * e + l;
            if (i > a) below += h[e].x * h[e].x + h[e].y * h[e].y;
            if (i == a) {
                ax = h[e].x;
                ay = h[e].y;
            }
        }
        below = row_sum(below);
        ax = row_sum(ax);
        ay = row_sum(ay);
        const double a2 = ax * ax + ay * ay;
        const bool keep = below < kTiny * kTiny;
        const double n2 = a2 + below;
        const double norm = n2 * rsqrt(n2);
        const double ia = a2 > 0.0 ? rsqrt(a2) : 0.0;
        const double top = a2 * ia;
        const double px = a2 > 0.0 ? ax * ia : 1.0, py = ay * ia;
        const double scale = rsqrt(norm * (norm + top));
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = 16 * e + l;
            double2 v = make_double2(0.0, 0.0);
            if (!keep && i >= a) {
                v = i > a ? make_double2(h[e].x * scale, h[e].y * scale)
                          : make_double2(px * (norm + top) * scale, py * (norm + top) * scale);
                if (i == a) h[e] = make_double2(-px * norm, -py * norm);
            }
            vbuf[a & 1][i] = v;
            ls.refl[(int64_t)a * N + i] = v;
        }
    };
    if (c == 0) form(0);
    for (int a = 0; a < sj; ++a) {
        lds_barrier();
        double2 v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = vbuf[a & 1][16 * e + l];
        auto reflect_rows = [&](double2 (&x)[E], bool on) {
            double2 d = make_double2(0.0, 0.0);
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const double2 y = cmulc(v[e], x[e]);
                d = make_double2(d.x + y.x, d.y + y.y);
            }
            d = make_double2(row_sum(d.x), row_sum(d.y));
            if (!on) d = make_double2(0.0, 0.0);
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const double2 y = cmul(v[e], d);
                x[e] = make_double2(x[e].x - y.x, x[e].y - y.y);
            }
        };
        if ((c | 3) > a && (c & ~3) < sj) reflect_rows(h, c > a);  // per wave: four columns
        if (c == a + 1 && c < sj) form(c);
        if ((c & ~3) < s) reflect_rows(r, true);
    }
    if (c < sj) {
        const int64_t column = (int64_t)p_start + c;
        double2* Rc = ls.R + column * (column + 1) / 2 + p_start;
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (16 * e + l <= c) Rc[16 * e + l] = h[e];
    }
    double tail = 0.0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = 16 * e + l;
        if (c < s && i < rows) ls.g[c * ls.ldg + p_start + i] = r[e];
        if (i >= sj && i < rows) tail += r[e].x * r[e].x + r[e].y * r[e].y;
    }
    tail = sqrt(row_sum(tail));
    if (c < s && l == 0) ls.host->tail[c] = tail;
    if (threadIdx.x == 0) {
        ls.groups[group] = make_int4(p_start - offset, offset + sj, s_next, 0);
        ls.host->next = s_next;
        ls.host->ok = 1;
    }
}

// The outcome of a block QR alone
__global__ void bk_qr_report_kernel(LsQr qr, int sj, BlockStep* host) {
    const int ok = qr.chain ? 1 : qr.chol->ok;
    host->ok = ok;
    host->next = ok ? qr.next(sj) : 0;
}

// g = [C0; 0]: C0 s1 x s row-major
__global__ void bk_ls_reset_kernel(const double2* __restrict__ c0, int s1, int s, double2* __restrict__ g,
                                   int64_t ldg) {
    for (int e = threadIdx.x; e < s1 * s; e += blockDim.x) g[(e % s) * ldg + e / s] = c0[e];
}

// y (cols x s, row-major) from R y = g by back substitution, one right-hand
// side per workgroup, column by column (solve_upper_triangular, gmres_common.rs:
// 110-127; a diagonal entry below its threshold gives y = 0).  The right-hand
// side stands in LDS where it fits, else in `work`.
template <bool LDS>
__global__ __launch_bounds__(256) void bk_ls_solve_kernel(LsState ls, int cols, int s, double2* __restrict__ work,
                                                          double2* __restrict__ y) {
    extern __shared__ double2 in_lds[];
    const int q = blockIdx.x;
    const int t = threadIdx.x;
    double2* b = LDS ? in_lds : work + (int64_t)q * ls.ldg;
    for (int i = t; i < cols; i += 256) b[i] = ls.g[q * ls.ldg + i];
    // columns in fours: their first 1024 rows and the inverses of their diagonal
    // entries are loaded a round ahead
    double2 ahead[4][4], ahead_inv[4];
    auto load = [&](int top) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = max(top - v, 0);
            const double2* Ri = ls.R + (int64_t)i * (i + 1) / 2;
#pragma unroll
            for (int u = 0; u < 4; ++u) ahead[v][u] = Ri[min(t + 256 * u, i)];
            ahead_inv[v] = Ri[i];
        }
    };
    load(cols - 1);
    __syncthreads();
    for (int top = cols - 1; top >= 0; top -= 4) {
        double2 col[4][4], inv[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
#pragma unroll
            for (int u = 0; u < 4; ++u) col[v][u] = ahead[v][u];
            const double2 d = ahead_inv[v];
            const double n2 = d.x * d.x + d.y * d.y;
            inv[v] = hypot(d.x, d.y) > 1e-30 ? make_double2(d.x / n2, -d.y / n2) : make_double2(0.0, 0.0);
        }
        load(max(top - 4, 0));
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = top - v;
            if (i < 0) break;
            const double2 yi = cmul(b[i], inv[v]);
            if (t == 0) y[(int64_t)i * s + q] = yi;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k = t + 256 * u;
                if (k < i) {
                    const double2 x = cmul(col[v][u], yi);
                    const double2 z = b[k];
                    b[k] = make_double2(z.x - x.x, z.y - x.y);
                }
            }
            for (int k = t + 1024; k < i; k += 256) {
                const double2 x = cmul(ls.R[(int64_t)i * (i + 1) / 2 + k], yi);
                const double2 z = b[k];
                b[k] = make_double2(z.x - x.x, z.y - x.y);
            }
            if constexpr (LDS)
                lds_barrier();
            else
                __syncthreads();
        }
    }
}

inline unsigned blocks_for(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

// ---------------------------------------------------------------- launchers

// Basis vectors of a Gram tile for sj columns: 32, or 16 where two tiles'
// sums would not leave registers for the loads ahead.
int bk_gram_tile(int sj) { return sj <= 32 ? 32 : 16; }

// K slices: about 1024 workgroups, as long as each of a slice's four waves
// has 32 rows (two rounds of loads ahead of the products).
int bk_gram_slices(int64_t n, int p, int tile) {
    const int itiles = (p + tile - 1) / tile;
    const int64_t want = (1024 + itiles - 1) / itiles;
    const int64_t most = n / 128;
    return (int)std::max<int64_t>(1, (std::min(want, most) + BK_XCD - 1) / BK_XCD) * BK_XCD;
}

// Partials of any Gram product of a solve: p <= max_basis, sj <= s
int64_t bk_gram_partial_elems(int64_t n, int max_basis, int s) {
    int64_t rows = 0;
    for (int p = 1; p <= max_basis; ++p)
        for (int tile = 16; tile <= 32; tile *= 2) rows = std::max(rows, (int64_t)bk_gram_slices(n, p, tile) * p);
    return rows * 2 * s;
}

// part: bk_gram_partial_elems; gram: p*sj; hacc: p*sj (hmode 0 none, 1 set, 2 add)
void bk_gram(sbh_context* ctx, const double2* V, int64_t ldv, int p, const double2* W, int64_t ldw, int sj,
             int64_t n, double* part, double2* gram, double2* hacc, int hmode, const int* flag) {
    SBH_REQUIRE(sj >= 1 && sj <= QR_MAXC && p >= 1, "block Gram shape");
    hipEvent_t ev;
    ctx->begin_timed(SBH_KERNEL_KRYLOV_VECTOR, &ev);
    const int tile = bk_gram_tile(sj);
    const int slices = bk_gram_slices(n, p, tile);
    const int itiles = (p + tile - 1) / tile;
    const int64_t kslice = ((n + slices - 1) / slices + 31) / 32 * 32;  // four waves, 8 rows a load
    const dim3 grid((unsigned)(slices * itiles));
#define SBH_BG(NT_, MB_)                                                                                           \
    hipLaunchKernelGGL((bk_gram_kernel<NT_, MB_>), grid, dim3(BK_THREADS), 0, ctx->stream, V, ldv, p, W, ldw, sj, n, \
                       kslice, itiles, part, flag)
    if (sj <= 8) SBH_BG(1, 2);
    else if (sj <= 16) SBH_BG(2, 2);
    else if (sj <= 24) SBH_BG(3, 2);
    else if (sj <= 32) SBH_BG(4, 2);
    else if (sj <= 48) SBH_BG(6, 1);
    else SBH_BG(8, 1);
#undef SBH_BG
    SBH_HIP(hipGetLastError());
    hipLaunchKernelGGL(bk_gram_reduce_kernel, dim3(blocks_for((int64_t)p * sj, 64)), dim3(64), 0,
                       ctx->stream, part, slices, p, sj, gram, hacc, hmode, flag);
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_KRYLOV_VECTOR, ev);
}

void bk_combine(sbh_context* ctx, const double2* V, int64_t ldv, int p, const double2* C, int ldc, int sj, int64_t n,
                double2* O, int64_t osc, int64_t osk, bool add, double alpha, const int* flag) {
    SBH_REQUIRE(sj >= 1 && sj <= QR_MAXC, "block combination width");
    if (p <= 0) return;
    hipEvent_t ev;
    ctx->begin_timed(SBH_KERNEL_KRYLOV_VECTOR, &ev);
    const dim3 grid(blocks_for(n, BK_CK));
    const int mt = (sj + 15) / 16;
#define SBH_BC(MT_)                                                                                             \
    hipLaunchKernelGGL(bk_combine_kernel<MT_>, grid, dim3(BK_THREADS), 0, ctx->stream, V, ldv, p, C, ldc, sj, n, O, \
                       osc, osk, add ? 1 : 0, alpha, flag)
    if (mt == 1) SBH_BC(1);
    else if (mt == 2) SBH_BC(2);
    else if (mt == 3) SBH_BC(3);
    else SBH_BC(4);
#undef SBH_BC
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_KRYLOV_VECTOR, ev);
}

size_t bk_cholesky_state_bytes(int m) { return offsetof(CholState, r) + sizeof(double2) * (size_t)m * m; }

// One Cholesky QR pass on the m x m Gram matrix G; T (m x m) = R^-1
void bk_cholesky(sbh_context* ctx, const double2* G, int m, double floor, int pass, void* state, double2* T) {
    SBH_REQUIRE(m >= 1 && m <= QR_MAXC, "block QR width");
    hipLaunchKernelGGL(bk_cholesky_kernel, dim3(1), dim3((unsigned)((m + 3) / 4 * 64)), 0, ctx->stream, G, m, floor, pass,
                       static_cast<CholState*>(state), T);
    SBH_HIP(hipGetLastError());
}

void bk_to_rowmajor(sbh_context* ctx, const double2* in, int64_t ld, int cols, int64_t n, double2* out) {
    hipLaunchKernelGGL(bk_to_rowmajor_kernel, dim3(blocks_for(n, 64), blocks_for(cols, 16)), dim3(BK_THREADS), 0,
                       ctx->stream, in, ld, cols, n, out);
    SBH_HIP(hipGetLastError());
}

void bk_to_colmajor(sbh_context* ctx, const double2* in, int cols, int64_t n, const double2* d, double2* out,
                    int64_t ld) {
    hipLaunchKernelGGL(bk_to_colmajor_kernel, dim3(blocks_for(n, 64), blocks_for(cols, 16)), dim3(BK_THREADS), 0,
                       ctx->stream, in, cols, n, d, out, ld);
    SBH_HIP(hipGetLastError());
}

void bk_residual_cm(sbh_context* ctx, const double2* B, const double2* AX, int s, int64_t n, const double2* d,
                    double2* R) {
    hipLaunchKernelGGL(bk_residual_cm_kernel, dim3(blocks_for(n, 64), blocks_for(s, 16)), dim3(BK_THREADS), 0,
                       ctx->stream, B, AX, s, n, d, R);
    SBH_HIP(hipGetLastError());
}

int bk_norm_chunks(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(256, (n + 4095) / 4096)); }

// out[c] = ||X_c|| for cols contiguous vectors (stride ld); part: chunks * cols doubles
void bk_colnorms(sbh_context* ctx, const double2* X, int64_t ld, int cols, int64_t n, double* part, double* out) {
    const int chunks = bk_norm_chunks(n);
    const int64_t len = (n + chunks - 1) / chunks;
    hipLaunchKernelGGL(bk_colnorm_partials_kernel, dim3(chunks, cols), dim3(BK_THREADS), 0, ctx->stream, X, ld, cols,
                       n, len, part);
    SBH_HIP(hipGetLastError());
    hipLaunchKernelGGL(bk_sum_sqrt_kernel, dim3(blocks_for(cols, 64)), dim3(64), 0, ctx->stream, part, chunks, cols,
                       out);
    SBH_HIP(hipGetLastError());
}

// squared Frobenius partials of one contiguous block (count complex values)
int bk_frob_partials(sbh_context* ctx, const double2* X, int64_t count, double* part) {
    const int chunks = bk_norm_chunks(count);
    const int64_t len = (count + chunks - 1) / chunks;
    hipLaunchKernelGGL(bk_colnorm_partials_kernel, dim3(chunks, 1), dim3(BK_THREADS), 0, ctx->stream, X, count, 1,
                       count, len, part);
    SBH_HIP(hipGetLastError());
    return chunks;
}

void bk_dgks_flag(sbh_context* ctx, const double* before, const double* after, int chunks, int* flag, double* frob) {
    hipLaunchKernelGGL(bk_dgks_flag_kernel, dim3(1), dim3(64), 0, ctx->stream, before, after, chunks, flag, frob);
    SBH_HIP(hipGetLastError());
}

// part: chunks * 3s doubles; returns the chunk count (partials to be summed by the caller's kernel)
void bk_true_metrics(sbh_context* ctx, const double2* B, const double2* AX, int s, int64_t n, double* part,
                     double* out) {
    const int chunks = bk_norm_chunks(n);
    const int64_t len = (n + chunks - 1) / chunks;
    hipLaunchKernelGGL(bk_true_partials_kernel, dim3(chunks, s), dim3(BK_THREADS), 0, ctx->stream, B, AX, s, n, len,
                       part);
    SBH_HIP(hipGetLastError());
    hipLaunchKernelGGL(bk_sum_sqrt_kernel, dim3(blocks_for(3 * s, 64)), dim3(64), 0, ctx->stream, part, chunks, 3 * s,
                       out);
    SBH_HIP(hipGetLastError());
}

size_t bk_qr_state_bytes() { return sizeof(QrState); }
int bk_qr_chunks(int64_t n) { return (int)((n + QR_CHUNK - 1) / QR_CHUNK); }
size_t bk_qr_partial_elems(int64_t n) { return (size_t)bk_qr_chunks(n) * QR_SLOTS; }

// Block QR with rank-drop deflation of the sj column-major vectors W into the
// directions Q (slots 0..); state (its counter zero between launches) and
// partials on the device.  Three launches per column plus one to write the
// last direction.
void bk_block_qr(sbh_context* ctx, double2* W, double2* Q, int64_t n, int sj, int budget, void* state,
                 double2* part) {
    SBH_REQUIRE(sj >= 1 && sj <= QR_MAXC, "block QR width");
    QrArgs a;
    a.W = W;
    a.Q = Q;
    a.n = n;
    a.sj = sj;
    a.budget = budget;
    a.defl_tol = std::sqrt(2.220446049250313e-16);
    a.st = static_cast<QrState*>(state);
    a.part = part;
    const int chunks = bk_qr_chunks(n);
    const dim3 grid((unsigned)chunks);
    hipEvent_t ev;
    ctx->begin_timed(SBH_KERNEL_KRYLOV_VECTOR, &ev);
    for (int c = 0; c <= sj; ++c) {
        hipLaunchKernelGGL(bk_qr_start_kernel, grid, dim3(BK_THREADS), 0, ctx->stream, a, c);
        if (c == sj) break;
        hipLaunchKernelGGL(bk_qr_project_kernel, grid, dim3(BK_THREADS), 0, ctx->stream, a, c, 0);
        hipLaunchKernelGGL(bk_qr_project_kernel, grid, dim3(BK_THREADS), 0, ctx->stream, a, c, 1);
    }
    SBH_HIP(hipGetLastError());
    ctx->end_timed(SBH_KERNEL_KRYLOV_VECTOR, ev);
}

size_t bk_ls_window(int s) { return s <= 32 ? 64 : 128; }

BlockLeastSquares::BlockLeastSquares(sbh_context* ctx, int64_t n, int s, int max_basis, int max_steps)
    : ctx_(ctx), n_(n), s_(s), max_basis_(max_basis), max_steps_(max_steps) {}

void BlockLeastSquares::allocate() {
    const size_t window = bk_ls_window(s_);
    refl_.allocate((size_t)s_ * window);
    window_.allocate((size_t)s_ * window);
    host_.allocate(1);
    make_room((int)std::min<int64_t>(max_steps_, n_ + 1), (int)std::min<int64_t>(max_basis_, n_ + 2 * s_));
}

// A step opens a group where the last one has more than window - 2 s columns.
int64_t BlockLeastSquares::most_groups(int s, int64_t steps, int64_t cols) {
    return std::min(steps, cols / ((int64_t)bk_ls_window(s) - 2 * s + 1) + 1);
}

int64_t BlockLeastSquares::room_bytes(int s, int64_t steps, int64_t cols) {
    const int64_t window = (int64_t)bk_ls_window(s);
    const int64_t groups = most_groups(s, steps, cols);
    return (int64_t)sizeof(int4) * groups +
           (int64_t)sizeof(double2) * (groups * window * window + cols * (cols + 1) / 2 + 2 * (cols + s) * s);
}

int64_t BlockLeastSquares::device_bytes(int64_t n, int s, int64_t restart) {
    const int64_t steps = std::min(restart, n + 1);
    const int64_t cols = std::min((steps + 1) * s, n + 2 * s);
    return room_bytes(s, steps, cols) + (int64_t)sizeof(double2) * 2 * s * (int64_t)bk_ls_window(s);
}

// Arrays for `steps` steps with `cols` columns; the columns added so far are kept.
void BlockLeastSquares::make_room(int steps, int cols) {
    const size_t window = bk_ls_window(s_);
    const int64_t ldg = cols + s_;
    const size_t most = (size_t)most_groups(s_, steps, cols);
    WorkArray<int4> groups(most);
    WorkArray<double2> qh(most * window * window), R((size_t)cols * (cols + 1) / 2), g((size_t)ldg * s_),
        work((size_t)ldg * s_);
    auto keep = [&](void* to, const void* from, size_t bytes) {
        if (bytes) SBH_HIP(hipMemcpyAsync(to, from, bytes, hipMemcpyDeviceToDevice, ctx_->stream));
    };
    keep(groups.ptr, groups_.ptr, sizeof(int4) * ngroups_);
    keep(qh.ptr, qh_.ptr, sizeof(double2) * ngroups_ * window * window);
    keep(R.ptr, R_.ptr, sizeof(double2) * ((size_t)cols_ * (cols_ + 1) / 2));
    if (ldg_)
        SBH_HIP(hipMemcpy2DAsync(g.ptr, sizeof(double2) * ldg, g_.ptr, sizeof(double2) * ldg_, sizeof(double2) * ldg_,
                                 s_, hipMemcpyDeviceToDevice, ctx_->stream));
    groups_.swap(groups);
    qh_.swap(qh);
    R_.swap(R);
    g_.swap(g);
    work_.swap(work);
    ldg_ = ldg;
    room_cols_ = cols;
    room_steps_ = steps;
}

namespace {
LsState ls_state(int4* groups, double2* refl, double2* qh, double2* R, double2* window, double2* g, int64_t ldg,
                 BlockStep* host) {
    return LsState{groups, refl, qh, R, window, g, ldg, host};
}
LsQr ls_qr(const void* chol, const void* chain) {
    return LsQr{static_cast<const CholState*>(chol), static_cast<const QrState*>(chain)};
}
}  // namespace

void BlockLeastSquares::report(const void* chol, const void* chain, int sj) {
    hipLaunchKernelGGL(bk_qr_report_kernel, dim3(1), dim3(1), 0, ctx_->stream, ls_qr(chol, chain), sj, host_.ptr);
    SBH_HIP(hipGetLastError());
}

void BlockLeastSquares::reset(const double2* c0, int s1) {
    done_ = 0;
    cols_ = 0;
    ngroups_ = 0;
    open_ = 0;
    hipLaunchKernelGGL(bk_ls_reset_kernel, dim3(1), dim3(BK_THREADS), 0, ctx_->stream, c0, s1, s_, g_.ptr, ldg_);
    SBH_HIP(hipGetLastError());
}

bool BlockLeastSquares::joins(int sj) const {
    return ngroups_ > 0 && open_ + 2 * sj <= (int)bk_ls_window(s_);
}

void BlockLeastSquares::accept(int sj) {
    if (joins(sj)) {
        open_ += sj;
    } else {
        ngroups_ += 1;
        open_ = sj;
    }
    done_ += 1;
    cols_ += sj;
}

void BlockLeastSquares::add(const void* chol, const void* chain, const double2* hacc, int sj) {
    SBH_REQUIRE(sj >= 1 && sj <= s_ && done_ < max_steps_ && cols_ + sj <= max_basis_, "block least-squares step");
    if (done_ + 1 > room_steps_ || cols_ + sj > room_cols_) {
        // without numbers the solve ends as a numerical error however long it goes on
        for (int c = 0; c < s_ && done_ > 0; ++c)
            if (!std::isfinite(host_.ptr->tail[c]))
                throw Error(SBH_ERR_NUMERICAL, "block GMRES generated NaN or infinity in its basis");
        auto grown = [](int room, int need, int most) {
            return need <= room ? room : (int)std::min<int64_t>(most, std::max<int64_t>(need, 2 * (int64_t)room));
        };
        const int steps = grown(room_steps_, done_ + 1, max_steps_), cols = grown(room_cols_, cols_ + sj, max_basis_);
        admit_device(ctx_, room_bytes(s_, steps, cols), "the block least squares", false);
        make_room(steps, cols);
    }
    hipEvent_t ev;
    ctx_->begin_timed(SBH_KERNEL_KRYLOV_VECTOR, &ev);
    const LsState st = ls_state(groups_.ptr, refl_.ptr, qh_.ptr, R_.ptr, window_.ptr, g_.ptr, ldg_, host_.ptr);
    const LsQr qr = ls_qr(chol, chain);
    const unsigned threads = (unsigned)((s_ + 3) / 4 * 64);  // sixteen lanes to a column
    const int group = joins(sj) ? ngroups_ - 1 : ngroups_, offset = joins(sj) ? open_ : 0;
    auto launch = [&](auto w) {
        constexpr int W = decltype(w)::value;
        hipLaunchKernelGGL(bk_ls_apply_kernel<W>, dim3(sj), dim3(256), 0, ctx_->stream, st, qr, hacc, sj, ngroups_, cols_);
        hipLaunchKernelGGL(bk_ls_factor_kernel<W>, dim3(1), dim3(threads), 0, ctx_->stream, st, qr, sj, s_, group, offset,
                           cols_);
        hipLaunchKernelGGL(bk_ls_form_kernel<W>, dim3(offset + 2 * sj), dim3(64), 0, ctx_->stream, st, qr, sj, group,
                           offset);
    };
    if (bk_ls_window(s_) == 64)
        launch(std::integral_constant<int, 1>());
    else
        launch(std::integral_constant<int, 2>());
    SBH_HIP(hipGetLastError());
    ctx_->end_timed(SBH_KERNEL_KRYLOV_VECTOR, ev);
}

void BlockLeastSquares::solve(double2* y) {
    const size_t bytes = sizeof(double2) * (size_t)cols_;
    const LsState st = ls_state(groups_.ptr, refl_.ptr, qh_.ptr, R_.ptr, window_.ptr, g_.ptr, ldg_, host_.ptr);
    if (bytes <= (64u << 10))  // what a launch may ask for
        hipLaunchKernelGGL(bk_ls_solve_kernel<true>, dim3(s_), dim3(256), bytes, ctx_->stream, st, cols_, s_, work_.ptr, y);
    else
        hipLaunchKernelGGL(bk_ls_solve_kernel<false>, dim3(s_), dim3(256), 0, ctx_->stream, st, cols_, s_, work_.ptr, y);
    SBH_HIP(hipGetLastError());
}

}  // namespace sbh
