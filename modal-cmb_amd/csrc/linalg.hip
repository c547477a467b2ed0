// FP64 orthonormalisation on the GPU (ortho_prim_mpi.c:198-284) and the
// Cholesky solve of the projection (eigenmode_mpi.c:195-219).
//
//   norm_i = sqrt(G_ii),  C = D^-1 G D^-1 = L L^T  (blocked right-looking
//   Cholesky, block OB: row-parallel substitution of the panel, SYRK update of
//   the trailing lower triangle on FP64 MFMA, whose first workgroup factors the
//   next diagonal block), L^-1 by joining inverted diagonal blocks pairwise,
//   X21 = -X22 L21 X11, on FP64 MFMA.
//   ortho  = symmetrised D L          (update_ortho, fixed_data.c:3285-3295)
//   lambda = symmetrised (D L)^-1     (update_lambda, fixed_data.c:3576-3586)
// A non-positive pivot sets a device flag (first failing column + 1); later
// kernels see it and return, and the host reports MCMB_ERR_NOT_SPD.
#include "mcmb_internal.h"
#include <algorithm>
#include <vector>

namespace mcmb {

constexpr int NB = 32;     // substitution block of many right-hand sides
constexpr int OB = 64;     // Cholesky, inverse and few-right-hand-side block

typedef double fd4 __attribute__((ext_vector_type(4)));

__global__ void la_norm_kernel(const double* __restrict__ G, int n, double* __restrict__ norm)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) norm[i] = sqrt(G[(size_t)i * n + i]);
}

__global__ void la_scale_kernel(const double* __restrict__ G, int n, const double* __restrict__ norm,
                                double* __restrict__ C)
{
    size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)n * n) return;
    int i = (int)(e / n), j = (int)(e % n);
    C[e] = G[e] / (norm[i] * norm[j]);
}

// value of a double in lane src (uniform) of the wave
__device__ __forceinline__ double lane_value(double x, int src)
{
    const int lo = __builtin_amdgcn_readlane(__double2loint(x), src);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(x), src);
    return __hiloint2double(hi, lo);
}

// s = sqrt(d), r = 1 / s by Goldschmidt's iteration from the hardware's
// reciprocal square root and a last residual step (d from 1e-280 up): a third
// of the dependent chain of a square root followed by a division.
__device__ __forceinline__ void sqrt_rcp(double d, double* s, double* r)
{
    if (d < 1e-280) {
        *s = sqrt(d);
        *r = 1.0 / *s;
        return;
    }
    const double y = __builtin_amdgcn_rsq(d);
    double g = d * y, h = 0.5 * y;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const double e = __builtin_fma(-h, g, 0.5);
        g = __builtin_fma(g, e, g);
        h = __builtin_fma(h, e, h);
    }
    *s = __builtin_fma(__builtin_fma(-g, g, d), h, g);
    *r = 2.0 * h;
}
// a / s with r = 1 / s to rounding
__device__ __forceinline__ double div_by(double a, double s, double r)
{
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-q, s, a), r, q);
}

// Cholesky of the OB x OB matrix in S (lower triangle, rows past nb the
// identity) by 256 threads, in panels of 16 columns: wave 0 factors a panel
// with lane = row and the panel's columns in registers (no barrier per column,
// the pivot row's values come by lane reads), then all waves update the
// columns right of it on FP64 MFMA.  A pivot that is not positive sets *flag
// to its column + 1 (k0 = the block's first column) and returns false in every
// thread.  About 20 us, 0.3 us a column, bound by the chain of lane reads and
// the square root; 0.77 us when each column took three barriers of a workgroup.
__device__ __forceinline__ bool potrf_block(double (*S)[OB + 1], int* bad, int nb, int k0, int* flag)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) *bad = 0;
    __syncthreads();
    for (int p = 0; p < 4; ++p) {
        const int c0 = 16 * p;
        if (wave == 0) {
            double a[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) a[j] = S[lane][c0 + j];
            int b = 0;
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const double d = lane_value(a[j], c0 + j);
                if (!(d > 0.0) && !b) b = k0 + c0 + j + 1;   // (the rest of the panel is not used)
                double s, r;
                sqrt_rcp(d, &s, &r);
                a[j] = lane == c0 + j ? s : div_by(a[j], s, r);
#pragma unroll
                for (int l = j + 1; l < 16; ++l) a[l] -= a[j] * lane_value(a[j], c0 + l);
            }
#pragma unroll
            for (int j = 0; j < 16; ++j)
                if (lane >= c0 + j) S[lane][c0 + j] = a[j];
            if (b && lane == 0) *bad = b;
        }
        __syncthreads();
        if (*bad) {
            if (tid == 0) atomicCAS(flag, 0, *bad);
            return false;
        }
        if (c0 + 16 >= nb) break;
        int t = 0;
        for (int bj = p + 1; bj < 4; ++bj)
            for (int bi = bj; bi < 4; ++bi, ++t) {
                if ((t & 3) != wave) continue;
                // the chain starts from the element, as in the panel's updates
                fd4 acc;
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[v] = S[16 * bi + 4 * v + (lane >> 4)][16 * bj + (lane & 15)];
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    const int k = c0 + 4 * ks + (lane >> 4);
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-S[16 * bi + (lane & 15)][k],
                                                              S[16 * bj + (lane & 15)][k], acc, 0, 0, 0);
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) S[16 * bi + 4 * v + (lane >> 4)][16 * bj + (lane & 15)] = acc[v];
            }
        __syncthreads();
    }
    return true;
}

// The OB x OB lower triangle at (k0, k0) of the row-major n x n matrix M, into
// S; rows and columns past nb: the identity, the upper triangle 0.
// (256 threads; all loads of a thread are in flight at once).  TR: transposed.
template <bool TR>
__device__ __forceinline__ void load_block(const double* __restrict__ M, int n, int k0, int nb, double (*S)[OB + 1])
{
    double v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int e = threadIdx.x + 256 * u, i = e / OB, j = e % OB;
        v[u] = (i < nb && j <= i) ? M[(size_t)(k0 + i) * n + k0 + j] : (i == j ? 1.0 : 0.0);
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int e = threadIdx.x + 256 * u, i = e / OB, j = e % OB;
        if (TR) S[j][i] = v[u];
        else S[i][j] = v[u];
    }
}

__device__ __forceinline__ void store_block(const double (*S)[OB + 1], int n, int k0, int nb, double* __restrict__ M)
{
    for (int e = threadIdx.x; e < OB * OB; e += 256) {
        const int i = e / OB, j = e % OB;
        if (i < nb && j <= i) M[(size_t)(k0 + i) * n + k0 + j] = S[i][j];
    }
}

// The first diagonal block (the others are factored by la_syrk).
__global__ __launch_bounds__(256) void la_potrf_first(double* __restrict__ C, int n, int* __restrict__ flag)
{
    __shared__ double S[OB][OB + 1];
    __shared__ int bad;
    const int nb = min(OB, n);
    load_block<false>(C, n, 0, nb, S);
    if (!potrf_block(S, &bad, nb, 0, flag)) return;
    store_block(S, n, 0, nb, C);
}

// Panel rows i >= k0 + OB: L[i, k0:k0+OB] = C[i, k0:k0+OB] L_kk^-T, 64 rows a
// workgroup, by substitution (backward stable whatever the condition of the
// block): all threads load, wave 0 solves with lane = row, the row in
// registers and L_kk read from LDS as broadcasts.  Columns j + 1.. are updated
// as soon as x_j is known, so the dependent chain per column is a product and
// a difference.  17.7 us for 64 columns (17.1 us for 32 with a row per thread
// of 256-row workgroups).
__global__ __launch_bounds__(256) void la_trsm_panel(double* __restrict__ C, int n, int k0, const int* __restrict__ flag)
{
    __shared__ double Lk[OB][OB + 1], X[64][OB + 1], rd[OB];
    if (*flag) return;
    const int tid = threadIdx.x, r0 = k0 + OB + 64 * blockIdx.x;
    double v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int e = tid + 256 * u, i = r0 + e / OB;
        v[u] = i < n ? C[(size_t)i * n + k0 + e % OB] : 0.0;
    }
    load_block<true>(C, n, k0, OB, Lk);   // column j of the block is a row of LDS
#pragma unroll
    for (int u = 0; u < 16; ++u) X[(tid + 256 * u) / OB][tid % OB] = v[u];
    __syncthreads();
    if (tid < OB) {
        rd[tid] = 1.0 / Lk[tid][tid];
        double x[OB];
#pragma unroll
        for (int j = 0; j < OB; ++j) x[j] = X[tid][j];
#pragma unroll
        for (int j = 0; j < OB; ++j) {
            x[j] = div_by(x[j], Lk[j][j], rd[j]);
#pragma unroll
            for (int l = j + 1; l < OB; ++l) x[l] -= x[j] * Lk[j][l];
        }
#pragma unroll
        for (int j = 0; j < OB; ++j) X[tid][j] = x[j];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int e = tid + 256 * u, i = r0 + e / OB;
        if (i < n) C[(size_t)i * n + k0 + e % OB] = X[e / OB][e % OB];
    }
}

// Tiles of 64 x 64: 128 x 128 ones, at two rounds of the CUs or fewer, took 79
// against 46 us for the trailing update at m = 4000 and 1.5 times as long for
// the joins of the inverse.
constexpr int LT = 64;

// acc += sum over k in [k0, k1) of A(i, k) B(j, k) on an LT x LT tile: rows i of A
// from ra (below ea), columns j from rb (below eb), A(i, k) = A[i lda + k] and
// B(j, k) = B[j ldb + k] (KN: B[k ldb + j]).  256 threads, wave w the 32 x 32
// quadrant (w >> 1, w & 1); 16 K rows per LDS stage, double-buffered, the next
// stage loaded during this one's products.  Rows of 17 doubles: fragment reads
// and stores are free of bank conflicts.
template <bool KN>
__device__ __forceinline__ void tile_product(const double* __restrict__ A, long lda, int ra, int ea,
                                             const double* __restrict__ B, long ldb, int rb, int eb, int k0, int k1,
                                             double (*As)[LT][17], double (*Bs)[LT][17], fd4 (&acc)[LT / 32][LT / 32])
{
    constexpr int U = LT / 16;   // elements a thread stages of either operand
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave >> 1) * (LT / 2), wn = (wave & 1) * (LT / 2);
    double va[U], vb[U];
    const int kk = tid & 15, r = tid >> 4;
    auto gload = [&](int k) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = ra + r + 16 * u;
            va[u] = (i < ea && k + kk < k1) ? A[(long)i * lda + k + kk] : 0.0;
            if (KN) {
                const int e = tid + 256 * u, kb = k + e / LT, j = rb + e % LT;
                vb[u] = (j < eb && kb < k1) ? B[(long)kb * ldb + j] : 0.0;
            } else {
                const int j = rb + r + 16 * u;
                vb[u] = (j < eb && k + kk < k1) ? B[(long)j * ldb + k + kk] : 0.0;
            }
        }
    };
    auto sstore = [&](int buf) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            As[buf][r + 16 * u][kk] = va[u];
            if (KN) Bs[buf][(tid + 256 * u) % LT][(tid + 256 * u) / LT] = vb[u];
            else Bs[buf][r + 16 * u][kk] = vb[u];
        }
    };
    if (k0 >= k1) return;
    gload(k0);
    sstore(0);
    __syncthreads();
    int buf = 0;
    for (int k = k0; k < k1; k += 16, buf ^= 1) {
        const bool more = k + 16 < k1;
        if (more) gload(k + 16);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int q = 4 * ks + (lane >> 4);
            double av[LT / 32], bv[LT / 32];
#pragma unroll
            for (int x = 0; x < LT / 32; ++x) {
                av[x] = As[buf][wm + 16 * x + (lane & 15)][q];
                bv[x] = Bs[buf][wn + 16 * x + (lane & 15)][q];
            }
#pragma unroll
            for (int x = 0; x < LT / 32; ++x)
#pragma unroll
                for (int y = 0; y < LT / 32; ++y)
                    acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[x], bv[y], acc[x][y], 0, 0, 0);
        }
        if (more) sstore(buf ^ 1);
        __syncthreads();
    }
}

// lower tile index t -> (I, J), I >= J
__device__ __forceinline__ void lower_tile(int t, int* I, int* J)
{
    int i = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
    while ((i + 1) * (i + 2) / 2 <= t) ++i;
    while (i * (i + 1) / 2 > t) --i;
    *I = i;
    *J = t - i * (i + 1) / 2;
}

// The trailing update C(i, j) -= sum_{k < OB} L(i, k0 + k) L(j, k0 + k), i >= j >=
// k1 = k0 + OB, on LT x LT tiles; the workgroup of the first tile, whose values
// are final then, goes on to factor the next diagonal block, so that its
// latency is hidden by the other tiles.  37 us on average over n = 4960: the
// traffic of C (read and written once per 64 columns) and, below m = 2000, the
// diagonal block.
__global__ __launch_bounds__(256) void la_syrk(double* __restrict__ C, int n, int k0, int* __restrict__ flag)
{
    // the diagonal block is factored where the operand stages were
    __shared__ double mem[4 * LT * 17];
    __shared__ int bad;
    static_assert(4 * LT * 17 >= OB * (OB + 1), "the diagonal block fits the stages");
    auto As = reinterpret_cast<double(*)[LT][17]>(mem), Bs = reinterpret_cast<double(*)[LT][17]>(mem + 2 * LT * 17);
    auto S = reinterpret_cast<double(*)[OB + 1]>(mem);
    if (*flag) return;
    int I, J;
    lower_tile(blockIdx.x, &I, &J);
    const int k1 = k0 + OB, ra = k1 + LT * I, rb = k1 + LT * J;
    fd4 acc[LT / 32][LT / 32];
#pragma unroll
    for (int x = 0; x < LT / 32; ++x)
#pragma unroll
        for (int y = 0; y < LT / 32; ++y) acc[x][y] = (fd4){0.0, 0.0, 0.0, 0.0};
    tile_product<false>(C, n, ra, n, C, n, rb, n, k0, k1, As, Bs, acc);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave >> 1) * (LT / 2), wn = (wave & 1) * (LT / 2);
    const int nb = min(OB, n - k1);
    if (blockIdx.x == 0)
        for (int e = threadIdx.x; e < OB * OB; e += 256) S[e / OB][e % OB] = e / OB == e % OB ? 1.0 : 0.0;
    __syncthreads();
#pragma unroll
    for (int x = 0; x < LT / 32; ++x)
#pragma unroll
        for (int y = 0; y < LT / 32; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int a = wm + 16 * x + 4 * v + (lane >> 4), b = wn + 16 * y + (lane & 15);
                const int i = ra + a, j = rb + b;
                if (i < n && j <= i) {
                    const double z = C[(size_t)i * n + j] - acc[x][y][v];
                    if (blockIdx.x == 0 && a < nb) S[a][b] = z;
                    else C[(size_t)i * n + j] = z;
                }
            }
    if (blockIdx.x != 0) return;
    __syncthreads();
    if (!potrf_block(S, &bad, nb, k1, flag)) return;
    store_block(S, n, k1, nb, C);
}

// X_bb = L_bb^-1 of every OB x OB diagonal block, lane = column of wave 0, by
// substitution; X row-major with zeros above the diagonal.
__global__ __launch_bounds__(256) void la_inv_diag(const double* __restrict__ L, int n, double* __restrict__ X)
{
    __shared__ double S[OB][OB + 1], E[64][OB + 1];
    const int k0 = OB * blockIdx.x, nb = min(OB, n - k0), c = threadIdx.x;
    load_block<true>(L, n, k0, nb, S);   // the column that x_i multiplies is contiguous
    __syncthreads();
    if (c >= 64) return;
    // 16 components at a time in registers, the finished ones in LDS
    for (int q = 0; q < OB; q += 16) {
        double x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = q + i == c ? 1.0 : 0.0;
        for (int j = 0; j < q; ++j) {
            const double xj = E[c][j];
#pragma unroll
            for (int i = 0; i < 16; ++i) x[i] -= xj * S[j][q + i];
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            x[j] = x[j] / S[q + j][q + j];
#pragma unroll
            for (int l = j + 1; l < 16; ++l) x[l] -= x[j] * S[q + j][q + l];
            E[c][q + j] = x[j];
            if (q + j < nb && c < nb) X[(size_t)(k0 + q + j) * n + k0 + c] = x[j];
        }
    }
}

// One level of the inverse: the blocks of size s on X's diagonal are done, and
// pairs of them are joined, X21 = -X22 (L21 X11), all pairs at once.  STEP 1:
// W21 = L21 X11 (into W, at the place of L21); STEP 2: X21 = -X22 W21.  The
// triangles bound the sums: k >= the tile's first column, k <= its last row.
// (n^3 / 3 products in 2 log2(n / 64) launches; the tiles of every column of
// X at once, where substitution column block by column block took 2 n / 32
// dependent launches.)
template <int STEP>
__global__ __launch_bounds__(256) void la_inv_join(const double* __restrict__ L, double* __restrict__ X,
                                                      double* __restrict__ W, int n, int s)
{
    __shared__ double As[2][LT][17], Bs[2][LT][17];
    const int nt = (s + LT - 1) / LT, o = 2 * s * blockIdx.y, m0 = o + s, m1 = min(o + 2 * s, n);
    // the longest sums first: the first columns in step 1, the last rows in step 2
    const int hi = blockIdx.x / nt, lo = blockIdx.x % nt, I = STEP == 1 ? lo : nt - 1 - hi, J = STEP == 1 ? hi : lo;
    const int ra = m0 + LT * I, rb = o + LT * J;
    if (ra >= m1 || rb >= m0) return;
    fd4 acc[LT / 32][LT / 32];
#pragma unroll
    for (int x = 0; x < LT / 32; ++x)
#pragma unroll
        for (int y = 0; y < LT / 32; ++y) acc[x][y] = (fd4){0.0, 0.0, 0.0, 0.0};
    if (STEP == 1) tile_product<true>(L, n, ra, m1, X, n, rb, m0, rb, m0, As, Bs, acc);
    else tile_product<true>(X, n, ra, m1, W, n, rb, m0, m0, min(m1, ra + LT), As, Bs, acc);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave >> 1) * (LT / 2), wn = (wave & 1) * (LT / 2);
    double* const out = STEP == 1 ? W : X;
#pragma unroll
    for (int x = 0; x < LT / 32; ++x)
#pragma unroll
        for (int y = 0; y < LT / 32; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = ra + wm + 16 * x + 4 * v + (lane >> 4), j = rb + wn + 16 * y + (lane & 15);
                if (i < m1 && j < m0) out[(size_t)i * n + j] = STEP == 1 ? acc[x][y][v] : -acc[x][y][v];
            }
}

// C(i, j) -= sum_{k < K} A(i, k) B(j, k) over 64 x 64 tiles of rows [i0, i1)
// and columns [j0, j1), on FP64 MFMA (v_mfma_f64_16x16x4f64), with
// A(i, k) = A[i ai + k ak], B(j, k) = B[j bj + k bk], C(i, j) = C[i ci + j cj]:
// the updates of a solve with many right-hand sides.  Four waves per tile, a
// 32 x 32 quadrant each (2 x 2 blocks of 16 x 16), operands straight from
// global memory, K in steps of 4.
__global__ __launch_bounds__(256) void la_mfma_update(const double* __restrict__ A, long ai, long ak,
                                                      const double* __restrict__ B, long bj, long bk,
                                                      double* __restrict__ C, long ci, long cj, int i0, int i1,
                                                      int j0, int j1, int K)
{
    const int ntj = (j1 - j0 + 63) / 64, I = blockIdx.x / ntj, J = blockIdx.x % ntj;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int rb = i0 + 64 * I + 32 * (w >> 1), cb = j0 + 64 * J + 32 * (w & 1);
    const int l16 = lane & 15, kq = lane >> 4;
    fd4 acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = (fd4){0.0, 0.0, 0.0, 0.0};
    const int r0 = rb + l16, r1 = rb + 16 + l16, c0 = cb + l16, c1 = cb + 16 + l16;
    for (int k0 = 0; k0 < K; k0 += 4) {
        const int k = k0 + kq;
        const bool kin = k < K;
        double a[2], b[2];
        a[0] = (kin && r0 < i1) ? A[r0 * ai + k * ak] : 0.0;
        a[1] = (kin && r1 < i1) ? A[r1 * ai + k * ak] : 0.0;
        b[0] = (kin && c0 < j1) ? B[c0 * bj + k * bk] : 0.0;
        b[1] = (kin && c1 < j1) ? B[c1 * bj + k * bk] : 0.0;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[x], b[y], acc[x][y], 0, 0, 0);
    }
    // element v of a block: row 4 v + lane / 16, column lane % 16
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = rb + 16 * x + 4 * v + kq, j = cb + 16 * y + l16;
                if (i < i1 && j < j1) C[i * ci + j * cj] -= acc[x][y][v];
            }
}

// Diagonal-block substitution on every RHS (one RHS per thread):
// lower (upper == 0): X[rb+j] = (X[rb+j] - sum_{l<j} L(rb+j, rb+l) X[rb+l]) / L(rb+j, rb+j)
// upper (upper == 1, U = L^T): backward over j.  L is row-major lower.
__global__ __launch_bounds__(256) void la_trsm_rhs(const double* __restrict__ Lm, int n, int upper,
                                                   double* __restrict__ X, int ldx, int nrhs, int rb)
{
    __shared__ double Lk[NB][NB + 1];
    const int nb = min(NB, n - rb);
    for (int e = threadIdx.x; e < NB * NB; e += 256) {
        int i = e / NB, j = e % NB;
        Lk[i][j] = (i < nb && j <= i) ? Lm[(size_t)(rb + i) * n + rb + j] : 0.0;
    }
    __syncthreads();
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= nrhs) return;
    double* x = X + (size_t)r * ldx + rb;
    double v[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) v[j] = j < nb ? x[j] : 0.0;
    if (!upper) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            double s = v[j];
#pragma unroll
            for (int l = 0; l < j; ++l) s -= Lk[j][l] * v[l];
            v[j] = j < nb ? s / Lk[j][j] : 0.0;
        }
    } else {
#pragma unroll
        for (int j = NB - 1; j >= 0; --j) {
            double s = v[j];
#pragma unroll
            for (int l = j + 1; l < NB; ++l) s -= Lk[l][j] * v[l];
            v[j] = j < nb ? s / Lk[j][j] : 0.0;
        }
    }
#pragma unroll
    for (int j = 0; j < NB; ++j)
        if (j < nb) x[j] = v[j];
}

// ortho[i][j] = ortho[j][i] = norm[i] L[i][j], lambda[i][j] = lambda[j][i] = X[i][j]
// / norm[j] (i >= j; X = L^-1), by 32 x 32 lower tiles: each is read once along
// its rows and written with its mirror image, both along rows through LDS.
__global__ __launch_bounds__(256) void la_outputs(const double* __restrict__ L, const double* __restrict__ X,
                                                  const double* __restrict__ norm, int n, double* __restrict__ ortho,
                                                  double* __restrict__ lambda)
{
    __shared__ double To[32][33], Tl[32][33];
    int I, J;
    lower_tile(blockIdx.x, &I, &J);
    const int c = threadIdx.x & 31, r0 = threadIdx.x >> 5;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = r0 + 8 * u, i = 32 * I + r, j = 32 * J + c;
        if (i < n && j <= i) {
            To[r][c] = norm[i] * L[(size_t)i * n + j];
            Tl[r][c] = X[(size_t)i * n + j] / norm[j];
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = r0 + 8 * u;
        int i = 32 * I + r, j = 32 * J + c;
        if (i < n && j < n && (I != J || j <= i)) {
            ortho[(size_t)i * n + j] = To[r][c];
            lambda[(size_t)i * n + j] = Tl[r][c];
        }
        i = 32 * J + r;   // the mirror image (on a diagonal tile: above the diagonal)
        j = 32 * I + c;
        if (i < n && j < n && (I != J || j > i)) {
            ortho[(size_t)i * n + j] = To[c][r];
            lambda[(size_t)i * n + j] = Tl[c][r];
        }
    }
}

// One block step of L y = b (UP false, ascending) or L^T y = b (UP true,
// descending) for up to RH right-hand sides of group blockIdx.y: every
// workgroup solves the OB x OB diagonal block at rb for the group (one wave per
// right-hand side, lane = row: a chain of OB broadcasts), and subtracts its
// product from 64 of the rows still to come; the first workgroup stores the
// block of y.  X is RHS-major with leading dimension n; Y another buffer, since
// other workgroups may still read this block of X.  The rows of L are loaded
// before the substitution, so a step costs about one memory latency and the
// chain.
constexpr int RH = 4;
template <bool UP>
__global__ __launch_bounds__(256) void la_solve_step(const double* __restrict__ L, int n, double* __restrict__ X,
                                                     double* __restrict__ Y, int nrhs, int rb)
{
    __shared__ double S[OB][OB + 1], ys[RH][OB], part[4][RH][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nb = min(OB, n - rb), g0 = RH * blockIdx.y, ng = min(RH, nrhs - g0);
    const int r0 = UP ? 64 * blockIdx.x : rb + nb + 64 * blockIdx.x;   // rows of the update
    const int r1 = min(r0 + 64, UP ? rb : n);
    // this thread's 16 elements of the update: forward row tid / 4, columns 16
    // (tid % 4) ..; backward row (of y) lane, block rows 16 wave ..
    double lv[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        if (UP) {
            const int k = 16 * wave + q, i = r0 + lane;
            lv[q] = (k < nb && i < r1) ? L[(size_t)(rb + k) * n + i] : 0.0;
        } else {
            const int k = 16 * (tid & 3) + q, i = r0 + (tid >> 2);
            lv[q] = (k < nb && i < r1) ? L[(size_t)i * n + rb + k] : 0.0;
        }
    }
    load_block<false>(L, n, rb, nb, S);
    __syncthreads();
    if (wave < ng) {
        const double x0 = lane < nb ? X[(size_t)(g0 + wave) * n + rb + lane] : 0.0;
        // Quotients by the pivot, rounded once (a product with the reciprocal
        // alone rounds twice); by the division itself where a pivot is near the
        // ends of the exponent range or a result is not finite.
        const double d = S[lane][lane], inv = 1.0 / d;
        auto solve = [&](double x, auto quotient) {
            for (int t = 0; t < OB; ++t) {
                const int j = UP ? OB - 1 - t : t;
                const double y = lane_value(quotient(x), j);
                if (UP ? lane < j : lane > j) x -= (UP ? S[j][lane] : S[lane][j]) * y;
            }
            return quotient(x);
        };
        double y = solve(x0, [&](double a) { return div_by(a, d, inv); });
        if (!__all(fabs(d) > 1e-280 && fabs(d) < 1e280 && fabs(y) < INFINITY))
            y = solve(x0, [&](double a) { return a / d; });
        ys[wave][lane] = y;
        if (blockIdx.x == 0 && lane < nb) Y[(size_t)(g0 + wave) * n + rb + lane] = y;
    } else {
        ys[wave][lane] = 0.0;
    }
    __syncthreads();
    if (UP) {
#pragma unroll
        for (int g = 0; g < RH; ++g) {
            double t = 0.0;
#pragma unroll
            for (int q = 0; q < 16; ++q) t += lv[q] * ys[g][16 * wave + q];
            part[wave][g][lane] = t;
        }
        __syncthreads();
        if (wave < ng && r0 + lane < r1)
            X[(size_t)(g0 + wave) * n + r0 + lane] -= (part[0][wave][lane] + part[1][wave][lane]) +
                                                      (part[2][wave][lane] + part[3][wave][lane]);
    } else {
        const int i = r0 + (tid >> 2);
#pragma unroll
        for (int g = 0; g < RH; ++g) {
            double t = 0.0;
#pragma unroll
            for (int q = 0; q < 16; ++q) t += lv[q] * ys[g][16 * (tid & 3) + q];
            t += __shfl_xor(t, 1);
            t += __shfl_xor(t, 2);
            if (g < ng && (tid & 3) == g && i < r1) X[(size_t)(g0 + g) * n + i] -= t;
        }
    }
}

// Forward (L y = b) or backward (L^T y = b) substitution on many RHS-major
// right-hand sides (X[r n + i]) in place, right-looking: per block of NB, the
// diagonal block's substitution, then the update of the rows after it (forward)
// or before it (backward) on FP64 MFMA.
static int la_solve_many(mcmb_ctx* c, const double* dL, int n, int upper, double* dX, int nrhs)
{
    const int nblk = (n + NB - 1) / NB;
    for (int b = 0; b < nblk; ++b) {
        const int kb = upper ? (nblk - 1 - b) : b;
        const int rb = kb * NB, nb = std::min(NB, n - rb);
        hipLaunchKernelGGL(la_trsm_rhs, dim3((unsigned)((nrhs + 255) / 256)), dim3(256), 0, c->stream, dL, n, upper, dX,
                           n, nrhs, rb);
        // rows [i0, i1) of the update
        const int i0 = upper ? 0 : rb + nb, i1 = upper ? rb : n;
        if (i1 > i0) {
            const unsigned tiles = (unsigned)(((i1 - i0 + 63) / 64) * ((nrhs + 63) / 64));
            // forward: A(i, k) = L(i, rb + k); backward: A(i, k) = L^T(i, rb + k) = L(rb + k, i)
            const double* A = upper ? dL + (size_t)rb * n : dL + rb;
            hipLaunchKernelGGL(la_mfma_update, dim3(tiles), dim3(256), 0, c->stream, A, upper ? 1l : (long)n,
                               upper ? (long)n : 1l, (const double*)(dX + rb), (long)n, 1l, dX, 1l, (long)n, i0, i1, 0,
                               nrhs, nb);
        }
    }
    MCMB_HIP(hipGetLastError());
    return MCMB_OK;
}

// The same for few right-hand sides, a launch per block of OB: x in X on
// entry, the solution in Y (X is used up).
static int la_solve_few(mcmb_ctx* c, const double* dL, int n, bool upper, double* dX, double* dY, int nrhs)
{
    const int nblk = (n + OB - 1) / OB, groups = (nrhs + RH - 1) / RH;
    for (int b = 0; b < nblk; ++b) {
        const int rb = OB * (upper ? nblk - 1 - b : b), nb = std::min(OB, n - rb);
        const int rows = upper ? rb : n - rb - nb;
        const dim3 grid((unsigned)std::max(1, (rows + 63) / 64), (unsigned)groups);
        if (upper) hipLaunchKernelGGL(la_solve_step<true>, grid, dim3(256), 0, c->stream, dL, n, dX, dY, nrhs, rb);
        else hipLaunchKernelGGL(la_solve_step<false>, grid, dim3(256), 0, c->stream, dL, n, dX, dY, nrhs, rb);
    }
    MCMB_HIP(hipGetLastError());
    return MCMB_OK;
}

// In-place Cholesky (lower) of the n x n matrix at dC; *bad = failing column+1.
// Per block of OB columns two launches: the panel, and the trailing update with
// the next diagonal block (78 x 2 at n = 4960 against 155 x 3 of blocks of 32).
static int la_potrf(mcmb_ctx* c, double* dC, int n, int* d_flag, int* bad)
{
    MCMB_HIP(hipMemsetAsync(d_flag, 0, sizeof(int), c->stream));
    hipLaunchKernelGGL(la_potrf_first, dim3(1), dim3(256), 0, c->stream, dC, n, d_flag);
    for (int k0 = 0; k0 + OB < n; k0 += OB) {
        const int m = n - k0 - OB;
        hipLaunchKernelGGL(la_trsm_panel, dim3((unsigned)((m + 63) / 64)), dim3(256), 0, c->stream, dC, n, k0, d_flag);
        const int t = (m + LT - 1) / LT;
        hipLaunchKernelGGL(la_syrk, dim3((unsigned)(t * (t + 1) / 2)), dim3(256), 0, c->stream, dC, n, k0, d_flag);
    }
    MCMB_HIP(hipGetLastError());
    MCMB_HIP(hipMemcpyAsync(bad, d_flag, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    MCMB_HIP(hipStreamSynchronize(c->stream));
    return MCMB_OK;
}

// X = L^-1 (row-major, lower; X zeroed on entry), W: work of n^2 doubles.
static int la_inverse(mcmb_ctx* c, const double* dL, int n, double* dX, double* dW)
{
    hipLaunchKernelGGL(la_inv_diag, dim3((unsigned)((n + OB - 1) / OB)), dim3(256), 0, c->stream, dL, n, dX);
    for (int s = OB; s < n; s *= 2) {
        const unsigned pairs = (unsigned)((n - s + 2 * s - 1) / (2 * s));
        const unsigned t = (s + LT - 1) / LT;
        hipLaunchKernelGGL(la_inv_join<1>, dim3(t * t, pairs), dim3(256), 0, c->stream, dL, dX, dW, n, s);
        hipLaunchKernelGGL(la_inv_join<2>, dim3(t * t, pairs), dim3(256), 0, c->stream, dL, dX, dW, n, s);
    }
    MCMB_HIP(hipGetLastError());
    return MCMB_OK;
}

}  // namespace mcmb

using namespace mcmb;

// Right-hand sides up to which a solve runs a launch per block of OB with the
// substitution in every workgroup (la_solve_few), host to host at n = 2900: 33
// right-hand sides 3.3 against 5.9 ms, 128 4.5 against 7.1 ms, 256 8.1 against
// 10.1 ms; beyond, L would be read again for every four of them.
constexpr int LA_FEW = 128;

namespace {
// The work buffer stays with the context between calls up to 2 GiB (four n x n
// matrices of n = 8000); a larger one is given back at the end of the call.
struct LaWork {
    mcmb_ctx* c;
    explicit LaWork(mcmb_ctx* ctx) : c(ctx) {}
    ~LaWork()
    {
        if (c->la_ws.bytes > ((size_t)2 << 30)) c->la_ws.release();
    }
};
}  // namespace

extern "C" int mcmb_orthonormalise(mcmb_ctx* c, int n, const double* gamma, double* ortho, double* lambda,
                                   double* norm, int* bad_pivot)
{
    if (!c || !gamma || n < 1) return fail(MCMB_ERR_ARG, "mcmb_orthonormalise: bad argument");
    MCMB_TRY(set_device(c));
    const size_t nn = (size_t)n * n;
    // four n x n buffers: Gamma then ortho, C then L, L^-1, work then lambda
    LaWork work(c);
    MCMB_TRY(c->la_ws.alloc((4 * nn + n) * sizeof(double) + sizeof(int)));
    double *const dG = c->la_ws.as<double>(), *const dC = dG + nn, *const dX = dC + nn, *const dW = dX + nn,
                  *const dN = dW + nn;
    int* const dF = reinterpret_cast<int*>(dN + n);
    MCMB_TRY(copy_to_device(c, dG, gamma, nn * sizeof(double)));
    hipLaunchKernelGGL(la_norm_kernel, dim3((n + 255) / 256), dim3(256), 0, c->stream, (const double*)dG, n, dN);
    hipLaunchKernelGGL(la_scale_kernel, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, c->stream, (const double*)dG, n,
                       (const double*)dN, dC);
    MCMB_HIP(hipGetLastError());
    MCMB_HIP(hipEventRecord(c->ev0, c->stream));
    int bad = 0;
    MCMB_TRY(la_potrf(c, dC, n, dF, &bad));
    if (bad_pivot) *bad_pivot = bad ? bad - 1 : -1;
    if (bad) return fail(MCMB_ERR_NOT_SPD, "Cholesky: non-positive pivot at column %d of %d (normalised Gram not "
                                           "positive definite in FP64)", bad - 1, n);
    MCMB_HIP(hipMemsetAsync(dX, 0, nn * sizeof(double), c->stream));
    MCMB_TRY(la_inverse(c, dC, n, dX, dW));
    MCMB_HIP(hipEventRecord(c->ev1, c->stream));
    const unsigned t = (unsigned)((n + 31) / 32);
    hipLaunchKernelGGL(la_outputs, dim3(t * (t + 1) / 2), dim3(256), 0, c->stream, (const double*)dC, (const double*)dX,
                       (const double*)dN, n, dG, dW);
    MCMB_HIP(hipGetLastError());
    if (ortho) MCMB_TRY(copy_to_host(c, ortho, dG, nn * sizeof(double)));
    if (lambda) MCMB_TRY(copy_to_host(c, lambda, dW, nn * sizeof(double)));
    if (norm) MCMB_TRY(copy_to_host(c, norm, dN, n * sizeof(double)));
    float ms = 0.f;
    MCMB_HIP(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    c->last_launches = 0;
    return MCMB_OK;
}

extern "C" int mcmb_cholesky_solve(mcmb_ctx* c, int n, const double* ortho, int nrhs, const double* alpha,
                                   double* beta)
{
    if (!c || !ortho || !alpha || !beta || n < 1 || nrhs < 1) return fail(MCMB_ERR_ARG, "mcmb_cholesky_solve: bad argument");
    MCMB_TRY(set_device(c));
    const size_t nn = (size_t)n * n, nx = (size_t)n * nrhs;
    LaWork work(c);
    MCMB_TRY(c->la_ws.alloc((nn + 2 * nx) * sizeof(double)));
    double *const dF = c->la_ws.as<double>(), *const dX = dF + nn, *const dY = dX + nx;
    MCMB_TRY(copy_to_device(c, dF, ortho, nn * sizeof(double)));
    MCMB_TRY(copy_to_device(c, dX, alpha, nx * sizeof(double)));
    if (nrhs <= LA_FEW) {
        MCMB_TRY(la_solve_few(c, dF, n, false, dX, dY, nrhs));
        MCMB_TRY(la_solve_few(c, dF, n, true, dY, dX, nrhs));
    } else {
        MCMB_TRY(la_solve_many(c, dF, n, 0, dX, nrhs));
        MCMB_TRY(la_solve_many(c, dF, n, 1, dX, nrhs));
    }
    MCMB_TRY(copy_to_host(c, beta, dX, nx * sizeof(double)));
    return MCMB_OK;
}
