// Shape projection on the Gauss-Legendre k-tetrapyd, with tangent (forward)
// and adjoint (reverse) derivatives in (omega, phi), for the feature shape
// S = sin(omega (k1+k2+k3) + phi) / (k1 k2 k3)^2 (calculate_shape.c:933-946).
//
//   alpha_n(theta) = sum_{cube} W_ijk sin(omega K_ijk + phi) Q_n(i,j,k)
//   W_ijk = mask_ijk w_i w_j w_k / (k_i + k_j + k_k)
// restates calculate_eigen (calculate_eigen.c:86-145) on the GL grid: its
// integrand is shape3/K = (k1k2k3)^2 S / K.  W and S are symmetric, so
// alpha_n = A[r][s][t] with A_rst = sum_ijk F_ijk q_r(i) q_s(j) q_t(k), F = W S.
//
// With A_ij = omega (k_i + k_j) + phi and B_k = omega k_k,
//   sin(A + B) = sin A cos B + cos A sin B,
// the k-sum separates:  Y[(i,j)][x,t] = sum_k W_ijk Z[k][x,t] with the two
// column sets Z = {cos B, sin B} q_t(k)  -- one MFMA GEMM (W resident in HBM,
// N^2 / 2 x N) for a batch of shapes.  Then per shape
//   G_sin = sA Yc + cA Ys   (sin(A+B): the value)
//   G_cos = cA Yc - sA Ys   (cos(A+B): the derivatives)
//   H_x[i][s][t] = sum_j q_s(j) G_x[i][j][t],  A_x[r][s][t] = sum_i q_r(i) H_x[i][s][t],
// and d/domega, which brings K = k_i + k_j + k_k, from the k_i-weighted sum
// over i with each leg in turn on i.
// H_x[i] is symmetric in (s, t) (W and the shape are symmetric in the legs j
// and k), so it is formed and kept for s <= t only.
// The adjoint (VJP) of gbar = dL/dalpha contracts it with the two derivative
// tensors of the same k-, j- and i-sums: dL/dphi = sum_n gbar_n dalpha_n/dphi,
// dL/domega = sum_n gbar_n dalpha_n/domega.
#include "mcmb_internal.h"
#include <type_traits>
#include <cstring>
#include <algorithm>
#include <cmath>
#include <vector>

namespace mcmb {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int PT = 128;     // GEMM tile (M and N)
constexpr int WT = 64;      // the same of stage 1's GEMM
constexpr int PK = 16;      // GEMM K chunk
constexpr int PBATCH = 32;  // shapes per batch

// ---- full-cube weight ------------------------------------------------------
// W[(i*N + j)*Kp + k]; the mask compares the sorted triple exactly as the
// oracle does: k_c <= k_a + k_b (FP64).
template <class T>
__global__ void proj_build_W(const double* __restrict__ kn, const double* __restrict__ kw, int N, int Kp,
                             const int2* __restrict__ rowij, long M, T* __restrict__ W)
{
    // W[(i,j) pair row][k], pair rows i <= j only (W is symmetric in i, j)
    size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t tot = (size_t)M * Kp;
    if (e >= tot) return;
    int k = (int)(e % Kp);
    const int2 ij = rowij[e / Kp];
    double w = 0.0;
    if (k < N) {
        int a = ij.x, b = ij.y, c = k, t;
        if (a > b) { t = a; a = b; b = t; }
        if (b > c) { t = b; b = c; c = t; if (a > b) { t = a; a = b; b = t; } }
        if (kn[c] <= kn[a] + kn[b]) w = kw[a] * kw[b] * kw[c] / (kn[a] + kn[b] + kn[c]);
    }
    W[e] = (T)w;
}

// The K chunks of each WT-row tile of W that hold a nonzero weight: tiles[t]
// = (first chunk, chunk count) over the tile's rows (an all-zero tile keeps
// chunk 0).  The stage-1 GEMMs run only over those chunks: the others add
// exact zeros.
template <class T>
__global__ __launch_bounds__(256) void proj_w_tiles(const T* __restrict__ W, long M, int Kp,
                                                    int2* __restrict__ tiles)
{
    __shared__ int lo, hi;
    if (threadIdx.x == 0) {
        lo = Kp;
        hi = -1;
    }
    __syncthreads();
    const long r0 = (long)blockIdx.x * WT, ne = (long)min((long)WT, M - r0) * Kp;
    int mlo = Kp, mhi = -1;
    for (long e = threadIdx.x; e < ne; e += 256)
        if (W[r0 * Kp + e] != (T)0) {
            const int k = (int)(e % Kp);
            mlo = min(mlo, k);
            mhi = max(mhi, k);
        }
    atomicMin(&lo, mlo);
    atomicMax(&hi, mhi);
    __syncthreads();
    if (threadIdx.x == 0) {
        const int c0 = hi < 0 ? 0 : lo / PK, c1 = hi < 0 ? 0 : hi / PK;
        tiles[blockIdx.x] = make_int2(c0, c1 - c0 + 1);
    }
}

// The R basis columns as stage 2 takes them: NT = 1 or 2 matrix tiles (R > 16)
// of Rh columns, t = a Rh + c (a < NT, c < Rh <= 16).  A shape has the 2 NT Rh
// columns (c, a, cos / sin) of Z and Y, so that what lane c of stage 2 needs of
// a Y row is one vector of 2 NT elements.
struct BasisTiles {
    int NT, Rh, cols;   // tiles, columns of each, Z columns of a shape
};
__host__ __device__ __forceinline__ BasisTiles basis_tiles(int R)
{
    const int NT = R > 16 ? 2 : 1, Rh = (R + NT - 1) / NT;
    return BasisTiles{NT, Rh, 2 * NT * Rh};
}

// Z[k][col], col = ((b Rh + c) NT + a) 2 + x for shapes b < nb of the batch:
// x = 0 cos(omega_b k) q_t(k), x = 1 sin(omega_b k) q_t(k), t = a Rh + c (zero
// past R); Kp x ldz.
template <class T>
__global__ void proj_build_Z(const double* __restrict__ kn, const double* __restrict__ q, int ldq, int N, int R,
                             const double* __restrict__ theta, int nb, int Kp, int ldz, T* __restrict__ Z)
{
    size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)Kp * ldz) return;
    int k = (int)(e / ldz), col = (int)(e % ldz);
    double z = 0.0;
    const BasisTiles bt = basis_tiles(R);
    const int a = (col >> 1) % bt.NT, e1 = (col >> 1) / bt.NT, t = a * bt.Rh + e1 % bt.Rh, b = e1 / bt.Rh;
    if (k < N && b < nb && t < R) {
        const int c = col & 1;
        double om = theta[2 * b];
        double sb, cb;
        sincos(om * kn[k], &sb, &cb);
        z = (c ? sb : cb) * q[(size_t)k * ldq + t];
    }
    Z[e] = (T)z;
}

// ---- MFMA GEMM  C[M][Nc] = A[M][Kp] B[Kp][ldb]  (A row-major lda = Kp) ------
template <class T> struct MF;
template <> struct MF<double> {
    typedef d4 V;
    static __device__ __forceinline__ V mma(double a, double b, V c)
    { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    // output row of element v for lane: 4v + lane/16
    static __device__ __forceinline__ int row(int v, int lane) { return 4 * v + (lane >> 4); }
};
template <> struct MF<float> {
    typedef f4 V;
    static __device__ __forceinline__ V mma(float a, float b, V c)
    { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    // output row of element v for lane: 4 (lane/16) + v
    static __device__ __forceinline__ int row(int v, int lane) { return 4 * (lane >> 4) + v; }
};

template <class T>
__global__ __launch_bounds__(256, 2) void proj_gemm(const T* __restrict__ A, const T* __restrict__ B, int M, int Kp,
                                                    int Nc, int ldb, T* __restrict__ C, int ldc)
{
    __shared__ T As[2][PK][PT + 4];
    __shared__ T Bs[2][PK][PT + 4];
    const int m0 = blockIdx.y * PT, n0 = blockIdx.x * PT;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    typename MF<T>::V acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[a][b][v] = 0;
    // staging: thread loads 8 elements of A (rows r, k chunk) and 8 of B
    T ra[8], rb[8];
    auto gload = [&](int k0) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            int e = tid + u * 256;                  // 0..2047
            int r = e >> 4, kk = e & 15;            // A: 128 rows x 16
            int gm = m0 + r;
            ra[u] = (gm < M) ? A[(size_t)gm * Kp + k0 + kk] : (T)0;
            int kb = e >> 7, cc = e & 127;          // B: 16 x 128
            int gn = n0 + cc;
            rb[u] = (gn < Nc) ? B[(size_t)(k0 + kb) * ldb + gn] : (T)0;
        }
    };
    auto sstore = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            int e = tid + u * 256;
            As[buf][e & 15][e >> 4] = ra[u];
            Bs[buf][e >> 7][e & 127] = rb[u];
        }
    };
    gload(0);
    sstore(0);
    __syncthreads();
    const int nk = Kp / PK;
    for (int kc = 0; kc < nk; ++kc) {
        const int buf = kc & 1;
        if (kc + 1 < nk) gload((kc + 1) * PK);
#pragma unroll
        for (int ks = 0; ks < PK / 4; ++ks) {
            const int kk = ks * 4 + (lane >> 4);
            T av[4], bv[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) av[a] = As[buf][kk][wm * 64 + a * 16 + (lane & 15)];
#pragma unroll
            for (int b = 0; b < 4; ++b) bv[b] = Bs[buf][kk][wn * 64 + b * 16 + (lane & 15)];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[a][b] = MF<T>::mma(av[a], bv[b], acc[a][b]);
        }
        if (kc + 1 < nk) sstore(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                int gm = m0 + wm * 64 + a * 16 + MF<T>::row(v, lane);
                int gn = n0 + wn * 64 + b * 16 + (lane & 15);
                if (gm < M && gn < Nc) C[(size_t)gm * ldc + gn] = acc[a][b][v];
            }
}

// sin and cos of omega_b k_j for the shapes of a batch: scb[b][j] = (sin,
// cos), zero for N <= j < Np.  Stage 2 forms sin / cos of A_ij = (omega k_i +
// phi) + omega k_j by the angle-addition formulas from these and one sincos
// per workgroup.
__global__ void proj_sincos_tab(const double* __restrict__ kn, const double* __restrict__ theta, int N, int Np, int nb,
                                double* __restrict__ scb)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nb * Np) return;
    const int b = e / Np, j = e % Np;
    double sb = 0.0, cb = 0.0;
    if (j < N) sincos(theta[2 * b] * kn[j], &sb, &cb);
    scb[2 * e] = sb;
    scb[2 * e + 1] = cb;
}

// Column of (s, t) among the pairs s <= t of R functions; the symmetric
// planes below keep PP = the count rounded up to whole 16-column blocks.
__host__ __device__ __forceinline__ int sym_col(int s, int t, int R)
{
    const int lo = s < t ? s : t, hi = s < t ? t : s;
    return lo * (2 * R - lo - 1) / 2 + hi;
}
static int sym_cols(int R) { return (R * (R + 1) / 2 + 15) / 16 * 16; }

// ---- stage 2: per (shape b, node i) ----------------------------------------
// H[b][x][i][st] = sum_j q_s(j) G_x(i, j, t), s <= t, with G_x(i, j, t) =
// sum_k W_ijk {sin, cos}(omega K + phi) q_t(k): sin for the value, cos for the
// derivatives.  X selects the planes: 1 sin, 2 cos, 3 both (in that order).
// From stage 1's Yc, Ys (cos / sin omega k_k columns) by angle addition:
// G_sin = sin A Yc + cos A Ys, G_cos = cos A Yc - sin A Ys, A = omega (k_i +
// k_j) + phi.  Y's row of the pair (i, j) is wrow[stage2_row(i, j)] (stage 1
// runs over W's rows in their own order).
//
// On FP64 MFMA 16x16x4, A = Q^T (s x j), B = G_x (j x t); of the tiles of (s,
// t) only those on and above the diagonal (NP = 3 of 4 for NT = 2).  The four
// waves of a workgroup take every fourth K-step (4 nodes j) each and are
// summed through LDS at the end: a lane forms the B operand of its own (j, t)
// from its own loads, so the loop has no LDS traffic and no barrier, and the
// loads of the next group of K-steps run under this one's products.
//
// What bounds it besides the products is the address unit of the CU's vector
// loads, about 16 cycles an instruction whatever its width: with one load
// per element of Y and q and one for the row number (7 a K-step) that unit was
// 78% busy.  So a lane's Y, q and (sin, cos) of a K-step are one vector each
// (the layouts of Z and of the basis table), a lane's row numbers
// of a group lie next to each other, and the tables are padded with zeros to Np nodes so that nothing is
// clamped or masked.
//
// XCD x (workgroups are dealt to the 8 XCDs in turn) takes the nodes i = x
// mod 8, and the shapes go in groups of SG, node by node: neighbouring shapes'
// pieces of a Y row, which share cache lines, meet in one L2, and a group's
// part of Y is read the second time (for the pair's other node) out of cache.
//
// 32 shapes, 300 nodes, 30 functions, FP32 Y (347 MB; the products alone are
// 120 us, or 60 for one plane): both planes 373 -> 200 us, cos alone (with the
// sums that replaced the adjoint's own) 284 -> 137.  One shape of 200 nodes,
// FP64: 14 -> 7.4.
constexpr int SG = 4;    // shapes of a group
// Nodes of a workgroup: two share the basis and the (sin, cos) loads and halve
// the workgroups.  With one plane to form the address unit is the bound and
// two are faster from S2_PAIR (shape, node) pairs on: 3200 pairs (FP64) 36.2
// us with one, 36.8 with two; 6400 65.3, 64.6; 9600 (FP32) 157, 137.  With both
// planes the products are (9600: 195, 199), so there it stays one.
constexpr long S2_PAIR = 4800;
constexpr int S2U = 2;   // K-steps a wave loads ahead
// nodes of the padded tables: two groups of S2U K-steps past the last
__host__ __device__ __forceinline__ int stage2_nodes(int N) { return (N + 16 * S2U - 1) / (16 * S2U) * (16 * S2U) + 32 * S2U; }
// place of the pair (i, j) in the row table: a lane's nodes j = 16 m + r (r its own) in order of m
static size_t stage2_row(int i, int j, int Np) { return (size_t)i * Np + (size_t)(j % 16) * (Np / 16) + j / 16; }

template <class T, int X, int NT, int NI>
__global__ __launch_bounds__(256, NI * NT == 4 ? 3 : 4) void proj_stage2(const T* __restrict__ Y, int ldy, const int* __restrict__ wrow,
                                                      const double* __restrict__ kn, const double* __restrict__ qt,
                                                      int N, int R, int PP, const double* __restrict__ theta, int nb,
                                                      const double* __restrict__ scb, double* __restrict__ H)
{
    typedef T TV __attribute__((ext_vector_type(2 * NT)));
    typedef double D2 __attribute__((ext_vector_type(2)));
    typedef int I2 __attribute__((ext_vector_type(2)));
    static_assert(S2U == 2, "a group's row numbers are one int2");
    constexpr int NX = (X & 1) + (X >> 1), NP = NT * (NT + 1) / 2, U = S2U;
    __shared__ double red[4][NP][256];
    const int ni = (N + NI - 1) / NI, slot = blockIdx.x >> 3;
    const int per = SG * ((ni + 7) / 8);   // workgroups of a whole shape group on an XCD
    const int g0 = slot / per * SG, ns = min(SG, nb - g0), e0 = slot % per;
    const int b = g0 + e0 % ns, i0 = NI * (8 * (e0 / ns) + (blockIdx.x & 7));   // nodes i0 .. i0 + NI - 1
    if (i0 >= N) return;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15,
              kg = lane >> 4;
    const int Np = stage2_nodes(N), Rh = (R + NT - 1) / NT;
    double sa[NI], ca[NI];   // sin, cos of omega k_i + phi
#pragma unroll
    for (int z = 0; z < NI; ++z)
        sincos(theta[2 * b] * kn[min(i0 + z, N - 1)] + theta[2 * b + 1], &sa[z], &ca[z]);
    // the wave's K-step m has the nodes j = 16 m + 4 w + kg
    const I2* rw[NI];   // a node past N: the last one again, not stored
#pragma unroll
    for (int z = 0; z < NI; ++z)
        rw[z] = reinterpret_cast<const I2*>(wrow + (size_t)min(i0 + z, N - 1) * Np + (4 * w + kg) * (Np / 16));
    const D2* const sc = reinterpret_cast<const D2*>(scb) + (size_t)b * Np + 4 * w + kg;
    const double* const qj = qt + ((4 * w + kg) * 16 + c) * NT;
    const T* const Yb = Y + (size_t)b * 2 * NT * Rh + 2 * NT * min(c, Rh - 1);   // lanes past Rh: not stored
    d4 acc[NI][NX][NP];
#pragma unroll
    for (int z = 0; z < NI; ++z)
#pragma unroll
        for (int x = 0; x < NX; ++x)
#pragma unroll
            for (int p = 0; p < NP; ++p) acc[z][x][p] = (d4){0.0, 0.0, 0.0, 0.0};
    const int ng = (N + 16 * U - 1) / (16 * U);   // groups of U K-steps a wave
    I2 rows[NI];
    TV yv[NI][U];
    D2 sv[U];
    double qv[U][NT];
    auto load_rows = [&](int g) {
#pragma unroll
        for (int z = 0; z < NI; ++z) rows[z] = rw[z][g];
    };
    auto load = [&](int g) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int m = g * U + u;
#pragma unroll
            for (int z = 0; z < NI; ++z)
                yv[z][u] = *reinterpret_cast<const TV*>(Yb + (size_t)(unsigned)rows[z][u] * (unsigned)ldy);
            sv[u] = sc[16 * m];
            if (NT == 2) {
                const D2 v = *reinterpret_cast<const D2*>(qj + (size_t)m * 256 * NT);
                qv[u][0] = v[0];
                qv[u][NT - 1] = v[1];
            } else
                qv[u][0] = qj[(size_t)m * 256 * NT];
        }
    };
    load_rows(0);
    load(0);
    load_rows(1);
    for (int g = 0; g < ng; ++g) {
        double A[U][NT], B[NI][U][NX][NT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int a = 0; a < NT; ++a) A[u][a] = qv[u][a];
#pragma unroll
            for (int z = 0; z < NI; ++z) {
                const double sA = sa[z] * sv[u][1] + ca[z] * sv[u][0], cA = ca[z] * sv[u][1] - sa[z] * sv[u][0];
#pragma unroll
                for (int a = 0; a < NT; ++a) {
                    const double yc = (double)yv[z][u][2 * a], ys = (double)yv[z][u][2 * a + 1];
                    if (X & 1) B[z][u][0][a] = sA * yc + cA * ys;
                    if (X & 2) B[z][u][NX - 1][a] = cA * yc - sA * ys;
                }
            }
        }
        load(g + 1);
        load_rows(g + 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int z = 0; z < NI; ++z)
#pragma unroll
                for (int x = 0; x < NX; ++x) {
                    int p = 0;
#pragma unroll
                    for (int a = 0; a < NT; ++a)
#pragma unroll
                        for (int t = a; t < NT; ++t, ++p)
                            acc[z][x][p] =
                                __builtin_amdgcn_mfma_f64_16x16x4f64(A[u][a], B[z][u][x][t], acc[z][x][p], 0, 0, 0);
                }
    }
    // sum over the waves, a plane at a time; element v of a lane is row 4 v +
    // lane / 16, column lane % 16 of its tile, and thread tid stores element
    // (tid / 16, tid % 16).  A tile on the diagonal holds (s, t) and (t, s): of
    // these the mean, whose stage-1 roundings are independent.
#pragma unroll
    for (int z = 0; z < NI; ++z)
#pragma unroll
        for (int x = 0; x < NX; ++x) {
            if (x || z) __syncthreads();
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int v = 0; v < 4; ++v) red[w][p][64 * v + lane] = acc[z][x][p][v];
            __syncthreads();
            if (i0 + z >= N) continue;   // uniform over the workgroup
            double* const h = H + (((size_t)b * NX + x) * N + i0 + z) * PP;
            int p = 0;
#pragma unroll
            for (int a = 0; a < NT; ++a)
#pragma unroll
                for (int t = a; t < NT; ++t, ++p) {
                    const int sc = tid >> 4, tc = tid & 15, ss = a * Rh + sc, tt = t * Rh + tc, tr = 16 * tc + sc;
                    if (sc < Rh && tc < Rh && ss <= tt && tt < R) {
                        double v = (red[0][p][tid] + red[1][p][tid]) + (red[2][p][tid] + red[3][p][tid]);
                        if (a == t)
                            v = 0.5 * (v + ((red[0][p][tr] + red[1][p][tr]) + (red[2][p][tr] + red[3][p][tr])));
                        h[sym_col(ss, tt, R)] = v;
                    }
                }
        }
}

// D[b][d][r][st] (st a column s <= t) on FP64 MFMA 16x16x4:
//   d = 0: sum_i q_r(i) H_sin[i][st]       (alpha)
//   d = 1: sum_i q_r(i) H_cos[i][st]       (d alpha / d phi)
//   d = 2: sum_i k_i q_r(i) H_cos[i][st]   (E, the k_i-weighted cos form)
// One workgroup per (shape b, plane of H, block of 16 columns st): the sin
// plane makes d = 0, the cos plane d = 1 and 2 from the same B loads (each H
// element is read once); the r tiles share them too.  The four waves take a
// quarter of the nodes' K-steps each (a chain of N / 64 dependent loads instead
// of N / 16) and are summed through LDS.  32 shapes, 300 nodes, 30 functions:
// 70 -> 34 us (half of it from s <= t), one shape of 200 nodes 19 -> 7.9.
//
// E gives d alpha / d omega = sum W K cos(omega K + phi) q_r q_s q_t: W and
// the cos term are symmetric in the three legs, so each of k_j and k_k can
// be moved onto leg i by relabelling, and d alpha / d omega [r][s][t] =
// E[r][s][t] + E[s][r][t] + E[t][s][r].
template <int X, int NT>
__global__ __launch_bounds__(256) void proj_stage3(const double* __restrict__ H, const double* __restrict__ q, int ldq,
                                                   const double* __restrict__ kn, int N, int R, int PP,
                                                   double* __restrict__ D)
{
    constexpr int NX = (X & 1) + (X >> 1), NW = X >> 1, U = 4;
    __shared__ double red[4][(1 + NW) * NT][256];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c = lane & 15, kg = lane >> 4;
    const int nblk = PP / 16, by = blockIdx.x / nblk, st0 = 16 * (blockIdx.x % nblk);
    const int b = by / NX, y = X == 2 ? 1 : by % NX;   // y: 0 sin, 1 cos
    const double* const h = H + (size_t)by * N * PP + st0 + c;
    d4 acc[1 + NW][NT];   // [0 plain, 1 k-weighted][r tile]
#pragma unroll
    for (int d = 0; d <= NW; ++d)
#pragma unroll
        for (int a = 0; a < NT; ++a) acc[d][a] = (d4){0.0, 0.0, 0.0, 0.0};
    const int nks = (N + 3) / 4;
    for (int k0 = U * w; k0 < nks; k0 += 4 * U) {
        double bv[U], av[U][NT], kf[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = 4 * (k0 + u) + kg, ic = min(i, N - 1);
            bv[u] = h[(size_t)ic * PP];
            kf[u] = kn[ic];
#pragma unroll
            for (int a = 0; a < NT; ++a) av[u][a] = q[(size_t)ic * ldq + min(16 * a + c, R - 1)];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = 4 * (k0 + u) + kg < N;
#pragma unroll
            for (int a = 0; a < NT; ++a) {
                const double qa = in ? av[u][a] : 0.0;
                acc[0][a] = __builtin_amdgcn_mfma_f64_16x16x4f64(qa, bv[u], acc[0][a], 0, 0, 0);
                if (NW && y) acc[NW][a] = __builtin_amdgcn_mfma_f64_16x16x4f64(kf[u] * qa, bv[u], acc[NW][a], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int d = 0; d <= NW; ++d)
#pragma unroll
        for (int a = 0; a < NT; ++a)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[w][d * NT + a][64 * v + lane] = acc[d][a][v];
    __syncthreads();
#pragma unroll
    for (int d = 0; d <= NW; ++d)
        if (d <= y)
#pragma unroll
            for (int a = 0; a < NT; ++a) {
                const int r = 16 * a + (tid >> 4), e = d * NT + a;
                if (r < R)
                    D[(((size_t)b * 3 + y + d) * R + r) * PP + st0 + (tid & 15)] =
                        (red[0][e][tid] + red[1][e][tid]) + (red[2][e][tid] + red[3][e][tid]);
            }
}

// The sum of a plane of D over the three legs that a mode (r, s, t) may have
// on the node i: d alpha / d omega from E = D[b][2], and three times alpha and d
// alpha / d phi from D[b][0] and D[b][1], where the three are equal but for
// their stage-1 roundings.
__device__ __forceinline__ double legs(const double* __restrict__ E, int r, int s, int t, int R, int PP)
{
    return E[(size_t)r * PP + sym_col(s, t, R)] + E[(size_t)s * PP + sym_col(r, t, R)] +
           E[(size_t)t * PP + sym_col(s, r, R)];
}

// alpha[b][m], d alpha / d omega and d alpha / d phi of the modes (r, s, t) =
// order[m], written in the caller's layout: alpha[b][m] and dalpha[b][x][m] (x =
// 0: omega, 1: phi); nx = 3, or 1 for alpha alone.
__global__ void proj_stage3_modes(const double* __restrict__ D, int R, int PP, const int* __restrict__ modes, int n,
                                  int nb, int nx, double* __restrict__ alpha, double* __restrict__ dalpha)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nb * nx * n) return;
    const int m = e % n, x = (e / n) % nx, b = e / (nx * n);
    const int pk = modes[m], r = pk & 255, s = (pk >> 8) & 255, t = (pk >> 16) & 255;
    const double v = legs(D + ((size_t)b * 3 + x) * R * PP, r, s, t, R, PP);
    if (x == 0) alpha[(size_t)b * n + m] = v / 3.0;
    else if (x == 1) dalpha[((size_t)b * 2 + 1) * n + m] = v / 3.0;
    else dalpha[(size_t)b * 2 * n + m] = v;
}

// ---- adjoint ---------------------------------------------------------------
// dtheta[b] = sum_m gbar[b][m] (d alpha_m / d omega, d alpha_m / d phi), one
// workgroup per shape: thread l sums m = l, l + 512, ..., then the waves and
// the workgroup are summed in a fixed order.  (32 shapes of 4960 modes: 14 us;
// the contraction of gbar with the basis that this replaces, 62.)
__global__ __launch_bounds__(512) void proj_dtheta(const double* __restrict__ D, int R, int PP,
                                                   const int* __restrict__ modes, int n,
                                                   const double* __restrict__ gbar, double* __restrict__ out)
{
    __shared__ double part[8][2];
    const int b = blockIdx.x, tid = threadIdx.x;
    const size_t plane = (size_t)R * PP;
    const double* const P = D + ((size_t)b * 3 + 1) * plane;
    const double* const E = P + plane;
    double so = 0.0, sp = 0.0;
#pragma unroll 4
    for (int m = tid; m < n; m += 512) {
        const int pk = modes[m], r = pk & 255, s = (pk >> 8) & 255, t = (pk >> 16) & 255;
        const double g = gbar[(size_t)b * n + m];
        so += g * legs(E, r, s, t, R, PP);
        sp += g * (legs(P, r, s, t, R, PP) / 3.0);
    }
    for (int d = 32; d > 0; d >>= 1) {
        so += __shfl_xor(so, d);
        sp += __shfl_xor(sp, d);
    }
    if ((tid & 63) == 0) {
        part[tid >> 6][0] = so;
        part[tid >> 6][1] = sp;
    }
    __syncthreads();
    if (tid < 2) {
        double v = 0.0;
        for (int w = 0; w < 8; ++w) v += part[w][tid];
        out[2 * b + tid] = v;
    }
}

static int ensure_W(mcmb_ctx* c, int prec)
{
    PointSet& K = c->ks;
    const int N = K.lmax + 1, Kp = (N + PK - 1) / PK * PK;
    if (c->w_ready == prec + 1) return MCMB_OK;
    const long M = (long)N * (N + 1) / 2;
    // The pair rows i <= j in an order that groups rows of like nonzero k
    // range: W_ijk is nonzero only for k_k in [k_j - k_i, k_i + k_j] (the
    // triangle), so with the rows sorted by (upper end / PK, lower end) most
    // K chunks of a WT-row tile are zero throughout, and the GEMMs skip them
    // (43% of the chunks remain at 300 nodes, against 87% in i-major pair
    // order).  Each row's k-sum is unchanged, so Y holds the same values in
    // W's row order; wrow[stage2_row(i, j)] is the row of (i, j) or (j, i).
    const std::vector<double>& kn = K.kn;
    std::vector<int2> rowij;
    std::vector<long> key;
    rowij.reserve(M);
    key.reserve(M);
    for (int i = 0; i < N; ++i)
        for (int j = i; j < N; ++j) {
            const long lo = std::lower_bound(kn.begin(), kn.end(), kn[j] - kn[i]) - kn.begin();
            const long hi = std::upper_bound(kn.begin(), kn.end(), kn[i] + kn[j]) - kn.begin();
            key.push_back((hi / PK) * (N + 1) + lo);
            rowij.push_back(make_int2(i, j));
        }
    std::vector<long> ord(M);
    for (long r = 0; r < M; ++r) ord[r] = r;
    std::stable_sort(ord.begin(), ord.end(), [&](long a, long b) { return key[a] < key[b]; });
    std::vector<int2> rows(M);
    const int Np = stage2_nodes(N);
    std::vector<int> rowof(M), wrow((size_t)N * Np);
    for (long r = 0; r < M; ++r) {
        rows[r] = rowij[ord[r]];
        rowof[ord[r]] = (int)r;   // rowij is in i-major pair order
    }
    {
        long m = 0;
        for (int i = 0; i < N; ++i)
            for (int j = i; j < N; ++j, ++m)
                wrow[stage2_row(i, j, Np)] = wrow[stage2_row(j, i, Np)] = rowof[m];
        for (int i = 0; i < N; ++i)
            for (int j = N; j < Np; ++j) wrow[stage2_row(i, j, Np)] = wrow[stage2_row(i, N - 1, Np)];
    }
    // stage 2's basis operand: (j, c) -> the columns a Rh + c of its NT tiles,
    // zero past the nodes and the columns
    const BasisTiles bt = basis_tiles(K.R);
    std::vector<double> qt((size_t)Np * 16 * bt.NT, 0.0);
    for (int j = 0; j < N; ++j)
        for (int c = 0; c < bt.Rh; ++c)
            for (int a = 0; a < bt.NT; ++a)
                if (a * bt.Rh + c < K.R)
                    qt[((size_t)j * 16 + c) * bt.NT + a] = K.q[(size_t)j * K.ldq + a * bt.Rh + c];
    MCMB_TRY(c->d_pq.alloc(sizeof(double) * qt.size()));
    MCMB_HIP(hipMemcpyAsync(c->d_pq.p, qt.data(), sizeof(double) * qt.size(), hipMemcpyHostToDevice, c->stream));
    DevBuf d_ij;
    MCMB_TRY(d_ij.alloc(sizeof(int2) * (size_t)M));
    MCMB_HIP(hipMemcpyAsync(d_ij.p, rows.data(), sizeof(int2) * (size_t)M, hipMemcpyHostToDevice, c->stream));
    MCMB_TRY(c->d_wrow.alloc(sizeof(int) * wrow.size()));
    MCMB_HIP(hipMemcpyAsync(c->d_wrow.p, wrow.data(), sizeof(int) * wrow.size(), hipMemcpyHostToDevice, c->stream));
    const unsigned ntile = (unsigned)((M + WT - 1) / WT);
    MCMB_TRY(c->d_wtile.alloc(sizeof(int2) * ntile));
    size_t tot = (size_t)M * Kp;
    MCMB_TRY(launch_guard("projection weight cube", (tot + 255) / 256, 256));
    if (prec == MCMB_FP64) {
        MCMB_TRY(c->d_W.alloc(tot * sizeof(double)));
        hipLaunchKernelGGL(proj_build_W<double>, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, c->stream,
                           K.d_kn.as<double>(), K.d_kw.as<double>(), N, Kp, d_ij.as<int2>(), M,
                           c->d_W.as<double>());
        hipLaunchKernelGGL(proj_w_tiles<double>, dim3(ntile), dim3(256), 0, c->stream,
                           (const double*)c->d_W.as<double>(), M, Kp, c->d_wtile.as<int2>());
    } else {
        MCMB_TRY(c->d_W.alloc(tot * sizeof(float)));
        hipLaunchKernelGGL(proj_build_W<float>, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, c->stream,
                           K.d_kn.as<double>(), K.d_kw.as<double>(), N, Kp, d_ij.as<int2>(), M,
                           c->d_W.as<float>());
        hipLaunchKernelGGL(proj_w_tiles<float>, dim3(ntile), dim3(256), 0, c->stream,
                           (const float*)c->d_W.as<float>(), M, Kp, c->d_wtile.as<int2>());
    }
    MCMB_HIP(hipGetLastError());
    MCMB_HIP(hipStreamSynchronize(c->stream));   // the host tables go out of scope
    c->w_ready = prec + 1;
    return MCMB_OK;
}

// Leading dimension of stage 1's Z and Y for a batch of nb shapes (whole GEMM
// tiles).
static int stage1_ld(int nb, int R)
{
    return (nb * basis_tiles(R).cols + WT - 1) / WT * WT;
}

// Stage-1 GEMM C[m][ldc] = A[m][Kp] B[Kp][ldb] (B zero-padded to ldb columns
// and Kp rows, A to Kp columns): 64 x 64 tiles, 4 waves of 32
// x 32 on v_mfma_{f32,f64}_16x16x4, K chunks of 16 in
// double-buffered LDS, over the chunks ktiles[row tile] = (first, count)
// only (A is zero in the others).  Operands come in as 16-byte loads two chunks
// ahead of their use (two register sets), A stored [m][k] and B [k][n] with row
// strides that keep both the 16-byte stores and the MFMA operand reads free of
// bank conflicts.  The chunks run in K order.
//
// 64 x 64 tiles were never slower than 128 x 128 (two of those fit a CU): one
// shape of 200 nodes and 20 functions, 40 columns of which a 128-wide tile
// pads two thirds, 15.9 against 36.6 us in FP64; 8 shapes 33 against 54; 32
// shapes 98 against 111; 32 shapes of 300 nodes and 30 functions in FP32 259
// both.
template <class T>
__global__ __launch_bounds__(256, 4) void proj_gemm_w(const T* __restrict__ A, const T* __restrict__ B, int M, int Kp,
                                                      int ldb, T* __restrict__ C, int ldc,
                                                      const int2* __restrict__ ktiles)
{
    constexpr int TL = WT / 32;                                  // 16 x 16 tiles of a wave, each way
    constexpr int EV = 16 / sizeof(T);                           // elements of a load
    constexpr int LDA = PK + EV, LDB = WT + 64 / sizeof(T);      // LDS row strides
    constexpr int NL = WT * PK / EV / 256;                       // loads of A (and of B) a thread and chunk
    constexpr int QA = PK / EV, QB = WT / EV;                    // loads of an A row, of a B row
    typedef T TV __attribute__((ext_vector_type(EV)));
    typedef typename MF<T>::V Acc;
    __shared__ __align__(16) T As[2][WT][LDA];
    __shared__ __align__(16) T Bs[2][PK][LDB];
    const int m0 = blockIdx.y * WT, n0 = blockIdx.x * WT;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    Acc acc[TL][TL];
#pragma unroll
    for (int a = 0; a < TL; ++a)
#pragma unroll
        for (int b = 0; b < TL; ++b) acc[a][b] = (Acc){0, 0, 0, 0};
    // load e = tid + 256 u of a chunk: A row e / QA, k = EV (e % QA); B row k =
    // e / QB, n = EV (e % QB).  Rows of A past M repeat the last one (not stored).
    auto gload = [&](int k0, TV (&ra)[NL], TV (&rb)[NL]) {
#pragma unroll
        for (int u = 0; u < NL; ++u) {
            const int e = tid + 256 * u;
            ra[u] = *reinterpret_cast<const TV*>(A + (size_t)min(m0 + e / QA, M - 1) * Kp + k0 + EV * (e % QA));
            rb[u] = *reinterpret_cast<const TV*>(B + (size_t)(k0 + e / QB) * ldb + n0 + EV * (e % QB));
        }
    };
    auto sstore = [&](int buf, const TV (&ra)[NL], const TV (&rb)[NL]) {
#pragma unroll
        for (int u = 0; u < NL; ++u) {
            const int e = tid + 256 * u;
            *reinterpret_cast<TV*>(&As[buf][e / QA][EV * (e % QA)]) = ra[u];
            *reinterpret_cast<TV*>(&Bs[buf][e / QB][EV * (e % QB)]) = rb[u];
        }
    };
    auto compute = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < PK / 4; ++ks) {
            const int kk = ks * 4 + (lane >> 4);
            T av[TL], bv[TL];
#pragma unroll
            for (int a = 0; a < TL; ++a) av[a] = As[buf][(wm * TL + a) * 16 + (lane & 15)][kk];
#pragma unroll
            for (int b = 0; b < TL; ++b) bv[b] = Bs[buf][kk][(wn * TL + b) * 16 + (lane & 15)];
#pragma unroll
            for (int a = 0; a < TL; ++a)
#pragma unroll
                for (int b = 0; b < TL; ++b) acc[a][b] = MF<T>::mma(av[a], bv[b], acc[a][b]);
        }
    };
    // the tile's chunks c0 .. c0 + nk - 1 (the rest of W's rows here are
    // zero); chunk kc is in LDS buffer kc & 1, chunk kc + 1 in registers and
    // chunk kc + 2 loading; loads past the last chunk repeat it (unused), so
    // every load is unconditional
    const int2 kr = ktiles[blockIdx.y];
    const int c0 = kr.x, nk = kr.y;
    TV ra0[NL], rb0[NL], ra1[NL], rb1[NL];
    gload(c0 * PK, ra0, rb0);
    gload((c0 + min(1, nk - 1)) * PK, ra1, rb1);
    sstore(0, ra0, rb0);
    __syncthreads();
    for (int kc = 0;; kc += 2) {
        gload((c0 + min(kc + 2, nk - 1)) * PK, ra0, rb0);
        compute(0);
        sstore(1, ra1, rb1);
        __syncthreads();
        if (kc + 1 >= nk) break;
        gload((c0 + min(kc + 3, nk - 1)) * PK, ra1, rb1);
        compute(1);
        sstore(0, ra0, rb0);
        __syncthreads();
        if (kc + 2 >= nk) break;
    }
#pragma unroll
    for (int a = 0; a < TL; ++a)
#pragma unroll
        for (int b = 0; b < TL; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int gm = m0 + (wm * TL + a) * 16 + MF<T>::row(v, lane);
                const int gn = n0 + (wn * TL + b) * 16 + (lane & 15);
                if (gm < M) C[(size_t)gm * ldc + gn] = acc[a][b][v];
            }
}

template <class T>
static int run_stage1(mcmb_ctx* c, const double* d_theta, int nb, int& ldy, DevBuf& Yb)
{
    DevBuf& Zb = c->pz;
    PointSet& K = c->ks;
    const int N = K.lmax + 1, R = K.R, Kp = (N + PK - 1) / PK * PK;
    const int ldz = stage1_ld(nb, R);
    ldy = ldz;
    MCMB_TRY(Zb.alloc(sizeof(T) * (size_t)Kp * ldz));
    const long M = (long)N * (N + 1) / 2;   // pair rows i <= j
    MCMB_TRY(Yb.alloc(sizeof(T) * (size_t)M * ldy));
    size_t ze = (size_t)Kp * ldz;
    hipLaunchKernelGGL(proj_build_Z<T>, dim3((unsigned)((ze + 255) / 256)), dim3(256), 0, c->stream,
                       K.d_kn.as<double>(), K.d_q.as<double>(), K.ldq, N, R, d_theta, nb, Kp, ldz, Zb.as<T>());
    const dim3 grid((unsigned)(ldz / WT), (unsigned)((M + WT - 1) / WT));
    hipLaunchKernelGGL(proj_gemm_w<T>, grid, dim3(256), 0, c->stream, (const T*)c->d_W.as<T>(), (const T*)Zb.as<T>(),
                       (int)M, Kp, ldz, Yb.as<T>(), ldy, (const int2*)c->d_wtile.as<int2>());
    MCMB_HIP(hipGetLastError());
    return MCMB_OK;
}

// sin / cos of omega_b k_j for the nb shapes of a batch into c->psc
static int sincos_table(mcmb_ctx* c, const double* d_theta, int nb)
{
    const int N = c->ks.lmax + 1, Np = stage2_nodes(N);
    MCMB_TRY(c->psc.alloc(sizeof(double) * 2 * (size_t)PBATCH * Np));
    hipLaunchKernelGGL(proj_sincos_tab, dim3((unsigned)((nb * Np + 255) / 256)), dim3(256), 0, c->stream,
                       c->ks.d_kn.as<double>(), d_theta, N, Np, nb, c->psc.as<double>());
    MCMB_HIP(hipGetLastError());
    return MCMB_OK;
}

// Stages 2 and 3 of a batch from its stage-1 product: D[b][d] (c->pdm) for the
// planes X (1 sin, 2 cos, 3 both).
template <class T, int X, int NT>
static int run_stages23(mcmb_ctx* c, const double* d_theta, int nb, const T* Y, int ldy)
{
    PointSet& K = c->ks;
    constexpr int NX = (X & 1) + (X >> 1);
    const int N = K.lmax + 1, R = K.R, PP = sym_cols(R);
    MCMB_TRY(c->ph.alloc(sizeof(double) * (size_t)PBATCH * NX * N * PP));
    MCMB_TRY(c->pdm.alloc(sizeof(double) * (size_t)PBATCH * 3 * R * PP));
    MCMB_TRY(sincos_table(c, d_theta, nb));
    const bool two = X != 3 && (long)nb * N >= S2_PAIR;
    const int ni = two ? (N + 1) / 2 : N;
    const dim3 grid((unsigned)((ni + 7) / 8 * 8 * nb));
    auto* const k2 = two ? proj_stage2<T, X, NT, X != 3 ? 2 : 1> : proj_stage2<T, X, NT, 1>;
    hipLaunchKernelGGL(k2, grid, dim3(256), 0, c->stream, Y, ldy, (const int*)c->d_wrow.as<int>(), K.d_kn.as<double>(),
                       (const double*)c->d_pq.as<double>(), N, R, PP, d_theta, nb, (const double*)c->psc.as<double>(),
                       c->ph.as<double>());
    hipLaunchKernelGGL((proj_stage3<X, NT>), dim3((unsigned)(nb * NX * (PP / 16))), dim3(256), 0, c->stream,
                       (const double*)c->ph.as<double>(), K.d_q.as<double>(), K.ldq, K.d_kn.as<double>(), N, R, PP,
                       c->pdm.as<double>());
    MCMB_HIP(hipGetLastError());
    return MCMB_OK;
}

// Y is stage 1's product buffer (the context's batch buffer, or a slot of
// the forward cache).  d_dalpha null: alpha alone.
template <class T>
static int project_fwd_batch(mcmb_ctx* c, const double* d_theta, int nb, double* d_alpha /* [nb][n] */,
                             double* d_dalpha /* [nb][2][n] */, DevBuf& Yb)
{
    PointSet& K = c->ks;
    const int R = K.R, n = K.n, nx = d_dalpha ? 3 : 1;
    int ldy = 0;
    MCMB_TRY(run_stage1<T>(c, d_theta, nb, ldy, Yb));
    const T* const Y = Yb.as<T>();
    if (d_dalpha)
        MCMB_TRY(R > 16 ? (run_stages23<T, 3, 2>(c, d_theta, nb, Y, ldy)) : (run_stages23<T, 3, 1>(c, d_theta, nb, Y, ldy)));
    else
        MCMB_TRY(R > 16 ? (run_stages23<T, 1, 2>(c, d_theta, nb, Y, ldy)) : (run_stages23<T, 1, 1>(c, d_theta, nb, Y, ldy)));
    const int ne = nb * nx * n;
    hipLaunchKernelGGL(proj_stage3_modes, dim3((ne + 255) / 256), dim3(256), 0, c->stream,
                       (const double*)c->pdm.as<double>(), R, sym_cols(R), K.d_modes.as<int>(), n, nb, nx, d_alpha,
                       d_dalpha);
    MCMB_HIP(hipGetLastError());
    return MCMB_OK;
}

// Ycached: stage 1's product of this batch from the forward cache, or null to
// compute it.
template <class T>
static int project_bwd_batch(mcmb_ctx* c, const double* d_theta, int nb, const double* d_gbar, double* d_dtheta,
                             DevBuf* Ycached)
{
    PointSet& K = c->ks;
    const int N = K.lmax + 1, R = K.R, n = K.n;
    // a cached product is this batch's own: same shape count, so the same
    // leading dimension; anything smaller than that is recomputed
    const long M = (long)N * (N + 1) / 2;
    int ldy = stage1_ld(nb, R);
    if (Ycached && Ycached->bytes < sizeof(T) * (size_t)M * ldy) Ycached = nullptr;
    DevBuf& Yb = Ycached ? *Ycached : c->py;
    if (!Ycached) MCMB_TRY(run_stage1<T>(c, d_theta, nb, ldy, Yb));
    const T* const Y = Yb.as<T>();
    MCMB_TRY(R > 16 ? (run_stages23<T, 2, 2>(c, d_theta, nb, Y, ldy)) : (run_stages23<T, 2, 1>(c, d_theta, nb, Y, ldy)));
    hipLaunchKernelGGL(proj_dtheta, dim3((unsigned)nb), dim3(512), 0, c->stream, (const double*)c->pdm.as<double>(), R,
                       sym_cols(R), K.d_modes.as<int>(), n, d_gbar, d_dtheta);
    MCMB_HIP(hipGetLastError());
    return MCMB_OK;
}

// The forward cache holds every batch's stage-1 product when they fit in
// PCACHE_BYTES together.
constexpr size_t PCACHE_BYTES = 24ull << 30;

// Host threads that move a batch's slot: starting one costs more (about 15 us)
// than it saves below 256 KiB.
static int transfer_threads(size_t slot_bytes)
{
    return (int)std::min<size_t>(std::min(8, host_threads()), 1 + slot_bytes / (256u << 10));
}

static size_t ybytes(const mcmb_ctx* c, int prec)
{
    const PointSet& K = c->ks;
    const int N = K.lmax + 1, R = K.R;
    const long M = (long)N * (N + 1) / 2;
    return (prec == MCMB_FP64 ? sizeof(double) : sizeof(float)) * (size_t)M * stage1_ld(PBATCH, R);
}

}  // namespace mcmb

using namespace mcmb;

extern "C" {

int mcmb_kspace_set(mcmb_ctx* c, int N, const double* kn, const double* kw, int ldq, const double* q, int nmodes,
                    const int* order)
{
    if (!c || !kn || !kw || !q || !order) return fail(MCMB_ERR_ARG, "mcmb_kspace_set: null argument");
    if (N < 2 || N > 4096) return fail(MCMB_ERR_ARG, "mcmb_kspace_set: N %d not in [2,4096]", N);
    if (ldq < 1 || ldq > 32) return fail(MCMB_ERR_ARG, "mcmb_kspace_set: ldq %d not in [1,32]", ldq);
    if (nmodes < 1 || nmodes > 65536) return fail(MCMB_ERR_ARG, "mcmb_kspace_set: nmodes %d", nmodes);
    for (int a = 1; a < N; ++a)
        if (!(kn[a] > kn[a - 1]) || !(kn[0] > 0.0))
            return fail(MCMB_ERR_ARG, "mcmb_kspace_set: nodes must be positive and strictly ascending");
    int R = 0;
    for (int m = 0; m < nmodes; ++m)
        for (int a = 0; a < 3; ++a) {
            int p = order[3 * m + a];
            if (p < 0 || p >= ldq)
                return fail(MCMB_ERR_ORDER, "mcmb_kspace_set: order[%d][%d] = %d outside [0,%d)", m, a, p, ldq);
            if (p + 1 > R) R = p + 1;
        }
    MCMB_TRY(set_device(c));
    PointSet& K = c->ks;
    K.ready = false;
    K.kspace = true;
    K.kstep = 1;
    K.lmin = 0;
    K.lmax = N - 1;
    K.ldq = ldq;
    K.n = nmodes;
    K.R = R;
    K.order.assign(order, order + 3 * (size_t)nmodes);
    K.q.assign(q, q + (size_t)N * ldq);
    K.kn.assign(kn, kn + N);
    K.kw.assign(kw, kw + N);
    // ordered masked points a <= b <= c, k_c <= k_a + k_b (nodes ascending)
    K.rows.clear();
    K.npoints = 0;
    for (int a = 0; a < N; ++a)
        for (int b = a; b < N; ++b) {
            int cmax = b;
            while (cmax + 1 < N && kn[cmax + 1] <= kn[a] + kn[b]) ++cmax;
            K.rows.push_back(RowDesc{a, b, b, cmax - b + 1});
            K.npoints += cmax - b + 1;
        }
    MCMB_TRY(K.d_kn.alloc(sizeof(double) * N));
    MCMB_TRY(K.d_kw.alloc(sizeof(double) * N));
    MCMB_HIP(hipMemcpyAsync(K.d_kn.p, kn, sizeof(double) * N, hipMemcpyHostToDevice, c->stream));
    MCMB_HIP(hipMemcpyAsync(K.d_kw.p, kw, sizeof(double) * N, hipMemcpyHostToDevice, c->stream));
    MCMB_TRY(upload_pointset(c, K, K.order));
    c->w_ready = 0;
    K.ready = true;
    K.generation = next_generation();
    return MCMB_OK;
}

long mcmb_kspace_npoints(mcmb_ctx* c)
{
    if (!c || !c->ks.ready) return fail(MCMB_ERR_STATE, "mcmb_kspace_npoints: no k-space setup");
    return c->ks.npoints;
}

int mcmb_kgram(mcmb_ctx* c, int precision, double* gamma_host, double* gamma_dev)
{
    if (!c) return fail(MCMB_ERR_ARG, "mcmb_kgram: null context");
    if (!c->ks.ready) return fail(MCMB_ERR_STATE, "mcmb_kgram: call mcmb_kspace_set first");
    if (precision != MCMB_FP64 && precision != MCMB_MIXED) return fail(MCMB_ERR_ARG, "mcmb_kgram: precision %d", precision);
    MCMB_TRY(set_device(c));
    const int n = c->ks.n;
    double* dst = gamma_dev;
    if (!dst) {
        MCMB_TRY(c->d_gamma_tmp.alloc(sizeof(double) * (size_t)n * n));
        dst = c->d_gamma_tmp.as<double>();
    }
    MCMB_TRY(gram_tet_launch(c, c->ks, precision, dst, 0, (int)c->ks.rows.size()));
    if (gamma_host)
        MCMB_TRY(copy_to_host(c, gamma_host, dst, sizeof(double) * (size_t)n * n));
    MCMB_HIP(hipStreamSynchronize(c->stream));
    return MCMB_OK;
}

int mcmb_project_fwd(mcmb_ctx* c, int precision, int ntheta, const double* theta, double* alpha, double* dalpha)
{
    if (!c || !theta || !alpha || ntheta < 1) return fail(MCMB_ERR_ARG, "mcmb_project_fwd: bad argument");
    if (!c->ks.ready) return fail(MCMB_ERR_STATE, "mcmb_project_fwd: call mcmb_kspace_set first");
    if (precision != MCMB_FP64 && precision != MCMB_FP32) return fail(MCMB_ERR_ARG, "mcmb_project_fwd: precision %d", precision);
    MCMB_TRY(set_device(c));
    const int n = c->ks.n;
    MCMB_TRY(ensure_W(c, precision));
    const int nbat = (ntheta + PBATCH - 1) / PBATCH;
    // keep each batch's stage-1 product for a backward call on the same shapes
    const bool cache = (size_t)nbat * ybytes(c, precision) <= PCACHE_BYTES;
    c->ycache_gen = -1;
    if (cache && (int)c->ycache.size() < nbat) c->ycache.resize(nbat);
    // device arrays of the call: theta [ntheta][2], alpha [ntheta][n], dalpha [ntheta][2][n]
    MCMB_TRY(c->pio.alloc(sizeof(double) * (2 + 3 * (size_t)n) * ntheta));
    double* const dth = c->pio.as<double>();
    double* const dal = dth + 2 * (size_t)ntheta;
    double* const ddal = dal + (size_t)ntheta * n;
    // Each batch's results go to the host while later batches compute: once
    // the batch's kernels are done, the copy stream moves its alpha (and
    // dalpha) into slot bi % nslot of the pinned staging, and host threads
    // move the slots on to the caller's arrays in batch order, so only the
    // last batch's transfer follows the GPU work.
    const int nout = dalpha ? 3 : 1;
    const size_t slot_bytes = sizeof(double) * (size_t)std::min(PBATCH, ntheta) * n * nout;
    const int nslot = (int)std::min<size_t>(PSLOTS, 2 * STAGE_BYTES / slot_bytes);
    const char* cenv = getenv("MCMB_HOST_COPY");
    const bool staged = nslot >= 1 && !(cenv && !strcmp(cenv, "direct"));
    if (staged) MCMB_TRY(copy_stream_ready(c));
    const int nth = transfer_threads(slot_bytes);
    auto drain = [&](int bi) -> int {
        MCMB_HIP(hipEventSynchronize(c->slot_ev[1][bi % nslot]));
        const int b0 = bi * PBATCH, nb = std::min(PBATCH, ntheta - b0);
        const double* sl = reinterpret_cast<const double*>(static_cast<char*>(c->stage) + (bi % nslot) * slot_bytes);
        const size_t na = (size_t)nb * n;
        run_threads(nth, [&](int t) {
            const size_t a = na * t / nth, b = na * (t + 1) / nth;
            memcpy(alpha + (size_t)b0 * n + a, sl + a, sizeof(double) * (b - a));
            if (dalpha) memcpy(dalpha + (size_t)b0 * 2 * n + 2 * a, sl + na + 2 * a, sizeof(double) * 2 * (b - a));
        });
        return MCMB_OK;
    };
    MCMB_HIP(hipEventRecord(c->ev0, c->stream));
    MCMB_HIP(hipMemcpyAsync(dth, theta, sizeof(double) * 2 * (size_t)ntheta, hipMemcpyHostToDevice, c->stream));
    for (int b0 = 0, bi = 0; b0 < ntheta; b0 += PBATCH, ++bi) {
        const int nb = std::min(PBATCH, ntheta - b0);
        DevBuf& Yb = cache ? c->ycache[bi] : c->py;
        double* d_al = dal + (size_t)b0 * n;
        double* d_dal = dalpha ? ddal + (size_t)b0 * 2 * n : nullptr;
        if (precision == MCMB_FP64)
            MCMB_TRY(project_fwd_batch<double>(c, dth + 2 * b0, nb, d_al, d_dal, Yb));
        else
            MCMB_TRY(project_fwd_batch<float>(c, dth + 2 * b0, nb, d_al, d_dal, Yb));
        if (staged) {
            if (bi >= nslot) MCMB_TRY(drain(bi - nslot));   // the slot's previous batch
            const int k = bi % nslot;
            char* sl = static_cast<char*>(c->stage) + k * slot_bytes;
            MCMB_HIP(hipEventRecord(c->slot_ev[0][k], c->stream));
            MCMB_HIP(hipStreamWaitEvent(c->cstream, c->slot_ev[0][k], 0));
            MCMB_HIP(hipMemcpyAsync(sl, d_al, sizeof(double) * (size_t)nb * n, hipMemcpyDeviceToHost, c->cstream));
            if (dalpha)
                MCMB_HIP(hipMemcpyAsync(sl + sizeof(double) * (size_t)nb * n, d_dal, sizeof(double) * 2 * (size_t)nb * n,
                                        hipMemcpyDeviceToHost, c->cstream));
            MCMB_HIP(hipEventRecord(c->slot_ev[1][k], c->cstream));
        }
    }
    MCMB_HIP(hipEventRecord(c->ev1, c->stream));
    if (staged) {
        for (int bi = std::max(0, nbat - nslot); bi < nbat; ++bi) MCMB_TRY(drain(bi));
    } else {
        // the device arrays already have the caller's layout: one contiguous copy each
        MCMB_HIP(hipMemcpyAsync(alpha, dal, sizeof(double) * (size_t)ntheta * n, hipMemcpyDeviceToHost, c->stream));
        if (dalpha)
            MCMB_HIP(hipMemcpyAsync(dalpha, ddal, sizeof(double) * (size_t)ntheta * 2 * n, hipMemcpyDeviceToHost,
                                    c->stream));
    }
    MCMB_HIP(hipStreamSynchronize(c->stream));
    if (cache) {
        c->ycache_theta.assign(theta, theta + 2 * (size_t)ntheta);
        c->ycache_prec = precision;
        c->ycache_gen = c->ks.generation;
    }
    float ms = 0.f;
    MCMB_HIP(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    c->last_launches = nbat;
    return MCMB_OK;
}

int mcmb_project_bwd(mcmb_ctx* c, int precision, int ntheta, const double* theta, const double* gbar, double* dtheta)
{
    if (!c || !theta || !gbar || !dtheta || ntheta < 1) return fail(MCMB_ERR_ARG, "mcmb_project_bwd: bad argument");
    if (!c->ks.ready) return fail(MCMB_ERR_STATE, "mcmb_project_bwd: call mcmb_kspace_set first");
    if (precision != MCMB_FP64 && precision != MCMB_FP32) return fail(MCMB_ERR_ARG, "mcmb_project_bwd: precision %d", precision);
    MCMB_TRY(set_device(c));
    PointSet& K = c->ks;
    const int n = K.n, R = K.R;
    MCMB_TRY(ensure_W(c, precision));
    // a triple may be listed once only
    std::vector<char> seen((size_t)R * R * R, 0);
    for (int m = 0; m < n; ++m) {
        int r = K.order[3 * m], s = K.order[3 * m + 1], t = K.order[3 * m + 2];
        char& sl = seen[((size_t)r * R + s) * R + t];
        if (sl) return fail(MCMB_ERR_ORDER, "mcmb_project_bwd: repeated mode (%d,%d,%d)", r, s, t);
        sl = 1;
    }
    // device arrays of the call: theta [ntheta][2], gbar [ntheta][n], dtheta [ntheta][2]
    MCMB_TRY(c->pio.alloc(sizeof(double) * (4 + (size_t)n) * ntheta));
    double* const dth = c->pio.as<double>();
    double* const dg = dth + 2 * (size_t)ntheta;
    double* const dd = dg + (size_t)ntheta * n;
    // the last forward's stage-1 products, when it ran on exactly these shapes
    const bool cached = c->ycache_gen == K.generation && c->ycache_prec == precision &&
                        c->ycache_theta.size() == 2 * (size_t)ntheta &&
                        !memcmp(c->ycache_theta.data(), theta, sizeof(double) * 2 * (size_t)ntheta);
    // gbar goes up batch by batch through slots of the pinned staging: host
    // threads fill slot bi % nslot while the GPU works on earlier batches
    const size_t slot_bytes = sizeof(double) * (size_t)std::min(PBATCH, ntheta) * n;
    const int nslot = (int)std::min<size_t>(PSLOTS, 2 * STAGE_BYTES / slot_bytes);
    const char* cenv = getenv("MCMB_HOST_COPY");
    const bool staged = nslot >= 1 && !(cenv && !strcmp(cenv, "direct"));
    if (staged) MCMB_TRY(copy_stream_ready(c));
    const int nth = transfer_threads(slot_bytes);
    MCMB_HIP(hipEventRecord(c->ev0, c->stream));
    MCMB_HIP(hipMemcpyAsync(dth, theta, sizeof(double) * 2 * (size_t)ntheta, hipMemcpyHostToDevice, c->stream));
    if (!staged)
        MCMB_HIP(hipMemcpyAsync(dg, gbar, sizeof(double) * (size_t)ntheta * n, hipMemcpyHostToDevice, c->stream));
    for (int b0 = 0, bi = 0; b0 < ntheta; b0 += PBATCH, ++bi) {
        const int nb = std::min(PBATCH, ntheta - b0);
        DevBuf* Yc = cached ? &c->ycache[bi] : nullptr;
        const double* th = dth + 2 * b0;
        double* gb = dg + (size_t)b0 * n;
        double* dt = dd + 2 * b0;
        if (staged) {
            const int k = bi % nslot;
            // the slot's previous upload has been read
            if (bi >= nslot) MCMB_HIP(hipEventSynchronize(c->slot_ev[0][k]));
            double* sl = reinterpret_cast<double*>(static_cast<char*>(c->stage) + k * slot_bytes);
            const size_t na = (size_t)nb * n;
            run_threads(nth, [&](int t) {
                const size_t a = na * t / nth, b = na * (t + 1) / nth;
                memcpy(sl + a, gbar + (size_t)b0 * n + a, sizeof(double) * (b - a));
            });
            MCMB_HIP(hipMemcpyAsync(gb, sl, sizeof(double) * na, hipMemcpyHostToDevice, c->stream));
            MCMB_HIP(hipEventRecord(c->slot_ev[0][k], c->stream));
        }
        if (precision == MCMB_FP64)
            MCMB_TRY(project_bwd_batch<double>(c, th, nb, gb, dt, Yc));
        else
            MCMB_TRY(project_bwd_batch<float>(c, th, nb, gb, dt, Yc));
    }
    MCMB_HIP(hipMemcpyAsync(dtheta, dd, sizeof(double) * 2 * (size_t)ntheta, hipMemcpyDeviceToHost, c->stream));
    MCMB_HIP(hipEventRecord(c->ev1, c->stream));
    MCMB_HIP(hipStreamSynchronize(c->stream));
    float ms = 0.f;
    MCMB_HIP(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    c->last_launches = (ntheta + PBATCH - 1) / PBATCH;
    return MCMB_OK;
}

}  // extern "C"

// ---- Gamma post-processing (gamma_mpi.c:260-295, 801-840) -------------------
// orthoinv = lambda^T lambda, Gamma' = orthoinv Gamma, FP64 MFMA products
// (proj_gemm<double>: A n x Kp, B Kp x n, both zero-padded in K).
__global__ void la_pad(const double* __restrict__ src, int n, int trans, int rows, int cols,
                       double* __restrict__ dst)
{
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (long)rows * cols) return;
    const int r = (int)(e / cols), c = (int)(e % cols);
    dst[e] = (r < n && c < n) ? (trans ? src[(long)c * n + r] : src[(long)r * n + c]) : 0.0;
}

extern "C" int mcmb_gamma_post(mcmb_ctx* c, int n, const double* lambda, const double* gamma, double* orthoinv,
                               double* gamma_out)
{
    if (!c || n < 1 || !lambda || !gamma || !gamma_out) return fail(MCMB_ERR_ARG, "mcmb_gamma_post: bad arguments");
    MCMB_TRY(set_device(c));
    const int Kp = (n + PK - 1) / PK * PK;
    const size_t nn = (size_t)n * n, np = (size_t)n * Kp;
    DevBuf dL, dG, dA, dB, dC;
    MCMB_TRY(dL.alloc(sizeof(double) * nn));
    MCMB_TRY(dG.alloc(sizeof(double) * nn));
    MCMB_TRY(dA.alloc(sizeof(double) * np));
    MCMB_TRY(dB.alloc(sizeof(double) * np));
    MCMB_TRY(dC.alloc(sizeof(double) * nn));
    MCMB_TRY(copy_to_device(c, dL.p, lambda, sizeof(double) * nn));
    MCMB_TRY(copy_to_device(c, dG.p, gamma, sizeof(double) * nn));
    const unsigned gp = (unsigned)((np + 255) / 256);
    const dim3 grid((unsigned)((n + PT - 1) / PT), (unsigned)((n + PT - 1) / PT));
    MCMB_HIP(hipEventRecord(c->ev0, c->stream));
    // orthoinv[i][j] = sum_k lambda[k][i] lambda[k][j]
    hipLaunchKernelGGL(la_pad, dim3(gp), dim3(256), 0, c->stream, dL.as<double>(), n, 1, n, Kp, dA.as<double>());
    hipLaunchKernelGGL(la_pad, dim3(gp), dim3(256), 0, c->stream, dL.as<double>(), n, 0, Kp, n, dB.as<double>());
    hipLaunchKernelGGL(proj_gemm<double>, grid, dim3(256), 0, c->stream, dA.as<double>(), dB.as<double>(), n, Kp, n,
                       n, dC.as<double>(), n);
    // Gamma'[i][j] = sum_m orthoinv[i][m] Gamma[m][j]
    hipLaunchKernelGGL(la_pad, dim3(gp), dim3(256), 0, c->stream, dC.as<double>(), n, 0, n, Kp, dA.as<double>());
    hipLaunchKernelGGL(la_pad, dim3(gp), dim3(256), 0, c->stream, dG.as<double>(), n, 0, Kp, n, dB.as<double>());
    hipLaunchKernelGGL(proj_gemm<double>, grid, dim3(256), 0, c->stream, dA.as<double>(), dB.as<double>(), n, Kp, n,
                       n, dG.as<double>(), n);
    MCMB_HIP(hipGetLastError());
    MCMB_HIP(hipEventRecord(c->ev1, c->stream));
    if (orthoinv) MCMB_TRY(copy_to_host(c, orthoinv, dC.p, sizeof(double) * nn));
    MCMB_TRY(copy_to_host(c, gamma_out, dG.p, sizeof(double) * nn));
    MCMB_HIP(hipStreamSynchronize(c->stream));
    float ms = 0.f;
    MCMB_HIP(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    c->last_launches = 2;
    return MCMB_OK;
}
