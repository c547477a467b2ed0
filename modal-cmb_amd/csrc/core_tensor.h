// Core tensor of triple products over nodes, FP64 MFMA: used by the
// Gauss-Legendre cross-Gamma (samples of x) and Gram (chunks of nodes).
//
//   H_u[f][g][h] = sum over the unit's samples x and nodes k of
//                  wk[x wstride + k] sc[x] M[x][f][k] M[x][g][k] M[x][h][k]
//
// a GEMM over the nodes with A = (w M_b) M_a formed in registers; M[x][f][k] is
// of one field or (f, g) of one and h of another.
//
// Tiles of 16 functions.  SAME (one field): f <= g <= h, tile ta of a, one b
// in tile tb >= ta, tiles tc >= tb of c, stored tile by tile (cx_tile).
// Otherwise the pair (a, b) is of one field and c, any tile, of the other.
// One workgroup per (tb, ta, four tiles of c): wave w has b = 16 tb + 4w ..+3,
// 16 accumulator tiles, per K-step of 4 nodes 16 MFMAs on 9 LDS reads.
#pragma once
#include <hip/hip_runtime.h>

namespace mcmb {

typedef double d4 __attribute__((ext_vector_type(4)));

__host__ __device__ __forceinline__ int cx_jobs(int tb, int NTC, bool same)
{
    return (tb + 1) * ((NTC - (same ? tb : 0) + 3) / 4);
}
// tiles before the first of b-tile tb
__host__ __device__ __forceinline__ long cx_base(int tb, int NTC, bool same)
{
    long o = 0;
    for (int t = 0; t < tb; ++t) o += 16l * (t + 1) * (NTC - (same ? t : 0));
    return o;
}
__device__ __forceinline__ long cx_tile(long base, int ta, int b, int tc, int NTC, bool same)
{
    const int tb = b >> 4, lo = same ? tb : 0;
    return base + (long)((b & 15) * (tb + 1) + ta) * (NTC - lo) + (tc - lo);
}

// Samples of unit u: the ng groups of g samples from nm on, then the nm single ones.
__device__ __forceinline__ int cx_unit(int u, int nm, int ng, int g, int nx, int* n)
{
    if (u >= ng) {
        *n = 1;
        return u - ng;
    }
    *n = min(g, nx - nm - u * g);
    return nm + u * g;
}

template <bool SAME>
__global__ __launch_bounds__(256, 2) void cx_core(const double* __restrict__ MA, int FA, const double* __restrict__ MC,
                                                  int FC, int K, const double* __restrict__ wk,
                                                  long wstride, const double* __restrict__ sc, int nm, int ng, int g, int nx, int u0,
                                                  double* __restrict__ H, long us)
{
    __shared__ double S[2][96][17];   // 16 a, 16 b, 64 c rows of 16 nodes
    __shared__ double Ws[2][16];
    const int NTC = (FC + 15) >> 4;
    int tb = 0, job = blockIdx.x;
    for (int nj; job >= (nj = cx_jobs(tb, NTC, SAME)); ++tb) job -= nj;
    const int ta = job % (tb + 1), tc0 = (SAME ? tb : 0) + 4 * (job / (tb + 1)), nct = min(4, NTC - tc0);
    int nxu;
    const int xb = cx_unit(u0 + blockIdx.y, nm, ng, g, nx, &nxu);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int b0 = 16 * tb + 4 * wave;
    const bool live = b0 < FA;
    d4 acc[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[r][t] = d4{0.0, 0.0, 0.0, 0.0};
    // the six elements a thread stages: row e >> 4, node e & 15
    const double* src[6];
    double rs[6], rw = 0.0;
    const int kk = tid & 15;
#pragma unroll
    for (int u = 0; u < 6; ++u) {
        const int row = (tid >> 4) + 16 * u;
        const int f = u == 0 ? 16 * ta + row : u == 1 ? 16 * tb + row - 16 : 16 * tc0 + row - 32;
        src[u] = u < 2 ? (f < FA ? MA + ((long)xb * FA + f) * K + kk : nullptr)
                       : (f < FC ? MC + ((long)xb * FC + f) * K + kk : nullptr);
    }
    const int nk = K / 16;
    int lx = 0, lk = 0;   // sample and stage of the next load
    auto gload = [&]() {
        const long oa = (long)lx * FA * K + 16l * lk, oc = (long)lx * FC * K + 16l * lk;
#pragma unroll
        for (int u = 0; u < 6; ++u) rs[u] = src[u] ? src[u][u < 2 ? oa : oc] : 0.0;
        if (tid < 16) rw = wk[(xb + lx) * wstride + 16 * lk + kk] * (sc ? sc[xb + lx] : 1.0);
        if (++lk == nk) {
            lk = 0;
            ++lx;
        }
    };
    auto sstore = [&](int buf) {
#pragma unroll
        for (int u = 0; u < 6; ++u) S[buf][(tid >> 4) + 16 * u][kk] = rs[u];
        if (tid < 16) Ws[buf][kk] = rw;
    };
    gload();
    sstore(0);
    __syncthreads();
    const int nst = nxu * nk;
    for (int st = 0; st < nst; ++st) {
        const int buf = st & 1;
        if (st + 1 < nst) gload();
        if (live)
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                const int k = 4 * ks + (lane >> 4), col = lane & 15;
                const double ma = S[buf][col][k], w = Ws[buf][k];
                double mb[4], mc[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) mb[r] = ma * (S[buf][16 + 4 * wave + r][k] * w);
#pragma unroll
                for (int t = 0; t < 4; ++t) mc[t] = S[buf][32 + 16 * t + col][k];
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (t < nct)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            acc[r][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(mb[r], mc[t], acc[r][t], 0, 0, 0);
            }
        if (st + 1 < nst) sstore(buf ^ 1);
        __syncthreads();
    }
    if (!live) return;
    double* const Hu = H + (long)blockIdx.y * us;
    const long base = cx_base(tb, NTC, SAME);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (b0 + r < FA && t < nct) {
                double* const o = Hu + cx_tile(base, ta, b0 + r, tc0 + t, NTC, SAME) * 256;
#pragma unroll
                for (int v = 0; v < 4; ++v) o[16 * (4 * v + (lane >> 4)) + (lane & 15)] = acc[r][t][v];
            }
}

}  // namespace mcmb
