// The exact l-space Gram as a node sum over the compressed pair basis, in
// double-double arithmetic.
//
// With int P_l1 P_l2 P_l3 = 2 (l1 l2 l3; 0 0 0)^2 the tetrapyd sum over the
// basis columns (gram_sep.hip) is
//   H[a][b][c] = (3 / 4 pi) sum_s w_s Phi_a Phi_b Phi_c(x_s),
//   Phi_a(x)   = sum_l T[l][a] P_l(x),  T[l][a] = (2l + 1) v_l P[l][a],
// exact with Gauss-Legendre nodes of degree 3 lmax: the selection rules of the
// 3j symbols, which the tetrapyd's walk spells out point by point, come from
// the orthogonality of the P_l.  The work falls from N_tet r + rows r^2
// (lmax 2500, r = 59: 5e10 multiply-adds) to r L npt / 2 + r^3 npt / 6
// (4.1e8), but the sum cancels: the terms the rules forbid are as large as
// L^2 times the result, which is why the FP64 node sum (mcmb_gamma_gl) keeps
// only ten digits.  So the nodes, P_l, Phi and the node sum are carried in
// double-double (T, as in the tetrapyd order, is rounded once), and H is
// rounded once at the end.  What double-double leaves of the forbidden terms is
// alike for all entries, so an entry that the rules make small (columns of
// local support or of one parity) or zero would be lost in it: gl_gate
// compares it with what the rules allow, entry by entry, on the first call of a
// setup, and a setup with an entry that does not pass takes the tetrapyd
// contraction.  Measured, core tensor by the tetrapyd contraction -> as a node
// sum: lmax 2500, r = 59: 2.20 -> 0.18 ms; lmax 2000, r = 39: 1.22 -> 0.07 ms.
//
// Both parities of l are summed apart (P_l(-x) = (-1)^l P_l(x)), so the table
// holds the nodes x >= 0 only, and the columns at +x and -x are E + O and
// E - O.
#include "core_tensor.h"
#include "dd.h"
#include "mcmb_internal.h"
#include <cmath>
#include <vector>

namespace mcmb {

// cl[l] = (l - 1) / l for 2 <= l <= n
__global__ void gl_coef(int n, dd* __restrict__ cl)
{
    const int l = blockIdx.x * 256 + threadIdx.x;
    if (l <= n) cl[l] = l >= 2 ? dd{l - 1.0, 0.0} / dd{(double)l, 0.0} : dd{0.0, 0.0};
}

// Stages the coefficients l0 <= l < l0 + GN_CK of a recurrence in LDS.
constexpr int GN_CK = 512;
__device__ __forceinline__ int stage_coef(const dd* __restrict__ cl, int l0, int lmax, dd* sc)
{
    const int nl = min(GN_CK, lmax - l0 + 1);
    __syncthreads();
    for (int e = threadIdx.x; e < nl; e += 64) sc[e] = cl[l0 + e];
    __syncthreads();
    return nl;
}

// Nodes and weights of the rule of order n, x >= 0 ascending (the middle node
// of an odd rule at s = 0 with half its weight: it is summed at +x and -x).
// Newton's method in FP64 from the asymptotic root leaves x0 within an ulp;
// P_n(x0) in double-double (the recurrence P_l = t + c_l (t - P_{l-2}), t = x
// P_{l-1}) and the next Taylor term, from (1 - x^2) P'' = 2 x P' - n (n + 1)
// P, make the step to a root good to 1e-32.  One thread per node: a serial
// chain of n steps per evaluation (0.58 ms at 3751 nodes, once per rule).
__global__ __launch_bounds__(64) void gl_rule(int n, int half, int SH, const dd* __restrict__ cl, dd* __restrict__ x,
                                              dd* __restrict__ w)
{
#pragma clang fp contract(off)
    __shared__ dd sc[GN_CK];
    const int s = blockIdx.x * 64 + threadIdx.x;
    const bool mid = (n & 1) && s == 0;
    const int i = max(0, n - 1 - (n / 2 + s));   // from the largest root down (past half: the largest again)
    double x0 = mid ? 0.0 : cos(M_PI * (4.0 * i + 3.0) / (4.0 * n + 2.0)) * (1.0 - (n - 1.0) / (8.0 * n * (double)n * n));
    for (int it = 0; it < 3; ++it) {
        double p0 = 1.0, p1 = x0;
        for (int l0 = 2; l0 <= n; l0 += GN_CK) {
            const int nl = stage_coef(cl, l0, n, sc);
#pragma unroll 8
            for (int e = 0; e < nl; ++e) {
                const double t = x0 * p1, p = __builtin_fma(sc[e].hi, t - p0, t);
                p0 = p1;
                p1 = p;
            }
        }
        const double step = mid ? 0.0 : p1 * (x0 * x0 - 1.0) / (n * (x0 * p1 - p0));
        x0 -= step;
        if (__all(fabs(step) < 1e-15)) break;
    }
    dd p0{1.0, 0.0}, p1{x0, 0.0};
    for (int l0 = 2; l0 <= n; l0 += GN_CK) {
        const int nl = stage_coef(cl, l0, n, sc);
#pragma unroll 4
        for (int e = 0; e < nl; ++e) {
            const dd t = x0 * p1, p = t + sc[e] * (t - p0);
            p0 = p1;
            p1 = p;
        }
    }
    const dd x0d{x0, 0.0}, nn{(double)n, 0.0};
    const dd om = dd{1.0, 0.0} - two_prod(x0, x0);               // 1 - x0^2
    const dd f1 = nn * (p0 - x0d * p1) / om;                       // P'
    const dd f2 = (2.0 * (x0d * f1) - ((n * (n + 1.0)) * p1)) / om; // P''
    const double u = p1.hi / f1.hi;                                // Newton step, to the second order
    const double d = mid ? 0.0 : -u * (1.0 + 0.5 * u * (f2.hi / f1.hi));
    const dd xr = quick_two_sum(x0, d);
    // P' at the root: Taylor from x0 (P''' from the derivative of the equation)
    const double f3 = (4.0 * x0 * f2.hi - ((double)n * (n + 1.0) - 2.0) * f1.hi) / om.hi;
    const dd fr = f1 + d * f2 + dd{0.5 * d * d * f3, 0.0};
    const dd omr = dd{1.0, 0.0} - xr * xr;
    const dd wr = dd{mid ? 1.0 : 2.0, 0.0} / (omr * (fr * fr));
    x[s] = dd_sel(s < half, xr, dd{0.0, 0.0});
    w[s] = dd_sel(s < half, wr, dd{0.0, 0.0});
}

// P[l][s] = P_l(x_s), l <= lmax (0 past half); one thread per node (0.34 ms at
// lmax 2500, a serial chain, once per rule).
__global__ __launch_bounds__(64) void gl_ptab(int lmax, int half, int SH, const dd* __restrict__ cl,
                                              const dd* __restrict__ x, dd* __restrict__ P)
{
    __shared__ dd sc[GN_CK];
    const int s = blockIdx.x * 64 + threadIdx.x;
    const bool in = s < half;
    const dd zero{0.0, 0.0};
    const dd xs = x[s];
    dd p0{1.0, 0.0}, p1 = xs;
    P[s] = dd_sel(in, p0, zero);
    if (lmax >= 1) P[SH + s] = dd_sel(in, p1, zero);
    for (int l0 = 2; l0 <= lmax; l0 += GN_CK) {
        const int nl = stage_coef(cl, l0, lmax, sc);
#pragma unroll 4
        for (int e = 0; e < nl; ++e) {
            const dd t = xs * p1, p = t + sc[e] * (t - p0);
            p0 = p1;
            p1 = p;
            P[(long)(l0 + e) * SH + s] = dd_sel(in, p, zero);
        }
    }
}

// T[l][a] = (2l + 1) v_l P[l][a] for a < r; 0 for lmin > l and for r <= a <
// ldt.  One workgroup per 32 l (Pc is stored by columns, T by rows), which
// leaves the sum over its l of (2l + 1) |v_l| max_a |P[l][a]| in Sp (if given).
__global__ __launch_bounds__(256) void gl_ttab(const double* __restrict__ Pc, int nlp, int nl, int r, int lmin,
                                               const double* __restrict__ v, int ldt, double* __restrict__ T,
                                               double* __restrict__ Sp)
{
    __shared__ double S[GN_RMAX][33];
    const int l0 = blockIdx.x * 32, tl = threadIdx.x & 31;
    for (int a = threadIdx.x >> 5; a < r; a += 8) S[a][tl] = l0 + tl < nl ? Pc[(long)a * nlp + l0 + tl] : 0.0;
    __syncthreads();
    if (threadIdx.x < 32) {
        double m = 0.0;
        for (int a = 0; a < r; ++a) m = fmax(m, fabs(S[a][tl]));
        const int l = l0 + tl;
        double g = l < nl && l >= lmin ? m * fabs((2.0 * l + 1.0) * v[l]) : 0.0;
        for (int o = 16; o >= 1; o >>= 1) g += __shfl_xor(g, o);
        if (Sp && tl == 0) Sp[blockIdx.x] = g;
    }
    for (int e = threadIdx.x; e < 32 * ldt; e += 256) {
        const int l = l0 + e / ldt, a = e % ldt;
        if (l >= nl) break;
        T[(long)l * ldt + a] = (l < lmin || a >= r) ? 0.0 : S[a][l - l0] * ((2.0 * l + 1.0) * v[l]);
    }
}

// S = sum_l max_a |T[l][a]| from gl_ttab's parts, alike in every lane of every wave:
// no column's sum of |T[l][a] P_l| exceeds it (|P_l| <= 1).
__device__ __forceinline__ double gl_sbound(const double* __restrict__ Sp, int nsp, int lane)
{
    double s = 0.0;
    for (int b = lane; b < nsp; b += 64) s += Sp[b];
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o);
    return s;
}

// Phi[a][k] for CA columns from a0 on at 64 nodes: k = s is +x_s, k = SH + s
// is -x_s.  16 waves: waves 0..7 take the even l, 8..15 the odd ones, l =
// parity + 2 wave' + 16 i, and their sums are added pairwise in LDS in a fixed
// order.  Lane = node; the T row is uniform (scalar loads).  5 FP64 operations
// per (l, node, column): at 2501 l, 1876 nodes, 60 columns 0.081 ms, 0.157
// with the 11 of an error-free running sum.  CA columns share a P load.
// GATE: PhiA[a][k] = sum_l |T[l][a]| P_l(x_k) in FP64 beside them.
constexpr int GN_W = 16;
template <int CA, bool GATE>
__global__ __launch_bounds__(64 * GN_W) void gl_phi(const dd* __restrict__ P, int SH, const double* __restrict__ T,
                                                    int ldt, int nl, int nc, const double* __restrict__ Sp, int nsp,
                                                    dd* __restrict__ Phi, double* __restrict__ PhiA)
{
    __shared__ dd R[GN_W / 2][CA][64];
    __shared__ double RA[GATE ? GN_W : 1][CA][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // block b: node block nb and column group cg with b = 8 (ncg (nb / 8) + cg)
    // + nb % 8, so the column groups of a node block share an XCD (b % 8) and
    // read its slice of P from one L2
    const int ncg = (nc + CA - 1) / CA, q8 = blockIdx.x >> 3;
    const int nb = 8 * (q8 / ncg) + (blockIdx.x & 7), a0 = CA * (q8 % ncg);
    if (64 * nb >= SH) return;
    const int s = 64 * nb + lane;
    const int par = wave >> 3, ww = wave & 7;
    const double B = dd_bias(gl_sbound(Sp, nsp, lane));
    dd acc[CA];
#pragma unroll
    for (int k = 0; k < CA; ++k) acc[k] = dd{B, 0.0};
    double aa[CA] = {};
    const dd* const p = P + s;
#pragma unroll 4
    for (int l = par + 2 * ww; l < nl; l += GN_W) {
        const dd pl = p[(long)l * SH];
        const double* const t = T + (long)l * ldt + a0;
#pragma unroll
        for (int k = 0; k < CA; ++k) {
            dd_bmac(acc[k], t[k], pl);
            if (GATE) aa[k] = __builtin_fma(fabs(t[k]), pl.hi, aa[k]);
        }
    }
    if (GATE)
#pragma unroll
        for (int k = 0; k < CA; ++k) RA[wave][k][lane] = aa[k];
#pragma unroll
    for (int k = 0; k < CA; ++k) acc[k] = dd_unbias(acc[k], B);
    // 8 -> 4 -> 2 -> 1 waves per parity
#pragma unroll
    for (int h = 4; h >= 1; h >>= 1) {
        if (ww >= h && ww < 2 * h)
#pragma unroll
            for (int k = 0; k < CA; ++k) R[par * h + ww - h][k][lane] = acc[k];
        __syncthreads();
        if (ww < h)
#pragma unroll
            for (int k = 0; k < CA; ++k) acc[k] = acc[k] + R[par * h + ww][k][lane];
        __syncthreads();
    }
    if (par == 1 && ww == 0)
#pragma unroll
        for (int k = 0; k < CA; ++k) R[0][k][lane] = acc[k];
    __syncthreads();
    if (wave == 0)
#pragma unroll
        for (int k = 0; k < CA; ++k)
            if (a0 + k < nc) {
                const dd o = R[0][k][lane];
                dd* const out = Phi + (long)(a0 + k) * 2 * SH;
                out[s] = acc[k] + o;
                out[SH + s] = acc[k] - o;
            }
    if (GATE && wave < CA && a0 + wave < nc) {
        double e = 0.0, o = 0.0;
#pragma unroll
        for (int w = 0; w < GN_W / 2; ++w) {
            e += RA[w][wave][lane];
            o += RA[GN_W / 2 + w][wave][lane];
        }
        double* const out = PhiA + (long)(a0 + wave) * 2 * SH;
        out[s] = e + o;
        out[SH + s] = e - o;
    }
}

// Sum the 32 accumulators of a wave over its lanes, halving their number with
// each exchange: lane 2 i (and 2 i + 1) ends with the total of accumulator i.
__device__ __forceinline__ dd wave_totals(dd (&acc)[32], int lane)
{
#pragma unroll
    for (int o = 32, n = 16; n >= 1; o >>= 1, n >>= 1) {
        const bool up = lane & o;
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (i < n) {
                const dd x = acc[i], y = acc[i + n];
                acc[i] = dd_sel(up, y, x) + dd_shfl_xor(dd_sel(up, x, y), o);
            }
    }
    return acc[0] + dd_shfl_xor(acc[0], 1);
}

// H[g][a r + b] = scale sum_k w_k Phi_g Phi_a Phi_b over all K = 2 SH nodes.
// One workgroup per job: a in a tile of four columns ta, two b of tile tb >=
// ta, c in tile tc >= tb (a <= b <= c covers every entry; the entry is written
// at all its orders).  Wave q takes a quarter of the 64-node steps, lane =
// node: per step 10 columns are read for 32 products (6 operations each plus
// the pair products; the reads come from L2): 0.088 ms at 3752 nodes and 59
// columns, 0.120 with 12 operations each.
__device__ __forceinline__ void core_job(int job, int NT, int* ta, int* tb, int* tc, int* h)
{
    int t = 0;
    for (int nj; job >= (nj = 2 * (t + 1) * (NT - t)); ++t) job -= nj;
    *tb = t;
    *h = job & 1;
    job >>= 1;
    *ta = job % (t + 1);
    *tc = t + job / (t + 1);
}

__global__ __launch_bounds__(256, 2) void gl_core_dd(const dd* __restrict__ Phi, int SH, const dd* __restrict__ w,
                                                     int r, double scale, double* __restrict__ H, long ldh,
                                                     const double* __restrict__ Sp, int nsp)
{
    __shared__ dd R[4][32];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, K = 2 * SH;
    const double S = gl_sbound(Sp, nsp, lane);
    if (blockIdx.x == 0 && ldh > (long)r * r)   // H's padding (r^2 odd)
        for (int g = threadIdx.x; g < r; g += 256) H[(long)g * ldh + (long)r * r] = 0.0;
    int ta, tb, tc, h;
    core_job(blockIdx.x, (r + 3) / 4, &ta, &tb, &tc, &h);
    // |Phi| <= S and sum w = 2
    const double B = dd_bias(2.0 * S * S * S);
    dd acc[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) acc[i] = dd{B, 0.0};
    // columns past r repeat the last one (their products are not stored);
    // uniform row bases and one lane offset, the next step's columns loaded
    // before this step's products
    const char *fa[4], *fb[2], *fc[4];
    auto row = [&](int f) { return reinterpret_cast<const char*>(Phi + (size_t)min(f, r - 1) * K); };
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        fa[i] = row(4 * ta + i);
        fc[i] = row(4 * tc + i);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) fb[i] = row(4 * tb + 2 * h + i);
    const char* const wb = reinterpret_cast<const char*>(w);
    struct Step {
        dd a[4], b[2], c[4], w;
    };
    auto load = [&](int k0, Step& S) {
        const unsigned o = (unsigned)(k0 + lane) * (unsigned)sizeof(dd);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            S.a[i] = *reinterpret_cast<const dd*>(fa[i] + o);
            S.c[i] = *reinterpret_cast<const dd*>(fc[i] + o);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) S.b[i] = *reinterpret_cast<const dd*>(fb[i] + o);
        S.w = *reinterpret_cast<const dd*>(wb + (unsigned)((k0 < SH ? k0 : k0 - SH) + lane) * (unsigned)sizeof(dd));
    };
    Step cur, nxt;
    const int kw = __builtin_amdgcn_readfirstlane(64 * wave);
    load(kw < K ? kw : 0, cur);
#pragma unroll 1
    for (int k0 = kw; k0 < K; k0 += 256) {
        load(k0 + 256 < K ? k0 + 256 : k0, nxt);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const dd u = cur.w * cur.b[j];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const dd t = u * cur.a[i];
#pragma unroll
                for (int q = 0; q < 4; ++q) dd_bmac(acc[16 * j + 4 * i + q], t, cur.c[q]);
            }
        }
        cur = nxt;
    }
#pragma unroll
    for (int i = 0; i < 32; ++i) acc[i] = dd_unbias(acc[i], B);
    const dd tot = wave_totals(acc, lane);
    if (!(lane & 1)) R[wave][lane >> 1] = tot;
    __syncthreads();
    if (threadIdx.x < 32) {
        const int e = threadIdx.x;
        const dd t = scale * ((R[0][e] + R[1][e]) + (R[2][e] + R[3][e]));
        const double v = t.hi + t.lo;
        const int b = 4 * tb + 2 * h + (e >> 4), a = 4 * ta + ((e >> 2) & 3), c = 4 * tc + (e & 3);
        if (a <= b && b <= c && c < r) {
            const int o[6][3] = {{a, b, c}, {a, c, b}, {b, a, c}, {b, c, a}, {c, a, b}, {c, b, a}};
#pragma unroll
            for (int p = 0; p < 6; ++p) H[(long)o[p][0] * ldh + (long)o[p][1] * r + o[p][2]] = v;
        }
    }
}

// The gate of every entry a <= b <= c (gl_gate): A = sum_k w_k PhiA_a PhiA_b
// PhiA_c is, but for H's factor, the sum over the allowed multipole triples of
// the magnitudes of the entry's terms; gate[0] is set where margin S^3 exceeds
// it (or either is not a number), and gate[1] = S.  FP64: A cancels as H does,
// and keeps 1e-14 of S^3, a hundredth and less of what it is compared with.
// Jobs as gl_core_dd's; 256 nodes a stage in LDS, 32 threads for four entries (one
// entry to eight threads, with three LDS reads a product, took twice as long).
// On the first call of a setup alone: 3752 nodes and 59 columns 51 us, 1856 and
// 25 12.
__global__ __launch_bounds__(256) void gl_core_gate(const double* __restrict__ PhiA, int SH, const dd* __restrict__ w,
                                                    int r, double margin, const double* __restrict__ Sp, int nsp,
                                                    double* __restrict__ gate)
{
    __shared__ double F[10][256];   // 4 a, 4 c, 2 b with the node's weight
    const int tid = threadIdx.x, K = 2 * SH;
    int ta, tb, tc, h;
    core_job(blockIdx.x, (r + 3) / 4, &ta, &tb, &tc, &h);
    // columns past r repeat the last one (their entries are not looked at)
    const double* row[10];
#pragma unroll
    for (int u = 0; u < 10; ++u) {
        const int f = u < 4 ? 4 * ta + u : u < 8 ? 4 * tc + u - 4 : 4 * tb + 2 * h + u - 8;
        row[u] = PhiA + (long)min(f, r - 1) * K;
    }
    double v[10];
    auto load = [&](int k) {   // node k, of weight 0 past the last
        const double wk = k < K ? w[k < SH ? k : k - SH].hi : 0.0;
        const int kc = min(k, K - 1);
#pragma unroll
        for (int u = 0; u < 10; ++u) v[u] = row[u][kc];
        v[8] *= wk;
        v[9] *= wk;
    };
    const int n = tid & 31, i = (tid >> 5) & 3, q = 2 * (tid >> 7);   // a = i; b = 0, 1; c = q, q + 1
    double t[4] = {0.0, 0.0, 0.0, 0.0};
    load(tid);
    for (int k0 = 0; k0 < K; k0 += 256) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 10; ++u) F[u][tid] = v[u];
        __syncthreads();
        load(k0 + 256 + tid);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const double fa = F[i][32 * u + n], c0 = F[4 + q][32 * u + n], c1 = F[5 + q][32 * u + n];
#pragma unroll
            for (int z = 0; z < 2; ++z) {
                const double p = F[8 + z][32 * u + n] * fa;
                t[2 * z] = __builtin_fma(p, c0, t[2 * z]);
                t[2 * z + 1] = __builtin_fma(p, c1, t[2 * z + 1]);
            }
        }
    }
    const double S = gl_sbound(Sp, nsp, tid & 63);
    if (blockIdx.x == 0 && tid == 0) gate[1] = S;
#pragma unroll
    for (int z = 0; z < 4; ++z) {
        for (int o = 16; o >= 1; o >>= 1) t[z] += __shfl_xor(t[z], o);
        const int a = 4 * ta + i, b = 4 * tb + 2 * h + (z >> 1), c = 4 * tc + q + (z & 1);
        if (n == 0 && a <= b && b <= c && c < r && !(margin * (S * S * S) <= t[z])) gate[0] = 1.0;
    }
}

// The double-double rule of order npt and P_l at its nodes up to lmax, kept by
// the context for the last (npt, lmax): they depend on nothing else.
int gl_table(mcmb_ctx* c, int npt, int lmax)
{
    GlTable& G = c->glt;
    if (G.npt == npt && G.lmax >= lmax) return MCMB_OK;
    G.npt = 0;
    G.half = (npt + 1) / 2;
    G.SH = (G.half + 63) & ~63;   // whole waves of nodes, the padding with weight 0
    const int nc = std::max(npt, lmax) + 1;
    const size_t nx = (size_t)2 * G.SH, np = (size_t)(lmax + 1) * G.SH;
    MCMB_TRY(G.buf.alloc(sizeof(dd) * (nx + nc + np)));
    dd* const x = G.buf.as<dd>();
    dd *const w = x + G.SH, *const cl = w + G.SH, *const P = cl + nc;
    hipLaunchKernelGGL(gl_coef, dim3((nc + 255) / 256), dim3(256), 0, c->stream, nc - 1, cl);
    hipLaunchKernelGGL(gl_rule, dim3(G.SH / 64), dim3(64), 0, c->stream, npt, G.half, G.SH, (const dd*)cl, x, w);
    hipLaunchKernelGGL(gl_ptab, dim3(G.SH / 64), dim3(64), 0, c->stream, lmax, G.half, G.SH, (const dd*)cl,
                       (const dd*)x, P);
    MCMB_HIP(hipGetLastError());
    G.w = w;
    G.P = P;
    G.npt = npt;
    G.lmax = lmax;
    return MCMB_OK;
}

// Whether the node form may take this setup's whole Gram (see the header
// comment; then gl_gate decides).  Up to GN_LMIN the tetrapyd contraction
// stays the default not for its time (a repeated call takes 150 us at lmax 500
// with 10 functions against 82, 184 against 114 with 20, 435 against 335 with
// 30, 101 against 78 at lmax 200 with 10) but for its bits, which are the same
// for all its kernel variants and on which callers of those sizes may rely.
// Above GN_TABMAX the table of P_l would be kept at the expense of the caller's
// memory.
bool gram_nodes_supported(const PointSet& L, int r, int row_lo, int row_hi, bool any_lmax)
{
    if (L.kspace || L.uniform || L.h2mode != MCMB_H2_EXACT || L.kstep != 2) return false;
    if (row_lo != 0 || row_hi != (int)L.rows.size()) return false;
    if (r < 1 || r >= GN_RMAX || (L.lmax <= GN_LMIN && !any_lmax)) return false;
    const size_t half = (3 * (size_t)L.lmax / 2 + 2) / 2 + 64;
    return sizeof(dd) * half * (L.lmax + 1) <= GN_TABMAX;
}

// The gate.  The terms of an entry of H are at most 2 S^3 in sum, S = sum_l max_a
// |T[l][a]| (|P_l| <= 1, sum w = 2), and the roundings of the node form are
// shares of that whatever the entry.  The sums A of gl_core_gate, over the
// magnitudes of the terms that the rules allow, must be at least margin S^3: an
// error of 2^-101 (lmax + 64) 2 S^3 is then within 2^-54 of A, where FP64
// itself rounds.  That error is an estimate with room, no bound: against 113
// bits the entries of six Legendre columns are off by 2^-98.3 of 2 S^3 at most at
// lmax 2500 (2^-99.3 at 600, 2^-98.6 at 6000; the estimate is 2^-89.7, 2^-91.6
// and 2^-88.4), while rests of a biased sum that were all of one sign would grow
// as the square of a wave's terms (dd_bmac), to 2^-83.  The benchmark's
// spectra pass with a factor 140 to spare at lmax 2500 with 59 columns, 3e4 at
// 600 with 19; bins, hat functions, Gaussians of a width of lmax / 20 and bases
// of one parity do not pass.
static double gl_margin(int lmax) { return 0x1p-46 * (lmax + 64.0); }

// After the stream has been waited for.
bool gl_gate(const mcmb_ctx* c)
{
    const double S = c->gn_gate[1], b = 2.0 * S * S * S;
    // (within reach of overflow or of subnormal rests the bias does not hold)
    return c->gn_gate[0] == 0.0 && (S == 0.0 || (b > 1e-250 && b < 1e300));
}

// H (r x ldh) of the exact tetrapyd Gram over the r columns Pc (by columns,
// leading dimension nlp).  phase: called with the name of each part.  gate: the
// sums of gl_gate too.
int gram_nodes_core(mcmb_ctx* c, const PointSet& L, const double* Pc, int nlp, int nl, int r, double* H, long ldh,
                    bool gate, const std::function<int(const char*)>& phase)
{
    const int npt = 3 * L.lmax / 2 + 1;
    if (!(c->glt.npt == npt && c->glt.lmax >= L.lmax)) MCMB_TRY(phase("Legendre table"));
    MCMB_TRY(gl_table(c, npt, L.lmax));
    const GlTable& G = c->glt;
    const int K = 2 * G.SH;
    // columns per thread: four (eight share a P load among more, but leave one
    // workgroup a CU at lmax 2500: 100 us against 81), or two where four give
    // fewer than about one workgroup per CU (lmax 2000, 40 columns, 240
    // workgroups: 38 us with four, 53 with two)
    int ca = 4;
    const int nbx = G.SH / 64;
    while (ca > 2 && nbx * ((r + ca - 1) / ca) < 200) ca >>= 1;
    const int ldt = (r + 7) & ~7;
    const int nsp = (nl + 31) / 32;
    MCMB_TRY(c->gn_ws.alloc(sizeof(dd) * (size_t)r * K +
                            sizeof(double) * ((size_t)nl * ldt + nsp + (gate ? (size_t)r * K : 0))));
    dd* const Phi = c->gn_ws.as<dd>();
    double* const T = reinterpret_cast<double*>(Phi + (size_t)r * K);
    double* const Sp = T + (size_t)nl * ldt;
    double* const PhiA = Sp + nsp;
    if (!c->gn_gate) MCMB_HIP(hipHostMalloc((void**)&c->gn_gate, 2 * sizeof(double), hipHostMallocDefault));
    MCMB_TRY(phase("basis at the nodes"));
    hipLaunchKernelGGL(gl_ttab, dim3((nl + 31) / 32), dim3(256), 0, c->stream, Pc, nlp, nl, r, L.lmin,
                       (const double*)L.d_v.as<double>(), ldt, T, Sp);
    const dim3 grid(8 * ((nbx + 7) / 8) * ((r + ca - 1) / ca)), block(64 * GN_W);
    auto* const phi = ca == 4 ? (gate ? gl_phi<4, true> : gl_phi<4, false>) : (gate ? gl_phi<2, true> : gl_phi<2, false>);
    hipLaunchKernelGGL(phi, grid, block, 0, c->stream, (const dd*)G.P, G.SH, (const double*)T, ldt, nl, r,
                       (const double*)Sp, nsp, Phi, PhiA);
    MCMB_HIP(hipGetLastError());
    MCMB_TRY(phase("node sum"));
    const int NT = (r + 3) / 4;
    int njobs = 0;
    for (int t = 0; t < NT; ++t) njobs += 2 * (t + 1) * (NT - t);
    if (gate) {
        c->gn_gate[0] = 0.0;   // (the stream has been waited for since a kernel last wrote it)
        hipLaunchKernelGGL(gl_core_gate, dim3(njobs), dim3(256), 0, c->stream, (const double*)PhiA, G.SH,
                           (const dd*)G.w, r, gl_margin(L.lmax), (const double*)Sp, nsp, c->gn_gate);
    }
    hipLaunchKernelGGL(gl_core_dd, dim3(njobs), dim3(256), 0, c->stream, (const dd*)Phi, G.SH, (const dd*)G.w, r,
                       3.0 / (4.0 * M_PI), H, ldh, (const double*)Sp, nsp);
    MCMB_HIP(hipGetLastError());
    return MCMB_OK;
}

// ---- the FP64 node sum (mcmb_gamma_gl, mcmb_gamma_gl_pol) over compressed bases ----
//
// The Gauss-Legendre Gram keeps its FP64 nodes and recurrence (its results are
// those of the direct node sum to rounding).  P_l at the nodes x >= 0 depends
// on (npt, lmax) alone and is kept with the context; Phi is then a GEMM on the
// matrix cores instead of a recurrence per column group (lmax 2000, r = 39:
// 0.356 -> 0.035 ms, bound by its loads' latency: 94 workgroups), and the core
// tensor is cx_core's (0.072 -> 0.030 ms with gl_hsum, whose sums over the units
// wait for memory once per 16 of them).

// P[l][s] = P_l(x_s) by the three-term recurrence of the direct node sum, l <=
// lmax; 0 past half.  One thread per node, a serial chain.
__global__ __launch_bounds__(64) void gl_ptab64(int lmax, int half, int SH, const double* __restrict__ x,
                                                double* __restrict__ P)
{
    const int s = blockIdx.x * 64 + threadIdx.x;
    const bool in = s < half;
    const double xs = x[s];
    double p0 = 1.0, p1 = xs;   // P_{l-2}, P_{l-1}
    P[s] = in ? 1.0 : 0.0;
    if (lmax >= 1) P[SH + s] = in ? xs : 0.0;
    for (int l = 2; l <= lmax; ++l) {
        const double pl = ((2.0 * l - 1.0) * xs * p1 - (l - 1.0) * p0) / l;
        p0 = p1;
        p1 = pl;
        P[(long)l * SH + s] = in ? pl : 0.0;
    }
}

// Phi[k / 64][a][k % 64] = sum_l T[l][a] P_l(+-x_s), a < r (k = s: +x_s, SH + s:
// -x_s): one workgroup per 16 nodes, FP64 MFMA with up to four 16-column tiles;
// waves 0..7 take the even l, 8..15 the odd ones, 4 of a parity per step, and
// their sums are added pairwise in LDS in a fixed order.
__global__ __launch_bounds__(1024) void gl_phi64(const double* __restrict__ P, int SH, const double* __restrict__ T,
                                                 int ldt, int nl, int r, double* __restrict__ Phi)
{
    __shared__ d4 R[8][4][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int par = wave >> 3, ww = wave & 7, col = lane & 15, nct = (r + 15) >> 4;
    const double* const p = P + 16 * blockIdx.x + col;
    d4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = d4{0.0, 0.0, 0.0, 0.0};
    for (int l0 = par + 8 * ww; l0 < nl; l0 += 64) {
        const int l = l0 + 2 * (lane >> 4), lc = min(l, nl - 1);
        const double pv = l < nl ? p[(long)lc * SH] : 0.0;
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (t < nct)
                acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(T[(long)lc * ldt + 16 * t + col], pv, acc[t], 0, 0, 0);
    }
#pragma unroll
    for (int h = 4; h >= 1; h >>= 1) {
        if (ww >= h && ww < 2 * h)
#pragma unroll
            for (int t = 0; t < 4; ++t) R[par * h + ww - h][t][lane] = acc[t];
        __syncthreads();
        if (ww < h)
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] += R[par * h + ww][t][lane];
        __syncthreads();
    }
    if (par == 1 && ww == 0)
#pragma unroll
        for (int t = 0; t < 4; ++t) R[0][t][lane] = acc[t];
    __syncthreads();
    if (wave == 0) {
        const int s = 16 * blockIdx.x + col, km = SH + s;
        double* const fp = Phi + (long)(s >> 6) * r * 64 + (s & 63);
        double* const fm = Phi + (long)(km >> 6) * r * 64 + (km & 63);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const d4 o = R[0][t][lane];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int a = 16 * t + 4 * v + (lane >> 4);
                if (a < r) {
                    fp[64 * a] = acc[t][v] + o[v];
                    fm[64 * a] = acc[t][v] - o[v];
                }
            }
        }
    }
}

// The core H from the units' tile tensors (cx_core), added in order: H[g][a r
// + b] of one field, or H[b][g rP + a] with (a, b) of the pair's field.
template <bool SAME>
__global__ __launch_bounds__(64) void gl_hsum(const double* __restrict__ Hu, long us, int nu, int rP, int rS,
                                               double scale, double* __restrict__ H, long ldh)
{
    __shared__ long base[8];
    const int NTC = (rS + 15) >> 4, NTB = (rP + 15) >> 4;
    if (threadIdx.x < NTB) base[threadIdx.x] = cx_base(threadIdx.x, NTC, SAME);
    __syncthreads();
    const long e = (long)blockIdx.x * 64 + threadIdx.x;
    if (e >= (long)rP * ldh) return;
    const int x = (int)(e / ldh), rem = (int)(e % ldh), y = rem / rP, z = rem % rP;
    if (rem >= (SAME ? rP : rS) * rP) {
        H[e] = 0.0;
        return;
    }
    int a, b, c;
    if (SAME) {
        a = min(x, min(y, z));
        c = max(x, max(y, z));
        b = x + y + z - a - c;
    } else {
        a = min(x, z);
        b = max(x, z);
        c = y;
    }
    const double* const h = Hu + cx_tile(base[b >> 4], a >> 4, b, c >> 4, NTC, SAME) * 256 + 16 * (a & 15) + (c & 15);
    double t = 0.0;
    for (int u0 = 0; u0 < nu; u0 += 16) {   // 16 loads in flight, added in order
        double v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] = u0 + k < nu ? h[(long)(u0 + k) * us] : 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) t += v[k];
    }
    H[e] = scale * t;
}

// The FP64 rule's nodes x >= 0 and weights (the middle node of an odd rule
// with half its weight, at +x and -x), and P_l at the nodes up to lmax.
int gl_half_table(mcmb_ctx* c, int npt, int lmax, const double* x, const double* w)
{
    GlHalf& G = c->glh;
    if (G.npt == npt && G.lmax >= lmax) return MCMB_OK;
    G.npt = 0;
    const int half = (npt + 1) / 2, SH = (half + 63) & ~63;
    MCMB_TRY(G.buf.alloc(sizeof(double) * ((size_t)3 * SH + (size_t)(lmax + 1) * SH)));
    std::vector<double> h((size_t)3 * SH, 0.0);
    for (int s = 0; s < half; ++s) {
        const int i = npt / 2 + s;
        h[s] = x[i];
        h[SH + s] = h[2 * SH + s] = (npt & 1) && s == 0 ? 0.5 * w[i] : w[i];
    }
    double* const d = G.buf.as<double>();
    MCMB_HIP(hipMemcpyAsync(d, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL(gl_ptab64, dim3(SH / 64), dim3(64), 0, c->stream, lmax, half, SH, (const double*)d, d + 3 * SH);
    MCMB_HIP(hipGetLastError());
    MCMB_HIP(hipStreamSynchronize(c->stream));   // h
    G.w = d + SH;
    G.P = d + 3 * SH;
    G.SH = SH;
    G.npt = npt;
    G.lmax = lmax;
    return MCMB_OK;
}

// Doubles of T and of Phi for r columns over nl multipoles.
static int gl_ldt(int r) { return std::max(16 * ((r + 15) / 16), (r + 8) & ~7); }
size_t gl_phi64_size(const mcmb_ctx* c, int nl, int r) { return (size_t)nl * gl_ldt(r) + (size_t)2 * c->glh.SH * r; }

// Phi of r compressed columns Pc (by columns) with per-leg weight v into the
// second part of ws (gl_phi64_size doubles); *phi points there.
int gl_phi64_launch(mcmb_ctx* c, const double* Pc, int nlp, int nl, int r, int lmin, const double* v, double* ws,
                    double** phi)
{
    const GlHalf& G = c->glh;
    const int ldt = gl_ldt(r);
    *phi = ws + (size_t)nl * ldt;
    hipLaunchKernelGGL(gl_ttab, dim3((nl + 31) / 32), dim3(256), 0, c->stream, Pc, nlp, nl, r, lmin, v, ldt, ws,
                       (double*)nullptr);
    hipLaunchKernelGGL(gl_phi64, dim3(G.SH / 16), dim3(1024), 0, c->stream, (const double*)G.P, G.SH, (const double*)ws,
                       ldt, nl, r, *phi);
    MCMB_HIP(hipGetLastError());
    return MCMB_OK;
}

// Units of the core: chunks of 64 nodes, grouped to about 512 workgroups.
static void gl_units(const mcmb_ctx* c, int rP, int rS, bool same, long* jobs, int* g, int* ng, long* us)
{
    const int NTB = (rP + 15) / 16, NTC = (rS + 15) / 16, nch = 2 * c->glh.SH / 64;
    *jobs = 0;
    for (int t = 0; t < NTB; ++t) *jobs += cx_jobs(t, NTC, same);
    const int want = (int)std::min<long>(nch, (511 + *jobs) / *jobs);
    *g = (nch + want - 1) / want;
    *ng = (nch + *g - 1) / *g;
    *us = cx_base(NTB, NTC, same) * 256;
}
size_t gl_core64_size(const mcmb_ctx* c, int rP, int rS, bool same)
{
    long jobs, us;
    int g, ng;
    gl_units(c, rP, rS, same, &jobs, &g, &ng, &us);
    return (size_t)ng * us;
}

// H (rP x ldh) = scale sum_k w_k Phi Phi Phi from phP (and phS unless it is the
// same field); ws: gl_core64_size doubles.
int gl_core64_launch(mcmb_ctx* c, const double* phP, int rP, const double* phS, int rS, double scale, double* ws,
                     double* H, long ldh)
{
    const bool same = phP == phS;
    long jobs, us;
    int g, ng;
    gl_units(c, rP, rS, same, &jobs, &g, &ng, &us);
    const int nch = 2 * c->glh.SH / 64;
    const dim3 grid((unsigned)jobs, ng), hgrid((unsigned)(((long)rP * ldh + 63) / 64));
#define GL_CORE64(SAME)                                                                                          \
    do {                                                                                                         \
        hipLaunchKernelGGL(cx_core<SAME>, grid, dim3(256), 0, c->stream, phP, rP, phS, rS, 64,                   \
                           (const double*)c->glh.w, 64l, (const double*)nullptr, 0, ng, g, nch, 0, ws, us);      \
        hipLaunchKernelGGL(gl_hsum<SAME>, hgrid, dim3(64), 0, c->stream, (const double*)ws, us, ng, rP, rS, scale, H, \
                           ldh);                                                                                 \
    } while (0)
    if (same) GL_CORE64(true);
    else GL_CORE64(false);
#undef GL_CORE64
    MCMB_HIP(hipGetLastError());
    return MCMB_OK;
}

}  // namespace mcmb
