// syev.hip -- eigen-decomposition of a symmetric positive semi-definite
// Gram matrix (c <= 128) for the Gram route of the right-to-left truncation
// step: G = U diag(sigma^2) U^T.
//
// The step needs the left singular vectors and values of a bond matrix M
// from its Gram G = M M^T.  A one-sided Jacobi SVD of a Cholesky factor of
// G performs about 8 sweeps x 127 rounds of pair rotations (~100 MFLOP at
// c = 128) on one CU; this solver does ~7 MFLOP:
//   1. k_sytrd: Householder tridiagonalisation G = Q T Q^T, one workgroup,
//      G held in registers (two lanes per row), one reflector per step with
//      two workgroup barriers;
//   2. k_stedc: Cuppen's divide and conquer on T (split into 1 x 1 blocks,
//      merged bottom-up by rank-one updates), with the deflation rules of
//      Dongarra and Sorensen, the secular-equation iteration of Li's "middle
//      way" (SIAM J. Sci. Comput. 1994, as in LAPACK's dlaed4) from the
//      nearer pole, and the eigenvectors of Gu and Eisenstat (SIAM J. Matrix
//      Anal. Appl. 16, 1995): z is recomputed from the computed roots, which
//      makes the vectors numerically orthogonal without reorthogonalisation;
//   3. k_ormtr: Q applied to the eigenvectors of T below the top merge, one
//      wave per column, the reflectors staged in LDS;
//   4. the top merge's product (W times the rank-one eigenvector matrix,
//      padded with the identity for deflated columns) on the MFMA GEMM.
// G is scaled by an even power of two so that its largest entry is O(1)
// (bond matrices of deep trains reach 1e-60 and below); sigma is scaled back.
// Eigenvectors of the Gram carry the Gram's rounding (~ c u ||G||), as the
// Cholesky route does; callers decide whether that resolution suffices.
#include "common.hpp"

#include <cmath>
#include <type_traits>

using namespace ptt;

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr double EPSU = 0x1.0p-53;
constexpr int EIG_NMAX = 128;

__device__ __forceinline__ double quad_prod(double x) {
    x *= dppd<0xB1>(x);
    x *= dppd<0x4E>(x);
    return x;
}
// Sum / product over each aligned group of 8 lanes (quad, then half-row mirror).
__device__ __forceinline__ double oct_sum(double x) {
    x = quad_sum(x);
    x += dppd<0x141>(x);
    return x;
}
__device__ __forceinline__ double oct_prod(double x) {
    x = quad_prod(x);
    x *= dppd<0x141>(x);
    return x;
}
// Sum / product over aligned groups of L = 1, 2, 4 or 8 lanes.
template <int L>
__device__ __forceinline__ double grp_sum(double x) {
    if constexpr (L == 2) x += dppd<0xB1>(x);
    if constexpr (L == 4) x = quad_sum(x);
    if constexpr (L == 8) x = oct_sum(x);
    return x;
}
template <int L>
__device__ __forceinline__ double grp_prod(double x) {
    if constexpr (L == 2) x *= dppd<0xB1>(x);
    if constexpr (L == 4) x = quad_prod(x);
    if constexpr (L == 8) x = oct_prod(x);
    return x;
}
__device__ __forceinline__ double wave_max(double x) {
    for (int o = 32; o > 0; o >>= 1) x = fmax(x, __shfl_xor(x, o));
    return x;
}
// 1/x from the hardware reciprocal and two Newton steps (a few ulp; x != 0).
__device__ __forceinline__ double rcp_nr(double x) {
    double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    e = fma(-x, r, 1.0);
    return fma(r, e, r);
}
__device__ __forceinline__ double uniform_d(double x) {
    const int lo = __builtin_amdgcn_readfirstlane(__double2loint(x));
    const int hi = __builtin_amdgcn_readfirstlane(__double2hiint(x));
    return __hiloint2double(hi, lo);
}

// Workgroup barrier that orders LDS traffic only: outstanding global stores
// (the reflectors written as they are formed) do not hold the barrier.
__device__ __forceinline__ void lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Inclusive suffix sum over the 64 lanes of a wave: x_lane + ... + x_63.
__device__ __forceinline__ double suffix_sum(double x) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double y = __shfl_down(x, o);
        if (lane + o < 64) x += y;
    }
    return x;
}

// Largest even e with 2^e <= a (a > 0, finite); 0 otherwise.
__device__ __forceinline__ int even_exp(double a) {
    if (!(a > 0.0) || !(a < INFINITY)) return 0;
    int e = ilogb(a);
    return (e >= 0) ? (e / 2) * 2 : -(((-e) + 1) / 2) * 2;
}

// ---- 1. tridiagonalisation ------------------------------------------------
// Register tiles: G is cut into 16 x 16 tiles; row wave I (NB = NMAX/16 of
// them) holds tile row I.  Lane l (a = l/16, j = l%16) holds rows
// 16I + a + 4v (v = 0..3) of column 16J + j of every tile J: g[J][v].
// Entries beyond n are zero and stay zero.  A lane thus needs only the NB
// entries of v (and of p) at its columns and four at its rows, which keeps
// the LDS traffic of a step at a few KB.
//
// Step k applies the reflector H_k = I - tau v v^T (v_{k+1} = 1, LAPACK
// dlarfg convention beta = -sign(x0) ||x||) built from column k below the
// diagonal: p = tau G v, K = tau/2 p^T v and G <- G - v p^T - (p - 2K v) v^T,
// per element g -= v_r p_c + v_c (p_r - 2K v_r).  The row sums of G v are
// reduced over the 16 lanes of a DPP row by a reduce-scatter (each lane ends
// with one of its four rows); K is formed by every row wave from p and v.
//
// One more wave (the reflector wave) forms the reflectors.  It holds the
// next row, k+1, two entries per lane: the lanes that own that row copied it
// to LDS one step earlier, after their own update.  Once p is complete it
// applies step k's update to that row, reduces it across the wave and writes
// v_{k+1} to LDS, while the row waves update their tiles and the
// owner of row k+2 copies its row out.  A step is thus the product G v on
// the row waves, a barrier, the reflector wave's short chain (beside the
// row waves' update) and a barrier.  Row waves whose rows all lie at or
// before k hold nothing later steps read and skip the products.
//
// Outputs: d (diagonal), e (off-diagonal), tau, the reflectors in the
// columns of Vh (n x n, ld n; rows <= k zero, v_{k+1} = 1), the exponent of
// the power-of-two scaling, max |G| (dinfo[6]) and the trace of G (dinfo[7]).
// Only the upper triangle of G is read.
__device__ __forceinline__ double readlane_d(double v, int l) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double sel(bool c, double x, double y) { return c ? x : y; }

template <int NMAX>
__global__ __launch_bounds__(NMAX * 4 + 64) void k_sytrd(int n, const double *__restrict__ G,
                                                         long ldg, double *__restrict__ Vh,
                                                         double *__restrict__ tau_out,
                                                         double *__restrict__ d_out,
                                                         double *__restrict__ e_out,
                                                         int *__restrict__ eexp,
                                                         double *__restrict__ dinfo) {
    constexpr int NB = NMAX / 16, NTM = 64 * NB, NT = NTM + 64, NW = NT / 64;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const bool star = (tid >= NTM);  // the reflector wave
    const int I = wv, ga = lane >> 4, gj = lane & 15;
    __shared__ double vb[2][NMAX];    // v of the current / next step
    __shared__ double pp[NMAX];       // p
    __shared__ double rowb[2][NMAX];  // the next rows, for the reflector wave
    __shared__ double tkb[2];
    __shared__ double sd[NMAX], se[NMAX], st[NMAX];
    __shared__ double s_max[NW], s_tr[NW];
    __shared__ int s_e;

    double g[NB][4];
    double amax = 0.0, tr = 0.0;
#pragma unroll
    for (int J = 0; J < NB; J++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = 16 * I + ga + 4 * v, col = 16 * J + gj;
            double x = 0.0;
            if (!star && row < n && col < n)
                x = (row <= col) ? G[row + (long)col * ldg] : G[col + (long)row * ldg];
            g[J][v] = x;
            amax = fmax(amax, fabs(x));
            if (row == col) tr += x;
        }
    amax = wave_max(amax);
    tr = wave_sum(tr);
    if (lane == 0) {
        s_max[wv] = amax;
        s_tr[wv] = tr;
    }
    __syncthreads();
    if (tid == 0) {
        double m = 0.0, t = 0.0;
        for (int w = 0; w < NW; w++) {
            m = fmax(m, s_max[w]);
            t += s_tr[w];
        }
        s_e = even_exp(m);
        dinfo[6] = m;
        dinfo[7] = t;
        *eexp = s_e;
    }
    __syncthreads();
    const int es = s_e;
#pragma unroll
    for (int J = 0; J < NB; J++)
#pragma unroll
        for (int v = 0; v < 4; v++) g[J][v] = ldexp(g[J][v], -es);

    // Row i of this wave's tile row into rowb[slot] (called by the whole
    // wave; i wave-uniform, held by the lanes with a = i % 4 in register
    // v = (i % 16) / 4).
    auto copy_row = [&](int i, int slot) {
        const int v = (i & 15) >> 2;
        if (ga == (i & 3)) {
            // g[J][v] by a 0/1 mask (exact: one term is nonzero), so every
            // register index stays constant and g stays in registers
            const double m0 = (v == 0) ? 1.0 : 0.0, m1 = (v == 1) ? 1.0 : 0.0;
            const double m2 = (v == 2) ? 1.0 : 0.0, m3 = (v == 3) ? 1.0 : 0.0;
#pragma unroll
            for (int J = 0; J < NB; J++)
                rowb[slot][16 * J + gj] =
                    fma(g[J][3], m3, fma(g[J][2], m2, fma(g[J][1], m1, g[J][0] * m0)));
        }
    };
    // The reflector wave turns row p (entries a0 = row[lane], a1 =
    // row[lane + 64]) into the reflector for step p, from column p below the
    // diagonal: v into vb[slot], tau, d_p, e_p = beta (the row waves copy v
    // to Vh at the start of step p).
    // x0 = row[p+1] and dp = row[p] arrive as wave-uniform values (formed by
    // every lane with the owner lane's arithmetic, so no lane reads).
    auto reflector = [&](int p, int slot, double a0, double a1, double x0, double dp) {
        const int i0 = lane, i1 = lane + 64;
        double s2 = (i0 >= p + 2 ? a0 * a0 : 0.0) + (i1 >= p + 2 && i1 < NMAX ? a1 * a1 : 0.0);
        s2 = wave_sum(s2);
        double beta, tk, scl;
        if (s2 == 0.0) {
            beta = x0;
            tk = 0.0;
            scl = 0.0;
        } else {
            beta = -copysign(sqrt(x0 * x0 + s2), x0);
            tk = (beta - x0) * rcp_nr(beta);
            scl = rcp_nr(x0 - beta);
        }
        const double w0 = (i0 == p + 1) ? 1.0 : (i0 > p + 1 ? a0 * scl : 0.0);
        const double w1 = (i1 == p + 1) ? 1.0 : (i1 > p + 1 ? a1 * scl : 0.0);
        if (i0 < NMAX) vb[slot][i0] = w0;
        if (i1 < NMAX) vb[slot][i1] = w1;
        if (lane == 0) {
            tkb[slot] = tk;
            sd[p] = dp;
            se[p] = beta;
            st[p] = tk;
        }
    };
    // entries of an LDS row vector at columns lane and lane + 64
    auto lrow = [&](const double *v, double &x0, double &x1) {
        x0 = v[lane];
        x1 = (lane + 64 < NMAX) ? v[lane + 64 < NMAX ? lane + 64 : 0] : 0.0;
    };

    if (!star && I == 0) {
        copy_row(0, 1);
        copy_row(1, 0);
    }
    lds_sync();
    if (star) {
        double a0, a1;
        lrow(rowb[1], a0, a1);
        reflector(0, 0, a0, a1, rowb[1][1 < NMAX ? 1 : 0], rowb[1][0]);
    }
    lds_sync();

    for (int k = 0; k + 2 < n; k++) {
        const double *vk = vb[k & 1];
        const double tk = tkb[k & 1];
        if (!star) {
            for (int i = tid; i < n; i += NTM) Vh[i + (long)k * n] = vk[i];
            const bool act = (16 * I + 15 > k);
            if (tk != 0.0) {
                double vJ[NB];
                if (act) {
                    double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int J = 0; J < NB; J++) {
                        vJ[J] = vk[16 * J + gj];
#pragma unroll
                        for (int v = 0; v < 4; v++) acc[v] = fma(g[J][v], vJ[J], acc[v]);
                    }
                    // reduce-scatter over the 16 lanes of the row: lane j
                    // ends with the sum for v = 2 (j / 8 % 2) + (j / 4 % 2)
                    const bool h8 = (gj & 8) != 0, h4 = (gj & 4) != 0;
                    const double k0 = sel(h8, acc[2], acc[0]), k1 = sel(h8, acc[3], acc[1]);
                    const double s0 = sel(h8, acc[0], acc[2]), s1 = sel(h8, acc[1], acc[3]);
                    const double u0 = k0 + dppd<0x128>(s0);  // row_ror:8
                    const double u1 = k1 + dppd<0x128>(s1);
                    const double kk2 = sel(h4, u1, u0), ss2 = sel(h4, u0, u1);
                    double x = kk2 + dppd<0x141>(ss2);  // half-row mirror: 4-lane groups swap
                    x = quad_sum(x);
                    if ((gj & 3) == 0) {
                        const int vi = 2 * (int)h8 + (int)h4;
                        pp[16 * I + ga + 4 * vi] = tk * x;
                    }
                }
                lds_sync();
                if (act) {
                    double pJ[NB];
                    double dot = 0.0;
#pragma unroll
                    for (int J = 0; J < NB; J++) {
                        pJ[J] = pp[16 * J + gj];
                        dot = fma(pJ[J], vJ[J], dot);
                    }
                    // p^T v over the 16 columns j of the row (each DPP row
                    // forms the same sum)
                    dot = quad_sum(dot);
                    dot += dppd<0x141>(dot);
                    dot += dppd<0x140>(dot);
                    const double kk = 0.5 * tk * dot;
                    double vr[4], wr[4];
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const int row = 16 * I + ga + 4 * v;
                        vr[v] = vk[row];
                        wr[v] = pp[row] - 2.0 * kk * vr[v];
                    }
#pragma unroll
                    for (int J = 0; J < NB; J++)
#pragma unroll
                        for (int v = 0; v < 4; v++)
                            g[J][v] = fma(-vr[v], pJ[J], fma(-vJ[J], wr[v], g[J][v]));
                }
            }
            // row k+2 (now updated through step k) for the reflector wave
            if (I == (k + 2) >> 4) copy_row(k + 2, (k + 1) & 1);
        } else {
            // row k+1, updated through step k-1 (copied before the last barrier),
            // and its entries k+1 (the diagonal) and k+2 as uniform values
            const int k1 = k + 1, k2 = (k + 2 < NMAX) ? k + 2 : k + 1;
            const double *rk = rowb[k & 1];
            double a0, a1;
            lrow(rk, a0, a1);
            double dp = rk[k1];
            double x0 = (k + 2 < NMAX) ? rk[k2] : 0.0;
            if (tk != 0.0) {
                double v0, v1;
                lrow(vk, v0, v1);
                const double vx = vk[k2];
                lds_sync();
                double p0, p1;
                lrow(pp, p0, p1);
                const double pk = pp[k1], px = pp[k2];
                const double kk = 0.5 * tk * wave_sum(fma(p0, v0, p1 * v1));
                const double w = pk - 2.0 * kk;  // v_{k+1} = 1
                a0 = fma(-1.0, p0, fma(-v0, w, a0));
                a1 = fma(-1.0, p1, fma(-v1, w, a1));
                // the owner lanes' arithmetic for entries k+1 and k+2
                dp = fma(-1.0, pk, fma(-1.0, w, dp));
                if (k + 2 < NMAX) x0 = fma(-1.0, px, fma(-vx, w, x0));
            }
            reflector(k1, k1 & 1, a0, a1, x0, dp);
        }
        lds_sync();
    }
    // the last diagonal entry: row n-1, updated through step n-3
    if (star && n >= 2 && lane == 0) sd[n - 1] = rowb[(n - 2) & 1][n - 1];
    lds_sync();
    for (int i = tid; i < n; i += NT) {
        d_out[i] = sd[i];
        e_out[i] = (i + 1 < n) ? se[i] : 0.0;
        tau_out[i] = (i + 2 < n) ? st[i] : 0.0;
    }
}

// ---- 2. divide and conquer on the tridiagonal -----------------------------
// Blocks of size s = 2, 4, ... are merged bottom-up; block [lo, hi) splits
// at m = lo + s/2 with coupling beta = e[m-1]:
//   T = diag(T1 - |beta| e_last e_last^T, T2 - |beta| e_1 e_1^T) + |beta| v v^T,
//   v = [e_last; sign(beta) e_1],
// so the 1 x 1 leaves start from d_i - |e_{i-1}| - |e_i|.  The eigenvectors of
// the blocks live in the block-diagonal Z (global, n x n, ld n); the
// eigenvalues in sD.  At a merge z = [last row of Z1; sign * first row of
// Z2] / sqrt(2) and rho = 2 |beta|.
//
// Deflation (one wave per block): entries with rho |z| <= tol are deflated;
// consecutive remaining entries whose poles are closer than the tolerance
// allows (|t c s| <= tol for the rotation that zeroes one z) are combined by
// that rotation.  When no such pair exists -- the common case -- the
// non-deflated list is formed by ballots; otherwise one lane walks the block
// in order.  Secular-equation roots: eight lanes per root.  Lower merges stage
// the block's columns in LDS and form Z[:, nd] * U in registers.
//
// The top merge stops after the rank-one eigenvector matrix and leaves Z
// as the lower merges left it: column c of Um (n x n, ld n) is the update's
// eigenvector c (non-deflated first, then the deflated unit vectors) with
// its rows in the order of Z's columns, and the top merge's deflating
// rotations of Z's column pairs are applied to Um's rows instead (last
// first), so U = (Q Z) Um.  Also written: sigma (descending, scaled back),
// colidx (descending rank -> U column), numrank, rho, and colmap (U column
// c's pole: Z column colmap[c]).
//
// part 0 runs every merge; part 1 the merges below the top one, then saves
// the poles and the iteration count in dsave (n + 1 doubles) and exits;
// part 2 the top merge and the decisions from that state.  Between the two
// launches Z is final, so the back transformation Q Z can run beside part 2.
//
// Threads: NT = 8 NMAX.  Dynamic LDS: NMAX * NMAX doubles (the lower merges'
// eigenvector matrices in the first half, the staged columns in the second;
// the top merge's Um).
template <int NMAX>
__global__ __launch_bounds__(8 * NMAX) void k_stedc(
    int n, const double *__restrict__ dd, const double *__restrict__ ee,
    const int *__restrict__ eexp, double *__restrict__ Z, double *__restrict__ Um,
    int *__restrict__ colmap, int *__restrict__ colidx, double *__restrict__ sig,
    int *__restrict__ iout, double *__restrict__ dinfo, double delta, int cap, double budget,
    int part, double *__restrict__ dsave) {
    constexpr int NT = 8 * NMAX;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    extern __shared__ __align__(16) double lds[];
    double *ums = lds;                            // NMAX * NMAX / 2
    double *zs = lds + (NMAX * NMAX) / 2;         // NMAX * NMAX / 2
    __shared__ double sD[NMAX], sz[NMAX], sdl[NMAX], szl[NMAX], stau[NMAX], szh[NMAX],
        sinv[NMAX], rc[NMAX], rs[NMAX], srho[NMAX], slam[NMAX];
    __shared__ int sperm[NMAX], snd[NMAX], sorg[NMAX], ra[NMAX], rb[NMAX], sKn[NMAX],
        sNrot[NMAX], sflag[NMAX], spos[NMAX], scm[NMAX];
    __shared__ int s_iters;

    if (part == 2) {
        // the state part 1 left: poles, iteration count; Z in place
        for (int i = tid; i < n; i += NT) sD[i] = dsave[i];
        if (tid == 0) s_iters = (int)dsave[n];
    } else {
        if (tid == 0) s_iters = 0;
        for (int i = tid; i < n; i += NT) {
            double di = dd[i];
            if (i > 0) di -= fabs(ee[i - 1]);
            if (i + 1 < n) di -= fabs(ee[i]);
            sD[i] = di;
        }
        for (int j = tid / NMAX; j < n; j += NT / NMAX)
            for (int i = tid % NMAX; i < n; i += NMAX) Z[i + (long)j * n] = (i == j) ? 1.0 : 0.0;
    }
    __syncthreads();

    bool top_done = false;
    int s0 = 2;
    if (part == 2)
        while (s0 < n) s0 *= 2;
    for (int s = s0; s / 2 < n; s *= 2) {
        const bool top = (s >= n);
        if (part == 1 && top) break;
        const int ls = __builtin_ctz(s);  // all index arithmetic by shifts
        const int nblk = (n + s - 1) >> ls;
        // A: z and the ascending order of the eigenvalues of each block, the
        // rank of entry j counted by eight lanes (ties by index)
        {
            const int j = tid >> 3, sub = tid & 7;
            const int b = j >> ls, lo = b << ls, hi = min(lo + s, n), m = lo + s / 2;
            if (j < n && m < hi) {
                if (sub == 0) {
                    const double bt = ee[m - 1];
                    const double sg = (bt >= 0.0) ? 1.0 : -1.0;
                    sz[j] = (j < m ? Z[(m - 1) + (long)j * n] : sg * Z[m + (long)j * n]) * M_SQRT1_2;
                }
                const double dj = sD[j];
                int pos = 0;
                for (int q = lo + sub; q < hi; q += 8) {
                    const double dq = sD[q];
                    pos += (dq < dj) || (dq == dj && q < j);
                }
                pos = (int)oct_sum((double)pos);
                if (sub == 0) sperm[lo + pos] = j;
            }
        }
        __syncthreads();
        // B: deflation, a group of GL = min(s, 64) lanes per block (each lane
        // one or two sorted positions)
        {
            const int GL = s < 64 ? s : 64;
            const int gl = tid & (GL - 1);
            const int gbase = lane - gl;
            const unsigned long long gmask = (GL == 64) ? ~0ULL : (((1ULL << GL) - 1) << gbase);
            const int lgl = __builtin_ctz(GL);
            for (int b = tid >> lgl; b < nblk; b += NT >> lgl) {
                const int lo = b << ls, hi = min(lo + s, n), m = lo + s / 2, K = hi - lo;
                if (m >= hi) {
                    if (gl == 0) sKn[b] = -1;
                    continue;
                }
                const double rho = 2.0 * fabs(ee[m - 1]);
                if (rho == 0.0) {
                    if (gl == 0) {
                        srho[b] = rho;
                        sKn[b] = 0;
                        sNrot[b] = 0;
                    }
                    continue;
                }
                // sorted positions q0 = gl, q1 = gl + 64 (only when s = 128)
                const int q0 = gl, q1 = gl + 64;
                const int j0 = (q0 < K) ? sperm[lo + q0] : -1;
                const int j1 = (s > 64 && q1 < K) ? sperm[lo + q1] : -1;
                const double z0 = j0 >= 0 ? sz[j0] : 0.0, z1 = j1 >= 0 ? sz[j1] : 0.0;
                const double d0 = j0 >= 0 ? sD[j0] : 0.0, d1 = j1 >= 0 ? sD[j1] : 0.0;
                double dmax = fmax(fabs(d0), fabs(d1)), zmax = fmax(fabs(z0), fabs(z1));
                for (int o = 1; o < GL; o <<= 1) {
                    dmax = fmax(dmax, __shfl_xor(dmax, o, GL));
                    zmax = fmax(zmax, __shfl_xor(zmax, o, GL));
                }
                const double tol = 8.0 * EPSU * fmax(dmax, zmax);
                const bool k0 = j0 >= 0 && !(rho * fabs(z0) <= tol);
                const bool k1 = j1 >= 0 && !(rho * fabs(z1) <= tol);
                // kept positions of the group, bit = sorted position
                const unsigned long long m0 = (__ballot(k0) & gmask) >> gbase;
                const unsigned long long m1 = (__ballot(k1) & gmask) >> gbase;
                const unsigned long long below = (gl == 0) ? 0ULL : ((~0ULL) >> (64 - gl));
                bool close = false;
                if (k0) {
                    const unsigned long long mm = m0 & below;
                    if (mm) {
                        const int jp = sperm[lo + 63 - __clzll(mm)];
                        const double zp = sz[jp], t = d0 - sD[jp];
                        close = fabs(t * z0 * zp) <= tol * (z0 * z0 + zp * zp);
                    }
                }
                if (k1) {
                    const unsigned long long mm = m1 & below;
                    const int p = mm ? 64 + 63 - __clzll(mm) : (m0 ? 63 - __clzll(m0) : -1);
                    if (p >= 0) {
                        const int jp = sperm[lo + p];
                        const double zp = sz[jp], t = d1 - sD[jp];
                        close = close || (fabs(t * z1 * zp) <= tol * (z1 * z1 + zp * zp));
                    }
                }
                if ((__ballot(close) & gmask) == 0ULL) {
                    const int c0 = __popcll(m0);
                    if (k0) {
                        const int pos = __popcll(m0 & below);
                        snd[lo + pos] = j0;
                        sdl[lo + pos] = d0;
                        szl[lo + pos] = z0;
                    }
                    if (k1) {
                        const int pos = c0 + __popcll(m1 & below);
                        snd[lo + pos] = j1;
                        sdl[lo + pos] = d1;
                        szl[lo + pos] = z1;
                    }
                    if (gl == 0) {
                        srho[b] = rho;
                        sKn[b] = c0 + __popcll(m1);
                        sNrot[b] = 0;
                    }
                } else if (gl == 0) {
                    // one lane walks the sorted entries; the pending entry's
                    // (z, d) are carried in registers and the next entry is
                    // loaded while the current one is decided (entries not
                    // reached yet are never written, so the early loads hold)
                    int Kn = 0, nrot = 0, prev = -1;
                    double zp = 0.0, dp = 0.0;
                    int jn = sperm[lo];
                    double zn = sz[jn], dn = sD[jn];
                    for (int qq = lo; qq < hi; qq++) {
                        const int j = jn;
                        const double zj = zn, dj = dn;
                        if (qq + 1 < hi) {
                            jn = sperm[qq + 1];
                            zn = sz[jn];
                            dn = sD[jn];
                        }
                        if (rho * fabs(zj) <= tol) continue;
                        if (prev < 0) {
                            prev = j;
                            zp = zj;
                            dp = dj;
                            continue;
                        }
                        const double t = dj - dp;
                        const double t2 = zj * zj + zp * zp;
                        // |t c s| <= tol with c = zj/tau, s = -zp/tau, tau^2 = t2
                        if (fabs(t * zj * zp) <= tol * t2) {
                            const double ta = sqrt(t2);
                            const double c = zj / ta, sn = -zp / ta;
                            sz[prev] = 0.0;
                            sD[prev] = dp * c * c + dj * sn * sn;
                            ra[lo + nrot] = prev;
                            rb[lo + nrot] = j;
                            rc[lo + nrot] = c;
                            rs[lo + nrot] = sn;
                            nrot++;
                            prev = j;
                            zp = ta;
                            dp = dp * sn * sn + dj * c * c;
                        } else {
                            sz[prev] = zp;
                            sD[prev] = dp;
                            snd[lo + Kn] = prev;
                            sdl[lo + Kn] = dp;
                            szl[lo + Kn] = zp;
                            Kn++;
                            prev = j;
                            zp = zj;
                            dp = dj;
                        }
                    }
                    if (prev >= 0) {
                        sz[prev] = zp;
                        sD[prev] = dp;
                        snd[lo + Kn] = prev;
                        sdl[lo + Kn] = dp;
                        szl[lo + Kn] = zp;
                        Kn++;
                    }
                    srho[b] = rho;
                    sKn[b] = Kn;
                    sNrot[b] = nrot;
                }
            }
        }
        __syncthreads();
        // C: the deflating rotations on the rows of Z (column pairs, in
        // order); the top merge's go to its Um instead
        for (int rr = tid; rr < n && !top; rr += NT) {
            const int b = rr >> ls, lo = b << ls;
            if (sKn[b] < 0) continue;
            const int nrot = sNrot[b];
            for (int t = 0; t < nrot; t++) {
                const long ia = rr + (long)ra[lo + t] * n, ib = rr + (long)rb[lo + t] * n;
                const double qa = Z[ia], qb = Z[ib], c = rc[lo + t], sn = rs[lo + t];
                Z[ia] = c * qa + sn * qb;
                Z[ib] = c * qb - sn * qa;
            }
        }
        // D: secular equation 1/rho + sum_j zl_j^2 / (dl_j - lambda) = 0 for
        // the root in (dl_i, dl_{i+1}) (the last one in (dl_K-1, dl_K-1 + rho
        // |z|^2)), L lanes per root (L = 1..8 by block size), from the nearer pole;
        // two poles: the root of the quadratic, no iteration
        auto secular = [&](auto Ltag) {
            constexpr int L = decltype(Ltag)::value;
            const int ri = tid / L, sub = tid & (L - 1);
            int b = 0, lo = 0, i = 0, Kn = 0;
            if (ri < n) {
                b = ri >> ls;
                lo = b << ls;
                i = ri - lo;
                Kn = sKn[b];
            }
            if (Kn > 0 && i < Kn) {
                const double rho = srho[b];
                const double *dl = sdl + lo, *zl = szl + lo;
                int org;
                double tau;
                int it = 0;
                if (Kn == 1) {
                    org = 0;
                    tau = rho * zl[0] * zl[0];
                } else if (Kn == 2) {
                    // the roots of the quadratic, each from its nearer pole
                    const double rinv = 1.0 / rho, gap = dl[1] - dl[0];
                    const double z02 = zl[0] * zl[0], z12 = zl[1] * zl[1];
                    if (i == 0) {
                        // the sign of the secular function at the midpoint
                        // picks the nearer pole
                        if (rinv + 2.0 * (z12 - z02) / gap >= 0.0) {
                            // tau in (0, gap/2]: rinv tau^2 - a tau + b = 0
                            // (discriminant as a sum of non-negative terms)
                            const double rg = rinv * gap, a = rg + z02 + z12, bq = z02 * gap;
                            const double dm = rg - z02;
                            org = 0;
                            tau = 2.0 * bq / (a + sqrt(dm * dm + z12 * (z12 + 2.0 * (rg + z02))));
                        } else {
                            // tau in (-gap/2, 0) from the upper pole: rinv tau^2 + a tau - b = 0
                            const double a = rinv * gap - z02 - z12, bq = z12 * gap;
                            org = 1;
                            tau = (a < 0.0) ? 2.0 * bq / (a - sqrt(fabs(a * a + 4.0 * bq * rinv)))
                                            : -(a + sqrt(fabs(a * a + 4.0 * bq * rinv))) / (2.0 * rinv);
                        }
                    } else {
                        // tau > 0 beyond the upper pole: rinv tau^2 - A tau - z1^2 gap = 0
                        const double A = z02 + z12 - rinv * gap;
                        const double Dq = sqrt(A * A + 4.0 * rinv * z12 * gap);
                        org = 1;
                        tau = (A >= 0.0) ? (A + Dq) / (2.0 * rinv) : 2.0 * z12 * gap / (Dq - A);
                    }
                } else {
                    const double rinv = 1.0 / rho;
                    double tlo, thi;
                    if (i < Kn - 1) {
                        const double gap = dl[i + 1] - dl[i];
                        const double mid = 0.5 * gap;
                        // w at the midpoint, and the part of it from the poles
                        // other than i, i+1 (initial guess of LAPACK's dlaed4)
                        double w = 0.0;
                        for (int j = sub; j < Kn; j += L)
                            w = fma(zl[j] * zl[j], rcp_nr((dl[j] - dl[i]) - mid), w);
                        w = grp_sum<L>(w) + rinv;
                        const double zi2 = zl[i] * zl[i], zi12 = zl[i + 1] * zl[i + 1];
                        const double c0 = w - zi2 / (-mid) - zi12 / (gap - mid);
                        double t0;
                        if (w >= 0.0) {
                            org = i;
                            tlo = 0.0;
                            thi = mid;
                            const double a = c0 * gap + zi2 + zi12, bq = zi2 * gap;
                            if (c0 == 0.0) t0 = bq / a;
                            else if (a <= 0.0) t0 = (a - sqrt(fabs(a * a - 4.0 * bq * c0))) / (2.0 * c0);
                            else t0 = 2.0 * bq / (a + sqrt(fabs(a * a - 4.0 * bq * c0)));
                        } else {
                            org = i + 1;
                            tlo = -(gap - mid);
                            thi = 0.0;
                            // c0 t^2 + a t - bq = 0, the root in (-mid, 0)
                            const double a = c0 * gap - zi2 - zi12, bq = zi12 * gap;
                            if (c0 == 0.0) t0 = bq / a;
                            else if (a < 0.0) t0 = 2.0 * bq / (a - sqrt(fabs(a * a + 4.0 * bq * c0)));
                            else t0 = -(a + sqrt(fabs(a * a + 4.0 * bq * c0))) / (2.0 * c0);
                        }
                        tau = (t0 > tlo && t0 < thi) ? t0 : 0.5 * (tlo + thi);
                    } else {
                        double zz = 0.0;
                        for (int j = sub; j < Kn; j += L) zz = fma(zl[j], zl[j], zz);
                        zz = grp_sum<L>(zz);
                        org = i;
                        tlo = 0.0;
                        thi = rho * zz * (1.0 + 8.0 * EPSU) + 0x1.0p-1000;
                        tau = 0.5 * thi;
                    }
                    const double dorg = dl[org];
                    for (it = 0; it < 100; it++) {
                        // poles up to i (psi) and beyond (phi), split by lane
                        double psi = 0.0, dpsi = 0.0, phi = 0.0, dphi = 0.0;
                        double psi2 = 0.0, dpsi2 = 0.0, phi2 = 0.0, dphi2 = 0.0;
                        int j = sub;
                        for (; j + L <= i; j += 2 * L) {
                            const double t = zl[j] * rcp_nr((dl[j] - dorg) - tau);
                            const double t2 = zl[j + L] * rcp_nr((dl[j + L] - dorg) - tau);
                            psi = fma(zl[j], t, psi);
                            dpsi = fma(t, t, dpsi);
                            psi2 = fma(zl[j + L], t2, psi2);
                            dpsi2 = fma(t2, t2, dpsi2);
                        }
                        for (; j <= i; j += L) {
                            const double t = zl[j] * rcp_nr((dl[j] - dorg) - tau);
                            psi = fma(zl[j], t, psi);
                            dpsi = fma(t, t, dpsi);
                        }
                        for (; j + L < Kn; j += 2 * L) {
                            const double t = zl[j] * rcp_nr((dl[j] - dorg) - tau);
                            const double t2 = zl[j + L] * rcp_nr((dl[j + L] - dorg) - tau);
                            phi = fma(zl[j], t, phi);
                            dphi = fma(t, t, dphi);
                            phi2 = fma(zl[j + L], t2, phi2);
                            dphi2 = fma(t2, t2, dphi2);
                        }
                        for (; j < Kn; j += L) {
                            const double t = zl[j] * rcp_nr((dl[j] - dorg) - tau);
                            phi = fma(zl[j], t, phi);
                            dphi = fma(t, t, dphi);
                        }
                        psi += psi2;
                        dpsi += dpsi2;
                        phi += phi2;
                        dphi += dphi2;
                        psi = grp_sum<L>(psi);
                        dpsi = grp_sum<L>(dpsi);
                        phi = grp_sum<L>(phi);
                        dphi = grp_sum<L>(dphi);
                        const double w = rinv + psi + phi;
                        if (w == 0.0) break;
                        if (w < 0.0) tlo = tau;
                        else thi = tau;
                        // rounding bound of w: LAPACK's dlaed4 adds the running
                        // partial sums, at most Kn times the sum of |terms|
                        const double errm = (8.0 + Kn) * (phi - psi) + 2.0 * rinv +
                                            3.0 * fabs(tau) * (dpsi + dphi);
                        if (fabs(w) <= EPSU * errm) break;
                        // the step's quotients by the hardware reciprocal (a
                        // few ulp): the step only steers the iteration, whose
                        // stopping test is on w, and a step outside the
                        // bracket falls back to bisection below
                        double eta;
                        if (i < Kn - 1) {
                            const double Di = (dl[i] - dorg) - tau, Di1 = (dl[i + 1] - dorg) - tau;
                            const double c = w - Di * dpsi - Di1 * dphi;
                            const double a = (Di + Di1) * w - Di * Di1 * (dpsi + dphi);
                            const double bq = Di * Di1 * w;
                            if (c == 0.0)
                                eta = (a != 0.0) ? bq * rcp_nr(a) : 0.5 * (tlo + thi) - tau;
                            else if (a <= 0.0)
                                eta = (a - sqrt(fabs(a * a - 4.0 * bq * c))) * rcp_nr(2.0 * c);
                            else
                                eta = 2.0 * bq * rcp_nr(a + sqrt(fabs(a * a - 4.0 * bq * c)));
                        } else {
                            const double Dl = (dl[i] - dorg) - tau;
                            const double den = w - Dl * dpsi;
                            eta = (den > 0.0) ? Dl + Dl * Dl * dpsi * rcp_nr(den)
                                              : 0.5 * (tlo + thi) - tau;
                        }
                        if (w * eta >= 0.0) eta = -w * rcp_nr(dpsi + dphi);
                        double tn = tau + eta;
                        if (!(tn > tlo && tn < thi)) tn = 0.5 * (tlo + thi);
                        if (tn == tau) break;
                        tau = tn;
                    }
                }
                if (sub == 0) {
                    sorg[lo + i] = org;
                    stau[lo + i] = tau;
                    if (it > 0) atomicMax(&s_iters, it);
                }
            }
        };
        {
            const int L = s >= 8 ? 8 : (s == 4 ? 4 : 1);
            if (L == 8) secular(std::integral_constant<int, 8>{});
            else if (L == 4) secular(std::integral_constant<int, 4>{});
            else if (L == 2) secular(std::integral_constant<int, 2>{});
            else secular(std::integral_constant<int, 1>{});
        }
        __syncthreads();
        // E: Gu-Eisenstat z from the computed roots, L lanes per entry:
        // zhat_q^2 = (lambda_K-1 - d_q)/rho * prod_{i<q} (lambda_i - d_q)/(d_i - d_q)
        //            * prod_{q<=i<K-1} (lambda_i - d_q)/(d_{i+1} - d_q),
        // every factor in (0, 1) except the first
        auto zhat = [&](auto Ltag) {
            constexpr int L = decltype(Ltag)::value;
            const int jq = tid / L, sub = tid & (L - 1);
            int lo = 0, q = 0, Kn = 0;
            if (jq < n) {
                const int b = jq >> ls;
                lo = b << ls;
                q = jq - lo;
                Kn = sKn[b];
            }
            if (Kn > 0 && q < Kn) {
                const double *dl = sdl + lo;
                const double dq = dl[q];
                double prod = 1.0;
                for (int i = sub; i < Kn; i += L) {
                    const double num = (dl[sorg[lo + i]] - dq) + stau[lo + i];
                    const double den = (i == Kn - 1) ? srho[jq >> ls] : (i < q ? dl[i] - dq : dl[i + 1] - dq);
                    prod *= num * rcp_nr(den);
                }
                prod = grp_prod<L>(prod);
                if (sub == 0) szh[lo + q] = copysign(sqrt(fmax(prod, 0.0)), szl[lo + q]);
            }
        };
        {
            const int L = s >= 8 ? 8 : (s == 4 ? 4 : 1);
            if (L == 8) zhat(std::integral_constant<int, 8>{});
            else if (L == 4) zhat(std::integral_constant<int, 4>{});
            else if (L == 2) zhat(std::integral_constant<int, 2>{});
            else zhat(std::integral_constant<int, 1>{});
        }
        __syncthreads();
        if (!top) {
            // F: eigenvector matrix of each rank-one update, column i of
            // block b at ums[lo*s + i + q*s] (i fastest: one row of U per q)
            for (int t = tid; t < nblk << (2 * ls); t += NT) {
                const int b = t >> (2 * ls);
                const int rem = t & ((1 << (2 * ls)) - 1);
                const int q = rem >> ls, i = rem & (s - 1);
                const int lo = b << ls, Kn = sKn[b];
                if (Kn <= 0 || q >= Kn || i >= Kn) continue;
                const double *dl = sdl + lo;
                ums[lo * s + i + q * s] =
                    szh[lo + q] * rcp_nr((dl[q] - dl[sorg[lo + i]]) - stau[lo + i]);
            }
            // stage the non-deflated columns of each block: zs[lo*s + r + q*s]
            {
                const int tot = nblk << (2 * ls);
                for (int t0 = tid; t0 < tot; t0 += 4 * NT) {
                    double v[4];
                    int dst[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const int t = t0 + u * NT;
                        v[u] = 0.0;
                        dst[u] = -1;
                        if (t >= tot) continue;
                        const int b = t >> (2 * ls);
                        const int rem = t & ((1 << (2 * ls)) - 1);
                        const int q = rem >> ls, rl = rem & (s - 1);
                        const int lo = b << ls, hi = min(lo + s, n), Kn = sKn[b];
                        if (Kn <= 0 || q >= Kn || lo + rl >= hi) continue;
                        v[u] = Z[lo + rl + (long)snd[lo + q] * n];
                        dst[u] = t;
                    }
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        if (dst[u] >= 0) zs[dst[u]] = v[u];
                }
            }
            __syncthreads();
            // G: column norms of the update's eigenvectors, eight lanes per column
            {
                const int ci = tid >> 3, sub = tid & 7;
                int lo = 0, i = 0, Kn = 0, b = 0;
                if (ci < n) {
                    b = ci >> ls;
                    lo = b << ls;
                    i = ci - lo;
                    Kn = sKn[b];
                }
                if (Kn > 0 && i < Kn) {
                    const double *u = ums + lo * s + i;
                    double ss = 0.0;
                    for (int q = sub; q < Kn; q += 8) ss = fma(u[q * s], u[q * s], ss);
                    ss = oct_sum(ss);
                    if (sub == 0) sinv[lo + i] = 1.0 / sqrt(ss);
                }
            }
            __syncthreads();
            // H: Z[:, nd_i] = (staged columns) * u_i * sinv_i over the block's
            // rows.  Blocks of 16 and more: 16 x 16 output tiles on the FP64
            // matrix cores, issued as (U^T)(ZS^T) so that a tile's lanes hold 16
            // consecutive rows of one column (128-byte stores); a wave per tile,
            // the k steps beyond Kn zeroed in both operands.  Smaller blocks: a
            // thread per (block, group of 16 columns, row), rows fastest.
            if (s >= 16) {
                const int lt = ls - 4;
                const int tiles = nblk << (2 * lt);
                for (int t = wv; t < tiles; t += NT / 64) {
                    const int b = t >> (2 * lt), rem = t & ((1 << (2 * lt)) - 1);
                    const int rb = (rem >> lt) * 16, cb = (rem & ((1 << lt) - 1)) * 16;
                    const int lo = b << ls, hi = min(lo + s, n), Kn = sKn[b];
                    if (Kn <= 0 || cb >= Kn || lo + rb >= hi) continue;
                    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
                    const double *ub = ums + lo * s + cb + (lane & 15);
                    const double *zb = zs + lo * s + rb + (lane & 15);
                    for (int k0 = 0; k0 < Kn; k0 += 4) {
                        const int q = k0 + (lane >> 4);
                        const bool kin = q < Kn;
                        const double ua = kin ? ub[q * s] : 0.0;  // U[q][cb + l%16]
                        const double zb2 = kin ? zb[q * s] : 0.0;  // ZS[rb + l%16][q]
                        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(ua, zb2, acc, 0, 0, 0);
                    }
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const int col = cb + (lane >> 4) + 4 * v, row = lo + rb + (lane & 15);
                        if (col < Kn && row < hi)
                            Z[row + (long)snd[lo + col] * n] = acc[v] * sinv[lo + col];
                    }
                }
            } else
            {
                const int lcg = (ls > 4) ? ls - 4 : 0;  // column groups of 16: s/16 of them
                const int tot = nblk << (lcg + ls);
                for (int t = tid; t < tot; t += NT) {
                    const int rl = t & (s - 1);
                    const int bc = t >> ls;
                    const int cg = bc & ((1 << lcg) - 1), b = bc >> lcg;
                    const int lo = b << ls, hi = min(lo + s, n), Kn = sKn[b];
                    const int i0 = cg * 16;
                    if (Kn <= 0 || i0 >= Kn || lo + rl >= hi) continue;
                    const int nc = min(16, Kn - i0);
                    double acc[16];
#pragma unroll
                    for (int c = 0; c < 16; c++) acc[c] = 0.0;
                    const double *zb = zs + lo * s + rl;
                    const double *ub = ums + lo * s + i0;
                    for (int q = 0; q < Kn; q++) {
                        const double zv = zb[q * s];
                        // 16-byte aligned: lo * s, q * s and i0 are even
                        const double2 *uq = reinterpret_cast<const double2 *>(ub + q * s);
#pragma unroll
                        for (int c = 0; c < 8; c++) {
                            const double2 u2 = uq[c];
                            acc[2 * c] = fma(zv, u2.x, acc[2 * c]);
                            acc[2 * c + 1] = fma(zv, u2.y, acc[2 * c + 1]);
                        }
                    }
#pragma unroll
                    for (int c = 0; c < 16; c++)
                        if (c < nc)
                            Z[lo + rl + (long)snd[lo + i0 + c] * n] = acc[c] * sinv[lo + i0 + c];
                }
            }
            for (int t = tid; t < n; t += NT) {
                const int b = t >> ls, lo = b << ls, i = t - lo, Kn = sKn[b];
                if (Kn <= 0 || i >= Kn) continue;
                sD[snd[lo + i]] = sdl[lo + sorg[lo + i]] + stau[lo + i];
            }
            __syncthreads();
        } else {
            // top merge: column order (non-deflated first), eigenvalues per
            // column, and the padded, normalised eigenvector matrix of the update
            const int Kn = sKn[0] > 0 ? sKn[0] : 0;
            for (int j = tid; j < n; j += NT) sflag[j] = 0;
            __syncthreads();
            for (int q = tid; q < Kn; q += NT) sflag[snd[q]] = 1;
            __syncthreads();
            // column c's pole: Z column scm[c]; Z column j's column: spos[j]
            for (int j = tid; j < n; j += NT) {
                if (sflag[j]) continue;
                int pos = Kn;
                for (int q = 0; q < j; q++) pos += !sflag[q];
                colmap[pos] = j;
                scm[pos] = j;
                spos[j] = pos;
                slam[pos] = sD[j];
            }
            for (int q = tid; q < Kn; q += NT) {
                colmap[q] = snd[q];
                scm[q] = snd[q];
                spos[snd[q]] = q;
                slam[q] = sdl[sorg[q]] + stau[q];
            }
            __syncthreads();
            // Um in LDS (ld n), row r = Z column r
            double *um = lds;
            {
                const int i = tid >> 3, sub = tid & 7;
                if (i < Kn) {
                    const double li = sdl[sorg[i]], ti = stau[i];
                    double ss = 0.0;
                    for (int q = sub; q < Kn; q += 8) {
                        const double u = szh[q] * rcp_nr((sdl[q] - li) - ti);
                        ss = fma(u, u, ss);
                    }
                    ss = oct_sum(ss);
                    const double iv = 1.0 / sqrt(ss);
                    for (int r = sub; r < n; r += 8) {
                        const int q = spos[r];
                        um[r + i * n] = (q < Kn) ? szh[q] * rcp_nr((sdl[q] - li) - ti) * iv : 0.0;
                    }
                } else if (i < n) {
                    const int j = scm[i];
                    for (int r = sub; r < n; r += 8) um[r + i * n] = (r == j) ? 1.0 : 0.0;
                }
            }
            __syncthreads();
            // Z G_0 ... G_{k-1} Um = Z (G_0 (... (G_{k-1} Um))): each rotation
            // of Z's columns (a, b) acts on Um's rows a and b, last first
            const int nrot = sNrot[0];
            for (int i = tid; i < n && nrot > 0; i += NT) {
                double *col = um + i * n;
                for (int t = nrot - 1; t >= 0; t--) {
                    const int a = ra[t], b = rb[t];
                    const double c = rc[t], sn = rs[t];
                    const double ua = col[a], ub = col[b];
                    col[a] = c * ua - sn * ub;
                    col[b] = sn * ua + c * ub;
                }
            }
            __syncthreads();
            for (int e = tid; e < n * n; e += NT) Um[e] = um[e];
            top_done = true;
            __syncthreads();
            break;
        }
    }
    if (part == 1) {
        // the poles after the lower merges and their iteration count
        __syncthreads();
        for (int i = tid; i < n; i += NT) dsave[i] = sD[i];
        if (tid == 0) dsave[n] = (double)s_iters;
        return;
    }
    if (!top_done) {
        // n == 1: no merge at all
        for (int j = tid; j < n; j += NT) {
            colmap[j] = j;
            slam[j] = sD[j];
            Um[j + (long)j * n] = 1.0;
        }
        __syncthreads();
    }
    // final order (descending), dropped tail, numerical rank, tail rule
    __shared__ int s_keep;
    {
        // rank of column c in descending order, eight lanes per column
        const int c = tid >> 3, sub = tid & 7;
        if (c < n) {
            const double lc = slam[c];
            int pos = 0;
            for (int q = sub; q < n; q += 8) {
                const double lq = slam[q];
                pos += (lq > lc) || (lq == lc && q < c);
            }
            pos = (int)oct_sum((double)pos);
            if (sub == 0) {
                colidx[pos] = c;
                sdl[pos] = lc;  // sdl reused: eigenvalues in descending order (scaled)
            }
        }
    }
    __syncthreads();
    const int es = *eexp;
    // Wave 0 holds the descending values two per lane and decides:
    //  - the smallest eigenvalues are dropped while their running sum stays
    //    within lim = budget * lmax: the suffix sums S(q) and the values grow
    //    as q falls, so the dropped set is {q >= keep} with keep the least q
    //    where S(q) <= lim and v_q < lmax;
    //  - the numerical rank counts the kept values above (sqrt(n) u sigma_0)^2
    //    (a prefix, the values being sorted);
    //  - tail rule on the scaled values, sqrt(tail) * 2^(es/2) < delta, with
    //    the tail T(q) over [q, numrank) shrinking as q grows.
    // The suffix sums are wave scans; the least q of each rule is the first
    // set bit of a ballot.
    if (wv == 0) {
        const bool in0 = lane < n, in1 = lane + 64 < n;
        const double h0 = in0 ? fmax(sdl[lane], 0.0) : 0.0;
        const double h1 = in1 ? fmax(sdl[lane + 64 < NMAX ? lane + 64 : 0], 0.0) : 0.0;
        const double lmax = readlane_d(h0, 0);
        const double lim = budget * lmax;
        const double S1 = suffix_sum(h1);
        const double S0 = suffix_sum(h0) + readlane_d(S1, 0);
        const unsigned long long b0 = __ballot(in0 && S0 <= lim && h0 < lmax);
        const unsigned long long b1 = __ballot(in1 && S1 <= lim && h1 < lmax);
        const int keep = b0 ? __ffsll((long long)b0) - 1 : (b1 ? 63 + __ffsll((long long)b1) : n);
        const double cum = (keep >= n) ? 0.0 : (keep < 64 ? readlane_d(S0, keep) : readlane_d(S1, keep - 64));
        const double thr2 = (double)n * EPSU * EPSU * lmax;  // (sqrt(n) u sigma_0)^2
        int numrank = 0;
        if (lmax > 0.0)
            numrank = __popcll(__ballot(lane < keep && h0 > thr2)) +
                      __popcll(__ballot(lane + 64 < keep && h1 > thr2));
        const double dl2 =
            (delta > 0.0) ? exp(2.0 * (log(delta) - (es / 2) * 0.6931471805599453)) : -1.0;
        const double T1 = suffix_sum(lane + 64 < numrank ? h1 : 0.0);
        const double T0 = suffix_sum(lane < numrank ? h0 : 0.0) + readlane_d(T1, 0);
        const unsigned long long c0 = __ballot(lane < numrank && T0 < dl2);
        const unsigned long long c1 = __ballot(lane + 64 < numrank && T1 < dl2);
        int rho = c0 ? __ffsll((long long)c0) - 1 : (c1 ? 63 + __ffsll((long long)c1) : numrank);
        if (rho > n) rho = n;
        if (rho > cap) rho = cap;
        if (rho < 1) rho = 1;
        if (lane == 0) {
            iout[0] = numrank;
            iout[1] = rho;
            iout[2] = s_iters;
            dinfo[5] = ldexp(cum, es);
            s_keep = keep;
        }
    }
    __syncthreads();
    const int keep = s_keep;
    for (int q = tid; q < n; q += NT) sig[q] = (q < keep) ? ldexp(sqrt(fmax(sdl[q], 0.0)), es / 2) : 0.0;
}

// ---- 3. back transformation -----------------------------------------------
// W = H_0 H_1 ... H_{n-3} Z, the reflectors applied last first.  Sixteen lanes (one DPP row) own a column, each holding the rows
// l, l+16, ..., so a reflector's dot product reduces inside the row; a
// workgroup of four waves owns 16 columns and stages the reflectors in LDS.
constexpr int ORM_RPL = EIG_NMAX / 16;  // rows per lane
__global__ __launch_bounds__(256) void k_ormtr(int n, const double *__restrict__ Vh,
                                               const double *__restrict__ tau,
                                               const double *__restrict__ Z,
                                               double *__restrict__ W) {
    extern __shared__ double vs[];  // n x n reflectors, then n taus
    const int tid = threadIdx.x;
    const long nn = (long)n * n;
    for (long e0 = tid; e0 < nn; e0 += 4 * 256) {
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const long e = e0 + (long)u * 256;
            v[u] = (e < nn) ? Vh[e] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const long e = e0 + (long)u * 256;
            if (e < nn) vs[e] = v[u];
        }
    }
    for (int i = tid; i < n; i += 256) vs[nn + i] = tau[i];
    __syncthreads();
    const int l = tid & 15;
    const int c = blockIdx.x * 16 + (tid >> 4);
    const bool live = c < n;  // rows of 16 lanes: uniform per DPP row
    const double *zc = Z + (long)(live ? c : 0) * n;
    double x[ORM_RPL];
#pragma unroll
    for (int m = 0; m < ORM_RPL; m++) {
        const int i = l + 16 * m;
        x[m] = (live && i < n) ? zc[i] : 0.0;
    }
    for (int k = n - 3; k >= 0; k--) {
        const double tk = vs[nn + k];
        if (tk == 0.0) continue;
        const double *v = vs + (long)k * n;
        double vr[ORM_RPL];
        double d0 = 0.0, d1 = 0.0;
#pragma unroll
        for (int m = 0; m < ORM_RPL; m++) {
            const int i = l + 16 * m;
            vr[m] = (i < n) ? v[i] : 0.0;
            if (m & 1) d1 = fma(vr[m], x[m], d1);
            else d0 = fma(vr[m], x[m], d0);
        }
        double dt = quad_sum(d0 + d1);
        dt += dppd<0x141>(dt);
        dt += dppd<0x140>(dt);
        dt *= tk;
#pragma unroll
        for (int m = 0; m < ORM_RPL; m++) x[m] = fma(-dt, vr[m], x[m]);
    }
    if (live)
#pragma unroll
        for (int m = 0; m < ORM_RPL; m++) {
            const int i = l + 16 * m;
            if (i < n) W[i + (long)c * n] = x[m];
        }
}

__global__ void k_svd_factors_perm(int m, int rho, const int *__restrict__ colidx,
                                   const double *__restrict__ U, long ldu,
                                   const double *__restrict__ sig, double wscale,
                                   double *__restrict__ W, double *__restrict__ US) {
    const long total = (long)m * rho;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total;
         e += (long)gridDim.x * blockDim.x) {
        const int j = (int)(e / m), i = (int)(e - (long)j * m);
        const double u = U[i + (long)colidx[j] * ldu], s = sig[j];
        if (US) US[i + (long)j * m] = u * s;
        if (W) W[j + (long)i * rho] = (s > 0.0) ? wscale * u / s : 0.0;
    }
}

void ormtr_attr() {
    static bool done = false;
    if (done) return;
    HIPCHECK(hipFuncSetAttribute((const void *)k_ormtr, hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (EIG_NMAX * EIG_NMAX + EIG_NMAX) * (int)sizeof(double)));
    done = true;
}

void launch_ormtr(int c, const double *Vh, const double *tau, const double *Z, double *W) {
    const double cc = (double)c * c;
    PTT_LAUNCH_FB("syev_ormtr", 4.0 * cc * c, 8.0 * 3.0 * cc, k_ormtr, dim3(cdiv(c, 16)),
                  dim3(256), ((size_t)c * c + c) * sizeof(double), c, Vh, tau, Z, W);
}

// Tridiagonalisation, divide and conquer and back transformation, W = Q Z.
// With the side stream on, the back transformation runs there beside the
// top merge (the merges below it leave Z final); the main stream waits for
// it before returning.
template <int NMAX>
void launch_syev(int c, const double *G, double *Vh, double *tau, double *d, double *e, int *ex,
                 double *Z, double *Um, double *W, int *colmap, int *colidx, double *sig,
                 int *iout, double *dinfo, double delta, int cap, double budget, double *dsave) {
    static bool attr = false;
    if (!attr) {
        HIPCHECK(hipFuncSetAttribute((const void *)k_stedc<NMAX>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                     NMAX * NMAX * (int)sizeof(double)));
        attr = true;
    }
    ormtr_attr();
    const double cc = (double)c;
    const size_t shm = (size_t)NMAX * NMAX * sizeof(double);
    PTT_LAUNCH_FB("syev_sytrd", 4.0 * cc * cc * cc / 3.0, 8.0 * cc * cc * 2.0, k_sytrd<NMAX>,
                  dim3(1), dim3(4 * NMAX + 64), 0, c, G, (long)c, Vh, tau, d, e, ex, dinfo);
    if (!ptt_hip_side_enabled()) {
        PTT_LAUNCH_FB("syev_stedc", 2.0 * cc * cc * cc / 3.0, 8.0 * cc * cc * 3.0, k_stedc<NMAX>,
                      dim3(1), dim3(8 * NMAX), shm, c, d, e, ex, Z, Um, colmap, colidx, sig, iout,
                      dinfo, delta, cap, budget, 0, dsave);
        launch_ormtr(c, Vh, tau, Z, W);
        return;
    }
    PTT_LAUNCH_FB("syev_stedc", cc * cc * cc / 3.0, 8.0 * cc * cc * 2.0, k_stedc<NMAX>, dim3(1),
                  dim3(8 * NMAX), shm, c, d, e, ex, Z, Um, colmap, colidx, sig, iout, dinfo,
                  delta, cap, budget, 1, dsave);
    ptt_hip_side_begin();
    launch_ormtr(c, Vh, tau, Z, W);
    ptt_hip_side_end(0);
    PTT_LAUNCH_FB("syev_stedc_top", cc * cc * cc / 3.0, 8.0 * cc * cc * 2.0, k_stedc<NMAX>,
                  dim3(1), dim3(8 * NMAX), shm, c, d, e, ex, Z, Um, colmap, colidx, sig, iout,
                  dinfo, delta, cap, budget, 2, dsave);
    ptt_hip_side_wait(0);
}

// Workspace of one eigen-decomposition of order c: reflectors, divide and
// conquer vectors, the top update's matrix, the back-transformed vectors
// (c x c each), then tau, d, e, two int vectors and the c + 1 doubles that
// pass the divide and conquer's state to its top merge.
constexpr size_t syev_ws_doubles(size_t c) { return 4 * c * c + 8 * c + 8; }

void syev_run(int c, const double *G, double *sig, double *U, long ldu, int *colidx, int *iout,
              double *dinfo, double delta, int cap, double budget, double *ws) {
    const size_t cc = (size_t)c * c;
    double *Vh = ws, *Z = Vh + cc, *Um = Z + cc, *W = Um + cc;
    double *tau = W + cc, *d = tau + c, *e = d + c;
    int *colmap = (int *)(e + c);
    int *ex = colmap + c;
    double *dsave = (double *)(colmap + 2 * (size_t)c);  // c + 1 doubles
    if (c <= 64)
        launch_syev<64>(c, G, Vh, tau, d, e, ex, Z, Um, W, colmap, colidx, sig, iout, dinfo,
                        delta, cap, budget, dsave);
    else
        launch_syev<128>(c, G, Vh, tau, d, e, ex, Z, Um, W, colmap, colidx, sig, iout, dinfo,
                         delta, cap, budget, dsave);
    ptt_hip_dgemm('N', 'N', c, c, c, 1.0, W, c, Um, c, 0.0, U, ldu);
}

// Fixed workspace of the entry point that allocates nothing: one copy per
// GPU, held until the process ends.  Host code reaches it only through the
// device address from hipGetSymbolAddress (the name is a host stand-in).
constexpr int NOALLOC_CMAX = EIG_NMAX;
__device__ __align__(256) double scratch[syev_ws_doubles(NOALLOC_CMAX)];
constexpr int NOALLOC_MAXDEV = 64;
double *g_scratch_dev[NOALLOC_MAXDEV] = {nullptr};

// The device address of `scratch` on the current device (looked up once per
// device; no allocation).  Returns nullptr for a device index beyond the table.
double *scratch_address() {
    int dev = 0;
    HIPCHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= NOALLOC_MAXDEV) return nullptr;
    if (!g_scratch_dev[dev]) {
        void *p = nullptr;
        HIPCHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_dev[dev] = (double *)p;
    }
    return g_scratch_dev[dev];
}

}  // namespace

extern "C" {

// Called by ptt_hip_init with the library's device current.
void ptt_hip_noalloc_setup(void) { (void)scratch_address(); }

void ptt_hip_syev_gram(int c, const double *G, double *sig, double *U, long ldu, int *colidx,
                       int *iout, double *dinfo, double delta, int cap, double budget) {
    ptt_hip_init();
    if (c <= 0) return;
    if (c > EIG_NMAX) {
        fprintf(stderr, "ptt_hip_syev_gram: c = %d exceeds %d\n", c, EIG_NMAX);
        exit(1);
    }
    double *ws = (double *)ptt_hip_scratch(PTT_WS_EIG, sizeof(double) * syev_ws_doubles(c));
    syev_run(c, G, sig, U, ldu, colidx, iout, dinfo, delta, cap, budget, ws);
}

int ptt_hip_syev_gram_noalloc(int c, const double *G, double *sig, double *U, long ldu,
                              int *colidx, int *iout, double *dinfo, double delta, int cap,
                              double budget) {
    if (!ptt_hip_initialized()) {
        fprintf(stderr, "ptt_hip_syev_gram_noalloc: call ptt_hip_init() first (set-up may "
                        "allocate; this entry point does not)\n");
        return -2;
    }
    if (c <= 0) return 0;
    if (c > NOALLOC_CMAX) {
        fprintf(stderr, "ptt_hip_syev_gram_noalloc: c = %d exceeds the fixed workspace's "
                        "maximum order %d\n", c, NOALLOC_CMAX);
        return -1;
    }
    double *ws = scratch_address();
    if (!ws) {
        fprintf(stderr, "ptt_hip_syev_gram_noalloc: device index beyond %d\n", NOALLOC_MAXDEV);
        return -3;
    }
    syev_run(c, G, sig, U, ldu, colidx, iout, dinfo, delta, cap, budget, ws);
    return 0;
}

void ptt_hip_svd_factors_perm(int m, int rho, const int *colidx, const double *U, long ldu,
                              const double *sig, double wscale, double *W, double *US) {
    ptt_hip_init();
    const long total = (long)m * rho;
    if (total <= 0) return;
    PTT_LAUNCH("svd_factors", k_svd_factors_perm, dim3(stream_blocks(total, 256)), dim3(256), 0,
               m, rho, colidx, U, ldu, sig, wscale, W, US);
}

}  // extern "C"
