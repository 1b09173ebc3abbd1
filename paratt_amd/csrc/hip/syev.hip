// syev.hip -- eigen-decomposition of a symmetric positive semi-definite
// Gram matrix (c <= 192) for the Gram route of the right-to-left truncation
// step: G = U diag(sigma^2) U^T.
//
// The step needs the left singular vectors and values of a bond matrix M
// from its Gram G = M M^T.  A one-sided Jacobi SVD of a Cholesky factor of
// G performs about 8 sweeps x 127 rounds of pair rotations (~100 MFLOP at
// c = 128) on one CU; this solver does ~7 MFLOP:
//   1. k_sytrd: Householder tridiagonalisation G = Q T Q^T, one workgroup,
//      G held in registers (16 x 16 tiles), one reflector per step with two
//      workgroup barriers;
//   2. k_dc_leaf, k_dc_roots, k_dc_vecs, k_dc_top: Cuppen's divide and conquer
//      on T (split into 2 x 2 blocks, merged bottom-up by rank-one updates), over
//      several workgroups, with the deflation rules of Dongarra and Sorensen,
//      the secular-equation iteration of Li's "middle way" (SIAM J. Sci.
//      Comput. 1994, as in LAPACK's dlaed4) from the
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
// A Gram with an entry that is not finite is taken as zero and its sigma come out
// as NaN: the orders and lists of the divide and conquer are permutations only of
// values that compare, and index memory.
#include "common.hpp"

#include <cmath>
#include <type_traits>

using namespace ptt;

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr double EPSU = 0x1.0p-53;
constexpr int EIG_NMAX = 192;
constexpr int EIG_NONFINITE = 0x7fffffff;  // in place of the scaling's exponent

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
// Sum over aligned groups of L = 2, 4, ..., 32 lanes, product of 2, 4 or 8.
template <int L>
__device__ __forceinline__ double grp_sum(double x) {
    if constexpr (L == 2) x += dppd<0xB1>(x);
    if constexpr (L == 4) x = quad_sum(x);
    if constexpr (L >= 8) x = oct_sum(x);
    if constexpr (L >= 16) x += dppd<0x140>(x);
    if constexpr (L == 32) x = xor16_sum(x);
    return x;
}
template <int L>
__device__ __forceinline__ double grp_prod(double x) {
    if constexpr (L == 2) x *= dppd<0xB1>(x);
    if constexpr (L == 4) x = quad_prod(x);
    if constexpr (L == 8) x = oct_prod(x);
    return x;
}
// sqrt(x) for x >= 0 to a few ulp; 0 below 2^-900 (x not far above 1 otherwise).
__device__ __forceinline__ double sqrt_pos(double x) {
    return x > 0x1.0p-900 ? sqrt_nr(x) : 0.0;
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
// Register tiles: G is cut into 16 x 16 tiles; row wave I holds tile row I (NB =
// NMAX/16 of them), beyond 128 rows tile rows I and I + NB/2.  Lane l (a = l/16, j = l%16) holds rows
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
// the power-of-two scaling (EIG_NONFINITE: an entry of G is not finite), max |G|
// (dinfo[6], infinite then) and the trace of G (dinfo[7]).
// Only the upper triangle of G is read.
//
// Bound by the chain of a step (about 1 us: the product's lane sums, two barriers,
// the reflector wave's two reductions and its root); at 192 rows also by the row
// waves' FP64 issue (288 multiply-adds a lane a step).  Measured: 26 us at 32 rows,
// 43 at 59, 124 at 128, 395 at 192 (734 when v and p were held in registers, which
// spilled).  A raised priority of the reflector wave made no difference.
__device__ __forceinline__ double readlane_d(double v, int l) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double sel(bool c, double x, double y) { return c ? x : y; }

// Tile rows a row wave holds: two beyond 128 rows (row wave I: I and I + NB / 2),
// so that the workgroup keeps 256 registers a lane.
template <int NMAX>
struct sytrd_geom {
    static constexpr int NB = NMAX / 16, TR = NMAX > 128 ? 2 : 1, NWR = NB / TR;
    static constexpr int E = (NMAX + 63) / 64;  // entries of a row a lane of the reflector wave
    static constexpr int NT = 64 * NWR + 64;
};

template <int NMAX>
__global__ __launch_bounds__(sytrd_geom<NMAX>::NT) void k_sytrd(int n, const double *__restrict__ G,
                                                         long ldg, double *__restrict__ Vh,
                                                         double *__restrict__ tau_out,
                                                         double *__restrict__ d_out,
                                                         double *__restrict__ e_out,
                                                         int *__restrict__ eexp,
                                                         double *__restrict__ dinfo) {
    using geom = sytrd_geom<NMAX>;
    constexpr int NB = geom::NB, TR = geom::TR, NWR = geom::NWR, E = geom::E;
    constexpr int NTM = 64 * NWR, NT = NTM + 64, NW = NT / 64;
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

    double g[TR][NB][4];
    double amax = 0.0, tr = 0.0;
#pragma unroll
    for (int t = 0; t < TR; t++)
#pragma unroll
        for (int J = 0; J < NB; J++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = 16 * (I + NWR * t) + ga + 4 * v, col = 16 * J + gj;
                double x = 0.0;
                if (!star && row < n && col < n)
                    x = (row <= col) ? G[row + (long)col * ldg] : G[col + (long)row * ldg];
                g[t][J][v] = x;
                amax = fmax(amax, fabs(x) < INFINITY ? fabs(x) : INFINITY);
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
        if (!(m < INFINITY)) s_e = EIG_NONFINITE;
        *eexp = s_e;
    }
    __syncthreads();
    const int es = s_e;
#pragma unroll
    for (int t = 0; t < TR; t++)
#pragma unroll
        for (int J = 0; J < NB; J++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                g[t][J][v] = es == EIG_NONFINITE ? 0.0 : ldexp(g[t][J][v], -es);

    // Row i of this wave's tile row t into rowb[slot] (called by the whole
    // wave; i wave-uniform, held by the lanes with a = i % 4 in register
    // v = (i % 16) / 4).
    auto copy_row = [&](int i, int slot) {
        const int v = (i & 15) >> 2;
#pragma unroll
        for (int t = 0; t < TR; t++)
            if (I + NWR * t == i >> 4 && ga == (i & 3)) {
                // g[t][J][v] by a 0/1 mask (exact: one term is nonzero), so every
                // register index stays constant and g stays in registers
                const double m0 = (v == 0) ? 1.0 : 0.0, m1 = (v == 1) ? 1.0 : 0.0;
                const double m2 = (v == 2) ? 1.0 : 0.0, m3 = (v == 3) ? 1.0 : 0.0;
#pragma unroll
                for (int J = 0; J < NB; J++)
                    rowb[slot][16 * J + gj] = fma(
                        g[t][J][3], m3, fma(g[t][J][2], m2, fma(g[t][J][1], m1, g[t][J][0] * m0)));
            }
    };
    // The reflector wave turns row p (entries a[u] = row[lane + 64 u]) into the
    // reflector for step p, from column p below the diagonal: v into vb[slot],
    // tau, d_p, e_p = beta (the row waves copy v to Vh at the start of step p).
    // x0 = row[p+1] and dp = row[p] arrive as wave-uniform values (formed by
    // every lane with the owner lane's arithmetic, so no lane reads).
    auto reflector = [&](int p, int slot, const double(&a)[E], double x0, double dp) {
        double s2 = 0.0;
#pragma unroll
        for (int u = 0; u < E; u++) {
            const int i = lane + 64 * u;
            const double x = (i >= p + 2 && i < NMAX) ? a[u] : 0.0;
            s2 = fma(x, x, s2);
        }
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
#pragma unroll
        for (int u = 0; u < E; u++) {
            const int i = lane + 64 * u;
            const double w = (i == p + 1) ? 1.0 : (i > p + 1 ? a[u] * scl : 0.0);
            if (i < NMAX) vb[slot][i] = w;
        }
        if (lane == 0) {
            tkb[slot] = tk;
            sd[p] = dp;
            se[p] = beta;
            st[p] = tk;
        }
    };
    // entries of an LDS row vector at columns lane + 64 u
    auto lrow = [&](const double *v, double(&x)[E]) {
#pragma unroll
        for (int u = 0; u < E; u++)
            x[u] = (lane + 64 * u < NMAX) ? v[lane + 64 * u < NMAX ? lane + 64 * u : 0] : 0.0;
    };

    // p starts as zero: a wave whose rows stop mattering before the first reflector
    // (leading zero or diagonal rows) never writes its entries, which later steps
    // multiply by v = 0
    for (int i = tid; i < NMAX; i += NT) pp[i] = 0.0;
    if (!star && I == 0) {
        copy_row(0, 1);
        copy_row(1, 0);
    }
    lds_sync();
    if (star) {
        double a[E];
        lrow(rowb[1], a);
        reflector(0, 0, a, rowb[1][1 < NMAX ? 1 : 0], rowb[1][0]);
    }
    lds_sync();

    for (int k = 0; k + 2 < n; k++) {
        const double *vk = vb[k & 1];
        const double tk = tkb[k & 1];
        if (!star) {
            for (int i = tid; i < n; i += NTM) Vh[i + (long)k * n] = vk[i];
            const bool act = (16 * (I + NWR * (TR - 1)) + 15 > k);
            if (tk != 0.0) {
                // two tile rows leave no registers for v and p: they are read where
                // they are used
                constexpr bool HOLD = TR == 1;
                double vJ[HOLD ? NB : 1], dot = 0.0;
                if (act) {
                    double acc[TR][4];
#pragma unroll
                    for (int t = 0; t < TR; t++)
#pragma unroll
                        for (int v = 0; v < 4; v++) acc[t][v] = 0.0;
#pragma unroll
                    for (int J = 0; J < NB; J++) {
                        const double vj = vk[16 * J + gj];
                        if (HOLD) vJ[HOLD ? J : 0] = vj;
#pragma unroll
                        for (int t = 0; t < TR; t++)
#pragma unroll
                            for (int v = 0; v < 4; v++) acc[t][v] = fma(g[t][J][v], vj, acc[t][v]);
                        if (!HOLD && J % 3 == 2) __asm__ __volatile__("" ::: "memory");
                    }
#pragma unroll
                    for (int t = 0; t < TR; t++) {
                        // reduce-scatter over the 16 lanes of the row: lane j
                        // ends with the sum for v = 2 (j / 8 % 2) + (j / 4 % 2)
                        const bool h8 = (gj & 8) != 0, h4 = (gj & 4) != 0;
                        const double k0 = sel(h8, acc[t][2], acc[t][0]);
                        const double k1 = sel(h8, acc[t][3], acc[t][1]);
                        const double s0 = sel(h8, acc[t][0], acc[t][2]);
                        const double s1 = sel(h8, acc[t][1], acc[t][3]);
                        const double u0 = k0 + dppd<0x128>(s0);  // row_ror:8
                        const double u1 = k1 + dppd<0x128>(s1);
                        const double kk2 = sel(h4, u1, u0), ss2 = sel(h4, u0, u1);
                        double x = kk2 + dppd<0x141>(ss2);  // half-row mirror: 4-lane groups swap
                        x = quad_sum(x);
                        if ((gj & 3) == 0) {
                            const int vi = 2 * (int)h8 + (int)h4;
                            pp[16 * (I + NWR * t) + ga + 4 * vi] = tk * x;
                        }
                    }
                }
                lds_sync();
                if (act) {
                    double pJ[HOLD ? NB : 1];
#pragma unroll
                    for (int J = 0; J < NB; J++) {
                        const double pj = pp[16 * J + gj];
                        if (HOLD) pJ[HOLD ? J : 0] = pj;
                        dot = fma(pj, HOLD ? vJ[HOLD ? J : 0] : vk[16 * J + gj], dot);
                        if (!HOLD && J % 3 == 2) __asm__ __volatile__("" ::: "memory");
                    }
                    // p^T v over the 16 columns j of the row (each DPP row
                    // forms the same sum)
                    dot = quad_sum(dot);
                    dot += dppd<0x141>(dot);
                    dot += dppd<0x140>(dot);
                    const double kk = 0.5 * tk * dot;
#pragma unroll
                    for (int t = 0; t < TR; t++) {
                        double vr[4], wr[4];
#pragma unroll
                        for (int v = 0; v < 4; v++) {
                            const int row = 16 * (I + NWR * t) + ga + 4 * v;
                            vr[v] = vk[row];
                            wr[v] = pp[row] - 2.0 * kk * vr[v];
                        }
#pragma unroll
                        for (int J = 0; J < NB; J++) {
                            const double pj = HOLD ? pJ[HOLD ? J : 0] : pp[16 * J + gj];
                            const double vj = HOLD ? vJ[HOLD ? J : 0] : vk[16 * J + gj];
#pragma unroll
                            for (int v = 0; v < 4; v++)
                                g[t][J][v] = fma(-vr[v], pj, fma(-vj, wr[v], g[t][J][v]));
                            // (limits how many reads are hoisted)
                            if (!HOLD && J % 3 == 2) __asm__ __volatile__("" ::: "memory");
                        }
                    }
                }
            }
            // row k+2 (now updated through step k) for the reflector wave
            copy_row(k + 2, (k + 1) & 1);
        } else {
            // row k+1, updated through step k-1 (copied before the last barrier),
            // and its entries k+1 (the diagonal) and k+2 as uniform values
            const int k1 = k + 1, k2 = (k + 2 < NMAX) ? k + 2 : k + 1;
            const double *rk = rowb[k & 1];
            double a[E];
            lrow(rk, a);
            double dp = rk[k1];
            double x0 = (k + 2 < NMAX) ? rk[k2] : 0.0;
            if (tk != 0.0) {
                double v[E];
                lrow(vk, v);
                const double vx = vk[k2];
                lds_sync();
                double p[E];
                lrow(pp, p);
                const double pk = pp[k1], px = pp[k2];
                // fma from zero: a bare product could be contracted into the first
                // addition across lanes, whose result would then differ by lane
                double pv = 0.0;
#pragma unroll
                for (int u = E - 1; u >= 0; u--) pv = fma(p[u], v[u], pv);
                const double kk = 0.5 * tk * wave_sum(pv);
                const double w = pk - 2.0 * kk;  // v_{k+1} = 1
#pragma unroll
                for (int u = 0; u < E; u++) a[u] = fma(-1.0, p[u], fma(-v[u], w, a[u]));
                // the owner lanes' arithmetic for entries k+1 and k+2
                dp = fma(-1.0, pk, fma(-1.0, w, dp));
                if (k + 2 < NMAX) x0 = fma(-1.0, px, fma(-vx, w, x0));
            }
            reflector(k1, k1 & 1, a, x0, dp);
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
// so a leaf's d_i loses the |e| of the couplings that were cut beside it.  The eigenvectors of
// the blocks live in the block-diagonal Z (n x n, ld n).  At a merge z =
// [last row of Z1; sign * first row of Z2] / sqrt(2) and rho = 2 |beta|.
//
// The merges up to 32 rows run in k_dc_leaf, a workgroup per 32 rows with its Z
// in LDS; each merge beyond takes two launches, k_dc_roots and k_dc_vecs, a
// workgroup per 16 columns: what a merge decides once (order, deflation, the
// vector zhat) every workgroup repeats, the roots and the eigenvectors, where
// the work is, are divided.  The last merge (`top`) always takes this form.
// All merges in one workgroup of 1024 threads, with Z in memory, were bound by
// the FP64 instructions of one CU: 178 us at n = 128, 95 at 59, 62 at 32; this
// form takes 98, 65 and 44 (with the gaps between its launches).  Half of the leaf
// kernel's time is its roots: 1500 cycles an iteration, 4 to 8 iterations a level.
//
// Deflation (one wave per block): entries with rho |z| <= tol are deflated;
// consecutive remaining entries whose poles are closer than the tolerance
// allows (|t c s| <= tol for the rotation that zeroes one z) are combined by
// that rotation.  The pairs are found by all lanes at once; one lane visits those
// and, after each rotation, the entry that follows (a walk over every entry, with
// the same outcome, took 10 us at 128 of them); the lists are formed by ballots.
//
// The top merge stops after the rank-one eigenvector matrix and leaves Z
// as the lower merges left it: column c of Um (n x n, ld n) is the update's
// eigenvector c (non-deflated first, then the deflated unit vectors) with
// its rows in the order of Z's columns, and the top merge's deflating
// rotations of Z's column pairs are applied to Um's rows instead (last
// first), so U = (Q Z) Um.  Also written: sigma (descending, scaled back),
// colidx (descending rank -> U column) and numrank, rho.  Z is final before the
// top merge, so the back transformation Q Z runs beside it.

// Deflation of one block by GL lanes (gl: lane in the group, which starts at
// lane gbase of the wave); K entries at the sorted positions sperm[0 .. K).  A
// lane takes the positions gl + 64 w, w < NW.  Lists snd, sdl, szl and rotations
// ra, rb, rc, rs; Kn and nrot as lane 0 has them.
template <int NW>
__device__ __forceinline__ void deflate(int GL, int gl, int gbase, int K, double rho,
                                        const int *sperm, double *sz, double *sD, int *snd,
                                        double *sdl, double *szl, int *ra, int *rb, double *rc,
                                        double *rs, int &Kn_out, int &nrot_out) {
    typedef unsigned long long u64;
    const u64 gmask = (GL == 64) ? ~0ULL : (((1ULL << GL) - 1) << gbase);
    const u64 below = (gl == 0) ? 0ULL : ((~0ULL) >> (64 - gl));
    int jw[NW];
    double zw[NW], dw[NW], dmax = 0.0, zmax = 0.0;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        const int q = gl + 64 * w;
        jw[w] = (q < K) ? sperm[q] : -1;
        zw[w] = jw[w] >= 0 ? sz[jw[w]] : 0.0;
        dw[w] = jw[w] >= 0 ? sD[jw[w]] : 0.0;
        dmax = fmax(dmax, fabs(dw[w]));
        zmax = fmax(zmax, fabs(zw[w]));
    }
    for (int o = 1; o < GL; o <<= 1) {
        dmax = fmax(dmax, __shfl_xor(dmax, o, GL));
        zmax = fmax(zmax, __shfl_xor(zmax, o, GL));
    }
    const double tol = 8.0 * EPSU * fmax(dmax, zmax);
    // kept positions of the group, bit = sorted position; the position kept
    // before q, and the first one of a mask after q (-1: none)
    u64 m[NW], f[NW], r[NW];
    bool keep[NW];
#pragma unroll
    for (int w = 0; w < NW; w++) {
        keep[w] = jw[w] >= 0 && !(rho * fabs(zw[w]) <= tol);
        m[w] = (__ballot(keep[w]) & gmask) >> gbase;
        r[w] = 0;
    }
    auto before = [&](int q) {
        int p = -1;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const int l = q - 64 * w;  // bits below l
            const u64 x = l >= 64 ? m[w] : l > 0 ? m[w] & (~0ULL >> (64 - l)) : 0ULL;
            if (x) p = 64 * w + 63 - __clzll((long long)x);
        }
        return p;
    };
    auto next = [&](const u64(&a)[NW], int q) {
        int p = -1;
#pragma unroll
        for (int w = NW - 1; w >= 0; w--) {
            const int l = q + 1 - 64 * w;  // bits from l
            const u64 x = l <= 0 ? a[w] : l < 64 ? a[w] & (~0ULL << l) : 0ULL;
            if (x) p = 64 * w + __ffsll((long long)x) - 1;
        }
        return p;
    };
    u64 any = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        bool close = false;
        if (keep[w]) {
            const int p = before(gl + 64 * w);
            if (p >= 0) {
                const int jp = sperm[p];
                const double zp = sz[jp], t = dw[w] - sD[jp];
                close = fabs(t * zw[w] * zp) <= tol * (zw[w] * zw[w] + zp * zp);
            }
        }
        f[w] = (__ballot(close) & gmask) >> gbase;
        any |= f[w];
    }
    int nrot = 0;
    if (any) {
        if (gl == 0) {
            int q = next(f, -1), p = before(q);
            while (q >= 0) {
                const int j = sperm[q], prev = sperm[p];
                const double zj = sz[j], dj = sD[j], zp = sz[prev], dp = sD[prev];
                const double t = dj - dp, t2 = zj * zj + zp * zp;
                // |t c s| <= tol with c = zj/tau, s = -zp/tau, tau^2 = t2
                if (fabs(t * zj * zp) <= tol * t2) {
                    const double ta = sqrt(t2);
                    const double c = zj / ta, sn = -zp / ta;
                    sz[prev] = 0.0;
                    sD[prev] = dp * c * c + dj * sn * sn;
                    sz[j] = ta;
                    sD[j] = dp * sn * sn + dj * c * c;
                    ra[nrot] = prev;
                    rb[nrot] = j;
                    rc[nrot] = c;
                    rs[nrot] = sn;
                    nrot++;
#pragma unroll
                    for (int w = 0; w < NW; w++)
                        if (p >> 6 == w) r[w] |= 1ULL << (p & 63);
                    // the combined entry against the next one
                    p = q;
                    q = next(m, q);
                } else {
                    q = next(f, q);
                    if (q >= 0) p = before(q);
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int w = 0; w < NW; w++) r[w] = __shfl(r[w], 0, GL);
    }
    int c0 = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        const u64 nw = m[w] & ~r[w];
        if ((nw >> gl) & 1) {
            const int pos = c0 + __popcll(nw & below);
            snd[pos] = jw[w];
            sdl[pos] = sD[jw[w]];
            szl[pos] = sz[jw[w]];
        }
        c0 += __popcll(nw);
    }
    Kn_out = c0;
    nrot_out = nrot;
}

// Secular equation 1/rho + sum_j zl_j^2 / (dl_j - lambda) = 0: root i of Kn, in
// (dl_i, dl_{i+1}) (the last one in (dl_K-1, dl_K-1 + rho |z|^2)), as tau from
// the nearer pole org, by L lanes (lane sub of them).  Two poles: the root of the
// quadratic, no iteration.  Bound by an iteration's chain, so a lane keeps its M
// poles and weights in registers (padded with weight 0 at 1e300) and runs
// straight-line code: no branch on a root's position, one reciprocal and one
// square root a step.
template <int L, int M>
__device__ __forceinline__ void secular_root(int i, int Kn, int sub, double rho,
                                             const double *dl, const double *zl, int &org,
                                             double &tau, int &it) {
    it = 0;
    if (Kn == 1) {
        org = 0;
        tau = rho * zl[0] * zl[0];
        return;
    }
    if (Kn == 2) {
        // the roots of the quadratic, each from its nearer pole
        const double rinv = 1.0 / rho, gap = dl[1] - dl[0];
        const double z02 = zl[0] * zl[0], z12 = zl[1] * zl[1];
        if (i == 0) {
            // the sign of the secular function at the midpoint picks the nearer pole
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
        return;
    }
    const double rinv = rcp_nr(rho);
    const bool last = i == Kn - 1;
    const int i1 = last ? i : i + 1;
    const double di = dl[i], di1 = dl[i1];
    const double zi2 = zl[i] * zl[i], zi12 = zl[i1] * zl[i1];
    const double gap = di1 - di, mid = 0.5 * gap;
    // this lane's poles (from pole i) and weights, the latter apart for the
    // poles up to i (psi) and beyond (phi)
    double dj[M], zp[M], zq[M];
    double zz = 0.0, wm = 0.0;
#pragma unroll
    for (int m = 0; m < M; m++) {
        const int j = sub + m * L;
        const bool in = j < Kn;
        const double z = in ? zl[in ? j : 0] : 0.0;
        const double z2 = z * z;
        dj[m] = in ? dl[in ? j : 0] - di : 1e300;
        zp[m] = j <= i ? z2 : 0.0;
        zq[m] = j <= i ? 0.0 : z2;
        zz += z2;
        // w at the midpoint (the last root has none)
        wm = fma(z2, rcp_nr(last ? 1.0 : dj[m] - mid), wm);
    }
    zz = grp_sum<L>(zz);
    wm = grp_sum<L>(wm) + rinv;
    double tlo, thi;
    org = i;
    if (last) {
        tlo = 0.0;
        thi = rho * zz * (1.0 + 8.0 * EPSU) + 0x1.0p-1000;
        tau = 0.5 * thi;
    } else {
        // the quadratic through the poles i and i+1 with the rest of w at the
        // midpoint (initial guess of LAPACK's dlaed4)
        const bool up = !(wm >= 0.0);  // nearer to pole i+1
        const double c0 = wm + (zi2 - zi12) * rcp_nr(mid);
        if (up) org = i1;
        tlo = up ? -(gap - mid) : 0.0;
        thi = up ? 0.0 : mid;
        // lower pole: c0 t^2 - a t + bq = 0; upper: c0 t^2 + a t - bq = 0
        const double a = c0 * gap + (up ? -(zi2 + zi12) : zi2 + zi12);
        const double bq = (up ? zi12 : zi2) * gap;
        const double sq = sqrt_pos(fabs(fma(a, a, (up ? 4.0 : -4.0) * bq * c0)));
        const bool div = up ? a < 0.0 : a > 0.0;  // divide by a +- sq
        const double num = div ? 2.0 * bq : (up ? -(a + sq) : a - sq);
        const double den = div ? (up ? a - sq : a + sq) : 2.0 * c0;
        const double t0 = num * rcp_nr(den);
        tau = (t0 > tlo && t0 < thi) ? t0 : 0.5 * (tlo + thi);
    }
    // poles from the origin: dl - dl[org] (differences of the stored poles, as
    // where the roots are used)
    const double dorg = dl[org];
#pragma unroll
    for (int m = 0; m < M; m++) {
        const int j = sub + m * L;
        if (j < Kn) dj[m] = dl[j] - dorg;
    }
    const double ei = di - dorg, ei1 = di1 - dorg;
    for (it = 0; it < 100; it++) {
        double psi = 0.0, dpsi = 0.0, phi = 0.0, dphi = 0.0;
#pragma unroll
        for (int m = 0; m < M; m++) {
            const double r = rcp_nr(dj[m] - tau);
            const double tp = zp[m] * r, tq = zq[m] * r;
            psi += tp;
            phi += tq;
            dpsi = fma(tp, r, dpsi);
            dphi = fma(tq, r, dphi);
        }
        psi = grp_sum<L>(psi);
        dpsi = grp_sum<L>(dpsi);
        phi = grp_sum<L>(phi);
        dphi = grp_sum<L>(dphi);
        const double w = rinv + psi + phi;
        if (w == 0.0) break;
        if (w < 0.0) tlo = tau;
        else thi = tau;
        // rounding bound of w: LAPACK's dlaed4 adds the running partial sums, at
        // most Kn times the sum of |terms|
        const double errm =
            (8.0 + Kn) * (phi - psi) + 2.0 * rinv + 3.0 * fabs(tau) * (dpsi + dphi);
        if (fabs(w) <= EPSU * errm) break;
        // the step's quotient by the hardware reciprocal and the square root by
        // its estimate, with Newton steps: the step only steers the iteration,
        // whose stopping test is on w, and a step outside the bracket (or not a
        // number) falls back to bisection below
        const double Di = ei - tau, Di1 = ei1 - tau;
        const double c = w - Di * dpsi - Di1 * dphi;
        const double a = (Di + Di1) * w - Di * Di1 * (dpsi + dphi);
        const double bq = Di * Di1 * w;
        const double sq = sqrt_pos(fabs(fma(a, a, -4.0 * bq * c)));
        const bool neg = a <= 0.0;
        double num = neg ? a - sq : 2.0 * bq, den = neg ? 2.0 * c : a + sq;
        if (last) {  // the last pole's own term and a constant: Di + Di^2 dpsi / den
            den = w - Di * dpsi;
            num = den > 0.0 ? Di * w : NAN;
        } else if (c == 0.0) {
            num = bq;
            den = a;
        }
        double eta = num * rcp_nr(den);
        if (w * eta >= 0.0) eta = -w * rcp_nr(dpsi + dphi);
        double tn = tau + eta;
        if (!(tn > tlo && tn < thi)) tn = 0.5 * (tlo + thi);
        if (tn == tau) break;
        tau = tn;
    }
}

// Gu-Eisenstat z from the computed roots, entry q by L lanes:
// zhat_q^2 = (lambda_K-1 - d_q)/rho * prod_{i<q} (lambda_i - d_q)/(d_i - d_q)
//            * prod_{q<=i<K-1} (lambda_i - d_q)/(d_{i+1} - d_q),
// every factor in (0, 1) except the first (dorg: the roots' origins, lambda_i =
// dorg_i + tau_i).
template <int L>
__device__ __forceinline__ double zhat_entry(int q, int Kn, int sub, double rho, const double *dl,
                                             const double *dorg, const double *tau, double zq) {
    const double dq = dl[q];
    double prod = 1.0;
#pragma unroll 4
    for (int i = sub; i < Kn; i += L) {
        const double num = (dorg[i] - dq) + tau[i];
        const double dd = dl[i + (i >= q && i + 1 < Kn)] - dq;
        prod *= num * rcp_nr(i + 1 == Kn ? rho : dd);
    }
    prod = grp_prod<L>(prod);
    return copysign(sqrt(fmax(prod, 0.0)), zq);
}

// What k_dc_roots leaves for k_dc_vecs: per block of a level (index lo + .) the
// non-deflated poles, weights, roots and deflating rotations, in block-local
// column numbers; kn < 0: the block was not merged.
struct DcState {
    double *dl, *zl, *tau, *dorg, *rc, *rs, *rho;
    int *snd, *ra, *rb, *kn, *nrot, *iters;
};

// The merges of four to smax <= 32 rows, workgroup b on rows and columns 32 b ...
// Z's columns are written whole (zero outside the block).
constexpr int DCL = 32, DCP = 33;
__global__ __launch_bounds__(256) void k_dc_leaf(int n, const double *__restrict__ dd,
                                                 const double *__restrict__ ee,
                                                 double *__restrict__ Z, double *__restrict__ lam,
                                                 int smax, int *iters) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int b0 = DCL * blockIdx.x, nb = min(DCL, n - b0);
    __shared__ double Zs[DCL * DCP], ums[DCL * DCP];  // Z[r + DCP j]; U[q][i] at q DCP + i
    __shared__ double sD[DCL], sz[DCL], sdl[DCL], szl[DCL], stau[DCL], sdo[DCL], szh[DCL], sinv[DCL],
        rc[DCL], rs[DCL], srho[DCL];
    __shared__ int sperm[DCL], snd[DCL], ra[DCL], rb[DCL], sKn[DCL], sNrot[DCL];
    __shared__ int s_iters;
    if (tid == 0) s_iters = 0;
    for (int e = tid; e < DCL * DCL; e += 256) Zs[(e & 31) + DCP * (e >> 5)] = (e & 31) == (e >> 5);
    lds_sync();
    // Leaves of two rows (of one if even those are left to the top merge), torn
    // off their neighbours: the 2 x 2 blocks by their Jacobi rotation.
    if (tid < DCL && b0 + tid < n) {
        const int i = b0 + tid;
        const bool two = smax >= 2, pair = two && (tid ^ 1) < nb;
        auto leaf_d = [&](int q) {
            double x = dd[q];
            if (q > 0 && !(two && (q & 1))) x -= fabs(ee[q - 1]);
            if (q + 1 < n && !(two && !(q & 1))) x -= fabs(ee[q]);
            return x;
        };
        const double x = leaf_d(i);
        sD[tid] = x;
        if (pair && ee[i & ~1] != 0.0) {
            const double y = leaf_d(i ^ 1), off = ee[i & ~1];
            const double a = (i & 1) ? y : x, b = (i & 1) ? x : y;
            const double th = (b - a) / (2.0 * off);
            const double t = copysign(1.0 / (fabs(th) + sqrt(1.0 + th * th)), th);
            const double c = 1.0 / sqrt(1.0 + t * t), sn = t * c;
            // columns (c, -s) for a - t e and (s, c) for b + t e
            sD[tid] = (i & 1) ? b + t * off : a - t * off;
            Zs[(tid & ~1) + DCP * tid] = (i & 1) ? sn : c;
            Zs[(tid | 1) + DCP * tid] = (i & 1) ? c : -sn;
        }
    }
    lds_sync();
    for (int s = 4; s <= smax && s / 2 < nb; s *= 2) {
        const int ls = __builtin_ctz(s);
        const int nblk = (nb + s - 1) >> ls;
        // z and the ascending order of the eigenvalues of each block, the rank
        // of entry j counted by eight lanes (ties by index)
        {
            const int j = tid >> 3, sub = tid & 7;
            const int lo = (j >> ls) << ls, hi = min(lo + s, nb), m = lo + s / 2;
            if (j < nb && m < hi) {
                if (sub == 0) {
                    const double sg = (ee[b0 + m - 1] >= 0.0) ? 1.0 : -1.0;
                    sz[j] = (j < m ? Zs[(m - 1) + DCP * j] : sg * Zs[m + DCP * j]) * M_SQRT1_2;
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
        lds_sync();
        {
            const int b = tid >> ls, gl = tid & (s - 1), lo = b << ls;
            if (b < nblk) {
                const int hi = min(lo + s, nb), m = lo + s / 2;
                int Kn = -1, nrot = 0;
                double rho = 0.0;
                if (m < hi) {
                    rho = 2.0 * fabs(ee[b0 + m - 1]);
                    Kn = 0;
                    if (rho != 0.0)
                        deflate<1>(s, gl, lane - gl, hi - lo, rho, sperm + lo, sz, sD,
                                       snd + lo, sdl + lo, szl + lo, ra + lo, rb + lo, rc + lo,
                                       rs + lo, Kn, nrot);
                }
                if (gl == 0) {
                    srho[b] = rho;
                    sKn[b] = Kn;
                    sNrot[b] = nrot;
                }
            }
        }
        lds_sync();
        // the deflating rotations on the rows of Z (column pairs, in order)
        if (tid < nb) {
            const int b = tid >> ls, lo = b << ls;
            const int nrot = sKn[b] < 0 ? 0 : sNrot[b];
            for (int t = 0; t < nrot; t++) {
                const int ia = tid + DCP * ra[lo + t], ib = tid + DCP * rb[lo + t];
                const double qa = Zs[ia], qb = Zs[ib], c = rc[lo + t], sn = rs[lo + t];
                Zs[ia] = c * qa + sn * qb;
                Zs[ib] = c * qb - sn * qa;
            }
        }
        auto roots = [&](auto Ltag, auto Mtag) {
            constexpr int L = decltype(Ltag)::value, M = decltype(Mtag)::value;
            const int ri = tid / L, sub = tid & (L - 1);
            const int b = ri >> ls, lo = b << ls, i = ri - lo;
            const int Kn = ri < nb ? sKn[b] : 0;
            if (i < Kn) {
                int org, it;
                double tau;
                secular_root<L, M>(i, Kn, sub, srho[b], sdl + lo, szl + lo, org, tau, it);
                if (sub == 0) {
                    sdo[lo + i] = sdl[lo + org];
                    stau[lo + i] = tau;
                    if (it > 0) atomicMax(&s_iters, it);
                }
            }
        };
        if (s == 4) roots(std::integral_constant<int, 4>{}, std::integral_constant<int, 1>{});
        else if (s == 8) roots(std::integral_constant<int, 8>{}, std::integral_constant<int, 1>{});
        else if (s == 16) roots(std::integral_constant<int, 8>{}, std::integral_constant<int, 2>{});
        else roots(std::integral_constant<int, 8>{}, std::integral_constant<int, 4>{});
        lds_sync();
        {
            const int jq = tid >> 3, sub = tid & 7, b = jq >> ls, lo = b << ls, q = jq - lo;
            const int Kn = jq < nb ? sKn[b] : 0;
            if (q < Kn) {
                const double z = zhat_entry<8>(q, Kn, sub, srho[b], sdl + lo, sdo + lo, stau + lo,
                                               szl[jq]);
                if (sub == 0) szh[jq] = z;
            }
        }
        lds_sync();
        // eigenvectors of the rank-one updates, and their norms
        for (int t = tid; t < nblk << (2 * ls); t += 256) {
            const int jq = t >> ls, i = t & (s - 1), b = jq >> ls, lo = b << ls, q = jq - lo;
            const int Kn = sKn[b];
            if (q < Kn && i < Kn)
                ums[jq * DCP + i] =
                    szh[jq] * rcp_nr((sdl[jq] - sdo[lo + i]) - stau[lo + i]);
        }
        lds_sync();
        {
            const int ci = tid >> 3, sub = tid & 7, b = ci >> ls, lo = b << ls, i = ci - lo;
            const int Kn = ci < nb ? sKn[b] : 0;
            if (i < Kn) {
                double ss = 0.0;
                for (int q = sub; q < Kn; q += 8) {
                    const double u = ums[(lo + q) * DCP + i];
                    ss = fma(u, u, ss);
                }
                ss = oct_sum(ss);
                if (sub == 0) sinv[ci] = 1.0 / sqrt(ss);
            }
        }
        lds_sync();
        // Z[:, snd_i] = Z[:, snd] u_i over the block's rows, read by every thread
        // before any writes.  Blocks of 16 and 32: 16 x 16 tiles on the matrix
        // cores, issued as (U^T)(Z^T) so that a tile's lanes hold 16 consecutive
        // rows of one column; smaller blocks: a thread an entry.
        if (s >= 16) {
            const int lt = ls - 4, tiles = nblk << (2 * lt);
            const int b = wv >> (2 * lt), rem = wv & ((1 << (2 * lt)) - 1);
            const int rb0 = (rem >> lt) * 16, cb = (rem & ((1 << lt) - 1)) * 16;
            const int lo = b << ls, Kn = wv < tiles ? sKn[b] : 0;
            f64x4 acc = {0.0, 0.0, 0.0, 0.0};
            for (int k0 = 0; k0 < Kn; k0 += 4) {
                const int q = k0 + (lane >> 4);
                const bool kin = q < Kn;
                const int qi = kin ? q : 0;
                const double ua = kin && cb + (lane & 15) < Kn
                                      ? ums[(lo + qi) * DCP + cb + (lane & 15)] : 0.0;
                const double zb = kin ? Zs[lo + rb0 + (lane & 15) + DCP * snd[lo + qi]] : 0.0;
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(ua, zb, acc, 0, 0, 0);
            }
            lds_sync();
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int col = cb + (lane >> 4) + 4 * v;
                if (col < Kn)
                    Zs[lo + rb0 + (lane & 15) + DCP * snd[lo + col]] = acc[v] * sinv[lo + col];
            }
        } else {
            const int r = tid & 31, i = tid >> 5, b = r >> ls, lo = b << ls;
            const int Kn = r < nb ? sKn[b] : 0;
            double acc = 0.0;
            if (i < Kn)
                for (int q = 0; q < Kn; q++)
                    acc = fma(Zs[r + DCP * snd[lo + q]], ums[(lo + q) * DCP + i], acc);
            lds_sync();
            if (i < Kn) Zs[r + DCP * snd[lo + i]] = acc * sinv[lo + i];
        }
        if (tid < nb) {
            const int b = tid >> ls, lo = b << ls, i = tid - lo;
            if (i < sKn[b]) sD[snd[tid]] = sdo[tid] + stau[tid];
        }
        lds_sync();
    }
    for (int j = tid >> 5; j < nb; j += 8)
        for (int r = tid & 31; r < n; r += 32)
            Z[r + (long)(b0 + j) * n] = (r >= b0 && r < b0 + nb) ? Zs[r - b0 + DCP * j] : 0.0;
    if (tid < nb) lam[b0 + tid] = sD[tid];
    if (tid == 0) {
        iters[blockIdx.x] = s_iters;
        if (blockIdx.x == 0) iters[8] = 0;
    }
}

// One merge of blocks of s <= S rows, first half: workgroup g of a block's
// ceil(s/16) finds roots 16 g .. 16 g + 15, L lanes a root; the block's
// first also leaves the deflation's outcome.
template <int S, int L>
__global__ __launch_bounds__(16 * L) void k_dc_roots(int n, int s, const double *__restrict__ ee,
                                                  const double *__restrict__ Z,
                                                  const double *__restrict__ lam_in,
                                                  double *__restrict__ lam_out, DcState st) {
    const int tid = threadIdx.x;
    const int gpb = (s + 15) >> 4, b = blockIdx.x / gpb, g = blockIdx.x - b * gpb;
    const int lo = b * s, hi = min(lo + s, n), m = lo + s / 2, K = hi - lo;
    __shared__ double sD[S], sz[S], sdl[S], szl[S], rc[S], rs[S];
    __shared__ int sperm[S], snd[S], ra[S], rb[S], sflag[S];
    __shared__ int s_kn, s_nrot;
    if (m >= hi) {  // nothing to merge with
        if (g == 0) {
            if (tid < K) lam_out[lo + tid] = lam_in[lo + tid];
            if (tid == 0) {
                st.kn[b] = -1;
                st.nrot[b] = 0;
            }
        }
        return;
    }
    const double bt = ee[m - 1], rho = 2.0 * fabs(bt);
    if (tid < K) {
        const int j = lo + tid;
        sD[tid] = lam_in[j];
        sz[tid] = (j < m ? Z[(m - 1) + (long)j * n]
                         : (bt >= 0.0 ? 1.0 : -1.0) * Z[m + (long)j * n]) * M_SQRT1_2;
        sflag[tid] = 0;
    }
    __syncthreads();
    {
        constexpr int LP = 16 * L / S > 8 ? 8 : 16 * L / S;
        const int j = tid / LP, sub = tid & (LP - 1);
        if (j < K) {
            const double dj = sD[j];
            int pos = 0;
#pragma unroll 8
            for (int q = sub; q < K; q += LP) {
                const double dq = sD[q];
                pos += (dq < dj) || (dq == dj && q < j);
            }
            pos = (int)grp_sum<LP>((double)pos);
            if (sub == 0) sperm[pos] = j;
        }
    }
    __syncthreads();
    if (tid < 64) {
        int Kn = 0, nrot = 0;
        if (rho != 0.0)
            deflate<(S + 63) / 64>(64, tid, 0, K, rho, sperm, sz, sD, snd, sdl, szl, ra, rb, rc, rs, Kn,
                              nrot);
        if (tid == 0) {
            s_kn = Kn;
            s_nrot = nrot;
        }
    }
    __syncthreads();
    const int Kn = s_kn;
    const int i = 16 * g + tid / L, sub = tid & (L - 1);
    if (i < Kn) {
        int org, it;
        double tau;
        secular_root<L, S / L>(i, Kn, sub, rho, sdl, szl, org, tau, it);
        if (sub == 0) {
            st.dorg[lo + i] = sdl[org];
            st.tau[lo + i] = tau;
            lam_out[lo + snd[i]] = sdl[org] + tau;
            if (it > 0) atomicMax(st.iters + 8, it);
        }
    }
    if (g != 0) return;
    if (tid < Kn) sflag[snd[tid]] = 1;
    __syncthreads();
    if (tid < K && !sflag[tid]) lam_out[lo + tid] = sD[tid];
    if (tid < Kn) {
        st.dl[lo + tid] = sdl[tid];
        st.zl[lo + tid] = szl[tid];
        st.snd[lo + tid] = snd[tid];
    }
    if (tid < s_nrot) {
        st.ra[lo + tid] = ra[tid];
        st.rb[lo + tid] = rb[tid];
        st.rc[lo + tid] = rc[tid];
        st.rs[lo + tid] = rs[tid];
    }
    if (tid == 0) {
        st.rho[b] = rho;
        st.kn[b] = Kn;
        st.nrot[b] = s_nrot;
    }
}

// Second half, of a merge below the top: workgroup g of a block forms the new
// columns of Z at roots 16 g .. 16 g + 15 and copies the deflated ones among the
// block's columns 16 g .. 16 g + 15, from Zin into Zout (whole columns, zero
// outside the block).  A workgroup takes 64 rows of the block's.
template <int S>
__global__ __launch_bounds__(256) void k_dc_vecs(int n, int s, const double *__restrict__ Zin,
                                                 double *__restrict__ Zout, DcState st) {
    constexpr int LD = 65, NCH = S / 64;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int gpb = (s + 15) >> 4, r0 = 64 * (blockIdx.x % NCH), bg = blockIdx.x / NCH;
    const int b = bg / gpb, g = bg - b * gpb;
    const int lo = b * s, hi = min(lo + s, n), K = hi - lo;
    extern __shared__ double vlds[];
    double *Zs = vlds;          // Zs[r - r0 + LD j]
    double *us = Zs + S * LD;   // U[q][c] of the 16 own columns
    __shared__ double sdl[S], szl[S], stau[S], sdo[S], szh[S], sinv[16], rc[S], rs[S];
    __shared__ int snd[S], sflag[S], ra[S], rb[S];
    const int Kn = max(st.kn[b], 0), nrot = Kn > 0 || st.kn[b] == 0 ? st.nrot[b] : 0;
    const double rho = Kn > 0 ? st.rho[b] : 0.0;
    {
        double z[S / 4];
#pragma unroll
        for (int t = 0; t < S / 4; t++) {
            const int j = wv + 4 * t;
            z[t] = (r0 + lane < K && j < K) ? Zin[lo + r0 + lane + (long)(lo + j) * n] : 0.0;
        }
#pragma unroll
        for (int t = 0; t < S / 4; t++) Zs[lane + LD * (wv + 4 * t)] = z[t];
    }
    if (tid < S) sflag[tid] = 0;
    if (tid < Kn) {
        sdl[tid] = st.dl[lo + tid];
        szl[tid] = st.zl[lo + tid];
        stau[tid] = st.tau[lo + tid];
        snd[tid] = st.snd[lo + tid];
        sdo[tid] = st.dorg[lo + tid];
    }
    if (tid < nrot) {
        ra[tid] = st.ra[lo + tid];
        rb[tid] = st.rb[lo + tid];
        rc[tid] = st.rc[lo + tid];
        rs[tid] = st.rs[lo + tid];
    }
    __syncthreads();
    if (tid < Kn) sflag[snd[tid]] = 1;
    if (tid >= 192) {  // the deflating rotations, a thread a row
        const int r = tid - 192;
        for (int t = 0; t < nrot; t++) {
            const int ia = r + LD * ra[t], ib = r + LD * rb[t];
            const double qa = Zs[ia], qb = Zs[ib], c = rc[t], sn = rs[t];
            Zs[ia] = c * qa + sn * qb;
            Zs[ib] = c * qb - sn * qa;
        }
    }
    {
        constexpr int LP = 256 / S;
        const int q = tid / LP, sub = tid & (LP - 1);
        if (q < Kn) {
            const double z = zhat_entry<LP>(q, Kn, sub, rho, sdl, sdo, stau, szl[q]);
            if (sub == 0) szh[q] = z;
        }
    }
    __syncthreads();
    for (int e = tid; e < S * 16; e += 256) {
        const int q = e >> 4, c = e & 15, i = 16 * g + c;
        us[q * 17 + c] = (q < Kn && i < Kn)
                             ? szh[q] * rcp_nr((sdl[q] - sdo[i]) - stau[i]) : 0.0;
    }
    __syncthreads();
    {
        const int c = tid >> 4, sub = tid & 15;
        double ss = 0.0;
#pragma unroll
        for (int m = 0; m < S / 16; m++) {
            const double u = us[(sub + 16 * m) * 17 + c];
            ss = fma(u, u, ss);
        }
        ss = grp_sum<16>(ss);
        if (sub == 0) sinv[c] = 16 * g + c < Kn ? 1.0 / sqrt(ss) : 0.0;
    }
    __syncthreads();
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < Kn; k0 += 4) {
        const int q = k0 + (lane >> 4);
        const bool kin = q < Kn;
        const double ua = us[q * 17 + (lane & 15)];  // zero beyond Kn
        const double zb = kin ? Zs[16 * wv + (lane & 15) + LD * snd[kin ? q : 0]] : 0.0;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(ua, zb, acc, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int c = (lane >> 4) + 4 * v, i = 16 * g + c, r = r0 + 16 * wv + (lane & 15);
        if (i < Kn && r < K) Zout[lo + r + (long)(lo + snd[i]) * n] = acc[v] * sinv[c];
    }
    // deflated columns, and the zeros outside the block of every column written
    for (int c = wv; c < 16; c += 4) {
        const int i = 16 * g + c;
        if (i < K && !sflag[i] && r0 + lane < K)
            Zout[lo + r0 + lane + (long)(lo + i) * n] = Zs[lane + LD * i];
        if (r0 != 0) continue;
        for (int r = lane; r < n; r += 64)
            if (r < lo || r >= hi) {
                if (i < Kn) Zout[r + (long)(lo + snd[i]) * n] = 0.0;
                if (i < K && !sflag[i]) Zout[r + (long)(lo + i) * n] = 0.0;
            }
    }
}

// Second half, of the top merge: workgroup g < ceil(n/16) forms columns 16 g ..
// of Um; the last one orders the eigenvalues (lam, by Z column) and decides.
template <int S>
__global__ __launch_bounds__(256) void k_dc_top(int n, DcState st, const double *__restrict__ lam,
                                                const int *__restrict__ eexp,
                                                double *__restrict__ Um, int *__restrict__ colidx,
                                                double *__restrict__ sig, int *__restrict__ iout,
                                                double *__restrict__ dinfo, double delta, int cap,
                                                double budget) {
    constexpr int LD = S + 1;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int g = blockIdx.x;
    __shared__ double um[16 * LD];  // own columns, um[r + LD c]
    __shared__ double sdl[S], szl[S], stau[S], sdo[S], szh[S], slam[S], rc[S], rs[S];
    __shared__ int snd[S], sflag[S], spos[S], scm[S], ra[S], rb[S];
    const int Kn = max(st.kn[0], 0), nrot = st.nrot[0];
    if (tid < n) sflag[tid] = 0;
    if (tid < Kn) {
        sdl[tid] = st.dl[tid];
        szl[tid] = st.zl[tid];
        stau[tid] = st.tau[tid];
        snd[tid] = st.snd[tid];
        sdo[tid] = st.dorg[tid];
    }
    if (tid < nrot) {
        ra[tid] = st.ra[tid];
        rb[tid] = st.rb[tid];
        rc[tid] = st.rc[tid];
        rs[tid] = st.rs[tid];
    }
    __syncthreads();
    if (tid < Kn) {
        sflag[snd[tid]] = 1;
        scm[tid] = snd[tid];
        spos[snd[tid]] = tid;
    }
    __syncthreads();
    // column c's pole: Z column scm[c]; Z column j's column: spos[j]
    if (tid < n && !sflag[tid]) {
        int pos = Kn;
#pragma unroll 8
        for (int q = 0; q < tid; q++) pos += !sflag[q];
        scm[pos] = tid;
        spos[tid] = pos;
    }
    if (g + 1 < (int)gridDim.x) {
        const double rho = Kn > 0 ? st.rho[0] : 0.0;
        constexpr int LP = 256 / S > 8 ? 8 : 256 / S;
        const int q = tid / LP, sub = tid & (LP - 1);
        if (q < Kn) {
            const double z = zhat_entry<LP>(q, Kn, sub, rho, sdl, sdo, stau, szl[q]);
            if (sub == 0) szh[q] = z;
        }
        __syncthreads();
        {
            const int c = tid >> 4, sb = tid & 15, i = 16 * g + c;
            if (i < Kn) {
                const double li = sdo[i], ti = stau[i];
                double u[S / 16 > 0 ? S / 16 : 1];
                double ss = 0.0;
#pragma unroll
                for (int m = 0; m < S / 16; m++) {
                    const int r = sb + 16 * m;
                    const int p = r < n ? spos[r] : S;
                    u[m] = p < Kn ? szh[p] * rcp_nr((sdl[p] - li) - ti) : 0.0;
                    ss = fma(u[m], u[m], ss);
                }
                ss = grp_sum<16>(ss);
                const double iv = 1.0 / sqrt(ss);
#pragma unroll
                for (int m = 0; m < S / 16; m++) um[sb + 16 * m + LD * c] = u[m] * iv;
            } else if (i < n) {
                const int j = scm[i];
#pragma unroll
                for (int m = 0; m < S / 16; m++) um[sb + 16 * m + LD * c] = (sb + 16 * m == j) ? 1.0 : 0.0;
            }
        }
        __syncthreads();
        // Z G_0 ... G_{k-1} Um = Z (G_0 (... (G_{k-1} Um))): each rotation
        // of Z's columns (a, b) acts on Um's rows a and b, last first
        if (nrot > 0) {
            if (tid < 16 && 16 * g + tid < n) {
                double *col = um + LD * tid;
                for (int t = nrot - 1; t >= 0; t--) {
                    const int a = ra[t], b = rb[t];
                    const double c = rc[t], sn = rs[t];
                    const double ua = col[a], ub = col[b];
                    col[a] = c * ua - sn * ub;
                    col[b] = sn * ua + c * ub;
                }
            }
            __syncthreads();
        }
        for (int c = wv; c < 16; c += 4)
            for (int r = lane; r < n; r += 64)
                if (16 * g + c < n) Um[r + (long)(16 * g + c) * n] = um[r + LD * c];
        return;
    }
    __syncthreads();
    // final order (descending), dropped tail, numerical rank, tail rule
    if (tid < n) slam[tid] = lam[scm[tid]];
    __syncthreads();
    {
        // rank of column c in descending order
        constexpr int LP = 256 / S > 8 ? 8 : 256 / S;
        const int c = tid / LP, sub = tid & (LP - 1);
        if (c < n) {
            const double lc = slam[c];
            int pos = 0;
#pragma unroll 8
            for (int q = sub; q < n; q += LP) {
                const double lq = slam[q];
                pos += (lq > lc) || (lq == lc && q < c);
            }
            pos = (int)grp_sum<LP>((double)pos);
            if (sub == 0) {
                colidx[pos] = c;
                sdl[pos] = lc;  // sdl reused: eigenvalues in descending order (scaled)
            }
        }
    }
    __syncthreads();
    const bool finite = *eexp != EIG_NONFINITE;
    const int es = finite ? *eexp : 0;
    // Wave 0 holds the descending values lane + 64 w and decides:
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
    __shared__ int s_keep;
    if (wv == 0) {
        constexpr int NW = (S + 63) / 64;
        double h[NW], suf[NW];
#pragma unroll
        for (int w = 0; w < NW; w++)
            h[w] = lane + 64 * w < n ? fmax(sdl[lane + 64 * w < S ? lane + 64 * w : 0], 0.0) : 0.0;
        const double lmax = readlane_d(h[0], 0);
        const double lim = budget * lmax;
        // suffix sums of x over all words, into suf
        auto suffix = [&](const double(&x)[NW]) {
            double rest = 0.0;
#pragma unroll
            for (int w = NW - 1; w >= 0; w--) {
                suf[w] = w == NW - 1 ? suffix_sum(x[w]) : suffix_sum(x[w]) + rest;
                rest = readlane_d(suf[w], 0);
            }
        };
        suffix(h);
        int keep = n;
        double cum = 0.0;
#pragma unroll
        for (int w = NW - 1; w >= 0; w--) {
            const unsigned long long k =
                __ballot(lane + 64 * w < n && suf[w] <= lim && h[w] < lmax);
            if (k) {
                keep = 64 * w + __ffsll((long long)k) - 1;
                cum = readlane_d(suf[w], keep & 63);
            }
        }
        const double thr2 = (double)n * EPSU * EPSU * lmax;  // (sqrt(n) u sigma_0)^2
        int numrank = 0;
        if (lmax > 0.0)
#pragma unroll
            for (int w = 0; w < NW; w++)
                numrank += __popcll(__ballot(lane + 64 * w < keep && h[w] > thr2));
        const double dl2 =
            (delta > 0.0) ? exp(2.0 * (log(delta) - (es / 2) * 0.6931471805599453)) : -1.0;
#pragma unroll
        for (int w = 0; w < NW; w++) h[w] = lane + 64 * w < numrank ? h[w] : 0.0;
        suffix(h);
        int rho = numrank;
#pragma unroll
        for (int w = NW - 1; w >= 0; w--) {
            const unsigned long long k = __ballot(lane + 64 * w < numrank && suf[w] < dl2);
            if (k) rho = 64 * w + __ffsll((long long)k) - 1;
        }
        if (rho > n) rho = n;
        if (rho > cap) rho = cap;
        if (rho < 1) rho = 1;
        if (lane == 0) {
            int it = st.iters[8];
            for (int q = 0; 32 * q < n; q++) it = max(it, st.iters[q]);
            iout[0] = numrank;
            iout[1] = rho;
            iout[2] = it;
            dinfo[5] = ldexp(cum, es);
            s_keep = keep;
        }
    }
    __syncthreads();
    const int keep = s_keep;
    if (tid < n)
        sig[tid] = !finite ? NAN : (tid < keep) ? ldexp(sqrt(fmax(sdl[tid], 0.0)), es / 2) : 0.0;
}

// ---- 3. back transformation -----------------------------------------------
// W = H_0 H_1 ... H_{n-3} Z, the reflectors applied last first.  Sixteen lanes (one DPP row) own a column, each holding the rows
// l, l+16, ..., so a reflector's dot product reduces inside the row; a
// workgroup of four waves owns 16 columns and stages the reflectors in LDS, `ch`
// at a time (all of them up to 128 rows).
template <int RPL>  // rows per lane
__global__ __launch_bounds__(256) void k_ormtr(int n, int ch, const double *__restrict__ Vh,
                                               const double *__restrict__ tau,
                                               const double *__restrict__ Z,
                                               double *__restrict__ W) {
    extern __shared__ double vs[];  // ch x n reflectors, then n taus
    const int tid = threadIdx.x;
    const int l = tid & 15;
    const int c = blockIdx.x * 16 + (tid >> 4);
    const bool live = c < n;  // rows of 16 lanes: uniform per DPP row
    const double *zc = Z + (long)(live ? c : 0) * n;
    double x[RPL];
#pragma unroll
    for (int m = 0; m < RPL; m++) {
        const int i = l + 16 * m;
        x[m] = (live && i < n) ? zc[i] : 0.0;
    }
    double *ts = vs + (long)ch * n;
    for (int i = tid; i < n; i += 256) ts[i] = tau[i];
    for (int k1 = n; k1 > 0; k1 -= ch) {  // reflectors kb .. k1 - 1
        const int kb = k1 > ch ? k1 - ch : 0;
        const long cnt = (long)(k1 - kb) * n;
        const double *src = Vh + (long)kb * n;
        if (k1 < n) __syncthreads();
        for (long e0 = tid; e0 < cnt; e0 += 4 * 256) {
            double v[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const long e = e0 + (long)u * 256;
                v[u] = (e < cnt) ? src[e] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const long e = e0 + (long)u * 256;
                if (e < cnt) vs[e] = v[u];
            }
        }
        __syncthreads();
        for (int k = min(k1 - 1, n - 3); k >= kb; k--) {
            const double tk = ts[k];
            if (tk == 0.0) continue;
            const double *v = vs + (long)(k - kb) * n;
            double vr[RPL];
            double d0 = 0.0, d1 = 0.0;
#pragma unroll
            for (int m = 0; m < RPL; m++) {
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
            for (int m = 0; m < RPL; m++) x[m] = fma(-dt, vr[m], x[m]);
        }
    }
    if (live)
#pragma unroll
        for (int m = 0; m < RPL; m++) {
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

constexpr int ORM_LDS_DOUBLES = 128 * 128 + 256;

void syev_attr() {
    static bool done = false;
    if (done) return;
    auto set = [](const void *f, int doubles) {
        HIPCHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     doubles * (int)sizeof(double)));
    };
    set((const void *)k_ormtr<8>, ORM_LDS_DOUBLES);
    set((const void *)k_ormtr<12>, ORM_LDS_DOUBLES);
    set((const void *)k_dc_vecs<128>, 128 * (65 + 17));
    done = true;
}

void launch_ormtr(int c, const double *Vh, const double *tau, const double *Z, double *W) {
    const double cc = (double)c * c;
    const int ch = c * c + c <= ORM_LDS_DOUBLES ? c : (ORM_LDS_DOUBLES - c) / c;
    const size_t shm = ((size_t)ch * c + c) * sizeof(double);
    if (c <= 128)
        PTT_LAUNCH_FB("syev_ormtr", 4.0 * cc * c, 8.0 * 3.0 * cc, k_ormtr<8>, dim3(cdiv(c, 16)),
                      dim3(256), shm, c, ch, Vh, tau, Z, W);
    else
        PTT_LAUNCH_FB("syev_ormtr", 4.0 * cc * c, 8.0 * 3.0 * cc, k_ormtr<12>, dim3(cdiv(c, 16)),
                      dim3(256), shm, c, ch, Vh, tau, Z, W);
}

// Workspace of one eigen-decomposition of order c: reflectors, Z twice (a merge
// below the top reads one and writes the other), the top update's matrix and the
// back-transformed vectors (c x c each), then tau, d, e, the poles twice and the
// state between a merge's launches.
constexpr size_t syev_ws_doubles(size_t c) { return 5 * c * c + 13 * c + 64; }

// Top merge and decisions (n <= S).
template <int S>
void launch_top(int n, int s, const double *e, const double *Z, const double *lam, double *lam2,
                const DcState &st, const int *ex, double *Um, int *colidx, double *sig, int *iout,
                double *dinfo, double delta, int cap, double budget) {
    constexpr int L = S > 64 ? 32 : 16;
    const double nn = (double)n;
    PTT_LAUNCH_FB("syev_roots", 60.0 * nn * nn, 8.0 * 4.0 * nn, (k_dc_roots<S, L>),
                  dim3(cdiv(s, 16)), dim3(16 * L), 0, n, s, e, Z, lam, lam2, st);
    PTT_LAUNCH_FB("syev_top", 10.0 * nn * nn, 8.0 * nn * nn, k_dc_top<S>, dim3(cdiv(n, 16) + 1),
                  dim3(256), 0, n, st, lam2, ex, Um, colidx, sig, iout, dinfo, delta, cap, budget);
}

// Tridiagonalisation, divide and conquer, back transformation W = Q Z, and
// U = W Um.  With the side stream on, the back transformation of more than 64 rows
// runs there beside the top merge (the merges below it leave Z final); the main stream waits for
// it before the product.
void syev_run(int c, const double *G, double *sig, double *U, long ldu, int *colidx, int *iout,
              double *dinfo, double delta, int cap, double budget, double *ws) {
    const size_t cc = (size_t)c * c;
    double *Vh = ws, *Z = Vh + cc, *Z2 = Z + cc, *Um = Z2 + cc, *W = Um + cc;
    double *tau = W + cc, *d = tau + c, *e = d + c, *lam = e + c, *lam2 = lam + c;
    DcState st;
    st.dl = lam2 + c;
    st.zl = st.dl + c;
    st.tau = st.zl + c;
    st.dorg = st.tau + c;
    st.rc = st.dorg + c;
    st.rs = st.rc + c;
    st.rho = st.rs + c;  // up to 4 blocks
    st.snd = (int *)(st.rho + 4);
    st.ra = st.snd + c;
    st.rb = st.ra + c;
    st.kn = st.rb + c;
    st.nrot = st.kn + 4;
    st.iters = st.nrot + 4;  // one per leaf workgroup (up to 8), then the larger merges'
    int *ex = st.iters + 10;
    syev_attr();
    const double n = (double)c;
    if (c <= 64)
        PTT_LAUNCH_FB("syev_sytrd", 4.0 * n * n * n / 3.0, 8.0 * n * n * 2.0, k_sytrd<64>, dim3(1),
                      dim3(4 * 64 + 64), 0, c, G, (long)c, Vh, tau, d, e, ex, dinfo);
    else if (c <= 128)
        PTT_LAUNCH_FB("syev_sytrd", 4.0 * n * n * n / 3.0, 8.0 * n * n * 2.0, k_sytrd<128>, dim3(1),
                      dim3(4 * 128 + 64), 0, c, G, (long)c, Vh, tau, d, e, ex, dinfo);
    else
        PTT_LAUNCH_FB("syev_sytrd", 4.0 * n * n * n / 3.0, 8.0 * n * n * 2.0, k_sytrd<192>, dim3(1),
                      dim3(2 * 192 + 64), 0, c, G, (long)c, Vh, tau, d, e, ex, dinfo);
    int top = 2;
    while (top < c) top *= 2;
    PTT_LAUNCH_FB("syev_leaf", 2.0 * 32.0 * 32.0 * n, 8.0 * n * n, k_dc_leaf, dim3(cdiv(c, DCL)),
                  dim3(256), 0, c, d, e, Z, lam, top / 2 < DCL ? top / 2 : DCL, st.iters);
    auto swap = [](double *&a, double *&b) {
        double *t = a;
        a = b;
        b = t;
    };
    if (top >= 128) {  // blocks of 64
        const int nb = (int)cdiv(c, 64);
        PTT_LAUNCH_FB("syev_roots", 60.0 * 64.0 * n, 8.0 * 4.0 * n, (k_dc_roots<64, 16>),
                      dim3(nb * 4), dim3(256), 0, c, 64, e, Z, lam, lam2, st);
        PTT_LAUNCH_FB("syev_vecs", 2.0 * 64.0 * 64.0 * n, 8.0 * 2.0 * n * n, k_dc_vecs<64>,
                      dim3(nb * 4), dim3(256), 64 * (65 + 17) * sizeof(double), c, 64, Z, Z2, st);
        swap(Z, Z2);
        swap(lam, lam2);
    }
    if (top == 256) {  // blocks of 128 (the second may hold no more than 64 rows)
        PTT_LAUNCH_FB("syev_roots", 60.0 * 128.0 * n, 8.0 * 4.0 * n, (k_dc_roots<128, 32>),
                      dim3(2 * 8), dim3(512), 0, c, 128, e, Z, lam, lam2, st);
        PTT_LAUNCH_FB("syev_vecs", 2.0 * 128.0 * 128.0 * n, 8.0 * 2.0 * n * n, k_dc_vecs<128>,
                      dim3(2 * 8 * 2), dim3(256), 128 * (65 + 17) * sizeof(double), c, 128, Z, Z2,
                      st);
        swap(Z, Z2);
        swap(lam, lam2);
    }
    // Up to 64 rows the back transformation (9 us at 32, 17 at 59) costs less than the
    // streams' events: roundings at 32 columns 3.64 -> 3.52 ms, at 59 3.75 -> 3.67.
    // At 128 it takes 40 us, beside 20 of the top merge.
    const bool side = ptt_hip_side_enabled() && c > 64;
    if (side) {
        ptt_hip_side_begin();
        launch_ormtr(c, Vh, tau, Z, W);
        ptt_hip_side_end(0);
    }
    if (top == 256)
        launch_top<EIG_NMAX>(c, top, e, Z, lam, lam2, st, ex, Um, colidx, sig, iout, dinfo, delta,
                             cap, budget);
    else if (top == 128)
        launch_top<128>(c, top, e, Z, lam, lam2, st, ex, Um, colidx, sig, iout, dinfo, delta, cap,
                        budget);
    else if (top == 64)
        launch_top<64>(c, top, e, Z, lam, lam2, st, ex, Um, colidx, sig, iout, dinfo, delta, cap,
                       budget);
    else
        launch_top<32>(c, top, e, Z, lam, lam2, st, ex, Um, colidx, sig, iout, dinfo, delta, cap,
                       budget);
    if (side) ptt_hip_side_wait(0);
    else launch_ormtr(c, Vh, tau, Z, W);
    ptt_hip_dgemm('N', 'N', c, c, c, 1.0, W, c, Um, c, 0.0, U, ldu);
}

// Fixed workspace of the entry point that allocates nothing: one copy per
// GPU, held until the process ends.  Host code reaches it only through the
// device address from hipGetSymbolAddress (the name is a host stand-in).
constexpr int NOALLOC_CMAX = 128;
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
