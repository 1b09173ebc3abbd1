// dense.hip -- small dense FP64 factorizations on one workgroup (gfx950).
//
// ptt_hip_chol_qr_factor: the r x r step of Cholesky-QR.  The Gram matrix is
// Jacobi-scaled (unit diagonal) so column scaling never costs accuracy, the
// factorization guards tiny pivots (the index is marked deficient: its row
// of R and column of R^-1 become zero, so A*T has a zero column there and
// A = (A*T)*R still holds to rounding), and the inverse is formed in place.
//
// ptt_hip_svd_jacobi: one-sided (Hestenes) Jacobi SVD with round-robin
// parallel pairing; each pair is owned by a lane group that reduces its
// three inner products with cross-lane shuffles.  Up to 56 columns that fit in
// the LDS of one CU (160 KB on gfx950) are rotated there by one wave or one
// workgroup; otherwise many workgroups take pairs of blocks of columns into LDS
// in turn, and columns too long for that stay in global memory.
// The reference's rank rule (pattac.c:468-481) is applied on the device.
#include "common.hpp"

#include <cmath>

using namespace ptt;

namespace {

constexpr int NT = 1024;
// Doubles of columns in the one-workgroup Jacobi's LDS (135 KB of the CU's 160).
constexpr int SVD_LDS_DOUBLES = 17280;
// Columns beyond which the Jacobi SVD runs over many workgroups.  Measured with
// V (us; flat spectrum, square): k = 48: 658 on one workgroup, 760 on many;
// 59: 942 / 826; 96: 1830 / 1315; 128: 2370 / 2030; 192: 37600 / 4140 (the
// columns of one workgroup are then in HBM).
constexpr int SVD_ONE_WG_MAX = 56;
constexpr int SVD_NT = 1024;  // Jacobi SVD workgroup: at most 16 waves, four per SIMD
constexpr int SVD_RV = 8;     // rows per lane held in registers by a Jacobi pair

// ---- factors of more than 128 columns ----------------------------------------
// Blocks of 128 columns: the scaled Gram (k_chol_scale) is factored block row by
// block row, the diagonal block by k_chol_blk (with its inverse), the rest of
// the block row as T_PP^T S and the trailing update as matrix products on the
// matrix cores; the inverse's off-diagonal blocks are two products each.  One
// workgroup eliminating column by column through global memory took 1680 us at
// 192 columns.

// D and its inverse (c each), S = D^-1 G D^-1 + shift I (ld c; rows and columns of a zero diagonal
// are zero).
__global__ void k_chol_scale(int c, const double *__restrict__ G, double shift,
                             double *__restrict__ D, double *__restrict__ iD,
                             double *__restrict__ S) {
    const long total = (long)c * c;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total;
         e += (long)gridDim.x * blockDim.x) {
        const int k = (int)(e / c), i = (int)(e - (long)k * c);
        const double gi = G[i + (long)i * c], gk = G[k + (long)k * c];
        const double di = gi > 0.0 ? sqrt(gi) : 0.0, dk = gk > 0.0 ? sqrt(gk) : 0.0;
        double v = (di > 0.0 && dk > 0.0) ? G[e] / (di * dk) : 0.0;
        if (i == k) {
            D[i] = di;
            iD[i] = di > 0.0 ? 1.0 / di : 0.0;
            if (di > 0.0) v += shift;
        }
        S[e] = v;
    }
}

// R = Rs D, T = D^-1 Ts in place (zeros below the diagonal), T NULL for R only.
__global__ void k_chol_unscale(int c, const double *__restrict__ D, double *__restrict__ R,
                               double *__restrict__ T) {
    const long total = (long)c * c;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total;
         e += (long)gridDim.x * blockDim.x) {
        const int k = (int)(e / c), i = (int)(e - (long)k * c);
        R[e] = (i <= k) ? R[e] * D[k] : 0.0;
        if (T) T[e] = (i <= k && D[i] > 0.0) ? T[e] / D[i] : 0.0;
    }
}

// Orders up to which k_chol_report iterates from registers: 16 waves of 12 rows.
constexpr int CR_REG = 192;

// Deficient pivots and the condition estimates, from G, D, R and T as the
// smaller factors' kernels report them: Gershgorin's bound, else the pivots
// where they decide, else power iterations.  binfo[b]: deficient pivots of
// block b.  y, z: c doubles of scratch each.  One workgroup.
__global__ __launch_bounds__(NT) void k_chol_report(int c, const double *__restrict__ G,
                                                    const double *__restrict__ D,
                                                    const double *__restrict__ iD,
                                                    const double *__restrict__ R,
                                                    const double *__restrict__ T, int nblk,
                                                    const int *__restrict__ binfo,
                                                    double *__restrict__ y,
                                                    double *__restrict__ z, int *info,
                                                    double *dinfo, int want_kappa) {
    __shared__ double s_red[NT / 64], s_part[NT];
    __shared__ double s_x[CR_REG], s_y[CR_REG], s_q[NT / 64][CR_REG];
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    const int cpad = c < NT ? c : NT, parts = NT / cpad;
    auto block_sum = [&](double v) -> double {
        v = wave_sum(v);
        __syncthreads();
        if (lane == 0) s_red[wv] = v;
        __syncthreads();
        double t = 0.0;
        for (int i = 0; i < NT / 64; i++) t += s_red[i];
        return t;
    };
    auto block_max = [&](double v) -> double {
        for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
        __syncthreads();
        if (lane == 0) s_red[wv] = v;
        __syncthreads();
        double t = 0.0;
        for (int i = 0; i < NT / 64; i++) t = fmax(t, s_red[i]);
        return t;
    };
    double dmax = 0.0, pmax = 0.0, pneg = -INFINITY;
    for (int j = tid; j < c; j += NT) {
        dmax = fmax(dmax, D[j] * D[j]);
        const double r = R[j + (long)j * c] * iD[j], p = r * r;
        if (p > 0.0) {
            pmax = fmax(pmax, p);
            pneg = fmax(pneg, -p);
        }
    }
    dmax = block_max(dmax);
    pmax = block_max(pmax);
    {
        for (int o = 32; o > 0; o >>= 1) pneg = fmax(pneg, __shfl_xor(pneg, o));
        __syncthreads();
        if (lane == 0) s_red[wv] = pneg;
        __syncthreads();
        for (int i = 0; i < NT / 64; i++) pneg = fmax(pneg, s_red[i]);
    }
    const double pmin = -pneg;
    int ndef = 0;
    for (int b = 0; b < nblk; b++) ndef += binfo[b];
    double fr = 0.0, ft = 0.0, eoff = 0.0, lmax = 0.0, lminv = 0.0;
    bool gersh = false, decided = false;
    if (T) {
        // one wave a column
        for (int k = wv; k < c; k += NT / 64) {
            const double dk = iD[k];
            double rs = 0.0;
#pragma unroll 4
            for (int i = lane; i < c; i += 64) {
                const double r = R[i + (long)k * c] * dk, t = T[i + (long)k * c] * D[i];
                fr += r * r;
                ft += t * t;
                if (i != k) rs += fabs(G[i + (long)k * c]) * iD[i] * dk;
            }
            eoff = fmax(eoff, wave_sum(rs));
        }
        fr = block_sum(fr);
        ft = block_sum(ft);
        eoff = block_max(eoff);
        gersh = want_kappa && eoff < 0.5;
        decided = ndef > 0 || !(pmax <= 1e12 * pmin);
        // Ten products a side: the estimate comes from below and sets the number of
        // passes, one up to 30 (130 columns of condition 34 read 29.0 after six products,
        // 30.7 after ten).  192 columns: 76 us with six, 88 with ten.
        const int PIT = (want_kappa && !gersh && !decided) ? 10 : 0;
        if (PIT > 0 && c <= CR_REG) {
            // the matrix in registers, rows 12 wv + 3 lg + v, columns li + 16 q; S
            // first, then Ts^T (beyond this order every product reads it from
            // memory: 635 us at 256 columns)
            const int li = lane & 15, lg = lane >> 4, r0 = 12 * wv + 3 * lg;
            double m[3][12];
            auto load = [&](const double *__restrict__ A, const double *__restrict__ cs,
                            const double *__restrict__ rs) {
#pragma unroll
                for (int v = 0; v < 3; v++)
#pragma unroll
                    for (int q = 0; q < 12; q++) {
                        const int r = r0 + v, k = li + 16 * q;
                        m[v][q] = (r < c && k < c)
                                      ? A[k + (long)r * c] * cs[k] * (rs ? rs[r] : 1.0) : 0.0;
                    }
            };
            // y = m x, by rows
            auto rows = [&](const double *x, double *y) {
                double t[3] = {0.0, 0.0, 0.0};
#pragma unroll
                for (int q = 0; q < 12; q++) {
                    const double xq = x[li + 16 * q];
#pragma unroll
                    for (int v = 0; v < 3; v++) t[v] = fma(m[v][q], xq, t[v]);
                }
#pragma unroll
                for (int v = 0; v < 3; v++) t[v] = row16_sum(t[v]);
                if (li < 3) y[r0 + li] = li == 0 ? t[0] : li == 1 ? t[1] : t[2];
                __syncthreads();
            };
            // y = f m^T x, by columns
            auto cols = [&](const double *x, double *y, double f) {
                const double x0 = x[r0], x1 = x[r0 + 1], x2 = x[r0 + 2];
#pragma unroll
                for (int q = 0; q < 12; q++) {
                    double t = fma(m[2][q], x2, fma(m[1][q], x1, fma(m[0][q], x0, 0.0)));
                    t = xor32_sum(xor16_sum(t));
                    if (lane < 16) s_q[wv][lane + 16 * q] = t;
                }
                __syncthreads();
                if (tid < CR_REG) {
                    double t = 0.0;
#pragma unroll
                    for (int w = 0; w < NT / 64; w++) t += s_q[w][tid];
                    y[tid] = f * t;
                }
                __syncthreads();
            };
            auto norm2 = [&](const double *x) {
                double t = 0.0;
                for (int i = lane; i < CR_REG; i += 64) t = fma(x[i], x[i], t);
                return wave_sum(t);
            };
            auto start = [&](int period) {
                if (tid < CR_REG) s_x[tid] = tid < c ? 1.0 + 0.01 * (tid % period) : 0.0;
                __syncthreads();
            };
            // lambda_max(S) <= c: no scaling between the products
            load(G, iD, iD);
            start(7);
            for (int it = 0; it < PIT; it += 2) {
                rows(s_x, s_y);
                rows(s_y, s_x);
            }
            lmax = sqrt(norm2(s_x) / norm2(s_y));
            __syncthreads();
            // lambda_max(Ts Ts^T) <= ft, divided out of every product
            load(T, D, nullptr);
            start(5);
            double prev = 1.0;
            for (int it = 0; it < PIT; it++) {
                if (it == PIT - 1) prev = norm2(s_x);
                rows(s_x, s_y);
                cols(s_y, s_x, 1.0 / ft);
            }
            lminv = ft * sqrt(norm2(s_x) / prev);
        }
        for (int side = 0; side < 2 && c > CR_REG; side++) {
            for (int i = tid; i < c; i += NT) y[i] = 1.0 + 0.01 * (i % (side == 0 ? 7 : 5));
            __syncthreads();
            for (int it = 0; it < PIT; it++) {
                double xn = 0.0;
                for (int i = tid; i < c; i += NT) xn += y[i] * y[i];
                xn = block_sum(xn);
                const double is = xn > 0.0 ? 1.0 / sqrt(xn) : 0.0;
                // side 0: z = S y; side 1: z = Ts^T y, then y = Ts z
                for (int k = wv; k < c; k += NT / 64) {
                    double acc = 0.0;
                    if (side == 0)
#pragma unroll 4
                        for (int i = lane; i < c; i += 64)
                            acc += G[i + (long)k * c] * iD[i] * y[i];
                    else
#pragma unroll 4
                        for (int i = lane; i <= k; i += 64) acc += T[i + (long)k * c] * D[i] * y[i];
                    acc = wave_sum(acc);
                    if (lane == 0) z[k] = acc * is * (side == 0 ? iD[k] : 1.0);
                }
                __syncthreads();
                if (side == 1) {
                    // rows on consecutive lanes, the columns split over parts
                    for (int i0 = 0; i0 < c; i0 += cpad) {
                        const int i = i0 + tid % cpad, part = tid / cpad;
                        double acc = 0.0;
                        if (i < c && part < parts) {
                            const int per = (c - i0 + parts - 1) / parts;
                            const int k0 = i0 + part * per, k1 = min(c, k0 + per);
#pragma unroll 8
                            for (int k = k0; k < k1; k++) acc += T[i + (long)k * c] * z[k];
                        }
                        __syncthreads();
                        s_part[tid] = acc;
                        __syncthreads();
                        if (part == 0 && i < c) {
                            for (int q = 1; q < parts; q++) acc += s_part[tid + q * cpad];
                            y[i] = acc * D[i];
                        }
                    }
                } else {
                    for (int i = tid; i < c; i += NT) y[i] = z[i];
                }
                __syncthreads();
                double nn = 0.0;
                for (int i = tid; i < c; i += NT) nn += y[i] * y[i];
                nn = block_sum(nn);
                (side == 0 ? lmax : lminv) = sqrt(nn);
            }
            __syncthreads();
        }
    }
    if (tid == 0) {
        dinfo[0] = sqrt(fr) * sqrt(ft);
        dinfo[1] = !(T && want_kappa) ? 0.0
                   : gersh            ? sqrt((1.0 + eoff) / (1.0 - eoff))
                   : decided          ? (pmin > 0.0 && pmin < INFINITY ? sqrt(pmax / pmin) : 0.0)
                                      : sqrt(lmax * lminv);
        dinfo[2] = (double)ndef;
        dinfo[3] = dmax;
        info[0] = ndef;
    }
}

// ---- Cholesky of a scaled Gram, c <= 128, on one workgroup ------------------
// Scaled Gram S = D^-1 G D^-1 with unit diagonal, shifted pivots, dead pivots
// skipped, R = Rs D and T = D^-1 Ts, Frobenius and 2-norm condition estimates.
// Bound by its serial chain (a pivot, a reciprocal, an update, c times over), so
// everything else is kept off that chain.  NB blocks of 16 columns, a wave each:
//   1. panel P is factored in LDL^T form by the wave (or two) whose lanes hold
//      its rows, one row a lane.  Each of them keeps the diagonal block as well,
//      once in every 16 lanes, so that the pivot and the multipliers come by a
//      DPP row broadcast: a step has no LDS access and no barrier (through LDS it
//      took about twice as long).  The columns are scaled by 1/sqrt(pivot) after
//      the panel, the roots taken by one lane each;
//   2. A22 -= L21 L21^T by 16 x 16 tiles on the FP64 matrix cores, the next
//      panel's column of tiles first; the other tiles and the inverse of the
//      diagonal block run beside the next panel's factorisation.
//   3. with the inverse wanted, row I of X = L^-1, X_IJ = -X_II sum_{K<I} L_IK
// X_KJ, on the matrix cores, beside the panel after next; the last two rows
// after the factorisation.  Ts = X^T is kept in the upper triangle of S (the
// diagonal blocks separately).  R's rows are written beside the panels too.  S lives in LDS
// column-major with an odd stride.  The power iterations hold their matrix in
// registers, 4 rows x NB columns a thread, with one barrier a product.
// Measured (us, well conditioned / with the iterations; before: column by column
// with a workgroup barrier a column up to 48, panels through LDS beyond):
// c = 16: 15 / 31 -> 7 / 10, 32: 20 / 35 -> 12 / 17, 48: 37 / 60 -> 16 / 21,
// 64: 47 / 70 -> 20 / 26, 128: 96 / 146 -> 39 / 49, of which the panels are 24.
template <int NB>
struct chol_geom {
    static constexpr int N = 16 * NB;            // padded order
    static constexpr int LD = N + 1;
    static constexpr int XS = 16 * 17;           // one diagonal block of X, row-major, stride 17
    static constexpr int LDS_DOUBLES = N * LD + NB * XS + 6 * N;  // 153 KB at NB = 8
};

typedef double f64x4_t __attribute__((ext_vector_type(4)));

// One panel in registers: dg the diagonal block's row lane % 16, pw the lane's
// own row, psel the pivot of row lane % 16.  (Forming the next reciprocal between
// a step's updates made no difference: the updates' issue bounds a step.)
template <int J, int M>
__device__ __forceinline__ void chol_update(double (&dg)[16], double (&pw)[16], double w0,
                                            double w1) {
    if constexpr (M < 16) {
        const double um = row_bcast<M>(dg[J]);
        dg[M] = fma(-w0, um, dg[M]);
        pw[M] = fma(-w1, um, pw[M]);
        // formed here, not sunk to its use
        __asm__ __volatile__("" : "+v"(dg[M]), "+v"(pw[M]));
        chol_update<J, M + 1>(dg, pw, w0, w1);
    }
}
template <int J>
__device__ __forceinline__ void chol_steps(double (&dg)[16], double (&pw)[16], int r,
                                           unsigned alive, double shift, double tiny,
                                           double &psel) {
    if constexpr (J < 16) {
        const double p = row_bcast<J>(dg[J]) + shift;
        const bool live = ((alive >> J) & 1u) && p > tiny;
        const double ip = live ? rcp_nr(p) : 0.0;
        if (r == J) psel = live ? p : 0.0;
        // multipliers (unscaled column / pivot) of the rows below row J
        const double w0 = r > J ? dg[J] * ip : 0.0, w1 = pw[J] * ip;
        chol_update<J, J + 1>(dg, pw, w0, w1);
        chol_steps<J + 1>(dg, pw, r, alive, shift, tiny, psel);
    }
}
template <int M>
__device__ __forceinline__ void chol_scale_cols(double (&dg)[16], double (&pw)[16], double isq) {
    if constexpr (M < 16) {
        const double f = row_bcast<M>(isq);
        dg[M] *= f;
        pw[M] *= f;
        chol_scale_cols<M + 1>(dg, pw, isq);
    }
}
// Inverse of a 16 x 16 lower triangle by columns: lane r of 16 holds row r of it
// in l and column r of the inverse in x; idg the reciprocal of row r's diagonal.
template <int K, int I>
__device__ __forceinline__ void tri_update(const double (&l)[16], double (&x)[16]) {
    if constexpr (I < 16) {
        x[I] = fma(-row_bcast<I>(l[K]), x[K], x[I]);
        __asm__ __volatile__("" : "+v"(x[I]));
        tri_update<K, I + 1>(l, x);
    }
}
template <int K>
__device__ __forceinline__ void tri_inverse(const double (&l)[16], double (&x)[16], double idg) {
    if constexpr (K < 16) {
        x[K] *= row_bcast<K>(idg);
        tri_update<K, K + 1>(l, x);
        tri_inverse<K + 1>(l, x, idg);
    }
}

// Tile t of a lower triangle of tiles, row by row.
__device__ __forceinline__ void tri_tile(int t, int &I, int &J) {
    I = 0;
    while ((I + 1) * (I + 2) / 2 <= t) I++;
    J = t - I * (I + 1) / 2;
}

// With `unit` the input is already scaled (a diagonal block of a larger scaled
// Gram, ptt_hip_chol_qr_factor beyond 128 columns): D = 1, pivots are tested as
// they come.  ldg, ldo: leading dimensions of G and of R and T.
template <int NB, bool WT>
__global__ __launch_bounds__(64 * NB) void k_chol_blk(int c, const double *__restrict__ G, long ldg,
                                                      double shift, double tiny,
                                                      double *__restrict__ R,
                                                      double *__restrict__ T, long ldo, int *info,
                                                      double *dinfo, int want_kappa, int unit) {
    using geom = chol_geom<NB>;
    constexpr int N = geom::N, LD = geom::LD, XS = geom::XS;
    extern __shared__ double lds[];
    double *S = lds;            // N x N, S[i + j * LD]
    double *Xd = S + N * LD;    // diagonal blocks of X = L^-1
    double *D = Xd + NB * XS;   // Jacobi scaling
    double *iD = D + N;         // 1 / D (0 where D is)
    double *tdg = iD + N;       // pivots (0 when dead)
    double *idg = tdg + N;      // 1 / sqrt(pivot) (0 when dead)
    double *pv = idg + N;       // power-iteration vectors (2 x N)
    __shared__ double s_red[2 * NB];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int li = lane & 15, lg = lane >> 4;
    // row ti, columns tj, tj + 4, ... of the copies in and out
    const int ti = tid % N, tj = tid / N;
    const int npn = (c + 15) >> 4;

    // S = D^-1 G D^-1 from the lower tiles of G, all loads of a thread in flight
    // at once (one CU's loads of 128 KB took a tenth of the whole)
    double eoff = 0.0, dmax = 0.0;
    {
        // wave w's tiles: the pairs (w, w + u mod NB), each pair once
        constexpr int PER = NB / 2 + 1;
        auto tile = [&](int u, int &I, int &J) {
            const int o = wv + u < NB ? wv + u : wv + u - NB;
            I = o > wv ? o : wv;
            J = o > wv ? wv : o;
            return 2 * u < NB || wv < NB / 2 || u == 0;
        };
        double gv[PER][4];
#pragma unroll
        for (int u = 0; u < PER; u++) {
            int I, J;
            const bool mine = tile(u, I, J);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int i = 16 * I + li, j = 16 * J + 4 * q + lg;
                gv[u][q] = (mine && i < c && j < c) ? G[i + (long)j * ldg] : 0.0;
            }
        }
        if (tid < N) {
            double dj = 0.0;
            if (tid < c) {
                const double g = G[tid + (long)tid * ldg];
                dj = unit ? 1.0 : g > 0.0 ? sqrt(g) : 0.0;
            }
            D[tid] = dj;
            iD[tid] = dj > 0.0 ? 1.0 / dj : 0.0;
            tdg[tid] = 0.0;
            idg[tid] = 0.0;
            pv[tid] = tid < c ? 1.0 + 0.01 * (tid % 7) : 0.0;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < PER; u++) {
            int I, J;
            if (tile(u, I, J)) {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int i = 16 * I + li, j = 16 * J + 4 * q + lg;
                    const double s = gv[u][q] * iD[i] * iD[j];
                    S[i + j * LD] = s;
                    if (I != J) S[j + i * LD] = s;
                }
            }
        }
    }
    __syncthreads();
    if (want_kappa) {
        // row sums of |S - I|, a quarter of the columns a thread
        double rs = 0.0;
#pragma unroll 8
        for (int u = 0; u < 4 * NB; u++) {
            const int j = tj + 4 * u;
            rs += j != ti ? fabs(S[ti + j * LD]) : 0.0;
        }
        Xd[tj * N + ti] = rs;  // free until the inverse
        lds_sync();
        for (int i = lane; i < N; i += 64)
            eoff = fmax(eoff, (Xd[i] + Xd[N + i]) + (Xd[2 * N + i] + Xd[3 * N + i]));
    }
    for (int i = lane; i < N; i += 64) dmax = fmax(dmax, D[i] * D[i]);
    // Gershgorin certificate: S = I + E with ||E||_inf = e < 1/2 has kappa_2 <=
    // (1+e)/(1-e), and the power iterations are skipped
    eoff = wave_max(eoff);
    dmax = wave_max(dmax);
    const bool gersh = want_kappa && eoff < 0.5;
    // y = M x for the N x N matrix whose rows 16 wv + 4 lg + v, columns li + 16 q
    // a thread holds in m
    auto matvec = [&](const double (&m)[4][NB], const double *x, double *y) {
        double xv[NB], s[4];
#pragma unroll
        for (int q = 0; q < NB; q++) xv[q] = x[li + 16 * q];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            s[v] = 0.0;
#pragma unroll
            for (int q = 0; q < NB; q++) s[v] = fma(m[v][q], xv[q], s[v]);
        }
        // the four rows' sums over the 16 lanes at once: lane li ends with row
        // 2 (li / 8 % 2) + (li / 4 % 2) (four sums by turns: 32
        // columns 18.1 us instead of 16.7)
        const bool h8 = (li & 8) != 0, h4 = (li & 4) != 0;
        const double u0 = (h8 ? s[2] : s[0]) + dppd<0x128>(h8 ? s[0] : s[2]);  // row_ror:8
        const double u1 = (h8 ? s[3] : s[1]) + dppd<0x128>(h8 ? s[1] : s[3]);
        // half-row mirror: the 4-lane groups swap
        const double t = quad_sum((h4 ? u1 : u0) + dppd<0x141>(h4 ? u0 : u1));
        if ((li & 3) == 0) y[16 * wv + 4 * lg + 2 * (int)h8 + (int)h4] = t;
        lds_sync();
    };
    auto norm2 = [&](const double *x) {
        double s = 0.0;
        for (int i = lane; i < N; i += 64) s = fma(x[i], x[i], s);
        return wave_sum(s);
    };
    constexpr int PIT = 6;
    double lmax = 0.0, lminv = 0.0;
    if (WT && want_kappa && !gersh) {
        // lambda_max(S) <= c: six products need no scaling in between
        double m[4][NB];
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
            for (int q = 0; q < NB; q++) m[v][q] = S[(li + 16 * q) + (16 * wv + 4 * lg + v) * LD];
        for (int it = 0; it < PIT; it++) matvec(m, pv + (it & 1) * N, pv + (~it & 1) * N);
        lmax = sqrt(norm2(pv) / norm2(pv + N));  // PIT is even: the last product is in pv
    }
    lds_sync();

    // A tile (I, J) of the trailing matrix less L_IP L_JP^T
    auto update_tile = [&](int I, int J, int P) {
        const int bi = 16 * I, bj = 16 * J;
        f64x4_t acc;
#pragma unroll
        for (int v = 0; v < 4; v++) acc[v] = S[(bi + lg + 4 * v) + (bj + li) * LD];
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            const int kc = 16 * P + 4 * kk + lg;
            const double a = -S[(bi + li) + kc * LD];
            const double b = S[(bj + li) + kc * LD];
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < 4; v++) S[(bi + lg + 4 * v) + (bj + li) * LD] = acc[v];
    };
    auto invert_diag = [&](int B) {
        double l[16], x[16];
#pragma unroll
        for (int k = 0; k < 16; k++) {
            l[k] = S[(16 * B + li) + (16 * B + k) * LD];
            x[k] = k == li ? 1.0 : 0.0;
        }
        tri_inverse<0>(l, x, idg[16 * B + li]);
        if (lane < 16) {
#pragma unroll
            for (int i = 0; i < 16; i++) Xd[B * XS + i * 17 + li] = x[i];
        }
    };

    // X_IJ, J < I, stored transposed: Ts[16J + j][16I + i] = X_IJ[i][j]
    auto x_tile = [&](int I, int J) {
        f64x4_t acc = {0.0, 0.0, 0.0, 0.0};
        for (int K = J; K < I; K++) {
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                const int k = 4 * kk + lg;
                const double a = S[(16 * I + li) + (16 * K + k) * LD];
                const double b =
                    (K == J) ? Xd[J * XS + k * 17 + li] : S[(16 * J + li) + (16 * K + k) * LD];
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
            }
        }
        // X_IJ = -X_II acc: register kk of acc is the B operand of step kk
        f64x4_t x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            const double a = -Xd[I * XS + li * 17 + 4 * kk + lg];
            x = __builtin_amdgcn_mfma_f64_16x16x4f64(a, acc[kk], x, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < 4; v++) S[(16 * J + li) + (16 * I + lg + 4 * v) * LD] = x[v];
    };
    double fr = 0.0, ft = 0.0;
    // rows of R (and the zeros of T left of them) of block B, by wave w of nw
    auto put_rows = [&](int B, int w, int nw) {
        const int i = 16 * B + li;
        for (int k = 4 * w + lg; k < c; k += 4 * nw) {
            const double rv = k >= i ? S[k + i * LD] : 0.0;
            if (i < c) {
                fr = fma(rv, rv, fr);
                R[i + (long)k * ldo] = rv * D[k];
                if (WT && k < 16 * B) T[i + (long)k * ldo] = 0.0;
            }
        }
    };

    // ---- factorization, panel by panel
    for (int P = 0; P < npn; P++) {
        const int rb0 = 16 * P;
        // waves that hold the rows below the panel's diagonal block
        const int fw = 16 * (npn - P - 1) > 64 ? 2 : 1;
        double dg[16], pw[16];
        double sq = 0.0;
        if (wv < fw) {
            const int r = rb0 + 16 + 64 * wv + lane;
#pragma unroll
            for (int m = 0; m < 16; m++) {
                dg[m] = S[(rb0 + li) + (rb0 + m) * LD];
                pw[m] = r < N ? S[r + (rb0 + m) * LD] : 0.0;
            }
            double psel = 0.0;
            const unsigned alive = (unsigned)__ballot(rb0 + li < c && D[rb0 + li] > 0.0);
            chol_steps<0>(dg, pw, li, alive, shift, tiny, psel);
            sq = psel > 0.0 ? sqrt_nr(psel) : 0.0;
            const double isq = psel > 0.0 ? rcp_nr(sq) : 0.0;
            chol_scale_cols<0>(dg, pw, isq);
            if (wv == 0 && lane < 16) {
                tdg[rb0 + li] = psel;
                idg[rb0 + li] = isq;
            }
            if (r < N) {
#pragma unroll
                for (int m = 0; m < 16; m++) S[r + (rb0 + m) * LD] = pw[m];
            }
        } else if (P > 0) {
            // beside it: the rest of the previous panel's update, its diagonal
            // block's inverse, the row of X above it, and its rows of R
            const int nb = npn - (P + 1), nt = nb * (nb + 1) / 2;
            const int w = wv - fw, nw = NB - fw;
            for (int t = w; t < nt; t += nw) {
                int I, J;
                tri_tile(t, I, J);
                update_tile(P + 1 + I, P + 1 + J, P - 1);
            }
            if (WT) {
                if (w == nw - 1) invert_diag(P - 1);
                for (int J = w; J < P - 2; J += nw) x_tile(P - 2, J);
            }
            put_rows(P - 1, w, nw);
        }
        lds_sync();
        // the diagonal block of L: every wave that factored has read S's
        if (wv == 0 && lane < 16) {
#pragma unroll
            for (int m = 0; m < 16; m++)
                if (m <= li) S[(rb0 + li) + (rb0 + m) * LD] = m == li ? sq : dg[m];
        }
        for (int I = P + 1 + wv; I < npn; I += NB) update_tile(I, P + 1, P);
        lds_sync();
    }
    double pmax = 0.0, pmin = INFINITY;
    int ndef = 0;
    for (int i0 = 0; i0 < N; i0 += 64) {
        const double p = (i0 + lane < c) ? tdg[i0 + lane] : 0.0;
        pmax = fmax(pmax, p);
        if (p > 0.0) pmin = fmin(pmin, p);
        ndef += __popcll(__ballot(i0 + lane < c && !(p > 0.0)));
    }
    pmax = wave_max(pmax);
    pmin = -wave_max(-pmin);

    put_rows(npn - 1, wv, NB);
    if (WT) {
        if (wv == NB - 1) invert_diag(npn - 1);
        for (int J = wv; J < npn - 2; J += NB) x_tile(npn - 2, J);
        lds_sync();
        for (int J = wv; J < npn - 1; J += NB) x_tile(npn - 1, J);
        lds_sync();
    }
    // Ts(i, k), 0 below the diagonal
    auto tget = [&](int i, int k) -> double {
        const int ib = i >> 4, kb = k >> 4;
        const double off = S[i + k * LD], dia = Xd[ib * XS + (k & 15) * 17 + (i & 15)];
        // a block beyond c has no diagonal block
        return ib < kb ? off : (ib == kb && i <= k && k < c) ? dia : 0.0;
    };
    if (WT) {
        // the upper tiles of T (put_rows wrote the zeros of the others)
        for (int t = wv; t < npn * (npn + 1) / 2; t += NB) {
            int I, J;
            tri_tile(t, I, J);
            const int i = 16 * J + li;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int k = 16 * I + 4 * q + lg;
                const double tv = tget(i, k);
                if (i < c && k < c) {
                    ft = fma(tv, tv, ft);
                    T[i + (long)k * ldo] = tv * iD[i];
                }
            }
        }
    }
    const bool decided = ndef > 0 || !(pmax <= 1e12 * pmin);
    if (WT) {
        fr = wave_sum(fr);
        ft = wave_sum(ft);
        if (lane == 0) {
            s_red[2 * wv] = fr;
            s_red[2 * wv + 1] = ft;
        }
        if (tid < N) pv[tid] = tid < c ? 1.0 + 0.01 * (tid % 7) : 0.0;
        lds_sync();
        fr = 0.0;
        ft = 0.0;
        for (int w = 0; w < NB; w++) {
            fr += s_red[2 * w];
            ft += s_red[2 * w + 1];
        }
        if (want_kappa && !gersh && !decided) {
            // lambda_max(Ts Ts^T) <= ft = ||Ts||_F^2, divided out of every product.
            // (kappa_2 of S is at least the ratio of two pivots, each of which lies
            // between lambda_min and lambda_max: beyond 1e12, or with a dead pivot,
            // it is known to be too large without the iterations.)
            const double ift = 1.0 / ft;
            double m[4][NB], mt[4][NB];
#pragma unroll
            for (int v = 0; v < 4; v++)
#pragma unroll
                for (int q = 0; q < NB; q++) {
                    const int r = 16 * wv + 4 * lg + v, k = li + 16 * q;
                    m[v][q] = tget(r, k);
                    mt[v][q] = tget(k, r) * ift;
                }
            double prev = 1.0;
            for (int it = 0; it < PIT; it++) {
                if (it == PIT - 1) prev = norm2(pv);
                matvec(mt, pv, pv + N);
                matvec(m, pv + N, pv);
            }
            lminv = ft * sqrt(norm2(pv) / prev);
        }
    }
    if (tid == 0) {
        dinfo[0] = WT ? sqrt(fr) * sqrt(ft) : 0.0;
        dinfo[1] = !(WT && want_kappa) ? 0.0
                   : gersh             ? sqrt((1.0 + eoff) / (1.0 - eoff))
                   : decided           ? (pmax > 0.0 && pmin < INFINITY ? sqrt(pmax / pmin) : 0.0)
                                       : sqrt(lmax * lminv);
        dinfo[2] = (double)ndef;
        dinfo[3] = dmax;
        info[0] = ndef;
    }
}

// Rotation of a double across the 16 lanes of a DPP row (row_ror:N).
template <int N>
__device__ __forceinline__ double row_ror(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_update_dpp(0, lo, 0x120 + N, 0xF, 0xF, false);
    hi = __builtin_amdgcn_update_dpp(0, hi, 0x120 + N, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

// Sum of three values over each aligned group of G lanes (G a power of two
// <= 64), every lane receiving the sums.  Groups of 16 and 64 use row
// rotations (DPP) inside each 16-lane row.
__device__ __forceinline__ void group_allreduce3(double &x, double &y, double &z, int G) {
    if (G == 16 || G == 64) {
        x += row_ror<8>(x); y += row_ror<8>(y); z += row_ror<8>(z);
        x += row_ror<4>(x); y += row_ror<4>(y); z += row_ror<4>(z);
        x += row_ror<2>(x); y += row_ror<2>(y); z += row_ror<2>(z);
        x += row_ror<1>(x); y += row_ror<1>(y); z += row_ror<1>(z);
        if (G == 64) {
            for (int o = 16; o < 64; o <<= 1) {
                x += __shfl_xor(x, o);
                y += __shfl_xor(y, o);
                z += __shfl_xor(z, o);
            }
        }
    } else {
        for (int o = 1; o < G; o <<= 1) {
            x += __shfl_xor(x, o);
            y += __shfl_xor(y, o);
            z += __shfl_xor(z, o);
        }
    }
}

// DPP move of a double inside a quad / row (dpp_ctrl CTRL).  Every lane's
// source is a valid lane for the quad permutations and mirrors used here, so
// no "old" value needs to be materialised.
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xF, 0xF, false);
    hi = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

// Sum of three values over each aligned group of G lanes (G a power of two
// <= 64), every lane receiving the sums: quad permutations (xor 1, xor 2),
// then the half-row and row mirrors, then the cross-row lane swaps.
__device__ __forceinline__ void group_allreduce3_q(double &x, double &y, double &z, int G) {
    if (G >= 2) { x += dpp_d<0xB1>(x); y += dpp_d<0xB1>(y); z += dpp_d<0xB1>(z); }
    if (G >= 4) { x += dpp_d<0x4E>(x); y += dpp_d<0x4E>(y); z += dpp_d<0x4E>(z); }
    if (G >= 8) { x += dpp_d<0x141>(x); y += dpp_d<0x141>(y); z += dpp_d<0x141>(z); }
    if (G >= 16) { x += dpp_d<0x140>(x); y += dpp_d<0x140>(y); z += dpp_d<0x140>(z); }
    if (G >= 32) { x = xor16_sum(x); y = xor16_sum(y); z = xor16_sum(z); }
    if (G >= 64) { x = xor32_sum(x); y = xor32_sum(y); z = xor32_sum(z); }
}

// Round-robin pairing as rr_pair, without integer division.
__device__ __forceinline__ void rr_pair_fast(int kp, int t, int p, int &a, int &b) {
    const int m = kp - 1;
    if (p == 0) {
        a = m;
        b = t;
    } else {
        a = t + p;
        if (a >= m) a -= m;
        b = t - p;
        if (b < 0) b += m;
    }
}

// Jacobi rotation (c, s) zeroing the off-diagonal of [[al, ga], [ga, be]].
// The tangent only steers convergence and is formed from the hardware
// reciprocal / reciprocal-square-root approximations; c = 1/sqrt(1+t^2) is
// refined by two Newton steps so that c^2 + s^2 = 1 to working accuracy,
// which is what keeps the accumulated transformations orthogonal.
__device__ __forceinline__ void jacobi_cs(double al, double be, double ga, double &c, double &s) {
    const double zeta = (be - al) * 0.5 * __builtin_amdgcn_rcp(ga);
    const double az = fabs(zeta);
    double t;
    if (az > 1.0e150) {
        t = 0.5 * __builtin_amdgcn_rcp(zeta);
    } else {
        const double q = 1.0 + zeta * zeta;
        const double root = q * __builtin_amdgcn_rsq(q);  // ~sqrt(q)
        t = __builtin_amdgcn_rcp(az + root);
        if (zeta < 0.0) t = -t;
    }
    const double w = 1.0 + t * t;
    double y = __builtin_amdgcn_rsq(w);
    y = y * (1.5 - 0.5 * w * y * y);
    y = y * (1.5 - 0.5 * w * y * y);
    c = y;
    s = y * t;
}

// One Jacobi pair step with the lane-group width GG and rows per lane RR
// known at compile time (m == GG * RR): the LDS offsets of a lane's rows are
// immediates, so the round spends no VALU work on addresses.  Returns whether
// the pair rotated; cs / sn / unsettled as in the generic path.
template <int GG, int RR>
__device__ __forceinline__ bool jacobi_pair_fixed(double *ca, double *cb, bool valid, double tol,
                                                  double &cs, double &sn, bool &unsettled,
                                                  bool &big) {
    double xa[RR], xb[RR];
    double al = 0.0, be = 0.0, ga = 0.0;
    if (valid) {
#pragma unroll
        for (int q = 0; q < RR; q++) {
            xa[q] = ca[q * GG];
            xb[q] = cb[q * GG];
        }
#pragma unroll
        for (int q = 0; q < RR; q++) {
            al += xa[q] * xa[q];
            be += xb[q] * xb[q];
            ga += xa[q] * xb[q];
        }
    }
    group_allreduce3_q(al, be, ga, GG);
    // |cos| > tol compared as ga^2 > tol^2 al be (no square roots; the
    // columns are scaled to O(1), and products that underflow belong to
    // columns too small to matter)
    const double g2 = ga * ga, ab = al * be;
    const bool rot = valid && g2 > (tol * tol) * ab && al > 0.0 && be > 0.0;
    cs = 1.0;
    sn = 0.0;
    if (rot) jacobi_cs(al, be, ga, cs, sn);
    unsettled = rot && g2 > (4.0 * tol * tol) * ab;
    big = rot && g2 > 1e-16 * ab;
    if (rot) {
#pragma unroll
        for (int q = 0; q < RR; q++) {
            ca[q * GG] = cs * xa[q] - sn * xb[q];
            cb[q * GG] = sn * xa[q] + cs * xb[q];
        }
    }
    return rot;
}

__device__ __forceinline__ void rr_pair(int kp, int t, int p, int &a, int &b) {
    // Round-robin (circle) schedule over kp players, round t in [0, kp-1).
    const int m = kp - 1;
    if (p == 0) {
        a = m;
        b = t;
    } else {
        a = (t + p) % m;
        b = (t - p + m) % m;
    }
}

// The columns of A and, when wanted, of V live in LDS.
__global__ __launch_bounds__(SVD_NT) void k_svd_jacobi(int m, int k, const double *__restrict__ A,
                                                   long lda, double *__restrict__ sig,
                                                   double *__restrict__ U, long ldu,
                                                   double *__restrict__ V, long ldv,
                                                   double log_scale, double delta, int cap,
                                                   int *iout) {
    extern __shared__ double lds[];
    const int tid = threadIdx.x;
    const int nth = blockDim.x;  // chosen by the launcher for the problem size
    // Columns in LDS use an odd stride (in doubles) so that the 16 pairs a
    // wave touches start in distinct banks.
    const int ldw = m | 1;
    double *W = lds;  // m x k, ld ldw
    double *Vw = V ? lds + (long)ldw * k : nullptr;
    const int ldvw = k | 1;
    __shared__ int s_rot;
    __shared__ double s_sig[SVD_ONE_WG_MAX];
    __shared__ double s_sorted[SVD_ONE_WG_MAX];
    __shared__ int s_pos[SVD_ONE_WG_MAX];

    // Exactly-zero columns (deficient directions) take no part in the
    // rotations: nonzero columns are packed first, in their original order.
    __shared__ int s_perm[SVD_ONE_WG_MAX];
    __shared__ int s_knz;
    // The columns are scaled by 2^-e (exact) so that the largest entry is
    // O(1): bond matrices of deep trains reach 1e-60 and below, where the
    // products of squared norms would underflow.
    __shared__ int s_exp;
    for (int j = tid; j < k; j += nth) {
        double s = 0.0;
        for (int i = 0; i < m; i++) s = fmax(s, fabs(A[i + (long)j * lda]));
        s_sig[j] = s;
    }
    __syncthreads();
    if (tid == 0) {
        int q = 0;
        double amax = 0.0;
        for (int j = 0; j < k; j++) {
            if (s_sig[j] > 0.0) s_perm[q++] = j;
            amax = fmax(amax, s_sig[j]);
        }
        s_exp = (amax > 0.0) ? ilogb(amax) : 0;
        s_knz = q;
        for (int j = 0; j < k; j++)
            if (!(s_sig[j] > 0.0)) s_perm[q++] = j;
    }
    __syncthreads();
    for (long e = tid; e < (long)m * k; e += nth) {
        long j = e / m, i = e - j * m;
        W[i + j * ldw] = ldexp(A[i + (long)s_perm[j] * lda], -s_exp);
    }
    if (Vw)
        for (long e = tid; e < (long)k * k; e += nth) {
            long j = e / k, i = e - j * k;
            Vw[i + j * ldvw] = (i == s_perm[j]) ? 1.0 : 0.0;
        }
    __syncthreads();
    const int knz = s_knz;

    const int kp = knz + (knz & 1);
    const int P = kp / 2;
    int G = 64;
    while (G > 1 && G * P > nth) G >>= 1;
    // about SVD_RV rows per lane: wider groups only add redundant reduction
    // and rotation-parameter work (idle groups skip the round below)
    int Gr = 1;
    while (Gr < 64 && Gr * SVD_RV < m) Gr <<= 1;
    if (Gr < G) G = Gr;
    const int ngroups = nth / G;
    const int g = tid / G, gl = tid - g * G;
    // Rotate only when the pair's cosine exceeds the rounding noise of an
    // m-term dot product; below that the columns are orthogonal to working
    // accuracy (stricter thresholds never settle).
    const double tol = 0x1.0p-53 * (double)m;
    __shared__ int s_big, s_bad;
    int sweep = 0;
    const int max_sweeps = 40;
    for (; sweep < max_sweeps && knz >= 2; sweep++) {
        if (tid == 0) {
            s_rot = 0;
            s_big = 0;
            s_bad = 0;
        }
        __syncthreads();
        int rot_local = 0, big_local = 0;
        for (int t = 0; t < kp - 1; t++) {
            for (int p0 = 0; p0 < P; p0 += ngroups) {
                int p = p0 + g;
                // groups without a pair this round (all lanes of a group agree;
                // nothing below reaches across groups)
                if (p >= P) continue;
                int a = -1, b = -1;
                if (p < P) rr_pair_fast(kp, t, p, a, b);
                bool valid = (p < P) && a < knz && b < knz;
                // Column segments of the pair stay in registers between the
                // dot products and the rotation when they fit (m <= 8 G).
                const bool inreg = (m <= SVD_RV * G);
                double xa[SVD_RV], xb[SVD_RV];
                double al = 0.0, be = 0.0, ga = 0.0;
                double *ca = W + (long)(valid ? a : 0) * ldw, *cb = W + (long)(valid ? b : 0) * ldw;
                // exactly SVD_RV rows per lane (the common m = 8 G case): no
                // per-row guards, one branch on the pair's validity
                const bool full = (m == SVD_RV * G);
                // the common shapes get compile-time strides
                const bool fix16 = (G == 16 && m == 16 * SVD_RV);
                const bool fix32 = (G == 32 && m == 32 * (SVD_RV / 2));
                if (fix16 || fix32) {
                    // loads, dots and rotation inside jacobi_pair_fixed
                } else if (full) {
                    if (valid) {
#pragma unroll
                        for (int q = 0; q < SVD_RV; q++) {
                            xa[q] = ca[gl + q * G];
                            xb[q] = cb[gl + q * G];
                        }
#pragma unroll
                        for (int q = 0; q < SVD_RV; q++) {
                            al += xa[q] * xa[q];
                            be += xb[q] * xb[q];
                            ga += xa[q] * xb[q];
                        }
                    }
                } else if (inreg) {
#pragma unroll
                    for (int q = 0; q < SVD_RV; q++) {
                        const int i = gl + q * G;
                        double x = 0.0, y = 0.0;
                        if (valid && i < m) {
                            x = ca[i];
                            y = cb[i];
                        }
                        xa[q] = x;
                        xb[q] = y;
                        al += x * x;
                        be += y * y;
                        ga += x * y;
                    }
                } else if (valid) {
                    for (int i = gl; i < m; i += G) {
                        double x = ca[i], y = cb[i];
                        al += x * x;
                        be += y * y;
                        ga += x * y;
                    }
                }
                double cs = 1.0, sn = 0.0;
                bool rot, unsettled, big;
                if (fix16) {
                    rot = jacobi_pair_fixed<16, SVD_RV>(ca + gl, cb + gl, valid, tol, cs, sn,
                                                        unsettled, big);
                } else if (fix32) {
                    rot = jacobi_pair_fixed<32, SVD_RV / 2>(ca + gl, cb + gl, valid, tol, cs, sn,
                                                            unsettled, big);
                } else {
                group_allreduce3_q(al, be, ga, G);
                const double nab = sqrt(al) * sqrt(be);
                rot = valid && fabs(ga) > tol * nab && al > 0.0 && be > 0.0;
                if (rot) jacobi_cs(al, be, ga, cs, sn);
                // The computed cosine carries rounding up to ~m u even for
                // exactly orthogonal columns, so rotations start above tol
                // but only cosines above 2 tol keep the sweeps going;
                // otherwise noise-triggered rotations never settle.
                unsettled = rot && fabs(ga) > 2.0 * tol * nab;
                big = rot && ga * ga > 1e-16 * (al * be);
                }
                if (big) big_local = 1;
                if (rot && !fix16 && !fix32) {
                    if (full) {
#pragma unroll
                        for (int q = 0; q < SVD_RV; q++) {
                            ca[gl + q * G] = cs * xa[q] - sn * xb[q];
                            cb[gl + q * G] = sn * xa[q] + cs * xb[q];
                        }
                    } else if (inreg) {
#pragma unroll
                        for (int q = 0; q < SVD_RV; q++) {
                            const int i = gl + q * G;
                            if (i < m) {
                                ca[i] = cs * xa[q] - sn * xb[q];
                                cb[i] = sn * xa[q] + cs * xb[q];
                            }
                        }
                    } else {
                        for (int i = gl; i < m; i += G) {
                            double x = ca[i], y = cb[i];
                            ca[i] = cs * x - sn * y;
                            cb[i] = sn * x + cs * y;
                        }
                    }
                }
                if (rot) {
                    if (Vw) {
                        double *va = Vw + (long)a * ldvw, *vb = Vw + (long)b * ldvw;
                        for (int i = gl; i < k; i += G) {
                            double x = va[i], y = vb[i];
                            va[i] = cs * x - sn * y;
                            vb[i] = sn * x + cs * y;
                        }
                    }
                }
                if (unsettled) rot_local = 1;
            }
            __syncthreads();
        }
        if (rot_local) s_rot = 1;
        if (big_local) s_big = 1;
        __syncthreads();
        if (!s_rot) break;
        // When no pair of this sweep rotated by a cosine above 1e-8,
        // quadratic convergence has usually left every pair orthogonal to
        // working accuracy.  A direct test of every pair with the sweep's own
        // criterion (unsettled: cos > 2 tol) then replaces the rotation-free
        // sweep that would confirm it; if a pair fails, the sweeps go on.
        // (The skipped sweep would only rotate pairs with tol < cos <= 2 tol.)
        if (!s_big) {
            double *nrm = s_sorted;  // free until the singular values are sorted
            for (int j = tid; j < knz; j += nth) {
                const double *cj = W + (long)j * ldw;
                double a0 = 0.0, a1 = 0.0;
                int i = 0;
                for (; i + 1 < m; i += 2) {
                    a0 += cj[i] * cj[i];
                    a1 += cj[i + 1] * cj[i + 1];
                }
                if (i < m) a0 += cj[i] * cj[i];
                nrm[j] = a0 + a1;
            }
            __syncthreads();
            // 2 x 4 blocks of pair products over the upper triangle
            const int nb2 = (knz + 1) >> 1, nb4 = (knz + 3) >> 2;
            for (int t = tid; t < nb2 * nb4; t += nth) {
                const int bi = t / nb4, bj = t - bi * nb4;
                if (2 * bi > 4 * bj + 3) continue;
                int oi[2], oj[4];
#pragma unroll
                for (int q = 0; q < 2; q++) oi[q] = min(2 * bi + q, knz - 1) * ldw;
#pragma unroll
                for (int q = 0; q < 4; q++) oj[q] = min(4 * bj + q, knz - 1) * ldw;
                double acc[2][4];
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int b = 0; b < 4; b++) acc[a][b] = 0.0;
                for (int r = 0; r < m; r++) {
                    double x[2], y[4];
#pragma unroll
                    for (int q = 0; q < 2; q++) x[q] = W[oi[q] + r];
#pragma unroll
                    for (int q = 0; q < 4; q++) y[q] = W[oj[q] + r];
#pragma unroll
                    for (int a = 0; a < 2; a++)
#pragma unroll
                        for (int b = 0; b < 4; b++) acc[a][b] += x[a] * y[b];
                }
                bool bad = false;
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int b = 0; b < 4; b++) {
                        const int ia = 2 * bi + a, jb = 4 * bj + b;
                        if (ia < jb && jb < knz) {
                            const double g2 = acc[a][b] * acc[a][b], ab = nrm[ia] * nrm[jb];
                            bad = bad || (g2 > (4.0 * tol * tol) * ab);
                        }
                    }
                if (bad) s_bad = 1;
            }
            __syncthreads();
            if (!s_bad) break;
        }
        __syncthreads();
    }
    // column norms
    for (int j = g; j < k; j += ngroups) {
        const double *cj = W + (long)j * ldw;
        double s = 0.0;
        for (int i = gl; i < m; i += G) s += cj[i] * cj[i];
        for (int o = 1; o < G; o <<= 1) s += __shfl_xor(s, o);
        if (gl == 0) s_sig[j] = sqrt(s);
    }
    __syncthreads();
    // descending order by rank counting (ties by index)
    for (int j = tid; j < k; j += nth) {
        double sj = s_sig[j];
        int pos = 0;
        for (int i = 0; i < k; i++) {
            double si = s_sig[i];
            pos += (si > sj) || (si == sj && i < j);
        }
        s_pos[j] = pos;
    }
    __syncthreads();
    for (int j = tid; j < k; j += nth) {
        sig[s_pos[j]] = ldexp(s_sig[j], s_exp);
        s_sorted[s_pos[j]] = s_sig[j];  // scaled by 2^-e
    }
    for (long e = tid; e < (long)m * k; e += nth) {
        long j = e / m, i = e - j * m;
        double sj = s_sig[j];
        U[i + (long)s_pos[j] * ldu] = sj > 0.0 ? W[i + j * ldw] / sj : 0.0;
    }
    if (Vw)
        for (long e = tid; e < (long)k * k; e += nth) {
            long j = e / k, i = e - j * k;
            V[i + (long)s_pos[j] * ldv] = Vw[i + j * ldvw];
        }
    __syncthreads();
    if (tid == 0) {
        const double s0 = s_sorted[0];
        const double thr = sqrt((double)k) * 0x1.0p-53 * s0;
        int numrank = 0;
        for (int j = 0; j < k; j++) numrank += (s_sorted[j] > thr) && (s0 > 0.0);
        int rho = numrank;
        double tail = 0.0;
        const double ld = delta > 0.0 ? log(delta) : -INFINITY;
        for (int q = numrank - 1; q >= 0; q--) {
            double v = s_sorted[q];
            tail += v * v;
            double lhs = (tail > 0.0) ? 0.5 * log(tail) + log_scale + s_exp * 0.6931471805599453
                                      : -INFINITY;
            if (delta > 0.0 && lhs < ld) rho = q;
            else break;
        }
        if (rho > k) rho = k;
        if (rho > cap) rho = cap;
        if (rho < 1) rho = 1;
        iout[0] = numrank;
        iout[1] = rho;
        iout[2] = (sweep < max_sweeps) ? sweep + 1 : max_sweeps;
    }
}

// ---- one-sided Jacobi on one wave: k <= 32 columns, m <= 64 rows ---------
// The bonds of low-rank trains (the orthogonal route at ranks ~20) are too
// small for a workgroup: the one-workgroup kernel spends ~1.6 us per round on
// its barriers and group reductions.  Here one wave holds the columns in LDS;
// a round gives each pair G = 64 / (pairs, rounded up to a power of two)
// lanes, the three dot products are reduced inside the lane group, and the
// round ends with the wave's own barrier.  Same scaling, rotation rule,
// tolerance, ordering and rank decisions as k_svd_jacobi.
constexpr int SVW_K = 32, SVW_M = 64;
constexpr int SVW_LDW = SVW_M + 1, SVW_LDV = SVW_K + 1;
constexpr int SVW_LDS_DOUBLES = SVW_LDW * SVW_K + SVW_LDV * SVW_K;

// DPP move of a double inside a row (every source lane is in the same row).
template <int CTRL>
__device__ __forceinline__ double svw_dpp(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xF, 0xF, false);
    hi = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
// Sum over aligned groups of G = 2, 4, 8 or 16 lanes: quad xor 1 and xor 2,
// then the half-row mirror (lane i with 7 - i) and the row mirror (i, 15 - i).
template <int G>
__device__ __forceinline__ double svw_sum(double x) {
    x += svw_dpp<0xB1>(x);
    if constexpr (G >= 4) x += svw_dpp<0x4E>(x);
    if constexpr (G >= 8) x += svw_dpp<0x141>(x);
    if constexpr (G >= 16) x += svw_dpp<0x140>(x);
    return x;
}

// G lanes per pair (64 / G pairs at most), R rows per lane (G R <= 64 covers
// m).  Columns sit at a fixed stride of 65 (V at 33) with zero rows beyond m (k),
// so every lane handles exactly R rows without predication and the loads of
// a round issue together.
template <int G, int R>
__global__ __launch_bounds__(64) void k_svd_jacobi_wave(int m, int k, const double *__restrict__ A,
                                                        long lda, double *__restrict__ sig,
                                                        double *__restrict__ U, long ldu,
                                                        double *__restrict__ V, long ldv,
                                                        double log_scale, double delta, int cap,
                                                        int *iout) {
    extern __shared__ double lds[];
    double *W = lds, *Vs = lds + SVW_LDW * SVW_K;
    __shared__ double nrm[SVW_K], srt[SVW_K];
    __shared__ int pos[SVW_K];
    // rows of V per lane: k <= 2 (64 / G) columns, so 128 / G^2 rows cover them
    constexpr int RV = (128 / (G * G)) > 0 ? 128 / (G * G) : 1;
    static_assert(G >= 4, "k <= 32: at most 16 pairs");
    const int lane = threadIdx.x;
    // columns scaled by 2^-e (exact) so that the largest entry is O(1)
    double amax = 0.0;
    for (int e = lane; e < m * k; e += 64) {
        const int j = e / m, i = e - j * m;
        amax = fmax(amax, fabs(A[i + (long)j * lda]));
    }
    for (int o = 32; o >= 1; o >>= 1) amax = fmax(amax, __shfl_xor(amax, o));
    const int ex = (amax > 0.0) ? ilogb(amax) : 0;
    for (int e = lane; e < SVW_LDW * SVW_K; e += 64) W[e] = 0.0;
    for (int e = lane; e < SVW_LDV * SVW_K; e += 64) {
        const int j = e / SVW_LDV, i = e - j * SVW_LDV;
        Vs[e] = (V && i == j && j < k) ? 1.0 : 0.0;
    }
    __syncthreads();
    for (int e = lane; e < m * k; e += 64) {
        const int j = e / m, i = e - j * m;
        W[i + j * SVW_LDW] = ldexp(A[i + (long)j * lda], -ex);
    }
    __syncthreads();
    const int kp = k + (k & 1), P = kp / 2;
    const int g = lane / G, gl = lane - g * G;
    const double tol = 0x1.0p-53 * (double)m;
    int sweep = 0;
    const int max_sweeps = 40;
    for (; sweep < max_sweeps && k >= 2; sweep++) {
        bool unsettled = false;
        for (int t = 0; t < kp - 1; t++) {
            int a = 0, b = 0;
            if (g < P) rr_pair_fast(kp, t, g, a, b);
            const bool valid = g < P && a < k && b < k;
            // invalid lanes read column 0 twice and rotate nothing
            const int ca = valid ? a * SVW_LDW : 0, cb = valid ? b * SVW_LDW : 0;
            const int va = valid ? a * SVW_LDV : 0, vb = valid ? b * SVW_LDV : 0;
            double x[R], y[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                x[r] = W[gl + r * G + ca];
                y[r] = W[gl + r * G + cb];
            }
            double al = 0.0, be = 0.0, ga = 0.0;
#pragma unroll
            for (int r = 0; r < R; r++) {
                al += x[r] * x[r];
                be += y[r] * y[r];
                ga += x[r] * y[r];
            }
            al = svw_sum<G>(al);
            be = svw_sum<G>(be);
            ga = svw_sum<G>(ga);
            const double g2 = ga * ga, ab = al * be;
            const bool rot = valid && g2 > (tol * tol) * ab && al > 0.0 && be > 0.0;
            if (rot) {
                double cs, sn;
                jacobi_cs(al, be, ga, cs, sn);
                unsettled = unsettled || g2 > (4.0 * tol * tol) * ab;
#pragma unroll
                for (int r = 0; r < R; r++) {
                    W[gl + r * G + ca] = cs * x[r] - sn * y[r];
                    W[gl + r * G + cb] = sn * x[r] + cs * y[r];
                }
                if (V) {
                    double p[RV], q[RV];
#pragma unroll
                    for (int r = 0; r < RV; r++) {
                        p[r] = Vs[gl + r * G + va];
                        q[r] = Vs[gl + r * G + vb];
                    }
#pragma unroll
                    for (int r = 0; r < RV; r++) {
                        Vs[gl + r * G + va] = cs * p[r] - sn * q[r];
                        Vs[gl + r * G + vb] = sn * p[r] + cs * q[r];
                    }
                }
            }
            __syncthreads();
        }
        if (!__any(unsettled)) break;
    }
    // column norms, descending order by rank counting (ties by index)
    for (int j = lane; j < k; j += 64) {
        double s = 0.0;
        for (int i = 0; i < m; i++) s += W[i + j * SVW_LDW] * W[i + j * SVW_LDW];
        nrm[j] = sqrt(s);
    }
    __syncthreads();
    for (int j = lane; j < k; j += 64) {
        const double sj = nrm[j];
        int p = 0;
        for (int i = 0; i < k; i++) p += (nrm[i] > sj) || (nrm[i] == sj && i < j);
        pos[j] = p;
    }
    __syncthreads();
    for (int j = lane; j < k; j += 64) {
        sig[pos[j]] = ldexp(nrm[j], ex);
        srt[pos[j]] = nrm[j];
    }
    for (int e = lane; e < m * k; e += 64) {
        const int j = e / m, i = e - j * m;
        const double s = nrm[j];
        U[i + (long)pos[j] * ldu] = s > 0.0 ? W[i + j * SVW_LDW] / s : 0.0;
    }
    if (V)
        for (int e = lane; e < k * k; e += 64) {
            const int j = e / k, i = e - j * k;
            V[i + (long)pos[j] * ldv] = Vs[i + j * SVW_LDV];
        }
    __syncthreads();
    if (lane == 0) {
        const double s0 = srt[0];
        const double thr = sqrt((double)k) * 0x1.0p-53 * s0;
        int numrank = 0;
        for (int j = 0; j < k; j++) numrank += (srt[j] > thr) && (s0 > 0.0);
        int rho = numrank;
        double tail = 0.0;
        const double ld = delta > 0.0 ? log(delta) : -INFINITY;
        for (int q = numrank - 1; q >= 0; q--) {
            const double v = srt[q];
            tail += v * v;
            const double lhs =
                (tail > 0.0) ? 0.5 * log(tail) + log_scale + ex * 0.6931471805599453 : -INFINITY;
            if (delta > 0.0 && lhs < ld) rho = q;
            else break;
        }
        if (rho > k) rho = k;
        if (rho > cap) rho = cap;
        if (rho < 1) rho = 1;
        iout[0] = numrank;
        iout[1] = rho;
        iout[2] = (sweep < max_sweeps) ? sweep + 1 : max_sweeps;
    }
}

// ---- one-sided Jacobi over many workgroups ---------------------------------
// For column counts whose rotations one CU's LDS bandwidth or size would bound
// (the line: SVD_ONE_WG_MAX).  The columns are cut into blocks of
// B; a launch is one round of the circle schedule over the blocks, workgroup p
// taking its pair of blocks (2 B columns of W, and of V) into LDS and rotating
// every pair of columns across the two blocks, one wave a pair, B steps; the
// first round of a sweep also takes the pairs inside the blocks.  A sweep is
// thus k / B - 1 launches, each column read and written once a launch.  Same
// rotation rule, threshold, scaling and rank decisions as the one-workgroup
// kernel; the host checks once per sweep whether any pair was still unsettled.
// Columns too long for 4 of them to fit in LDS (m + k above 4800) go through
// HBM: one launch a round of single columns, one workgroup a pair (k_lj_round).
constexpr int LJ_NT = 256;
constexpr int LJ_LDS_DOUBLES = 19456;  // 152 KB

__device__ __forceinline__ void lj_sum3(double &x, double &y, double &z, double *red) {
    for (int o = 32; o >= 1; o >>= 1) {
        x += __shfl_xor(x, o);
        y += __shfl_xor(y, o);
        z += __shfl_xor(z, o);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[3 * w] = x;
        red[3 * w + 1] = y;
        red[3 * w + 2] = z;
    }
    __syncthreads();
    x = red[0] + red[3] + red[6] + red[9];
    y = red[1] + red[4] + red[7] + red[10];
    z = red[2] + red[5] + red[8] + red[11];
}

// colmax[j] = max_i |A[i, j]|
__global__ __launch_bounds__(LJ_NT) void k_lj_colmax(int m, const double *__restrict__ A,
                                                     long lda, double *__restrict__ colmax) {
    __shared__ double red[4];
    const int j = blockIdx.x;
    double s = 0.0;
    for (int i = threadIdx.x; i < m; i += LJ_NT) s = fmax(s, fabs(A[i + (long)j * lda]));
    for (int o = 32; o >= 1; o >>= 1) s = fmax(s, __shfl_xor(s, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) colmax[j] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

// exponent e with the largest entry scaled by 2^-e into [1, 2)
__global__ __launch_bounds__(LJ_NT) void k_lj_exponent(int k, const double *__restrict__ colmax,
                                                       int *__restrict__ dexp) {
    __shared__ double red[4];
    double s = 0.0;
    for (int j = threadIdx.x; j < k; j += LJ_NT) s = fmax(s, colmax[j]);
    for (int o = 32; o >= 1; o >>= 1) s = fmax(s, __shfl_xor(s, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double a = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
        *dexp = (a > 0.0) ? ilogb(a) : 0;
    }
}

// W = 2^-e A (exact), V = I (when wanted)
__global__ void k_lj_load(int m, int k, const double *__restrict__ A, long lda,
                          const int *__restrict__ dexp, double *__restrict__ W,
                          double *__restrict__ V) {
    const int e = *dexp;
    const long mk = (long)m * k, kk = V ? (long)k * k : 0;
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < mk + kk;
         t += (long)gridDim.x * blockDim.x) {
        if (t < mk) {
            const long j = t / m, i = t - j * m;
            W[t] = ldexp(A[i + j * lda], -e);
        } else {
            const long u = t - mk, j = u / k, i = u - j * k;
            V[u] = (i == j) ? 1.0 : 0.0;
        }
    }
}

// one round t of the circle schedule over kp players (k columns, a dummy
// player when k is odd); flag[0] is set when a pair was still unsettled
__global__ __launch_bounds__(LJ_NT) void k_lj_round(int m, int k, int kp, int t,
                                                    double *__restrict__ W,
                                                    double *__restrict__ V, double tol,
                                                    int *__restrict__ flag) {
    __shared__ double red[12];
    int a, b;
    rr_pair(kp, t, blockIdx.x, a, b);
    if (a >= k || b >= k) return;  // the dummy player's pair (uniform per workgroup)
    double *ca = W + (long)a * m, *cb = W + (long)b * m;
    double al = 0.0, be = 0.0, ga = 0.0;
    for (int i = threadIdx.x; i < m; i += LJ_NT) {
        const double x = ca[i], y = cb[i];
        al += x * x;
        be += y * y;
        ga += x * y;
    }
    lj_sum3(al, be, ga, red);
    const double g2 = ga * ga, ab = al * be;
    if (!(g2 > (tol * tol) * ab && al > 0.0 && be > 0.0)) return;
    if (threadIdx.x == 0 && g2 > (4.0 * tol * tol) * ab) atomicOr(flag, 1);
    double cs, sn;
    jacobi_cs(al, be, ga, cs, sn);
    for (int i = threadIdx.x; i < m; i += LJ_NT) {
        const double x = ca[i], y = cb[i];
        ca[i] = cs * x - sn * y;
        cb[i] = sn * x + cs * y;
    }
    if (V) {
        double *va = V + (long)a * k, *vb = V + (long)b * k;
        for (int i = threadIdx.x; i < k; i += LJ_NT) {
            const double x = va[i], y = vb[i];
            va[i] = cs * x - sn * y;
            vb[i] = sn * x + cs * y;
        }
    }
}

// Round t of the circle schedule over nblk (even) blocks of B columns, G lanes
// a pair.  NR > 0: the columns are padded with zeros to G NR rows in LDS (no
// guards; a lane holds NR rows of its pair in registers), and between the
// blocks' pairs column g of the first block stays in its group's registers, so
// only the second block goes through LDS.  NR = 0: columns of any length.  The
// rotation's scalar work (about 60 FP64 instructions, a chain of some 600
// cycles) is done by every lane of a group: sixteen lanes a pair, four pairs a
// wave, keeps it from filling the FP64 pipes, which a wave a pair did (192
// columns: 326 us a sweep that way).  ldc (odd): LDS stride of a column.
template <int B, int G, int NR>
__global__ __launch_bounds__(B * G) void k_lj_block(int m, int k, int nblk, int t, int ldc,
                                                    double *__restrict__ W,
                                                    double *__restrict__ V, double tol,
                                                    int *__restrict__ flag) {
    extern __shared__ double lds[];
    const int g = threadIdx.x / G, gl = threadIdx.x % G;
    int I, J;
    rr_pair(nblk, t, blockIdx.x, I, J);
    // columns beyond k belong to no pair; without a second block only the
    // pairs inside the first one are left (round 0)
    auto gcol = [&](int c) { return c < B ? I * B + c : J * B + (c - B); };
    if ((I * B >= k || J * B >= k) && t != 0) return;  // uniform per workgroup
    const int voff = NR > 0 ? G * NR : m;              // V's rows follow W's
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int c = g + h * B, gc = gcol(c);
        double *d = lds + (long)c * ldc;
        if (gc < k) {
            const double *w = W + (long)gc * m;
            for (int i = gl; i < (NR > 0 ? G * NR : m); i += G) d[i] = (i < m) ? w[i] : 0.0;
            if (V) {
                const double *v = V + (long)gc * k;
                for (int i = gl; i < (NR > 0 ? G * NR : k); i += G)
                    d[voff + i] = (i < k) ? v[i] : 0.0;
            }
        }
    }
    __syncthreads();
    bool open = false;
    const double tol2 = tol * tol;
    if (NR > 0 && t != 0) {
        constexpr int R = NR > 0 ? NR : 1;
        double *ca = lds + (long)g * ldc + gl;
        double x[R], v[R];
#pragma unroll
        for (int q = 0; q < R; q++) {
            x[q] = ca[G * q];
            v[q] = V ? ca[G * R + G * q] : 0.0;
        }
        for (int s = 0; s < B; s++) {
            const int b = B + ((g + s) & (B - 1));
            if (gcol(g) < k && gcol(b) < k) {  // uniform per group
                double *cb = lds + (long)b * ldc + gl;
                double y[R];
#pragma unroll
                for (int q = 0; q < R; q++) y[q] = cb[G * q];
                double al = 0.0, be = 0.0, ga = 0.0;
#pragma unroll
                for (int q = 0; q < R; q++) {
                    al += x[q] * x[q];
                    be += y[q] * y[q];
                    ga += x[q] * y[q];
                }
                group_allreduce3_q(al, be, ga, G);
                const double g2 = ga * ga, ab = al * be;
                if (g2 > tol2 * ab && al > 0.0 && be > 0.0) {
                    open = open || g2 > 4.0 * tol2 * ab;
                    double cs, sn;
                    jacobi_cs(al, be, ga, cs, sn);
#pragma unroll
                    for (int q = 0; q < R; q++) {
                        cb[G * q] = sn * x[q] + cs * y[q];
                        x[q] = cs * x[q] - sn * y[q];
                    }
                    if (V) {
#pragma unroll
                        for (int q = 0; q < R; q++) y[q] = cb[G * R + G * q];
#pragma unroll
                        for (int q = 0; q < R; q++) {
                            cb[G * R + G * q] = sn * v[q] + cs * y[q];
                            v[q] = cs * v[q] - sn * y[q];
                        }
                    }
                }
            }
            __syncthreads();
        }
#pragma unroll
        for (int q = 0; q < R; q++) {
            ca[G * q] = x[q];
            if (V) ca[G * R + G * q] = v[q];
        }
        __syncthreads();
    } else {
        const int len = NR > 0 ? (V ? 2 : 1) * G * NR : m + (V ? k : 0);
        const int steps = (t == 0) ? 2 * B - 1 : B;
        for (int s = 0; s < steps; s++) {
            int a, b;
            if (t == 0) {
                rr_pair_fast(2 * B, s, g, a, b);
            } else {
                a = g;
                b = B + ((g + s) & (B - 1));
            }
            if (gcol(a) < k && gcol(b) < k) {  // uniform per group
                double *ca = lds + (long)a * ldc, *cb = lds + (long)b * ldc;
                double al = 0.0, be = 0.0, ga = 0.0;
#pragma unroll 4
                for (int i = gl; i < m; i += G) {
                    const double x = ca[i], y = cb[i];
                    al += x * x;
                    be += y * y;
                    ga += x * y;
                }
                group_allreduce3_q(al, be, ga, G);
                const double g2 = ga * ga, ab = al * be;
                if (g2 > tol2 * ab && al > 0.0 && be > 0.0) {
                    open = open || g2 > 4.0 * tol2 * ab;
                    double cs, sn;
                    jacobi_cs(al, be, ga, cs, sn);
#pragma unroll 4
                    for (int i = gl; i < len; i += G) {
                        const double x = ca[i], y = cb[i];
                        ca[i] = cs * x - sn * y;
                        cb[i] = sn * x + cs * y;
                    }
                }
            }
            __syncthreads();
        }
    }
    if (open && gl == 0) atomicOr(flag, 1);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int c = g + h * B, gc = gcol(c);
        if (gc < k) {
            const double *d = lds + (long)c * ldc;
            double *w = W + (long)gc * m;
            for (int i = gl; i < m; i += G) w[i] = d[i];
            if (V) {
                double *v = V + (long)gc * k;
                for (int i = gl; i < k; i += G) v[i] = d[voff + i];
            }
        }
    }
}

// nrm[j] = ||W[:, j]||
__global__ __launch_bounds__(LJ_NT) void k_lj_colnorm(int m, const double *__restrict__ W,
                                                      double *__restrict__ nrm) {
    __shared__ double red[12];
    const int j = blockIdx.x;
    double s = 0.0, y = 0.0, z = 0.0;
    for (int i = threadIdx.x; i < m; i += LJ_NT) s += W[i + (long)j * m] * W[i + (long)j * m];
    lj_sum3(s, y, z, red);
    if (threadIdx.x == 0) nrm[j] = sqrt(s);
}

// descending order by rank counting (ties by index)
__global__ void k_lj_rank(int k, const double *__restrict__ nrm, int *__restrict__ pos) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= k) return;
    const double sj = nrm[j];
    int p = 0;
    for (int i = 0; i < k; i++) {
        const double si = nrm[i];
        p += (si > sj) || (si == sj && i < j);
    }
    pos[j] = p;
}

// sig, U (and V) in descending order
__global__ void k_lj_emit(int m, int k, const double *__restrict__ W,
                          const double *__restrict__ Vw, const double *__restrict__ nrm,
                          const int *__restrict__ pos, const int *__restrict__ dexp,
                          double *__restrict__ sig, double *__restrict__ sorted,
                          double *__restrict__ U, long ldu, double *__restrict__ V, long ldv) {
    const long mk = (long)m * k, kk = V ? (long)k * k : 0;
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < mk + kk;
         t += (long)gridDim.x * blockDim.x) {
        if (t < mk) {
            const long j = t / m, i = t - j * m;
            const double s = nrm[j];
            U[i + (long)pos[j] * ldu] = s > 0.0 ? W[t] / s : 0.0;
            if (i == 0) {
                sig[pos[j]] = ldexp(s, *dexp);
                sorted[pos[j]] = s;
            }
        } else {
            const long u = t - mk, j = u / k, i = u - j * k;
            V[i + (long)pos[j] * ldv] = Vw[u];
        }
    }
}

// numerical rank (sqrt(k) u s0) and the tail rule, as the one-workgroup kernel
__global__ void k_lj_finish(int k, const double *__restrict__ sorted, const int *__restrict__ dexp,
                            double log_scale, double delta, int cap, int sweeps,
                            int *__restrict__ iout) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const double s0 = sorted[0];
    const double thr = sqrt((double)k) * 0x1.0p-53 * s0;
    int numrank = 0;
    for (int j = 0; j < k; j++) numrank += (sorted[j] > thr) && (s0 > 0.0);
    int rho = numrank;
    double tail = 0.0;
    const double ld = delta > 0.0 ? log(delta) : -INFINITY;
    for (int q = numrank - 1; q >= 0; q--) {
        const double v = sorted[q];
        tail += v * v;
        const double lhs =
            (tail > 0.0) ? 0.5 * log(tail) + log_scale + *dexp * 0.6931471805599453 : -INFINITY;
        if (delta > 0.0 && lhs < ld) rho = q;
        else break;
    }
    if (rho > k) rho = k;
    if (rho > cap) rho = cap;
    if (rho < 1) rho = 1;
    iout[0] = numrank;
    iout[1] = rho;
    iout[2] = sweeps;
}

__global__ void k_svd_factors(int m, int rhomax, const int *__restrict__ drho,
                              const double *__restrict__ U, long ldu,
                              const double *__restrict__ sig, double wscale, double *W,
                              double *US) {
    const int rho = drho ? *drho : rhomax;
    long total = (long)m * rhomax;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total;
         e += (long)gridDim.x * blockDim.x) {
        int j = (int)(e / m), i = (int)(e - (long)j * m);
        if (j >= rho) continue;
        double u = U[i + (long)j * ldu], s = sig[j];
        if (US) US[i + (long)j * m] = u * s;
        if (W) W[j + (long)i * rho] = (s > 0.0) ? wscale * u / s : 0.0;
    }
}

// Symmetric permutation of a c x c Gram by descending diagonal (ties by
// index; NaN sorts last): perm[pos] = j, Gp = G[perm, perm].  Cholesky of Gp
// then yields a factor whose columns are ordered by decreasing norm, which
// cuts the one-sided Jacobi sweeps on its transpose (the diagonal-pivoting
// preconditioner of Drmac and Veselic, SIAM J. Matrix Anal. Appl. 29, 2008,
// applied statically).
constexpr int SORT_MAXC = 1024;
__global__ __launch_bounds__(1024) void k_sym_sort_perm(int c, const double *__restrict__ G,
                                                         double *__restrict__ Gp,
                                                         int *__restrict__ perm) {
    __shared__ double sd[SORT_MAXC];
    __shared__ int sp[SORT_MAXC];
    const int tid = threadIdx.x, hw = tid >> 5, hl = tid & 31, nhw = blockDim.x >> 5;
    for (int j = tid; j < c; j += blockDim.x) {
        double v = G[j + (long)j * c];
        sd[j] = (v == v) ? v : -INFINITY;
    }
    __syncthreads();
    for (int j = tid; j < c; j += blockDim.x) {
        const double dj = sd[j];
        int pos = 0;
        for (int i = 0; i < c; i++) {
            const double di = sd[i];
            pos += (di > dj) || (di == dj && i < j);
        }
        sp[pos] = j;
        perm[pos] = j;
    }
    __syncthreads();
    // one half-wave per column of Gp, 32 consecutive rows per pass
    for (int k = hw; k < c; k += nhw) {
        const double *gk = G + (long)sp[k] * c;
        for (int i = hl; i < c; i += 32) Gp[i + (long)k * c] = gk[sp[i]];
    }
}

// Zeroes the columns of L (m x k, ld) of smallest norm whose squared norms
// sum to at most budget * max_j ||L_j||^2; the sum dropped is written to
// *dropped.  Exactly-zero columns take no part in the Jacobi rotations, so
// columns whose content is below the Gram's own rounding stop costing sweeps.
__global__ __launch_bounds__(1024) void k_drop_small_cols(int m, int k, double *__restrict__ L,
                                                           long ld, double budget,
                                                           double *__restrict__ dropped) {
    __shared__ double sn[SORT_MAXC];
    __shared__ int so[SORT_MAXC];
    __shared__ int sdrop[SORT_MAXC];
    const int tid = threadIdx.x, hw = tid >> 5, hl = tid & 31, nhw = blockDim.x >> 5;
    // squared column norms, one half-wave per column (coalesced rows)
    for (int j = hw; j < k; j += nhw) {
        double s = 0.0;
        for (int i = hl; i < m; i += 32) {
            const double v = L[i + j * ld];
            s += v * v;
        }
        for (int o = 16; o > 0; o >>= 1) s += __shfl_xor(s, o, 32);
        if (hl == 0) {
            sn[j] = (s == s) ? s : INFINITY;
            sdrop[j] = 0;
        }
    }
    __syncthreads();
    // ascending order (ties by index); the largest norm is the last one
    for (int j = tid; j < k; j += blockDim.x) {
        const double sj = sn[j];
        int pos = 0;
        for (int i = 0; i < k; i++) pos += (sn[i] < sj) || (sn[i] == sj && i < j);
        so[pos] = j;
    }
    __syncthreads();
    if (tid == 0) {
        const double mx = fmax(sn[so[k - 1]], 0.0);
        const double lim = budget * mx;
        double cum = 0.0;
        for (int q = 0; q < k; q++) {
            const double v = sn[so[q]];
            if (!(cum + v <= lim) || v >= mx) break;
            cum += v;
            sdrop[so[q]] = 1;
        }
        *dropped = cum;
    }
    __syncthreads();
    for (int j = hw; j < k; j += nhw)
        if (sdrop[j])
            for (int i = hl; i < m; i += 32) L[i + j * ld] = 0.0;
}

// dst[perm[i] + j*ldd] = src[i + j*lds], i < m, j < n.
__global__ void k_unpermute_rows(int m, int n, const int *__restrict__ perm,
                                 const double *__restrict__ src, long lds,
                                 double *__restrict__ dst, long ldd) {
    const long total = (long)m * n;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total;
         e += (long)gridDim.x * blockDim.x) {
        const long j = e / m, i = e - j * m;
        dst[perm[i] + j * ldd] = src[i + j * lds];
    }
}

__global__ void k_permute_rows(int m, int n, const int *__restrict__ perm,
                               const double *__restrict__ src, long lds,
                               double *__restrict__ dst, long ldd) {
    const long total = (long)m * n;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total;
         e += (long)gridDim.x * blockDim.x) {
        const long j = e / m, i = e - j * m;
        dst[i + j * ldd] = src[perm[i] + j * lds];
    }
}

// 0: small SVDs on the one-workgroup kernel too (PARATT_AMD_SVD_NO_WAVE=1)
int g_svd_wave = [] {
    const char *e = getenv("PARATT_AMD_SVD_NO_WAVE");
    return (e && e[0] == '1') ? 0 : 1;
}();

template <typename KF>
void set_lds_attr(KF kern, int ndoubles) {
    HIPCHECK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                 ndoubles * (int)sizeof(double)));
}

void allow_big_lds() {
    static bool done = false;
    if (done) return;
    set_lds_attr(k_chol_blk<8, true>, chol_geom<8>::LDS_DOUBLES);
    set_lds_attr(k_chol_blk<8, false>, chol_geom<8>::LDS_DOUBLES);
    set_lds_attr(k_svd_jacobi, SVD_LDS_DOUBLES);
    set_lds_attr(k_svd_jacobi_wave<4, 2>, SVW_LDS_DOUBLES);
    set_lds_attr(k_svd_jacobi_wave<4, 4>, SVW_LDS_DOUBLES);
    set_lds_attr(k_svd_jacobi_wave<4, 8>, SVW_LDS_DOUBLES);
    set_lds_attr(k_svd_jacobi_wave<4, 16>, SVW_LDS_DOUBLES);
    set_lds_attr(k_svd_jacobi_wave<8, 2>, SVW_LDS_DOUBLES);
    set_lds_attr(k_svd_jacobi_wave<8, 4>, SVW_LDS_DOUBLES);
    set_lds_attr(k_svd_jacobi_wave<8, 8>, SVW_LDS_DOUBLES);
    set_lds_attr(k_svd_jacobi_wave<16, 2>, SVW_LDS_DOUBLES);
    set_lds_attr(k_svd_jacobi_wave<16, 4>, SVW_LDS_DOUBLES);
    set_lds_attr(k_lj_block<16, 16, 8>, LJ_LDS_DOUBLES);
    set_lds_attr(k_lj_block<16, 16, 12>, LJ_LDS_DOUBLES);
    set_lds_attr(k_lj_block<16, 16, 16>, LJ_LDS_DOUBLES);
    set_lds_attr(k_lj_block<8, 32, 0>, LJ_LDS_DOUBLES);
    set_lds_attr(k_lj_block<2, 64, 0>, LJ_LDS_DOUBLES);
    done = true;
}

// k_chol_blk with NB blocks of 16 columns, with the inverse when T is given.
template <int NB>
void launch_chol(const char *nm, double fl, double by, int c, const double *G, long ldg,
                 double shift, double tiny, double *R, double *T, long ldo, int *info,
                 double *dinfo, int want_kappa, int unit) {
    const size_t need = chol_geom<NB>::LDS_DOUBLES * sizeof(double);
    if (T)
        PTT_LAUNCH_FB(nm, fl, by, (k_chol_blk<NB, true>), dim3(1), dim3(64 * NB), need, c, G, ldg,
                      shift, tiny, R, T, ldo, info, dinfo, want_kappa, unit);
    else
        PTT_LAUNCH_FB(nm, fl, by, (k_chol_blk<NB, false>), dim3(1), dim3(64 * NB), need, c, G, ldg,
                      shift, tiny, R, T, ldo, info, dinfo, want_kappa, unit);
}

// One launch a round of block pairs (see k_lj_block).
template <int B, int G, int NR>
void lj_block_sweep(int m, int k, double *W, double *V, double tol, int *flag) {
    const int ldc = (NR > 0 ? (V ? 2 : 1) * G * NR : m + (V ? k : 0)) | 1;
    int nblk = (k + B - 1) / B;
    nblk += nblk & 1;
    const size_t shm = sizeof(double) * 2 * B * (size_t)ldc;
    for (int t = 0; t < nblk - 1; t++)
        PTT_LAUNCH("lj_block", (k_lj_block<B, G, NR>), dim3(nblk / 2), dim3(B * G), shm, m, k, nblk,
                   t, ldc, W, V, tol, flag);
}

// Jacobi SVD of an m x k matrix over many workgroups (outputs as ptt_hip_svd_jacobi).
// Sweeps run until one sweep leaves no pair unsettled (one flag read per
// sweep), at most 40 as in the one-workgroup kernel.
void svd_jacobi_large(int m, int k, const double *A, long lda, double *sig, double *U, long ldu,
                      double *V, long ldv, double log_scale, double delta, int cap, int *iout) {
    const size_t mk = (size_t)m * k, kk = V ? (size_t)k * k : 0;
    const size_t doubles = mk + kk + 3 * (size_t)k;
    char *ws = (char *)ptt_hip_scratch(PTT_WS_SKETCH,
                                       doubles * sizeof(double) + sizeof(int) * ((size_t)k + 8));
    double *W = (double *)ws, *Vw = V ? W + mk : nullptr;
    double *colmax = W + mk + kk, *nrm = colmax + k, *sorted = nrm + k;
    int *flag = (int *)(sorted + k), *dexp = flag + 2, *pos = flag + 4;  // flag 8-byte aligned
    const long total = (long)(mk + kk);
    PTT_LAUNCH("lj_colmax", k_lj_colmax, dim3(k), dim3(LJ_NT), 0, m, A, lda, colmax);
    PTT_LAUNCH("lj_exponent", k_lj_exponent, dim3(1), dim3(LJ_NT), 0, k, colmax, dexp);
    PTT_LAUNCH("lj_load", k_lj_load, dim3(stream_blocks(total, 256)), dim3(256), 0, m, k, A, lda,
               dexp, W, Vw);
    const int kp = k + (k & 1), P = kp / 2;
    const long ldc = (m + (V ? k : 0)) | 1;  // LDS stride of a column
    const int most = m > k ? m : k;
    const double tol = 0x1.0p-53 * (double)m;
    const int max_sweeps = 40;
    int sweep = 0;
    for (; sweep < max_sweeps; sweep++) {
        ptt_hip_zero(flag, sizeof(double));
        // blocks of 16 columns while two of them fit in LDS, then 8, then 2
        if (most <= 128)
            lj_block_sweep<16, 16, 8>(m, k, W, Vw, tol, flag);
        else if (most <= 192)
            lj_block_sweep<16, 16, 12>(m, k, W, Vw, tol, flag);
        else if (most <= 256)
            lj_block_sweep<16, 16, 16>(m, k, W, Vw, tol, flag);
        else if (16 * ldc <= LJ_LDS_DOUBLES)
            lj_block_sweep<8, 32, 0>(m, k, W, Vw, tol, flag);
        else if (4 * ldc <= LJ_LDS_DOUBLES)
            lj_block_sweep<2, 64, 0>(m, k, W, Vw, tol, flag);
        else
            for (int t = 0; t < kp - 1; t++)
                PTT_LAUNCH("lj_round", k_lj_round, dim3(P), dim3(LJ_NT), 0, m, k, kp, t, W, Vw, tol,
                           flag);
        int f = 0;
        ptt_hip_d2h(&f, flag, sizeof(int));
        if (!f) break;
    }
    const int sweeps = (sweep < max_sweeps) ? sweep + 1 : max_sweeps;
    PTT_LAUNCH("lj_colnorm", k_lj_colnorm, dim3(k), dim3(LJ_NT), 0, m, W, nrm);
    PTT_LAUNCH("lj_rank", k_lj_rank, dim3((k + 255) / 256), dim3(256), 0, k, nrm, pos);
    PTT_LAUNCH("lj_emit", k_lj_emit, dim3(stream_blocks(total, 256)), dim3(256), 0, m, k, W, Vw,
               nrm, pos, dexp, sig, sorted, U, ldu, V, ldv);
    PTT_LAUNCH("lj_finish", k_lj_finish, dim3(1), dim3(64), 0, k, sorted, dexp, log_scale, delta,
               cap, sweeps, iout);
}

}  // namespace

extern "C" {

void ptt_hip_chol_qr_factor(int c, const double *G, double shift, double tiny, double *R,
                            double *T, int *info, double *dinfo, int want_kappa) {
    ptt_hip_init();
    allow_big_lds();
    if (c <= 128) {
        const char *nm = T ? "chol_qr_factor" : "chol_factor_only";
        const double fl = 2.0 * c * (double)c * c / 3.0, by = 8.0 * 3.0 * c * (double)c;
        const int wk = T ? want_kappa : 0;
        // the fewest waves whose blocks hold c columns; beyond four blocks all eight
        // waves, whose spare ones take part in the tile products
        if (c <= 16)
            launch_chol<1>(nm, fl, by, c, G, c, shift, tiny, R, T, c, info, dinfo, wk, 0);
        else if (c <= 32)
            launch_chol<2>(nm, fl, by, c, G, c, shift, tiny, R, T, c, info, dinfo, wk, 0);
        else if (c <= 48)
            launch_chol<3>(nm, fl, by, c, G, c, shift, tiny, R, T, c, info, dinfo, wk, 0);
        else if (c <= 64)
            launch_chol<4>(nm, fl, by, c, G, c, shift, tiny, R, T, c, info, dinfo, wk, 0);
        else
            launch_chol<8>(nm, fl, by, c, G, c, shift, tiny, R, T, c, info, dinfo, wk, 0);
        return;
    }
    // blocks of 128 columns
    const int nblk = (c + 127) / 128;
    const size_t cc = (size_t)c * c;
    double *ws = (double *)ptt_hip_scratch(
        PTT_WS_SKETCH, sizeof(double) * (2 * cc + 128 * (size_t)c + 4 * (size_t)c + 4 * nblk) +
                           sizeof(int) * (size_t)nblk);
    double *S = ws, *Tw = S + cc, *X = Tw + cc, *D = X + 128 * (size_t)c, *iD = D + c, *y = iD + c,
           *z = y + c;
    double *bd = z + c;
    int *bi = (int *)(bd + 4 * nblk);
    double *Ti = T ? T : Tw;  // the diagonal blocks' inverses are needed either way
    if (T && nblk > 2) ptt_hip_zero(T, sizeof(double) * cc);  // its lower blocks are operands
    PTT_LAUNCH("chol_scale", k_chol_scale, dim3(stream_blocks((long)cc, 256)), dim3(256), 0, c, G,
               shift, D, iD, S);
    for (int b = 0; b < nblk; b++) {
        const int b0 = 128 * b, cb = c - b0 < 128 ? c - b0 : 128, rest = c - b0 - cb;
        const size_t dg = (size_t)b0 + (size_t)b0 * c;
        launch_chol<8>("chol_qr_factor", 2.0 * cb * (double)cb * cb / 3.0, 24.0 * cb * (double)cb, cb,
                       S + dg, c, 0.0, tiny, R + dg, Ti + dg, c, bi + b, bd + 4 * b, 0, 1);
        if (rest > 0) {
            const size_t right = dg + (size_t)cb * c, trail = right + cb;
            ptt_hip_dgemm('T', 'N', cb, rest, cb, 1.0, Ti + dg, c, S + right, c, 0.0, R + right, c);
            ptt_hip_dgemm('T', 'N', rest, rest, cb, -1.0, R + right, c, R + right, c, 1.0,
                          S + trail, c);
        }
        if (T && b > 0) {
            // T[0:b0, b] = -T[0:b0, 0:b0] R[0:b0, b] T_bb
            const size_t up = (size_t)b0 * c;
            ptt_hip_dgemm('N', 'N', b0, cb, cb, -1.0, R + up, c, Ti + dg, c, 0.0, X, b0);
            ptt_hip_dgemm('N', 'N', b0, cb, b0, 1.0, T, c, X, b0, 0.0, T + up, c);
        }
    }
    PTT_LAUNCH("chol_unscale", k_chol_unscale, dim3(stream_blocks((long)cc, 256)), dim3(256), 0, c,
               D, R, T);
    PTT_LAUNCH("chol_report", k_chol_report, dim3(1), dim3(NT), 0, c, G, D, iD, R, T, nblk, bi, y, z,
               info, dinfo, want_kappa);
}

void ptt_hip_svd_jacobi(int m, int k, double *A, long lda, double *sig, double *U, long ldu,
                        double *V, long ldv, double log_scale, double delta, int cap,
                        int *iout) {
    ptt_hip_init();
    allow_big_lds();
    if (m <= 0 || k <= 0) return;
    // LDS footprint of the one-workgroup kernel's padded columns
    const size_t lds_need = (size_t)(m | 1) * k + (V ? (size_t)(k | 1) * k : 0);
    if (k > SVD_ONE_WG_MAX || (lds_need > (size_t)SVD_LDS_DOUBLES && !(k <= SVW_K && m <= SVW_M))) {
        svd_jacobi_large(m, k, A, lda, sig, U, ldu, V, ldv, log_scale, delta, cap, iout);
        return;
    }
    if (k <= SVW_K && m <= SVW_M && g_svd_wave) {
        // G lanes per pair: 4 for up to 16 pairs, 8 for 8, 16 for 4; R rows
        // per lane.  (Two lanes per pair for k up to 64 measured slower than
        // the one-workgroup kernel: every round's LDS traffic then sits on
        // two lanes' critical path.)
        const int P = (k + 1) / 2;
        const int G = P > 8 ? 4 : (P > 4 ? 8 : 16);
        const int Rneed = (m + G - 1) / G;
        const int R = Rneed <= 2 ? 2 : (Rneed <= 4 ? 4 : (Rneed <= 8 ? 8 : 16));
        const size_t shm = (size_t)SVW_LDS_DOUBLES * sizeof(double);
        const double fl = 4.0 * m * (double)k * k + (V ? 9.0 * k * (double)k * k : 0.0);
        const double by = 8.0 * (2.0 * m * (double)k + k);
#define PTT_SVW(G_, R_)                                                                     \
    PTT_LAUNCH_FB("svd_jacobi_wave", fl, by, (k_svd_jacobi_wave<G_, R_>), dim3(1), dim3(64), shm, \
                  m, k, A, lda, sig, U, ldu, V, ldv, log_scale, delta, cap, iout)
        if (G == 4) {
            if (R == 2) PTT_SVW(4, 2);
            else if (R == 4) PTT_SVW(4, 4);
            else if (R == 8) PTT_SVW(4, 8);
            else PTT_SVW(4, 16);
        } else if (G == 8) {
            if (R == 2) PTT_SVW(8, 2);
            else if (R == 4) PTT_SVW(8, 4);
            else PTT_SVW(8, 8);
        } else {
            if (R == 2) PTT_SVW(16, 2);
            else PTT_SVW(16, 4);
        }
#undef PTT_SVW
        return;
    }
    // algorithmic work of a dense SVD with left vectors (Golub-Reinsch
    // count 4 m k^2 + 8 k^3, 9 k^3 for the right vectors)
    const double svd_flops = 4.0 * m * (double)k * k + 8.0 * (double)k * k * k;
    const double svd_bytes = 8.0 * (2.0 * m * (double)k + k);
    // threads: each Jacobi pair gets G lanes with about SVD_RV rows per lane, the
    // whole workgroup holding all pairs of a round (one wave at least)
    const int kp0 = k + (k & 1), P0 = kp0 / 2;
    int Gw = 1;
    while (Gw < 64 && Gw * SVD_RV < m) Gw <<= 1;
    int nth = P0 * Gw;
    nth = ((nth + 63) / 64) * 64;
    if (nth > SVD_NT) nth = SVD_NT;
    if (nth < 64) nth = 64;
    PTT_LAUNCH_FB("svd_jacobi", svd_flops + (V ? 9.0 * k * (double)k * k : 0.0), svd_bytes,
                  k_svd_jacobi, dim3(1), dim3(nth), lds_need * sizeof(double), m, k, A, lda, sig, U,
                  ldu, V, ldv, log_scale, delta, cap, iout);
}

void ptt_hip_svd_factors(int m, int rhomax, const int *drho, const double *U, long ldu,
                         const double *sig, double wscale, double *W, double *US) {
    ptt_hip_init();
    long total = (long)m * rhomax;
    if (total <= 0) return;
    PTT_LAUNCH("svd_factors", k_svd_factors, dim3(stream_blocks(total, 256)), dim3(256), 0, m,
               rhomax, drho, U, ldu, sig, wscale, W, US);
}

void ptt_hip_sym_sort_perm(int c, const double *G, double *Gp, int *perm) {
    ptt_hip_init();
    if (c <= 0) return;
    if (c > SORT_MAXC) {
        fprintf(stderr, "ptt_hip_sym_sort_perm: c = %d exceeds %d\n", c, SORT_MAXC);
        exit(1);
    }
    PTT_LAUNCH("sym_sort_perm", k_sym_sort_perm, dim3(1), dim3(1024), 0, c, G, Gp, perm);
}

void ptt_hip_drop_small_cols(int m, int k, double *L, long ld, double budget, double *dropped) {
    ptt_hip_init();
    if (m <= 0 || k <= 0) return;
    if (k > SORT_MAXC) {
        fprintf(stderr, "ptt_hip_drop_small_cols: k = %d exceeds %d\n", k, SORT_MAXC);
        exit(1);
    }
    PTT_LAUNCH("drop_small_cols", k_drop_small_cols, dim3(1), dim3(1024), 0, m, k, L, ld, budget,
               dropped);
}

void ptt_hip_unpermute_rows(int m, int n, const int *perm, const double *src, long lds,
                            double *dst, long ldd) {
    ptt_hip_init();
    long total = (long)m * n;
    if (total <= 0) return;
    PTT_LAUNCH("unpermute_rows", k_unpermute_rows, dim3(stream_blocks(total, 256)), dim3(256), 0,
               m, n, perm, src, lds, dst, ldd);
}

void ptt_hip_permute_rows(int m, int n, const int *perm, const double *src, long lds,
                          double *dst, long ldd) {
    ptt_hip_init();
    const long total = (long)m * n;
    if (total <= 0) return;
    PTT_LAUNCH("permute_rows", k_permute_rows, dim3(stream_blocks(total, 256)), dim3(256), 0,
               m, n, perm, src, lds, dst, ldd);
}

void ptt_hip_trmm_small(int c, const double *A, const double *B, double *C) {
    ptt_hip_dgemm('N', 'N', c, c, c, 1.0, A, c, B, c, 0.0, C, c);
}

}  // extern "C"
