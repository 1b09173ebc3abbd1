// tsqr.hip -- rounding of low-rank trains (bond ranks up to 32) without a host
// round trip per bond, gfx950.
//
// A bond matrix of at most 32 columns is factored by Householder reflectors in
// a tree: a workgroup holds a block of rows in registers, its reflectors V stay
// where the rows were, and the c x c factors of the blocks are stacked and
// factored in turn until one block is left.  Q is never formed: it is applied
// to a small matrix X from the root down, each block as [X; 0] - V (F X) with
// F = T V_top^T (T the block's compact WY factor), whose tall product runs on
// the matrix cores.  The root of a right-to-left bond also takes the small SVD
// (column-pivoted QR, then one-sided Jacobi on the transposed factor), the
// reference's rank rule, and the application of its own reflectors, so a bond
// is a fixed sequence of launches and every rank stays on the device until the
// sweep ends.
//
// What bounds it: the chain of reflectors (one barrier each; measured 0.4 us a
// reflector at 16 columns, 0.75-1.2 at 32) and of Jacobi rounds (0.45 us each).
// A block of 512 rows takes 16 us at 16 columns and 43 at 32, the root with its
// SVD 55-75 us at 16 columns and 120-180 at 32.  The Cholesky-QR passes it
// replaces cost a Gram, a reduction, a factorisation (25 us at 20 columns), a
// host read and a product each, three or four passes on rank-deficient sums;
// Householder needs one pass whatever the condition.
#include "common.hpp"

#include <type_traits>

using namespace ptt;

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int TQ_NT = 256;  // threads of a block's workgroup
constexpr int TQ_C = 32;    // columns at most; also ld of F and X
constexpr int TQ_LD = 33;   // LDS stride of small matrices

// Layout of a block: a row of 16 lanes holds one part's rows, part + 16 s for
// s < RP; lane li of it columns li + 16 k, k < NC.  The pivot column's rows thus
// reach every column by a lane broadcast inside the 16-lane row (one
// instruction a value): no LDS and no barrier.  (Published through LDS, by 512
// threads with a column each, a reflector took 2.1 us at 512 x 32.)
template <int NC, int RP>
struct Lay {
    static constexpr int ROWS = 16 * RP;
    static constexpr int RW = 16 * NC;                   // columns held
    static constexpr int QR_LDS = 2 * RW + 2 * 4 * RW;   // rowj, red
    static constexpr int MAT = RW * TQ_LD;               // a small matrix in LDS
    static_assert(NC <= RP, "the rows of R are the first NC of every part");
};

// Householder QR of the block held in a (c <= 16 NC columns; rows beyond the
// block are zero).  On return a holds the reflectors V (unnormalised, H_j = I -
// tau_j v_j v_j^T; zero above the diagonal), Rm (LDS, row-major stride TQ_LD) R,
// Mm (LDS, the same) the products v_l . v_j above the diagonal, tau (LDS, RW)
// the scalars.  H_0 ... H_{c-1} = I - V T V^T with T^-1 = diag(1 / tau) +
// striu(Mm).  One barrier a reflector: the partial products of every column
// with the pivot column, summed over the parts of a wave, meet in LDS
// (double-buffered).
template <int NC, int RP>
__device__ __forceinline__ void qr_block(double (&a)[NC][RP], int c, double *lds, double *Rm,
                                         double *Mm, double *tau) {
    typedef Lay<NC, RP> L;
    double *rowj = lds, *red = lds + 2 * L::RW;
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    __syncthreads();
    for (int e = tid; e < L::MAT; e += TQ_NT) {
        Rm[e] = 0.0;
        Mm[e] = 0.0;
    }
    if (tid < L::RW) tau[tid] = 0.0;
    __syncthreads();
    // columns 16 h .. 16 h + 15 are set 0 during turn h: the sets rotate by one a
    // turn and are back in place after NC
    for (int h = 0; h < NC; h++) {
        auto step = [&](auto jc) {
            constexpr int JJ = decltype(jc)::value, B = JJ & 1;
            const int j = 16 * h + JJ;
            if (j >= c) return;  // uniform
            int li = tid & 15, part = tid >> 4;
            // the comparisons below are made where they are used: hoisted, the
            // sixteen steps' masks fill the scalar registers and spill
            __asm__ volatile("" : "+v"(li), "+v"(part));
            double v[RP];
#pragma unroll
            for (int s = 0; s < RP; s++) v[s] = row_bcast<JJ>(a[0][s]);
            double t[NC];
#pragma unroll
            for (int k = 0; k < NC; k++) {
                double t0 = 0.0, t1 = 0.0, t2 = 0.0, t3 = 0.0;
#pragma unroll
                for (int s = 0; s < RP; s += 4) {
                    t0 += v[s] * a[k][s];
                    t1 += v[s + 1] * a[k][s + 1];
                    t2 += v[s + 2] * a[k][s + 2];
                    t3 += v[s + 3] * a[k][s + 3];
                }
                t[k] = xor32_sum(xor16_sum((t0 + t1) + (t2 + t3)));
            }
            if (lane < 16) {
#pragma unroll
                for (int k = 0; k < NC; k++) red[(B * 4 + wv) * L::RW + li * NC + k] = t[k];
            }
            if (part == JJ) {
#pragma unroll
                for (int s = 0; s < NC; s++)
                    if (s == h) {
#pragma unroll
                        for (int k = 0; k < NC; k++) rowj[B * L::RW + li * NC + k] = a[k][s];
                    }
            }
            __syncthreads();
            double S[NC], aj[NC];
#pragma unroll
            for (int k = 0; k < NC; k++) {
                S[k] = 0.0;
                aj[k] = rowj[B * L::RW + li * NC + k];
            }
#pragma unroll
            for (int w = 0; w < 4; w++)
#pragma unroll
                for (int k = 0; k < NC; k++) S[k] += red[(B * 4 + w) * L::RW + li * NC + k];
            const double sj = row_bcast<JJ>(S[0]), alpha = row_bcast<JJ>(aj[0]);
            double beta = alpha, v0 = 0.0, tj = 0.0;
            if (sj > 0x1.0p-1000) {  // below: the column is zero to working accuracy
                const double nrm = sqrt_nr(sj);
                beta = alpha > 0.0 ? -nrm : nrm;
                v0 = alpha - beta;
                tj = rcp_nr(sj + fabs(alpha) * nrm);  // 2 / v^T v
            }
            double dot[NC], f[NC];
#pragma unroll
            for (int k = 0; k < NC; k++) {
                dot[k] = S[k] - beta * aj[k];  // v has v0 = alpha - beta in row j
                const bool after = k == 0 ? li > JJ : h + k < NC;
                f[k] = after ? tj * dot[k] : 0.0;
                if (k == 0 || h + k < NC) {
#pragma unroll
                    for (int s = 0; s < RP; s++) a[k][s] -= f[k] * v[s];
                }
            }
            // row j leaves the block: R's row for the later columns (zero here from
            // now on, so that no later pivot column reaches above its diagonal), v0
            // for the pivot column, the earlier columns' reflectors stay
            if (part == JJ) {
#pragma unroll
                for (int k = 0; k < NC; k++) {
                    const int col = ((h + k) % NC) * 16 + li;
                    const bool after = k == 0 ? li > JJ : h + k < NC;
                    const bool piv = k == 0 && li == JJ;
                    if (after || piv) Rm[j * TQ_LD + col] = piv ? beta : aj[k] - f[k] * v0;
                    if (!after && !piv) Mm[col * TQ_LD + j] = dot[k];
#pragma unroll
                    for (int s = 0; s < NC; s++)
                        if (s == h) a[k][s] = piv ? v0 : after ? 0.0 : a[k][s];
                }
                if (li == JJ) tau[j] = tj;
            }
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
        step(std::integral_constant<int, 4>{});
        step(std::integral_constant<int, 5>{});
        step(std::integral_constant<int, 6>{});
        step(std::integral_constant<int, 7>{});
        step(std::integral_constant<int, 8>{});
        step(std::integral_constant<int, 9>{});
        step(std::integral_constant<int, 10>{});
        step(std::integral_constant<int, 11>{});
        step(std::integral_constant<int, 12>{});
        step(std::integral_constant<int, 13>{});
        step(std::integral_constant<int, 14>{});
        step(std::integral_constant<int, 15>{});
        if constexpr (NC > 1) {
#pragma unroll
            for (int s = 0; s < RP; s++) {
                const double x = a[0][s];
#pragma unroll
                for (int k = 0; k + 1 < NC; k++) a[k][s] = a[k + 1][s];
                a[NC - 1][s] = x;
            }
        }
    }
    __syncthreads();
}

// Power of two that brings a block whose largest entry is amax into the range
// where squares neither overflow nor underflow; 0 for ordinary magnitudes.
__device__ __forceinline__ int block_exp(double amax) {
    if (!(amax > 0.0) || !(amax < INFINITY)) return 0;
    const int e = ilogb(amax);
    return (e > 400 || e < -400) ? e : 0;
}

// Largest value over the workgroup (red4: 4 doubles of LDS).
__device__ __forceinline__ double block_max(double m, double *red4) {
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red4[threadIdx.x >> 6] = m;
    __syncthreads();
    return fmax(fmax(red4[0], red4[1]), fmax(red4[2], red4[3]));
}
template <int NC, int RP>
__device__ __forceinline__ double block_absmax(const double (&a)[NC][RP], double *red4) {
    double m = 0.0;
#pragma unroll
    for (int k = 0; k < NC; k++)
#pragma unroll
        for (int s = 0; s < RP; s++) m = fmax(m, fabs(a[k][s]));
    return block_max(m, red4);
}

// F = T V_top^T (c x c) of the block into Fg (ld TQ_C): back substitution with
// T^-1, RW columns on consecutive lanes, the rows dealt to 256 / RW groups.
// vt: MAT doubles of LDS.
template <int NC, int RP>
__device__ __forceinline__ void form_f(const double (&a)[NC][RP], int c, const double *Mm,
                                       const double *tau, double *vt, double *__restrict__ Fg) {
    typedef Lay<NC, RP> L;
    constexpr int GR = TQ_NT / L::RW, PER = L::RW / GR;  // groups, rows of each
    const int tid = threadIdx.x, li = tid & 15, part = tid >> 4;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NC; k++)
#pragma unroll
        for (int s = 0; s < NC; s++)
            vt[(part + 16 * s) * TQ_LD + li + 16 * k] = a[k][s];
    __syncthreads();
    const int x = tid % L::RW, g = tid / L::RW;
    double w[PER > 0 ? PER : 1];  // V_top^T, rows g + GR q of column x: V[x][row]
#pragma unroll
    for (int q = 0; q < PER; q++) w[q] = vt[x * TQ_LD + g + GR * q];
    __syncthreads();
    for (int i = c - 1; i >= 0; i--) {
        if (g == i % GR) {
            double y = 0.0;
#pragma unroll
            for (int q = 0; q < PER; q++)
                if (q == i / GR) y = w[q];
            y *= tau[i];
            vt[(i & 1) * L::RW + x] = y;
            if (x < c) Fg[i + x * TQ_C] = y;
        }
        __syncthreads();
        const double y = vt[(i & 1) * L::RW + x];
#pragma unroll
        for (int q = 0; q < PER; q++) w[q] -= Mm[(g + GR * q) * TQ_LD + i] * y;
    }
}

struct QrArgs {
    double *A;              // the matrix, overwritten by the reflectors
    long rs, cs;            // element (row, col) at row * rs + col * cs
    long rows;              // rows, or rows per rank when drho is given
    const int *drho;        // device rank multiplying rows (NULL: 1)
    int c;                  // columns
    double *F;              // c x c per block, ld TQ_C, TQ_C^2 apart
    double *R;              // stacked factors: block b's row i at (b c + i) * c, or,
                            // for the root, c x c column-major (ld c)
    int root;               // 1: R column-major, brought into range with *escale
    int *escale;            // device exponent taken out of R (root)
};

// One level of the tree: block b of 16 RP rows -> V in place, R, F.
// COLMAJOR: rows contiguous (rs = 1), staged through LDS 16 columns at a time
// so that global accesses follow the rows while lanes own columns.
template <int NC, int RP, bool COLMAJOR>
__global__ __launch_bounds__(TQ_NT) void k_qr_block(QrArgs g) {
    typedef Lay<NC, RP> L;
    constexpr int TL = L::ROWS + 1;
    extern __shared__ double lds[];
    __shared__ double red4[4];
    const int tid = threadIdx.x, li = tid & 15, part = tid >> 4;
    const int c = g.c;
    const long rows = g.drho ? g.rows * (long)*g.drho : g.rows;
    const long r0 = (long)blockIdx.x * L::ROWS;
    const int nr = (int)(rows - r0 < L::ROWS ? rows - r0 : L::ROWS);
    double *R = g.root ? g.R : g.R + (long)blockIdx.x * c * c;
    double *Fg = g.F + (long)blockIdx.x * TQ_C * TQ_C;
    if (nr <= 0) {  // beyond a train whose rank came out smaller: an empty block
        for (int e = tid; e < c * c; e += TQ_NT) R[e] = 0.0;
        for (int e = tid; e < TQ_C * TQ_C; e += TQ_NT) Fg[e] = 0.0;
        return;
    }
    double a[NC][RP];
#pragma unroll
    for (int k = 0; k < NC; k++) {
        if constexpr (COLMAJOR) {
            if (k > 0) __syncthreads();
            for (int q = tid / 64; q < 16; q += TQ_NT / 64) {
                if (16 * k + q >= c) continue;
                const double *p = g.A + r0 + (16 * k + q) * g.cs;
#pragma unroll
                for (int r = tid % 64; r < L::ROWS; r += 64)
                    lds[q * TL + r] = (r < nr) ? p[r] : 0.0;
            }
            __syncthreads();
#pragma unroll
            for (int s = 0; s < RP; s++)
                a[k][s] = (li + 16 * k < c) ? lds[li * TL + part + 16 * s] : 0.0;
        } else {
            const int col = li + 16 * k;
            const double *p = g.A + r0 * g.rs + col * g.cs;
#pragma unroll
            for (int s = 0; s < RP; s++) {
                const int r = part + 16 * s;
                a[k][s] = (col < c && r < nr) ? p[r * g.rs] : 0.0;
            }
        }
    }
    const int ex = block_exp(block_absmax<NC, RP>(a, red4));
    if (ex != 0) {
#pragma unroll
        for (int k = 0; k < NC; k++)
#pragma unroll
            for (int s = 0; s < RP; s++) a[k][s] = ldexp(a[k][s], -ex);
    }
    double *Rm = lds + L::QR_LDS, *Mm = Rm + L::MAT, *tau = Mm + L::MAT, *vt = tau + L::RW;
    qr_block<NC, RP>(a, c, lds, Rm, Mm, tau);
    int eo = ex;
    if (g.root) {
        double m = 0.0;
        for (int e = tid; e < L::MAT; e += TQ_NT) m = fmax(m, fabs(Rm[e]));
        m = block_max(m, red4);
        if (m > 0.0 && m < INFINITY) {
            const int em = ilogb(m) + ex;  // exponent of R's largest entry
            if (em > 400 || em < -400) {
                eo = ex - em;
                if (tid == 0) atomicAdd(g.escale, em);
            }
        }
    }
    for (int e = tid; e < c * L::RW; e += TQ_NT) {
        const int i = e % L::RW, q = e / L::RW;
        if (i >= c) continue;
        // root: column q, row i; stacked: row q, column i (both contiguous)
        const double v = g.root ? Rm[i * TQ_LD + q] : Rm[q * TQ_LD + i];
        R[(long)q * c + i] = eo != 0 ? ldexp(v, eo) : v;
    }
    form_f<NC, RP>(a, c, Mm, tau, vt, Fg);
    // V in place
#pragma unroll
    for (int k = 0; k < NC; k++) {
        if constexpr (COLMAJOR) {
            __syncthreads();
#pragma unroll
            for (int s = 0; s < RP; s++) lds[li * TL + part + 16 * s] = a[k][s];
            __syncthreads();
            for (int q = tid / 64; q < 16; q += TQ_NT / 64) {
                if (16 * k + q >= c) continue;
                double *p = g.A + r0 + (16 * k + q) * g.cs;
#pragma unroll
                for (int r = tid % 64; r < L::ROWS; r += 64)
                    if (r < nr) p[r] = lds[q * TL + r];
            }
        } else {
            const int col = li + 16 * k;
            double *p = g.A + r0 * g.rs + col * g.cs;
#pragma unroll
            for (int s = 0; s < RP; s++) {
                const int r = part + 16 * s;
                if (col < c && r < nr) p[r * g.rs] = a[k][s];
            }
        }
    }
}

struct ApplyArgs {
    const double *V;   // reflectors, element (row, col) at row * rs + col * cs
    long rs, cs, rows;
    const int *drho;   // as in QrArgs
    int c, brows;      // columns, rows of a block
    const double *F;
    const double *X;   // c x p per block: block b's row i at (b c + i) * xr + q * xc
    long xr, xc;
    const int *p;      // device: columns of X
    double *Y;         // rows x p: element (row, q) at row * yr + q * yc; yr 0: yr = p
    long yr, yc;
    double alpha;
    int plain;         // V is an explicit Q: Y = alpha V X
};

// Y = alpha (I - V T V^T) [X; 0] for one block: Z = -F X in LDS, then V Z on
// the matrix cores, 16 rows a wave and step.  z: 3 TQ_C TQ_LD doubles of LDS.
// TR: the rows lie on the lanes of a store (yr = 1), else the columns do.
template <bool TR>
__device__ __forceinline__ void apply_block(const ApplyArgs &g, long blk, double *z) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    constexpr int nw = TQ_NT / 64;
    const int c = g.c, p = *g.p;
    const long rows = g.drho ? g.rows * (long)*g.drho : g.rows;
    const long r0 = blk * g.brows;
    const int nr = (int)(rows - r0 < g.brows ? rows - r0 : g.brows);
    if (nr <= 0) return;
    const double *F = g.plain ? nullptr : g.F + blk * TQ_C * TQ_C;
    const double *X = g.X + (g.plain ? 0 : blk * c * g.xr);
    const long yr = g.yr ? g.yr : p;
    double *x = z + TQ_C * TQ_LD, *f = x + TQ_C * TQ_LD;
#pragma unroll
    for (int e = tid; e < TQ_C * TQ_C; e += TQ_NT) {
        const int q = e % TQ_C, i = e / TQ_C;
        x[i * TQ_LD + q] = (i < c && q < p) ? X[i * g.xr + q * g.xc] : 0.0;
        f[i * TQ_LD + q] = (!g.plain && i < c && q < c) ? F[q + i * TQ_C] : 0.0;  // F^T
        if (g.plain) z[i * TQ_LD + q] = x[i * TQ_LD + q];
    }
    __syncthreads();
    if (!g.plain)
#pragma unroll
    for (int e = tid; e < TQ_C * TQ_C; e += TQ_NT) {
        const int q = e % TQ_C, i = e / TQ_C;
        double s0 = 0.0, s1 = 0.0;
#pragma unroll 8
        for (int l = 0; l < TQ_C; l += 2) {
            s0 += f[l * TQ_LD + i] * x[l * TQ_LD + q];
            s1 += f[(l + 1) * TQ_LD + i] * x[(l + 1) * TQ_LD + q];
        }
        z[i * TQ_LD + q] = -(s0 + s1);
    }
    __syncthreads();
    const int ks = (c + 3) >> 2, nq = (p + 15) >> 4;
    double zf[2][8];  // Z fragments: Z[4 kk + lane/16][16 h + lane%16]
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int kk = 0; kk < 8; kk++)
            zf[h][kk] = z[(4 * kk + (lane >> 4)) * TQ_LD + 16 * h + (lane & 15)];
    const double *V = g.V + r0 * g.rs;
    double *Y = g.Y + r0 * yr;
    for (int t = wv; 16 * t < nr; t += nw) {
        const int row = 16 * t + (lane & 15);
        double vf[8];
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
            const int k = 4 * kk + (lane >> 4);
            vf[kk] = (kk < ks && k < c && row < nr) ? V[row * g.rs + k * g.cs] : 0.0;
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (h >= nq) continue;
            f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int kk = 0; kk < 8; kk++)
                if (kk < ks)
                    acc = TR ? __builtin_amdgcn_mfma_f64_16x16x4f64(zf[h][kk], vf[kk], acc, 0, 0, 0)
                             : __builtin_amdgcn_mfma_f64_16x16x4f64(vf[kk], zf[h][kk], acc, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                // D[lane/16 + 4v][lane%16]
                const int rr = 16 * t + (TR ? (lane & 15) : (lane >> 4) + 4 * v);
                const int q = 16 * h + (TR ? (lane >> 4) + 4 * v : (lane & 15));
                if (rr < nr && q < p) {
                    double y = acc[v];
                    if (rr < c && !g.plain) y += x[rr * TQ_LD + q];
                    Y[rr * yr + q * g.yc] = g.alpha * y;
                }
            }
        }
    }
}

// Up to two independent applications a launch: blocks of the first, then of
// the second (a finished core and the next bond's matrix).
__global__ __launch_bounds__(TQ_NT) void k_qr_apply(ApplyArgs g0, ApplyArgs g1, int n0) {
    __shared__ double z[3 * TQ_C * TQ_LD];
    const bool second = (int)blockIdx.x >= n0;
    const ApplyArgs &g = second ? g1 : g0;
    const long blk = second ? (int)blockIdx.x - n0 : (int)blockIdx.x;
    if (g.yr == 1)
        apply_block<true>(g, blk, z);
    else
        apply_block<false>(g, blk, z);
}

// ---- the small SVD of a bond, on the workgroup of the tree's root -------------
// R (c x c upper, LDS): L = R^T = Q4 X^T by column-pivoted QR (stopped where the
// remaining columns fall below u |R_11|, far below the numerical rank's line),
// then one-sided Jacobi on X (c x r): X = U Sigma V^T, so U holds L's right
// singular vectors and no V is accumulated.  (Drmac and Veselic, SIAM J. Matrix
// Anal. Appl. 29, 2008: the transposed factor of a pivoted QR takes few sweeps.)
// The pivoted QR runs on one wave (columns on 16 lanes, two each; rows on its
// four parts; sums by lane swaps, no barriers), the rotations on sixteen lanes a
// pair, two rows a lane, one barrier a round.
constexpr int SV_LD = 33;

// Jacobi rotation zeroing the off-diagonal of [[al, ga], [ga, be]]: the tangent
// t = 2 ga / (d + sign(d) hypot(d, 2 ga)), d = be - al, only steers convergence
// (hardware reciprocals; columns of order one down to u, so nothing under- or
// overflows); c is refined so that c^2 + s^2 = 1 to working accuracy.
__device__ __forceinline__ void sv_rotation(double al, double be, double ga, double &c, double &s) {
    const double d = be - al, g2 = ga + ga;
    const double h2 = fma(d, d, g2 * g2);
    const double hyp = h2 * __builtin_amdgcn_rsq(h2);
    double t = g2 * __builtin_amdgcn_rcp(fabs(d) + hyp);
    if (d < 0.0) t = -t;
    const double w = fma(t, t, 1.0);
    double y = __builtin_amdgcn_rsq(w);
    y = y * (1.5 - 0.5 * w * y * y);
    y = y * (1.5 - 0.5 * w * y * y);
    c = y;
    s = y * t;
}

// Jacobi sweeps over the r <= 32 columns (32 rows, LDS stride SV_LD) of X by the
// workgroup, sixteen lanes a pair.  nrm (32 doubles of LDS) carries the squared
// norms through a sweep (al - t ga, be + t ga), so a round reduces one product;
// flag: 4 ints of LDS.  A sweep whose largest cosine is below 1e-8 is followed
// by a test of every pair instead of another sweep.  Returns the sweeps taken.
__device__ int sv_sweeps(double *X, int r, int c, double *nrm, int *flag) {
    const int tid = threadIdx.x, g = tid >> 4, gl = tid & 15;
    const int kp = r + (r & 1), P = kp / 2, m = kp - 1;
    const double tol = 0x1.0p-53 * (double)c, tol2 = tol * tol;
    int sweep = 0;
    for (; sweep < 40 && r >= 2; sweep++) {
        for (int j = g; j < r; j += TQ_NT / 16) {
            const double x0 = X[j * SV_LD + gl], x1 = X[j * SV_LD + gl + 16];
            const double n = row16_sum(x0 * x0 + x1 * x1);
            if (gl == 0) nrm[j] = n;
        }
        if (tid < 4) flag[tid] = 0;
        __syncthreads();
        bool open = false, big = false;
        int a = g == 0 ? m : g, b = g == 0 ? 0 : m - g;  // the pair of round 0
        if (b == m) b = 0;
        for (int t = 0; t < m; t++) {
            if (g < P && a < r && b < r) {
                double *ca = X + a * SV_LD + gl, *cb = X + b * SV_LD + gl;
                const double x0 = ca[0], x1 = ca[16], y0 = cb[0], y1 = cb[16];
                const double al = nrm[a], be = nrm[b];
                const double ga = row16_sum(x0 * y0 + x1 * y1);
                const double g2 = ga * ga, ab = al * be;
                if (g2 > tol2 * ab && al > 0.0 && be > 0.0) {
                    open = open || g2 > 4.0 * tol2 * ab;
                    big = big || g2 > 1e-16 * ab;
                    double cs, sn;
                    sv_rotation(al, be, ga, cs, sn);
                    ca[0] = cs * x0 - sn * y0;
                    ca[16] = cs * x1 - sn * y1;
                    cb[0] = sn * x0 + cs * y0;
                    cb[16] = sn * x1 + cs * y1;
                    if (gl == 0) {
                        const double e = sn * (sn * (be - al) - 2.0 * cs * ga);
                        nrm[a] = fmax(al + e, 0.0);
                        nrm[b] = fmax(be - e, 0.0);
                    }
                }
            }
            // the next round's pair: player m stays, the others move on by one
            if (g != 0 && ++a == m) a = 0;
            if (++b == m) b = 0;
            __syncthreads();
        }
        if (open) flag[0] = 1;
        if (big) flag[1] = 1;
        __syncthreads();
        if (!flag[0]) break;
        if (!flag[1]) {
            // every pair, sixteen columns b a step, one lane a pair
            for (int e = tid; e < r * r; e += TQ_NT) {
                const int i = e / r, j = e - i * r;
                if (i >= j) continue;
                double p = 0.0, n0 = 0.0, n1 = 0.0;
#pragma unroll 8
                for (int q = 0; q < 32; q++) {
                    const double x = X[i * SV_LD + q], y = X[j * SV_LD + q];
                    p += x * y;
                    n0 += x * x;
                    n1 += y * y;
                }
                if (p * p > 4.0 * tol2 * (n0 * n1)) flag[2] = 1;
            }
            __syncthreads();
            if (!flag[2]) break;
        }
        __syncthreads();
    }
    __syncthreads();
    return sweep < 40 ? sweep + 1 : 40;
}

// Column-pivoted QR of L (c x c, L(x, q) = R[q * SV_LD + x]) by one wave: lane
// (q, half) holds rows 16 half + s of column q.  Row i of the factor goes to
// column i of X.  vc: 36 doubles of LDS.  Returns the rows formed.
__device__ int sv_pivoted_qr(const double *R, int c, double *X, double *vc) {
    const int lane = threadIdx.x & 63, q = lane & 31, half = lane >> 5;
    double a[16];  // finished rows are zero
#pragma unroll
    for (int s = 0; s < 16; s++) {
        const int x = 16 * half + s;
        a[s] = (q < c && x < c) ? R[q * SV_LD + x] : 0.0;
    }
    bool done = q >= c, stop = false;
    double first = 0.0;
    int r = 0;
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int s0 = 0; s0 < 16; s0++) {
            const int j = 16 * h + s0;
            if (stop || j >= c) continue;  // uniform
            double u = 0.0, w = 0.0;
#pragma unroll
            for (int s = 0; s < 16; s += 2) {
                u += a[s] * a[s];
                w += a[s + 1] * a[s + 1];
            }
            double n = xor32_sum(u + w);
            if (done) n = -1.0;
            double best = n;
            best = fmax(best, dppd<0xB1>(best));
            best = fmax(best, dppd<0x4E>(best));
            best = fmax(best, dppd<0x141>(best));
            best = fmax(best, dppd<0x140>(best));
            best = fmax(best, xor16_other(best));
            if (j == 0) first = best;
            // stop where nothing above u |R_11| is left (also: all zero, NaN)
            if (!(best > first * 0x1.0p-106) || !(best > 0x1.0p-1000)) {
                stop = true;
                continue;
            }
            const int p = (__ffsll((unsigned long long)__ballot(n == best)) - 1) & 31;
            if (q == p) {
#pragma unroll
                for (int s = 0; s < 16; s++) vc[half * 18 + s] = a[s];
            }
            __asm__ __volatile__("" ::: "memory");  // a wave's LDS accesses complete in order
            double v[16];
#pragma unroll
            for (int s = 0; s < 16; s++) v[s] = vc[half * 18 + s];
            const double alpha = vc[h * 18 + s0];
            const double nrm = sqrt_nr(best), beta = alpha > 0.0 ? -nrm : nrm, v0 = alpha - beta;
            const double tau = rcp_nr(best + fabs(alpha) * nrm);
            const double ajj = a[s0];
            u = 0.0;
            w = 0.0;
#pragma unroll
            for (int s = 0; s < 16; s += 2) {
                u += v[s] * a[s];
                w += v[s + 1] * a[s + 1];
            }
            u += w;
            if (half == h) u -= beta * ajj;  // v has v0 = alpha - beta in row j
            const double f = tau * xor32_sum(u);
#pragma unroll
            for (int s = 0; s < 16; s++) a[s] -= f * v[s];
            if (half == h) {
                X[j * SV_LD + q] = q == p ? beta : done ? 0.0 : ajj - f * v0;
                a[s0] = 0.0;
            }
            if (q == p) {
                done = true;
#pragma unroll
                for (int s = 0; s < 16; s++) a[s] = 0.0;
            }
            r = j + 1;
        }
    }
    return r;
}

struct SvdOut {
    double *sig;   // 32 singular values, descending, zeros beyond
    int *info;     // numerical rank, rank kept, sweeps, columns factored
    double *X;     // right singular vectors, c x rho (ld TQ_C)
    double *US;    // U Sigma of L = R^T V: c x rho, row i at i * TQ_C
    int *rho;      // the rank kept
    double delta;  // tail threshold
    int cap;
};

// R: LDS, c x c, row-major stride SV_LD, scaled by 2^-ex to entries of order
// one.  lds: SV_LDS doubles.
constexpr int SV_LDS = 2 * 32 * SV_LD + 32 + 32 + 16 + 8 + 40 + 32;
__device__ void svd_root(const double *R, int c, int ex, double *lds, const SvdOut &o) {
    double *X = lds, *U = X + 32 * SV_LD, *sv = U + 32 * SV_LD, *sorted = sv + 32;
    int *pos = (int *)(sorted + 32), *sint = pos + 32;
    double *vc = sorted + 32 + 16 + 8, *cn = vc + 40;
    const int tid = threadIdx.x;
    for (int e = tid; e < 32 * SV_LD; e += TQ_NT) X[e] = 0.0;
    __syncthreads();
    if (tid < 64) {
        const int rr = sv_pivoted_qr(R, c, X, vc);
        if (tid == 0) sint[1] = rr;
    }
    __syncthreads();
    const int r = sint[1];
    const int sw = sv_sweeps(X, r, c, cn, sint + 2);
    // singular values, descending order by rank counting (ties by index)
    if (tid < 32) {
        double s = 0.0;
        if (tid < r)
            for (int i = 0; i < 32; i++) s += X[tid * SV_LD + i] * X[tid * SV_LD + i];
        sv[tid] = sqrt(s);
    }
    __syncthreads();
    if (tid < 32) {
        int ps = 0;
        for (int i = 0; i < 32; i++) ps += (sv[i] > sv[tid]) || (sv[i] == sv[tid] && i < tid);
        pos[tid] = ps;
        sorted[ps] = sv[tid];
    }
    __syncthreads();
    if (tid == 0) {
        const double s0 = sorted[0], thr = sqrt((double)c) * 0x1.0p-53 * s0;
        const double dl = ldexp(o.delta, -ex);
        int nk = 0;
        for (int j = 0; j < 32; j++) nk += (sorted[j] > thr) && (s0 > 0.0);
        int rho = nk;
        double tail = 0.0;
        for (int j = nk - 1; j >= 0; j--) {
            tail += sorted[j] * sorted[j];
            if (o.delta > 0.0 && sqrt(tail) < dl) rho = j;
            else break;
        }
        if (rho > o.cap) rho = o.cap;
        if (rho < 1) rho = 1;
        sint[1] = rho;
        o.info[0] = nk;
        o.info[1] = rho;
        o.info[2] = sw;
        o.info[3] = r;
        *o.rho = rho;
    }
    __syncthreads();
    const int rho = sint[1];
    if (tid < 32) o.sig[tid] = ldexp(sorted[tid], ex);
    for (int e = tid; e < 32 * 32; e += TQ_NT) {
        const int i = e & 31, j = e >> 5, ps = pos[j];
        if (ps < rho) {
            const double s = sv[j];
            // an all-zero bond keeps one (arbitrary) unit direction
            const double u = s > 0.0 ? X[j * SV_LD + i] / s : (i == ps && ps == 0 ? 1.0 : 0.0);
            U[i * SV_LD + ps] = u;
            if (i < c) o.X[i + ps * TQ_C] = u;
        }
    }
    __syncthreads();
    for (int e = tid; e < 32 * 32; e += TQ_NT) {
        const int p = e & 31, x = e >> 5;
        if (p < rho && x < c) {
            double s = 0.0;
            for (int i = 0; i <= x; i++) s += R[i * SV_LD + x] * U[i * SV_LD + p];
            o.US[x * TQ_C + p] = ldexp(s, ex);
        }
    }
    __syncthreads();
}

// The root of a right-to-left bond: its block's factorisation, the SVD, and the
// application of its reflectors to the right singular vectors (ap.X = svd.X).
// A bond of one block writes the new core itself.
template <int NC, int RP>
__global__ __launch_bounds__(TQ_NT) void k_qr_svd(QrArgs g, SvdOut o, ApplyArgs ap) {
    extern __shared__ double lds[];
    __shared__ double red4[4];
    __shared__ double Rm[32 * SV_LD];
    typedef Lay<NC, RP> L;
    const int tid = threadIdx.x, li = tid & 15, part = tid >> 4;
    const int c = g.c;
    const long rows = g.drho ? g.rows * (long)*g.drho : g.rows;
    const int nr = (int)(rows < L::ROWS ? rows : L::ROWS);
    double a[NC][RP];
#pragma unroll
    for (int k = 0; k < NC; k++)
#pragma unroll
        for (int s = 0; s < RP; s++) {
            const int r = part + 16 * s, col = li + 16 * k;
            a[k][s] = (col < c && r < nr) ? g.A[r * g.rs + col * g.cs] : 0.0;
        }
    int ex = 0;
    {
        // the SVD works on entries of order one
        const double m = block_absmax<NC, RP>(a, red4);
        if (m > 0.0 && m < INFINITY) ex = ilogb(m);
    }
#pragma unroll
    for (int k = 0; k < NC; k++)
#pragma unroll
        for (int s = 0; s < RP; s++) a[k][s] = ldexp(a[k][s], -ex);
    double *Mm = lds + L::QR_LDS, *tau = Mm + L::MAT, *vt = tau + L::RW;
    for (int e = tid; e < 32 * SV_LD; e += TQ_NT) Rm[e] = 0.0;
    qr_block<NC, RP>(a, c, lds, Rm, Mm, tau);
    form_f<NC, RP>(a, c, Mm, tau, vt, g.F);
#pragma unroll
    for (int k = 0; k < NC; k++)
#pragma unroll
        for (int s = 0; s < RP; s++) {
            const int r = part + 16 * s, col = li + 16 * k;
            if (col < c && r < nr) g.A[r * g.rs + col * g.cs] = a[k][s];
        }
    __syncthreads();
    svd_root(Rm, c, ex, lds, o);
    __threadfence_block();  // V, F, X and the rank were written by this workgroup
    __syncthreads();
    apply_block<false>(ap, 0, lds);
}

template <int NC, int RP>
constexpr size_t qr_lds(bool colmajor) {
    typedef Lay<NC, RP> L;
    size_t d = L::QR_LDS + 3 * L::MAT + L::RW;
    const size_t tile = 16 * (L::ROWS + 1), app = 3 * TQ_C * TQ_LD;
    if (colmajor && tile > d) d = tile;
    if (SV_LDS > d) d = SV_LDS;
    if (app > d) d = app;
    return d * sizeof(double);
}

template <typename K>
void lds_attr(K kern, size_t bytes) {
    HIPCHECK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)bytes));
}

void allow_lds() {
    static bool done = false;
    if (done) return;
#define TQ_ATTR(NC, RP)                                             \
    lds_attr(k_qr_block<NC, RP, true>, qr_lds<NC, RP>(true));       \
    lds_attr(k_qr_block<NC, RP, false>, qr_lds<NC, RP>(false));     \
    lds_attr(k_qr_svd<NC, RP>, qr_lds<NC, RP>(false))
    TQ_ATTR(1, 8);
    TQ_ATTR(1, 16);
    TQ_ATTR(1, 32);
    TQ_ATTR(2, 8);
    TQ_ATTR(2, 16);
    TQ_ATTR(2, 32);
#undef TQ_ATTR
    done = true;
}

// Rows of a block by columns and rows of the matrix: the smallest layout that
// takes them all, 512 rows for larger ones.
int block_rows(int c, long rows) {
    (void)c;
    return rows <= 128 ? 128 : rows <= 256 ? 256 : 512;
}

#define TQ_DISPATCH(c, br, M)             \
    do {                                  \
        if ((c) <= 16) {                  \
            if ((br) == 128) M(1, 8);     \
            else if ((br) == 256) M(1, 16); \
            else M(1, 32);                \
        } else {                          \
            if ((br) == 128) M(2, 8);     \
            else if ((br) == 256) M(2, 16); \
            else M(2, 32);                \
        }                                 \
    } while (0)

void launch_qr(const QrArgs &g, int nblk, int br, bool colmajor) {
    const double fl = 4.0 * (double)br * nblk * g.c * g.c;
#define TQ_QR(NC, RP)                                                                          \
    do {                                                                                       \
        if (colmajor)                                                                          \
            PTT_LAUNCH_FB("tsqr_block", fl, 0.0, (k_qr_block<NC, RP, true>), dim3(nblk),        \
                          dim3(TQ_NT), (qr_lds<NC, RP>(true)), g);                              \
        else                                                                                   \
            PTT_LAUNCH_FB("tsqr_block", fl, 0.0, (k_qr_block<NC, RP, false>), dim3(nblk),       \
                          dim3(TQ_NT), (qr_lds<NC, RP>(false)), g);                             \
    } while (0)
    TQ_DISPATCH(g.c, br, TQ_QR);
#undef TQ_QR
}

}  // namespace

extern "C" {

// Levels of the tree over `rows` rows of c columns.
int ptt_hip_tsqr_plan(int c, long rows, ptt_tsqr_plan *pl) {
    pl->c = c;
    pl->rows = rows;
    pl->levels = 0;
    pl->fsize = pl->ssize = 0;
    long r = rows;
    for (;;) {
        if (pl->levels == PTT_TSQR_LEVELS) return -1;
        const int br = block_rows(c, r);
        const long nb = (r + br - 1) / br;
        const int l = pl->levels++;
        pl->brows[l] = br;
        pl->nblk[l] = (int)nb;
        pl->lrows[l] = r;
        pl->foff[l] = pl->fsize;
        pl->soff[l] = pl->ssize;  // the stack this level factors (level 0: the matrix)
        pl->fsize += nb * TQ_C * TQ_C;
        if (l > 0) pl->ssize += r * c;
        if (nb == 1) break;
        r = nb * c;
    }
    return 0;
}

// The matrix behind level l's blocks.
static void level_matrix(const ptt_tsqr_plan *pl, int l, double *A, long rs, long cs, double *S,
                         double **M, long *mr, long *mc) {
    if (l == 0) {
        *M = A;
        *mr = rs;
        *mc = cs;
    } else {
        *M = S + pl->soff[l];
        *mr = pl->c;
        *mc = 1;
    }
}

void ptt_hip_tsqr_factor(const ptt_tsqr_plan *pl, double *A, long rs, long cs, const int *drho,
                         long rows_per_rank, double *F, double *S, double *R, int *escale) {
    ptt_hip_init();
    allow_lds();
    const int last = pl->levels - 1;
    for (int l = 0; l <= last; l++) {
        if (l == last && !R) break;  // the root belongs to ptt_hip_tsqr_svd
        QrArgs g;
        level_matrix(pl, l, A, rs, cs, S, &g.A, &g.rs, &g.cs);
        g.rows = (l == 0 && drho) ? rows_per_rank : pl->lrows[l];
        g.drho = l == 0 ? drho : nullptr;
        g.c = pl->c;
        g.F = F + pl->foff[l];
        g.root = l == last;
        g.R = l == last ? R : S + pl->soff[l + 1];
        g.escale = escale;
        launch_qr(g, pl->nblk[l], pl->brows[l], l == 0 && rs == 1);
    }
}

static ApplyArgs level_apply(const ptt_tsqr_plan *pl, int l, const double *A, long rs, long cs,
                             const int *drho, long rows_per_rank, const double *F,
                             const double *S, const double *X, long xr, long xc, const int *p,
                             double *Y, long yr, long yc, double alpha) {
    ApplyArgs g;
    double *M;
    level_matrix(pl, l, (double *)A, rs, cs, (double *)S, &M, &g.rs, &g.cs);
    g.V = M;
    g.rows = (l == 0 && drho) ? rows_per_rank : pl->lrows[l];
    g.drho = l == 0 ? drho : nullptr;
    g.c = pl->c;
    g.brows = pl->brows[l];
    g.F = F ? F + pl->foff[l] : nullptr;
    g.X = X;
    g.xr = xr;
    g.xc = xc;
    g.p = p;
    g.Y = Y;
    g.yr = yr;
    g.yc = yc;
    g.alpha = alpha;
    g.plain = 0;
    return g;
}

// Work rows handed down the tree are row-major with stride TQ_C; two buffers
// of pl->lrows[1] * TQ_C doubles (none for a single level) alternate.
static const double *apply_upper(const ptt_tsqr_plan *pl, int from, const double *A, long rs,
                                 long cs, const double *F, const double *S, const double *X,
                                 long xr, long xc, const int *p, double *W) {
    // levels from .. 1; returns the rows that level 0 takes
    const long wsz = pl->levels > 1 ? pl->lrows[1] * TQ_C : 0;
    const double *x = X;
    for (int l = from; l >= 1; l--) {
        double *y = W + (l & 1) * wsz;
        const ApplyArgs g = level_apply(pl, l, A, rs, cs, nullptr, 0, F, S, x, xr, xc, p, y,
                                        TQ_C, 1, 1.0);
        PTT_LAUNCH("tsqr_apply", k_qr_apply, dim3(pl->nblk[l]), dim3(TQ_NT), 0, g, g, pl->nblk[l]);
        x = y;
        xr = TQ_C;
        xc = 1;
    }
    return x;
}

void ptt_hip_tsqr_svd(const ptt_tsqr_plan *pl, double *A, long rs, long cs, const int *drho,
                      long rows_per_rank, double *F, double *S, double delta, int cap,
                      double *sig, int *info, int *rho, double *X, double *US, double *W,
                      double *Y, double alpha) {
    ptt_hip_init();
    allow_lds();
    const int last = pl->levels - 1;
    QrArgs g;
    level_matrix(pl, last, A, rs, cs, S, &g.A, &g.rs, &g.cs);
    g.rows = (last == 0 && drho) ? rows_per_rank : pl->lrows[last];
    g.drho = last == 0 ? drho : nullptr;
    g.c = pl->c;
    g.F = F + pl->foff[last];
    g.root = 1;
    g.R = nullptr;
    g.escale = nullptr;
    SvdOut o;
    o.sig = sig;
    o.info = info;
    o.X = X;
    o.US = US;
    o.rho = rho;
    o.delta = delta;
    o.cap = cap;
    const long wsz = pl->levels > 1 ? pl->lrows[1] * TQ_C : 0;
    // a single level writes the new core (rho x w): element (t, p) at p + rho t
    ApplyArgs ap = level_apply(pl, last, A, rs, cs, drho, rows_per_rank, F, S, X, 1, TQ_C, rho,
                               last == 0 ? Y : W + (last & 1) * wsz, last == 0 ? 0 : TQ_C, 1,
                               last == 0 ? alpha : 1.0);
#define TQ_SVD(NC, RP)                                                                        \
    PTT_LAUNCH_FB("tsqr_svd", 4.0 * pl->brows[last] * g.c * g.c, 0.0, (k_qr_svd<NC, RP>), dim3(1), \
                  dim3(TQ_NT), (qr_lds<NC, RP>(false)), g, o, ap)
    TQ_DISPATCH(g.c, pl->brows[last], TQ_SVD);
#undef TQ_SVD
}

void ptt_hip_tsqr_finish(const ptt_tsqr_plan *pl0, const double *A0, const int *drho0,
                         long rows_per_rank0, const double *F0, const double *S0,
                         const int *rho0, double *W0, double *Y0, double alpha0,
                         const ptt_tsqr_plan *pl1, const double *A1, const double *F1,
                         const double *S1, const double *US1, const int *p1, double *W1,
                         double *Y1, double alpha1) {
    ptt_hip_init();
    allow_lds();
    ApplyArgs g[2];
    int nb[2] = {0, 0};
    if (pl0 && pl0->levels > 1) {
        // below the root, whose rows ptt_hip_tsqr_svd left in W0
        const int last = pl0->levels - 1;
        const long wsz = pl0->lrows[1] * TQ_C;
        const double *x = apply_upper(pl0, last - 1, A0, pl0->c, 1, F0, S0, W0 + (last & 1) * wsz,
                                      TQ_C, 1, rho0, W0);
        g[0] = level_apply(pl0, 0, A0, pl0->c, 1, drho0, rows_per_rank0, F0, S0, x, TQ_C, 1, rho0,
                           Y0, 0, 1, alpha0);
        nb[0] = pl0->nblk[0];
    }
    if (pl1 && !F1) {
        // an explicit Q: every block takes US1 itself
        g[1] = level_apply(pl1, 0, A1, 1, pl1->rows, nullptr, 0, nullptr, S1, US1, TQ_C, 1, p1, Y1,
                           1, pl1->rows, alpha1);
        g[1].plain = 1;
        nb[1] = pl1->nblk[0];
    } else if (pl1) {
        const double *x = apply_upper(pl1, pl1->levels - 1, A1, 1, pl1->rows, F1, S1, US1, TQ_C, 1,
                                      p1, W1);
        g[1] = level_apply(pl1, 0, A1, 1, pl1->rows, nullptr, 0, F1, S1, x, TQ_C, 1, p1, Y1, 1,
                           pl1->rows, alpha1);
        nb[1] = pl1->nblk[0];
    }
    if (nb[0] + nb[1] == 0) return;
    if (!nb[0]) g[0] = g[1];
    if (!nb[1]) g[1] = g[0];
    PTT_LAUNCH("tsqr_apply", k_qr_apply, dim3(nb[0] + nb[1]), dim3(TQ_NT), 0, g[0], g[1], nb[0]);
}

}  // extern "C"
