// svdr.hip -- singular values and right singular vectors of a bond's factor
// L = R^T (R upper triangular, up to 128 columns; 192 from approximate vectors),
// gfx950.
//
// Two kernels, one workgroup each:
//   k_pivoted_qr   column-pivoted Householder QR of L, L = Q4 X^T, stopped where
//                  the remaining columns fall below u |R_11|: X is k x r with r
//                  the columns that carry information (a rank-deficient sum of
//                  100 columns leaves some 35);
//   k_right_jacobi (beyond 64 columns of content: the SVD over many workgroups)
//                  one-sided Jacobi on the columns of X: X = U S W^T, so U holds
//                  L's right singular vectors.  The transposed factor of a
//                  pivoted QR takes few sweeps (Drmac and Veselic, SIAM J. Matrix
//                  Anal. Appl. 29, 2008) and no vectors are accumulated: half
//                  the LDS traffic and rotations of an SVD of L with V.
// L's left factor is L U, one product on the matrix cores.  Where the caller has
// approximate left vectors of L (ptt_hip_svd_right_from), the rotations start from
// R times them and k_pivoted_qr is left out: 59 columns of flat spectrum 52 us
// against 400.
//
// What bounds them: the chain of reflectors (1.7 us each at 59 columns, 3.4 at
// 128) and of rotation rounds (a barrier, an LDS round trip, a lane reduction
// and about 45 dependent FP64 instructions each, 0.7 us).  Measured against the
// SVD of L with V that these replace (us): 59 columns of flat spectrum 436 (was
// 942 on one workgroup, 826 over many), graded 244 (453), a third of the columns
// carrying information 83; 100: 1556 flat (1681), 258 deficient (about 900).
// Beyond 128 columns the pivoted QR leaves the registers (9 us a reflector).
#include "common.hpp"

using namespace ptt;

namespace {

constexpr int SR_K = 128;
constexpr int SR_KMAX = 192;  // started from approximate vectors
constexpr int RJ_NT = 512;  // Jacobi

// Column q of L is row q of R.  Lane li of a 16-lane row holds columns li + 16
// kk, kk < NC, the row's part rows part + PARTS s.  Row j of the factor leaves
// the registers for column j of X (k x k in global memory, ld k) as it is
// finished; finished rows and columns are zero.  Column norms are formed anew at
// every step.  Sums over the waves go through one total per column (TWO: with
// many waves or columns, reading every wave's partials would be what bounds a
// step: 4.8 us at 128 columns).
template <int NC, int NTH>
__global__ __launch_bounds__(NTH) void k_pivoted_qr(int k, const double *__restrict__ R, long ldr,
                                                    double *__restrict__ X,
                                                    int *__restrict__ nform) {
    constexpr int W = 16 * NC, PARTS = NTH / 16, NW = NTH / 64;
    constexpr int RS = (W + PARTS - 1) / PARTS, VS = (RS + 1) / 2 * 2 + 2;
    constexpr bool TWO = NC > 4;
    __shared__ double red[2][NW][W], tot[2][W], vc[PARTS * VS], rowj[W], redw[NW];
    const int tid = threadIdx.x, li = tid & 15, part = tid >> 4, wv = tid >> 6, lane = tid & 63;
    double a[NC][RS];
#pragma unroll
    for (int kk = 0; kk < NC; kk++)
#pragma unroll
        for (int s = 0; s < RS; s++) {
            const int q = li + 16 * kk, x = part + PARTS * s;
            a[kk][s] = (q <= x && x < k) ? R[q + x * ldr] : 0.0;
        }
    // entries of order one (exact power of two): products of tiny bonds' entries
    // would underflow
    double m = 0.0;
#pragma unroll
    for (int kk = 0; kk < NC; kk++)
#pragma unroll
        for (int s = 0; s < RS; s++) m = fmax(m, fabs(a[kk][s]));
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    if (lane == 0) redw[wv] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; w++) m = fmax(m, redw[w]);
    const int ex = (m > 0.0 && m < INFINITY) ? ilogb(m) : 0;
#pragma unroll
    for (int kk = 0; kk < NC; kk++)
#pragma unroll
        for (int s = 0; s < RS; s++) a[kk][s] = ldexp(a[kk][s], -ex);
    unsigned done = 0;  // bit kk: column li + 16 kk pivoted (or none)
#pragma unroll
    for (int kk = 0; kk < NC; kk++)
        if (li + 16 * kk >= k) done |= 1u << kk;
    // this thread's columns' sums over the waves of the partials in red[b]
    auto sums = [&](int b, double(&t)[NC]) {
        if constexpr (TWO) {
            __syncthreads();
            if (tid < W) {
                double u = 0.0;
#pragma unroll
                for (int w = 0; w < NW; w++) u += red[b][w][tid];
                tot[b][tid] = u;
            }
            __syncthreads();
#pragma unroll
            for (int kk = 0; kk < NC; kk++) t[kk] = tot[b][li * NC + kk];
        } else {
            __syncthreads();
#pragma unroll
            for (int kk = 0; kk < NC; kk++) {
                t[kk] = 0.0;
#pragma unroll
                for (int w = 0; w < NW; w++) t[kk] += red[b][w][li * NC + kk];
            }
        }
    };
    double first = 0.0;
    int r = 0;
    for (int j = 0; j < k; j++) {
#pragma unroll
        for (int kk = 0; kk < NC; kk++) {
            double u = 0.0;
#pragma unroll
            for (int s = 0; s < RS; s++) u += a[kk][s] * a[kk][s];
            u = xor32_sum(xor16_sum(u));
            if (lane < 16) red[0][wv][li * NC + kk] = u;
        }
        double n[NC], best = -1.0;
        sums(0, n);
#pragma unroll
        for (int kk = 0; kk < NC; kk++) {
            if (done >> kk & 1) n[kk] = -1.0;
            best = fmax(best, n[kk]);
        }
        best = fmax(best, dppd<0xB1>(best));
        best = fmax(best, dppd<0x4E>(best));
        best = fmax(best, dppd<0x141>(best));
        best = fmax(best, dppd<0x140>(best));
        if (j == 0) first = best;
        // nothing above u |R_11| is left (also: all zero, NaN); uniform
        if (!(best > first * 0x1.0p-106) || !(best > 0x1.0p-1000)) break;
        int set = -1, p = 0;
#pragma unroll
        for (int kk = NC - 1; kk >= 0; kk--) {
            const unsigned long long hit = __ballot(n[kk] == best);
            if (hit) {
                set = kk;
                p = (__ffsll(hit) - 1) & 15;
            }
        }
        const bool jp = part == j % PARTS;
        const int js = j / PARTS;
        if (li == p) {
#pragma unroll
            for (int kk = 0; kk < NC; kk++)
                if (kk == set) {
#pragma unroll
                    for (int s = 0; s < RS; s++) vc[part * VS + s] = a[kk][s];
                }
        }
        if (jp) {
#pragma unroll
            for (int s = 0; s < RS; s++)
                if (s == js) {
#pragma unroll
                    for (int kk = 0; kk < NC; kk++) rowj[li * NC + kk] = a[kk][s];
                }
        }
        __syncthreads();
        double v[RS];
#pragma unroll
        for (int s = 0; s < RS; s++) v[s] = vc[part * VS + s];
        const double alpha = vc[(j % PARTS) * VS + js];
#pragma unroll
        for (int kk = 0; kk < NC; kk++) {
            double u = 0.0;
#pragma unroll
            for (int s = 0; s < RS; s++) u += v[s] * a[kk][s];
            u = xor32_sum(xor16_sum(u));
            if (lane < 16) red[1][wv][li * NC + kk] = u;
        }
        const double nrm = sqrt_nr(best), beta = alpha > 0.0 ? -nrm : nrm, v0 = alpha - beta;
        const double tau = rcp_nr(best + fabs(alpha) * nrm);
        double aj[NC], d[NC];
#pragma unroll
        for (int kk = 0; kk < NC; kk++) aj[kk] = rowj[li * NC + kk];
        sums(1, d);
#pragma unroll
        for (int kk = 0; kk < NC; kk++) {
            const double f = tau * (d[kk] - beta * aj[kk]);  // v has v0 = alpha - beta in row j
            const bool piv = kk == set && li == p;
#pragma unroll
            for (int s = 0; s < RS; s++) a[kk][s] = piv ? 0.0 : a[kk][s] - f * v[s];
            if (jp) {
                const int q = li + 16 * kk;
                if (q < k) X[q + (long)j * k] = piv ? beta : (done >> kk & 1) ? 0.0 : aj[kk] - f * v0;
#pragma unroll
                for (int s = 0; s < RS; s++)
                    if (s == js) a[kk][s] = 0.0;
            }
            if (piv) done |= 1u << kk;
        }
        r = j + 1;
    }
    if (tid == 0) {
        nform[0] = r;
        nform[1] = ex;
    }
}

__device__ __forceinline__ void rotation(double al, double be, double ga, double &c, double &s) {
    // tangent 2 ga / (d + sign(d) hypot(d, 2 ga)) from hardware reciprocals (it
    // only steers convergence), c refined so that c^2 + s^2 = 1 to working
    // accuracy; the columns are of order one down to u
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

template <int G>
__device__ __forceinline__ double group_sum(double x) {
    x = quad_sum(x);
    if constexpr (G >= 8) x += dppd<0x141>(x);
    if constexpr (G >= 16) x += dppd<0x140>(x);
    return x;
}

// Sweeps over the r columns (G RR rows, zeros beyond the true ones, LDS stride
// ld) of X, G lanes a pair.  nrm carries the squared norms through a sweep (al +
// e, be - e), so a round reduces one product; flag: 4 ints.  A sweep whose
// largest cosine is below 1e-8 is followed by a test of every pair instead of
// another sweep.  Pairs are rotated down to a cosine of 4 u although k u ends the
// sweeps: from nearly orthogonal columns no later sweep would square what is left
// (the cores of a rounding at n = 301, 59 columns were 2.1e-12 from LAPACK's, and are
// 1.2e-12).
template <int G, int RR>
__device__ int right_sweeps(double *X, int ld, int r, int k, double *nrm, int *flag) {
    constexpr int NG = RJ_NT / G;
    const int tid = threadIdx.x, g = tid / G, gl = tid % G;
    const int kp = r + (r & 1), P = kp / 2, m = kp - 1;
    const double tol = 0x1.0p-53 * (double)k, tol2 = tol * tol;
    const double rot2 = 0x1.0p-102;  // (4 u)^2
    int sweep = 0;
    for (; sweep < 40 && r >= 2; sweep++) {
        for (int j = g; j < r; j += NG) {
            double n = 0.0;
#pragma unroll
            for (int q = 0; q < RR; q++) n += X[j * ld + gl + G * q] * X[j * ld + gl + G * q];
            n = group_sum<G>(n);
            if (gl == 0) nrm[j] = n;
        }
        if (tid < 4) flag[tid] = 0;
        __syncthreads();
        bool open = false, big = false;
        int a = g == 0 ? m : g, b = g == 0 ? 0 : m - g;  // the pair of round 0
        for (int t = 0; t < m; t++) {
            if (g < P && a < r && b < r) {
                double *ca = X + a * ld + gl, *cb = X + b * ld + gl;
                double x[RR], y[RR];
#pragma unroll
                for (int q = 0; q < RR; q++) {
                    x[q] = ca[G * q];
                    y[q] = cb[G * q];
                }
                const double al = nrm[a], be = nrm[b];
                double g0 = 0.0, g1 = 0.0;
#pragma unroll
                for (int q = 0; q < RR; q += 2) {
                    g0 += x[q] * y[q];
                    if (q + 1 < RR) g1 += x[q + 1] * y[q + 1];
                }
                const double ga = group_sum<G>(g0 + g1);
                const double g2 = ga * ga, ab = al * be;
                if (g2 > rot2 * ab && al > 0.0 && be > 0.0) {
                    open = open || g2 > 4.0 * tol2 * ab;
                    big = big || g2 > 1e-16 * ab;
                    double cs, sn;
                    rotation(al, be, ga, cs, sn);
#pragma unroll
                    for (int q = 0; q < RR; q++) {
                        ca[G * q] = cs * x[q] - sn * y[q];
                        cb[G * q] = sn * x[q] + cs * y[q];
                    }
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
            for (int j = g; j < r; j += NG) {
                double n = 0.0;
#pragma unroll
                for (int q = 0; q < RR; q++) n += X[j * ld + gl + G * q] * X[j * ld + gl + G * q];
                n = group_sum<G>(n);
                if (gl == 0) nrm[j] = n;
            }
            __syncthreads();
            for (int e = tid; e < r * r; e += RJ_NT) {
                const int i = e / r, j = e - i * r;
                if (i >= j) continue;
                double p0 = 0.0, p1 = 0.0;
#pragma unroll 8
                for (int q = 0; q < G * RR; q += 2) {
                    p0 += X[i * ld + q] * X[j * ld + q];
                    p1 += X[i * ld + q + 1] * X[j * ld + q + 1];
                }
                const double p = p0 + p1;
                if (p * p > 4.0 * tol2 * (nrm[i] * nrm[j])) flag[2] = 1;
            }
            __syncthreads();
            if (!flag[2]) break;
        }
        __syncthreads();
    }
    __syncthreads();
    return sweep < 40 ? sweep + 1 : 40;
}

// X (k x k, k <= 64) to entries of order one by an exact power of two; all of its
// columns count.  One workgroup.
__global__ __launch_bounds__(256) void k_right_start(int k, double *__restrict__ X,
                                                     int *__restrict__ nform) {
    __shared__ double red[4];
    double x[16], m = 0.0;
#pragma unroll
    for (int t = 0; t < 16; t++) {
        const int e = threadIdx.x + 256 * t;
        x[t] = e < k * k ? X[e] : 0.0;
        m = fmax(m, fabs(x[t]));
    }
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
    const int ex = (m > 0.0 && m < INFINITY) ? ilogb(m) : 0;
#pragma unroll
    for (int t = 0; t < 16; t++) {
        const int e = threadIdx.x + 256 * t;
        if (e < k * k) X[e] = ldexp(x[t], -ex);
    }
    if (threadIdx.x == 0) {
        nform[0] = k;
        nform[1] = ex;
    }
}

// r <= 64 columns; KR: rows of a column in LDS (k rounded up to 64 or 128).
template <int KR>
__global__ __launch_bounds__(RJ_NT) void k_right_jacobi(int k, const double *__restrict__ Xg,
                                                        const int *__restrict__ nform,
                                                        double *__restrict__ sig,
                                                        double *__restrict__ V, long ldv,
                                                        double delta, int cap,
                                                        int *__restrict__ iout) {
    extern __shared__ double lds[];
    constexpr int ld = KR + 1;
    __shared__ double nrm[SR_K], sv[SR_K], sorted[SR_K];
    __shared__ int pos[SR_K], flag[4], s_nk;
    const int tid = threadIdx.x, r = nform[0], ex = nform[1];
    for (int e = tid; e < r * KR; e += RJ_NT) {
        const int j = e / KR, i = e - j * KR;
        lds[j * ld + i] = i < k ? Xg[i + (long)j * k] : 0.0;
    }
    if (tid == 0) s_nk = 0;
    __syncthreads();
    const int sw = right_sweeps<16, KR / 16>(lds, ld, r, k, nrm, flag);
    for (int j = tid; j < SR_K; j += RJ_NT) {
        double s0 = 0.0, s1 = 0.0;
        if (j < r)
#pragma unroll 8
            for (int i = 0; i < KR; i += 2) {
                s0 += lds[j * ld + i] * lds[j * ld + i];
                s1 += lds[j * ld + i + 1] * lds[j * ld + i + 1];
            }
        sv[j] = sqrt(s0 + s1);
    }
    __syncthreads();
    // descending order by rank counting (ties by index)
    for (int j = tid; j < SR_K; j += RJ_NT) {
        const double s = sv[j];
        int p = 0;
#pragma unroll 8
        for (int i = 0; i < SR_K; i++) p += (sv[i] > s) || (sv[i] == s && i < j);
        pos[j] = p;
        sorted[p] = s;
    }
    __syncthreads();
    const double s0 = sorted[0], thr = sqrt((double)k) * 0x1.0p-53 * s0;
    if (tid < SR_K && s0 > 0.0 && sorted[tid] > thr) atomicAdd(&s_nk, 1);
    __syncthreads();
    if (tid == 0) {
        const int nk = s_nk;
        const double dl = ldexp(delta, -ex);
        int rho = nk;
        double tail = 0.0;
        for (int j = nk - 1; j >= 0; j--) {
            tail += sorted[j] * sorted[j];
            if (delta > 0.0 && sqrt(tail) < dl) rho = j;
            else break;
        }
        if (rho > k) rho = k;
        if (rho > cap) rho = cap;
        if (rho < 1) rho = 1;
        iout[0] = nk;
        iout[1] = rho;
        iout[2] = sw;
    }
    for (int j = tid; j < k; j += RJ_NT) sig[j] = ldexp(sorted[j], ex);
    for (int e = tid; e < k * k; e += RJ_NT) {
        const int j = e / k, i = e - j * k, p = pos[j];
        const double s = sv[j];
        double u = 0.0;
        if (s > 0.0)
            u = lds[j * ld + i] / s;
        else if (r == 0 && p == 0 && i == 0)
            u = 1.0;  // an all-zero bond keeps one (arbitrary) unit direction
        V[i + p * ldv] = u;
    }
}

// k_right_jacobi on the nform[0] <= 64 columns of X.
void right_jacobi(int k, const double *X, const int *nform, double *sig, double *V, long ldv,
                  double delta, int cap, int *iout) {
    static bool attr = false;
    if (!attr) {
        auto set = [](const void *f, int rows) {
            HIPCHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                         64 * (rows + 1) * (int)sizeof(double)));
        };
        set((const void *)k_right_jacobi<64>, 64);
        set((const void *)k_right_jacobi<128>, 128);
        attr = true;
    }
    const double jf = 12.0 * k * (double)k * k, jb = 16.0 * k * (double)k;
#define PTT_RJ(KR)                                                                          \
    PTT_LAUNCH_FB("svd_right_jacobi", jf, jb, k_right_jacobi<KR>, dim3(1), dim3(RJ_NT),        \
                  64 * (KR + 1) * sizeof(double), k, X, nform, sig, V, ldv, delta, cap, iout)
    if (k <= 64) PTT_RJ(64);
    else PTT_RJ(128);
#undef PTT_RJ
}

}  // namespace

extern "C" {

// Beyond 64 columns of content the rotations go over many workgroups
// (ptt_hip_svd_jacobi): one CU's LDS then bounds a round (100 columns of flat
// spectrum: 1520 us here, 1680 there with V, some 1200 without).
void ptt_hip_svd_right(int k, const double *R, long ldr, double *X, double *sig, double *V,
                      long ldv, double delta, int cap, int *iout) {
    ptt_hip_init();
    if (k < 1 || k > SR_K) {
        fprintf(stderr, "ptt_hip_svd_right: k = %d out of range\n", k);
        exit(1);
    }
    int *nform = iout + 3;
    const double fl = 4.0 / 3.0 * k * (double)k * k;
#define PTT_PQ(NC, NTH)                                                                     \
    PTT_LAUNCH_FB("svd_pivoted_qr", fl, 16.0 * k * (double)k, (k_pivoted_qr<NC, NTH>), dim3(1), \
                  dim3(NTH), 0, k, R, ldr, X, nform)
    if (k <= 32) PTT_PQ(2, 256);
    else if (k <= 48) PTT_PQ(3, 256);
    else if (k <= 64) PTT_PQ(4, 256);
    else if (k <= 96) PTT_PQ(6, 512);
    else PTT_PQ(8, 512);
#undef PTT_PQ
    if (k > 64) {
        int h[2];
        ptt_hip_d2h(h, nform, sizeof h);
        if (h[0] > 64) {
            // the vectors beyond the columns formed belong to zero values
            ptt_hip_zero(V, sizeof(double) * (size_t)ldv * k);
            ptt_hip_zero(sig, sizeof(double) * (size_t)k);
            ptt_hip_svd_jacobi(k, h[0], X, k, sig, V, ldv, nullptr, 0, h[1] * 0.6931471805599453,
                               delta, cap, iout);
            if (h[1] != 0) ptt_hip_scale(sig, h[0], ldexp(1.0, h[1]));
            return;
        }
    }
    right_jacobi(k, X, nform, sig, V, ldv, delta, cap, iout);
}

// The rotations start from U, orthogonal up to rounding, whose columns approximate
// L's left singular vectors: the columns of X = R U are then nearly orthogonal
// already (R U = V Sigma for the exact ones), two or three sweeps instead of six to
// ten, and no pivoted QR.
void ptt_hip_svd_right_from(int k, const double *R, long ldr, const double *U, long ldu, double *X,
                            double *sig, double *V, long ldv, double delta, int cap, int *iout) {
    ptt_hip_init();
    if (k < 1 || k > SR_KMAX) {
        fprintf(stderr, "ptt_hip_svd_right_from: k = %d out of range\n", k);
        exit(1);
    }
    ptt_hip_dgemm('N', 'N', k, k, k, 1.0, R, ldr, U, ldu, 0.0, X, k);
    if (k > 64) {
        ptt_hip_svd_jacobi(k, k, X, k, sig, V, ldv, nullptr, 0, 0.0, delta, cap, iout);
        return;
    }
    PTT_LAUNCH("svd_right_start", k_right_start, dim3(1), dim3(256), 0, k, X, iout + 3);
    right_jacobi(k, X, iout + 3, sig, V, ldv, delta, cap, iout);
}

}  // extern "C"
