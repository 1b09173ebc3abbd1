// dot.hip -- one mode of the inner product of two trains, ranks up to 64 (gfx950).
//
//   a'(p, q) = s sum_{j, i, k} x(i, j, p) a(i, k) y(k, j, q)
//
// as a' = s sum_j X_j^T (a Y_j): both products of a mode index j stay in the
// registers of the waves that take it, so x and y are read once and the product
// a Y (as large as y) is neither written nor read.  Bound by the FP64 matrix
// cores (1.07 GFLOP a mode at n = 1024, ranks 64: 13.7 us at their peak, against
// 13 us for its 67 MB at 5.2 TB/s).
//
// Operands come straight from global memory into the MFMA layout: the order of k
// within a product is free, so lane group g of a wave takes rows 16 b + 4 g + v of
// a column for the four steps v of block b, 32 consecutive bytes (a column's 16
// rows are one 128-byte line).  The rows of a are permuted to match
// (i = 4 (m % 4) + m / 4), so that register v of the first product is the second
// operand of step v of the second one.  No LDS until the waves' sums are added.
// X_j is loaded beside the first product, Y_{j+1} beside the second.
// Measured (us a mode, with the sum over workgroups): n = 1024, ranks 64: 33 (two
// tiled products and a reduction over the splits of K, which this replaces: 60),
// 48: 19, 40: 24, 32: 11, 16: 7; n = 300, ranks 64: 22.  At 64 a mode index costs
// 6.1 us a CU against 5.0 at the 53 TFLOP/s that the matrix cores hold under such a
// load, and a mode some 6 us for a's operands and the sums.  Loading a product and a
// half ahead (35 us) and handing the indices out round robin (34) gave nothing.
#include "common.hpp"

using namespace ptt;

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
// two doubles at any multiple of 8 bytes
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));

constexpr int DOT_R = 64;  // ranks at most

// Rows r0 .. r0 + 3 of a column of `rows` rows; RAG: zero beyond them, else
// there are that many.  col: byte offset from base.  Nothing outside the column
// is read.
template <bool RAG>
__device__ __forceinline__ void load4(const double *__restrict__ base, unsigned col, int r0,
                                      int rows, double (&v)[4]) {
    const char *b = (const char *)base;
    if (RAG && rows == 1) {
        const double a = *(const double *)(b + col);
#pragma unroll
        for (int t = 0; t < 4; t++) v[t] = r0 + t == 0 ? a : 0.0;
        return;
    }
#pragma unroll
    for (int t = 0; t < 4; t += 2) {
        const int r = r0 + t;
        // a pair that straddles the end is read one row up
        const f64x2u a = *(const f64x2u *)(b + (col + 8u * (unsigned)(RAG ? min(r, rows - 2) : r)));
        v[t] = RAG ? (r + 1 < rows ? a.x : r < rows ? a.y : 0.0) : a.x;
        v[t + 1] = RAG ? (r + 1 < rows ? a.y : 0.0) : a.y;
    }
}

// How a workgroup takes mode indices: RB column blocks of y (a wave each) times HB
// halves of x's rows, JW indices at once.
template <int RB>
struct dot_geom {
    static constexpr int HB = RB % 2 ? 1 : 2, IB = RB / HB, WJ = RB * HB;
    static constexpr int JW = RB == 1 ? 8 : RB == 2 ? 2 : RB == 3 ? 2 : 1;
    static constexpr int NTH = 64 * WJ * JW;
};

// Ranks up to 16 RB.  Workgroup z takes mode indices z per .. (z + 1) per - 1 and
// writes its sum to out + z rx1 ry1, scaled by s.
template <int RB, bool RAG>
__global__ __launch_bounds__(dot_geom<RB>::NTH) void k_dot_mode(int n, int per, int rx0, int rx1,
                                                                int ry0, int ry1, const double *a,
                                                                const double *__restrict__ x,
                                                                const double *__restrict__ y,
                                                                double s, double *out) {
    using geom = dot_geom<RB>;
    constexpr int HB = geom::HB, IB = geom::IB, WJ = geom::WJ, JW = geom::JW, NTH = geom::NTH;
    constexpr int W = 16 * RB;
    __shared__ double lds[W * (W + 1)];
    const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int jw = wv / WJ, h = wv % WJ / RB, qb = wv % RB;
    const int j0 = blockIdx.x * per, j1 = min(n, j0 + per);

    // operand of step k, row block b: al[(b * 4 RB + k) * 64 + lane] (in registers it
    // would leave none for X_j)
    {
        constexpr int PER = (W * W + NTH - 1) / NTH;
        double av[PER];
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int e = threadIdx.x + u * NTH;
            const int l = e & 63, k = (e >> 6) % (4 * RB), b = (e >> 6) / (4 * RB);
            const int i = 16 * b + 4 * (l & 3) + ((l & 15) >> 2);
            const int c = 16 * (k >> 2) + 4 * (l >> 4) + (k & 3);
            av[u] = (i < rx0 && c < ry0) ? a[i + rx0 * c] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < PER; u++)
            if (threadIdx.x + u * NTH < W * W) lds[threadIdx.x + u * NTH] = av[u];
    }
    const double *al = lds + h * IB * 4 * RB * 64 + lane;
    __syncthreads();
    // columns beyond the ranks repeat the last one: their results are not used
    const unsigned yc = 8u * ry0 * n * (unsigned)min(16 * qb + li, ry1 - 1);
    unsigned xc[RB];
#pragma unroll
    for (int p = 0; p < RB; p++) xc[p] = 8u * rx0 * n * (unsigned)min(16 * p + li, rx1 - 1);

    f64x4 acc[RB];
#pragma unroll
    for (int p = 0; p < RB; p++) acc[p] = f64x4{0.0, 0.0, 0.0, 0.0};
    double yv[RB][4];
    auto load_y = [&](int j) {
#pragma unroll
        for (int b = 0; b < RB; b++)
            load4<RAG>(y + (long)ry0 * j, yc, 16 * b + 4 * lg, ry0, yv[b]);
    };
    if (j0 + jw < j1) load_y(j0 + jw);
    for (int j = j0 + jw; j < j1; j += JW) {
        __asm__ __volatile__("" ::: "memory");  // a's operands stay in LDS
        double xv[RB][IB][4];
#pragma unroll
        for (int p = 0; p < RB; p++)
#pragma unroll
            for (int b = 0; b < IB; b++)
                load4<RAG>(x + (long)rx0 * j, xc[p], 16 * (h * IB + b) + 4 * lg, rx0, xv[p][b]);
        __builtin_amdgcn_sched_barrier(0);  // issued here, not at their use
        f64x4 w[IB];
#pragma unroll
        for (int b = 0; b < IB; b++) w[b] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 4 * RB; k++)
#pragma unroll
            for (int b = 0; b < IB; b++)
                w[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(al[(b * 4 * RB + k) * 64],
                                                            yv[k >> 2][k & 3], w[b], 0, 0, 0);
        load_y(j + JW < j1 ? j + JW : j);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < IB; b++)
#pragma unroll
            for (int v = 0; v < 4; v++)
#pragma unroll
                for (int p = 0; p < RB; p++)
                    acc[p] = __builtin_amdgcn_mfma_f64_16x16x4f64(xv[p][b][v], w[b][v], acc[p], 0, 0,
                                                                  0);
    }
    __syncthreads();
    // acc[p][v]: row 16 p + lg + 4 v, column 16 qb + li
    for (int g = 0; g < HB * JW; g++) {
        if (jw * HB + h == g) {
#pragma unroll
            for (int p = 0; p < RB; p++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    double *t = &lds[16 * p + lg + 4 * v + (16 * qb + li) * (W + 1)];
                    *t = g == 0 ? acc[p][v] : *t + acc[p][v];
                }
        }
        __syncthreads();
    }
    double *o = out + (long)blockIdx.x * rx1 * ry1;
    for (int e = threadIdx.x; e < rx1 * ry1; e += NTH) {
        const int q = e / rx1, p = e - q * rx1;
        o[e] = s * lds[p + q * (W + 1)];
    }
}

// out[e] = sum over z of part[z * total + e]: 32 elements a workgroup, 32 parts a
// round, so a thread's loads are all in flight at once up to 256 parts.
__global__ __launch_bounds__(1024) void k_dot_sum(int total, int nz, const double *__restrict__ part,
                                                  double *__restrict__ out) {
    __shared__ double red[32][33];
    const int el = threadIdx.x & 31, zl = threadIdx.x >> 5;
    const int e = blockIdx.x * 32 + el;
    double s = 0.0;
    if (e < total) {
#pragma unroll 8
        for (int z = zl; z < nz; z += 32) s += part[(long)z * total + e];
    }
    red[zl][el] = s;
    __syncthreads();
    if (threadIdx.x < 32 && e < total) {
        double t = 0.0;
#pragma unroll
        for (int z = 0; z < 32; z++) t += red[z][el];
        out[e] = t;
    }
}

template <int RB>
void dot_mode(int n, int rx0, int rx1, int ry0, int ry1, const double *a, const double *x,
              const double *y, double s, double *out) {
    constexpr int JW = dot_geom<RB>::JW, NTH = dot_geom<RB>::NTH;
    // one workgroup a CU at most; a few indices a wave stay on one workgroup, which
    // needs no second launch
    const int cap = 256 * JW;
    int per = n <= 4 * JW ? n : (n + cap - 1) / cap * JW;
    const int nz = (n + per - 1) / per;
    const double fl = 2.0 * n * (double)rx0 * ry1 * (ry0 + rx1);
    const double by = 8.0 * n * ((double)rx0 * rx1 + (double)ry0 * ry1);
    double *part = out;
    if (nz > 1)
        part = (double *)ptt_hip_scratch(PTT_WS_GRAM, sizeof(double) * (size_t)nz * rx1 * ry1);
    // ranks of whole blocks need no masks
    if (rx0 == 16 * RB && ry0 == 16 * RB)
        PTT_LAUNCH_FB("dot_mode", fl, by, (k_dot_mode<RB, false>), dim3(nz), dim3(NTH), 0, n, per,
                      rx0, rx1, ry0, ry1, a, x, y, s, part);
    else
        PTT_LAUNCH_FB("dot_mode", fl, by, (k_dot_mode<RB, true>), dim3(nz), dim3(NTH), 0, n, per,
                      rx0, rx1, ry0, ry1, a, x, y, s, part);
    if (nz > 1)
        PTT_LAUNCH("dot_sum", k_dot_sum, dim3(cdiv((long)rx1 * ry1, 32)), dim3(1024), 0, rx1 * ry1,
                   nz, part, out);
}

}  // namespace

extern "C" {

int ptt_hip_dot_mode(int n, int rx0, int rx1, int ry0, int ry1, const double *a, const double *x,
                     const double *y, double s, double *out) {
    ptt_hip_init();
    int r = rx0;
    if (rx1 > r) r = rx1;
    if (ry0 > r) r = ry0;
    if (ry1 > r) r = ry1;
    // a core's byte offsets fit 32 bits
    if ((double)n * r * r * 8.0 >= 4.0e9) return 0;
    if (r > DOT_R || n < 1 || rx0 < 1 || rx1 < 1 || ry0 < 1 || ry1 < 1) return 0;
    if (r <= 16) dot_mode<1>(n, rx0, rx1, ry0, ry1, a, x, y, s, out);
    else if (r <= 32) dot_mode<2>(n, rx0, rx1, ry0, ry1, a, x, y, s, out);
    else if (r <= 48) dot_mode<3>(n, rx0, rx1, ry0, ry1, a, x, y, s, out);
    else dot_mode<4>(n, rx0, rx1, ry0, ry1, a, x, y, s, out);
    return 1;
}

}  // extern "C"
