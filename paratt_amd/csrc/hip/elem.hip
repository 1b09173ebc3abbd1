// elem.hip -- streaming (HBM-bound) kernels on TT cores for gfx950.
//
// Core k is column-major r0 x n x r1; element (a, j, b) at a + r0*(j + n*b).
// Every kernel is output-stationary with the fastest-varying rank index a
// mapped to consecutive lanes, so loads and stores coalesce.  The stencil,
// flux and diagonal kernels compile with FP contraction off so each output
// is rounded exactly as the reference's scalar C loops round it.
#include "common.hpp"

using namespace ptt;

namespace {

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

__global__ void k_gauss_fill(double *dst, long count, uint64_t h, double scale) {
    long npair = (count + 1) / 2;
    for (long p = blockIdx.x * (long)blockDim.x + threadIdx.x; p < npair;
         p += (long)gridDim.x * blockDim.x) {
        uint64_t a = mix64(h + 2 * (uint64_t)p), b = mix64(h + 2 * (uint64_t)p + 1);
        double u1 = ((double)(a >> 11) + 0.5) * 0x1.0p-53;
        double u2 = (double)(b >> 11) * 0x1.0p-53;
        double rad = sqrt(-2.0 * log(u1));
        double th = 6.283185307179586476925286766559 * u2;
        double s, c;
        sincos(th, &s, &c);
        dst[2 * p] = rad * c * scale;
        if (2 * p + 1 < count) dst[2 * p + 1] = rad * s * scale;
    }
}

__global__ void k_scale(double *p, long count, double alpha) {
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < count;
         e += (long)gridDim.x * blockDim.x)
        p[e] *= alpha;
}

__global__ void k_zero(double *p, long count) {
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < count;
         e += (long)gridDim.x * blockDim.x)
        p[e] = 0.0;
}

// Division of 32-bit indices by a divisor fixed for the launch: the
// round-up multiply-high method (Granlund and Montgomery, PLDI 1994, Fig.
// 4.1): with l = ceil(log2 d) and m = floor(2^32 (2^l - d) / d) + 1,
// n / d = (mulhi(n, m) + n) >> l for every 32-bit n (the sum taken in 64
// bits).  The streaming kernels below split a core's element index into
// (row of the column, column) by their 2D grid and the row into (rank
// index, mode index) this way, with no 64-bit division per element.
struct FastDiv {
    unsigned m;
    unsigned l;
};

FastDiv make_fastdiv(unsigned d) {
    unsigned l = 0;
    while (l < 32 && (1ull << l) < d) l++;
    const unsigned long long m = (((1ull << l) - d) << 32) / d + 1;
    return FastDiv{(unsigned)m, l};
}

__device__ __forceinline__ unsigned fdiv(unsigned n, FastDiv f) {
    const unsigned t = __umulhi(n, f.m);
    return (unsigned)(((unsigned long long)t + n) >> f.l);
}

// Grid of a core-shaped launch: y over the columns (the right rank), x over
// the rows r0 * n of a column; both grid-stride.
dim3 grid_core(long rows, long cols) {
    const unsigned gy = (unsigned)(cols < 65535 ? cols : 65535);
    long gx = (rows + 255) / 256;
    long cap = (256L * 16 + gy - 1) / gy;  // about 4096 workgroups in all
    if (gx > cap) gx = cap;
    if (gx < 1) gx = 1;
    return dim3((unsigned)gx, gy < 1 ? 1 : gy);
}

// VW consecutive doubles moved as one 16-byte access (VW = 2).
template <int VW>
struct Vd {
    double v[VW];
};

template <int VW>
__device__ __forceinline__ Vd<VW> ld_vd(const double *p) {
    Vd<VW> r;
    if constexpr (VW == 2) {
        const double2 t = *reinterpret_cast<const double2 *>(p);
        r.v[0] = t.x;
        r.v[1] = t.y;
    } else {
        r.v[0] = *p;
    }
    return r;
}

template <int VW>
__device__ __forceinline__ void st_vd(double *p, const Vd<VW> &r) {
    if constexpr (VW == 2)
        *reinterpret_cast<double2 *>(p) = make_double2(r.v[0], r.v[1]);
    else
        *p = r.v[0];
}

// ---- whole trains per launch -------------------------------------------------
// The formal sum, the stencil sum and the copy write every core of
// a train independently: one launch takes up to TRAIN_CHUNK cores (descriptors
// in the kernel arguments), with gridDim.z over the cores, y over a core's
// columns and x over the rows of a column.  Trains of low rank are bound by
// launches (about 3 us each on the stream), large ones by HBM.  Two rank
// indices are moved per lane where ranks and addresses allow 16-byte accesses.
// The headline sum (d = 40, n = 1024, 64 + 64 -> 128) is at the card's copy
// rate (4.7 TB/s) either way.
constexpr int TRAIN_CHUNK = 32;

// Grid of a train launch: rows and cols are the largest of its cores; about
// 16384 workgroups in all, each grid-stride.
dim3 grid_train(long rows, long cols, int ncores, int vw) {
    const unsigned gy = (unsigned)(cols < 1 ? 1 : cols < 65535 ? cols : 65535);
    long gx = (rows + 256L * vw - 1) / (256L * vw);
    const long cap = (16384L + (long)gy * ncores - 1) / ((long)gy * ncores);
    if (gx > cap) gx = cap;
    if (gx < 1) gx = 1;
    return dim3((unsigned)gx, gy, (unsigned)ncores);
}

struct SumCore {
    const double *x, *y;
    double *z;
    double a, b;
    int kind, n, rx0, rx1, ry0, ry1;
    FastDiv drz0;  // division by z's left rank
};
struct SumChunk {
    SumCore c[TRAIN_CHUNK];
};

// z = a*x (+) b*y.  kind 0 first core (cols concat), 1 interior (block
// diagonal), 2 last (rows concat).  attac.c:81-112.  VW rank indices per
// thread (both left ranks even, 16-byte aligned cores).
template <int VW>
__global__ __launch_bounds__(256) void k_axpby_train(SumChunk ch) {
    const SumCore &s = ch.c[blockIdx.z];
    const int kind = s.kind, n = s.n, rx0 = s.rx0, rx1 = s.rx1, ry0 = s.ry0, ry1 = s.ry1;
    const double *__restrict__ x = s.x;
    const double *__restrict__ y = s.y;
    const int rz0 = (kind == 0) ? 1 : rx0 + ry0;
    const int rz1 = (kind == 2) ? 1 : rx1 + ry1;
    const unsigned rows = (unsigned)rz0 * (unsigned)n;
    for (int col = blockIdx.y; col < rz1; col += gridDim.y) {
        double *__restrict__ zc = s.z + (long)col * rows;
        for (unsigned m = VW * (blockIdx.x * blockDim.x + threadIdx.x); m < rows;
             m += VW * gridDim.x * blockDim.x) {
            const int j = (int)fdiv(m, s.drz0);
            const int al = (int)m - j * rz0;
            Vd<VW> v;
#pragma unroll
            for (int q = 0; q < VW; q++) v.v[q] = 0.0;
            if (kind == 0) {
                const bool left = col < rx1;
                v = ld_vd<VW>(left ? x + j + (long)n * col : y + j + (long)n * (col - rx1));
#pragma unroll
                for (int q = 0; q < VW; q++) v.v[q] = v.v[q] * (left ? s.a : s.b);
            } else if (kind == 2) {
                v = ld_vd<VW>((al < rx0) ? x + al + (long)rx0 * j : y + (al - rx0) + (long)ry0 * j);
            } else {
                if (al < rx0 && col < rx1)
                    v = ld_vd<VW>(x + al + (long)rx0 * (j + (long)n * col));
                else if (al >= rx0 && col >= rx1)
                    v = ld_vd<VW>(y + (al - rx0) + (long)ry0 * (j + (long)n * (col - rx1)));
            }
            st_vd<VW>(zc + m, v);
        }
    }
}

struct CopyCore {
    const double *src;
    double *dst;
    long count;
};
struct CopyChunk {
    CopyCore c[TRAIN_CHUNK];
};

// Copies of whole cores (y over the cores): 16 bytes a lane, the odd element by
// the first lane.  Unaligned cores go element by element.
__global__ __launch_bounds__(256) void k_copy_train(CopyChunk ch) {
    const CopyCore &c = ch.c[blockIdx.y];
    const long stride = (long)gridDim.x * blockDim.x;
    const long t0 = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if ((((uintptr_t)c.src | (uintptr_t)c.dst) & 15) == 0) {
        const double2 *s2 = reinterpret_cast<const double2 *>(c.src);
        double2 *d2 = reinterpret_cast<double2 *>(c.dst);
        const long half = c.count >> 1;
        for (long e = t0; e < half; e += stride) d2[e] = s2[e];
        if (t0 == 0 && (c.count & 1)) c.dst[c.count - 1] = c.src[c.count - 1];
    } else {
        for (long e = t0; e < c.count; e += stride) c.dst[e] = c.src[e];
    }
}

struct ModeSumCore {
    const double *u;
    double *s;
    int kind, r0, n, r1;  // kind 0 first, 1 interior, 2 last, 3 the only core
    FastDiv ds0;          // division by s's left rank
};
struct ModeSumChunk {
    ModeSumCore c[TRAIN_CHUNK];
    double st[3];
};

// z[(ry0*ax+ay), j, (ry1*bx+by)] = x[ax,j,bx] * y[ay,j,by] (utilities.c:112-129)
__global__ void k_hadamard_core(int n, int rx0, int rx1, const double *__restrict__ x,
                                int ry0, int ry1, const double *__restrict__ y,
                                double *__restrict__ z, FastDiv drz0, FastDiv dry0) {
    const int rz0 = rx0 * ry0, rz1 = rx1 * ry1;
    const unsigned rows = (unsigned)rz0 * (unsigned)n;
    for (int col = blockIdx.y; col < rz1; col += gridDim.y) {
        const int bx = col / ry1, by = col - bx * ry1;
        const double *xc = x + (long)rx0 * n * bx, *yc = y + (long)ry0 * n * by;
        double *zc = z + (long)col * rows;
        for (unsigned m = blockIdx.x * blockDim.x + threadIdx.x; m < rows;
             m += gridDim.x * blockDim.x) {
            const int j = (int)fdiv(m, drz0);
            const int al = (int)m - j * rz0;
            const int ax = (int)fdiv((unsigned)al, dry0), ay = al - ax * ry0;
            zc[m] = xc[ax + rx0 * j] * yc[ay + ry0 * j];
        }
    }
}

#pragma clang fp contract(off)

__global__ void k_diag_core(int r0, int n, int r1, const double *__restrict__ v,
                            double *__restrict__ f, FastDiv dr0) {
    const unsigned rows = (unsigned)r0 * (unsigned)n;
    for (int col = blockIdx.y; col < r1; col += gridDim.y) {
        double *fc = f + (long)col * rows;
        for (unsigned m = blockIdx.x * blockDim.x + threadIdx.x; m < rows;
             m += gridDim.x * blockDim.x)
            fc[m] *= v[fdiv(m, dr0)];
    }
}

// Mode stencils: paratt.c:584-661 (kind 1), :665-770 (kind 0), :772-923 (kind 2).
// VW consecutive rank indices (same mode index) per thread, loaded and
// stored as one vector when the leading rank is even: the arithmetic of each
// is the scalar path's, in the same order.
template <int VW>
__global__ void k_stencil_core(int kind, int r0, int n, int r1,
                               const double *__restrict__ sten, int slen,
                               const double *__restrict__ f, double *__restrict__ g,
                               FastDiv dr0) {
    const int h = (slen - 1) / 2;
    const unsigned rows = (unsigned)r0 * (unsigned)n;
    for (int col = blockIdx.y; col < r1; col += gridDim.y)
    for (unsigned m = VW * (blockIdx.x * blockDim.x + threadIdx.x); m < rows;
         m += VW * gridDim.x * blockDim.x) {
        const long e = (long)col * rows + m;
        const int i = (int)fdiv(m, dr0);
        const int al = (int)m - i * r0;
        const double *fb = f + al + (long)col * rows;  // fiber base; stride r0
#define FV(jj) ld_vd<VW>(fb + (long)r0 * (jj))
        Vd<VW> acc;
#pragma unroll
        for (int q = 0; q < VW; q++) acc.v[q] = 0.0;
        auto add = [&](double st, const Vd<VW> &x) {
#pragma unroll
            for (int q = 0; q < VW; q++) acc.v[q] += st * x.v[q];
        };
        if (kind == 1) {
            // exact periodic wrap, summed in stencil order
            for (int t = 0; t < slen; t++) {
                int jj = i + t - h;
                jj = jj < 0 ? jj + n : (jj >= n ? jj - n : jj);
                add(sten[t], FV(jj));
            }
        } else {
            int sc = 0, gc = 0;
            for (int jj = i - h; jj < i; jj++) {
                Vd<VW> v;
                if (jj < 0) {
                    v = (kind == 0) ? FV(n - h + gc) : FV(h - 1 - gc);
                    gc++;
                } else {
                    v = FV(jj);
                }
                add(sten[sc++], v);
            }
            add(sten[sc++], FV(i));
            gc = 0;
            for (int jj = i + 1; jj <= i + h; jj++) {
                Vd<VW> v;
                if (jj < n) {
                    v = FV(jj);
                } else {
                    v = (kind == 0) ? FV(gc) : FV(n - 1 - gc);
                    gc++;
                }
                add(sten[sc++], v);
            }
        }
        st_vd<VW>(g + e, acc);
#undef FV
    }
}

// S = sum_i D_i u as a rank-2r train (first core [D u | u], interior
// [[u, 0], [D u, u]], last [u; D u]), every block of S written in one pass
// with the 3-point periodic stencil of kind 0 applied on the way (same order of
// operations as k_stencil_core).  Written block by block (the stencil to a
// buffer, a zero fill, three placements) S was passed over more than twice: the
// whole operator at d = 20, n = 1024, r = 32 took 739 us and takes 248 us, 180 of
// them this kernel (756 MB read and written once, 4.2 TB/s; bound by HBM and the
// call's launch and wait).
template <int VW>
__global__ __launch_bounds__(256) void k_mode_sum_train(ModeSumChunk ch) {
    const ModeSumCore &c = ch.c[blockIdx.z];
    const int kind = c.kind, r0 = c.r0, n = c.n, r1 = c.r1;
    const double *__restrict__ u = c.u;
    const int s0 = (kind == 0 || kind == 3) ? r0 : 2 * r0;
    const int s1 = (kind >= 2) ? r1 : 2 * r1;
    const unsigned rows = (unsigned)s0 * (unsigned)n;
    for (int col = blockIdx.y; col < s1; col += gridDim.y) {
        double *__restrict__ sc = c.s + (long)col * rows;
        const bool right = col >= r1;  // the right half of the columns
        const double *uc = u + (long)(right ? col - r1 : col) * r0 * n;
        for (unsigned m = VW * (blockIdx.x * blockDim.x + threadIdx.x); m < rows;
             m += VW * gridDim.x * blockDim.x) {
            const int j = (int)fdiv(m, c.ds0);
            const int al = (int)m - j * s0;
            const bool low = al >= r0;  // the lower half of the rows
            const int a = low ? al - r0 : al;
            Vd<VW> v;
#pragma unroll
            for (int q = 0; q < VW; q++) v.v[q] = 0.0;
            const bool du = (kind == 0 || kind == 3) ? !right : (low && !right);
            const double *fb = uc + a;
            if (du) {
                const int jl = (j > 0) ? j - 1 : n - 1, jr = (j + 1 < n) ? j + 1 : 0;
                const Vd<VW> x = ld_vd<VW>(fb + (long)r0 * jl), y = ld_vd<VW>(fb + (long)r0 * j),
                             z = ld_vd<VW>(fb + (long)r0 * jr);
#pragma unroll
                for (int q = 0; q < VW; q++) {
                    double acc = 0.0;
                    acc += ch.st[0] * x.v[q];
                    acc += ch.st[1] * y.v[q];
                    acc += ch.st[2] * z.v[q];
                    v.v[q] = acc;
                }
            } else if (kind != 1 || low || !right) {
                v = ld_vd<VW>(fb + (long)r0 * j);
            }
            st_vd<VW>(sc + m, v);
        }
    }
}

// paratt.c:926-1093 at one rank; coef = [c(n), gc(2), s(n)].
__global__ void k_lf_flux_core(int r0, int n, int r1, const double *__restrict__ coef,
                               double dx, const double *__restrict__ f,
                               double *__restrict__ g, FastDiv dr0) {
    const double *c = coef, *gcw = coef + n, *s = coef + n + 2;
    const double s0 = -0.5 / dx, s2 = 0.5 / dx;
    const unsigned rows = (unsigned)r0 * (unsigned)n;
    for (int col = blockIdx.y; col < r1; col += gridDim.y)
    for (unsigned m = blockIdx.x * blockDim.x + threadIdx.x; m < rows;
         m += gridDim.x * blockDim.x) {
        const long e = (long)col * rows + m;
        const int i = (int)fdiv(m, dr0);
        const int al = (int)m - i * r0;
        const double *fb = f + al + (long)col * rows;
#define FV(jj) fb[(long)r0 * (jj)]
        double v = (i - 1 < 0) ? -gcw[0] * FV(0) : -c[i - 1] * FV(i - 1);
        double acc = 0.0;
        acc += s0 * v;
        v = (i + 1 < n) ? -c[i + 1] * FV(i + 1) : -gcw[1] * FV(n - 1);
        acc += s2 * v;
        g[e] = acc + s[i] * FV(i);
#undef FV
    }
}

// paratt.c:1096-1250 at one rank; coef = [c(n), gc(2), bw(n+1), s(n)].
__global__ void k_lw_rhs_core(int r0, int n, int r1, const double *__restrict__ coef,
                              double dt, double dx, const double *__restrict__ f,
                              double *__restrict__ g, FastDiv dr0) {
    const double *c = coef, *gcw = coef + n, *bw = coef + n + 2, *s = coef + 2 * n + 3;
    const unsigned rows = (unsigned)r0 * (unsigned)n;
    for (int col = blockIdx.y; col < r1; col += gridDim.y)
    for (unsigned m = blockIdx.x * blockDim.x + threadIdx.x; m < rows;
         m += gridDim.x * blockDim.x) {
        const long e = (long)col * rows + m;
        const int i = (int)fdiv(m, dr0);
        const int al = (int)m - i * r0;
        const double *fb = f + al + (long)col * rows;
#define FV(jj) fb[(long)r0 * (jj)]
        double uh0, uh1;
        if (i == 0) {
            double g0 = FV(0);
            uh0 = 0.5 * (g0 + FV(0)) - ((c[0] * FV(0) - g0 * gcw[0]) * dt / (2.0 * dx));
        } else {
            uh0 = 0.5 * (FV(i) + FV(i - 1)) -
                  ((c[i] * FV(i) - c[i - 1] * FV(i - 1)) * dt / (2.0 * dx));
        }
        if (i + 1 < n) {
            uh1 = 0.5 * (FV(i + 1) + FV(i)) -
                  ((c[i + 1] * FV(i + 1) - c[i] * FV(i)) * dt / (2.0 * dx));
        } else {
            double g1 = FV(n - 1);
            uh1 = 0.5 * (g1 + FV(i)) - ((g1 * gcw[1] - c[i] * FV(i)) * dt / (2.0 * dx));
        }
        g[e] = -(bw[i + 1] * uh1 - bw[i] * uh0) / dx + s[i] * FV(i);
#undef FV
    }
}

#pragma clang fp contract(on)

__global__ void k_copy2d(int m, int n, const double *__restrict__ A, long lda,
                         double *__restrict__ B, long ldb, double alpha) {
    long total = (long)m * n;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total;
         e += (long)gridDim.x * blockDim.x) {
        long j = e / m, i = e - j * m;
        B[i + j * ldb] = alpha * A[i + j * lda];
    }
}

// B (n x m) = alpha * A^T, A is m x n; 32x32 tiles through LDS.
__global__ void k_transpose(int m, int n, const double *__restrict__ A, long lda,
                            double *__restrict__ B, long ldb, double alpha) {
    __shared__ double tile[32][33];
    int bi = blockIdx.x * 32, bj = blockIdx.y * 32;
    int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 256 threads: ty 0..7
    for (int yy = ty; yy < 32; yy += 8) {
        int i = bi + tx, j = bj + yy;
        tile[yy][tx] = (i < m && j < n) ? A[i + (long)j * lda] : 0.0;
    }
    __syncthreads();
    for (int yy = ty; yy < 32; yy += 8) {
        int j = bj + tx, i = bi + yy;  // B(j, i) = A(i, j)
        if (j < n && i < m) B[j + (long)i * ldb] = alpha * tile[tx][yy];
    }
}

__global__ void k_fill(double *p, long count, double v) {
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < count;
         e += (long)gridDim.x * blockDim.x)
        p[e] = v;
}

__global__ void k_set_diag(double *A, int m, long lda, double alpha) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x)
        A[i + (long)i * lda] = alpha;
}

// Two-stage deterministic sum of squares: stage 1 gives one partial per
// workgroup (grid-stride over the block), stage 2 adds the partials in order.
__global__ __launch_bounds__(256) void k_sumsq_partial(int m, int n, const double *__restrict__ A,
                                                       long lda, double *__restrict__ part) {
    __shared__ double red[4];
    double s = 0.0;
    long total = (long)m * n;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total;
         e += (long)gridDim.x * blockDim.x) {
        long j = e / m, i = e - j * m;
        double v = A[i + j * lda];
        s += v * v;
    }
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ __launch_bounds__(256) void k_sum_final(int np, const double *__restrict__ part,
                                                   double *out) {
    __shared__ double red[4];
    double s = 0.0;
    for (int i = threadIdx.x; i < np; i += blockDim.x) s += part[i];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) *out = (red[0] + red[1]) + (red[2] + red[3]);
}

uint64_t mix64_host(uint64_t z) {
    z += 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}
uint64_t mix64_host_seed(uint64_t seed, int core) {
    return mix64_host(mix64_host(seed) + (uint64_t)core);
}

}  // namespace

extern "C" {

void ptt_hip_zero(void *p, size_t bytes) {
    ptt_hip_init();
    long cnt = (long)(bytes / sizeof(double));
    if (cnt <= 0) return;
    PTT_LAUNCH("zero", k_zero, dim3(stream_blocks(cnt, 256)), dim3(256), 0, (double *)p, cnt);
}

void ptt_hip_gauss_fill(double *dst, long count, uint64_t seed, int core, double scale) {
    ptt_hip_init();
    if (count <= 0) return;
    uint64_t h = mix64_host_seed(seed, core);
    long np = (count + 1) / 2;
    PTT_LAUNCH("gauss_fill", k_gauss_fill, dim3(stream_blocks(np, 256)), dim3(256), 0, dst,
               count, h, scale);
}

void ptt_hip_scale(double *p, long count, double alpha) {
    ptt_hip_init();
    if (count <= 0) return;
    PTT_LAUNCH("scale", k_scale, dim3(stream_blocks(count, 256)), dim3(256), 0, p, count, alpha);
}

void ptt_hip_axpby_train(int d, const int *kind, const int *n, const int *rx,
                         double *const *x, const int *ry, double *const *y, double a, double b,
                         double *const *z) {
    ptt_hip_init();
    // two chunks: cores that move in pairs and cores that do not
    SumChunk ch[2];
    int cnt[2] = {0, 0};
    long rows[2] = {0, 0}, cols[2] = {0, 0};
    double bytes[2] = {0.0, 0.0};
    auto flush = [&](int v) {
        if (!cnt[v]) return;
        const dim3 grid = grid_train(rows[v], cols[v], cnt[v], v ? 2 : 1);
        if (v)
            PTT_LAUNCH_FB("axpby", 0.0, bytes[v], k_axpby_train<2>, grid, dim3(256), 0, ch[v]);
        else
            PTT_LAUNCH_FB("axpby", 0.0, bytes[v], k_axpby_train<1>, grid, dim3(256), 0, ch[v]);
        cnt[v] = 0;
        rows[v] = cols[v] = 0;
        bytes[v] = 0.0;
    };
    for (int k = 0; k < d; k++) {
        SumCore c;
        c.kind = kind[k];
        c.n = n[k];
        c.rx0 = rx[k];
        c.rx1 = rx[k + 1];
        c.ry0 = ry[k];
        c.ry1 = ry[k + 1];
        c.x = x[k];
        c.y = y[k];
        c.z = z[k];
        c.a = a;
        c.b = b;
        const long rz0 = (c.kind == 0) ? 1 : c.rx0 + c.ry0, rz1 = (c.kind == 2) ? 1 : c.rx1 + c.ry1;
        const long total = rz0 * c.n * rz1;
        if (total <= 0) continue;
        c.drz0 = make_fastdiv((unsigned)rz0);
        const bool even = c.kind == 0 ? (c.n & 1) == 0 : ((c.rx0 | c.ry0) & 1) == 0;
        const int v =
            (even && (((uintptr_t)c.x | (uintptr_t)c.y | (uintptr_t)c.z) & 15) == 0) ? 1 : 0;
        ch[v].c[cnt[v]++] = c;
        if (rz0 * c.n > rows[v]) rows[v] = rz0 * c.n;
        if (rz1 > cols[v]) cols[v] = rz1;
        bytes[v] += 8.0 * ((double)c.rx0 * c.n * c.rx1 + (double)c.ry0 * c.n * c.ry1 + (double)total);
        if (cnt[v] == TRAIN_CHUNK) flush(v);
    }
    flush(0);
    flush(1);
}

void ptt_hip_copy_train(int d, double *const *dst, double *const *src, const long *count) {
    ptt_hip_init();
    CopyChunk ch;
    int cnt = 0;
    long most = 0;
    double bytes = 0.0;
    for (int k = 0; k <= d; k++) {
        if (k < d && count[k] > 0 && dst[k] != src[k]) {
            ch.c[cnt].src = src[k];
            ch.c[cnt].dst = dst[k];
            ch.c[cnt].count = count[k];
            cnt++;
            most = count[k] > most ? count[k] : most;
            bytes += 16.0 * (double)count[k];
        }
        if (cnt == TRAIN_CHUNK || (k == d && cnt > 0)) {
            long gx = (most + 511) / 512;
            const long cap = (16384 + cnt - 1) / cnt;
            gx = gx < 1 ? 1 : gx > cap ? cap : gx;
            PTT_LAUNCH_FB("copy_train", 0.0, bytes, k_copy_train, dim3((unsigned)gx, (unsigned)cnt),
                          dim3(256), 0, ch);
            cnt = 0;
            most = 0;
            bytes = 0.0;
        }
    }
}

void ptt_hip_axpby_core(int kind, int n, int rx0, int rx1, const double *x, int ry0, int ry1,
                        const double *y, double a, double b, double *z) {
    const int rx[2] = {rx0, rx1}, ry[2] = {ry0, ry1};
    double *const xs = (double *)x, *const ys = (double *)y;
    ptt_hip_axpby_train(1, &kind, &n, rx, &xs, ry, &ys, a, b, &z);
}

void ptt_hip_mode_sum_train(int d, const int *n, const int *r, double *const *u,
                            const double *sten3, double *const *s) {
    ptt_hip_init();
    ModeSumChunk ch[2];
    int cnt[2] = {0, 0};
    long rows[2] = {0, 0}, cols[2] = {0, 0};
    double bytes[2] = {0.0, 0.0};
    for (int v = 0; v < 2; v++)
        for (int q = 0; q < 3; q++) ch[v].st[q] = sten3[q];
    auto flush = [&](int v) {
        if (!cnt[v]) return;
        const dim3 grid = grid_train(rows[v], cols[v], cnt[v], v ? 2 : 1);
        if (v)
            PTT_LAUNCH_FB("mode_sum", 0.0, bytes[v], k_mode_sum_train<2>, grid, dim3(256), 0, ch[v]);
        else
            PTT_LAUNCH_FB("mode_sum", 0.0, bytes[v], k_mode_sum_train<1>, grid, dim3(256), 0, ch[v]);
        cnt[v] = 0;
        rows[v] = cols[v] = 0;
        bytes[v] = 0.0;
    };
    for (int k = 0; k < d; k++) {
        ModeSumCore c;
        c.kind = d == 1 ? 3 : k == 0 ? 0 : k == d - 1 ? 2 : 1;
        c.r0 = r[k];
        c.n = n[k];
        c.r1 = r[k + 1];
        c.u = u[k];
        c.s = s[k];
        const long s0 = (c.kind == 0 || c.kind == 3) ? c.r0 : 2L * c.r0;
        const long s1 = (c.kind >= 2) ? c.r1 : 2L * c.r1;
        const long total = s0 * c.n * s1;
        if (total <= 0) continue;
        c.ds0 = make_fastdiv((unsigned)s0);
        const int v =
            ((c.r0 & 1) == 0 && (((uintptr_t)c.u | (uintptr_t)c.s) & 15) == 0) ? 1 : 0;
        ch[v].c[cnt[v]++] = c;
        if (s0 * c.n > rows[v]) rows[v] = s0 * c.n;
        if (s1 > cols[v]) cols[v] = s1;
        bytes[v] += 8.0 * ((double)c.r0 * c.n * c.r1 + (double)total);
        if (cnt[v] == TRAIN_CHUNK) flush(v);
    }
    flush(0);
    flush(1);
}

void ptt_hip_hadamard_core(int n, int rx0, int rx1, const double *x, int ry0, int ry1,
                           const double *y, double *z) {
    ptt_hip_init();
    long total = (long)rx0 * ry0 * n * rx1 * ry1;
    double bytes = 8.0 * ((double)rx0 * n * rx1 + (double)ry0 * n * ry1 + (double)total);
    if (total <= 0) return;
    PTT_LAUNCH_FB("hadamard", 0.0, bytes, k_hadamard_core,
                  grid_core((long)rx0 * ry0 * n, (long)rx1 * ry1), dim3(256), 0, n, rx0, rx1, x,
                  ry0, ry1, y, z, make_fastdiv((unsigned)(rx0 * ry0)), make_fastdiv((unsigned)ry0));
}

void ptt_hip_diag_core(int r0, int n, int r1, const double *v, double *f) {
    ptt_hip_init();
    long total = (long)r0 * n * r1;
    if (total <= 0) return;
    PTT_LAUNCH_FB("diag", (double)total, 16.0 * total, k_diag_core, grid_core((long)r0 * n, r1),
                  dim3(256), 0, r0, n, r1, v, f, make_fastdiv((unsigned)r0));
}

void ptt_hip_stencil_core(int kind, int r0, int n, int r1, const double *sten, int slen,
                          const double *f, double *g) {
    ptt_hip_init();
    long total = (long)r0 * n * r1;
    if (total <= 0) return;
    // pairs of rank indices per thread when the leading rank is even and
    // both cores are 16-byte aligned
    if ((r0 & 1) == 0 && (((uintptr_t)f | (uintptr_t)g) & 15) == 0)
        PTT_LAUNCH_FB("stencil", 2.0 * slen * total, 16.0 * total, k_stencil_core<2>,
                      grid_core((long)r0 * n / 2, r1), dim3(256), 0, kind, r0, n, r1, sten, slen,
                      f, g, make_fastdiv((unsigned)r0));
    else
        PTT_LAUNCH_FB("stencil", 2.0 * slen * total, 16.0 * total, k_stencil_core<1>,
                      grid_core((long)r0 * n, r1), dim3(256), 0, kind, r0, n, r1, sten, slen, f,
                      g, make_fastdiv((unsigned)r0));
}

void ptt_hip_lf_flux_core(int r0, int n, int r1, const double *coef, double dt, double dx,
                          const double *f, double *g) {
    ptt_hip_init();
    (void)dt;
    long total = (long)r0 * n * r1;
    if (total <= 0) return;
    PTT_LAUNCH("lf_flux", k_lf_flux_core, grid_core((long)r0 * n, r1), dim3(256), 0, r0, n, r1,
               coef, dx, f, g, make_fastdiv((unsigned)r0));
}

void ptt_hip_lw_rhs_core(int r0, int n, int r1, const double *coef, double dt, double dx,
                         const double *f, double *g) {
    ptt_hip_init();
    long total = (long)r0 * n * r1;
    if (total <= 0) return;
    PTT_LAUNCH("lw_rhs", k_lw_rhs_core, grid_core((long)r0 * n, r1), dim3(256), 0, r0, n, r1,
               coef, dt, dx, f, g, make_fastdiv((unsigned)r0));
}

void ptt_hip_copy2d(int m, int n, const double *A, long lda, double *B, long ldb,
                    double alpha) {
    ptt_hip_init();
    long total = (long)m * n;
    if (total <= 0) return;
    PTT_LAUNCH("copy2d", k_copy2d, dim3(stream_blocks(total, 256)), dim3(256), 0, m, n, A, lda,
               B, ldb, alpha);
}

void ptt_hip_transpose(int m, int n, const double *A, long lda, double *B, long ldb,
                       double alpha) {
    ptt_hip_init();
    if (m <= 0 || n <= 0) return;
    PTT_LAUNCH("transpose", k_transpose, dim3(cdiv(m, 32), cdiv(n, 32)), dim3(256), 0, m, n, A,
               lda, B, ldb, alpha);
}

void ptt_hip_fill(double *p, long count, double v) {
    ptt_hip_init();
    if (count <= 0) return;
    PTT_LAUNCH("fill", k_fill, dim3(stream_blocks(count, 256)), dim3(256), 0, p, count, v);
}

void ptt_hip_set_diag(double *A, int m, long lda, double alpha) {
    ptt_hip_init();
    if (m <= 0) return;
    PTT_LAUNCH("set_diag", k_set_diag, dim3(cdiv(m, 256)), dim3(256), 0, A, m, lda, alpha);
}

void ptt_hip_sumsq(int m, int n, const double *A, long lda, double *out) {
    ptt_hip_init();
    long total = (long)m * n;
    int nb = (int)stream_blocks(total, 256);
    if (nb > 1024) nb = 1024;
    static double *g_part = nullptr;
    if (!g_part) g_part = (double *)ptt_hip_malloc(sizeof(double) * 1024);
    PTT_LAUNCH_FB("sumsq", 2.0 * total, 8.0 * total, k_sumsq_partial, dim3(nb), dim3(256), 0, m, n,
                  A, lda, g_part);
    PTT_LAUNCH("sum_final", k_sum_final, dim3(1), dim3(256), 0, nb, g_part, out);
}

}  // extern "C"
