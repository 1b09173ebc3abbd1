// gram.hip -- Gram matrices of tall-skinny / short-wide cores on the matrix
// cores (gfx950): G = A^T A for A (len x c, column-major) or G = M M^T for
// M (c x len), c <= 128, split over the long dimension.
//
// A workgroup of eight waves owns one slab of the long dimension and the
// whole c x c Gram: the slab is staged through LDS in steps of 32 (two buffers,
// one barrier a step, the next step's loads in flight meanwhile).  The
// upper-triangular 16 x 16 blocks (36 for c = 128) are dealt round-robin to four
// waves, so the symmetry halves the work with every wave busy; the other four
// waves take the other half of each step's rows, so that each SIMD has two waves
// whose products cover each other's LDS reads (the accumulators are added at the
// end).  A wave reads each column block's fragment once per four rows and uses it
// in all its products.  Each block accumulates v_mfma_*_16x16x4 products: the
// first operand holds the block row's 16 columns of the slab, the second the
// block column's.
// Bound by the matrix cores (33 us for 131072 x 128 in FP64).  That size took
// 67 us with four waves, one buffer and two LDS reads a product, and takes 57;
// 128 x 65536 took 41 and takes 36; 131072 x 128 in FP32 took 136 and takes 41.
// Sixteen waves (half the registers) spill: 150 us.
//
// FP64 (v_mfma_f64_16x16x4f64, FP64 accumulation) for the plain rounding;
// FP32 (v_mfma_f32_16x16x4f32, FP32 accumulation within a slab) for the
// first Cholesky-QR pass of the mixed-precision rounding, with the input
// scaled by an exact power of two first (the bond matrices of deep trains
// lie far below FP32's range).  Slab partials are summed in FP64 by the
// split-K reduction, which also mirrors the upper triangle.
#include "common.hpp"

using namespace ptt;

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int KC = 32;   // long-dimension rows staged per step
constexpr int GPAD = 1;  // LDS row padding (elements)
constexpr int GRAM_NT = 512;

template <typename T>
struct Acc;
template <>
struct Acc<double> {
    typedef f64x4 V;
    static __device__ __forceinline__ V mfma(double a, double b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // lane l, register v holds D[l/16 + 4v][l%16]
    static __device__ __forceinline__ int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <>
struct Acc<float> {
    typedef f32x4 V;
    static __device__ __forceinline__ V mfma(float a, float b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    // lane l, register v holds D[4 (l/16) + v][l%16]
    static __device__ __forceinline__ int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

// Upper-triangular block pair number idx of an nb x nb block grid.
constexpr int pair_row(int idx, int nb) {
    int p = 0, rowlen = nb;
    while (idx >= rowlen) {
        idx -= rowlen;
        p++;
        rowlen--;
    }
    return p;
}
constexpr int pair_col(int idx, int nb) {
    int p = 0, rowlen = nb;
    while (idx >= rowlen) {
        idx -= rowlen;
        p++;
        rowlen--;
    }
    return p + idx;
}

// Power-of-two exponent bringing the largest |entry| (*dmax) to [1, 2); 0
// without a bound (dmax NULL) or for a zero / non-finite bound.
__device__ __forceinline__ int scale_exp(const double *dmax) {
    if (!dmax) return 0;
    const double m = *dmax;
    return (m > 0.0 && m < INFINITY) ? ilogb(m) : 0;
}

// The blocks of wave WQ of four: products of one K-group's four k-slices of a
// staged step (rows r0 .. r0 + 15 of s).
template <typename T, int CP, int WQ>
struct GramWave {
    typedef Acc<T> AC;
    typedef typename AC::V V;
    static constexpr int NB = CP / 16, NBLK = NB * (NB + 1) / 2, LD = CP + GPAD;
    static constexpr int MINE = (NBLK - WQ + 3) / 4;
    template <int B>
    static constexpr int row() { return pair_row(WQ + 4 * B, NB); }
    template <int B>
    static constexpr int col() { return pair_col(WQ + 4 * B, NB); }
    template <int B>
    static __device__ __forceinline__ void mul(const T (&f)[NB], V *acc) {
        if constexpr (B < MINE) {
            constexpr int p = row<B>(), q = col<B>();
            acc[B] = AC::mfma(f[p], f[q], acc[B]);
            mul<B + 1>(f, acc);
        }
    }
    static __device__ __forceinline__ void step(const T *s, int r0, int lane, V *acc) {
#pragma unroll
        for (int ks = 0; ks < KC / 8; ks++) {
            const T *row = s + (r0 + ks * 4 + (lane >> 4)) * LD + (lane & 15);
            T f[NB];
#pragma unroll
            for (int p = 0; p < NB; p++) f[p] = row[16 * p];
            mul<0>(f, acc);
        }
    }
    template <int B>
    static __device__ __forceinline__ void give(T *red, int lane, const V *acc) {
        if constexpr (B < MINE) {
#pragma unroll
            for (int v = 0; v < 4; v++) red[((WQ + 4 * B) * 4 + v) * 64 + lane] = acc[B][v];
            give<B + 1>(red, lane, acc);
        }
    }
    template <int B>
    static __device__ __forceinline__ void write(const T *red, int lane, int c, const V *acc,
                                                 double *out) {
        if constexpr (B < MINE) {
            constexpr int pb = row<B>() * 16, qb = col<B>() * 16;
            const int q = qb + (lane & 15);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int p = pb + AC::row(lane, v);
                const T x = acc[B][v] + red[((WQ + 4 * B) * 4 + v) * 64 + lane];
                if (p < c && q < c && p <= q) out[p + (long)q * c] = (double)x;
            }
            write<B + 1>(red, lane, c, acc, out);
        }
    }
};

// TR: G = A^T A with element (k, p) of the slab at A[k + p lda];
// otherwise G = M M^T with element (k, p) at M[p + k lda].  The slab's
// entries are scaled by 2^-scale_exp(dmax) before the conversion to T.
template <typename T, bool TR, int CP>
__global__ __launch_bounds__(GRAM_NT) void k_gram(int c, long len, long kchunk,
                                                  const double *__restrict__ A, long lda,
                                                  const double *__restrict__ dmax,
                                                  double *__restrict__ partial) {
    typedef typename Acc<T>::V V;
    constexpr int NB = CP / 16, NBLK = NB * (NB + 1) / 2, MAXB = (NBLK + 3) / 4;
    constexpr int LD = CP + GPAD;
    constexpr int PER = KC * CP / GRAM_NT;  // staged elements per thread
    extern __shared__ double lds_raw[];
    T *s = (T *)lds_raw;  // two buffers of KC x LD, then the accumulators' exchange
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int wq = wv & 3, r0 = (wv >> 2) * (KC / 2);
    const double prescale = ldexp(1.0, -scale_exp(dmax));
    const long kbeg = (long)blockIdx.x * kchunk;
    const long kend = min(len, kbeg + kchunk);

    V acc[MAXB];
#pragma unroll
    for (int b = 0; b < MAXB; b++) acc[b] = V{0, 0, 0, 0};

    double reg[PER];
    auto load = [&](long k0) {
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const int idx = tid + GRAM_NT * e;
            int kk, p;
            if (TR) {
                kk = idx % KC;
                p = idx / KC;
            } else {
                p = idx % CP;
                kk = idx / CP;
            }
            const long k = k0 + kk;
            const bool in = p < c && k < kend;  // an entry outside reads A[0] instead
            reg[e] = A[in ? (TR ? k + (long)p * lda : p + k * lda) : 0];
        }
    };
    // (nothing is done with what was loaded until here: it would wait for it)
    auto store = [&](T *buf, long k0) {
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const int idx = tid + GRAM_NT * e;
            int kk, p;
            if (TR) {
                kk = idx % KC;
                p = idx / KC;
            } else {
                p = idx % CP;
                kk = idx / CP;
            }
            buf[kk * LD + p] = p < c && k0 + kk < kend ? (T)(reg[e] * prescale) : (T)0;
        }
    };

    if (kbeg < kend) {
        load(kbeg);
        store(s, kbeg);
    }
    __syncthreads();
    int cur = 0;
    for (long k0 = kbeg; k0 < kend; k0 += KC) {
        const bool more = k0 + KC < kend;
        if (more) load(k0 + KC);
        const T *buf = s + cur * (KC * LD);
        if (wq == 0) GramWave<T, CP, 0>::step(buf, r0, lane, acc);
        else if (wq == 1) GramWave<T, CP, 1>::step(buf, r0, lane, acc);
        else if (wq == 2) GramWave<T, CP, 2>::step(buf, r0, lane, acc);
        else GramWave<T, CP, 3>::step(buf, r0, lane, acc);
        if (more) store(s + (cur ^ 1) * (KC * LD), k0 + KC);
        __syncthreads();
        cur ^= 1;
    }
    // the second K-group's accumulators through LDS, then the partial (c x c, ld
    // c) of this slab: the upper blocks only
    if (wv >= 4) {
        if (wq == 0) GramWave<T, CP, 0>::template give<0>(s, lane, acc);
        else if (wq == 1) GramWave<T, CP, 1>::template give<0>(s, lane, acc);
        else if (wq == 2) GramWave<T, CP, 2>::template give<0>(s, lane, acc);
        else GramWave<T, CP, 3>::template give<0>(s, lane, acc);
    }
    __syncthreads();
    if (wv < 4) {
        double *out = partial + (long)blockIdx.x * c * c;
        if (wq == 0) GramWave<T, CP, 0>::template write<0>(s, lane, c, acc, out);
        else if (wq == 1) GramWave<T, CP, 1>::template write<0>(s, lane, c, acc, out);
        else if (wq == 2) GramWave<T, CP, 2>::template write<0>(s, lane, c, acc, out);
        else GramWave<T, CP, 3>::template write<0>(s, lane, c, acc, out);
    }
}

template <typename T, int CP>
constexpr size_t gram_lds() {
    constexpr size_t nb = CP / 16, blk = nb * (nb + 1) / 2;
    constexpr size_t a = 2 * KC * (CP + GPAD), b = blk * 256;
    return sizeof(T) * (a > b ? a : b);
}

// Sum of the slab partials (upper triangle), times alpha, written to both
// triangles.  Workgroup (q, h) owns rows 16h..16h+15 of column q of the upper
// triangle (workgroups wholly below the diagonal exit at once), so only the
// upper partials are read, each coalesced along the rows; its 256 threads
// split the slabs sixteen ways (sixteen loads in flight per thread), then
// combine through LDS.
__global__ __launch_bounds__(256) void k_gram_reduce(int c, int nsplit,
                                                     const double *__restrict__ partial,
                                                     const double *__restrict__ dmax,
                                                     double *__restrict__ G) {
    __shared__ double red[16][17];
    const int nch = (c + 15) >> 4;
    const int q = blockIdx.x / nch, h = blockIdx.x - q * nch;
    if (16 * h > q) return;
    const double alpha = ldexp(1.0, 2 * scale_exp(dmax));
    const int o = threadIdx.x & 15, zs = threadIdx.x >> 4;
    const int p = 16 * h + o;
    const long total = (long)c * c;
    const long src = p + (long)q * c;
    double s = 0.0;
    if (p <= q) {
        double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
        int z = zs;
        for (; z + 48 < nsplit; z += 64) {
            a0 += partial[(long)z * total + src];
            a1 += partial[(long)(z + 16) * total + src];
            a2 += partial[(long)(z + 32) * total + src];
            a3 += partial[(long)(z + 48) * total + src];
        }
        for (; z < nsplit; z += 16) a0 += partial[(long)z * total + src];
        s = (a0 + a1) + (a2 + a3);
    }
    red[zs][o] = s;
    __syncthreads();
    if (zs == 0 && p <= q) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < 16; w++) t += red[w][o];
        G[src] = alpha * t;
        G[q + (long)p * c] = alpha * t;
    }
}

// Largest |A_i| over count entries into *out (which starts at 0): one atomic
// maximum per workgroup on the bit patterns (ordered like the values for
// non-negative doubles).
__global__ __launch_bounds__(256) void k_maxabs(long count, const double *__restrict__ A,
                                                unsigned long long *__restrict__ out) {
    double m = 0.0;
    for (long i = blockIdx.x * 256L + threadIdx.x; i < count; i += (long)gridDim.x * 256)
        m = fmax(m, fabs(A[i]));
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    __shared__ double sm[4];
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fmax(fmax(sm[0], sm[1]), fmax(sm[2], sm[3]));
        atomicMax(out, (unsigned long long)__double_as_longlong(m));
    }
}

template <typename T>
void launch_gram(char trans, int c, long len, const double *A, long lda, const double *dmax,
                 double *G, const char *name) {
    // about one slab per CU (each partial Gram costs a c x c write and read
    // in the reduction), each at least 64 long and a multiple of KC: a short
    // operand is spread over more workgroups, each with fewer dependent
    // staging steps (the Grams of low-rank trains are latency-bound)
    long nsplit = 256;  // 512 and 1024 measured no faster at cfg2 (the reduction grows)
    if (len / nsplit < 64) nsplit = (len + 63) / 64;
    if (nsplit < 1) nsplit = 1;
    long kchunk = (len + nsplit - 1) / nsplit;
    kchunk = (kchunk + KC - 1) / KC * KC;
    nsplit = (len + kchunk - 1) / kchunk;
    double *partial =
        (double *)ptt_hip_scratch(PTT_WS_GRAM, sizeof(double) * (size_t)nsplit * c * c);
    const bool tr = (trans == 'T' || trans == 't');
    // algorithmic work: the symmetric half, c (c+1) len flops; A read once
    const double fl = (double)c * (c + 1) * (double)len, by = 8.0 * ((double)c * len + (double)c * c);
    dim3 grid((unsigned)nsplit);
    static bool attr = false;
    if (!attr) {
        auto set = [](const void *f, size_t bytes) {
            HIPCHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
        };
        set((const void *)k_gram<T, true, 64>, gram_lds<T, 64>());
        set((const void *)k_gram<T, false, 64>, gram_lds<T, 64>());
        set((const void *)k_gram<T, true, 128>, gram_lds<T, 128>());
        set((const void *)k_gram<T, false, 128>, gram_lds<T, 128>());
        attr = true;
    }
#define PTT_GRAM(TR, CP)                                                                       \
    PTT_LAUNCH_FB(name, fl, by, (k_gram<T, TR, CP>), grid, dim3(GRAM_NT), (gram_lds<T, CP>()), c, \
                  len, kchunk, A, lda, dmax, partial)
    if (c <= 64) {
        if (tr) PTT_GRAM(true, 64);
        else PTT_GRAM(false, 64);
    } else {
        if (tr) PTT_GRAM(true, 128);
        else PTT_GRAM(false, 128);
    }
#undef PTT_GRAM
    PTT_LAUNCH("gram_reduce", k_gram_reduce, dim3((unsigned)(c * cdiv(c, 16))), dim3(256), 0, c,
               (int)nsplit, partial, dmax, G);
}

}  // namespace

extern "C" {

void ptt_hip_gram_syrk(char trans, int c, long len, const double *A, long lda, double *G) {
    ptt_hip_init();
    if (c <= 0) return;
    if (c > 128 || len <= 0) {
        fprintf(stderr, "ptt_hip_gram_syrk: c = %d, len = %ld out of range\n", c, len);
        exit(1);
    }
    launch_gram<double>(trans, c, len, A, lda, nullptr, G,
                        trans == 'T' || trans == 't' ? "gram_tn" : "gram_nt");
}

void ptt_hip_gram32(char trans, int c, long len, const double *A, long lda, double *G) {
    ptt_hip_init();
    if (c <= 0) return;
    if (c > 128 || len <= 0) {
        fprintf(stderr, "ptt_hip_gram32: c = %d, len = %ld out of range\n", c, len);
        exit(1);
    }
    // the largest |entry| sets the power-of-two scaling into FP32's range
    double *dmax = (double *)ptt_hip_scratch(PTT_WS_INT, sizeof(int) * 64) + 30;
    ptt_hip_zero(dmax, sizeof(double));
    const long count = (trans == 'T' || trans == 't') ? len * (long)c : len * (long)c;
    if ((trans == 'T' || trans == 't') ? lda != len : lda != c) {
        fprintf(stderr, "ptt_hip_gram32: leading dimension must equal the rows\n");
        exit(1);
    }
    PTT_LAUNCH_FB("maxabs", 0.0, 8.0 * (double)count, k_maxabs, dim3(stream_blocks(count, 256)),
                  dim3(256), 0, count, A, (unsigned long long *)dmax);
    launch_gram<float>(trans, c, len, A, lda, dmax, G,
                       trans == 'T' || trans == 't' ? "gram32_tn" : "gram32_nt");
}

double ptt_hip_maxabs(const double *A, long count) {
    ptt_hip_init();
    if (count <= 0) return 0.0;
    double *dmax = (double *)ptt_hip_scratch(PTT_WS_INT, sizeof(int) * 64) + 29;
    ptt_hip_zero(dmax, sizeof(double));
    PTT_LAUNCH_FB("maxabs", 0.0, 8.0 * (double)count, k_maxabs, dim3(stream_blocks(count, 256)),
                  dim3(256), 0, count, A, (unsigned long long *)dmax);
    double m = 0.0;
    ptt_hip_d2h(&m, dmax, sizeof(double));
    return m;
}

}  // extern "C"
