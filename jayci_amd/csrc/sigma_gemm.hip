// Dense-string full-CI sigma on MFMA (see sigma_gemm.h for the decomposition).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
#include "mfma.h"
#include "sigma_gemm.h"
#include "slater.h"

#define RCHECK(x)                      \
    do {                               \
        int rc_ = (x);                 \
        if (rc_) return rc_;           \
    } while (0)

#define GF_CHECK()                                                       \
    do {                                                                 \
        hipError_t e_ = hipGetLastError();                               \
        if (e_ != hipSuccess) {                                          \
            jci_set_error("%s:%d launch: %s", __FILE__, __LINE__,        \
                          hipGetErrorString(e_));                        \
            return -2;                                                   \
        }                                                                \
    } while (0)

// ---- set-up kernels ---------------------------------------------------------------------------
__global__ void k_gf_dense(long long nstr, const uint64_t *__restrict__ mask,
                           const long long *__restrict__ off1, const int2 *__restrict__ e1,
                           const double *__restrict__ v1, const long long *__restrict__ off2,
                           const int2 *__restrict__ e2, const double *__restrict__ v2,
                           const double *__restrict__ m1, const double *__restrict__ m2,
                           double *__restrict__ H)
{
    long long I = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (I >= nstr) return;
    const uint64_t s = mask[I];
    double d = 0.0;
    for (uint64_t x = s; x; x &= x - 1) {
        int i = jci_ctz(x);
        d += jci_h1(m1, i, i);
        for (uint64_t y = s & ((1ULL << i) - 1ULL); y; y &= y - 1) {
            int j = jci_ctz(y);
            d += jci_eri(m2, i, i, j, j) - jci_eri(m2, i, j, i, j);
        }
    }
    double *row = H + I * nstr;
    row[I] = d;
    for (long long e = off1[I]; e < off1[I + 1]; e++) {
        int2 en = e1[e];
        double v = v1[e];
        row[en.x] = (en.y & (1 << 12)) ? -v : v;
    }
    for (long long e = off2[I]; e < off2[I + 1]; e++) row[e2[e].x] = v2[e];
}

__global__ void k_gf_lists(long long nstr, const uint64_t *__restrict__ mask,
                           const long long *__restrict__ off1, const int2 *__restrict__ e1, int L,
                           int Lp, uint32_t pad, int diag_one, uint32_t *__restrict__ out)
{
    long long I = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (I >= nstr) return;
    uint32_t *o = out + I * Lp;
    for (int i = L; i < Lp; i++) o[i] = pad << 16;
    int n = 0;
    for (long long e = off1[I]; e < off1[I + 1] && n < L; e++) {
        int2 en = e1[e];
        int i = en.y & 63, f = (en.y >> 6) & 63;
        uint32_t P = (uint32_t)jci_tri(i, f);
        o[n++] = (uint32_t)en.x | (P << 16) | ((uint32_t)((en.y >> 12) & 1) << 31);
    }
    if (diag_one) {
        if (mask[I] && n < L) o[n++] = (uint32_t)I | ((uint32_t)GF_PDIAG << 16);
        return;
    }
    for (uint64_t x = mask[I]; x && n < L; x &= x - 1) {
        int k = jci_ctz(x);
        o[n++] = (uint32_t)I | ((uint32_t)jci_tri(k, k) << 16);
    }
}

// E row of each alpha-list entry: the position of the entry's pair in its target's list
__global__ void k_gf_rank(long long nstr, int L, const uint32_t *__restrict__ in,
                          uint32_t *__restrict__ out, int *__restrict__ missing)
{
    long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nstr * L) return;
    const uint32_t w = in[idx];
    const long long J = w & 0xFFFFu;
    const uint32_t P = (w >> 16) & 0xFFu;
    uint32_t pos = 0;
    bool found = false;
    if (J < nstr)
        for (int e = 0; e < L; e++)
            if (((in[J * L + e] >> 16) & 0xFFu) == P) { pos = (uint32_t)e; found = true; break; }
    if (!found) atomicAdd(missing, 1);
    out[idx] = (w & ~(0x7Fu << 24)) | (pos << 24);
}

__global__ void k_gf_diagrows(long long nstr, int MP, const uint64_t *__restrict__ mask,
                              const double *__restrict__ M64, double *__restrict__ o64,
                              float *__restrict__ o32)
{
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nstr * MP) return;
    const long long J = idx / MP;
    const int Q = (int)(idx - J * MP);
    double s = 0.0;
    for (uint64_t x = mask[J]; x; x &= x - 1) {
        const int k = jci_ctz(x);
        s += M64[jci_tri(k, k) * MP + Q];
    }
    o64[idx] = s;
    o32[idx] = (float)s;
}

__global__ void k_gf_m2pad(int m1, int MP, const double *__restrict__ sq, double *__restrict__ o64,
                           float *__restrict__ o32)
{
    int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= MP * MP) return;
    int P = idx / MP, Q = idx - P * MP;
    double v = (P < m1 && Q < m1) ? sq[(long long)P * m1 + Q] : 0.0;
    o64[idx] = v;
    o32[idx] = (float)v;
}


// ---- grouped kernels ------------------------------------------------------------------------
template <typename T> __device__ __forceinline__ const T *hmat(const GemmFci &g, int spin);
template <> __device__ __forceinline__ const double *hmat<double>(const GemmFci &g, int spin)
{
    return g.H64[spin];
}
template <> __device__ __forceinline__ const float *hmat<float>(const GemmFci &g, int spin)
{
    return g.H32[spin];
}
template <typename T> __device__ __forceinline__ const T *mpad(const GemmFci &g);
template <> __device__ __forceinline__ const double *mpad<double>(const GemmFci &g) { return g.M64; }
template <> __device__ __forceinline__ const float *mpad<float>(const GemmFci &g) { return g.M32; }
template <typename T> __device__ __forceinline__ const T *drows(const GemmFci &g);
template <> __device__ __forceinline__ const double *drows<double>(const GemmFci &g) { return g.D64; }
template <> __device__ __forceinline__ const float *drows<float>(const GemmFci &g) { return g.D32; }

// input vector k of a task in the arithmetic type
template <typename T> __device__ __forceinline__ const T *xin(const GfTask &t, int k);
template <> __device__ __forceinline__ const double *xin<double>(const GfTask &t, int k)
{
    return t.x64 + (long long)k * t.ldx64;
}
template <> __device__ __forceinline__ const float *xin<float>(const GfTask &t, int k)
{
    return t.x32 + (long long)k * t.g.na * t.g.nb;
}

// task owning flattened unit u of kernel `which` (tasks ordered by base)
__device__ __forceinline__ int find_task(const GfTask *__restrict__ T, int n, long long u, int which)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (T[mid].base[which] <= u) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// FP64 -> FP32 copies of the input vectors, 256 elements per unit
__global__ __launch_bounds__(256) void k_gcv(const GfHeader *__restrict__ H,
                                             const GfTask *__restrict__ tasks)
{
    const int n = H->n;
    const long long total = H->total[GF_CV];
    for (long long u = blockIdx.x; u < total; u += gridDim.x) {
        const GfTask &t = tasks[find_task(tasks, n, u, GF_CV)];
        const long long N = t.g.na * t.g.nb;
        const long long idx = (u - t.base[GF_CV]) * 256 + threadIdx.x;
        if (idx < N * t.K) {
            const long long k = idx / N, i = idx - k * N;
            t.x32[idx] = (float)t.x64[k * t.ldx64 + i];
        }
    }
}

// ---- same-spin products -----------------------------------------------------------------------
// four consecutive elements at an address aligned to one
template <typename T> struct Gs;
template <> struct Gs<double> {
    typedef double quad __attribute__((ext_vector_type(4), aligned(8)));
    typedef double pair __attribute__((ext_vector_type(2), aligned(8)));
};
template <> struct Gs<float> {
    typedef float quad __attribute__((ext_vector_type(4), aligned(4)));
    typedef float pair __attribute__((ext_vector_type(2), aligned(4)));
};
typedef double GsOut __attribute__((ext_vector_type(2), aligned(8)));

// operands of one 16-deep step of a wave's tile: rows m of A, columns n of B
template <typename T, int RT> struct GsStep { T a[RT][4], b[4][RT]; };

// acc += A B over reduction steps [s0, s1) of 16, A row-major (lda), B row-major (ldb): a wave's
// tile of RT x RT 16 x 16 tiles straight from memory, without LDS.  Lane group l / 16 takes the
// reduction indexes 4 (l / 16) .. + 3 of a step, four consecutive elements of a row of A; the
// columns are dealt out so that lane l % 16 has RT consecutive ones, one wide read of a row of
// B.  The operands of the next step are loaded during the products of this one.  Rows, columns
// and the last reduction indexes past the end are moved back inside (their results equal the
// ones that are stored twice; reduction indexes met before are taken with zero from A).
template <typename T, int RT>
__device__ __forceinline__ void gs_wave(typename Mf<T>::acc (&acc)[RT][RT], const T *A, int lda,
                                        const T *B, int ldb, int Kr, const int (&m)[RT], int n, int s0,
                                        int s1)
{
    typedef const __attribute__((address_space(1))) typename Gs<T>::quad *QP;
    typedef const __attribute__((address_space(1))) typename Gs<T>::pair *PP;
    const int part = (threadIdx.x & 63) >> 4;
    const auto Ag = gptr(A), Bg = gptr(B);
    uint32_t ao[RT];
#pragma unroll
    for (int i = 0; i < RT; i++) ao[i] = (uint32_t)m[i] * (uint32_t)lda;
    auto load = [&](int s, GsStep<T, RT> &o) __attribute__((always_inline)) {
        const int k = std::min(s * 16 + part * 4, Kr - 4);
#pragma unroll
        for (int i = 0; i < RT; i++) {
            const typename Gs<T>::quad v = *(QP)(Ag + (ao[i] + (uint32_t)k));
#pragma unroll
            for (int j = 0; j < 4; j++) o.a[i][j] = v[j];
        }
        const uint32_t bo = (uint32_t)k * (uint32_t)ldb + (uint32_t)n;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const auto row = Bg + (bo + (uint32_t)(j * ldb));
            if constexpr (RT == 4) {
                const typename Gs<T>::quad v = *(QP)row;
#pragma unroll
                for (int c = 0; c < 4; c++) o.b[j][c] = v[c];
            } else {
                const typename Gs<T>::pair v = *(PP)row;
#pragma unroll
                for (int c = 0; c < RT; c++) o.b[j][c] = v[c];
            }
        }
    };
    auto mul = [&](GsStep<T, RT> &o) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int c = 0; c < RT; c++) acc[i][c] = Mf<T>::mma(o.a[i][j], o.b[j][c], acc[i][c]);
    };
    // zero the reduction indexes of a moved quad that an earlier one has
    auto trim = [&](int s, GsStep<T, RT> &o) __attribute__((always_inline)) {
        const int over = s * 16 + part * 4 - (Kr - 4);
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (j < over) o.a[i][j] = (T)0;
    };
    if (s0 >= s1) return;
    GsStep<T, RT> o[2];
    load(s0, o[0]);
    int s = s0;
    for (; s + 2 < s1; s += 2) {
        load(s + 1, o[1]);
        mul(o[0]);
        load(s + 2, o[0]);
        mul(o[1]);
    }
    if (s + 1 < s1) {
        load(s + 1, o[1]);
        mul(o[0]);
        trim(s + 1, o[1]);
        mul(o[1]);
    } else {
        trim(s, o[0]);
        mul(o[0]);
    }
}

// y_k = Haa X_k + X_k Hbb on a tile of the block's (RT = 4: 64 x 64, RT = 2: 32 x 32), every
// wave over a quarter of the two reductions, the four sums added in LDS
template <typename T, int RT>
__device__ __forceinline__ void gs_split(const GfTask &t, const T *X, double *y, int m0, int n0, T *red)
{
    const GemmFci &g = t.g;
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, na = (int)g.na, nb = (int)g.nb;
    typename Mf<T>::acc acc[RT][RT];
    int m[RT];
#pragma unroll
    for (int i = 0; i < RT; i++) {
        m[i] = std::min(m0 + i * 16 + (l & 15), na - 1);
#pragma unroll
        for (int c = 0; c < RT; c++) acc[i][c] = Mf<T>::zero();
    }
    const int n = std::min(n0 + RT * (l & 15), nb - RT);
    const int ka = (na + 15) / 16, kb = (nb + 15) / 16, q0 = (ka + kb) * w / 4, q1 = (ka + kb) * (w + 1) / 4;
    gs_wave<T, RT>(acc, hmat<T>(g, 0), na, X, nb, na, m, n, q0, std::min(q1, ka));
    gs_wave<T, RT>(acc, X, nb, hmat<T>(g, 1), nb, nb, m, n, std::max(q0 - ka, 0), q1 - ka);
#pragma unroll
    for (int c = 0; c < RT; c++) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int v = 0; v < 4; v++) red[((w * RT + i) * 4 + v) * 64 + l] = acc[i][c][v];
        __syncthreads();
        // wave w finishes element w of every row tile
#pragma unroll
        for (int i = 0; i < RT; i++) {
            T sum = (T)0;
#pragma unroll
            for (int q = 0; q < 4; q++) sum += red[((q * RT + i) * 4 + w) * 64 + l];
            const int r = std::min(m0 + i * 16 + Mf<T>::row(l, w), na - 1);
            y[(long long)r * nb + n + c] = (double)sum;
        }
    }
}

// any shape with fewer than four strings of a spin: one element per lane
template <typename T>
__device__ __forceinline__ void gs_small(const GfTask &t, const T *X, double *y, int m0, int n0)
{
    const GemmFci &g = t.g;
    const int na = (int)g.na, nb = (int)g.nb;
    for (int e = threadIdx.x; e < 32 * 32; e += 256) {
        const int r = m0 + e / 32, c = n0 + e % 32;
        if (r >= na || c >= nb) continue;
        const T *Ha = hmat<T>(g, 0), *Hb = hmat<T>(g, 1);
        T sum = (T)0;
        for (int k = 0; k < na; k++) sum += Ha[(long long)r * na + k] * X[(long long)k * nb + c];
        for (int k = 0; k < nb; k++) sum += X[(long long)r * nb + k] * Hb[(long long)k * nb + c];
        y[(long long)r * nb + c] = (double)sum;
    }
}

// Same-spin parts: y_k = Haa X_k + X_k Hbb on tiles (k, alpha rows, beta columns) of the edge
// that gs_edge chooses.  128: four waves of 64 x 64 each over both reductions whole; 64 and 32:
// the four waves share the reductions of one tile, in the same four ranges, so that the two give
// the same sums to the last bit.
//
// Bound by the matrix cores (FP64 88 % busy, FP32 73 % at 1.8 GHz).  Operands straight from
// memory: a 16-deep step of a 64 x 64 tile is 16 (FP64) or 8 wide loads for 64 products, which
// the caches keep up with, and no wave waits at a barrier.  5a5b in 14 orbitals: FP64 one vector
// 720 -> 589 us, FP32 four vectors 2390 -> 1573 us against 64 x 64 tiles staged through LDS;
// 4a4b in 12 orbitals, where 64 x 64 tiles occupy a quarter of the chip, 67 -> 16 us.
template <typename T>
__device__ __forceinline__ void gf_same(const GfHeader *__restrict__ H, const GfTask *__restrict__ tasks,
                                        int block, int blocks)
{
    extern __shared__ __align__(16) unsigned char gf_smem[];
    T *red = (T *)gf_smem;                         // 4 x 4 x 4 x 64
    const int n = H->n;
    const long long total = H->total[GF_SS];
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (long long u = block; u < total; u += blocks) {
        const GfTask &t = tasks[find_task(tasks, n, u, GF_SS)];
        const GemmFci &g = t.g;
        const int na = (int)g.na, nb = (int)g.nb, edge = gs_edge(g.na, g.nb, t.K);
        const int tn = (nb + edge - 1) / edge, tm = (na + edge - 1) / edge;
        const int loc = (int)(u - t.base[GF_SS]), k = loc / (tm * tn), rem = loc - k * tm * tn;
        const int m0 = rem / tn * edge, n0 = rem % tn * edge;
        const T *X = xin<T>(t, k);
        double *y = t.y + (long long)k * t.ldy;
        if (na < 4 || nb < 4) {
            gs_small<T>(t, X, y, m0, n0);
        } else if (edge == 32) {
            gs_split<T, 2>(t, X, y, m0, n0, red);
        } else if (edge == 64) {
            gs_split<T, 4>(t, X, y, m0, n0, red);
        } else {
            typename Mf<T>::acc acc[4][4];
            int m[4];
            const int mw = m0 + (w >> 1) * 64;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                m[i] = std::min(mw + i * 16 + (l & 15), na - 1);
#pragma unroll
                for (int c = 0; c < 4; c++) acc[i][c] = Mf<T>::zero();
            }
            const int c0 = std::min(n0 + (w & 1) * 64 + 4 * (l & 15), nb - 4);
            gs_wave<T, 4>(acc, hmat<T>(g, 0), na, X, nb, na, m, c0, 0, (na + 15) / 16);
            gs_wave<T, 4>(acc, X, nb, hmat<T>(g, 1), nb, nb, m, c0, 0, (nb + 15) / 16);
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int r = std::min(mw + i * 16 + Mf<T>::row(l, v), na - 1);
                    const auto o = gptr_w(y + (long long)r * nb + c0);
#pragma unroll
                    for (int c = 0; c < 4; c += 2)
                        *(__attribute__((address_space(1))) GsOut *)(o + c) =
                            (GsOut){(double)acc[i][c][v], (double)acc[i][c + 1][v]};
                }
        }
    }
}

// ---- opposite-spin products -------------------------------------------------------------------
template <typename T> struct GeL;
template <> struct GeL<double> {
    // row padding, elements of a 16-byte read; waves per SIMD (work-groups per CU), their LDS
    static constexpr int PAD = 2, VK = 2, WPE = 1, LDS = 160 << 10;
    typedef double vec __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ double sgn(double v, uint32_t e)
    {
        return __hiloint2double(__double2hiint(v) ^ (int)(e & 0x80000000u), __double2loint(v));
    }
};
template <> struct GeL<float> {
    static constexpr int PAD = 4, VK = 4, WPE = 2, LDS = 80 << 10;
    typedef float vec __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ float sgn(float v, uint32_t e)
    {
        return __int_as_float(__float_as_int(v) ^ (int)(e & 0x80000000u));
    }
};

// element i past a uniform pointer, by a 32-bit offset per lane
template <typename T>
__device__ __forceinline__ void gf_put(__attribute__((address_space(1))) T *p, uint32_t i, T v)
{
    *(__attribute__((address_space(1))) T *)((__attribute__((address_space(1))) char *)p + i * (uint32_t)sizeof(T)) = v;
}

typedef uint32_t GfQuad __attribute__((ext_vector_type(4)));

// f(integral constant i) for i = A .. B - 1, written out
template <int A, int B, typename F> __device__ __forceinline__ void gf_each(F f)
{
    if constexpr (A < B) {
        f(std::integral_constant<int, A>{});
        gf_each<A + 1, B>(f);
    }
}

// E rows of alpha string Ja, vector k, column tiles tile0 .. tile1 - 1, by one wave: the (P|Q)
// fragments of its RT row tiles stay in registers, the D tile of 16 columns is in the wave's
// own part of LDS.  D sits column-major and the reduction index is permuted: step ks, lane
// group l / 16 takes Q = (l / 16) * KS + ks, so that a lane's B values of consecutive steps
// come in one 16-byte read.  A lane scatters a quarter of one column's list (4 entries per
// 16 bytes).
//
// A matrix product occupies the matrix core for 64 (FP64) or 32 cycles, in which the wave may
// issue other work: everything else a tile needs is cut into single operations that are dealt
// out between the products, in this order: the list of the tile after next (F), the clearing of
// the next tile's D (Z, the other of two buffers), the stores of the previous tile's results
// (S), the reads of the next tile's values (G) and their scatter (P).  Rows and columns past the
// end repeat the last one, results and all, so that nothing needs a mask; a span's first tile
// stores zeros where its results follow.
template <typename T, int KS, int RT, bool EX, bool ST>
__device__ __forceinline__ void gE_span(const GfTask &t, long long r, int Ja, int tile0, int tile1,
                                        int xo, const T *xg, int dofs)
{
    constexpr int KC = 4 * KS, LDC = KC + GeL<T>::PAD, VK = GeL<T>::VK, NG = KS / VK;
    constexpr int Lp = ge_pitch(KC), NL = Lp / 4, NZ = (LDC * (int)sizeof(T) + 63) / 64;
    typedef typename GeL<T>::vec V;
    typedef const __attribute__((address_space(1))) V *VP;
    typedef const __attribute__((address_space(1))) char *CP;
    typedef const __attribute__((address_space(1))) GfQuad *QP;
    // the lane and the row made opaque here: what the cases of the switch over the shapes have
    // in common would otherwise be computed ahead of it and held in registers all along
    int l = threadIdx.x & 63;
    asm volatile("" : "+v"(l));
    asm volatile("" : "+s"(r));
    asm volatile("" : "+s"(Ja));
    asm volatile("" : "+s"(tile0));
    asm volatile("" : "+s"(xo));
    asm volatile("" : "+s"(dofs));
    const int col = l & 15, part = l >> 4;
    extern __shared__ __align__(16) unsigned char gf_smem[];
    T *Dt = (T *)gf_smem + dofs;                   // two tiles of 16 columns
    const T *xs = (const T *)gf_smem + xo;         // staged row (ST; else gathered from memory)
    const GemmFci &g = t.g;
    const int La = wave_uni(g.La), nb = wave_uni((int)g.nb);
    T a[RT][KS];
#pragma unroll
    for (int i = 0; i < RT; i++) {
        const int p = std::min(i * 16 + col, La - 1 - (int)EX);
        const int P = (int)((gptr(g.la)[(long long)Ja * La + p] >> 16) & 0xFFu);
        const auto row = gptr(P == GF_PDIAG ? drows<T>(g) + (long long)Ja * KC : mpad<T>(g) + P * KC) + part * KS;
#pragma unroll
        for (int s = 0; s < NG; s++) {
            const V v = *(VP)(row + s * VK);
#pragma unroll
            for (int q = 0; q < VK; q++) a[i][s * VK + q] = v[q];
        }
    }
    T ar[EX ? KS : 1];                             // the row past the last tile, at this lane's steps
    if (EX) {
        const auto row = gptr(drows<T>(g) + (long long)Ja * KC) + part * KS;
#pragma unroll
        for (int s = 0; s < NG; s++) {
            const V v = *(VP)(row + s * VK);
#pragma unroll
            for (int q = 0; q < VK; q++) ar[s * VK + q] = v[q];
        }
    }
    const auto lb = gptr((const uint32_t *)wave_uni((long long)g.lb));
    const auto xr = gptr((const T *)wave_uni((long long)xg));
    const auto E = gptr_w((T *)wave_uni((long long)t.E)) + r * La * nb;
    // rows of a lane: LROW * part + VROW * v, in the last row tile up to the last one
    const uint32_t eofs = (uint32_t)(Mf<T>::LROW * part * nb);
    uint32_t elast[4];
#pragma unroll
    for (int v = 0; v < 4; v++)
        elast[v] = (uint32_t)(std::min((RT - 1) * 16 + Mf<T>::LROW * part + Mf<T>::VROW * v, La - 1 - (int)EX) * nb);
    uint32_t e[NL], en[NL];
    T v[NL];
    typename Mf<T>::acc acc[RT], res[RT];
    T d, dres = (T)0;                              // the extra row: a dot product per column
    uint32_t cres = 0;                             // column of res
    auto fetch = [&](int tile, int i) __attribute__((always_inline)) {
        const uint32_t o = ((uint32_t)std::min(tile * 16 + col, nb - 1) * Lp + (uint32_t)part * 4) * 4;
        const GfQuad q = *(QP)((CP)lb + o + i * 64);
#pragma unroll
        for (int j = 0; j < 4; j++) en[4 * i + j] = q[j];
    };
    auto clear = [&](T *D, int z) __attribute__((always_inline)) {
        const V zv = {};
        if (z * 64 + 64 <= LDC * (int)sizeof(T) || z * 64 + l < LDC * (int)sizeof(T)) ((V *)D)[z * 64 + l] = zv;
    };
    auto get = [&](int j) __attribute__((always_inline)) { v[j] = ST ? xs[e[j] & 0xFFFFu] : xr[e[j] & 0xFFFFu]; };
    auto put = [&](T *Dc, int j) __attribute__((always_inline)) {
        Dc[(e[j] >> 16) & 0xFFu] = GeL<T>::sgn(v[j], e[j]);
    };
    auto store = [&](int i, int q) __attribute__((always_inline)) {
        if (i + 1 < RT) gf_put(E + (i * 16 + Mf<T>::VROW * q) * nb, eofs + cres, res[i][q]);
        else gf_put(E, elast[q] + cres, res[i][q]);
    };
    // operation m of the M that go with a tile's products (order above)
    constexpr int GL = NL / 2, M = NL / 4 + NZ + 4 * RT + 2 * NL, NM = KS * RT;
    auto op = [&](auto mc, T *D, int tile) __attribute__((always_inline)) {
        constexpr int m = decltype(mc)::value, z = m - NL / 4, st = z - NZ, f = st - 4 * RT;
        T *Dc = D + col * LDC;
        if constexpr (z < 0) fetch(std::min(tile + 2, tile1 - 1), m);
        else if constexpr (st < 0) clear(D, z);
        else if constexpr (f < 0) store(st >> 2, st & 3);
        // half the reads, then a write and a read in turn, then the other writes
        else if constexpr (f < GL) get(f);
        else if constexpr (f >= GL + NL) put(Dc, f - NL);
        else if constexpr ((f - GL) & 1) get(GL + (f - GL) / 2);
        else put(Dc, (f - GL) / 2);
    };
#pragma unroll
    for (int i = 0; i < NL / 4; i++) fetch(tile0, i);
#pragma unroll
    for (int i = 0; i < NZ; i++) clear(Dt, i);
#pragma unroll
    for (int i = 0; i < NL; i++) e[i] = en[i];
#pragma unroll
    for (int i = 0; i < NL / 4; i++) fetch(std::min(tile0 + 1, tile1 - 1), i);
#pragma unroll
    for (int j = 0; j < NL; j++) get(j);
    wave_sync();
#pragma unroll
    for (int j = 0; j < NL; j++) put(Dt + col * LDC, j);
#pragma unroll
    for (int i = 0; i < RT; i++) res[i] = Mf<T>::zero();
    cres = (uint32_t)std::min(tile0 * 16 + col, nb - 1);
    int cur = 0;
    for (int tile = tile0; tile < tile1; tile++) {
        wave_sync();
        const T *b0 = Dt + cur + col * LDC + part * KS;
        T *Dn = Dt + (16 * LDC - cur);
#pragma unroll
        for (int i = 0; i < NL; i++) e[i] = en[i];
#pragma unroll
        for (int i = 0; i < RT; i++) acc[i] = Mf<T>::zero();
        d = (T)0;
        V b[2];
        b[0] = *(const V *)b0;
        gf_each<0, NM>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value, i = k % RT, st = k / RT, s = st / VK, q = st % VK;
            if constexpr (k % (RT * VK) == 0 && s + 1 < NG) b[(s + 1) & 1] = *(const V *)(b0 + (s + 1) * VK);
            acc[i] = Mf<T>::mma(a[i][st], b[s & 1][q], acc[i]);
            gf_each<(k * M + NM - 1) / NM, ((k + 1) * M + NM - 1) / NM>(
                [&](auto mc) __attribute__((always_inline)) { op(mc, Dn, tile); });
            if constexpr (EX && i == RT - 1) d += b[s & 1][q] * ar[st];
            __builtin_amdgcn_sched_barrier(0);
        });
        if (EX) {
            // the previous tile's extra row, and this one's sum over the four lane groups
            gf_put(E + (La - 1) * nb, cres, dres);
            d += __shfl_xor(d, 16);
            dres = d + __shfl_xor(d, 32);
        }
        cres = (uint32_t)std::min(tile * 16 + col, nb - 1);
#pragma unroll
        for (int i = 0; i < RT; i++) res[i] = acc[i];
        cur = 16 * LDC - cur;
    }
    if (EX) gf_put(E + (La - 1) * nb, cres, dres);
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) store(i, q);
}

// The depths KS, row tiles and extra rows that alpha lists of n <= 15 orbitals have
// (La = a (n - a) + 1 rows, KS = MP / 4); only n = 15 has rows too long to stage.
template <typename T>
__device__ __forceinline__ void gE_shape(const GfTask &t, long long r, int Ja, bool ex, int tile0,
                                         int tile1, int xo, const T *xg, int dofs)
{
    static_assert(GF_MAXMP == 128, "reduction depths below cover MP <= 128");
#define GE_CASE(KS, RT, EX) \
    case (KS) * 16 + (RT) * 2 + (EX): \
        gE_span<T, KS, RT, EX, true>(t, r, Ja, tile0, tile1, xo, xg, dofs); break
#define GE_CASE2(KS, RT) \
    case (KS) * 16 + (RT) * 2: \
        if (xo >= 0) gE_span<T, KS, RT, false, true>(t, r, Ja, tile0, tile1, xo, xg, dofs); \
        else gE_span<T, KS, RT, false, false>(t, r, Ja, tile0, tile1, xo, xg, dofs); \
        break
    switch (t.g.MP / 4 * 16 + (t.g.La - ex + 15) / 16 * 2 + ex) {
    GE_CASE(4, 1, 0);                                                      // n <= 5
    GE_CASE(8, 1, 0);                                                      // 6, 7
    GE_CASE(12, 1, 0); GE_CASE(12, 1, 1); GE_CASE(12, 2, 0);               // 8, 9
    GE_CASE(16, 1, 0); GE_CASE(16, 1, 1); GE_CASE(16, 2, 0);               // 10
    GE_CASE(20, 1, 0); GE_CASE(20, 2, 0); GE_CASE(20, 2, 1); GE_CASE(20, 3, 0);   // 11, 12
    GE_CASE(24, 1, 0); GE_CASE(24, 2, 0); GE_CASE(24, 3, 0);               // 13
    GE_CASE(28, 1, 0); GE_CASE(28, 2, 0); GE_CASE(28, 3, 0); GE_CASE(28, 3, 1); GE_CASE(28, 4, 0);   // 14
    GE_CASE2(32, 1); GE_CASE2(32, 2); GE_CASE2(32, 3); GE_CASE2(32, 4);    // 15
    }
#undef GE_CASE
#undef GE_CASE2
}

// E[p][c] = sum_Q (P_p|Q) D[Q][c] over columns c = (k, Ja, Ib), for the La rows p of the
// alpha string Ja (P_p = pair of entry p of Ja's alpha list).  Every wave works on its own 16
// columns of one row (k, Ja) and all of that string's row tiles, without barriers.  A row past
// the last full tile (a (n - a) a multiple of 16) is a dot product on the vector units instead
// of a tile.  The vector's rows that a work-group needs next are staged in LDS for the list
// gathers (as many as fit beside the D tiles; longer rows are gathered from memory).  A unit
// is `bn` columns of one row; work-groups take equal consecutive ranges of units.
//
// Bound by the matrix cores (70 % busy at the clock the power limit leaves, about 2 GHz).  FP64
// keeps one wave per SIMD: two D tiles a wave fill the LDS, and the fragments of four row tiles
// take half the registers.  5a5b in 14 orbitals: FP64 one vector 1362 -> 936 us, FP32 four
// vectors 3232 -> 1884 us against a work-group per tile with three barriers and a row tile per
// wave (the fourth wave idle at 46 rows); waves by themselves, two per SIMD and one D tile each,
// reached 1017 and 2220 us, two D tiles without the dealt-out order 1083 and 2151 us.  4a4b in
// 12 orbitals (33 rows): 81 -> 45 us, and the whole product 70 -> 67 with the 33rd row of (P|Q)
// in registers instead of LDS.
template <typename T>
__device__ __forceinline__ void gf_opposite(const GfHeader *__restrict__ H,
                                            const GfTask *__restrict__ tasks, int bn, int block,
                                            int blocks)
{
    extern __shared__ __align__(16) unsigned char gf_smem[];
    const int tid = threadIdx.x, S = bn >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = H->n;
    const long long total = H->total[GF_E];
    const long long u0 = total * block / blocks, u1 = total * (block + 1) / blocks;
    for (long long u = u0; u < u1;) {
        const int ti = find_task(tasks, n, u, GF_E);
        const GfTask &t = tasks[ti];
        const GemmFci &g = t.g;
        const bool ex = ge_extra(g.La);
        const int nct = (int)(g.nb + 15) / 16, per = (nct + S - 1) / S;
        const long long base = t.base[GF_E];
        const long long r0 = (u - base) / per;
        const int dw = 32 * (g.MP + GeL<T>::PAD);                 // one wave's D tiles
        T *xs = (T *)gf_smem + 4 * dw;
        const int room = (GeL<T>::LDS / (int)sizeof(T) - 4 * dw) / (int)g.nb;
        long long end = std::min(u1, ti + 1 < n ? tasks[ti + 1].base[GF_E] : total);
        if (room > 0) end = std::min(end, base + (r0 + room) * per);
        __syncthreads();   // the rows and tiles of the previous stage are read
        if (room > 0) {
            for (long long r = r0; r <= (end - 1 - base) / per; r++) {
                const long long k = r / g.na;
                const auto xr = gptr(xin<T>(t, (int)k) + (r - k * g.na) * g.nb);
                for (int i = tid; i < g.nb; i += 256) xs[(r - r0) * g.nb + i] = xr[i];
            }
            __syncthreads();
        }
        const long long w1 = u + ((end - u) * (w + 1) >> 2);
        for (long long q = u + ((end - u) * w >> 2); q < w1;) {
            const long long r = wave_uni((q - base) / per);
            const int k = wave_uni((int)(r / g.na)), Ja = wave_uni((int)(r - k * g.na));
            const int un = (int)(q - base - r * per), m = (int)std::min<long long>(w1 - q, per - un);
            const int xo = wave_uni(room > 0 ? 4 * dw + (int)(r - r0) * (int)g.nb : -1);
            const T *xg = xin<T>(t, k) + Ja * g.nb;
            const int t0 = wave_uni(un * S), t1 = wave_uni(std::min(nct, (un + m) * S)), dofs = wave_uni(w * dw);
            gE_shape<T>(t, r, Ja, ex, t0, t1, xo, xg, dofs);
            q += m;
        }
        u = end;
    }
}

// Both parts in one launch, the first `eblocks` work-groups on the opposite-spin products: they
// are independent of each other, and the one's last work-groups run beside the other's first.
// Small spaces, of which either part leaves most of the chip idle, take the time of the longer
// one and a launch less: 3a3b in 8 orbitals FP64 15.0 -> 10.3 us; 1 % or less from 4a4b in 12
// orbitals on.
template <typename T>
__global__ __launch_bounds__(256, GeL<T>::WPE) void k_gprod(const GfHeader *__restrict__ H,
                                                            const GfTask *__restrict__ tasks, int bn,
                                                            int eblocks)
{
    if ((int)blockIdx.x < eblocks) gf_opposite<T>(H, tasks, bn, blockIdx.x, eblocks);
    else gf_same<T>(H, tasks, blockIdx.x - eblocks, gridDim.x - eblocks);
}

// y_k[Ia][Ib] += sum over the alpha list of Ia of sign * E[p][k, Ja, Ib], p the entry's E row
// (bits 24..30); 256 elements per unit
template <typename T>
__global__ __launch_bounds__(256) void k_gga(const GfHeader *__restrict__ H,
                                             const GfTask *__restrict__ tasks)
{
    const int n = H->n;
    const long long total = H->total[GF_GA];
    for (long long u = blockIdx.x; u < total; u += gridDim.x) {
        const GfTask &t = tasks[find_task(tasks, n, u, GF_GA)];
        const GemmFci &g = t.g;
        const long long Nb = g.nb, N = g.na * g.nb, ncols = N * t.K;
        const int La = g.La;
        const long long idx = (u - t.base[GF_GA]) * 256 + threadIdx.x;
        if (idx >= ncols) continue;
        const long long k = idx / N, rem = idx - k * N;
        const long long Ia = rem / Nb, Ib = rem - Ia * Nb;
        const auto lst = gptr(g.la + Ia * La);
        const auto Ek = gptr((const T *)t.E + k * N * La + Ib);
        T acc = (T)0;
        int e = 0;
        // eight independent loads in flight per lane
        for (; e + 8 <= La; e += 8) {
            T v[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const uint32_t wd = lst[e + q];
                v[q] = Ek[(long long)((wd & 0xFFFFu) * (uint32_t)La + ((wd >> 24) & 0x7Fu)) * Nb];
            }
#pragma unroll
            for (int q = 0; q < 8; q++) acc += (lst[e + q] >> 31) ? -v[q] : v[q];
        }
        for (; e < La; e++) {
            const uint32_t wd = lst[e];
            const T v = Ek[(long long)((wd & 0xFFFFu) * (uint32_t)La + ((wd >> 24) & 0x7Fu)) * Nb];
            acc += (wd >> 31) ? -v : v;
        }
        t.y[k * t.ldy + rem] += (double)acc;
    }
}

// ---- launchers ------------------------------------------------------------------------------
int jk_gf_dense(long long nstr, const uint64_t *mask, const long long *off1, const int2 *e1,
                const double *v1, const long long *off2, const int2 *e2, const double *v2,
                const double *m1, const double *m2, double *H, hipStream_t st)
{
    if (hipMemsetAsync(H, 0, sizeof(double) * (size_t)nstr * nstr, st) != hipSuccess) {
        jci_set_error("gf_dense: memset failed");
        return -2;
    }
    hipLaunchKernelGGL(k_gf_dense, dim3((unsigned)((nstr + 127) / 128)), dim3(128), 0, st, nstr,
                       mask, off1, e1, v1, off2, e2, v2, m1, m2, H);
    GF_CHECK();
    return 0;
}

int jk_gf_lists(long long nstr, const uint64_t *mask, const long long *off1, const int2 *e1,
                int L, int Lp, int pad, int diag_one, uint32_t *out, hipStream_t st)
{
    hipLaunchKernelGGL(k_gf_lists, dim3((unsigned)((nstr + 127) / 128)), dim3(128), 0, st, nstr,
                       mask, off1, e1, L, Lp, (uint32_t)pad, diag_one, out);
    GF_CHECK();
    return 0;
}

int jk_gf_rank(long long nstr, int L, const uint32_t *in, uint32_t *out, int *missing,
               hipStream_t st)
{
    if (nstr * L == 0) return 0;
    hipLaunchKernelGGL(k_gf_rank, dim3((unsigned)((nstr * L + 255) / 256)), dim3(256), 0, st, nstr, L,
                       in, out, missing);
    GF_CHECK();
    return 0;
}

int jk_gf_m2pad(int m1, int MP, const double *m2sq, double *o64, float *o32, hipStream_t st)
{
    hipLaunchKernelGGL(k_gf_m2pad, dim3((MP * MP + 255) / 256), dim3(256), 0, st, m1, MP, m2sq,
                       o64, o32);
    GF_CHECK();
    return 0;
}

int jk_gf_diagrows(long long nstr, int MP, const uint64_t *mask, const double *M64, double *o64,
                   float *o32, hipStream_t st)
{
    if (nstr * MP == 0) return 0;
    hipLaunchKernelGGL(k_gf_diagrows, dim3((unsigned)((nstr * MP + 255) / 256)), dim3(256), 0, st,
                       nstr, MP, mask, M64, o64, o32);
    GF_CHECK();
    return 0;
}

int jk_gf_bn_valid(int prec, int bn)
{
    return prec == 64 ? (bn == 16 || bn == 32) : (bn == 32 || bn == 64);
}

void jk_gf_units(int prec, int bn, const GfTask &t, long long units[4])
{
    const long long na = t.g.na, nb = t.g.nb, N = na * nb, cols = N * t.K;
    units[GF_CV] = prec == 64 ? 0 : (cols + 255) / 256;
    const int edge = gs_edge(na, nb, t.K);
    units[GF_SS] = (long long)t.K * ((na + edge - 1) / edge) * ((nb + edge - 1) / edge);
    units[GF_E] = t.g.La ? (long long)t.K * na * ((nb + bn - 1) / bn) : 0;
    units[GF_GA] = (cols + 255) / 256;
}

// persistent grid caps of the grid-stride kernels (conversion, gather)
static const long long gf_cap[4] = {4096, 0, 0, 4096};

static long long device_cus()
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 256;
    return cus;
}

template <typename T>
static int gf_group_t(int bn, const GfHeader *d_hdr, const GfTask *d_tasks, const GfHeader *hh,
                      hipStream_t st)
{
    // Opposite-spin units go in equal consecutive ranges, one per work-group, same-spin tiles one
    // after another: each part as many work-groups as the device holds
    static const long long cap_p = device_cus() * GeL<T>::WPE;
    const long long cap[4] = {gf_cap[GF_CV], cap_p, cap_p, gf_cap[GF_GA]};
    unsigned g[4];
    for (int i = 0; i < 4; i++) {
        // an opposite-spin unit is one wave's, four to a work-group
        const long long units = !hh ? cap[i] : i == GF_E ? (hh->total[i] + 3) / 4 : hh->total[i];
        g[i] = (unsigned)std::max<long long>(1, std::min(units, cap[i]));
    }
    if (sizeof(T) == 4) {
        hipLaunchKernelGGL(k_gcv, dim3(g[GF_CV]), dim3(256), 0, st, d_hdr, d_tasks);
        GF_CHECK();
    }
    hipLaunchKernelGGL(k_gprod<T>, dim3(g[GF_E] + g[GF_SS]), dim3(256), GeL<T>::LDS, st, d_hdr, d_tasks,
                       bn, (int)g[GF_E]);
    GF_CHECK();
    hipLaunchKernelGGL(k_gga<T>, dim3(g[GF_GA]), dim3(256), 0, st, d_hdr, d_tasks);
    GF_CHECK();
    return 0;
}

int jk_gf_group(int prec, int bn, const GfHeader *d_hdr, const GfTask *d_tasks,
                const GfHeader *hdr_host, hipStream_t st)
{
    if (!jk_gf_bn_valid(prec, bn)) {
        jci_set_error("gf_sigma: E tile width %d not available for FP%d", bn, prec);
        return -1;
    }
    if (prec == 64) return gf_group_t<double>(bn, d_hdr, d_tasks, hdr_host, st);
    return gf_group_t<float>(bn, d_hdr, d_tasks, hdr_host, st);
}
