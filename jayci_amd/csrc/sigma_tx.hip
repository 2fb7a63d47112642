// Contraction form of the truncated-space sigma on MFMA (see sigma_tx.h).
#include <hip/hip_runtime.h>
#include <algorithm>
#include "mfma.h"
#include "sigma_tx.h"

#define TX_CHECK()                                                       \
    do {                                                                 \
        hipError_t e_ = hipGetLastError();                               \
        if (e_ != hipSuccess) {                                          \
            jci_set_error("%s:%d launch: %s", __FILE__, __LINE__,        \
                          hipGetErrorString(e_));                        \
            return -2;                                                   \
        }                                                                \
    } while (0)

// ---- set-up ------------------------------------------------------------------------------------

// first-spin lists and reverse ranks of one spin, one thread per string
__global__ void k_tx_lists(const SpaceDesc *__restrict__ d, int spin, long long nstr,
                           const uint64_t *__restrict__ M, const long long *__restrict__ off1,
                           const int2 *__restrict__ e1, const int *__restrict__ goff1,
                           const TxList *__restrict__ lists, uint32_t *__restrict__ lst,
                           uint16_t *__restrict__ rk)
{
    const long long I = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (I >= nstr) return;
    const SpinDesc &S = d->s[spin];
    int g = 0;
    while (g + 1 < S.ngrp && S.gstart[g + 1] <= I) g++;
    const TxList &t = lists[g];
    const long long loc = I - S.gstart[g];
    const long long iI = loc / t.nsv, w = loc % t.nsv;
    const uint64_t m = M[I], ext = m & d->vmask;
    uint32_t *out = lst + t.base + w * t.rows * t.nIp + iI;
    for (int s = 0; s < t.nsec; s++) {
        const int h = t.grp[s];
        if (h < 0) {
            int r = t.row0[s];
            for (uint64_t x = m; x; x &= x - 1, r++) {
                const int k = jci_ctz(x);
                out[(long long)r * t.nIp] = (uint32_t)loc | ((uint32_t)tx_kpos(d, ext, 0, k, k) << TX_JBITS);
            }
            continue;
        }
        const int dv = S.gv[h] == S.gv[g] ? 0 : S.gv[h] < S.gv[g] ? -1 : 1;
        const long long e0 = off1[I] + goff1[I * (S.ngrp + 1) + h];
        const int n = goff1[I * (S.ngrp + 1) + h + 1] - goff1[I * (S.ngrp + 1) + h];
        for (int k = 0; k < n && k < t.cnt[s]; k++) {
            const int2 en = e1[e0 + k];
            const int i = en.y & 63, f = (en.y >> 6) & 63;
            out[(long long)(t.row0[s] + k) * t.nIp] =
                (uint32_t)(en.x - S.gstart[h]) |
                ((uint32_t)tx_kpos(d, ext, dv, i, f) << TX_JBITS) |
                ((uint32_t)((en.y >> 12) & 1) << 31);
            rk[e0 + k] = (uint16_t)tx_single_rank(d, m ^ (1ULL << i) ^ (1ULL << f), f, i);
        }
    }
}

__global__ void k_tx_fill(long long n, uint32_t *__restrict__ p)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = TX_PAD;
}

int jk_tx_lists(const SpaceDesc *d, int spin, long long nstr, const uint64_t *mask,
                const long long *off1, const int2 *e1, const int *goff1, const TxList *lists,
                uint32_t *lst, uint16_t *rk, hipStream_t st)
{
    hipLaunchKernelGGL(k_tx_lists, dim3((unsigned)((nstr + 63) / 64)), dim3(64), 0, st, d, spin, nstr,
                       mask, off1, e1, goff1, lists, lst, rk);
    TX_CHECK();
    return 0;
}

int jk_tx_fill(long long n, uint32_t *p, hipStream_t st)
{
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_tx_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, p);
    TX_CHECK();
    return 0;
}

// the pairs of every string: its own list, and its entries in the lists of the N - 2 electron
// strings they leave; one thread per string
__global__ void k_tx_pairs(const SpaceDesc *__restrict__ d, int spin, long long nstr,
                           const uint64_t *__restrict__ M,
                           const unsigned long long *__restrict__ binom,
                           const TxPairGroup *__restrict__ pg, int npg, int npair,
                           int2 *__restrict__ kl, int2 *__restrict__ gl)
{
    const long long I = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (I >= nstr) return;
    const SpinDesc &S = d->s[spin];
    int g = 0;
    while (g + 1 < S.ngrp && S.gstart[g + 1] <= I) g++;
    const int e[3] = {S.gd[g], S.ga[g], S.gv[g]};
    const uint64_t m = M[I];
    int at = 0;
    for (int s0 = 0; s0 < 3; s0++)
        for (int s1 = s0; s1 < 3; s1++) {
            const int n = s0 == s1 ? e[s0] * (e[s0] - 1) / 2 : e[s0] * e[s1];
            if (n <= 0) continue;
            int o[3] = {e[0], e[1], e[2]};
            o[s0]--;
            o[s1]--;
            int q = 0;
            while (q < npg && !(pg[q].d == o[0] && pg[q].a == o[1] && pg[q].v == o[2])) q++;
            if (q == npg) return;
            const int ty = tx_type(s0, s1);
            for (uint64_t x = m & tx_submask(d, s0); x; x &= x - 1) {
                const int i = jci_ctz(x);
                for (uint64_t y = m & tx_submask(d, s1) & ~tx_below(i) & ~(1ULL << i); y; y &= y - 1) {
                    const int j = jci_ctz(y);
                    uint64_t k2;
                    int type, idx, neg;
                    tx_pair(d, m, i, j, &k2, &type, &idx, &neg);
                    const long long K = tx_pair_rank(d, k2, binom);
                    gl[I * npair + at++] = make_int2((int)K, idx | (int)((unsigned)neg << 31));
                    kl[pg[q].base + K * pg[q].R + pg[q].off[ty] + idx] =
                        make_int2((int)(I - S.gstart[g]),
                                  (j * (j - 1) / 2 + i) | (int)((unsigned)neg << 31));
                }
            }
        }
}

int jk_tx_pairs(const SpaceDesc *d, int spin, long long nstr, const uint64_t *mask,
                const unsigned long long *binom, const TxPairGroup *pg, int npg, int npair,
                int2 *kl, int2 *gl, hipStream_t st)
{
    hipLaunchKernelGGL(k_tx_pairs, dim3((unsigned)((nstr + 63) / 64)), dim3(64), 0, st, d, spin, nstr,
                       mask, binom, pg, npg, npair, kl, gl);
    TX_CHECK();
    return 0;
}

__device__ __forceinline__ void pair_of(int P, int *i, int *j)
{
    int b = (int)((1.0 + sqrt(1.0 + 8.0 * P)) * 0.5);
    while (b * (b - 1) / 2 > P) b--;
    while ((b + 1) * b / 2 <= P) b++;
    *j = b;
    *i = P - b * (b - 1) / 2;
}

__global__ void k_tx_w(int np, double sc, const double *__restrict__ m1,
                       const double *__restrict__ m2, double *__restrict__ w64,
                       float *__restrict__ w32)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)np * np) return;
    int i, j, k, l;
    pair_of((int)(t / np), &i, &j);
    pair_of((int)(t % np), &k, &l);
    double v = jci_eri(m2, i, k, j, l) - jci_eri(m2, i, l, j, k);
    double h = 0.0;
    if (j == l) h += jci_h1(m1, i, k);
    if (i == l) h -= jci_h1(m1, j, k);
    if (j == k) h -= jci_h1(m1, i, l);
    if (i == k) h += jci_h1(m1, j, l);
    v += h * sc;
    w64[t] = v;
    w32[t] = (float)v;
}

int jk_tx_w(int norb, int nelec, const double *m1, const double *m2, double *w64, float *w32,
            hipStream_t st)
{
    const int np = norb * (norb - 1) / 2;
    hipLaunchKernelGGL(k_tx_w, dim3((unsigned)(((long long)np * np + 255) / 256)), dim3(256), 0, st, np,
                       1.0 / (nelec - 1), m1, m2, w64, w32);
    TX_CHECK();
    return 0;
}

// integral rows (TxSpin::m64)
struct TxParts {
    int iI0[JCI_MAXG], nsv[JCI_MAXG];
    int ngrp;
};
__global__ void k_tx_rows(const SpaceDesc *__restrict__ d, int spin, TxParts p, int nparts,
                          const uint64_t *__restrict__ M, int m1, const double *__restrict__ m2sq,
                          double *__restrict__ m64, float *__restrict__ m32)
{
    const int ms = m1 + 1;
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)(m1 + nparts + 1) * ms) return;
    const int r = (int)(t / ms), Q = (int)(t % ms);
    double s = 0.0;
    if (Q < m1 && r < m1) {
        s = m2sq[(long long)r * m1 + Q];
    } else if (Q < m1 && r < m1 + nparts) {
        const int part = r - m1;
        int g = 0;
        while (g + 1 < p.ngrp && p.iI0[g + 1] <= part) g++;
        const uint64_t m = M[d->s[spin].gstart[g] + (long long)(part - p.iI0[g]) * p.nsv[g]];
        for (uint64_t x = m & ~d->vmask; x; x &= x - 1) {
            const int k = jci_ctz(x);
            s += m2sq[jci_tri(k, k) * m1 + Q];
        }
    }
    m64[t] = s;
    m32[t] = (float)s;
}

int jk_tx_rows(const SpaceDesc *d, const SpaceDesc &h, int spin, const uint64_t *mask, int m1,
               const double *m2sq, const TxPlan &P, double *m64, float *m32, hipStream_t st)
{
    TxParts p;
    p.ngrp = h.s[spin].ngrp;
    for (int g = 0; g < p.ngrp; g++) {
        p.iI0[g] = P.iI0[spin][g];
        p.nsv[g] = P.lists[spin][g].nsv;
    }
    const long long n = (long long)(m1 + P.nint_parts[spin] + 1) * (m1 + 1);
    hipLaunchKernelGGL(k_tx_rows, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, d, spin, p,
                       (int)P.nint_parts[spin], mask, m1, m2sq, m64, m32);
    TX_CHECK();
    return 0;
}

// ---- vectors in and out ------------------------------------------------------------------------

__device__ __forceinline__ int tx_block(const long long *__restrict__ off, int n, long long t)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= t) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// 16 x 16 element tiles of the blocks (tt: first tile of each block): the vector in the
// arithmetic type (xv, may be null) and its block-transposed copy.  Bound by memory: one read
// and one or two writes of the vector.
template <typename T>
__global__ __launch_bounds__(256) void k_tx_in(long long N, const SpaceDesc *__restrict__ d,
                                               const long long *__restrict__ tt,
                                               const double *__restrict__ x, long long xs,
                                               long long xk, T *__restrict__ xv, T *__restrict__ xT)
{
    __shared__ T t[16][17];
    const int b = tx_block(tt, d->nblk, blockIdx.x);
    const long long na = d->s[0].gn[d->bp[b]], nb = d->s[1].gn[d->bq[b]];
    const long long ntc = (nb + 15) / 16, rel = blockIdx.x - tt[b];
    const long long r0 = rel / ntc * 16, c0 = rel % ntc * 16, off = d->boff[b];
    const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
    const long long k = blockIdx.y;
    if (r0 + ty < na && c0 + tx < nb) {
        const long long n = off + (r0 + ty) * nb + c0 + tx;
        const T v = (T)x[n * xs + k * xk];
        t[ty][tx] = v;
        if (xv) xv[k * N + n] = v;
    }
    __syncthreads();
    if (c0 + ty < nb && r0 + tx < na) xT[k * N + off + (c0 + ty) * na + r0 + tx] = t[tx][ty];
}

__global__ __launch_bounds__(256) void k_tx_out(long long N, const SpaceDesc *__restrict__ d,
                                                const long long *__restrict__ tt,
                                                const double *__restrict__ yT,
                                                double *__restrict__ y, long long ys, long long yk)
{
    __shared__ double t[16][17];
    const int b = tx_block(tt, d->nblk, blockIdx.x);
    const long long na = d->s[0].gn[d->bp[b]], nb = d->s[1].gn[d->bq[b]];
    const long long ntc = (nb + 15) / 16, rel = blockIdx.x - tt[b];
    const long long r0 = rel / ntc * 16, c0 = rel % ntc * 16, off = d->boff[b];
    const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
    const long long k = blockIdx.y;
    if (c0 + ty < nb && r0 + tx < na) t[ty][tx] = yT[k * N + off + (c0 + ty) * na + r0 + tx];
    __syncthreads();
    if (r0 + ty < na && c0 + tx < nb) {
        const long long n = off + (r0 + ty) * nb + c0 + tx;
        y[n * ys + k * yk] += t[tx][ty];
    }
}

int jk_tx_in(int prec, int nvec, long long N, const SpaceDesc *d, const long long *tt, long long ntt,
             const double *x, long long xs, long long xk, void *xv, void *xT, hipStream_t st)
{
    const dim3 g((unsigned)ntt, (unsigned)nvec);
    if (prec == 64)
        hipLaunchKernelGGL(k_tx_in<double>, g, dim3(256), 0, st, N, d, tt, x, xs, xk, (double *)xv,
                           (double *)xT);
    else
        hipLaunchKernelGGL(k_tx_in<float>, g, dim3(256), 0, st, N, d, tt, x, xs, xk, (float *)xv,
                           (float *)xT);
    TX_CHECK();
    return 0;
}

int jk_tx_out(int nvec, long long N, const SpaceDesc *d, const long long *tt, long long ntt,
              const double *yT, double *y, long long ys, long long yk, hipStream_t st)
{
    hipLaunchKernelGGL(k_tx_out, dim3((unsigned)ntt, (unsigned)nvec), dim3(256), 0, st, N, d, tt, yT, y,
                       ys, yk);
    TX_CHECK();
    return 0;
}

// ---- same-spin part ----------------------------------------------------------------------------

template <typename T> __device__ __forceinline__ const T *tx_w(const TxSpin &s);
template <> __device__ __forceinline__ const double *tx_w<double>(const TxSpin &s) { return s.w64; }
template <> __device__ __forceinline__ const float *tx_w<float>(const TxSpin &s) { return s.w32; }

// E[p][K2, c] on 64 x 64 tiles (64 pairs of one N - 2 electron string, 64 columns): a wave owns
// 16 columns and all four row tiles, its B operand comes straight from the vector (rows of 16
// consecutive elements), the W tile is staged in LDS one 16-deep step ahead.
template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_tx_ess(TxDev A, TxRound R, const T *__restrict__ x0,
                                                long long ldx0, const T *__restrict__ x1,
                                                long long ldx1, T *__restrict__ E)
{
    extern __shared__ __align__(16) unsigned char tx_smem[];
    __shared__ T As[2][16][65];
    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6;
    int lo = 0, hi = R.ni - 1;
    const TxPairItem *__restrict__ items = A.pitem + R.i0;
    const long long u = blockIdx.x;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (items[mid].item0 <= u) lo = mid; else hi = mid - 1;
    }
    const TxPairItem &it = items[lo];
    const TxPairTask &t = A.ptask[it.task];
    const int loc = (int)(u - it.item0), rg = loc % it.rg, ct = loc / it.rg % it.ct;
    const long long K2 = loc / (it.rg * it.ct);
    const int Rr = t.R, r0 = rg * 64;
    const TxSpin &S = A.s[t.o];
    const long long k = blockIdx.y;
    const T *__restrict__ x = (t.o ? x1 + k * ldx1 : x0 + k * ldx0) + it.c0 + ct * 64;
    long long *__restrict__ off = (long long *)tx_smem;
    int *__restrict__ pr = (int *)(off + Rr);
    for (int r = tid; r < Rr; r += 256) {
        int s = 0;
        while (s + 1 < t.nsec && t.sr[s + 1] <= r) s++;
        const int2 en = S.kl[t.lbase + K2 * t.Rfull + t.so[s] + (r - t.sr[s])];
        off[r] = t.sx[s] + (long long)en.x * t.nb;
        pr[r] = en.y;
    }
    __syncthreads();
    const int np = A.np;
    const T *__restrict__ W = tx_w<T>(S);
    const int ar = tid >> 2, ak = (tid & 3) * 4;
    const bool aok = r0 + ar < Rr;
    const T *__restrict__ Wr = W + (long long)(aok ? pr[r0 + ar] & 0x7FFFFFFF : 0) * np;
    const int c = w * 16 + (l & 15), kk = l >> 4;
    const bool cok = ct * 64 + c < it.nc;
    T ra[4], rb[4];
    auto gload = [&](int k0) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int q = k0 + ak + j;
            ra[j] = aok && q < Rr ? Wr[pr[q] & 0x7FFFFFFF] : (T)0;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int q = k0 + j * 4 + kk;
            const bool ok = cok && q < Rr;
            const T v = ok ? x[off[ok ? q : 0] + c] : (T)0;
            rb[j] = ok && pr[q] < 0 ? -v : v;
        }
    };
    typename Mf<T>::acc acc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = Mf<T>::zero();
    const int nrt = (std::min(64, Rr - r0) + 15) / 16;
    gload(0);
#pragma unroll
    for (int j = 0; j < 4; j++) As[0][ak + j][ar] = ra[j];
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < Rr; k0 += 16) {
        T b[4];
#pragma unroll
        for (int j = 0; j < 4; j++) b[j] = rb[j];
        const bool more = k0 + 16 < Rr;
        if (more) gload(k0 + 16);
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (i < nrt) {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    acc[i] = Mf<T>::mma(As[buf][j * 4 + kk][i * 16 + (l & 15)], b[j], acc[i]);
            }
        if (more) {
#pragma unroll
            for (int j = 0; j < 4; j++) As[buf ^ 1][ak + j][ar] = ra[j];
        }
        __syncthreads();
        buf ^= 1;
    }
    if (ct * 64 + c < it.ncp) {
        T *__restrict__ Er = E + k * R.elems + it.ebase + K2 * Rr * it.ncp + ct * 64 + c;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = r0 + i * 16 + Mf<T>::row(l, v);
                if (r < Rr) Er[(long long)r * it.ncp] = acc[i][v];
            }
    }
}

// the same-spin sums: y(I, c) = sum over the pairs of I, one E row each (coalesced); the first
// writer of the result
template <typename T>
__global__ __launch_bounds__(256) void k_tx_gss(TxDev A, TxRound R, const T *__restrict__ E, double *y0,
                                                long long ys0, long long yk0, double *y1,
                                                long long ys1, long long yk1)
{
    int lo = 0, hi = R.no - 1;
    const TxPairOut *__restrict__ outs = A.pout + R.o0;
    const long long u = blockIdx.x;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (outs[mid].blk0 <= u) lo = mid; else hi = mid - 1;
    }
    const TxPairOut &t = outs[lo];
    const int loc = (int)(u - t.blk0), il = loc / t.cblk;
    const int c = (loc - il * t.cblk) * 256 + threadIdx.x;
    if (c >= t.nc) return;
    const TxSpin &S = A.s[t.o];
    const int2 *__restrict__ g = S.gl + (long long)(t.ls0 + il) * S.npair;
    const long long k = blockIdx.y;
    T acc = (T)0;
    for (int s = 0; s < t.nsec; s++) {
        const T *__restrict__ Es = E + k * R.elems + t.eb[s] + (long long)t.r0[s] * t.ncp + c;
        const long long st = (long long)t.R[s] * t.ncp;
        int m = 0;
        for (; m + 4 <= t.np[s]; m += 4) {
            T v[4];
            int2 e[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                e[j] = g[m + j];
                v[j] = Es[(long long)e[j].x * st + (long long)(e[j].y & 0x7FFFFFFF) * t.ncp];
            }
#pragma unroll
            for (int j = 0; j < 4; j++) acc += e[j].y < 0 ? -v[j] : v[j];
        }
        for (; m < t.np[s]; m++) {
            const int2 e = g[m];
            const T v = Es[(long long)e.x * st + (long long)(e.y & 0x7FFFFFFF) * t.ncp];
            acc += e.y < 0 ? -v : v;
        }
        g += t.np[s];
    }
    const long long n = t.yb + (long long)il * t.nb + t.c0 + c;
    if (t.o) y1[n * ys1 + k * yk1] = (double)acc;
    else y0[n * ys0 + k * yk0] = (double)acc;
}

// ---- opposite-spin part ------------------------------------------------------------------------

template <typename T> struct TxV;
template <> struct TxV<double> {
    static constexpr int VK = 2, PAD = 2, RT = TX_ROWS64 / 16, PREC = 0, EP = 12;
    typedef double2 vec;
    static __device__ __forceinline__ double at(const vec &v, int q) { return q ? v.y : v.x; }
    static __device__ __forceinline__ const double *rows(const TxSpin &s) { return s.m64; }
};
template <> struct TxV<float> {
    static constexpr int VK = 4, PAD = 4, RT = TX_ROWS32 / 16, PREC = 1, EP = 12;
    typedef float4 vec;
    static __device__ __forceinline__ float at(const vec &v, int q)
    {
        return q == 0 ? v.x : q == 1 ? v.y : q == 2 ? v.z : v.w;
    }
    static __device__ __forceinline__ const float *rows(const TxSpin &s) { return s.m32; }
};

// acc[i] += A (row tile i) . D over KS steps, straight-line; the B vectors of the next group of
// steps are read while the products of the current group run
template <typename T, int NR, int KS>
__device__ __forceinline__ void tx_mma(typename Mf<T>::acc *acc, const T (*a)[KS], const T *b0)
{
    constexpr int VK = TxV<T>::VK, NG = KS / VK;
    typedef typename TxV<T>::vec V;
    V b[2];
    b[0] = *(const V *)b0;
#pragma unroll
    for (int g = 0; g < NG; g++) {
        if (g + 1 < NG) b[(g + 1) & 1] = *(const V *)(b0 + (g + 1) * VK);
#pragma unroll
        for (int q = 0; q < VK; q++)
#pragma unroll
            for (int i = 0; i < NR; i++)
                acc[i] = Mf<T>::mma(a[i][g * VK + q], TxV<T>::at(b[g & 1], q), acc[i]);
    }
}

__device__ __forceinline__ void tx_wave_sync()
{
    // LDS accesses of one wave execute in order; this keeps the compiler from moving them
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// element i of an array of less than 4 GB: a uniform base and a 32-bit offset per lane
template <typename T> __device__ __forceinline__ T tx_at(const T *p, uint32_t i)
{
    return *(const T *)((const char *)p + i * (uint32_t)sizeof(T));
}

// a value that all lanes share, in scalar registers
__device__ __forceinline__ long long tx_uni(long long v)
{
    const unsigned lo = __builtin_amdgcn_readfirstlane((int)v);
    return (long long)(int)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 | lo;
}

// what one wave works on: one JL, one external part w, row tiles from r0, vectors k0 .. k1 - 1
struct TxUnit {
    int ja, w, r0, nrt, dr;          // dr: row of the diagonal pairs relative to r0 (or outside)
    int k0, k1;
};

// one chunk of the reduction for every column tile and vector of the wave
template <typename T, int KS>
__device__ __forceinline__ void tx_eab(const TxDev &A, const TxItem &it, const TxTask &t,
                                       const TxChunk &ch, const TxUnit &u, bool add,
                                       const T *__restrict__ x, long long ldx, T *__restrict__ Eo,
                                       long long lde, T *__restrict__ Dt)
{
    constexpr int RT = TxV<T>::RT, EP = TxV<T>::EP, KC = 4 * KS, LDC = KC + TxV<T>::PAD;
    typedef typename TxV<T>::vec V;
    const TxSpin &SL = A.s[t.o], &SF = A.s[1 - t.o];
    const int l = threadIdx.x & 63, col = l & 15, part = l >> 4;
    const int m1 = A.m1, La = t.La;
    const long long J = t.ls0 + u.ja;

    // integral fragments: row r0 + 16 i + col, steps part * KS .. part * KS + KS - 1
    T a[RT][KS];
    {
        const long long e0 = SL.off1[J];
        const int *__restrict__ go = SL.goff1 + J * (SL.G + 1);
        const T *__restrict__ M = TxV<T>::rows(SL);
        const int *__restrict__ qt = A.q + ch.q0 + (long long)u.w * KC + part * KS;
        const uint32_t zero = (uint32_t)SL.zrow * A.ms;
        uint32_t row[RT];
#pragma unroll
        for (int i = 0; i < RT; i++) {
            const int r = u.r0 + i * 16 + col;
            row[i] = zero;
            if (r < La - t.diag) {
                int s = 0;
                while (s + 1 < t.nsec && t.sr0[s + 1] <= r) s++;
                row[i] = (uint32_t)((SL.e1[e0 + go[t.sg[s]] + r - t.sr0[s]].y >> 18) & 4095) * A.ms;
            } else if (r < La) {
                row[i] = (uint32_t)(m1 + t.iI0 + u.ja / t.nsvL) * A.ms;
            }
        }
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const uint32_t Q = qt[s];
#pragma unroll
            for (int i = 0; i < RT; i++) a[i][s] = tx_at(M, row[i] + Q);
            if (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
        if (u.dr >= 0 && u.dr < RT * 16)
            // the external electrons of JL add to its diagonal row
            for (uint64_t z = A.nint >= 64 ? 0 : SL.mask[J] >> A.nint << A.nint; z; z &= z - 1) {
                const int o = jci_ctz(z);
#pragma unroll
                for (int i = 0; i < RT; i++)
                    row[i] = i * 16 + col == u.dr ? (uint32_t)jci_tri(o, o) * A.ms : zero;
#pragma unroll
                for (int s = 0; s < KS; s++) {
                    const uint32_t Q = qt[s];
#pragma unroll
                    for (int i = 0; i < RT; i++) a[i][s] += tx_at(M, row[i] + Q);
                    if (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
            }
    }

    const TxSlot *__restrict__ slots = A.slot + ch.slot0;
    const int nsl = ch.nslot, nep = std::min(nsl, EP);
    const uint32_t *__restrict__ lst =
        SF.lst + t.lbase + (long long)u.w * t.lrows * t.nIp + part * t.nIp + col;
    // vector base, list row and chunk steps of the first slots, in scalar registers
    long long xo[EP];
    int lo[EP], ki[EP];
#pragma unroll
    for (int j = 0; j < EP; j++) {
        const TxSlot &q = slots[j < nsl ? j : 0];
        xo[j] = tx_uni(q.xb + (long long)u.ja * q.nb);
        lo[j] = __builtin_amdgcn_readfirstlane(q.lrow * t.nIp);
        ki[j] = __builtin_amdgcn_readfirstlane(q.kinfo);
    }
    auto put = [&](int k, uint32_t e, T v) __attribute__((always_inline)) {
        const int s = (int)((e >> TX_JBITS) & TX_KMAX) - (k >> 16);
        if ((unsigned)s < (unsigned)((k >> 8) & 0xFF)) Dt[col * LDC + s + (k & 0xFF)] = e >> 31 ? -v : v;
    };
    const uint32_t jm = (1u << TX_JBITS) - 1;
    const int tile1 = it.t0 + it.nt, ntc = it.nt * 16;
    uint32_t le[EP], ln[EP];
    T xv[EP];
    V zv = {};
    for (int k = u.k0; k < u.k1; k++) {
        const T *__restrict__ xk = x + k * ldx;
#pragma unroll
        for (int j = 0; j < EP; j++) le[j] = j < nep ? lst[lo[j] + it.t0 * 16] : TX_PAD;
#pragma unroll
        for (int j = 0; j < EP; j++) xv[j] = j < nep ? tx_at(xk + xo[j], le[j] & jm) : (T)0;
#pragma unroll
        for (int j = 0; j < EP; j++)
            ln[j] = j < nep && it.t0 + 1 < tile1 ? lst[lo[j] + (it.t0 + 1) * 16] : TX_PAD;
        for (int tile = it.t0; tile < tile1; tile++) {
            for (int z = l; z < LDC * (int)sizeof(T); z += 64) ((V *)Dt)[z] = zv;
            tx_wave_sync();
#pragma unroll
            for (int j = 0; j < EP; j++)
                if (j < nep) put(ki[j], le[j], xv[j]);
            for (int j = EP; j < nsl; j++) {
                const TxSlot &q = slots[j];
                const uint32_t e = lst[q.lrow * t.nIp + tile * 16];
                put(q.kinfo, e, tx_at(xk + q.xb + (long long)u.ja * q.nb, e & jm));
            }
            tx_wave_sync();
            // entries and vector elements of the next tile, behind the products below
#pragma unroll
            for (int j = 0; j < EP; j++) {
                le[j] = ln[j];
                if (j < nep && tile + 1 < tile1) {
                    xv[j] = tx_at(xk + xo[j], le[j] & jm);
                    if (tile + 2 < tile1) ln[j] = lst[lo[j] + (tile + 2) * 16];
                }
            }
            T *__restrict__ Et = Eo + k * lde + (tile - it.t0) * 16 + col;
            typename Mf<T>::acc acc[RT];
#pragma unroll
            for (int i = 0; i < RT; i++) {
                acc[i] = Mf<T>::zero();
                if (add) {
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const int r = u.r0 + i * 16 + Mf<T>::row(l, v);
                        if (r < La) acc[i][v] = Et[(long long)r * ntc];
                    }
                }
            }
            const T *b0 = Dt + col * LDC + part * KS;
            if (u.nrt == 1) tx_mma<T, 1, KS>(acc, a, b0);
            else if (u.nrt == 2) tx_mma<T, 2, KS>(acc, a, b0);
            else if (RT > 2) tx_mma<T, RT, KS>(acc, a, b0);
            tx_wave_sync();
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int r = u.r0 + i * 16 + Mf<T>::row(l, v);
                    if (r < La) Et[(long long)r * ntc] = acc[i][v];
                }
        }
    }
}

// E[row][JL, w, column] for one JL, one external part w of the first spin and up to RT row
// tiles, by one wave on its own: the integral fragments stay in registers, the D tile of 16
// columns is zeroed, scattered and read in the wave's own part of LDS, so no wave waits for
// another and the products of one overlap the list walks of the next.  The vector entries of
// the next column tile are loaded during the products of this one.
template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_tx_eab(
    TxDev A, TxRound R, int nvec, int kper, const T *__restrict__ x0, long long ldx0,
    const T *__restrict__ x1, long long ldx1, T *__restrict__ E, int ldt)
{
    constexpr int RT = TxV<T>::RT, PREC = TxV<T>::PREC;
    extern __shared__ __align__(16) unsigned char tx_smem2[];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long u = (long long)blockIdx.x * 4 + wv;
    if (u >= R.items[PREC]) return;
    T *Dt = (T *)tx_smem2 + (size_t)wv * 16 * ldt;
    const TxItem *__restrict__ items = A.item + R.i0;
    int lo = 0, hi = R.ni - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (items[mid].item0[PREC] <= u) lo = mid; else hi = mid - 1;
    }
    const TxItem &it = items[lo];
    const TxTask &t = A.task[it.task];
    int loc = (int)(u - it.item0[PREC]);
    TxUnit n;
    n.r0 = loc % it.rg[PREC] * RT * 16;
    loc /= it.rg[PREC];
    n.ja = loc / it.nw;
    n.w = it.w0 + loc % it.nw;
    n.k0 = blockIdx.y * kper;
    n.k1 = std::min(nvec, n.k0 + kper);
    n.nrt = std::min(RT, (t.La - n.r0 + 15) / 16);
    n.dr = t.diag ? t.La - 1 - n.r0 : -1;
    const T *__restrict__ x = t.o ? x1 : x0;
    const long long ldx = t.o ? ldx1 : ldx0, lde = R.elems;
    T *__restrict__ Eo = E + it.ebase + ((long long)n.ja * it.nw + (n.w - it.w0)) * t.La * it.nt * 16;
    static_assert(TX_KC == 96, "reduction depths below cover chunks of up to 96");
    for (int c = 0; c < t.nch; c++) {
        const TxChunk &ch = A.chunk[t.ch0 + c];
        switch (ch.KS) {
        case 4: tx_eab<T, 4>(A, it, t, ch, n, c > 0, x, ldx, Eo, lde, Dt); break;
        case 8: tx_eab<T, 8>(A, it, t, ch, n, c > 0, x, ldx, Eo, lde, Dt); break;
        case 12: tx_eab<T, 12>(A, it, t, ch, n, c > 0, x, ldx, Eo, lde, Dt); break;
        case 16: tx_eab<T, 16>(A, it, t, ch, n, c > 0, x, ldx, Eo, lde, Dt); break;
        case 20: tx_eab<T, 20>(A, it, t, ch, n, c > 0, x, ldx, Eo, lde, Dt); break;
        default: tx_eab<T, 24>(A, it, t, ch, n, c > 0, x, ldx, Eo, lde, Dt); break;
        }
    }
}

// y(IL, w, column) += sum over the singles of IL that a task covers, one E row each; 256
// columns of one string per work-group, eight loads in flight per lane
template <typename T>
__global__ __launch_bounds__(256) void k_tx_gab(TxDev A, TxRound R, const T *__restrict__ E, double *y0,
                                                long long ys0, long long yk0, double *y1,
                                                long long ys1, long long yk1)
{
    int lo = 0, hi = R.no - 1;
    const TxOut *__restrict__ outs = A.out + R.o0;
    const long long u = blockIdx.x;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (outs[mid].blk0 <= u) lo = mid; else hi = mid - 1;
    }
    const TxOut &t = outs[lo];
    const int loc = (int)(u - t.blk0), il = loc / t.cblk;
    const int c = (loc - il * t.cblk) * 256 + threadIdx.x, ntc = t.nt * 16;
    const int wi = c / ntc, ci = c - wi * ntc, ib = t.t0 * 16 + ci;
    if (wi >= t.nw || ib >= t.nI) return;
    const TxSpin &S = A.s[t.o];
    const long long I = t.ls0 + il, k = blockIdx.y;
    const long long e00 = S.off1[I];
    const int *__restrict__ go = S.goff1 + I * (S.G + 1);
    T acc = (T)0;
    for (int s = 0; s < t.nsrc; s++) {
        const TxSrc &q = A.src[t.src0 + s];
        const long long st = (long long)t.nw * q.La * ntc;
        const T *__restrict__ Es = E + k * R.elems + q.ebase + (long long)wi * q.La * ntc + ci;
        if (q.r0 >= 0) {
            long long e = e00 + go[q.l1];
            const long long e1 = e00 + go[q.l1 + 1];
            const T *__restrict__ Er = Es + (long long)q.r0 * ntc;
            for (; e + 8 <= e1; e += 8) {
                T v[8];
                int2 en[8];
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    en[j] = S.e1[e + j];
                    v[j] = Er[(long long)(en[j].x - q.ls0) * st + (long long)S.rk[e + j] * ntc];
                }
#pragma unroll
                for (int j = 0; j < 8; j++) acc += en[j].y & (1 << 12) ? -v[j] : v[j];
            }
            for (; e < e1; e++) {
                const int2 en = S.e1[e];
                const T v = Er[(long long)(en.x - q.ls0) * st + (long long)S.rk[e] * ntc];
                acc += en.y & (1 << 12) ? -v : v;
            }
        }
        if (q.diag) acc += Es[(long long)il * st + (long long)(q.La - 1) * ntc];
    }
    const long long n = t.yb + (long long)il * t.nb + (long long)ib * t.nsv + t.w0 + wi;
    if (t.o) y1[n * ys1 + k * yk1] += (double)acc;
    else y0[n * ys0 + k * yk0] += (double)acc;
}

template <typename T>
static int tx_run(int nvec, const TxDev &D, const TxPlan &P, const TxVec &V, T *E, hipStream_t st)
{
    const T *x0 = (const T *)V.x0, *x1 = (const T *)V.x1;
    for (const TxRound &R : P.ss) {
        hipLaunchKernelGGL(k_tx_ess<T>, dim3((unsigned)R.items[0], nvec), dim3(256),
                           (unsigned)P.rmax * 12, st, D, R, x0, V.ldx0, x1, V.ldx1, E);
        TX_CHECK();
        hipLaunchKernelGGL(k_tx_gss<T>, dim3((unsigned)R.blocks, nvec), dim3(256), 0, st, D, R, E, V.y0,
                           V.ys0, V.yk0, V.y1, V.ys1, V.yk1);
        TX_CHECK();
    }
    const int ldt = P.ldt + TxV<T>::PAD;
    for (const TxRound &R : P.ab) {
        // the vectors share a wave's fragments where there are waves enough without them
        const int kper = R.items[TxV<T>::PREC] >= 8192 ? nvec : 1;
        hipLaunchKernelGGL(k_tx_eab<T>,
                           dim3((unsigned)((R.items[TxV<T>::PREC] + 3) / 4), (nvec + kper - 1) / kper),
                           dim3(256), (unsigned)(64 * ldt * sizeof(T)), st, D, R, nvec, kper, x0, V.ldx0,
                           x1, V.ldx1, E, ldt);
        TX_CHECK();
        hipLaunchKernelGGL(k_tx_gab<T>, dim3((unsigned)R.blocks, nvec), dim3(256), 0, st, D, R, E, V.y0,
                           V.ys0, V.yk0, V.y1, V.ys1, V.yk1);
        TX_CHECK();
    }
    return 0;
}

int jk_tx_run(int prec, int nvec, const TxDev &D, const TxPlan &P, const TxVec &V, void *E,
              hipStream_t st)
{
    if (prec == 64) return tx_run<double>(nvec, D, P, V, (double *)E, st);
    return tx_run<float>(nvec, D, P, V, (float *)E, st);
}
