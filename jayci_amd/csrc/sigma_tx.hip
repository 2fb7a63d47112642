// Contraction form of the truncated-space sigma on MFMA (see sigma_tx.h).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
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
        const int h = t.grp[s], cls = t.cls[s], n = t.cnt[s];
        if (t.own[s]) {
            int r = 0;
            for (uint64_t x = cls == TX_II ? m & ~d->vmask : ext; x && r < n; x &= x - 1, r++) {
                const int k = jci_ctz(x);
                out[(long long)(t.row0[s] + r) * t.nIp] =
                    (uint32_t)tx_col(loc, t.nI, t.nsv) | ((uint32_t)tx_kpos(d, ext, cls, k, k) << TX_JBITS);
            }
            continue;
        }
        const long long e0 = off1[I] + goff1[I * (S.ngrp + 1) + h] + t.first[s];
        const int left = goff1[I * (S.ngrp + 1) + h + 1] - goff1[I * (S.ngrp + 1) + h] - t.first[s];
        for (int k = 0; k < n && k < left; k++) {
            const int2 en = e1[e0 + k];
            const int i = en.y & 63, f = (en.y >> 6) & 63;
            const int r = cls == TX_INC ? k % t.nf * (n / t.nf) + k / t.nf : k;
            out[(long long)(t.row0[s] + r) * t.nIp] =
                (uint32_t)tx_col(en.x - S.gstart[h], lists[h].nI, lists[h].nsv) |
                ((uint32_t)tx_kpos(d, ext, cls, i, f) << TX_JBITS) |
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
                                  tx_pair_id(d, i, j) | (int)((unsigned)neg << 31));
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

__global__ void k_tx_w(const SpaceDesc *__restrict__ d, int np, double sc, const double *__restrict__ m1,
                       const double *__restrict__ m2, double *__restrict__ w64,
                       float *__restrict__ w32)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int ws = np + 1, P = (int)(t / ws), Q = (int)(t % ws);
    if (P > np) return;
    double v = 0.0;
    if (P < np && Q < np) {
        int i, j, k, l;
        tx_pair_orbs(d, P, &i, &j);
        tx_pair_orbs(d, Q, &k, &l);
        v = jci_eri(m2, i, k, j, l) - jci_eri(m2, i, l, j, k);
        double h = 0.0;
        if (j == l) h += jci_h1(m1, i, k);
        if (i == l) h -= jci_h1(m1, j, k);
        if (j == k) h -= jci_h1(m1, i, l);
        if (i == k) h += jci_h1(m1, j, l);
        v += h * sc;
    }
    w64[t] = v;
    w32[t] = (float)v;
}

int jk_tx_w(const SpaceDesc *d, int norb, int nelec, const double *m1, const double *m2,
            double *w64, float *w32, hipStream_t st)
{
    const int np = norb * (norb - 1) / 2;
    hipLaunchKernelGGL(k_tx_w, dim3((unsigned)(((long long)(np + 1) * (np + 1) + 255) / 256)), dim3(256), 0, st, d, np,
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

// the last i < n with at(i) <= u (at(0) <= u, ascending), by whole waves: 64 probes a round, one
// round up to 64 entries, two up to 4096
template <typename F> __device__ __forceinline__ int tx_find(int n, long long u, F at)
{
    const int l = threadIdx.x & 63;
    int lo = 0;
    while (n > 1) {
        const int st = (n + 63) / 64, i = l * st;
        const int c = __popcll(__ballot(i < n && at(lo + i) <= u)) - 1;
        lo += c * st;
        n = std::min(st, n - c * st);
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// work-groups in runs of `run` consecutive ones per XCD (they are dealt to the 8 XCDs round
// robin), so that neighbours share an L2; the grid is a multiple of 8 run
#define TX_RUN 16
__device__ __forceinline__ long long tx_xcd(long long b)
{
    const long long q = b / (8 * TX_RUN), r = b % (8 * TX_RUN);
    return q * (8 * TX_RUN) + (r & 7) * TX_RUN + (r >> 3);
}
static inline unsigned tx_grid(long long n)
{
    return (unsigned)((n + 8 * TX_RUN - 1) / (8 * TX_RUN) * (8 * TX_RUN));
}

// one 16 x 16 tile of a block: internal parts ia0 .. of external part wa, and so for columns
struct TxTile {
    int b, ia0, wa, ib0, wb, nIa, nsa, nIb, nsb;
    long long na, nb, off;
};
__device__ __forceinline__ TxTile tx_tile(const SpaceDesc *__restrict__ d,
                                          const long long *__restrict__ tt, long long u)
{
    TxTile t;
    t.b = tx_find(d->nblk, u, [&](int i) { return tt[i]; });
    const int p = d->bp[t.b], q = d->bq[t.b];
    t.na = d->s[0].gn[p];
    t.nb = d->s[1].gn[q];
    t.nsa = (int)(d->s[0].nsv[p] > 1 ? d->s[0].nsv[p] : 1);
    t.nsb = (int)(d->s[1].nsv[q] > 1 ? d->s[1].nsv[q] : 1);
    t.nIa = (int)(t.na / t.nsa);
    t.nIb = (int)(t.nb / t.nsb);
    const int ntc = (t.nIb + 15) / 16 * t.nsb;
    const long long rel = u - tt[t.b];
    const int rt = (int)(rel / ntc), ct = (int)(rel % ntc);
    t.wa = rt % t.nsa;
    t.ia0 = rt / t.nsa * 16;
    t.wb = ct % t.nsb;
    t.ib0 = ct / t.nsb * 16;
    t.off = d->boff[t.b];
    return t;
}

// LOOP: tiles in turns of the grid.  Spaces of few internal parts have about as many tiles as
// determinants, past what a grid may hold; up to TX_TILES each has a work-group of its own (in
// turns of 2^14, 16e/28o: 0.60 -> 0.67 and 0.69 -> 0.78 ms).
#define TX_TILES (1 << 20)

// The vector into tx_col order, straight and block-transposed.  Bound by memory: one read (in
// runs of 16 external parts of a string, neighbouring tiles sharing the lines) and two writes.
template <typename T, bool LOOP>
__global__ __launch_bounds__(256) void k_tx_in(long long N, long long ntt, const SpaceDesc *__restrict__ d,
                                               const long long *__restrict__ tt,
                                               const double *__restrict__ x, long long xs,
                                               long long xk, T *__restrict__ x0, T *__restrict__ x1)
{
    __shared__ T s[16][17];
    const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
    const long long k = blockIdx.y;
    for (long long b = blockIdx.x;; b += gridDim.x) {
        const long long u = tx_xcd(b);
        if (u >= ntt) {
            if (!LOOP || b - b % (8 * TX_RUN) >= ntt) return;   // no tile left in this run of work-groups
            continue;
        }
        const TxTile t = tx_tile(d, tt, u);
        if (LOOP && b != blockIdx.x) __syncthreads();           // the tile before is read
        if (t.ia0 + ty < t.nIa && t.ib0 + tx < t.nIb) {
            const long long r = (long long)(t.ia0 + ty) * t.nsa + t.wa, c = (long long)(t.ib0 + tx) * t.nsb + t.wb;
            const T v = (T)x[(t.off + r * t.nb + c) * xs + k * xk];
            s[ty][tx] = v;
            x0[k * N + t.off + r * t.nb + (long long)t.wb * t.nIb + t.ib0 + tx] = v;
        }
        __syncthreads();
        if (t.ib0 + ty < t.nIb && t.ia0 + tx < t.nIa) {
            const long long c = (long long)(t.ib0 + ty) * t.nsb + t.wb;
            x1[k * N + t.off + c * t.na + (long long)t.wa * t.nIa + t.ia0 + tx] = s[tx][ty];
        }
        if (!LOOP) return;
    }
}

template <bool LOOP>
__global__ __launch_bounds__(256) void k_tx_out(long long N, long long ntt, const SpaceDesc *__restrict__ d,
                                                const long long *__restrict__ tt,
                                                const double *__restrict__ y0,
                                                const double *__restrict__ y1,
                                                double *__restrict__ y, long long ys, long long yk)
{
    __shared__ double s[16][17];
    const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
    const long long k = blockIdx.y;
    for (long long b = blockIdx.x;; b += gridDim.x) {
        const long long u = tx_xcd(b);
        if (u >= ntt) {
            if (!LOOP || b - b % (8 * TX_RUN) >= ntt) return;   // no tile left in this run of work-groups
            continue;
        }
        const TxTile t = tx_tile(d, tt, u);
        if (LOOP && b != blockIdx.x) __syncthreads();           // the tile before is read
        if (t.ib0 + ty < t.nIb && t.ia0 + tx < t.nIa) {
            const long long c = (long long)(t.ib0 + ty) * t.nsb + t.wb;
            s[ty][tx] = y1[k * N + t.off + c * t.na + (long long)t.wa * t.nIa + t.ia0 + tx];
        }
        __syncthreads();
        if (t.ia0 + ty < t.nIa && t.ib0 + tx < t.nIb) {
            const long long r = (long long)(t.ia0 + ty) * t.nsa + t.wa, c = (long long)(t.ib0 + tx) * t.nsb + t.wb;
            y[(t.off + r * t.nb + c) * ys + k * yk] =
                y0[k * N + t.off + r * t.nb + (long long)t.wb * t.nIb + t.ib0 + tx] + s[tx][ty];
        }
        if (!LOOP) return;
    }
}

int jk_tx_in(int prec, int nvec, long long N, const SpaceDesc *d, const long long *tt, long long ntt,
             const double *x, long long xs, long long xk, void *x0, void *x1, hipStream_t st)
{
    const dim3 g(tx_grid(std::min<long long>(ntt, TX_TILES)), (unsigned)nvec);
    auto go = [&](auto loop) {
        constexpr bool L = decltype(loop)::value;
        if (prec == 64)
            hipLaunchKernelGGL((k_tx_in<double, L>), g, dim3(256), 0, st, N, ntt, d, tt, x, xs, xk,
                               (double *)x0, (double *)x1);
        else
            hipLaunchKernelGGL((k_tx_in<float, L>), g, dim3(256), 0, st, N, ntt, d, tt, x, xs, xk,
                               (float *)x0, (float *)x1);
    };
    if (ntt > TX_TILES) go(std::true_type{});
    else go(std::false_type{});
    TX_CHECK();
    return 0;
}

int jk_tx_out(int nvec, long long N, const SpaceDesc *d, const long long *tt, long long ntt,
              const double *y0, const double *y1, double *y, long long ys, long long yk,
              hipStream_t st)
{
    const dim3 g(tx_grid(std::min<long long>(ntt, TX_TILES)), (unsigned)nvec);
    if (ntt > TX_TILES)
        hipLaunchKernelGGL(k_tx_out<true>, g, dim3(256), 0, st, N, ntt, d, tt, y0, y1, y, ys, yk);
    else
        hipLaunchKernelGGL(k_tx_out<false>, g, dim3(256), 0, st, N, ntt, d, tt, y0, y1, y, ys, yk);
    TX_CHECK();
    return 0;
}

// ---- same-spin part ----------------------------------------------------------------------------

// element i of an array of less than 4 GB: a uniform base and a 32-bit offset per lane
template <typename T> __device__ __forceinline__ T tx_at(const T *p, uint32_t i)
{
    return *(const T *)((const char *)p + i * (uint32_t)sizeof(T));
}

template <typename T> __device__ __forceinline__ void tx_put(T *p, uint32_t i, T v)
{
    *(T *)((char *)p + i * (uint32_t)sizeof(T)) = v;
}

__device__ __forceinline__ void tx_load4(double *v, const double *p)
{
    const double2 a = *(const double2 *)p, b = *(const double2 *)(p + 2);
    v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
}
__device__ __forceinline__ void tx_load4(float *v, const float *p)
{
    const float4 a = *(const float4 *)p;
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
template <typename T> __device__ __forceinline__ const T *tx_w(const TxSpin &s);
template <> __device__ __forceinline__ const double *tx_w<double>(const TxSpin &s) { return s.w64; }
template <> __device__ __forceinline__ const float *tx_w<float>(const TxSpin &s) { return s.w32; }

// E[p][K2, c] on 64 x 64 tiles (64 pairs of one N - 2 electron string, 64 columns): a wave owns
// 16 columns and all four row tiles, its B operand comes straight from the vector (rows of 16
// consecutive elements).  Strings of up to TX_RMAX pairs (most of them, and few pairs at that)
// keep their whole W block in LDS for several column blocks, without barriers in between; the
// others stage W one 16-deep step ahead.  In a step lane group g takes the pairs
// 4 g .. 4 g + 3, so that its four W entries of a row are one or two 16-byte reads.  The pair
// list is padded to whole steps by the zero row of W and the last pair's row of the vector (an
// infinite element there makes NaN of the padding, in results it is connected to anyway).  Offsets
// are 32 bits while the vector is below 4 GB (BIG: 64).  16e/28o FP64 writes 31 GB in 17.6 ms (one
// 64-column block per work-group: 23.1 ms).
// RT: row tiles of a work-group, 4, or 2 for strings of up to 32 pairs, whose work-groups are the
// most and the shortest: with half the registers and a quarter of the LDS seven fit on a CU
// instead of four (7a6b/17o two vectors 1.33 -> 1.28 ms, 16e/20o FP64 three 53.3 -> 51.8, 16e/28o
// one 92.2 -> 90.0).
template <typename T, bool BIG, int RT>
__global__ __launch_bounds__(256, RT == 2 ? 6 : 4) void k_tx_ess(TxDev A, TxRound R, int i0, int ni, long long N,
                                                   const T *__restrict__ x0, const T *__restrict__ x1,
                                                   T *__restrict__ E)
{
    typedef typename std::conditional<BIG, long long, uint32_t>::type O;
    extern __shared__ __align__(16) unsigned char tx_smem[];
    // row stride: 16-byte reads, rows spread over the banks
    __shared__ __align__(16) T As[RT * 16][RT * 16 + 4];
    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6;
    const TxPairItem *__restrict__ items = A.pitem + i0;
    const long long u = blockIdx.x;
    const TxPairItem &it = items[tx_find(ni, u, [&](int i) { return items[i].item0; })];
    const TxPairTask &t = A.ptask[it.task];
    const int loc = (int)(u - it.item0), rg = loc % it.rg, ct = loc / it.rg % it.ct;
    const long long k2 = loc / (it.rg * it.ct), K2 = it.k0 + k2;
    const int Rr = t.R, Rp = (Rr + 15) / 16 * 16, r0 = rg * 64, nc = it.nc, ncp = it.ncp;
    const TxSpin &S = A.s[t.o];
    const long long k = blockIdx.y;
    const int np = A.np, ws = np + 1;
    // vector offset and W row of every pair, sign in bit 31
    O *__restrict__ off = (O *)tx_smem;
    int *__restrict__ pr = (int *)(off + Rp);
    for (int r = tid; r < Rp; r += 256) {
        const int q = std::min(r, Rr - 1);
        int s = 0;
        while (s + 1 < t.nsec && t.sr[s + 1] <= q) s++;
        const int2 en = S.kl[t.lbase + K2 * t.Rfull + t.so[s] + (q - t.sr[s])];
        off[r] = (O)(t.sx[s] + (long long)en.x * t.nb);
        pr[r] = r < Rr ? en.y : np;
    }
    __syncthreads();
    const T *__restrict__ W = tx_w<T>(S);
    // W tile: rows ar + 16 j, column ak (16 mostly consecutive columns of four rows a load)
    const int ar = tid >> 4, ak = tid & 15, kk = l >> 4;
    const int nrt = (std::min(RT * 16, Rr - r0) + 15) / 16;
    uint32_t wrow[RT];
#pragma unroll
    for (int j = 0; j < RT; j++) {
        const int r = r0 + ar + 16 * j;
        wrow[j] = (uint32_t)(r < Rp ? pr[r] & 0x7FFFFFFF : np) * ws;
    }
    const T *__restrict__ x = (t.o ? x1 : x0) + k * N + it.c0;
    T *__restrict__ Ek = E + k * R.elems + it.ebase + (k2 * Rr + r0) * ncp;
    const int cb0 = ct * it.cb, cb1 = std::min(cb0 + it.cb, (nc + 63) / 64);
    T ra[RT], rb[4];
    typename Mf<T>::acc acc[RT];
    auto load_w = [&](int k0) __attribute__((always_inline)) {
        const int p = pr[k0 + ak];
#pragma unroll
        for (int j = 0; j < RT; j++)
            if (j < nrt) {
                const T v = tx_at(W, wrow[j] + (uint32_t)(p & 0x7FFFFFFF));
                ra[j] = p < 0 ? -v : v;
            }
    };
    // the vector's rows of a step; columns past the end repeat the last one (their products are
    // not read)
    auto load_x = [&](int k0, uint32_t xc) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const O o = off[k0 + kk * 4 + j];
            rb[j] = BIG ? x[(long long)o + xc] : tx_at(x, (uint32_t)o + xc);
        }
    };
    auto store = [&](int c) __attribute__((always_inline)) {
        if (c >= ncp) return;
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = i * 16 + Mf<T>::row(l, v);
                if (r0 + r < Rr) Ek[(long long)r * ncp + c] = acc[i][v];
            }
    };
    const int cl = w * 16 + (l & 15);
    if (RT == 2 || Rp <= TX_RMAX) {
        for (int k0 = 0; k0 < Rp; k0 += 16) {
            load_w(k0);
#pragma unroll
            for (int j = 0; j < RT; j++) if (j < nrt) As[ar + 16 * j][k0 + ak] = ra[j];
        }
        __syncthreads();
        for (int cb = cb0; cb < cb1; cb++) {
            if (cb * 64 + w * 16 >= nc) break;
            const uint32_t xc = (uint32_t)std::min(cb * 64 + cl, nc - 1);
#pragma unroll
            for (int i = 0; i < RT; i++) acc[i] = Mf<T>::zero();
            load_x(0, xc);
            for (int k0 = 0; k0 < Rp; k0 += 16) {
                T b[4];
#pragma unroll
                for (int j = 0; j < 4; j++) b[j] = rb[j];
                if (k0 + 16 < Rp) load_x(k0 + 16, xc);
#pragma unroll
                for (int i = 0; i < RT; i++)
                    if (i < nrt) {
                        T a[4];
                        tx_load4(a, &As[i * 16 + (l & 15)][k0 + kk * 4]);
#pragma unroll
                        for (int j = 0; j < 4; j++) acc[i] = Mf<T>::mma(a[j], b[j], acc[i]);
                    }
            }
            store(cb * 64 + cl);
        }
        return;
    }
    // two 16-deep W tiles side by side in As, columns 0 .. 15 and 32 .. 47
    const uint32_t xc = (uint32_t)std::min(cb0 * 64 + cl, nc - 1);
#pragma unroll
    for (int i = 0; i < RT; i++) acc[i] = Mf<T>::zero();
    load_w(0);
    load_x(0, xc);
#pragma unroll
    for (int j = 0; j < RT; j++) if (j < nrt) As[ar + 16 * j][ak] = ra[j];
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < Rp; k0 += 16) {
        T b[4];
#pragma unroll
        for (int j = 0; j < 4; j++) b[j] = rb[j];
        const bool more = k0 + 16 < Rp;
        if (more) {
            load_w(k0 + 16);
            load_x(k0 + 16, xc);
        }
#pragma unroll
        for (int i = 0; i < RT; i++)
            if (i < nrt) {
                T a[4];
                tx_load4(a, &As[i * 16 + (l & 15)][buf + kk * 4]);
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i] = Mf<T>::mma(a[j], b[j], acc[i]);
            }
        buf ^= 32;
        if (more) {
#pragma unroll
            for (int j = 0; j < RT; j++) if (j < nrt) As[ar + 16 * j][buf + ak] = ra[j];
        }
        __syncthreads();
    }
    store(cb0 * 64 + cl);
}

// acc plus (or less, where the entry is complemented) E at the n offsets ent, each moved by w
// times its step, eight loads in flight
template <typename T>
__device__ __forceinline__ T tx_sum(T acc, const T *__restrict__ E, const long long *ent, int n,
                                    const int *step = nullptr, int w = 0)
{
    int m = 0;
    for (; m + 8 <= n; m += 8) {
        T v[8];
        long long o[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            o[j] = ent[m + j];
            v[j] = E[(o[j] ^ (o[j] >> 63)) + (step ? (long long)w * step[m + j] : 0)];
        }
#pragma unroll
        for (int j = 0; j < 8; j++) acc += o[j] < 0 ? -v[j] : v[j];
    }
    // the rest together: entry 0 in place of those past the end, their values unused
    if (m < n) {
        T v[8];
        long long o[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int i = m + j < n ? m + j : 0;
            o[j] = ent[i];
            v[j] = E[(o[j] ^ (o[j] >> 63)) + (step ? (long long)w * step[i] : 0)];
        }
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (m + j < n) acc += o[j] < 0 ? -v[j] : v[j];
    }
    return acc;
}

// of the work-group's 256 entries those to keep, in order: this thread's place and their number
__device__ __forceinline__ int tx_place(bool keep, int *cnt, int *n)
{
    const uint64_t b = __ballot(keep);
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (l == 0) cnt[w] = __popcll(b);
    __syncthreads();
    int at = __popcll(b & ((1ULL << l) - 1ULL));
    for (int i = 0; i < w; i++) at += cnt[i];
    *n = cnt[0] + cnt[1] + cnt[2] + cnt[3];
    return at;
}

// the same-spin sums: y(I, c) = sum over the pairs of I, one E row each (coalesced); the first
// writer of the result.  The rows' offsets are set up in LDS once for the string's columns.  PART:
// the round holds some of the N - 2 electron strings only, the entries of the others are left out
// and the sums of its successors are added.
#define TX_ENT 512
#define TX_SRC 64            // one wave's scan
template <typename T, bool PART>
__global__ __launch_bounds__(256) void k_tx_gss(TxDev A, TxRound R, long long N,
                                                const T *__restrict__ E, double *__restrict__ y0,
                                                double *__restrict__ y1)
{
    __shared__ long long ent[TX_ENT];
    __shared__ int cnt[4];
    const TxPairOut *__restrict__ outs = A.pout + R.o0;
    const long long u = blockIdx.x;
    const TxPairOut &t = outs[tx_find(R.no, u, [&](int i) { return outs[i].blk0; })];
    const int loc = (int)(u - t.blk0), il = loc / t.cblk;
    const int c = (loc - il * t.cblk) * 256 + threadIdx.x;
    const TxSpin &S = A.s[t.o];
    const int2 *__restrict__ g = S.gl + (long long)(t.ls0 + il) * S.npair;
    const long long k = blockIdx.y;
    int np = 0;
    for (int s = 0; s < t.nsec; s++) np += t.np[s];
    T acc = (T)0;
    // offset of entry r (complemented: less), false where its N - 2 string is not in the round
    auto entry = [&](int r, long long &o) __attribute__((always_inline)) {
        int s = 0, m = r;
        while (m >= t.np[s]) m -= t.np[s++];
        const int2 e = g[PART ? t.g0[s] + m : r];
        const int K = PART ? e.x - t.k0[s] : e.x;
        o = t.eb[s] + ((long long)K * t.R[s] + t.r0[s] + (e.y & 0x7FFFFFFF)) * t.ncp;
        if (e.y < 0) o = ~o;
        return !PART || (unsigned)K < (unsigned)t.nk[s];
    };
    if (!PART) {
        for (int m0 = 0; m0 < np; m0 += TX_ENT) {
            const int n = std::min(TX_ENT, np - m0);
            if (m0) __syncthreads();
            for (int m = threadIdx.x; m < n; m += 256) {
                long long o;
                entry(m0 + m, o);
                ent[m] = o;
            }
            __syncthreads();
            if (c < t.nc) acc = tx_sum(acc, E + k * R.elems + c, ent, n);
        }
    } else {
        for (int m0 = 0; m0 < np; m0 += 256) {
            const int m = m0 + threadIdx.x;
            long long o = 0;
            const bool in = m < np && entry(m, o);
            int n;
            if (m0) __syncthreads();
            const int at = tx_place(in, cnt, &n);
            if (in) ent[at] = o;
            __syncthreads();
            if (c < t.nc) acc = tx_sum(acc, E + k * R.elems + c, ent, n);
        }
    }
    if (c >= t.nc) return;
    const long long n = t.yb + (long long)il * t.nb + t.c0 + c;
    double *y = (t.o ? y1 : y0) + (k * N + n);
    *y = PART && t.add ? *y + (double)acc : (double)acc;
}

// ---- opposite-spin part ------------------------------------------------------------------------

template <typename T> struct TxV;
template <> struct TxV<double> {
    static constexpr int VK = 2, PAD = 2, EP = 4, WPE = 3;
    typedef double2 vec;
    static __device__ __forceinline__ double at(const vec &v, int q) { return q ? v.y : v.x; }
    static __device__ __forceinline__ const double *rows(const TxSpin &s) { return s.m64; }
};
template <> struct TxV<float> {
    static constexpr int VK = 4, PAD = 4, EP = 4, WPE = 4;
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
        __builtin_amdgcn_sched_barrier(0);   // one group of B vectors ahead, no more
    }
}

// what one wave works on: one JL, one external part w, row tiles from r0, vectors k0 .. k1 - 1
struct TxUnit {
    int ja, w, r0, nrt, dr;          // dr: row of the diagonal pairs relative to r0 (or outside)
    int k0, k1;
};

// one chunk of the reduction for every column tile and vector of the wave
template <typename T, int KS>
__device__ __forceinline__ void tx_eab(const TxDev &A, const TxItem &it, const TxTask &t,
                                       const TxChunk &ch, TxUnit u, bool add,
                                       const T *__restrict__ x, long long ldx, T *__restrict__ Eo,
                                       long long lde, T *__restrict__ Dt)
{
    constexpr int RT = TX_ROWS / 16, EP = TxV<T>::EP, KC = 4 * KS, LDC = KC + TxV<T>::PAD;
    typedef typename TxV<T>::vec V;
    // the lane and the unit made opaque here: what the reduction depths have in common would
    // otherwise be computed ahead of the switch over them and held in registers all along
    int l = threadIdx.x & 63;
    asm volatile("" : "+v"(l));
    asm volatile("" : "+s"(u.ja));
    asm volatile("" : "+s"(u.w));
    asm volatile("" : "+s"(u.r0));
    const int col = l & 15, part = l >> 4;
    const int La = wave_uni(t.La), nIp = wave_uni(t.nIp);

    // integral fragments: row r0 + 16 i + col, steps part * KS .. part * KS + KS - 1
    T a[RT][KS];
    {
        const TxSpin &SL = A.s[t.o];
        const long long J = t.ls0 + u.ja;
        const long long e0 = SL.off1[J];
        const int *__restrict__ go = SL.goff1 + J * (SL.G + 1);
        const T *__restrict__ M = TxV<T>::rows(SL);
        const int *__restrict__ qt = A.q + ch.q0 + (long long)u.w * KC;
        const uint32_t zero = (uint32_t)SL.zrow * A.ms;
        // the rows come through LDS, a row (a run of mostly consecutive pairs) per load
        uint32_t Q[2];
#pragma unroll
        for (int h = 0; h < 2; h++) Q[h] = qt[std::min(l + 64 * h, KC - 1)];
#pragma unroll
        for (int i = 0; i < RT; i++) {
            // (past the last row tile the rows of the one before are read again, and not used:
            // 20.4 -> 17 us at 4a4b/10o)
            if (i == 0 || u.nrt > 1) {
                const int r = u.r0 + i * 16 + col;
                uint32_t row = zero;
                if (r < La - t.diag) {
                    int s = 0;
                    while (s + 1 < t.nsec && t.sr0[s + 1] <= r) s++;
                    row = (uint32_t)((SL.e1[e0 + go[t.sg[s]] + r - t.sr0[s]].y >> 18) & 4095) * A.ms;
                } else if (r < La) {
                    row = (uint32_t)(A.m1 + t.iI0 + u.ja / t.nsvL) * A.ms;
                }
#pragma unroll
                for (int g = 0; g < 16; g += 8) {
                    T v[8][2];
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const T *__restrict__ Mr = M + (uint32_t)__builtin_amdgcn_readlane((int)row, g + j);
#pragma unroll
                        for (int h = 0; h < (KC > 64 ? 2 : 1); h++) v[j][h] = tx_at(Mr, Q[h]);
                    }
#pragma unroll
                    for (int j = 0; j < 8; j++)
#pragma unroll
                        for (int h = 0; h < (KC > 64 ? 2 : 1); h++)
                            if (l + 64 * h < KC) Dt[(g + j) * LDC + l + 64 * h] = v[j][h];
                }
                wave_sync();
                if (u.dr >> 4 == i && u.dr >= 0) {
                    // the external electrons of JL add to its diagonal row
                    for (uint64_t z = A.nint >= 64 ? 0 : SL.mask[J] >> A.nint << A.nint; z; z &= z - 1) {
                        const int o = jci_ctz(z);
                        const T *__restrict__ Mr = M + (uint32_t)jci_tri(o, o) * A.ms;
#pragma unroll
                        for (int h = 0; h < (KC > 64 ? 2 : 1); h++)
                            if (l + 64 * h < KC) Dt[(u.dr & 15) * LDC + l + 64 * h] += tx_at(Mr, Q[h]);
                    }
                    wave_sync();
                }
            }
#pragma unroll
            for (int s = 0; s < KS; s += TxV<T>::VK) {
                const V v = *(const V *)(Dt + col * LDC + part * KS + s);
#pragma unroll
                for (int q = 0; q < TxV<T>::VK; q++)
#pragma unroll
                    for (int ii = 0; ii < RT; ii++)
                        if (ii == i) a[ii][s + q] = TxV<T>::at(v, q);
            }
            wave_sync();
        }
    }

    // list of external part w; a lane reads row `part` of four, column `col` of a tile
    const uint32_t *__restrict__ lst = A.s[1 - t.o].lst + wave_uni(t.lbase + (long long)u.w * t.lrows * nIp);
    const uint32_t lofs = (uint32_t)(part * nIp + col);
    // vector base, list row and chunk steps of slot j in lane j (chunks hold at most 64 slots)
    const int nsl = wave_uni(ch.nslot);
    int vxl, vxh, vlo, vki;
    {
        const TxSlot &q = A.slot[ch.slot0 + std::min(l, nsl - 1)];
        const long long xo = q.xb + (long long)u.ja * q.nb;
        vxl = (int)xo;
        vxh = (int)(xo >> 32);
        vlo = q.lrow * nIp;
        vki = l < nsl ? q.kinfo : 0;
    }
    T *Dc = Dt + col * LDC;
    const uint32_t jm = (1u << TX_JBITS) - 1;
    const int tile0 = wave_uni(it.t0), tile1 = tile0 + wave_uni(it.nt);
    const int p0 = wave_uni(it.p0), ntc = wave_uni(it.pn) * 16;
    // a lane's rows are LROW * part + VROW v + 16 i from r0: one offset per lane, the rest scalar
    const uint32_t eofs = (uint32_t)(Mf<T>::LROW * part * ntc + col);
    const int rleft = La - u.r0 - Mf<T>::LROW * part;
    Eo += (long long)u.r0 * ntc;
    const T *__restrict__ xk = x;
    // four slots at a time (the slots past the last one repeat it and write nothing)
    auto entries = [&](int j0, int tile, uint32_t *e) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; j++)
            e[j] = tx_at(lst + (__builtin_amdgcn_readlane(vlo, j0 + j) + tile * 16), lofs);
    };
    auto values = [&](int j0, const uint32_t *e, T *v) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const long long xo = (long long)__builtin_amdgcn_readlane(vxh, j0 + j) << 32 |
                                 (unsigned)__builtin_amdgcn_readlane(vxl, j0 + j);
            v[j] = tx_at(xk + xo, e[j] & jm);
        }
    };
    auto puts = [&](int j0, const uint32_t *e, const T *v) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int k = __builtin_amdgcn_readlane(vki, j0 + j);
            const int s = (int)((e[j] >> TX_JBITS) & TX_KMAX) - (k >> 16);
            if ((unsigned)s < (unsigned)((k >> 8) & 0xFF)) Dc[s + (k & 0xFF)] = e[j] >> 31 ? -v[j] : v[j];
        }
    };
    constexpr int NP = EP / 4;                     // groups of slots loaded one tile ahead
    uint32_t le[EP + 1], ln[EP + 1];
    T xv[EP + 1];
    V zv = {};
    for (int k = u.k0; k < u.k1; k++) {
        xk = x + k * ldx;
#pragma unroll
        for (int g = 0; g < NP; g++)
            if (4 * g < nsl) entries(4 * g, tile0, le + 4 * g);
#pragma unroll
        for (int g = 0; g < NP; g++)
            if (4 * g < nsl) {
                values(4 * g, le + 4 * g, xv + 4 * g);
                if (tile0 + 1 < tile1) entries(4 * g, tile0 + 1, ln + 4 * g);
            }
        for (int tile = tile0; tile < tile1; tile++) {
            for (int z = l; z < LDC * (int)sizeof(T); z += 64) ((V *)Dt)[z] = zv;
            wave_sync();
#pragma unroll
            for (int g = 0; g < NP; g++)
                if (4 * g < nsl) puts(4 * g, le + 4 * g, xv + 4 * g);
            for (int j = EP; j < nsl; j += 4) {
                uint32_t e[4];
                T v[4];
                entries(j, tile, e);
                values(j, e, v);
                puts(j, e, v);
            }
            wave_sync();
            // entries and vector elements of the next tile, behind the products below
#pragma unroll
            for (int g = 0; g < NP; g++)
                if (4 * g < nsl && tile + 1 < tile1) {
#pragma unroll
                    for (int j = 0; j < 4; j++) le[4 * g + j] = ln[4 * g + j];
                    values(4 * g, le + 4 * g, xv + 4 * g);
                    if (tile + 2 < tile1) entries(4 * g, tile + 2, ln + 4 * g);
                }
            T *__restrict__ Et = Eo + k * lde + (tile - p0) * 16;
            typename Mf<T>::acc acc[RT];
#pragma unroll
            for (int i = 0; i < RT; i++) {
                acc[i] = Mf<T>::zero();
                if (add) {
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        if (i * 16 + Mf<T>::VROW * v < rleft)
                            acc[i][v] = tx_at(Et + (i * 16 + Mf<T>::VROW * v) * (long long)ntc, eofs);
                }
            }
            const T *b0 = Dc + part * KS;
            if (u.nrt == 1) tx_mma<T, 1, KS>(acc, a, b0);
            else if (u.nrt == 2) tx_mma<T, RT, KS>(acc, a, b0);
            wave_sync();
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (i * 16 + Mf<T>::VROW * v < rleft)
                        tx_put(Et + (i * 16 + Mf<T>::VROW * v) * (long long)ntc, eofs, acc[i][v]);
        }
    }
}

// E[row][JL, w, column] for one JL, one external part w of the first spin and up to RT row
// tiles, by one wave on its own: the integral fragments stay in registers, the D tile of 16
// columns is zeroed, scattered and read in the wave's own part of LDS, so no wave waits for
// another and the products of one overlap the list walks of the next.  The vector entries of
// the next column tile are loaded during the products of this one.
template <typename T>
__global__ __launch_bounds__(256, TxV<T>::WPE) void k_tx_eab(
    TxDev A, TxRound R, int nvec, int kper, long long N, const T *__restrict__ x0,
    const T *__restrict__ x1, T *__restrict__ E, int ldt)
{
    constexpr int RT = TX_ROWS / 16;
    extern __shared__ __align__(16) unsigned char tx_smem2[];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long u = tx_xcd(blockIdx.x) * 4 + wv;
    if (u >= R.items) return;
    T *Dt = (T *)tx_smem2 + (size_t)wv * 16 * ldt;
    const TxItem *__restrict__ items = A.item + R.i0;
    const TxItem &it = items[tx_find(R.ni, u, [&](int i) { return items[i].item0; })];
    const TxTask &t = A.task[it.task];
    int loc = (int)(u - it.item0);
    TxUnit n;
    n.r0 = loc % it.rg * RT * 16;
    loc /= it.rg;
    const int jl = loc / it.nw;
    n.ja = it.j0 + jl;
    n.w = it.w0 + loc % it.nw;
    n.k0 = blockIdx.y * kper;
    n.k1 = std::min(nvec, n.k0 + kper);
    n.nrt = std::min(RT, (t.La - n.r0 + 15) / 16);
    n.dr = t.diag ? t.La - 1 - n.r0 : -1;
    const T *__restrict__ x = t.o ? x1 : x0;
    const long long lde = R.elems;
    T *__restrict__ Eo = E + it.ebase + ((long long)jl * it.nw + (n.w - it.w0)) * t.La * it.pn * 16;
    static_assert(TX_KC == 96, "reduction depths below cover chunks of up to 96");
    for (int c = 0; c < t.nch; c++) {
        const TxChunk &ch = A.chunk[t.ch0 + c];
        switch (ch.KS) {
        case 4: tx_eab<T, 4>(A, it, t, ch, n, c > 0, x, N, Eo, lde, Dt); break;
        case 8: tx_eab<T, 8>(A, it, t, ch, n, c > 0, x, N, Eo, lde, Dt); break;
        case 12: tx_eab<T, 12>(A, it, t, ch, n, c > 0, x, N, Eo, lde, Dt); break;
        case 16: tx_eab<T, 16>(A, it, t, ch, n, c > 0, x, N, Eo, lde, Dt); break;
        case 20: tx_eab<T, 20>(A, it, t, ch, n, c > 0, x, N, Eo, lde, Dt); break;
        default: tx_eab<T, 24>(A, it, t, ch, n, c > 0, x, N, Eo, lde, Dt); break;
        }
    }
}

// y(IL, w, column) += sum over the singles of IL that the round's tasks cover, one E row each;
// 256 columns of one string per work-group.  The rows' offsets, over all sources, are set up in
// LDS first: the sum is then one stream of loads, eight in flight per lane, at the copy rate for
// large spaces, and small ones (chains of list loads before) take 16.2 -> 9.1 us at 4a4b/10o and
// 0.22 -> 0.19 ms at 7a6b/17o.  PART: the round holds some of a source's strings JL only, the entries
// of the others are left out.
template <typename T, bool PART>
__global__ __launch_bounds__(256) void k_tx_gab(TxDev A, TxRound R, long long N,
                                                const T *__restrict__ E, double *__restrict__ y0,
                                                double *__restrict__ y1)
{
    // per source: first of the string's singles, rows before it in the list (its singles, then its
    // diagonal row); the list's offsets and steps per external part
    __shared__ int first[TX_SRC], base[TX_SRC + 1];
    __shared__ long long ent[TX_ENT];
    __shared__ int step[TX_ENT], cnt[4];
    const TxOut *__restrict__ outs = A.out + R.o0;
    const long long u = blockIdx.x;
    const TxOut &t = outs[tx_find(R.no, u, [&](int i) { return outs[i].blk0; })];
    const int loc = (int)(u - t.blk0), il = loc / t.cblk;
    const int c = (loc - il * t.cblk) * 256 + threadIdx.x, ntc = t.nt * 16;
    const int wi = c / ntc, ci = c - wi * ntc, ib = t.t0 * 16 + ci;
    const bool in = wi < t.nw && ib < t.nI;
    const TxSpin &S = A.s[t.o];
    const long long I = t.ls0 + il, k = blockIdx.y;
    const long long e00 = S.off1[I];
    const int *__restrict__ go = S.goff1 + I * (S.G + 1);
    T acc = (T)0;
    for (int s0 = 0; s0 < t.nsrc; s0 += TX_SRC) {
        const int ns = std::min(TX_SRC, t.nsrc - s0);
        if (s0) __syncthreads();
        if (threadIdx.x < TX_SRC) {
            int n = 0;
            if ((int)threadIdx.x < ns) {
                const TxSrc &q = A.src[t.src0 + s0 + threadIdx.x];
                const int g0 = go[q.l1];
                first[threadIdx.x] = g0;
                n = (q.r0 >= 0 ? go[q.l1 + 1] - g0 : 0) + (q.diag ? 1 : 0);
            }
            for (int d = 1; d < 64; d <<= 1) {
                const int o = __shfl_up(n, d);
                if ((int)threadIdx.x >= d) n += o;
            }
            base[threadIdx.x + 1] = n;
            if (threadIdx.x == 0) base[0] = 0;
        }
        __syncthreads();
        const int all = base[ns];
        // offset and step of entry m of the list (complemented: less), false where its JL is not
        // in the round
        auto entry = [&](int m, long long &o, int &rows) __attribute__((always_inline)) {
            int s = 0;
            while (base[s + 1] <= m) s++;
            const TxSrc &q = A.src[t.src0 + s0 + s];
            rows = q.La * ntc;
            long long J = il, row = q.La - 1;
            bool neg = false;
            if (!q.diag || m + 1 < base[s + 1]) {
                const long long e = e00 + first[s] + (m - base[s]);
                const int2 en = S.e1[e];
                J = en.x - q.ls0;
                row = q.r0 + S.rk[e];
                neg = en.y & (1 << 12);
            }
            if (PART) J -= q.j0;
            o = q.ebase + J * t.nw * rows + row * ntc;
            if (neg) o = ~o;
            return !PART || (unsigned long long)J < (unsigned long long)q.nj;
        };
        if (!PART) {
            for (int m0 = 0; m0 < all; m0 += TX_ENT) {
                const int n = std::min(TX_ENT, all - m0);
                if (m0) __syncthreads();
                for (int m = threadIdx.x; m < n; m += 256) {
                    long long o;
                    int rows;
                    entry(m0 + m, o, rows);
                    ent[m] = o;
                    step[m] = rows;
                }
                __syncthreads();
                if (in) acc = tx_sum(acc, E + k * R.elems + ci, ent, n, step, wi);
            }
        } else {
            for (int m0 = 0; m0 < all; m0 += 256) {
                const int m = m0 + threadIdx.x;
                long long o = 0;
                int rows = 0, n;
                const bool held = m < all && entry(m, o, rows);
                if (m0) __syncthreads();
                const int at = tx_place(held, cnt, &n);
                if (held) {
                    ent[at] = o;
                    step[at] = rows;
                }
                __syncthreads();
                if (in) acc = tx_sum(acc, E + k * R.elems + ci, ent, n, step, wi);
            }
        }
    }
    if (!in) return;
    const long long n = t.yb + (long long)il * t.nb + (long long)(t.w0 + wi) * t.nI + ib;
    (t.o ? y1 : y0)[k * N + n] += (double)acc;
}

template <typename T>
static int tx_run(int nvec, const TxDev &D, const TxPlan &P, const TxVec &V, T *E, hipStream_t st)
{
    const T *x0 = (const T *)V.x0, *x1 = (const T *)V.x1;
    for (const TxRound &R : P.ss) {
        const unsigned rp = (unsigned)(P.rmax + 15) / 16 * 16;
        const bool big = (unsigned long long)V.N * sizeof(T) >= (1ULL << 32);
        if (R.nsmall) {
            const dim3 g((unsigned)R.small, nvec);
            const unsigned rs = TX_RSMALL;
            if (big) hipLaunchKernelGGL((k_tx_ess<T, true, 2>), g, dim3(256), rs * 12, st, D, R, R.i0, R.nsmall, V.N, x0, x1, E);
            else hipLaunchKernelGGL((k_tx_ess<T, false, 2>), g, dim3(256), rs * 8, st, D, R, R.i0, R.nsmall, V.N, x0, x1, E);
            TX_CHECK();
        }
        if (R.ni > R.nsmall) {
            const dim3 g((unsigned)R.items, nvec);
            const int i0 = R.i0 + R.nsmall, ni = R.ni - R.nsmall;
            if (big) hipLaunchKernelGGL((k_tx_ess<T, true, 4>), g, dim3(256), rp * 12, st, D, R, i0, ni, V.N, x0, x1, E);
            else hipLaunchKernelGGL((k_tx_ess<T, false, 4>), g, dim3(256), rp * 8, st, D, R, i0, ni, V.N, x0, x1, E);
            TX_CHECK();
        }
        if (R.part)
            hipLaunchKernelGGL((k_tx_gss<T, true>), dim3((unsigned)R.blocks, nvec), dim3(256), 0, st, D, R,
                               V.N, E, V.y0, V.y1);
        else
            hipLaunchKernelGGL((k_tx_gss<T, false>), dim3((unsigned)R.blocks, nvec), dim3(256), 0, st, D, R,
                               V.N, E, V.y0, V.y1);
        TX_CHECK();
    }
    const int ldt = P.ldt + TxV<T>::PAD;
    for (const TxRound &R : P.ab) {
        // the vectors share a wave's fragments where there are waves enough without them
        const int kper = R.items >= 8192 ? nvec : 1;
        hipLaunchKernelGGL(k_tx_eab<T>,
                           dim3(tx_grid((R.items + 3) / 4), (nvec + kper - 1) / kper),
                           dim3(256), (unsigned)(64 * ldt * sizeof(T)), st, D, R, nvec, kper, V.N, x0,
                           x1, E, ldt);
        TX_CHECK();
        if (R.part)
            hipLaunchKernelGGL((k_tx_gab<T, true>), dim3((unsigned)R.blocks, nvec), dim3(256), 0, st, D, R,
                               V.N, E, V.y0, V.y1);
        else
            hipLaunchKernelGGL((k_tx_gab<T, false>), dim3((unsigned)R.blocks, nvec), dim3(256), 0, st, D, R,
                               V.N, E, V.y0, V.y1);
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
