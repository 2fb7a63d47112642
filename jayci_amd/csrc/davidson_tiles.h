// Device parts that the Davidson vector kernels of one solve (kernels.hip) and of a batch
// (batch_kernels.hip) share: the Gram products and the rows of a residual.
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>
#include "jci_internal.h"
#include "mfma.h"

// two consecutive elements at an address aligned to one
typedef double DvTwo __attribute__((ext_vector_type(2), aligned(8)));

// acc += A^T B over the rows r0 + 16 (s0 + q ds) < r1, A of m and B of w columns (leading
// dimensions lda, ldb), by one wave on MT x WT tiles of 16 x 16.  Lane l holds column l % 16 of
// a tile and the four rows 4 (l / 16) .. + 3 of a step, 32 bytes of one column: the operands
// come straight from memory in 128-byte runs, the next step's during the products of this one.
// Columns past the last repeat it (their products are not written).
//
// Bound by the reads of A and B (m <= 64 columns: at most 16 products per element read).  Gram
// products of a two-root solve (one buffer pair) of 6a6b in 14 orbitals: 150 launches of 9.2 -> 1.9 ms in all
// (32-row tiles through LDS, one work-group per 2048 rows, before); of a batch of 12 full-CI
// solves in 8 to 12 orbitals: 8.4 -> 5.6 ms.
template <int MT, int WT>
__device__ __forceinline__ void gram_wave(Mf<double>::acc (&acc)[MT][WT], int m, int w,
                                          const double *A, long long lda, const double *B,
                                          long long ldb, long long r0, long long r1, int s0, int ds)
{
    typedef const __attribute__((address_space(1))) DvTwo *TP;
    const int l = threadIdx.x & 63, col = l & 15, part = l >> 4;
    const __attribute__((address_space(1))) double *ap[MT], *bp[WT];
#pragma unroll
    for (int i = 0; i < MT; i++) ap[i] = gptr(A) + (long long)(i * 16 + col < m ? i * 16 + col : m - 1) * lda + part * 4;
#pragma unroll
    for (int j = 0; j < WT; j++) bp[j] = gptr(B) + (long long)(j * 16 + col < w ? j * 16 + col : w - 1) * ldb + part * 4;
    double a[2][MT][4], b[2][WT][4];
    auto load = [&](long long r, double (&x)[MT][4], double (&y)[WT][4]) __attribute__((always_inline)) {
        if (r + 16 <= r1) {
#pragma unroll
            for (int h = 0; h < 4; h += 2) {
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const DvTwo v = *(TP)(ap[i] + r + h);
                    x[i][h] = v[0];
                    x[i][h + 1] = v[1];
                }
#pragma unroll
                for (int j = 0; j < WT; j++) {
                    const DvTwo v = *(TP)(bp[j] + r + h);
                    y[j][h] = v[0];
                    y[j][h + 1] = v[1];
                }
            }
        } else {
#pragma unroll
            for (int h = 0; h < 4; h++) {
                const bool in = r + part * 4 + h < r1;
#pragma unroll
                for (int i = 0; i < MT; i++) x[i][h] = in ? ap[i][r + h] : 0.0;
#pragma unroll
                for (int j = 0; j < WT; j++) y[j][h] = in ? bp[j][r + h] : 0.0;
            }
        }
    };
    auto mul = [&](const double (&x)[MT][4], const double (&y)[WT][4]) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 4; h++)
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < WT; j++) acc[i][j] = Mf<double>::mma(x[i][h], y[j][h], acc[i][j]);
    };
    const long long step = 16LL * ds;
    long long r = r0 + 16LL * s0;
    if (r < r1) load(r, a[0], b[0]);
    for (; r < r1; r += 2 * step) {
        if (r + step < r1) load(r + step, a[1], b[1]);
        mul(a[0], b[0]);
        if (r + step >= r1) break;
        if (r + 2 * step < r1) load(r + 2 * step, a[0], b[0]);
        mul(a[1], b[1]);
    }
}

// the block's four waves over rows [r0, r1), their sums added in a fixed order through `red`
// (1024 elements) and written to out[i * ldo + j], i < m, j < w
template <int MT, int WT>
__device__ __forceinline__ void gram_block(int m, int w, const double *A, long long lda, const double *B,
                                           long long ldb, long long r0, long long r1, double *out,
                                           int ldo, double *red)
{
    const int l = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Mf<double>::acc acc[MT][WT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < WT; j++) acc[i][j] = Mf<double>::zero();
    gram_wave<MT, WT>(acc, m, w, A, lda, B, ldb, r0, r1, wave, 4);
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < WT; j++) {
            __syncthreads();
#pragma unroll
            for (int v = 0; v < 4; v++) red[wave * 256 + v * 64 + l] = acc[i][j][v];
            __syncthreads();
            // thread: element `wave` of lane l
            const double s = (red[wave * 64 + l] + red[256 + wave * 64 + l]) +
                             (red[512 + wave * 64 + l] + red[768 + wave * 64 + l]);
            const int row = i * 16 + Mf<double>::row(l, wave), c = j * 16 + (l & 15);
            if (row < m && c < w) out[row * ldo + c] = s;
        }
}

// one row of K residuals: res_r = sum_i C[i * K + r] (S_i - th_r V_i), written as the corrections
// -res_r / (h - th_r); the squares are added to nrm.  Eight basis vectors' loads at a time, the
// sums in registers (K a constant).  Bound by the reads of V and S: 39 residuals of the solve
// above 2.06 -> 0.68 ms, 47 of the batch 5.2 -> 4.5 ms.
template <int K>
__device__ __forceinline__ void residual_row(int m, const double *__restrict__ V,
                                             const double *__restrict__ S, long long ld, long long n,
                                             const double *C, const double *th, double h,
                                             double *__restrict__ T, double (&nrm)[K])
{
    constexpr int U = 8;
    const auto Vg = gptr(V) + n, Sg = gptr(S) + n;
    double res[K], t[K];
#pragma unroll
    for (int r = 0; r < K; r++) {
        res[r] = 0.0;
        t[r] = th[r];
    }
    int i = 0;
    for (; i + U <= m; i += U) {
        double v[U], s[U];
#pragma unroll
        for (int q = 0; q < U; q++) {
            v[q] = Vg[(i + q) * ld];
            s[q] = Sg[(i + q) * ld];
        }
#pragma unroll
        for (int q = 0; q < U; q++)
#pragma unroll
            for (int r = 0; r < K; r++) res[r] += C[(i + q) * K + r] * (s[q] - t[r] * v[q]);
    }
    for (; i < m; i++) {
        const double v = Vg[i * ld], s = Sg[i * ld];
#pragma unroll
        for (int r = 0; r < K; r++) res[r] += C[i * K + r] * (s - t[r] * v);
    }
    const auto Tg = gptr_w(T) + n;
#pragma unroll
    for (int r = 0; r < K; r++) {
        nrm[r] += res[r] * res[r];
        double den = h - t[r];
        if (fabs(den) < 1e-8) den = den < 0 ? -1e-8 : 1e-8;
        Tg[r * ld] = -res[r] / den;
    }
}

// K residuals over the rows [r0, r1) by a work-group of 256; out[r]: sums of squares (fixed order)
template <int K>
__device__ __forceinline__ void residual_block(int m, const double *V, const double *S, long long ld,
                                               long long r0, long long r1, const double *C,
                                               const double *th, const double *hd, double *T,
                                               double *out, double *red)
{
    double nrm[K];
#pragma unroll
    for (int r = 0; r < K; r++) nrm[r] = 0.0;
    for (long long n = r0 + threadIdx.x; n < r1; n += 256)
        residual_row<K>(m, V, S, ld, n, C, th, gptr(hd)[n], T, nrm);
    // waves by shuffles, then the four waves' sums
#pragma unroll
    for (int r = 0; r < K; r++) {
        for (int o = 32; o > 0; o >>= 1) nrm[r] += __shfl_xor(nrm[r], o);
        if ((threadIdx.x & 63) == 0) red[r * 4 + (threadIdx.x >> 6)] = nrm[r];
    }
    __syncthreads();
    if (threadIdx.x < K)
        out[threadIdx.x] = (red[threadIdx.x * 4] + red[threadIdx.x * 4 + 1]) +
                           (red[threadIdx.x * 4 + 2] + red[threadIdx.x * 4 + 3]);
}

// f(integral constant k) for the k of 1 .. 8 that equals `k`
template <typename F> __host__ __device__ __forceinline__ void with_k(int k, F f)
{
    static_assert(JCI_MAXK == 8, "one case per number of vectors");
    switch (k) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    default: f(std::integral_constant<int, 8>{}); break;
    }
}
