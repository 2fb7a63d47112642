// Contraction form of the sigma on truncated spaces (several group blocks).
//
// Both parts of the Hamiltonian are written as products of dense integral blocks with
// gathered vector rows, so that the matrix cores do the work and an entry of the vector is
// read a few dozen times instead of once per connected pair.
//
// Same-spin part (one-electron part and diagonal included).  With K2 a string of N - 2
// electrons and a pair p = (i < j) of its empty orbitals,
//
//   D[q][K2, J'] = sign X(K2 + q, J')                 (rows of the vector)
//   E[p][K2, J'] = sum_q W(p, q) D[q][K2, J']         (MFMA; rows and columns: the pairs of
//                                                      K2 whose strings the block allows)
//   sigma(I, J') += sum_{p in I} sign E[p][I - p, J'] (a string has N (N - 1) / 2 pairs)
//   W((i,j),(k,l)) = (ik|jl) - (il|jk)
//                    + (h_ik d_jl - h_il d_jk - h_jk d_il + h_jl d_ik) / (N - 1)
//
// Two strings that differ by a double share one K2, by a single N - 1 and equal ones
// N (N - 1) / 2 of them, which is how often the spectators of their elements are counted.
// J' is the other spin's string, so the vector's rows are contiguous: alpha on the vector,
// beta on its block-transposed copy.
//
// Opposite-spin part.  Each connection (p, q) <- (p1, q1) of group blocks is contracted with
// one spin first and the other last, through strings (last spin of the source, first spin of
// the target), whichever order has the fewer of them:
//
//   D[Q][JL, IF] = sum_{JF: <IF|B_Q|JF> != 0} sign X(JL, JF)
//   E[P][JL, IF] = sum_Q (P|Q) D[Q][JL, IF]
//   sigma(IL, IF) += sum_{(JL, P) in the singles of IL} sign E[P][JL, IF]
//
// with B_Q = E_kl + E_lk of the pair Q = (k, l) and the diagonal pairs for the Coulomb terms.
// The connections that share (JL's group, IF's group) and their source groups form one task.
// A task's columns are the strings of IF's group, taken 16 internal (doubly occupied + active)
// parts at a time for one external part: all of them reach the same short list of pairs Q
// (the internal pairs, and those of the external part's orbitals), which is the reduction
// index.  The rows are the singles of JL towards the target groups, plus one for JL's own
// diagonal pairs together.
//
// Against the table kernels (one gather per connected entry, sigma_fast.hip), whole products:
// MRCI-SD 16e/28o FP64 one vector 304 -> 90 ms, 16e/20o FP64 three vectors 108 -> 52 ms, FP32
// two vectors 56 -> 21 ms, 7a6b/17o two vectors 3.3 -> 1.28 ms, 4a4b/10o 259 -> 44 us; error
// against 64 bits 2.4e-15 -> 3.3e-16 (FP64) and 1.2e-6 -> 7.9e-8 (FP32) at 16e/20o.
#pragma once
#include "jci_internal.h"
#include "sigma_fast.h"

#define TX_MAXG2 64          // groups of N - 2 electron strings per spin
#define TX_MAXSEC 8          // target groups of a single excitation (7)
#define TX_NTYPE 6           // orbital-pair types dd, da, dv, aa, av, vv
#define TX_KC 96             // reduction depth of one LDS tile (four waves: 50 KB in FP64)
// column tiles x chunks of one wave's item at most (about): fragments are loaded once per item,
// and short items let a launch end evenly (8, 64 and no limit were 1 - 4 % slower)
#define TX_PASSES 32
// rows of E a wave holds integral fragments for: two row tiles leave three (FP64) or four waves
// a SIMD.  More rows per scattered tile at two waves: 16e/28o FP64 93 -> 97 ms; 48 at three in
// FP32, two vectors 16e/20o: 22.0 -> 22.7 ms
#define TX_ROWS 32
// Spaces that keep the table kernels: those with few internal orbitals and many excitations, whose
// column tiles of 16 internal parts are mostly padding and whose blocks are few and large, which
// the tables suit.  Estimated times, FP64, one vector: an element of the intermediate 16 ps
// (opposite spin) and 7 ps (same spin); the tables 1.1 ps per opposite-spin connection and 0.25 us
// per connection of the best connected determinant, one after another.  Estimated and measured
// speed of the contraction form relative to the tables (FP64, one vector / three): 2a2b in 60
// orbitals (2 active, 4 excitations) 0.53, 0.23 / 0.24 (186 against 44 ms); 4a4b/20 (2, 6) 0.32,
// 0.31 / 0.29 (37.8 against 11.9); 5a5b/18 (4, 6) 0.81, 0.81 / 0.86 (31.9 against 25.9); 3a3b/20 (2,
// 4) 0.96, 1.01 / 0.72 (0.96 both); on the other side 4a4b/24 (4, 4) 1.17, 1.59 / 1.36 (6.7 against
// 10.6), 7a7b/14 (2 doubly occupied + 10, 2) 1.40, 2.49 / 1.58 (5.9 against 14.7), 16e/20o 1.89,
// 2.93 / 2.07 (18 against 53).  Of 87 spaces none on the tables' side was more than 1.1 times
// faster in the contraction form (FP64), none on the other more than 1.15 times slower.
#define TX_COST_AB 16e-12
#define TX_COST_SS 7e-12
#define TX_COST_ENTRY 1.1e-12
#define TX_COST_CHAIN 0.25e-6
// work-groups of a launch: 256 threads each, and a grid holds fewer than 2^32 threads
#define TX_GRID ((1LL << 24) - 1024)
#define TX_PAD 0x7FF00000u   // list entry of a padded row or column (no position, string 0)

// Order of the vectors' columns.  Inside a block's row the strings of the first spin are kept
// external part outermost (column w * nI + internal part, tx_col below), so that the targets of
// a column tile, which share few external parts, are neighbours in memory; the vectors are
// brought into this order, and their transpose likewise, on the way in, and back on the way out.

// list entry of the first spin: column of the target string in its group (bits 0..19), position
// of the pair in its class (20..30), sign (31)
#define TX_JBITS 20
#define TX_KMAX 0x7FF

// Classes of orbital pairs that a string's replacements reach: internal pairs; pairs of an
// external orbital of the string with any external one; an external orbital of the string with
// an internal one (the target has one external electron less); any external orbital with an
// internal one (one more).  A section of a list holds the replacements of one class towards one
// target group.
#define TX_II 0
#define TX_EE 1
#define TX_DEC 2
#define TX_INC 3

// lists of one first-spin group: per external part `rows` rows of nIp entries, every section
// padded to a multiple of four rows
struct TxList {
    long long base;                  // first entry
    int rows, nI, nIp, nsv;
    int nsec;
    int grp[TX_MAXSEC + 4], cls[TX_MAXSEC + 4];
    int own[TX_MAXSEC + 4];          // 1: the diagonal pairs (k, k) of the string's electrons
    int first[TX_MAXSEC + 4];        // first single of the section towards its group, in table order
    int row0[TX_MAXSEC + 4], cnt[TX_MAXSEC + 4];
    int nf;                          // TX_INC: external orbitals to go to; a section's rows run
                                     // over them with the leaving orbital inside
};

// four list rows of a task's chunk: where their targets sit in the vector and in the chunk.
// The rows' positions [k0, k0 + len) of their class are steps [base, base + len) of the chunk.
struct TxSlot {
    long long xb;                    // block offset of (JL's group, target group)
    int nb;                          // strings of the target group (stride of JL)
    int lrow;                        // first list row
    int kinfo;                       // base | len << 8 | k0 << 16
    int pad;
};
// at most TX_KC steps of a task's reduction; the chunks of a task add to E one after another
struct TxChunk {
    int KS;                          // reduction steps of 4 (a multiple of 4)
    int slot0, nslot;
    int q0;                          // pair Q of step s of external part w: q[q0 + w * 4 KS + s]
};

struct TxTask {
    int o;                           // 0: beta first, alpha last (the vector); 1: the reverse
    int l1, f;                       // groups of JL and IF
    int na, ls0;                     // strings of JL's group, the first one
    int nI, nIp, nsv;                // internal parts of IF's group (padded to 16), external
    int La;                          // rows of E
    int ch0, nch;                    // chunks of the reduction
    int lrows;                       // rows of the list
    int diag;                        // last row: JL's diagonal pairs
    int nsec, sg[TX_MAXSEC], sr0[TX_MAXSEC];   // target groups and their first rows
    int iI0, nsvL;                   // first internal part of l1 in the diagonal-row table,
                                     // external parts of JL's group
    long long lbase;
};

// one task's share of a round (a range of columns, of one column tile also a range of strings JL,
// small enough that E fits its buffer)
struct TxItem {
    int task, w0, nw, t0, nt;        // external parts, column tiles of the item
    int p0, pn;                      // column tiles of the whole piece (rows of E)
    int j0, nj;                      // strings JL
    int rg;                          // row groups
    long long item0;                 // first item of the round's launch: (JL, w, row group)
    long long ebase;                 // first element in E
};

// target block of a round's gather: sources are consecutive entries of the TxSrc table
struct TxOut {
    int o, p, f;                     // last-spin group, first-spin group
    int na, ls0, nI, nIp, nsv;
    int w0, nw, t0, nt;
    int src0, nsrc;
    int nb;                          // strings of the first-spin group
    long long yb;                    // block offset
    long long blk0;                  // first work-group of the launch
    int cblk;                        // work-groups per string
};
struct TxSrc {
    int l1, ls0, La, r0, diag;       // JL's group and its first string, rows, first row of this
                                     // target (-1: none); diag 1: also JL = IL
    int j0, nj;                      // strings of JL's group that the round holds
    long long ebase;
};

// ---- same-spin part ----
struct TxPairGroup {                 // group of N - 2 electron strings
    int d, a, v;
    long long n, base;               // strings; first list entry
    int R;                           // list entries per string
    int off[TX_NTYPE], cnt[TX_NTYPE], tgt[TX_NTYPE];   // per pair type: first, count, group (-1)
};
struct TxPairTask {
    int o, g2, f;                    // orientation, N - 2 group, column group
    int R;                           // pairs (rows and reduction index)
    int nsec, so[TX_NTYPE], sc[TX_NTYPE], sr[TX_NTYPE];  // list offset, count, first row
    long long sx[TX_NTYPE];          // vector offset of the section's strings
    long long lbase;                 // list base of the group
    int Rfull, n, nb;
};
#define TX_RSMALL 32         // pairs up to which a work-group has two row tiles, in rounds of at
#define TX_SMALL_GROUPS 4096 // least so many such work-groups (fewer are not worth a launch)
#define TX_RMAX 64           // pairs up to which a work-group keeps all of W in LDS
struct TxPairItem {
    int task, c0, nc, ncp;           // columns of the round, padded to 16
    int k0, nk;                      // N - 2 electron strings
    int rg, cb, ct;                  // row groups of 64, column blocks of 64 per work-group,
                                     // work-groups across
    long long item0, ebase;
};
struct TxPairOut {
    int o, p, f, na, ls0, nb;
    int c0, nc, ncp, cblk;
    long long yb, blk0;
    int nsec, np[TX_NTYPE], r0[TX_NTYPE], R[TX_NTYPE];   // pairs of I per type, rows of E
    long long eb[TX_NTYPE];
    // rounds in part: 1 adds to the result; first pair of the type in the string's list, N - 2
    // strings that the round holds
    int add, g0[TX_NTYPE], k0[TX_NTYPE], nk[TX_NTYPE];
};

// one spin's lists (device)
struct TxSpin {
    const uint64_t *mask;
    const long long *off1;
    const int2 *e1;
    const int *goff1;
    const uint32_t *lst;             // TxList lists of all groups
    const uint16_t *rk;              // per entry of e1: its reverse's position among the
                                     // target's singles towards this string's group
    const int2 *kl;                  // per N - 2 string: pairs {string in its group,
                                     // pair | sign << 31}
    const int2 *gl;                  // per string: its pairs {N - 2 string in its group,
                                     // position in the type | sign << 31}
    int npair;                       // N (N - 1) / 2
    int G;
    const double *w64;               // W, (np + 1) x (np + 1), the last row and column zero
    const float *w32;
    // integral rows of ms = m1 + 1 elements, the last one zero: (P|.) of every pair, then per
    // internal part the sum of (kk|.) over its electrons, then a row of zeros
    const double *m64;
    const float *m32;
    int zrow;                        // the row of zeros
};

struct TxDev {
    TxSpin s[2];
    const TxTask *task;
    const TxSlot *slot;
    const TxChunk *chunk;
    const TxItem *item;
    const TxOut *out;
    const TxSrc *src;
    const TxPairTask *ptask;
    const TxPairItem *pitem;
    const TxPairOut *pout;
    const int *q;
    int m1, ms, np, nint;
};

// one launch pair (E, gather) of either part
struct TxRound {
    int i0, ni, o0, no;              // items and outputs in their tables
    int part;                        // 1: some strings of a source only, or results to add to
    int nsmall;                      // same spin: first items, strings of up to TX_RSMALL pairs
    long long small;                 // their work-groups
    long long items, blocks;         // waves (opposite spin) or work-groups (same spin); gather
                                     // work-groups
    long long elems;                 // elements of E
};

// index arithmetic shared by the device kernels and host checks -------------------------------
#include "slater.h"

// orbital subspace of orbital x: 0 doubly occupied, 1 active, 2 external
JCI_HD int tx_sub(const SpaceDesc *d, int x)
{
    return x < d->ndocc ? 0 : x < d->ndocc + d->nactv ? 1 : 2;
}
JCI_HD uint64_t tx_submask(const SpaceDesc *d, int s)
{
    return s == 0 ? d->dmask : s == 1 ? d->amask : d->vmask;
}
JCI_HD uint64_t tx_below(int x) { return (1ULL << x) - 1ULL; }
JCI_HD int tx_type(int s0, int s1)   // s0 <= s1
{
    return s0 == 0 ? s1 : s0 == 1 ? 2 + s1 : 5;
}

// column of string loc of a group of nI internal x nsv external parts
JCI_HD long long tx_col(long long loc, int nI, int nsv) { return loc % nsv * nI + loc / nsv; }

// position of the single excitation x -> y of string m among its singles towards their target
// group (enumeration order of the excitation tables: x ascending, then y ascending)
JCI_HD int tx_single_rank(const SpaceDesc *d, uint64_t m, int x, int y)
{
    const int sx = tx_sub(d, x), sy = tx_sub(d, y);
    const uint64_t mx = tx_submask(d, sx), my = tx_submask(d, sy);
    const int occ = jci_popc(m & mx & tx_below(x));
    const int emp = jci_popc(~m & my & tx_below(y));
    int r = occ * jci_popc(~m & my & d->allmask) + emp;
    if (sx == sy)   // the three subspaces' own replacements share the target group
        for (int s = 0; s < sx; s++) {
            const uint64_t ms = tx_submask(d, s);
            r += jci_popc(m & ms) * jci_popc(~m & ms & d->allmask);
        }
    return r;
}

// position of the pair (x, y) in its class for a string with external part ext
JCI_HD int tx_kpos(const SpaceDesc *d, uint64_t ext, int cls, int x, int y)
{
    const int nint = d->ndocc + d->nactv;
    const int hi = x > y ? x : y, lo = x > y ? y : x;
    if (cls == TX_II) return hi * (hi + 1) / 2 + lo;
    if (cls == TX_INC) return (hi - nint) * nint + lo;
    if (cls == TX_DEC) return jci_popc(ext & tx_below(hi)) * nint + lo;
    const int b = (ext >> hi) & 1 ? hi : lo, c = b == hi ? lo : hi;
    return jci_popc(ext & tx_below(b)) * d->nvirt + (c - nint);
}

// its inverse: pair index tri of position s of a class for the external orbitals extorb
JCI_HD int tx_kpair(int nint, int nv, const int *extorb, int cls, int s)
{
    if (cls == TX_II) return s;
    if (cls == TX_EE) return (int)jci_tri(extorb[s / nv], nint + s % nv);
    if (cls == TX_DEC) return (int)jci_tri(extorb[s / nint], s % nint);
    return (int)jci_tri(nint + s / nint, s % nint);
}

// positions of a class for a string with v external electrons
JCI_HD int tx_class_size(int nint, int nv, int v, int cls)
{
    return cls == TX_II ? nint * (nint + 1) / 2 : cls == TX_EE ? v * nv : cls == TX_DEC ? v * nint : nv * nint;
}

// Numbering of orbital pairs i < j by type, the second orbital fastest in the mixed types: the
// pairs a string's list walks in order are then mostly consecutive columns of W.
JCI_HD int tx_pair_id(const SpaceDesc *d, int i, int j)
{
    const int n[3] = {d->ndocc, d->nactv, d->nvirt}, o[3] = {0, d->ndocc, d->ndocc + d->nactv};
    const int si = tx_sub(d, i), sj = tx_sub(d, j), a = i - o[si], b = j - o[sj];
    int base = 0;
    for (int s = 0; s < 3; s++)
        for (int t = s; t < 3; t++) {
            if (s == si && t == sj) return base + (s == t ? b * (b - 1) / 2 + a : a * n[t] + b);
            base += s == t ? n[s] * (n[s] - 1) / 2 : n[s] * n[t];
        }
    return -1;
}

// its inverse
JCI_HD void tx_pair_orbs(const SpaceDesc *d, int P, int *i, int *j)
{
    const int n[3] = {d->ndocc, d->nactv, d->nvirt}, o[3] = {0, d->ndocc, d->ndocc + d->nactv};
    for (int s = 0; s < 3; s++)
        for (int t = s; t < 3; t++) {
            const int c = s == t ? n[s] * (n[s] - 1) / 2 : n[s] * n[t];
            if (P >= c) {
                P -= c;
                continue;
            }
            if (s != t) {
                *i = o[s] + P / n[t];
                *j = o[t] + P % n[t];
                return;
            }
            int b = 1;
            while ((b + 1) * b / 2 <= P) b++;
            *i = o[s] + P - b * (b - 1) / 2;
            *j = o[s] + b;
            return;
        }
    *i = *j = 0;
}

// pair i < j of string m: the N - 2 string's mask, the pair's type, its position in the type's
// section of that string's list and the sign of a_j a_i
JCI_HD void tx_pair(const SpaceDesc *d, uint64_t m, int i, int j, uint64_t *k2, int *type,
                    int *idx, int *neg)
{
    const uint64_t k = m & ~(1ULL << i) & ~(1ULL << j);
    const int si = tx_sub(d, i), sj = tx_sub(d, j);
    const uint64_t mi = tx_submask(d, si), mj = tx_submask(d, sj);
    const int ei = jci_popc(~k & mi & tx_below(i)), ej = jci_popc(~k & mj & tx_below(j));
    *k2 = k;
    *type = tx_type(si, sj);
    *idx = si == sj ? ej * (ej - 1) / 2 + ei : ei * jci_popc(~k & mj & d->allmask) + ej;
    *neg = (jci_popc(m & tx_below(i)) + jci_popc(m & tx_below(j)) + 1) & 1;
}

// index of an N - 2 string in its group
JCI_HD long long tx_pair_rank(const SpaceDesc *d, uint64_t k, const unsigned long long *binom)
{
    const int nd = jci_popc(k & d->dmask), na = jci_popc(k & d->amask), nv = jci_popc(k & d->vmask);
    const int si = d->ndocc + d->nactv;
    const long long rd = jci_lex_rank(k & d->dmask, d->ndocc, nd, binom);
    const long long ra = jci_lex_rank(d->ndocc >= 64 ? 0 : (k & d->amask) >> d->ndocc, d->nactv, na, binom);
    const long long rv = jci_lex_rank(si >= 64 ? 0 : (k & d->vmask) >> si, d->nvirt, nv, binom);
    return (rd * (long long)binom[d->nactv * 65 + na] + ra) * (long long)binom[d->nvirt * 65 + nv] + rv;
}

// host tables of the contraction form: lists, tasks and rounds (tx_plan.cpp)
#include <vector>
struct TxPlan {
    std::vector<TxList> lists[2];          // per spin and group
    long long nlst[2];                     // list entries per spin
    std::vector<TxPairGroup> pg[2];
    long long nkl[2];                      // pair-list entries per spin
    std::vector<TxTask> task;
    std::vector<TxSlot> slot;
    std::vector<TxChunk> chunk;
    std::vector<TxItem> item;
    std::vector<TxOut> out;
    std::vector<TxSrc> src;
    std::vector<TxPairTask> ptask;
    std::vector<TxPairItem> pitem;
    std::vector<TxPairOut> pout;
    std::vector<int> q;
    std::vector<TxRound> ab, ss;           // rounds of the two parts
    long long elems, total;                // largest E of a round, sum over the rounds
    long long sum[2];                      // of the opposite-spin and the same-spin rounds
    long long grid;                        // most work-groups of a launch
    int split[5];                          // pieces that start past the first external part, column
                                           // tile, JL (opposite spin), column, N - 2 string (same spin)
    int ldt, rmax;                         // deepest reduction chunk; most pairs of a task
    long long nint_parts[2];               // internal parts over all groups
    int iI0[2][JCI_MAXG];
};
// budget: bound on a round's E (what one string of a task needs for one column tile, or one N - 2
// electron string for 64 columns, where that is more).
// 0: built; 1: the space is outside what the lists can index, or the tables are faster on it (the
// caller keeps them)
int tx_plan(const SpaceDesc &D, const SpaceDesc &T, long long budget, TxPlan *P);

// ---- kernels (sigma_tx.hip) ----
int jk_tx_lists(const SpaceDesc *d, int spin, long long nstr, const uint64_t *mask,
                const long long *off1, const int2 *e1, const int *goff1, const TxList *lists,
                uint32_t *lst, uint16_t *rk, hipStream_t st);
int jk_tx_fill(long long n, uint32_t *p, hipStream_t st);
int jk_tx_pairs(const SpaceDesc *d, int spin, long long nstr, const uint64_t *mask,
                const unsigned long long *binom, const TxPairGroup *pg, int npg, int npair,
                int2 *kl, int2 *gl, hipStream_t st);
int jk_tx_w(const SpaceDesc *d, int norb, int nelec, const double *m1, const double *m2,
            double *w64, float *w32, hipStream_t st);
int jk_tx_rows(const SpaceDesc *d, const SpaceDesc &h, int spin, const uint64_t *mask, int m1,
               const double *m2sq, const TxPlan &P, double *m64, float *m32, hipStream_t st);
// x (vector k at x + k * xk, element n at n * xs) -> x0 and x1 (every block transposed), both in
// the arithmetic type, vectors of stride N, columns in tx_col order; tt: first 16 x 16 tile of
// each block (tx_tiles)
int jk_tx_in(int prec, int nvec, long long N, const SpaceDesc *d, const long long *tt, long long ntt,
             const double *x, long long xs, long long xk, void *x0, void *x1, hipStream_t st);
// y = y0 and the transposed blocks of y1, in the caller's order
int jk_tx_out(int nvec, long long N, const SpaceDesc *d, const long long *tt, long long ntt,
              const double *y0, const double *y1, double *y, long long ys, long long yk,
              hipStream_t st);
// the rounds of both parts on vectors of stride N
struct TxVec {
    const void *x0, *x1;
    double *y0, *y1;
    long long N;
};
int jk_tx_run(int prec, int nvec, const TxDev &D, const TxPlan &P, const TxVec &V, void *E,
              hipStream_t st);
