// Host tables of the contraction form of the truncated-space sigma (see sigma_tx.h): lists,
// tasks, and the rounds that keep the intermediates inside a buffer.
#include "sigma_tx.h"
#include <algorithm>
#include <map>
#include <set>
#include <string.h>

typedef long long ll;

static ll choose(int n, int k)
{
    if (k < 0 || n < 0 || k > n) return 0;
    ll r = 1;
    for (int i = 1; i <= k; i++) r = r * (n - k + i) / i;
    return r;
}

// singles of one string of group g to strings of group h of the same spin; -1: no single
// excitation leads there
static ll singles(const SpaceDesc &D, const SpinDesc &S, int g, int h)
{
    const int size[3] = {D.ndocc, D.nactv, D.nvirt};
    const int o[3] = {S.gd[g], S.ga[g], S.gv[g]}, t[3] = {S.gd[h], S.ga[h], S.gv[h]};
    if (g == h) return o[0] * (size[0] - o[0]) + o[1] * (size[1] - o[1]) + o[2] * (size[2] - o[2]);
    int from = -1, to = -1;
    for (int s = 0; s < 3; s++) {
        if (t[s] == o[s]) continue;
        if (t[s] == o[s] - 1 && from < 0) from = s;
        else if (t[s] == o[s] + 1 && to < 0) to = s;
        else return -1;
    }
    if (from < 0 || to < 0) return -1;
    return (ll)o[from] * (size[to] - o[to]);
}

static ll up(ll n, ll m) { return (n + m - 1) / m * m; }

// lists of one spin as the first spin of a task
static int plan_lists(const SpaceDesc &D, const SpinDesc &S, std::vector<TxList> &L, ll *total)
{
    ll base = 0;
    for (int g = 0; g < S.ngrp; g++) {
        TxList t;
        memset(&t, 0, sizeof(t));
        t.base = base;
        t.nsv = (int)std::max(1LL, S.nsv[g]);
        t.nI = (int)(S.gn[g] / t.nsv);
        t.nIp = (int)up(t.nI, 16);
        const int v = S.gv[g], nint_e = S.nelec - v;
        auto add = [&](int h, int cls, int own, int first, int cnt) {
            if (cnt <= 0) return;
            t.grp[t.nsec] = h;
            t.cls[t.nsec] = cls;
            t.own[t.nsec] = own;
            t.first[t.nsec] = first;
            t.row0[t.nsec] = t.rows;
            t.cnt[t.nsec] = cnt;
            t.rows += (int)up(cnt, 4);
            t.nsec++;
        };
        t.nf = D.nvirt - v;
        for (int h = 0; h < S.ngrp; h++) {
            if (!S.gn[h] || !S.gn[g]) continue;
            const int c = (int)singles(D, S, g, h);
            if (c <= 0) continue;
            if (t.nsec >= TX_MAXSEC) return 1;
            if (h == g) {
                // table order: internal replacements, then the external ones
                const int ee = v * (D.nvirt - v);
                add(h, TX_II, 0, 0, c - ee);
                add(h, TX_EE, 0, c - ee, ee);
            } else {
                add(h, S.gv[h] == v ? TX_II : S.gv[h] < v ? TX_DEC : TX_INC, 0, 0, c);
            }
        }
        add(g, TX_II, 1, 0, nint_e);
        add(g, TX_EE, 1, nint_e, v);
        if (S.gn[g] >= (1LL << TX_JBITS)) return 1;
        base += (ll)t.nsv * t.rows * t.nIp;
        L.push_back(t);
    }
    *total = base;
    return 0;
}

// groups of N - 2 electron strings of one spin
static int plan_pairs(const SpaceDesc &D, const SpinDesc &S, std::vector<TxPairGroup> &P, ll *total)
{
    const int size[3] = {D.ndocc, D.nactv, D.nvirt};
    static const int ts[TX_NTYPE][2] = {{0, 0}, {0, 1}, {0, 2}, {1, 1}, {1, 2}, {2, 2}};
    ll base = 0;
    for (int g = 0; g < S.ngrp; g++) {
        if (!S.gn[g]) continue;
        for (int t = 0; t < TX_NTYPE; t++) {
            int o[3] = {S.gd[g], S.ga[g], S.gv[g]};
            o[ts[t][0]]--;
            o[ts[t][1]]--;
            if (o[0] < 0 || o[1] < 0 || o[2] < 0) continue;
            bool have = false;
            for (const TxPairGroup &k : P) have = have || (k.d == o[0] && k.a == o[1] && k.v == o[2]);
            if (have) continue;
            if ((int)P.size() >= TX_MAXG2) return 1;
            TxPairGroup k;
            memset(&k, 0, sizeof(k));
            k.d = o[0];
            k.a = o[1];
            k.v = o[2];
            k.n = choose(size[0], o[0]) * choose(size[1], o[1]) * choose(size[2], o[2]);
            k.base = base;
            for (int u = 0; u < TX_NTYPE; u++) {
                int f[3] = {o[0], o[1], o[2]};
                const int s0 = ts[u][0], s1 = ts[u][1];
                const int e0 = size[s0] - o[s0], e1 = size[s1] - o[s1];
                f[s0]++;
                f[s1]++;
                k.off[u] = k.R;
                k.tgt[u] = -1;
                for (int h = 0; h < S.ngrp; h++)
                    if (S.gn[h] && S.gd[h] == f[0] && S.ga[h] == f[1] && S.gv[h] == f[2]) k.tgt[u] = h;
                if (k.tgt[u] < 0) continue;
                k.cnt[u] = s0 == s1 ? e0 * (e0 - 1) / 2 : e0 * e1;
                k.R += k.cnt[u];
            }
            if (k.n >= (1LL << 31)) return 1;
            base += k.n * k.R;
            P.push_back(k);
        }
    }
    *total = base;
    return 0;
}

namespace {
struct Builder {
    const SpaceDesc *dd[2];
    ll budget;
    TxPlan *P;
    // tasks by (orientation, first-spin group)
    std::vector<int> by[2][JCI_MAXG], pby[2][JCI_MAXG];
    std::map<std::vector<int>, int> qtab;
    unsigned long long binom[65 * 65];

    // a chunk's steps: consecutive positions of one or more classes
    struct Seg { int cls, k0, len, base; };

    // reduction-index table of a chunk for first-spin group f: its first entry
    int pair_table(const SpaceDesc &D, int f, const std::vector<Seg> &seg, int depth)
    {
        const SpinDesc &S = D.s[1];
        std::vector<int> key = {S.gv[f], depth};
        for (const Seg &g : seg) key.insert(key.end(), {g.cls, g.k0, g.len});
        auto it = qtab.find(key);
        if (it != qtab.end()) return it->second;
        const int nint = D.ndocc + D.nactv, v = S.gv[f];
        const int at = (int)P->q.size();
        const int none = D.norbs * (D.norbs + 1) / 2;   // the zero column
        const int nsv = (int)std::max(1LL, S.nsv[f]);
        for (int w = 0; w < nsv; w++) {
            int ext[64], n = 0;
            for (uint64_t m = v ? jci_lex_unrank(w, D.nvirt, v, binom) : 0; m; m &= m - 1)
                ext[n++] = nint + jci_ctz(m);
            int put = 0;
            for (const Seg &g : seg)
                for (int s = 0; s < g.len; s++, put++)
                    P->q.push_back(tx_kpair(nint, D.nvirt, ext, g.cls, g.k0 + s));
            for (; put < depth; put++) P->q.push_back(none);
        }
        qtab[key] = at;
        return at;
    }

    int tasks()
    {
        // every connection of group blocks goes to the orientation with fewer intermediates
        std::map<std::vector<int>, std::map<int, std::set<int>>> T;   // (o, l1, f) -> l -> f1 set
        const SpaceDesc &D = *dd[0];
        auto linked = [&](const SpinDesc &S, int a, int b) { return a == b || singles(D, S, a, b) > 0; };
        for (int b = 0; b < D.nblk; b++)
            for (int c = 0; c < D.nblk; c++) {
                const int p = D.bp[b], q = D.bq[b], p1 = D.bp[c], q1 = D.bq[c];
                if (!linked(D.s[0], p, p1) || !linked(D.s[1], q, q1)) continue;
                const ll n0 = D.s[0].gn[p1] * D.s[1].gn[q], n1 = D.s[0].gn[p] * D.s[1].gn[q1];
                if (n0 <= n1) T[{0, p1, q}][p].insert(q1);
                else T[{1, q1, p}][q].insert(p1);
            }
        for (auto &kv : T) {
            const int o = kv.first[0], l1 = kv.first[1], f = kv.first[2];
            const SpaceDesc &O = *dd[o];
            const SpinDesc &L = O.s[0], &F = O.s[1];
            // targets with the same source set form one task
            std::map<std::set<int>, std::vector<int>> groups;
            for (auto &t : kv.second) groups[t.second].push_back(t.first);
            const TxList &li = P->lists[o == 0 ? 1 : 0][f];
            for (auto &gr : groups) {
                TxTask t;
                memset(&t, 0, sizeof(t));
                t.o = o;
                t.l1 = l1;
                t.f = f;
                t.na = (int)L.gn[l1];
                t.ls0 = (int)L.gstart[l1];
                t.nI = li.nI;
                t.nIp = li.nIp;
                t.nsv = li.nsv;
                t.lrows = li.rows;
                t.lbase = li.base;
                t.nsvL = (int)std::max(1LL, L.nsv[l1]);
                t.iI0 = P->iI0[o == 0 ? 0 : 1][l1];
                for (int l : gr.second) {
                    const ll c = singles(O, L, l1, l);
                    if (c <= 0) continue;
                    if (t.nsec >= TX_MAXSEC) return 1;
                    t.sg[t.nsec] = l;
                    t.sr0[t.nsec] = t.La;
                    t.nsec++;
                    t.La += (int)c;
                }
                for (int l : gr.second) if (l == l1) { t.diag = 1; t.La++; break; }
                if (!t.La) continue;
                // reduction index: the classes of the sources, in chunks of at most TX_KC
                // steps; a class that does not fit what is left of a chunk opens the next
                // one, and one deeper than a chunk is split (by external orbitals for TX_INC)
                const int v = F.gv[f], nint = O.ndocc + O.nactv;
                int has[4] = {0, 0, 0, 0};
                for (int s = 0; s < li.nsec; s++) if (gr.first.count(li.grp[s])) has[li.cls[s]] = 1;
                std::vector<std::vector<Seg>> chunks(1);
                int depth = 0;
                for (int cls = 0; cls < 4; cls++) {
                    if (!has[cls]) continue;
                    const int m = tx_class_size(nint, O.nvirt, v, cls);
                    if (m >= TX_KMAX) return 1;
                    const int unit = cls == TX_INC ? nint : 1;
                    if (unit > TX_KC) return 1;
                    const int most = TX_KC / unit * unit, np = (m + most - 1) / most;
                    const int len = np ? (int)up((m + np - 1) / np, unit) : 0;
                    for (int k0 = 0; k0 < m; k0 += len) {
                        const int n = std::min(len, m - k0);
                        if (depth + n > TX_KC) {
                            chunks.push_back(std::vector<Seg>());
                            depth = 0;
                        }
                        chunks.back().push_back(Seg{cls, k0, n, depth});
                        depth += n;
                    }
                }
                t.ch0 = (int)P->chunk.size();
                for (const std::vector<Seg> &seg : chunks) {
                    TxChunk ch;
                    memset(&ch, 0, sizeof(ch));
                    int d = 0;
                    for (const Seg &g : seg) d += g.len;
                    const int kc = (int)up(d, 16);
                    ch.KS = kc / 4;
                    P->ldt = std::max(P->ldt, kc);
                    ch.q0 = pair_table(O, f, seg, kc);
                    ch.slot0 = (int)P->slot.size();
                    for (const Seg &g : seg)
                        for (int s = 0; s < li.nsec; s++) {
                            if (li.cls[s] != g.cls || !gr.first.count(li.grp[s])) continue;
                            const int blk = O.blkid[l1][li.grp[s]];
                            if (blk < 0) return 1;
                            // rows of the section that can reach the segment: all, or those of
                            // its external orbitals (whose ranks among the free ones lag by up
                            // to v)
                            int r0 = 0, r1 = li.cnt[s];
                            if (g.cls == TX_INC) {
                                const int ni = li.cnt[s] / li.nf;
                                r0 = std::max(0, g.k0 / nint - v) * ni / 4 * 4;
                                r1 = std::min(li.nf, (g.k0 + g.len + nint - 1) / nint) * ni;
                            }
                            for (int r = r0; r < r1; r += 4) {
                                TxSlot w;
                                memset(&w, 0, sizeof(w));
                                w.xb = O.boff[blk];
                                w.nb = (int)F.gn[li.grp[s]];
                                w.lrow = li.row0[s] + r;
                                w.kinfo = g.base | g.len << 8 | g.k0 << 16;
                                P->slot.push_back(w);
                            }
                        }
                    ch.nslot = (int)P->slot.size() - ch.slot0;
                    if (!ch.nslot) continue;
                    if (ch.nslot > 64) return 1;
                    P->chunk.push_back(ch);
                    t.nch++;
                }
                if (!t.nch) continue;
                by[o][f].push_back((int)P->task.size());
                P->task.push_back(t);
            }
        }
        return 0;
    }

    // one piece of a round: external parts [w0, w0 + nw) and column tiles [t0, t0 + nt) of
    // first-spin group f, for some of its tasks; nj > 0: strings JL [j0, j0 + nj) of the only task
    void piece(int o, int f, const std::vector<int> &tasks, int w0, int nw, int t0, int nt, TxRound &R,
               int j0 = 0, int nj = 0)
    {
        P->split[0] += w0 > 0;
        P->split[1] += t0 > 0;
        P->split[2] += j0 > 0;
        const SpaceDesc &O = *dd[o];
        const SpinDesc &L = O.s[0];
        std::vector<ll> eb;
        for (int ti : tasks) {
            const TxTask &t = P->task[ti];
            TxItem it;
            memset(&it, 0, sizeof(it));
            it.task = ti;
            it.w0 = w0;
            it.nw = nw;
            it.p0 = t0;
            it.pn = nt;
            it.j0 = j0;
            it.nj = nj ? nj : t.na;
            it.rg = (t.La + TX_ROWS - 1) / TX_ROWS;
            it.ebase = R.elems;
            eb.push_back(R.elems);
            R.elems += (ll)it.nj * nw * t.La * nt * 16;
            // long rows of tiles in several items: the launch's last work-groups end sooner
            const int most = std::max(2, TX_PASSES / t.nch), parts = (nt + most - 1) / most;
            for (int k = 0; k < parts; k++) {
                it.t0 = t0 + nt * k / parts;
                it.nt = t0 + nt * (k + 1) / parts - it.t0;
                P->item.push_back(it);
                R.ni++;
            }
        }
        for (int l = 0; l < L.ngrp; l++) {
            const int blk = O.blkid[l][f];
            if (blk < 0) continue;
            TxOut u;
            memset(&u, 0, sizeof(u));
            u.src0 = (int)P->src.size();
            for (size_t i = 0; i < tasks.size(); i++) {
                const TxTask &t = P->task[tasks[i]];
                TxSrc s;
                memset(&s, 0, sizeof(s));
                s.l1 = t.l1;
                s.ls0 = t.ls0;
                s.La = t.La;
                s.r0 = -1;
                s.ebase = eb[i];
                s.j0 = j0;
                s.nj = nj ? nj : t.na;
                for (int k = 0; k < t.nsec; k++) if (t.sg[k] == l) s.r0 = t.sr0[k];
                s.diag = t.diag && t.l1 == l;
                if (s.r0 < 0 && !s.diag) continue;
                if (s.nj < t.na) R.part = 1;
                P->src.push_back(s);
                u.nsrc++;
            }
            if (!u.nsrc) continue;
            const TxTask &t = P->task[tasks[0]];
            u.o = o;
            u.p = l;
            u.f = f;
            u.na = (int)L.gn[l];
            u.ls0 = (int)L.gstart[l];
            u.nI = t.nI;
            u.nIp = t.nIp;
            u.nsv = t.nsv;
            u.w0 = w0;
            u.nw = nw;
            u.t0 = t0;
            u.nt = nt;
            u.nb = (int)O.s[1].gn[f];
            u.yb = O.boff[blk];
            u.blk0 = R.blocks;
            u.cblk = (nw * nt * 16 + 255) / 256;
            R.blocks += (ll)u.na * u.cblk;
            P->out.push_back(u);
            R.no++;
        }
    }

    void count(const TxRound &R, int part)
    {
        P->sum[part] += R.elems;
        P->elems = std::max(P->elems, R.elems);
        P->total += R.elems;
        P->grid = std::max(P->grid, std::max(std::max(R.items, R.small), R.blocks));
    }

    void rounds()
    {
        TxRound R;
        auto open = [&]() {
            memset(&R, 0, sizeof(R));
            R.i0 = (int)P->item.size();
            R.o0 = (int)P->out.size();
        };
        auto close = [&]() {
            if (R.ni) {
                // the longest items first, so that the launch ends on short ones
                auto first = P->item.begin() + R.i0;
                auto cost = [&](const TxItem &a) {
                    const TxTask &t = P->task[a.task];
                    ll c = 0;
                    for (int i = 0; i < t.nch; i++)
                        c += 4 * P->chunk[t.ch0 + i].KS * std::min(2, (t.La + 15) / 16) + 40 * P->chunk[t.ch0 + i].nslot;
                    return c * a.nt;
                };
                std::stable_sort(first, first + R.ni,
                                 [&](const TxItem &a, const TxItem &b) { return cost(a) > cost(b); });
                for (int i = 0; i < R.ni; i++) {
                    TxItem &a = first[i];
                    a.item0 = R.items;
                    R.items += (ll)a.nj * a.nw * a.rg;
                }
                P->ab.push_back(R);
                count(R, 0);
            }
            open();
        };
        open();
        for (int o = 0; o < 2; o++)
            for (int f = 0; f < dd[o]->s[1].ngrp; f++) {
                if (by[o][f].empty()) continue;
                const TxTask &t = P->task[by[o][f][0]];
                const int nt = t.nIp / 16;
                // elements of one external part for all tasks; where one alone exceeds the
                // buffer the tasks go one by one (their sums add up in the result), a single
                // one past the buffer by column tiles, and a column tile past it by strings JL
                ll all = 0;
                for (int ti : by[o][f]) all += (ll)P->task[ti].na * P->task[ti].La * 16 * nt;
                std::vector<std::vector<int>> sets;
                if (all <= budget) sets.push_back(by[o][f]);
                else for (int ti : by[o][f]) sets.push_back(std::vector<int>(1, ti));
                for (const std::vector<int> &set : sets) {
                    ll tile = 0;                 // elements of one column tile
                    for (int ti : set) tile += (ll)P->task[ti].na * P->task[ti].La * 16;
                    if (tile * nt <= budget) {
                        for (int w = 0; w < t.nsv;) {
                            const ll room = (budget - R.elems) / (tile * nt);
                            if (room <= 0) {
                                close();
                                continue;
                            }
                            const int n = (int)std::min<ll>(room, t.nsv - w);
                            piece(o, f, set, w, n, 0, nt, R);
                            w += n;
                        }
                    } else if (tile <= budget) {
                        for (int w = 0; w < t.nsv; w++)
                            for (int c = 0; c < nt;) {
                                const ll room = (budget - R.elems) / tile;
                                if (room <= 0) {
                                    close();
                                    continue;
                                }
                                const int n = (int)std::min<ll>(room, nt - c);
                                piece(o, f, set, w, 1, c, n, R);
                                c += n;
                            }
                    } else {
                        const TxTask &a = P->task[set[0]];
                        const ll most = std::max(1LL, budget / ((ll)a.La * 16)), parts = (a.na + most - 1) / most;
                        for (int w = 0; w < t.nsv; w++)
                            for (int c = 0; c < nt; c++)
                                for (ll k = 0; k < parts; k++) {
                                    const int j0 = (int)(a.na * k / parts), j1 = (int)(a.na * (k + 1) / parts);
                                    close();
                                    piece(o, f, set, w, 1, c, 1, R, j0, j1 - j0);
                                }
                        close();
                    }
                    // two pieces of one round may not add to the same results
                    if (sets.size() > 1) close();
                }
            }
        close();
    }

    void pair_tasks()
    {
        for (int o = 0; o < 2; o++) {
            const SpaceDesc &O = *dd[o];
            const SpinDesc &F = O.s[1];
            const std::vector<TxPairGroup> &pg = P->pg[o];
            for (int f = 0; f < F.ngrp; f++) {
                if (!F.gn[f]) continue;
                for (size_t g = 0; g < pg.size(); g++) {
                    TxPairTask t;
                    memset(&t, 0, sizeof(t));
                    t.o = o;
                    t.g2 = (int)g;
                    t.f = f;
                    for (int u = 0; u < TX_NTYPE; u++) {
                        if (pg[g].tgt[u] < 0 || !pg[g].cnt[u]) continue;
                        const int blk = O.blkid[pg[g].tgt[u]][f];
                        if (blk < 0) continue;
                        t.so[t.nsec] = pg[g].off[u];
                        t.sc[t.nsec] = pg[g].cnt[u];
                        t.sr[t.nsec] = t.R;
                        t.sx[t.nsec] = O.boff[blk];
                        t.nsec++;
                        t.R += pg[g].cnt[u];
                    }
                    if (!t.R) continue;
                    t.lbase = pg[g].base;
                    t.Rfull = pg[g].R;
                    t.n = (int)pg[g].n;
                    t.nb = (int)F.gn[f];
                    P->rmax = std::max(P->rmax, t.R);
                    pby[o][f].push_back((int)P->ptask.size());
                    P->ptask.push_back(t);
                }
            }
        }
    }

    // N - 2 electron strings [k0, k0 + nk) of a task
    struct Part { int task, k0, nk; };

    // one piece of a round: columns [c0, c0 + nc) of column group f for some strings of its tasks;
    // add: a piece before has written the results
    void pair_piece(int o, int f, int c0, int nc, const std::vector<Part> &parts, bool add, TxRound &R)
    {
        static const int ts[TX_NTYPE][2] = {{0, 0}, {0, 1}, {0, 2}, {1, 1}, {1, 2}, {2, 2}};
        const SpaceDesc &O = *dd[o];
        const SpinDesc &L = O.s[0];
        const int ncp = (int)up(nc, 16);
        std::vector<ll> eb;
        // (the gather takes a string's pairs as they come only where all tasks are there)
        if (add || parts.size() != pby[o][f].size()) R.part = 1;
        P->split[3] += c0 > 0;
        for (const Part &p : parts) {
            const TxPairTask &t = P->ptask[p.task];
            TxPairItem it;
            memset(&it, 0, sizeof(it));
            it.task = p.task;
            it.k0 = p.k0;
            it.nk = p.nk;
            P->split[4] += p.k0 > 0;
            if (p.nk < t.n) R.part = 1;
            it.c0 = c0;
            it.nc = nc;
            it.ncp = ncp;
            it.rg = (t.R + 63) / 64;
            // few pairs: many columns per work-group, for the list and the W tile it sets up
            it.cb = t.R <= 16 ? 16 : t.R <= 32 ? 8 : t.R <= TX_RMAX ? 4 : 1;
            it.ct = (nc + 64 * it.cb - 1) / (64 * it.cb);
            it.item0 = R.items;
            R.items += (ll)p.nk * it.rg * it.ct;
            it.ebase = R.elems;
            eb.push_back(R.elems);
            R.elems += (ll)p.nk * t.R * ncp;
            P->pitem.push_back(it);
            R.ni++;
        }
        for (int l = 0; l < L.ngrp; l++) {
            const int blk = O.blkid[l][f];
            if (blk < 0) continue;
            TxPairOut u;
            memset(&u, 0, sizeof(u));
            u.o = o;
            u.p = l;
            u.f = f;
            u.na = (int)L.gn[l];
            u.ls0 = (int)L.gstart[l];
            u.nb = (int)O.s[1].gn[f];
            u.c0 = c0;
            u.nc = nc;
            u.ncp = ncp;
            u.cblk = (nc + 255) / 256;
            u.yb = O.boff[blk];
            u.blk0 = R.blocks;
            R.blocks += (ll)u.na * u.cblk;
            u.add = add;
            const int e[3] = {L.gd[l], L.ga[l], L.gv[l]};
            int first = 0;
            for (int k = 0; k < TX_NTYPE; k++) {
                const int s0 = ts[k][0], s1 = ts[k][1];
                const int n = s0 == s1 ? e[s0] * (e[s0] - 1) / 2 : e[s0] * e[s1];
                if (n <= 0) continue;
                int o3[3] = {e[0], e[1], e[2]};
                o3[s0]--;
                o3[s1]--;
                for (size_t i = 0; i < parts.size(); i++) {
                    const TxPairTask &t = P->ptask[parts[i].task];
                    const TxPairGroup &g = P->pg[o][t.g2];
                    if (g.d != o3[0] || g.a != o3[1] || g.v != o3[2]) continue;
                    u.g0[u.nsec] = first;
                    u.k0[u.nsec] = parts[i].k0;
                    u.nk[u.nsec] = parts[i].nk;
                    u.np[u.nsec] = n;
                    u.R[u.nsec] = t.R;
                    u.eb[u.nsec] = eb[i];
                    for (int s = 0; s < t.nsec; s++)
                        if (t.so[s] == g.off[k] && t.sc[s] == g.cnt[k]) u.r0[u.nsec] = t.sr[s];
                    u.nsec++;
                }
                first += n;
            }
            if (add && !u.nsec) {
                R.blocks -= (ll)u.na * u.cblk;
                continue;
            }
            P->pout.push_back(u);
            R.no++;
        }
    }

    void pair_rounds()
    {
        TxRound R;
        auto open = [&]() {
            memset(&R, 0, sizeof(R));
            R.i0 = (int)P->pitem.size();
            R.o0 = (int)P->pout.size();
        };
        auto close = [&]() {
            if (R.ni) {
                // strings of few pairs first, in a launch of their own where they fill one
                auto groups = [&](const TxPairItem &it) { return (ll)it.nk * it.rg * it.ct; };
                auto few = [&](const TxPairItem &it) { return P->ptask[it.task].R <= TX_RSMALL; };
                const auto first = P->pitem.begin() + R.i0, end = P->pitem.end();
                ll small = 0;
                for (auto it = first; it != end; ++it) if (few(*it)) small += groups(*it);
                if (small >= TX_SMALL_GROUPS) {
                    R.nsmall = (int)(std::stable_partition(first, end, few) - first);
                    R.small = small;
                    R.items -= small;
                    ll at[2] = {0, 0};
                    for (int q = 0; q < R.ni; q++) {
                        TxPairItem &it = first[q];
                        ll &p = at[q >= R.nsmall];
                        it.item0 = p;
                        p += groups(it);
                    }
                }
                P->ss.push_back(R);
                count(R, 1);
            }
            open();
        };
        open();
        for (int o = 0; o < 2; o++)
            for (int f = 0; f < dd[o]->s[1].ngrp; f++) {
                if (pby[o][f].empty()) continue;
                ll col = 0;                      // elements of 16 columns
                for (int ti : pby[o][f]) col += (ll)P->ptask[ti].n * P->ptask[ti].R * 16;
                const int nb = P->ptask[pby[o][f][0]].nb;
                if (col * std::min(4, (nb + 15) / 16) <= budget) {
                    std::vector<Part> all;
                    for (int ti : pby[o][f]) all.push_back(Part{ti, 0, P->ptask[ti].n});
                    for (int c = 0; c < nb;) {
                        // whole 64-column blocks, or the rest of the group if it fits
                        const ll room = (budget - R.elems) / col * 16;
                        const ll n = room >= nb - c ? nb - c : room / 64 * 64;
                        if (n <= 0) {
                            close();
                            continue;
                        }
                        pair_piece(o, f, c, (int)n, all, false, R);
                        c += (int)n;
                    }
                    continue;
                }
                // 64 columns of all tasks past the buffer: a range of their strings at a time, the
                // sums of each added to those before
                for (int c = 0; c < nb; c += 64) {
                    const int nc = std::min(64, nb - c);
                    std::vector<Part> parts;
                    ll used = 0;
                    bool add = false;
                    auto flush = [&]() {
                        close();
                        pair_piece(o, f, c, nc, parts, add, R);
                        close();
                        parts.clear();
                        used = 0;
                        add = true;
                    };
                    for (int ti : pby[o][f]) {
                        const TxPairTask &t = P->ptask[ti];
                        const ll row = (ll)t.R * up(nc, 16);
                        for (int k = 0; k < t.n;) {
                            const ll room = (budget - used) / row;
                            if (room <= 0 && used) {
                                flush();
                                continue;
                            }
                            const int n = (int)std::min<ll>(std::max(1LL, room), t.n - k);
                            parts.push_back(Part{ti, k, n});
                            used += n * row;
                            k += n;
                        }
                    }
                    flush();
                }
            }
        close();
    }
};
}

int tx_plan(const SpaceDesc &D, const SpaceDesc &T, ll budget, TxPlan *P)
{
    if (D.s[0].nelec < 2 || D.s[1].nelec < 2 || D.norbs < 2) return 1;
    P->elems = P->total = P->grid = 0;
    P->ldt = P->rmax = 0;
    P->sum[0] = P->sum[1] = 0;
    memset(P->split, 0, sizeof(P->split));
    for (int s = 0; s < 2; s++) {
        if (plan_lists(D, D.s[s], P->lists[s], &P->nlst[s])) return 1;
        if (plan_pairs(D, D.s[s], P->pg[s], &P->nkl[s])) return 1;
        if (P->nlst[s] / 256 >= TX_GRID) return 1;   // one thread an entry fills them
        ll n = 0;
        for (int g = 0; g < D.s[s].ngrp; g++) {
            P->iI0[s][g] = (int)n;
            n += P->lists[s][g].nI;
        }
        P->nint_parts[s] = n;
    }
    Builder *B = new Builder();
    B->dd[0] = &D;
    B->dd[1] = &T;
    B->budget = budget;
    B->P = P;
    jci_binom_table(B->binom);
    int rc = B->tasks();
    if (!rc) {
        B->rounds();
        B->pair_tasks();
        B->pair_rounds();
    }
    delete B;
    if (P->grid > TX_GRID) rc = 1;
    // the table kernels' estimate: opposite-spin connections, and those of one determinant
    double entries = 0.0, chain = 0.0;
    for (int b = 0; b < D.nblk; b++) {
        double each = 0.0;
        for (int c = 0; c < D.nblk; c++)
            each += (double)std::max(0LL, singles(D, D.s[0], D.bp[b], D.bp[c])) *
                    (double)std::max(0LL, singles(D, D.s[1], D.bq[b], D.bq[c]));
        entries += each * (double)D.s[0].gn[D.bp[b]] * (double)D.s[1].gn[D.bq[b]];
        chain = std::max(chain, each);
    }
    if (TX_COST_AB * P->sum[0] + TX_COST_SS * P->sum[1] > TX_COST_ENTRY * entries + TX_COST_CHAIN * chain)
        rc = 1;
    return rc;
}
