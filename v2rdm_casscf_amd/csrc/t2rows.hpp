// t2rows.hpp -- the T2 rows (t2.cc:1251-1861) by unit: one row's columns of one chunk, a
// wavefront's work (t2maps.hip); the code runs on the host too (CPU tests).
//
// A T2 row (ijk) holds its own entry in every column (lmn) and a D2 or D1 term only where a
// column's orbital equals one of the row's: of n^3 columns each of the five or so
// conditions (l == i, n == k, ...) keeps n^2.  Asked of every column (rows::t2_terms), the
// conditions make nearly every wavefront walk all branches with a few lanes in each.  Here the
// columns with l == o, m == o and n == o are listed beforehand for every orbital o, and a
// unit walks the lists its row selects: every lane has a term.
//
// A^T y of the same rows is gathered, entry by entry: every term's row and column share
// one orbital t, so a D2 entry's part is a sum over t of some ten row elements whose places the
// triplets' ranks give, and a D1 entry's a sum over two orbitals.
#pragma once
#include <vector>

#include "layout.hpp"
#include "rowterms.hpp"

namespace v2g {

constexpr int kT2Chunk = 1024;   // columns of a unit at most: 8 KB of LDS a wavefront

// columns c0 .. c0 + n of a row's aab part (aba = 0) or aba part; its lists start at
// ptr[ptr0 + slot * amo + o], slot 0, 1, 2: l, m, n == o
struct T2Chunk {
    int32_t c0, n, aba, ptr0;
};

// the T2 rows of one block: `dim` rows in nchunk chunks each, units unit0 ..
struct T2Seg {
    int32_t kind, sub, h, dim, chunk0, nchunk;
    int64_t unit0, x0, row0;   // first unit, first entry of the own block, first row
};

struct T2Tab {
    const T2Seg *seg;
    const T2Chunk *chunk;
    const int32_t *ptr;
    const uint32_t *item;      // column within the chunk | the other two orbitals << 10, << 18
    const int32_t *aab, *aba;  // place of the triplet (i, j, k) in its irrep's list, amo^3 each
    int nseg;
    int64_t units;
};

struct T2Lists {
    std::vector<T2Seg> seg;
    std::vector<T2Chunk> chunk;
    std::vector<int32_t> ptr;
    std::vector<uint32_t> item;
    std::vector<int32_t> aab, aba;
    int64_t units = 0;
};

// the lists of a layout with T2 rows (t2lists.cc)
void make_t2_lists(const Layout &L, T2Lists &out);

namespace rows {

// the segment, row and chunk of a unit
V2G_HD inline const T2Seg &t2_unit(const T2Tab &T, int64_t unit, int &row, T2Chunk &ch)
{
    int lo = 0, hi = T.nseg;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (T.seg[mid].unit0 <= unit) lo = mid;
        else hi = mid;
    }
    const T2Seg &sg = T.seg[lo];
    const uint32_t u = (uint32_t)(unit - sg.unit0);
    row = (int)(u / (uint32_t)sg.nchunk);
    ch = T.chunk[sg.chunk0 + (int)(u % (uint32_t)sg.nchunk)];
    return sg;
}

// offset of the unit's first column within the block
V2G_HD inline int64_t t2_first(const DevLayout &L, const T2Seg &sg, int row, const T2Chunk &ch)
{
    return (int64_t)row * sg.dim + (ch.aba ? L.trip_aab[sg.h] : 0) + ch.c0;
}

// the D2 / D1 terms of a unit: f(column within the chunk, column of x, coefficient), list by
// list with phase() between them; within a list every column occurs once.  Lane `lane` of
// `lanes` takes its share.
template <class F, class B>
V2G_HD inline void t2_unit_terms(const DevLayout &L, const T2Tab &T, const T2Seg &sg, int row, const T2Chunk &ch,
                                 int lane, int lanes, F &f, const B &phase)
{
    const int amo = L.amo, h = sg.h, s = sg.sub;
    const int *gab = L.gab, *gaa = L.gaa, *sym = L.sym;
    const bool big = sg.kind == RF_T2BIG, rA = !big || row < L.trip_aab[h], cA = !ch.aba;
    const int pr = rA ? L.baab[L.baab_off[h] + row] : L.baba[L.baba_off[h] + (row - L.trip_aab[h])];
    const int i = T0(pr), j = T1(pr), k = T2i(pr);
    // the columns whose slot-th orbital is o: fn(column, the other two orbitals)
    auto list = [&](int slot, int o, auto fn) {
        const int32_t *p = T.ptr + ch.ptr0 + slot * amo + o;
        for (int t = p[0] + lane; t < p[1]; t += lanes) {
            const uint32_t it = T.item[t];
            fn((int)(it & 1023), (int)(it >> 10 & 255), (int)(it >> 18));
        }
        phase();
    };
    auto GAB = [&](int p, int q) -> int64_t { return gab[p * amo + q]; };
    auto GAA = [&](int p, int q) -> int64_t { return gaa[p * amo + q]; };
    auto D1 = [&](int w, int n) -> int64_t {   // D1 (n, k)
        const int h3 = sym[k];
        return L.xoff[w][h3] + (int64_t)(n - L.poff[h3]) * L.amopi[h3] + (k - L.poff[h3]);
    };
    auto AA = [&](int c, int w, int p, int q, int r, int v, double co) {   // D2aa / D2bb (pq|rv)
        if (p == q || r == v) return;
        const int hh = sym[p] ^ sym[q];
        f(c, L.xoff[w][hh] + GAA(p, q) * L.gems_aa[hh] + GAA(r, v), (p > q) == (r > v) ? co : -co);
    };
    // D2ab (pq|rv), alpha first; AX: the spins swapped when s (aab rows), when !s (AY)
    auto AB = [&](int c, int p, int q, int r, int v, double co) {
        const int hh = sym[p] ^ sym[q];
        f(c, L.xoff[XB_D2AB][hh] + GAB(p, q) * L.gems_ab[hh] + GAB(r, v), co);
    };
    auto AX = [&](int c, int p, int q, int r, int v, double co) { s ? AB(c, q, p, v, r, co) : AB(c, p, q, r, v, co); };
    auto AY = [&](int c, int p, int q, int r, int v, double co) { s ? AB(c, p, q, r, v, co) : AB(c, q, p, v, r, co); };
    const int w2 = s ? XB_D2BB : XB_D2AA, w2o = s ? XB_D2AA : XB_D2BB;
    const int wd = s ? XB_D1B : XB_D1A, wdo = s ? XB_D1A : XB_D1B;
    if (rA && cA) {
        const int hij = sym[i] ^ sym[j];
        const int64_t ij = L.xoff[w2][hij] + GAA(i, j) * L.gems_aa[hij];
        list(2, k, [&](int c, int l, int m) { f(c, ij + GAA(l, m), 1.0); });
        if (!big) {
            list(0, i, [&](int c, int m, int n) {
                AX(c, j, n, m, k, -1.0);
                if (m == j) f(c, D1(wdo, n), 1.0);
            });
            list(0, j, [&](int c, int m, int n) { AX(c, i, n, m, k, 1.0); });
            list(1, i, [&](int c, int l, int n) { AX(c, j, n, l, k, 1.0); });
            list(1, j, [&](int c, int l, int n) { AX(c, i, n, l, k, -1.0); });
        } else {
            list(0, i, [&](int c, int m, int n) {
                AA(c, w2, n, j, k, m, -1.0);
                if (m == j) f(c, D1(wd, n), 1.0);
            });
            list(0, j, [&](int c, int m, int n) { AA(c, w2, n, i, k, m, 1.0); });
            list(1, i, [&](int c, int l, int n) { AA(c, w2, n, j, k, l, 1.0); });
            list(1, j, [&](int c, int l, int n) { AA(c, w2, n, i, k, l, -1.0); });
        }
    } else if (rA) {
        list(0, i, [&](int c, int m, int n) { AX(c, j, n, k, m, 1.0); });
        list(0, j, [&](int c, int m, int n) { AX(c, i, n, k, m, -1.0); });
    } else if (cA) {
        list(0, i, [&](int c, int m, int n) { AY(c, j, n, k, m, 1.0); });
        list(1, i, [&](int c, int l, int n) { AY(c, j, n, k, l, -1.0); });
    } else {
        list(2, k, [&](int c, int l, int m) { AX(c, i, j, l, m, 1.0); });
        list(0, i, [&](int c, int m, int n) {
            AA(c, w2o, n, j, k, m, -1.0);
            if (m == j) f(c, D1(wdo, n), 1.0);
        });
        list(1, j, [&](int c, int l, int n) { AX(c, i, n, l, k, -1.0); });
    }
}

// ---- A^T y ---------------------------------------------------------------------
// elements of y by triplets: AAB(s; i j k | l m n), and of the big blocks with aab (A) or
// aba (B) rows and columns; aab triplets in either order of their first two
template <class Y>
struct T2Y {
    const DevLayout &L;
    const T2Tab &T;
    const Y &y;
    V2G_HD inline int64_t aab(int i, int j, int k) const
    {
        return T.aab[((i < j ? i : j) * L.amo + (i < j ? j : i)) * L.amo + k];
    }
    V2G_HD inline int64_t aba(int i, int j, int k) const { return T.aba[(i * L.amo + j) * L.amo + k]; }
    V2G_HD inline double A(int s, int h, int64_t row, int64_t col) const
    {
        return y[L.rowoff[RF_T2AAB][s][h] + row * L.trip_aab[h] + col];
    }
    // row and col of the whole block: aba triplets follow the aab ones
    V2G_HD inline double B(int s, int h, int64_t row, int64_t col) const
    {
        return y[L.rowoff[RF_T2BIG][s][h] + row * (L.trip_aab[h] + L.trip_aba[h]) + col];
    }
};

// the terms that share the orbital t of the D2ab entry (pq|rs), from the rows of spin sp
template <class Y>
V2G_HD inline double t2_at_ab(const DevLayout &L, const T2Tab &T, int sp, int t, int p, int q, int r, int s,
                              const Y &y)
{
    if (sp) {   // the other spin's rows read the entry with its spins exchanged
        int x = p;
        p = q;
        q = x;
        x = r;
        r = s;
        s = x;
    }
    const T2Y<Y> e{L, T, y};
    const int *sym = L.sym;
    const int h1 = sym[t] ^ sym[p] ^ sym[s], h2 = sym[t] ^ sym[p] ^ sym[r], h3 = sym[t] ^ sym[q] ^ sym[s],
              h4 = sym[t] ^ sym[p] ^ sym[q];
    const int a2 = L.trip_aab[h2], a3 = L.trip_aab[h3], a4 = L.trip_aab[h4], a1 = L.trip_aab[h1];
    double v = e.B(sp, h4, a4 + e.aba(p, q, t), a4 + e.aba(r, s, t)) -
               e.B(sp, h1, a1 + e.aba(p, t, s), a1 + e.aba(r, t, q));
    if (t != p) {
        const double b = e.B(sp, h2, e.aab(t, p, r), a2 + e.aba(t, s, q));
        v += t < p ? b : -b;
    }
    if (t != r) {
        const double b = e.B(sp, h3, a3 + e.aba(t, q, s), e.aab(t, r, p));
        v += t < r ? b : -b;
    }
    if (t != p && t != r) {
        const double b = e.A(sp, h1, e.aab(t, p, s), e.aab(t, r, q));
        v += (t < p) == (t < r) ? -b : b;
    }
    return v;
}

// the same of the D2aa (sp = 0) / D2bb entry of the pairs a < b, c < d
template <class Y>
V2G_HD inline double t2_at_aa(const DevLayout &L, const T2Tab &T, int sp, int t, int a, int b, int c, int d,
                              const Y &y)
{
    const T2Y<Y> e{L, T, y};
    const int *sym = L.sym;
    const int h0 = sym[t] ^ sym[a] ^ sym[b];
    double v = e.A(sp, h0, e.aab(a, b, t), e.aab(c, d, t)) + e.B(sp, h0, e.aab(a, b, t), e.aab(c, d, t));
    for (int k = 0; k < 4; k++) {
        // n, J of the bra and k, M of the ket in either order
        const int n = k & 1 ? b : a, J = k & 1 ? a : b, kk = k & 2 ? d : c, M = k & 2 ? c : d;
        const int h = sym[t] ^ sym[J] ^ sym[kk], ta = L.trip_aab[h];
        double w = -e.B(1 - sp, h, ta + e.aba(t, J, kk), ta + e.aba(t, M, n));
        if (t != J && t != M) {
            const double x = e.B(sp, h, e.aab(t, J, kk), e.aab(t, M, n));
            w += (t < J) == (t < M) ? -x : x;
        }
        v += (k & 1) == (k >> 1) ? w : -w;
    }
    return v;
}

// the terms that share the orbitals i, j of the D1a (sp = 0) / D1b entry (n, k)
template <class Y>
V2G_HD inline double t2_at_d1(const DevLayout &L, const T2Tab &T, int sp, int i, int j, int n, int k, const Y &y)
{
    const T2Y<Y> e{L, T, y};
    const int h = L.sym[i] ^ L.sym[j] ^ L.sym[k], ta = L.trip_aab[h];
    double v = e.B(1 - sp, h, ta + e.aba(i, j, k), ta + e.aba(i, j, n));
    if (i < j) v += e.A(1 - sp, h, e.aab(i, j, k), e.aab(i, j, n)) + e.B(sp, h, e.aab(i, j, k), e.aab(i, j, n));
    return v;
}

}  // namespace rows
}  // namespace v2g
