// redrows.hpp -- the rows of A in the reduced form of the plain CG (redcg.hip),
// as code that runs on the device and, unchanged, on the host (CPU tests).
//
// Most constraint rows (D200, Q1, Q2, G2) hold one entry +-1 in a primal block
// of their own ("self rows"); the rest of such a row, and every other row
// ("explicit rows"), only reads D2 and D1 entries.  With A = [B1 0; B2 S],
// S = diag(+-1), the operator of the CG on the self rows is
//
//     (A A^T p)_self = p_self + B2 t,   t = (A^T p)_D = B1^T p_expl + B2^T p_self,
//
// so every vector of a plain CG keeps the form  a s + B2 b  on the self rows,
// with s the self part of the first residual, a number a and a vector b of D2 /
// D1 length.  The maximal-spin rows also read G2ba entries of irrep 0; they add
// a third generator, - P m, with one number per maximal-spin row.
//
// The self parts of s are kept aligned with the D2 entry they read: a G2ab,
// G2ba or G2 super-block row reads exactly one D2ab (or D2aa) entry (pq|rs), so
// its slot is that entry's.  The entries in turn are stored by "cell": for a pair
// p > q and a pair r > s the four D2ab entries (pq|rs), (qp|rs), (pq|sr), (qp|sr)
// lie at the same place of four arrays, beside the cell's D2aa and D2bb entry.
// D200, the like-spin quadrants and the antisymmetry rows only mix what is in one
// cell, so on a cell whose pairs share no orbital the whole operator is a few
// multiply-adds on its own numbers: no index arithmetic and no gather.  Cells that
// share an orbital, and the entries with p == q or r == s, also meet D1, the
// traces, contractions, S^2 and the maximal-spin rows; they are listed.
#pragma once
#include "rowterms.hpp"

namespace v2g {

// families of self rows; the first kSfAb are aligned with the D2ab entries
// (pq|rs), the next two with the D2aa / D2bb entries, the last two with D1
enum SelfFam : int {
    SF_Q2AB = 0,
    SF_G2AB,      // row ((p,s),(r,q)) of G2ab
    SF_G2BA,      // row ((q,r),(s,p)) of G2ba
    SF_G2X,       // row ((p,r),(s,q)) of the alpha-beta quadrant of the super block
    SF_G2Y,       // row ((q,s),(r,p)) of the beta-alpha quadrant
    SF_G2A,       // row ((p,s),(r,q)) of the alpha-alpha quadrant
    SF_G2B,       // the same in the beta-beta quadrant
    SF_D0, SF_D1, SF_D2, SF_D3,   // D200 (singlet: SF_D0 only), quadrant 2 a + b
    kSfAb,
    SF_Q2AA = kSfAb, SF_Q2BB, SF_Q1A, SF_Q1B, SF_COUNT
};

struct RedLayout {
    // xoff of the D1 blocks in a D vector (the offsets count the entries; D, R and M
    // vectors end with one more, a zero, for indices that stand for no entry), rowoff of the explicit rows that are not
    // aligned with cells in an R vector; other blocks and rows absent
    DevLayout L;
    // positions of the D2ab entries: 4 gems_aa^2 from ab0[h] on (orientation
    // (p < q) + 2 (r < s), then the cell), the entries (pp|rs) from dA and (pq|rr),
    // p != q, from dB on.  A D vector is [D2ab: nAB][D2aa: nAA][D2bb: nAA][D1a][D1b]
    int64_t ab0[kMaxIrrep], aa0[kMaxIrrep], dA, dB, nAB, nAA;
    int64_t soff[SF_COUNT];              // first slot of a family, -1 absent
    int64_t nD, nR, nS;
    // cell-aligned explicit rows (singlets with spin rows): D2aa - D2bb, then the two
    // antisymmetry rows; nAA each from 0, or cells = 0
    int cells;
    int64_t nD1;     // D1a entries
    int nM;          // maximal-spin rows (2 gems_ab[0], or 0)
    int lanes;       // threads that share a row summed over the orbitals: 16, 32 or 64
    int nblk_d;      // D200 quadrants: 0 (spin off), 1 (singlet), 4
    const int32_t *rowtab;   // RT_COUNT tables of amo^2 entries (RowTab)
};

// A row of the full layout is the sum of two entries, by the row pair and by the column
// pair: the first with the block's offset and row length worked in.  (From the geminal
// numbers, with the irreps' offsets and lengths to look up as well, the start and the end of a
// solve spent 120 loads on an entry's 14 rows.)
enum RowTab : int {
    RT_AB,                 // column: the pair's number
    RT_GG,                 // column: behind the first half
    RT_Q2, RT_G2AB, RT_G2BA, RT_GA, RT_GB, RT_D0, RT_D1, RT_COUNT   // rows
};

// a D2ab entry outside the cells (p == q or r == s): where everything lies that its rows
// read, -1 never occurs (the zero at the end of the vector stands for an absent entry).  It
// has no D2aa entry and no antisymmetry row
struct AbRec {
    int32_t pos, p1, p2, p3;   // (pq|rs), (qp|rs), (pq|sr), (qp|sr)
    int32_t pr, rp;            // D1a entries (p,r), (r,p) when q == s
    int32_t qs, sq;            // D1b entries (q,s), (s,q) when p == r
    int32_t m0, m1;            // maximal-spin rows when s == p, q == r
    int32_t flags;             // AbFlag
};
enum AbFlag : int { AF_BRA = 1, AF_KET = 2, AF_QS = 4, AF_PR = 8, AF_S2 = 16 };

// a listed cell: its pairs share an orbital k, or both orbitals.  With i and j the others
// of the two pairs, a shared orbital puts D1a(i,j) into the rows of (ik|jk), D1b(i,j) into
// those of (ki|kj), and the maximal-spin rows into (ki|jk) and (ik|kj)
struct CellRec {
    int32_t pos, k;            // first D2ab entry, place among the cells
    int32_t ij[2], ji[2];      // D1a entries (i,j), (j,i)
    int32_t m0[2], m1[2];      // maximal-spin rows of (ki|jk), (ik|kj)
    int32_t row;               // place within the irrep (for checks)
    int32_t flags;             // orientation of (ik|jk) in bits 0-1 and 2-3, CellFlag, irrep << 8
};
enum CellFlag : int { CF_TWO = 16 };

namespace rows {

struct AbEntry {
    int p, q, r, s;
    int64_t pos;
    // of an entry inside a cell (cc = 0: outside): the cell's first entry, cells of the
    // irrep, orientation, place among the cells
    int64_t base = 0, cc = 0;
    int o = 0;
    int64_t k = 0;
};

V2G_HD inline int64_t ab_pos(const RedLayout &R, int p, int q, int r, int s)
{
    const DevLayout &L = R.L;
    if (p == q) return R.dA + (int64_t)p * L.gems_ab[0] + L.gab[r * L.amo + s];
    if (r == s) return R.dB + (int64_t)r * L.gems_ab[0] + L.gab[p * L.amo + q];
    const int h = L.sym[p] ^ L.sym[q];
    const int64_t ga = L.gems_aa[h];
    return R.ab0[h] + ((p < q) + 2 * (r < s)) * ga * ga + L.gaa[p * L.amo + q] * ga + L.gaa[r * L.amo + s];
}

// cell of (pq|rs), p != q, r != s: the place of its D2aa entry among the nAA
V2G_HD inline int64_t aa_pos(const RedLayout &R, int p, int q, int r, int s)
{
    const DevLayout &L = R.L;
    const int h = L.sym[p] ^ L.sym[q];
    return R.aa0[h] + (int64_t)L.gaa[p * L.amo + q] * L.gems_aa[h] + L.gaa[r * L.amo + s];
}

// the pairs p > q, r > s of cell c of irrep h
V2G_HD inline AbEntry cell_entry(const RedLayout &R, int h, int64_t c)
{
    const DevLayout &L = R.L;
    int I, K;
    split_index(c, L.gems_aa[h], I, K);
    const int b = L.baa[L.baa_off[h] + I], k = L.baa[L.baa_off[h] + K];
    const int64_t pos = R.ab0[h] + c;
    return {P0(b), P1(b), P0(k), P1(k), pos, pos, (int64_t)L.gems_aa[h] * L.gems_aa[h], 0, R.aa0[h] + c};
}

// entry number i (0 .. 4 gems_aa^2) of irrep h: by the bra pair in one order, then in the
// other, with both orders of the ket pair after each bra: together they touch whole lines of the
// rows, one order alone the r > s part of each
V2G_HD inline AbEntry cell_ab(const RedLayout &R, int h, int64_t i)
{
    const DevLayout &L = R.L;
    const int64_t ga = L.gems_aa[h], cc = ga * ga;
    const int o1 = i >= 2 * cc ? 1 : 0;
    int I, K;
    split_index(i - o1 * 2 * cc, 2 * ga, I, K);
    const int o = o1 + (K >= ga ? 2 : 0);
    AbEntry a = cell_entry(R, h, I * ga + (K >= ga ? K - ga : K));
    if (o & 1) { const int t = a.p; a.p = a.q; a.q = t; }
    if (o & 2) { const int t = a.r; a.r = a.s; a.s = t; }
    a.pos += o * cc;
    a.o = o;
    return a;
}

// position of the entry with the bra pair (x & 1), the ket pair (x & 2) exchanged
V2G_HD inline int64_t exchanged(const RedLayout &R, const AbEntry &a, int x)
{
    if (a.cc) return a.base + (a.o ^ x) * a.cc;
    return ab_pos(R, x & 1 ? a.q : a.p, x & 1 ? a.p : a.q, x & 2 ? a.s : a.r, x & 2 ? a.r : a.s);
}

// entry number i (0 .. 2 amo gems_ab[0]) of those with p == q or r == s; false: none
V2G_HD inline bool diag_ab(const RedLayout &R, int64_t i, AbEntry &a)
{
    const DevLayout &L = R.L;
    const int g0 = L.gems_ab[0];
    const int d = (int)(i / g0), pr = L.bab[L.bab_off[0] + i % g0];
    if (d < L.amo) {
        a = {d, d, P0(pr), P1(pr), R.dA + i};
        return true;
    }
    a = {P0(pr), P1(pr), d - L.amo, d - L.amo, R.dB + (i - (int64_t)L.amo * g0)};
    return a.p != a.q;
}

V2G_HD inline int64_t d1_col(const DevLayout &L, int w, int p, int q)
{
    const int h = L.sym[p];
    return L.xoff[w][h] + (int64_t)(p - L.poff[h]) * L.amopi[h] + (q - L.poff[h]);
}

// coefficients of a D200 row of quadrant 2 a + b on (pq|rs), (qp|rs), (pq|sr), (qp|sr)
V2G_HD inline void d200_coef(int blk, bool singlet, bool pq, bool rs, double (&c)[4])
{
    const double dp = pq ? 1.4142135623730951 : 1.0, dr = rs ? 1.4142135623730951 : 1.0;
    if (singlet || blk == 0) {
        c[0] = c[1] = c[2] = c[3] = -0.5 / (dp * dr);
    } else if (blk == 1) {
        const double v = 0.5 / dp;
        c[0] = c[1] = -v;
        c[2] = c[3] = v;
    } else if (blk == 2) {
        const double v = 0.5 / dr;
        c[0] = c[2] = -v;
        c[1] = c[3] = v;
    } else {
        c[0] = c[3] = -0.5;
        c[1] = c[2] = 0.5;
    }
}

// the D2 / D1 parts of the Q2 and G2 rows aligned with entry a; X is a D vector
template <class X>
struct SelfAb {
    double x, q2, g1, g2, ga, gb;   // x: the mixed-spin quadrants' part too
    V2G_HD inline SelfAb(const RedLayout &R, const AbEntry &a, const X &v)
    {
        const DevLayout &L = R.L;
        x = v[a.pos];
        q2 = x;
        g1 = g2 = -x;
        ga = gb = 0.0;
        if (L.g2 && a.p != a.q && a.r != a.s) {
            const int64_t k = R.nAB + a.k;
            const double sg = ((a.p < a.q) == (a.r < a.s)) ? -1.0 : 1.0;
            ga = sg * v[k];
            gb = sg * v[k + R.nAA];
        }
        if (a.q == a.s) {
            if (L.q2) q2 -= v[d1_col(L, XB_D1A, a.r, a.p)];
            if (L.g2) {
                const double da = v[d1_col(L, XB_D1A, a.p, a.r)];
                g1 += da;
                ga += da;
                gb += v[d1_col(L, XB_D1B, a.p, a.r)];
            }
        }
        if (a.p == a.r) {
            if (L.q2) q2 -= v[d1_col(L, XB_D1B, a.s, a.q)];
            if (L.g2) g2 += v[d1_col(L, XB_D1B, a.q, a.s)];
        }
    }
};

// the D2 parts of the D200 rows aligned with entry a
template <class X>
struct D200Ab {
    double v0, v1, v2, v3;          // x at (pq|rs), (qp|rs), (pq|sr), (qp|sr)
    V2G_HD inline D200Ab(const RedLayout &R, const AbEntry &a, const X &v)
    {
        v0 = v[a.pos];
        v1 = v[exchanged(R, a, 1)];
        v2 = v[exchanged(R, a, 2)];
        v3 = v[exchanged(R, a, 3)];
    }
    V2G_HD inline double row(const RedLayout &R, const AbEntry &a, int blk) const
    {
        double c[4];
        d200_coef(blk, R.L.singlet, a.p == a.q, a.r == a.s, c);
        return c[0] * v0 + c[1] * v1 + c[2] * v2 + c[3] * v3;
    }
};

// the D2 / D1 part of the Q2aa / Q2bb row (spin sp) of the cell a
template <class X>
V2G_HD inline double self_row_aa(const RedLayout &R, int sp, const AbEntry &a, const X &x)
{
    const DevLayout &L = R.L;
    const int i = a.p, j = a.q, k = a.r, l = a.s, wd = sp ? XB_D1B : XB_D1A;
    double v = x[R.nAB + sp * R.nAA + aa_pos(R, i, j, k, l)];
    if (j == l) v -= x[d1_col(L, wd, k, i)];
    if (j == k) v += x[d1_col(L, wd, l, i)];
    if (i == l) v += x[d1_col(L, wd, k, j)];
    if (i == k) v -= x[d1_col(L, wd, l, j)];
    return v;
}

// (P m)(e): the maximal-spin generator on the G2ba row aligned with (pq|rs)
// (s == p or q == r imply that the row lies in irrep 0)
template <class M>
V2G_HD inline double ms_part(const RedLayout &R, int p, int q, int r, int s, const M &m)
{
    const DevLayout &L = R.L;
    double v = 0.0;
    if (R.nM) {
        if (s == p) v += m[L.gab[q * L.amo + r]];
        if (q == r) v += m[L.gems_ab[0] + L.gab[s * L.amo + p]];
    }
    return v;
}

// whether ms_part has a term
V2G_HD inline bool ms_reads(const RedLayout &R, int p, int q, int r, int s) { return R.nM && (s == p || q == r); }

// B2^T (B2 x - P m) on a D1 entry: lane-strided share of R.lanes threads
template <class X, class M>
V2G_HD inline double gram_d1(const RedLayout &R, int sp, int h, int64_t item, int lane, const X &x,
                             const M &m)
{
    const DevLayout &L = R.L;
    const int n = L.amopi[h];
    const int A = (int)(item / n) + L.poff[h], B = (int)(item % n) + L.poff[h];
    const int wd = sp ? XB_D1B : XB_D1A, wo = sp ? XB_D1A : XB_D1B;
    // D1(A,B) itself: the D1 + Q1 row, then one Q2ab and two G2 rows for every t and a
    // like-spin Q2 row for every t that differs from A and B
    const double xd = x[L.xoff[wd][h] + item];
    const int others = L.amo - (A == B ? 1 : 2);
    double v = lane == 0 ? xd * (1.0 + (L.q2 ? L.amo + others : 0) + (L.g2 ? 2.0 * L.amo : 0.0)) : 0.0;
    for (int t = lane; t < L.amo; t += R.lanes) {
        const bool in = t != A && t != B;
        const double sg = ((A < t) == (B < t)) ? 1.0 : -1.0;
        const int64_t k = in ? R.nAB + sp * R.nAA : 0;
        if (L.q2) {
            v -= x[sp ? ab_pos(R, t, B, t, A) : ab_pos(R, B, t, A, t)];
            if (in) v -= sg * x[k + aa_pos(R, B, t, A, t)];
            if (A == B) v += x[d1_col(L, wo, t, t)] + (in ? x[d1_col(L, wd, t, t)] : 0.0);
        }
        if (L.g2) {
            v -= x[sp ? ab_pos(R, t, A, t, B) : ab_pos(R, A, t, B, t)];   // G2ab / G2ba
            if (in) v -= sg * x[k + aa_pos(R, A, t, B, t)];              // like-spin quadrant
            if (sp) v -= ms_part(R, t, A, t, B, m);
        }
    }
    return v;
}

// B2^T s: the self rows' share of A^T on a D2ab / D2aa / D1 entry from aligned slots
template <class S>
V2G_HD inline double self_at_ab(const RedLayout &R, const AbEntry &a, const S &s)
{
    const DevLayout &L = R.L;
    double t = 0.0;
    if (L.q2) t += s[R.soff[SF_Q2AB] + a.pos];
    if (L.g2)
        t += (s[R.soff[SF_G2X] + a.pos] + s[R.soff[SF_G2Y] + a.pos]) -
             (s[R.soff[SF_G2AB] + a.pos] + s[R.soff[SF_G2BA] + a.pos]);
    if (R.nblk_d) {
        const int64_t p1 = exchanged(R, a, 1), p2 = exchanged(R, a, 2), p3 = exchanged(R, a, 3);
        for (int k = 0; k < R.nblk_d; k++) {
            double c[4];
            d200_coef(k, L.singlet, a.p == a.q, a.r == a.s, c);
            const int64_t b = R.soff[SF_D0 + k];
            t += c[0] * s[b + a.pos] + c[1] * s[b + p1] + c[2] * s[b + p2] + c[3] * s[b + p3];
        }
    }
    return t;
}

template <class S>
V2G_HD inline double self_at_aa(const RedLayout &R, int sp, int h, const AbEntry &a, const S &s)
{
    const DevLayout &L = R.L;
    double t = L.q2 ? s[R.soff[sp ? SF_Q2BB : SF_Q2AA] + aa_pos(R, a.p, a.q, a.r, a.s)] : 0.0;
    if (L.g2) {
        const int64_t cc = (int64_t)L.gems_aa[h] * L.gems_aa[h];
        const int64_t b = R.soff[sp ? SF_G2B : SF_G2A] + a.pos;
        t += (s[b + cc] + s[b + 2 * cc]) - (s[b] + s[b + 3 * cc]);
    }
    return t;
}

template <class S>
V2G_HD inline double self_at_d1(const RedLayout &R, int sp, int h, int64_t item, int lane, const S &s)
{
    const DevLayout &L = R.L;
    const int n = L.amopi[h];
    const int A = (int)(item / n) + L.poff[h], B = (int)(item % n) + L.poff[h];
    double v = lane == 0 ? s[R.soff[sp ? SF_Q1B : SF_Q1A] + (L.xoff[sp ? XB_D1B : XB_D1A][h] -
                                                             L.xoff[sp ? XB_D1B : XB_D1A][0]) + item]
                         : 0.0;
    for (int t = lane; t < L.amo; t += 64) {
        if (L.q2) {
            v -= s[R.soff[SF_Q2AB] + (sp ? ab_pos(R, t, B, t, A) : ab_pos(R, B, t, A, t))];
            if (t != A && t != B) {
                const double sg = ((B > t) == (A > t)) ? 1.0 : -1.0;
                v -= sg * s[R.soff[sp ? SF_Q2BB : SF_Q2AA] + aa_pos(R, B, t, A, t)];
            }
        }
        if (L.g2) {
            v += s[R.soff[sp ? SF_G2BA : SF_G2AB] + (sp ? ab_pos(R, t, A, t, B) : ab_pos(R, A, t, B, t))];
            // the like-spin quadrant's row ((A,t),(B,t)) reads (At|Bt)
            v += s[R.soff[sp ? SF_G2B : SF_G2A] + ab_pos(R, A, t, B, t)];
        }
    }
    return v;
}

// (P^T P m) of maximal-spin row `item` of orientation o: lane-strided share
template <class M>
V2G_HD inline double ms_row_gram(const RedLayout &R, int o, int item, int lane, const M &m)
{
    const DevLayout &L = R.L;
    const int g0 = L.gems_ab[0];
    const int pr = L.bab[L.bab_off[0] + item];
    double v = lane == 0 ? L.amo * m[o * g0 + item] : 0.0;
    if (P0(pr) == P1(pr))
        for (int i = lane; i < L.amo; i += R.lanes) v += m[(1 - o) * g0 + L.gab[i * L.amo + i]];
    return v;
}

// maximal-spin row `item` of orientation o (0: G2ba entries (kl, ii), 1: (ii, kl)):
// lane-strided share of sum_i p_self over its G2ba rows, p_self = d s + B2 x - P m.  sq
// (optional): += the squares of those p_self, each G2ba row once over all maximal-spin rows
template <class S, class X, class M>
V2G_HD inline double ms_row_self(const RedLayout &R, int o, int item, int lane, double d, const S &s,
                                 const X &x, const M &m, double *sq = nullptr)
{
    const DevLayout &L = R.L;
    const int g0 = L.gems_ab[0];
    const int pr = L.bab[L.bab_off[0] + item], k = P0(pr), l = P1(pr);
    const double own = m[o * g0 + item];
    double v = 0.0;
    for (int i = lane; i < L.amo; i += R.lanes) {
        // the row's pairs are (q, r) and (s, p)
        const int64_t e = o ? ab_pos(R, l, i, i, k) : ab_pos(R, i, k, l, i);
        double q = d * s[R.soff[SF_G2BA] + e] - x[e] - own;
        if (k == l) q -= m[(1 - o) * g0 + L.gab[i * L.amo + i]];   // of both orientations
        if (i == l) q += o ? x[d1_col(L, XB_D1B, l, k)] : x[d1_col(L, XB_D1B, k, l)];   // p == r
        v += q;
        if (sq && !(o && k == l)) *sq += q * q;
    }
    return v;
}

// ---- explicit rows that are not aligned with cells: their value on a D vector --
// a trace, S^2 or contraction row: lane-strided share of `lanes` threads
template <class X>
V2G_HD inline double long_row(const RedLayout &R, const Segment &sg, int64_t item, int lane, int lanes,
                              const X &x)
{
    const DevLayout &L = R.L;
    const int amo = L.amo;
    double v = 0.0;
    if (sg.kind == RF_CONTR) {
        const int n = sg.dim, sub = sg.sub;
        const int i = (int)(item / n) + L.poff[sg.h], j = (int)(item % n) + L.poff[sg.h];
        const bool beta = sub == 1 || sub == 3 || sub == 5;
        if (lane == 0) {
            const double c = sub == 0 ? L.nb : sub == 1 ? L.na : sub == 2 ? L.na - 1.0
                           : sub == 3 ? L.nb - 1.0 : L.na + L.nb - 1.0;
            v += c * x[d1_col(L, beta ? XB_D1B : XB_D1A, i, j)];
        }
        for (int k = lane; k < amo; k += lanes) {
            if (sub < 2 || sub >= 4) v -= x[beta ? ab_pos(R, k, i, k, j) : ab_pos(R, i, k, j, k)];
            if (sub >= 2 && i != k && j != k) {
                const double s2 = ((i < k) == (j < k)) ? 1.0 : -1.0;
                v -= s2 * x[R.nAB + (beta ? R.nAA : 0) + aa_pos(R, i, k, j, k)];
            }
        }
        return v;
    }
    for (int pq = lane; pq < amo * amo; pq += lanes) {
        const int i = pq / amo, j = pq % amo;
        if (sg.kind == RF_S2) {
            v += x[ab_pos(R, i, j, j, i)];
            continue;
        }
        if (sg.sub == 0 || sg.sub == 3) v += (sg.sub ? 2.0 : 1.0) * x[ab_pos(R, i, j, i, j)];
        if (sg.sub > 0 && i != j) {
            const int64_t k = R.nAB + aa_pos(R, i, j, i, j);
            if (sg.sub != 2) v += x[k];
            if (sg.sub != 1) v += x[k + R.nAA];
        }
    }
    return v;
}

// ---- rows of the full layout -------------------------------------------------
V2G_HD inline int64_t row_tab(const RedLayout &R, int tab, int x, int y)
{
    return R.rowtab[(tab * R.L.amo + x) * R.L.amo + y];
}

// the row of the full layout that family f's slot of an aligned entry stands for
V2G_HD inline int64_t self_row_ab(const RedLayout &R, int f, const AbEntry &a)
{
    const int p = a.p, q = a.q, r = a.r, s = a.s;
    switch (f) {
    case SF_Q2AB: return row_tab(R, RT_Q2, p, q) + row_tab(R, RT_AB, r, s);
    case SF_G2AB: return row_tab(R, RT_G2AB, p, s) + row_tab(R, RT_AB, r, q);
    case SF_G2BA: return row_tab(R, RT_G2BA, q, r) + row_tab(R, RT_AB, s, p);
    case SF_G2X: return row_tab(R, RT_GA, p, r) + row_tab(R, RT_GG, s, q);
    case SF_G2Y: return row_tab(R, RT_GB, q, s) + row_tab(R, RT_AB, r, p);
    case SF_G2A: return row_tab(R, RT_GA, p, s) + row_tab(R, RT_AB, r, q);
    case SF_G2B: return row_tab(R, RT_GB, p, s) + row_tab(R, RT_GG, r, q);
    default: {
        const int k = f - SF_D0;
        return row_tab(R, k & 2 ? RT_D1 : RT_D0, p, q) + row_tab(R, k & 1 ? RT_GG : RT_AB, r, s);
    }
    }
}

// the D1 + Q1 row of D1 entry `item` of irrep h
V2G_HD inline int64_t self_row_d1(const DevLayout &Lo, int sp, int h, int64_t item)
{
    const int n = Lo.amopi[h];
    return Lo.rowoff[RF_D1Q1][sp][h] + (item % n) * n + item / n;
}

// A^T y on entry a of the D2ab blocks / the cell a of the D2aa, D2bb blocks, from full rows
// (y's rows of the full layout Lo)
template <class Y>
V2G_HD inline double full_at_ab(const RedLayout &R, const DevLayout &Lo, const AbEntry &a, const Y &y)
{
    const int p = a.p, q = a.q, r = a.r, s = a.s;
    double t = 0.0;
    if (p == r && q == s) t += Lo.sz ? y[Lo.rowoff[RF_TRACE][0][0]] : 2.0 * y[Lo.rowoff[RF_TRACE][3][0]];
    if (q == s) {   // D2ab -> D1a
        const int h = Lo.sym[p], n = Lo.amopi[h];
        t -= y[Lo.rowoff[RF_CONTR][Lo.sz ? 0 : 4][h] + (p - Lo.poff[h]) * n + (r - Lo.poff[h])];
    }
    if (p == r) {   // D2ab -> D1b
        const int h = Lo.sym[q], n = Lo.amopi[h];
        t -= y[Lo.rowoff[RF_CONTR][Lo.sz ? 1 : 5][h] + (q - Lo.poff[h]) * n + (s - Lo.poff[h])];
    }
    if (Lo.spin && p == s && q == r) t += y[Lo.rowoff[RF_S2][0][0]];
    if (R.cells && a.cc) {
        const int h = Lo.sym[p] ^ Lo.sym[q];
        const int64_t k = a.k - R.aa0[h];
        const double an = 0.5 * (y[Lo.rowoff[RF_SPIN_ANTI][0][h] + k] + y[Lo.rowoff[RF_SPIN_ANTI][1][h] + k]);
        t += (p > q) == (r > s) ? -an : an;
    }
    for (int b = 0; b < R.nblk_d; b++) {
        double c[4];
        d200_coef(b, Lo.singlet, p == q, r == s, c);
        const int tr = b & 2 ? RT_D1 : RT_D0, tc = b & 1 ? RT_GG : RT_AB;
        const int64_t pq = row_tab(R, tr, p, q), qp = row_tab(R, tr, q, p), rs = row_tab(R, tc, r, s),
                      sr = row_tab(R, tc, s, r);
        t += c[0] * y[pq + rs] + c[1] * y[qp + rs] + c[2] * y[pq + sr] + c[3] * y[qp + sr];
    }
    auto row = [&](int f) { return y[self_row_ab(R, f, a)]; };
    if (Lo.q2) t += row(SF_Q2AB);
    if (Lo.g2) t += (row(SF_G2X) + row(SF_G2Y)) - (row(SF_G2AB) + row(SF_G2BA));
    return t;
}

template <class Y>
V2G_HD inline double full_at_aa(const DevLayout &Lo, int sp, const AbEntry &a, const Y &y)
{
    Segment sg{};
    sg.h = Lo.sym[a.p] ^ Lo.sym[a.q];
    sg.sub = sp;
    sg.dim = Lo.gems_aa[sg.h];
    return atu_d2aa(Lo, sg, (int64_t)Lo.gaa[a.p * Lo.amo + a.q] * sg.dim + Lo.gaa[a.r * Lo.amo + a.s], y);
}

// ---- listed entries ------------------------------------------------------------
// p == q or r == s
V2G_HD inline AbRec make_ab_rec(const RedLayout &R, int p, int q, int r, int s)
{
    const DevLayout &L = R.L;
    AbRec a;
    a.pos = (int32_t)ab_pos(R, p, q, r, s);
    a.p1 = (int32_t)ab_pos(R, q, p, r, s);
    a.p2 = (int32_t)ab_pos(R, p, q, s, r);
    a.p3 = (int32_t)ab_pos(R, q, p, s, r);
    a.pr = (int32_t)(q == s ? d1_col(L, XB_D1A, p, r) : R.nD);
    a.rp = (int32_t)(q == s ? d1_col(L, XB_D1A, r, p) : R.nD);
    a.qs = (int32_t)(p == r ? d1_col(L, XB_D1B, q, s) : R.nD);
    a.sq = (int32_t)(p == r ? d1_col(L, XB_D1B, s, q) : R.nD);
    a.m0 = R.nM && s == p ? L.gab[q * L.amo + r] : R.nM;
    a.m1 = R.nM && q == r ? L.gems_ab[0] + L.gab[s * L.amo + p] : R.nM;
    a.flags = (p == q ? AF_BRA : 0) | (r == s ? AF_KET : 0) | (q == s ? AF_QS : 0) | (p == r ? AF_PR : 0) |
              (p == s && q == r ? AF_S2 : 0);
    return a;
}

// p > q, r > s with a common orbital
V2G_HD inline CellRec make_cell_rec(const RedLayout &R, int p, int q, int r, int s)
{
    const DevLayout &L = R.L;
    const int h = L.sym[p] ^ L.sym[q];
    CellRec c;
    c.pos = (int32_t)ab_pos(R, p, q, r, s);
    c.k = (int32_t)aa_pos(R, p, q, r, s);
    c.row = (int32_t)(c.k - R.aa0[h]);
    c.flags = h << 8;
    int n = 0;
    for (int u = 0; u < 2; u++)
        for (int w = 0; w < 2; w++) {
            // bra (i,l), ket (j,k) by orientation u + 2 w of the cell; l == k is shared
            const int i = u ? q : p, l = u ? p : q, j = w ? s : r, k = w ? r : s;
            if (k != l || n == 2) continue;
            c.ij[n] = (int32_t)d1_col(L, XB_D1A, i, j);
            c.ji[n] = (int32_t)d1_col(L, XB_D1A, j, i);
            c.m0[n] = R.nM ? L.gab[i * L.amo + j] : 0;
            c.m1[n] = R.nM ? L.gems_ab[0] + L.gab[j * L.amo + i] : 0;
            c.flags |= (u + 2 * w) << (2 * n);
            if (n) c.flags |= CF_TWO;
            n++;
        }
    if (n == 1) {
        c.ij[1] = c.ij[0];
        c.ji[1] = c.ji[0];
        c.m0[1] = c.m0[0];
        c.m1[1] = c.m1[0];
    }
    return c;
}

// what a listed D2ab entry reads of a D vector
struct AbVals {
    double x0, x1, x2, x3, arp, apr, bpr, bsq, bqs;
    template <class X>
    V2G_HD inline AbVals(const RedLayout &R, const AbRec &a, const X &x)
    {
        x0 = x[a.pos];
        x1 = x[a.p1];
        x2 = x[a.p2];
        x3 = x[a.p3];
        arp = x[a.rp];
        apr = x[a.pr];
        bpr = x[a.flags & AF_QS ? a.pr + (int32_t)R.nD1 : a.pr];
        bsq = x[a.sq];
        bqs = x[a.qs];
    }
    V2G_HD inline double q2() const { return x0 - arp - bsq; }
    V2G_HD inline double g1() const { return apr - x0; }
    V2G_HD inline double g2() const { return bqs - x0; }
    V2G_HD inline double ga(const AbRec &) const { return apr; }
    V2G_HD inline double gb(const AbRec &) const { return bpr; }
    V2G_HD inline double d200(const RedLayout &R, const AbRec &a, int blk) const
    {
        double c[4];
        d200_coef(blk, R.L.singlet, (a.flags & AF_BRA) != 0, (a.flags & AF_KET) != 0, c);
        return c[0] * x0 + c[1] * x1 + c[2] * x2 + c[3] * x3;
    }
    // B2^T B2 x (the maximal-spin part, nu[m0] + nu[m1], is the caller's)
    V2G_HD inline double gram(const RedLayout &R, const AbRec &a) const
    {
        double t = (R.L.q2 ? x0 - arp - bsq : 0.0) + (R.L.g2 ? 4.0 * x0 - apr - bqs : 0.0);
        if (R.nblk_d) {
            const double ip = a.flags & AF_BRA ? 0.5 : 1.0, ir = a.flags & AF_KET ? 0.5 : 1.0;
            t += (ip * ir) * ((x0 + x1) + (x2 + x3));
            if (!R.L.singlet) {
                t += ip * ((x0 + x1) - (x2 + x3));
                t += ir * ((x0 + x2) - (x1 + x3));
                t += (x0 + x3) - (x1 + x2);
            }
        }
        return t;
    }
};

// the explicit rows' share of A^T on a listed D2ab entry
template <class Y>
V2G_HD inline double rec_expl_ab(const RedLayout &R, const AbRec &a, const Y &y)
{
    const DevLayout &L = R.L;
    const bool A = a.flags & AF_QS, B = a.flags & AF_PR;
    const int64_t ca = L.rowoff[RF_CONTR][L.sz ? 0 : 4][0] + (a.pr - L.xoff[XB_D1A][0]);
    const int64_t cb = L.rowoff[RF_CONTR][L.sz ? 1 : 5][0] + (a.qs - L.xoff[XB_D1B][0]);
    const int64_t tr = L.rowoff[RF_TRACE][L.sz ? 0 : 3][0];
    double v = (L.sz ? 1.0 : 2.0) * y[A && B ? tr : R.nR] - y[A ? ca : R.nR] - y[B ? cb : R.nR];
    if (L.spin) v += y[a.flags & AF_S2 ? L.rowoff[RF_S2][0][0] : R.nR];
    return v;
}

// ---- a cell whose pairs share no orbital --------------------------------------
// its numbers in a D vector: the four D2ab entries by orientation, D2aa, D2bb
struct Cell {
    double ab[4], aa, bb;
};

template <class X>
V2G_HD inline Cell load_cell(const RedLayout &R, int64_t pos, int64_t cc, int64_t k, const X &x)
{
    Cell c;
    for (int o = 0; o < 4; o++) c.ab[o] = x[pos + o * cc];
    c.aa = x[R.nAB + k];
    c.bb = x[R.nAB + R.nAA + k];
    return c;
}

// t = d g + B2^T B2 v + B1^T p on the cell (pr: its three explicit rows' p)
V2G_HD inline Cell cell_at(bool q2, bool g2, int nd, bool cells, double d, const Cell &g, const Cell &v,
                           const double (&pr)[3])
{
    const double w = (q2 ? 1.0 : 0.0) + (g2 ? 4.0 : 0.0), wd = w + (nd == 4 ? 4.0 : 0.0);
    const double sum = nd == 1 ? (v.ab[0] + v.ab[1]) + (v.ab[2] + v.ab[3]) : 0.0;
    const double an = cells ? 0.5 * (pr[1] + pr[2]) : 0.0;
    Cell t;
    for (int o = 0; o < 4; o++)
        t.ab[o] = d * g.ab[o] + wd * v.ab[o] + sum + (o == 1 || o == 2 ? an : -an);
    t.aa = d * g.aa + w * v.aa + (cells ? pr[0] + pr[1] : 0.0);
    t.bb = d * g.bb + w * v.bb + (cells ? pr[2] - pr[0] : 0.0);
    return t;
}

// the cell's three explicit rows on t
V2G_HD inline void cell_rows(const Cell &t, double (&a)[3])
{
    const double an = 0.5 * ((t.ab[1] + t.ab[2]) - (t.ab[0] + t.ab[3]));
    a[0] = t.aa - t.bb;
    a[1] = t.aa + an;
    a[2] = t.bb + an;
}

// ---- a listed cell: what a shared orbital adds ---------------------------------
V2G_HD inline int shared_count(const CellRec &c) { return c.flags & CF_TWO ? 2 : 1; }
// orientation of (ik|jk); (ki|kj), (ki|jk), (ik|kj) are it xor 3, 1, 2
V2G_HD inline int shared_or(const CellRec &c, int n) { return c.flags >> (2 * n) & 3; }

// whether a maximal-spin row reads the G2ba row of orientation o of the cell
V2G_HD inline bool shared_ms(const RedLayout &R, const CellRec &c, int o)
{
    const int a = o ^ shared_or(c, 0), b = c.flags & CF_TWO ? o ^ shared_or(c, 1) : 0;
    return R.nM && (a == 1 || a == 2 || b == 1 || b == 2);
}

// a shared orbital's D1 and maximal-spin numbers
struct Shared {
    double aij, aji, bij, bji, m0, m1;
    template <class X, class M>
    V2G_HD inline Shared(const RedLayout &R, const CellRec &c, int n, const X &x, const M &m)
    {
        aij = x[c.ij[n]];
        aji = x[c.ji[n]];
        bij = x[c.ij[n] + (int32_t)R.nD1];
        bji = x[c.ji[n] + (int32_t)R.nD1];
        m0 = R.nM ? m[c.m0[n]] : 0.0;
        m1 = R.nM ? m[c.m1[n]] : 0.0;
    }
};

V2G_HD inline void add_or(double (&v)[4], int o, double x)
{
    for (int k = 0; k < 4; k++) v[k] += k == o ? x : 0.0;
}

// adds the terms of the shared orbitals, traces and S^2 to t = cell_at(...)
template <class X, class M, class Y>
V2G_HD inline void shared_at(const RedLayout &R, const CellRec &c, const X &x, const M &m, const Y &y, Cell &t)
{
    const DevLayout &L = R.L;
    const int64_t c0 = L.rowoff[RF_CONTR][L.sz ? 0 : 4][0] - L.xoff[XB_D1A][0];
    const int64_t c1 = L.rowoff[RF_CONTR][L.sz ? 1 : 5][0] - L.xoff[XB_D1A][0];
    const int64_t c2 = L.rowoff[RF_CONTR][L.sz ? 2 : 4][0] - L.xoff[XB_D1A][0];
    const int64_t c3 = L.rowoff[RF_CONTR][L.sz ? 3 : 5][0] - L.xoff[XB_D1A][0];
    const double q2 = L.q2 ? 1.0 : 0.0, g2 = L.g2 ? 1.0 : 0.0;
    for (int n = 0; n < shared_count(c); n++) {
        const Shared s(R, c, n, x, m);
        const int o = shared_or(c, n);
        add_or(t.ab, o, -(q2 * s.aji + g2 * s.aij + y[c0 + c.ij[n]]));
        add_or(t.ab, o ^ 3, -(q2 * s.bji + g2 * s.bij + y[c1 + c.ij[n]]));
        add_or(t.ab, o ^ 1, g2 * s.m0);
        add_or(t.ab, o ^ 2, g2 * s.m1);
        // like spins: the pairs' order decides the sign
        const double sg = o == 0 || o == 3 ? -1.0 : 1.0;
        t.aa += sg * (q2 * s.aji + g2 * s.aij + y[c2 + c.ij[n]]);
        t.bb += sg * (q2 * s.bji + g2 * s.bij + y[c3 + c.ij[n]]);
    }
    if (c.flags & CF_TWO) {   // the same pair twice: a diagonal entry
        const double tr = L.sz ? y[L.rowoff[RF_TRACE][0][0]] : 2.0 * y[L.rowoff[RF_TRACE][3][0]];
        t.ab[0] += tr;
        t.ab[3] += tr;
        if (L.spin) {
            const double s2 = y[L.rowoff[RF_S2][0][0]];
            t.ab[1] += s2;
            t.ab[2] += s2;
        }
        t.aa += 2.0 * y[L.rowoff[RF_TRACE][L.sz ? 1 : 3][0]];
        t.bb += 2.0 * y[L.rowoff[RF_TRACE][L.sz ? 2 : 3][0]];
    }
}

// the D1 / maximal-spin part that the shared orbitals add to a cell's self rows in
// orientation o: Q2ab, G2ab (and the alpha quadrant), G2ba, the beta quadrant
struct SharedAt {
    double q2 = 0.0, g1 = 0.0, g2 = 0.0, gb = 0.0;
    template <class X, class M>
    V2G_HD inline SharedAt(const RedLayout &R, const CellRec &c, int o, const X &x, const M &m)
    {
        const int32_t b = (int32_t)R.nD1;
        for (int n = 0; n < shared_count(c); n++) {
            const int rel = o ^ shared_or(c, n);
            if (rel == 0) {          // (ik|jk)
                q2 -= x[c.ji[n]];
                g1 += x[c.ij[n]];
                gb += x[c.ij[n] + b];
            } else if (rel == 3) {   // (ki|kj)
                q2 -= x[c.ji[n] + b];
                g2 += x[c.ij[n] + b];
            } else if (R.nM) {       // (ki|jk), (ik|kj)
                g2 -= m[rel == 1 ? c.m0[n] : c.m1[n]];
            }
        }
    }
};

// what they add to the cell's Q2aa (sp = 0) / Q2bb row
template <class X>
V2G_HD inline double shared_q2(const RedLayout &R, const CellRec &c, int sp, const X &x)
{
    const int32_t b = sp ? (int32_t)R.nD1 : 0;
    double v = 0.0;
    for (int n = 0; n < shared_count(c); n++) {
        const int o = shared_or(c, n);
        v += o == 0 || o == 3 ? -x[c.ji[n] + b] : x[c.ji[n] + b];
    }
    return v;
}

}  // namespace rows
}  // namespace v2g
