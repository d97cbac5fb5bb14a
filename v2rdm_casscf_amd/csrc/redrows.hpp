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
// its slot is that entry's, and all index permutations of the G2 maps vanish.
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
    // compact view: xoff of the D2 / D1 blocks in a vector of nD entries, rowoff
    // of the explicit rows in a vector of nR entries; other blocks and rows absent
    DevLayout L;
    int64_t soff[SF_COUNT][kMaxIrrep];   // slot ranges in the self vector, -1 absent
    int64_t nD, nR, nS;
    int nM;          // maximal-spin rows (2 gems_ab[0], or 0); their rowoff is compact too
    int nblk_d;      // D200 quadrants: 0 (spin off), 1 (singlet), 4
};

namespace rows {

struct AbEntry {
    int h, IJ, KL, p, q, r, s;
    int64_t e;       // IJ g + KL
};

V2G_HD inline AbEntry ab_entry(const DevLayout &L, int h, int64_t e)
{
    AbEntry a;
    a.h = h;
    a.e = e;
    split_index(e, L.gems_ab[h], a.IJ, a.KL);
    const int pij = L.bab[L.bab_off[h] + a.IJ], pkl = L.bab[L.bab_off[h] + a.KL];
    a.p = P0(pij);
    a.q = P1(pij);
    a.r = P0(pkl);
    a.s = P1(pkl);
    return a;
}

// slot of (pq|rs) within its irrep's aligned range
V2G_HD inline int64_t ab_slot(const DevLayout &L, int p, int q, int r, int s)
{
    return (int64_t)L.gab[p * L.amo + q] * L.gems_ab[L.sym[p] ^ L.sym[q]] + L.gab[r * L.amo + s];
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

// the D2 / D1 parts of the Q2 and G2 rows aligned with entry a; X is a vector of nD
// entries
template <class X>
struct SelfAb {
    double x, q2, g1, g2, ga, gb;   // x: the mixed-spin quadrants' part too
    V2G_HD inline SelfAb(const RedLayout &R, const AbEntry &a, const X &v)
    {
        const DevLayout &L = R.L;
        x = v[L.xoff[XB_D2AB][a.h] + a.e];
        q2 = x;
        g1 = g2 = -x;
        ga = gb = 0.0;
        if (L.g2 && a.p != a.q && a.r != a.s) {
            const int64_t k = (int64_t)L.gaa[a.p * L.amo + a.q] * L.gems_aa[a.h] + L.gaa[a.r * L.amo + a.s];
            const double sg = ((a.p < a.q) == (a.r < a.s)) ? -1.0 : 1.0;
            ga = sg * v[L.xoff[XB_D2AA][a.h] + k];
            gb = sg * v[L.xoff[XB_D2BB][a.h] + k];
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
        const DevLayout &L = R.L;
        const int64_t b = L.xoff[XB_D2AB][a.h], g = L.gems_ab[a.h];
        const int64_t qp = L.gab[a.q * L.amo + a.p], sr = L.gab[a.s * L.amo + a.r];
        v0 = v[b + a.e];
        v1 = v[b + qp * g + a.KL];
        v2 = v[b + a.IJ * g + sr];
        v3 = v[b + qp * g + sr];
    }
    V2G_HD inline double row(const RedLayout &R, const AbEntry &a, int blk) const
    {
        double c[4];
        d200_coef(blk, R.L.singlet, a.p == a.q, a.r == a.s, c);
        return c[0] * v0 + c[1] * v1 + c[2] * v2 + c[3] * v3;
    }
};

// the D2 / D1 part of a Q2aa / Q2bb row (spin sp) at entry e of irrep h
template <class X>
V2G_HD inline double self_row_aa(const RedLayout &R, int sp, int h, int64_t e, const X &x)
{
    const DevLayout &L = R.L;
    int IJ, KL;
    split_index(e, L.gems_aa[h], IJ, KL);
    const int pij = L.baa[L.baa_off[h] + IJ], pkl = L.baa[L.baa_off[h] + KL];
    const int i = P0(pij), j = P1(pij), k = P0(pkl), l = P1(pkl), wd = sp ? XB_D1B : XB_D1A;
    double v = x[L.xoff[sp ? XB_D2BB : XB_D2AA][h] + e];
    if (j == l) v -= x[d1_col(L, wd, k, i)];
    if (j == k) v += x[d1_col(L, wd, l, i)];
    if (i == l) v += x[d1_col(L, wd, k, j)];
    if (i == k) v -= x[d1_col(L, wd, l, j)];
    return v;
}

// (P m)(e): the maximal-spin generator on the G2ba row of the aligned entry a
// (non-zero on irrep 0 only: s == p or q == r imply it)
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

// (B2^T B2 x)(e) + (the G2ba rows' share of -B2^T P m, whose sign is +): a D2ab entry
template <class X, class M>
V2G_HD inline double gram_ab(const RedLayout &R, const AbEntry &a, const X &x, const M &m)
{
    const DevLayout &L = R.L;
    const double v = x[L.xoff[XB_D2AB][a.h] + a.e];
    double t = (L.q2 ? v : 0.0) + (L.g2 ? 4.0 * v : 0.0);
    if (a.q == a.s) {
        if (L.q2) t -= x[d1_col(L, XB_D1A, a.r, a.p)];
        if (L.g2) t -= x[d1_col(L, XB_D1A, a.p, a.r)];
    }
    if (a.p == a.r) {
        if (L.q2) t -= x[d1_col(L, XB_D1B, a.s, a.q)];
        if (L.g2) t -= x[d1_col(L, XB_D1B, a.q, a.s)];
    }
    if (L.g2) t += ms_part(R, a.p, a.q, a.r, a.s, m);
    if (R.nblk_d) {
        const D200Ab<X> w(R, a, x);
        // sum over a row's four source entries of (coefficient x row value)
        const double ip = a.p == a.q ? 0.5 : 1.0, ir = a.r == a.s ? 0.5 : 1.0;
        t += (ip * ir) * ((w.v0 + w.v1) + (w.v2 + w.v3));
        if (!L.singlet) {
            t += ip * ((w.v0 + w.v1) - (w.v2 + w.v3));
            t += ir * ((w.v0 + w.v2) - (w.v1 + w.v3));
            t += (w.v0 + w.v3) - (w.v1 + w.v2);
        }
    }
    return t;
}

// the same for a D2aa / D2bb entry (spin sp)
template <class X>
V2G_HD inline double gram_aa(const RedLayout &R, int sp, int h, int64_t e, const X &x)
{
    const DevLayout &L = R.L;
    double t = L.q2 ? self_row_aa(R, sp, h, e, x) : 0.0;
    if (L.g2) {
        int IJ, KL;
        split_index(e, L.gems_aa[h], IJ, KL);
        const int pij = L.baa[L.baa_off[h] + IJ], pkl = L.baa[L.baa_off[h] + KL];
        const int wd = sp ? XB_D1B : XB_D1A;
        t += 4.0 * x[L.xoff[sp ? XB_D2BB : XB_D2AA][h] + e];
        // rows ((i,j),(k,l)) of the like-spin quadrant, {i,l} = pair 1, {k,j} = pair 2
        for (int a = 0; a < 2; a++)
            for (int b = 0; b < 2; b++) {
                const int i = a ? P1(pij) : P0(pij), l = a ? P0(pij) : P1(pij);
                const int k = b ? P1(pkl) : P0(pkl), j = b ? P0(pkl) : P1(pkl);
                if (j != l) continue;
                const double sg = ((i < l) == (k < j)) ? 1.0 : -1.0;
                t -= sg * x[d1_col(L, wd, i, k)];
            }
    }
    return t;
}

// the same for a D1 entry: lane-strided share of one wavefront
template <class X, class M>
V2G_HD inline double gram_d1(const RedLayout &R, int sp, int h, int64_t item, int lane, const X &x,
                             const M &m)
{
    const DevLayout &L = R.L;
    const int amo = L.amo, n = L.amopi[h];
    const int A = (int)(item / n) + L.poff[h], B = (int)(item % n) + L.poff[h];
    const int wd = sp ? XB_D1B : XB_D1A, wo = sp ? XB_D1A : XB_D1B;
    const double xd = x[L.xoff[wd][h] + item];
    double v = lane == 0 ? xd : 0.0;   // D1 + Q1 row
    for (int t = lane; t < amo; t += 64) {
        const int ht = L.sym[B] ^ L.sym[t];
        const int64_t bt = sp ? L.gab[t * amo + B] : L.gab[B * amo + t];
        const int64_t at = sp ? L.gab[t * amo + A] : L.gab[A * amo + t];
        const int64_t g = L.gems_ab[ht], bab = L.xoff[XB_D2AB][ht];
        if (L.q2) {
            v -= x[bab + bt * g + at] - xd;
            if (A == B) v += x[d1_col(L, wo, t, t)];
            if (t != A && t != B) {
                const double sg = ((B > t) == (A > t)) ? 1.0 : -1.0;
                v -= sg * self_row_aa(R, sp, ht,
                                      (int64_t)L.gaa[B * amo + t] * L.gems_aa[ht] + L.gaa[A * amo + t], x);
            }
        }
        if (L.g2) {
            v += xd - x[bab + at * g + bt];     // G2ab (alpha) / G2ba (beta)
            if (sp) v -= ms_part(R, t, A, t, B, m);
            v += xd;                            // like-spin quadrant
            if (t != A && t != B) {
                const double sg = ((A < t) == (B < t)) ? 1.0 : -1.0;
                v -= sg * x[L.xoff[sp ? XB_D2BB : XB_D2AA][ht] +
                            (int64_t)L.gaa[A * amo + t] * L.gems_aa[ht] + L.gaa[B * amo + t]];
            }
        }
    }
    return v;
}

// B2^T s: the self rows' share of A^T on a D2ab / D2aa / D1 entry from aligned slots
template <class S>
V2G_HD inline double self_at_ab(const RedLayout &R, const AbEntry &a, const S &s)
{
    const DevLayout &L = R.L;
    const int64_t g = L.gems_ab[a.h];
    double t = 0.0;
    if (L.q2) t += s[R.soff[SF_Q2AB][a.h] + a.e];
    if (L.g2)
        t += (s[R.soff[SF_G2X][a.h] + a.e] + s[R.soff[SF_G2Y][a.h] + a.e]) -
             (s[R.soff[SF_G2AB][a.h] + a.e] + s[R.soff[SF_G2BA][a.h] + a.e]);
    if (R.nblk_d) {
        const int64_t qp = L.gab[a.q * L.amo + a.p], sr = L.gab[a.s * L.amo + a.r];
        for (int k = 0; k < R.nblk_d; k++) {
            double c[4];
            d200_coef(k, L.singlet, a.p == a.q, a.r == a.s, c);
            const int64_t b = R.soff[SF_D0 + k][a.h];
            t += c[0] * s[b + a.e] + c[1] * s[b + qp * g + a.KL] + c[2] * s[b + a.IJ * g + sr] +
                 c[3] * s[b + qp * g + sr];
        }
    }
    return t;
}

template <class S>
V2G_HD inline double self_at_aa(const RedLayout &R, int sp, int h, int64_t e, const S &s)
{
    const DevLayout &L = R.L;
    double t = L.q2 ? s[R.soff[sp ? SF_Q2BB : SF_Q2AA][h] + e] : 0.0;
    if (L.g2) {
        int IJ, KL;
        split_index(e, L.gems_aa[h], IJ, KL);
        const int pij = L.baa[L.baa_off[h] + IJ], pkl = L.baa[L.baa_off[h] + KL];
        const int64_t b0 = R.soff[sp ? SF_G2B : SF_G2A][h], g = L.gems_ab[h];
        for (int a = 0; a < 2; a++)
            for (int b = 0; b < 2; b++) {
                const int i = a ? P1(pij) : P0(pij), l = a ? P0(pij) : P1(pij);
                const int k = b ? P1(pkl) : P0(pkl), j = b ? P0(pkl) : P1(pkl);
                const double sg = ((i < l) == (k < j)) ? 1.0 : -1.0;
                t -= sg * s[b0 + (int64_t)L.gab[i * L.amo + l] * g + L.gab[k * L.amo + j]];
            }
    }
    return t;
}

template <class S>
V2G_HD inline double self_at_d1(const RedLayout &R, int sp, int h, int64_t item, int lane, const S &s)
{
    const DevLayout &L = R.L;
    const int amo = L.amo, n = L.amopi[h];
    const int A = (int)(item / n) + L.poff[h], B = (int)(item % n) + L.poff[h];
    double v = lane == 0 ? s[R.soff[sp ? SF_Q1B : SF_Q1A][h] + item] : 0.0;
    for (int t = lane; t < amo; t += 64) {
        const int ht = L.sym[B] ^ L.sym[t];
        const int64_t g = L.gems_ab[ht];
        const int64_t bt = sp ? L.gab[t * amo + B] : L.gab[B * amo + t];
        const int64_t at = sp ? L.gab[t * amo + A] : L.gab[A * amo + t];
        if (L.q2) {
            v -= s[R.soff[SF_Q2AB][ht] + bt * g + at];
            if (t != A && t != B) {
                const double sg = ((B > t) == (A > t)) ? 1.0 : -1.0;
                v -= sg * s[R.soff[sp ? SF_Q2BB : SF_Q2AA][ht] +
                            (int64_t)L.gaa[B * amo + t] * L.gems_aa[ht] + L.gaa[A * amo + t]];
            }
        }
        if (L.g2) {
            v += s[R.soff[sp ? SF_G2BA : SF_G2AB][ht] + at * g + bt];
            // the like-spin quadrant's row ((A,t),(B,t)) reads (At|Bt)
            v += s[R.soff[sp ? SF_G2B : SF_G2A][ht] + (int64_t)L.gab[A * amo + t] * g + L.gab[B * amo + t]];
        }
    }
    return v;
}

// maximal-spin row `item` of orientation o (0: G2ba entries (kl, ii), 1: (ii, kl)):
// lane-strided share of sum_i p_self over its G2ba rows, p_self = d s + B2 x - P m
template <class S, class X, class M>
V2G_HD inline double ms_row_self(const RedLayout &R, int o, int item, int lane, double d, const S &s,
                                 const X &x, const M &m)
{
    const DevLayout &L = R.L;
    const int pr = L.bab[L.bab_off[0] + item], k = P0(pr), l = P1(pr);
    double v = 0.0;
    for (int i = lane; i < L.amo; i += 64) {
        // the row's pairs are (q, r) and (s, p)
        const int q = o ? i : k, r = o ? i : l, ss = o ? k : i, p = o ? l : i;
        const int hh = L.sym[p] ^ L.sym[q];
        const int64_t e = ab_slot(L, p, q, r, ss);
        v += d * s[R.soff[SF_G2BA][hh] + e] - x[L.xoff[XB_D2AB][hh] + e] - ms_part(R, p, q, r, ss, m);
        if (p == r) v += x[d1_col(L, XB_D1B, q, ss)];
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
        for (int i = lane; i < L.amo; i += 64) v += m[(1 - o) * g0 + L.gab[i * L.amo + i]];
    return v;
}

// the row of the full layout Lo that the slot of family f at an aligned entry stands for
V2G_HD inline int64_t self_row_ab(const DevLayout &Lo, int f, const AbEntry &a)
{
    const int amo = Lo.amo;
    const int *gab = Lo.gab, *sym = Lo.sym;
    const int p = a.p, q = a.q, r = a.r, s = a.s;
    auto GAB = [&](int x, int y) -> int64_t { return gab[x * amo + y]; };
    switch (f) {
    case SF_Q2AB: return Lo.rowoff[RF_Q2AB][0][a.h] + a.e;
    case SF_G2AB: {
        const int h = sym[p] ^ sym[s];
        return Lo.rowoff[RF_G2AB][0][h] + GAB(p, s) * Lo.gems_ab[h] + GAB(r, q);
    }
    case SF_G2BA: {
        const int h = sym[q] ^ sym[r];
        return Lo.rowoff[RF_G2AB][1][h] + GAB(q, r) * Lo.gems_ab[h] + GAB(s, p);
    }
    case SF_G2X: {
        const int h = sym[p] ^ sym[r];
        const int64_t g = Lo.gems_ab[h];
        return Lo.rowoff[RF_G2AA][0][h] + GAB(p, r) * 2 * g + g + GAB(s, q);
    }
    case SF_G2Y: {
        const int h = sym[q] ^ sym[s];
        const int64_t g = Lo.gems_ab[h];
        return Lo.rowoff[RF_G2AA][0][h] + (g + GAB(q, s)) * 2 * g + GAB(r, p);
    }
    case SF_G2A: case SF_G2B: {
        const int h = sym[p] ^ sym[s];
        const int64_t g = Lo.gems_ab[h], b = f == SF_G2B ? g : 0;
        return Lo.rowoff[RF_G2AA][0][h] + (b + GAB(p, s)) * 2 * g + b + GAB(r, q);
    }
    default: {
        if (Lo.singlet) return Lo.rowoff[RF_SPIN_D200][0][a.h] + a.e;
        const int k = f - SF_D0;
        const int64_t g = Lo.gems_ab[a.h];
        return Lo.rowoff[RF_SPIN_D200_4][0][a.h] + (a.IJ + (k >> 1) * g) * 2 * g + a.KL + (k & 1) * g;
    }
    }
}

// the D1 + Q1 row of D1 entry `item` of irrep h
V2G_HD inline int64_t self_row_d1(const DevLayout &Lo, int sp, int h, int64_t item)
{
    const int n = Lo.amopi[h];
    return Lo.rowoff[RF_D1Q1][sp][h] + (item % n) * n + item / n;
}

}  // namespace rows
}  // namespace v2g
