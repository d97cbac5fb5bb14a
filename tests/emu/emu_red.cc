// emu_red.cc -- host execution of the reduced plain CG (csrc/redrows.hpp) with
// the device row code, for the CPU test suite: every vector read is checked
// against its buffer.
#include <cmath>
#include <cstdint>
#include <vector>

#include "../../v2rdm_casscf_amd/csrc/redcg.hpp"

using namespace v2g;
using namespace v2g::rows;

namespace {

long long g_viol;

struct Vec {
    std::vector<double> v;
    explicit Vec(int64_t n) : v((size_t)n, 0.0) {}
    double operator[](int64_t i) const
    {
        if (i < 0 || i >= (int64_t)v.size()) { g_viol++; return 0.0; }
        return v[i];
    }
    double &at(int64_t i)
    {
        static double sink;
        if (i < 0 || i >= (int64_t)v.size()) { g_viol++; return sink; }
        return v[i];
    }
};

struct View {
    const double *p;
    int64_t n;
    double operator[](int64_t i) const
    {
        if (i < 0 || i >= n) { g_viol++; return 0.0; }
        return p[i];
    }
};

struct VGather {
    const Vec &x;
    double acc = 0.0;
    void operator()(int64_t col, double c) { acc += c * x[col]; }
};

}  // namespace

extern "C" {

// maxiter iterations of CG on A A^T y = rhs (stops below tol); res: ||r|| after
// each; returns the iteration count (CGSolver::solve's), -1 for a layout that
// the reduced form does not cover, -2 when an index left its buffer
int emu_red_cg(int nirrep, const int *amopi, int na, int nb, int mult, int q2, int g2, int t2, int t1,
               int spin, int sz, const double *rhs_, double *y_, long long ncon, double tol,
               int maxiter, double *res)
{
    Options op;
    op.nirrep = nirrep;
    for (int h = 0; h < 8; h++) op.amopi[h] = h < nirrep ? amopi[h] : 0;
    op.nalpha = na;
    op.nbeta = nb;
    op.multiplicity = mult;
    op.q2 = q2;
    op.g2 = g2;
    op.t2 = t2;
    op.t1 = t1;
    op.spin = spin;
    op.sz = sz;
    Layout L(op);
    const DevLayout Lo = make_dev_layout(L, {L.sym.data(), L.gab.data(), L.gaa.data(), L.bab.data(),
                                             L.baa.data(), L.baab.data(), L.baba.data(),
                                             L.baaa.data(), L.b00.data()});
    RedLayout R;
    RedWork W;
    if (!make_red_layout(L, Lo, R, W)) return -1;
    if (R.nS + R.nR != L.ncon || ncon != L.ncon) return -3;
    g_viol = 0;
    const View rhs{rhs_, ncon}, y{y_, ncon};
    Vec t(R.nD), g(R.nD), u(R.nD), v(R.nD), wv(R.nD), s(R.nS), r(R.nR), p(R.nR), mu(R.nM), nu(R.nM),
        om(R.nM), ams(R.nM);
    const int64_t ms0 = R.nM ? R.L.rowoff[RF_MAXSPIN][0][0] : 0;
    // A^T y on the D entries, from the full rows
    for (const Segment &sg : W.p)
        for (int64_t e = 0; sg.kind <= XS_SELF && e < sg.count; e++) {
            double a = 0.0;
            if (sg.kind == XS_D2AB) a = atu_d2ab(Lo, sg, e, y);
            else if (sg.kind == XS_D2AA) a = atu_d2aa(Lo, sg, e, y);
            else for (int l = 0; l < 64; l++) a += atu_d1_wave(Lo, sg, e, l, y);
            t.at(sg.start + e) = a;
        }
    // visits every self slot: fn(slot, full row, D part of x, P part of m, is G2ba)
    auto each_self = [&](const Vec &x, const Vec &m, auto fn) {
        std::vector<char> seen((size_t)R.nS, 0);
        for (const Segment &sg : W.n)
            for (int64_t e = 0; e < sg.count; e++) {
                auto visit = [&](int64_t slot, int64_t row, double dx, double pm) {
                    if (slot < 0 || slot >= R.nS || seen[slot]++ || row < 0 || row >= ncon) { g_viol++; return; }
                    fn(slot, row, dx, pm);
                };
                if (sg.kind == XS_D2AB) {
                    const AbEntry a = ab_entry(R.L, sg.h, e);
                    const SelfAb<Vec> o(R, a, x);
                    auto one = [&](int f, double dx, double pm) { visit(R.soff[f][sg.h] + e, self_row_ab(Lo, f, a), dx, pm); };
                    if (R.L.q2) one(SF_Q2AB, o.q2, 0.0);
                    if (R.L.g2) {
                        one(SF_G2AB, o.g1, 0.0);
                        one(SF_G2BA, o.g2, ms_part(R, a.p, a.q, a.r, a.s, m));
                        one(SF_G2X, o.x, 0.0);
                        one(SF_G2Y, o.x, 0.0);
                        one(SF_G2A, o.ga, 0.0);
                        one(SF_G2B, o.gb, 0.0);
                    }
                    if (R.nblk_d) {
                        const D200Ab<Vec> d(R, a, x);
                        for (int k = 0; k < R.nblk_d; k++) one(SF_D0 + k, d.row(R, a, k), 0.0);
                    }
                } else if (sg.kind == XS_D2AA) {
                    const int f = sg.sub ? SF_Q2BB : SF_Q2AA;
                    if (R.soff[f][sg.h] >= 0)
                        visit(R.soff[f][sg.h] + e, Lo.rowoff[RF_Q2AA][sg.sub][sg.h] + e,
                              self_row_aa(R, sg.sub, sg.h, e, x), 0.0);
                } else {
                    visit(R.soff[sg.sub ? SF_Q1B : SF_Q1A][sg.h] + e, self_row_d1(Lo, sg.sub, sg.h, e),
                          x[sg.start + e], 0.0);
                }
            }
        for (char c : seen) if (c != 1) g_viol++;
    };
    // explicit rows of A t; the maximal-spin rows take theirs from msrow
    auto explicit_rows = [&](auto msrow, auto fn) {
        for (const Segment &sg : W.r) {
            if (sg.kind >= RK_ROWS) continue;
            for (int64_t e = 0; e < sg.count; e++) {
                double a = 0.0;
                if (sg.kind == RF_MAXSPIN) a = msrow(sg.sub, (int)e);
                else {
                    VGather f{t};
                    if (sg.wave == 0) elem_terms(R.L, sg, e, f);
                    else if (sg.wave == 1) for (int l = 0; l < 64; l++) wave_terms(R.L, sg, e, l, f);
                    else for (int l = 0; l < 512; l++) wave_terms(R.L, sg, e, l, f, 512);
                    a = f.acc;
                }
                fn(sg.start + e, sg.aux + e, a);
            }
        }
    };
    // s = rhs - y - B2 t + P y_ms on the self rows, r on the explicit ones
    Vec yms(R.nM), ys(R.nS), none(R.nM), zD(R.nD);
    for (int k = 0; k < R.nM; k++) yms.at(k) = y[Lo.rowoff[RF_MAXSPIN][0][0] + k];
    each_self(t, yms, [&](int64_t sl, int64_t row, double dx, double pm) {
        ys.at(sl) = y[row];
        s.at(sl) = rhs[row] - y[row] - dx + pm;
    });
    auto wave = [&](auto fn) { double a = 0.0; for (int l = 0; l < 64; l++) a += fn(l); return a; };
    explicit_rows([&](int o, int e) {
        return -wave([&](int l) { return ms_row_self(R, o, e, l, 1.0, ys, zD, none); }) +
               wave([&](int l) { return ms_row_gram(R, o, e, l, yms); });
    }, [&](int64_t i, int64_t row, double a) { r.at(i) = rhs[row] - a; });
    for (const Segment &sg : W.p)
        for (int64_t e = 0; sg.kind <= XS_SELF && e < sg.count; e++) {
            double a = 0.0;
            if (sg.kind == XS_D2AB) a = self_at_ab(R, ab_entry(R.L, sg.h, e), s);
            else if (sg.kind == XS_D2AA) a = self_at_aa(R, sg.sub, sg.h, e, s);
            else a = wave([&](int l) { return self_at_d1(R, sg.sub, sg.h, e, l, s); });
            g.at(sg.start + e) = a;
        }
    double c = 1.0, d = 1.0, e_ = 0.0, rz = 0.0, pp2 = 0.0;
    p = r;
    for (double a : r.v) rz += a * a;
    for (double a : s.v) pp2 += a * a;
    rz += pp2;
    int it = 0;
    while (it < maxiter) {
        double pap = pp2;
        for (const Segment &sg : W.p)
            for (int64_t e = 0; sg.kind <= XS_SELF && e < sg.count; e++) {
                double a = d * g[sg.start + e];
                if (sg.kind == XS_D2AB)
                    a += atu_d2ab<false, true>(R.L, sg, e, p) + gram_ab(R, ab_entry(R.L, sg.h, e), v, nu);
                else if (sg.kind == XS_D2AA)
                    a += atu_d2aa<false, true>(R.L, sg, e, p) + gram_aa(R, sg.sub, sg.h, e, v);
                else
                    a += wave([&](int l) { return atu_d1_wave<false, true>(R.L, sg, e, l, p) +
                                                  gram_d1(R, sg.sub, sg.h, e, l, v, nu); });
                t.at(sg.start + e) = a;
                pap += a * a;
            }
        struct Ms { const Vec &p; int64_t o; double operator[](int64_t i) const { return p[o + i]; } } pm{p, ms0};
        for (int k = 0; k < R.nM; k++) {
            const int g0 = R.nM / 2, o = k / g0, e = k % g0;
            const double self = wave([&](int l) { return ms_row_self(R, o, e, l, d, s, v, nu); });
            const double gr = wave([&](int l) { return ms_row_gram(R, o, e, l, pm); });
            ams.at(k) = gr - self;
            pap += pm[k] * (gr - 2.0 * self);
        }
        const double al = rz / pap;
        for (int64_t i = 0; i < R.nD; i++) {
            u.at(i) -= al * (v[i] + t[i]);
            wv.at(i) += al * v[i];
        }
        for (int k = 0; k < R.nM; k++) {
            mu.at(k) -= al * (nu[k] + pm[k]);
            om.at(k) += al * nu[k];
        }
        double rr = 0.0;
        explicit_rows([&](int o, int e) { return ams[o * (R.nM / 2) + e]; },
                      [&](int64_t i, int64_t row, double a) {
                          y_[row] += al * p[i];
                          r.at(i) -= al * a;
                          rr += r[i] * r[i];
                      });
        c -= al * d;
        e_ += al * d;
        double rr2 = 0.0, rp = 0.0, pp = 0.0;
        std::vector<double> rs((size_t)R.nS);
        each_self(u, mu, [&](int64_t sl, int64_t, double dx, double pmv) { rs[sl] = c * s[sl] + dx - pmv; });
        each_self(v, nu, [&](int64_t sl, int64_t, double dx, double pmv) {
            const double ps = d * s[sl] + dx - pmv;
            rr2 += rs[sl] * rs[sl];
            rp += rs[sl] * ps;
            pp += ps * ps;
        });
        rr += rr2;
        res[it] = std::sqrt(rr);
        if (res[it] < tol) break;
        const double be = rr / rz;
        for (int64_t i = 0; i < R.nR; i++) p.at(i) = r[i] + be * p[i];
        for (int64_t i = 0; i < R.nD; i++) v.at(i) = u[i] + be * v[i];
        for (int k = 0; k < R.nM; k++) nu.at(k) = mu[k] + be * nu[k];
        d = c + be * d;
        pp2 = rr2 + 2.0 * be * rp + be * be * pp;
        rz = rr;
        it++;
    }
    each_self(wv, om, [&](int64_t sl, int64_t row, double dx, double pmv) { y_[row] += e_ * s[sl] + dx - pmv; });
    return g_viol ? -2 : it;
}

}  // extern "C"
