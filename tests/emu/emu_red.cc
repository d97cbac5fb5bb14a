// emu_red.cc -- host execution of the reduced plain CG (csrc/redrows.hpp) with
// the device row code, for the CPU test suite: every vector read is checked
// against its buffer.
#include <cmath>
#include <cstdint>
#include <map>
#include <type_traits>
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
    R.rowtab = W.rowtab.data();
    if (ncon != L.ncon) return -3;
    g_viol = 0;
    const View rhs{rhs_, ncon}, y{y_, ncon};
    // D, R and M vectors end with a zero (the place of no entry)
    Vec t(R.nD + 1), g(R.nD + 1), u(R.nD + 1), v(R.nD + 1), wv(R.nD + 1), s(R.nS), r(R.nR + 1),
        p(R.nR + 1), mu(R.nM + 1), nu(R.nM + 1), om(R.nM), ams(R.nM);
    const int64_t ms0 = R.nM ? R.L.rowoff[RF_MAXSPIN][0][0] : 0;
    auto wave = [&](auto fn) { double a = 0.0; for (int l = 0; l < 64; l++) a += fn(l); return a; };
    auto group = [&](auto fn) { double a = 0.0; for (int l = 0; l < R.lanes; l++) a += fn(l); return a; };
    // every D2 / D1 entry once: ab(entry), aa(spin, cell, irrep, place), d1(segment, item)
    auto each_entry = [&](auto ab, auto aa, auto d1) {
        std::vector<char> seen((size_t)R.nD, 0);
        auto mark = [&](int64_t i) { if (i < 0 || i >= R.nD || seen[i]++) g_viol++; };
        for (const Segment &sg : W.start)
            for (int64_t i = 0; i < sg.count; i++) {
                AbEntry a;
                if (sg.kind == RK_AB || sg.kind == RK_DIAG) {
                    if (sg.kind == RK_AB) a = cell_ab(R, sg.h, i);
                    else if (!diag_ab(R, i, a)) continue;
                    if (a.pos != ab_pos(R, a.p, a.q, a.r, a.s)) g_viol++;
                    mark(a.pos);
                    ab(a);
                } else if (sg.kind == RK_AA) {
                    a = cell_entry(R, sg.h, i);
                    if (sg.start + i != aa_pos(R, a.p, a.q, a.r, a.s)) g_viol++;
                    for (int sp = 0; sp < 2; sp++) { mark(R.nAB + sp * R.nAA + sg.start + i); aa(sp, a, sg.h, sg.start + i); }
                } else if (sg.kind == XS_D1) {
                    mark(sg.start + i);
                    d1(sg, i);
                }
            }
        long long n = 0, want = 0;
        for (char c : seen) n += c;
        for (int h = 0; h < L.nirrep; h++)
            want += (int64_t)L.gems_ab[h] * L.gems_ab[h] + 2LL * L.gems_aa[h] * L.gems_aa[h] + 2LL * op.amopi[h] * op.amopi[h];
        if (n != want) g_viol++;
    };
    // every self slot once: fn(slot, full row, D part of x, P part of m)
    auto each_self = [&](const auto &x, const auto &m, auto fn) {
        std::vector<char> seen((size_t)ncon, 0);
        auto visit = [&](int64_t slot, int64_t row, double dx, double pm) {
            if (slot < 0 || slot >= R.nS || row < 0 || row >= ncon || seen[row]++) { g_viol++; return; }
            fn(slot, row, dx, pm);
        };
        each_entry([&](const AbEntry &a) {
            const SelfAb<std::decay_t<decltype(x)>> o(R, a, x);
            auto one = [&](int f, double dx, double pm) { visit(R.soff[f] + a.pos, self_row_ab(R, f, a), dx, pm); };
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
                const D200Ab<std::decay_t<decltype(x)>> d(R, a, x);
                for (int k = 0; k < R.nblk_d; k++) one(SF_D0 + k, d.row(R, a, k), 0.0);
            }
        }, [&](int sp, const AbEntry &a, int h, int64_t k) {
            if (R.L.q2) visit(R.soff[SF_Q2AA + sp] + k, Lo.rowoff[RF_Q2AA][sp][h] + k - R.aa0[h], self_row_aa(R, sp, a, x), 0.0);
        }, [&](const Segment &sg, int64_t i) {
            visit(R.soff[sg.sub ? SF_Q1B : SF_Q1A] + sg.start - R.L.xoff[sg.sub ? XB_D1B : XB_D1A][0] + i,
                  self_row_d1(Lo, sg.sub, sg.h, i), x[sg.start + i], 0.0);
        });
        long long n = 0;
        for (char c : seen) n += c;
        if (n + R.nR != ncon) g_viol++;
    };
    // every explicit row once, on the D vector t: fn(compact row, full row, value)
    auto explicit_rows = [&](auto msrow, auto fn) {
        std::vector<char> seen((size_t)R.nR, 0);
        auto visit = [&](int64_t k, int64_t row, double a) {
            if (k < 0 || k >= R.nR || seen[k]++ || row < 0 || row >= ncon) { g_viol++; return; }
            fn(k, row, a);
        };
        if (R.cells)
            for (int h = 0; h < L.nirrep; h++) {
                const int64_t cc = (int64_t)L.gems_aa[h] * L.gems_aa[h];
                for (int64_t i = 0; i < cc; i++) {
                    double at[3];
                    cell_rows(load_cell(R, R.ab0[h] + i, cc, R.aa0[h] + i, t), at);
                    for (int j = 0; j < 3; j++)
                        visit(j * R.nAA + R.aa0[h] + i,
                              (j ? Lo.rowoff[RF_SPIN_ANTI][j - 1][h] : Lo.rowoff[RF_SPIN_D2][0][h]) + i, at[j]);
                }
            }
        for (const Segment &sg : W.res)
            for (int64_t e = 0; sg.kind < RK_AB && e < sg.count; e++) {
                double a = 0.0;
                if (sg.kind == RF_MAXSPIN) a = msrow(sg.sub, (int)e);
                else if (sg.kind == RF_SPIN_D1) a = t[R.L.xoff[XB_D1A][sg.h] + e] - t[R.L.xoff[XB_D1B][sg.h] + e];
                else {
                    const int lanes = sg.wave == 3 ? R.lanes : 256;
                    for (int l = 0; l < lanes; l++) a += long_row(R, sg, e, l, lanes, t);
                }
                visit(sg.start + e, sg.aux + e, a);
            }
        for (char c : seen) if (c != 1) g_viol++;
    };
    each_entry([&](const AbEntry &a) { t.at(a.pos) = full_at_ab(R, Lo, a, y); },
               [&](int sp, const AbEntry &a, int, int64_t k) { t.at(R.nAB + sp * R.nAA + k) = full_at_aa(Lo, sp, a, y); },
               [&](const Segment &sg, int64_t i) { t.at(sg.start + i) = wave([&](int l) { return atu_d1_wave(Lo, sg, i, l, y); }); });
    // s = rhs - y - B2 t + P y_ms on the self rows, r on the explicit ones
    Vec yms(R.nM), ys(R.nS), none(R.nM), zD(R.nD + 1);
    for (int k = 0; k < R.nM; k++) yms.at(k) = y[Lo.rowoff[RF_MAXSPIN][0][0] + k];
    each_self(t, yms, [&](int64_t sl, int64_t row, double dx, double pm) {
        ys.at(sl) = y[row];
        s.at(sl) = rhs[row] - y[row] - dx + pm;
    });
    explicit_rows([&](int o, int e) {
        return -group([&](int l) { return ms_row_self(R, o, e, l, 1.0, ys, zD, none); }) +
               group([&](int l) { return ms_row_gram(R, o, e, l, yms); });
    }, [&](int64_t i, int64_t row, double a) { r.at(i) = rhs[row] - a; });
    each_entry([&](const AbEntry &a) { g.at(a.pos) = self_at_ab(R, a, s); },
               [&](int sp, const AbEntry &a, int h, int64_t k) { g.at(R.nAB + sp * R.nAA + k) = self_at_aa(R, sp, h, a, s); },
               [&](const Segment &sg, int64_t i) { g.at(sg.start + i) = wave([&](int l) { return self_at_d1(R, sg.sub, sg.h, i, l, s); }); });
    double c = 1.0, d = 1.0, e_ = 0.0, rz = 0.0, pp2 = 0.0;
    p = r;
    for (double a : r.v) rz += a * a;
    for (double a : s.v) pp2 += a * a;
    rz += pp2;
    int it = 0;
    while (it < maxiter) {
        double pap = pp2;
        auto keep = [&](int64_t k, double a) {
            t.at(k) = d * g[k] + a;
            pap += t[k] * t[k];
        };
        for (const Segment &sg : W.dir)
            for (int64_t i = 0; i < sg.count; i++) {
                if (sg.kind == RK_CELLS) {
                    const AbEntry a = cell_entry(R, sg.h, i);
                    const int64_t k = R.aa0[sg.h] + i, word = sg.aux + i / 64;
                    const uint64_t m = (uint64_t)1 << (i % 64);
                    const bool shares = W.bits.at((size_t)word) & m;
                    if (shares != (a.p == a.r || a.p == a.s || a.q == a.r || a.q == a.s)) g_viol++;
                    double pr[3] = {0.0, 0.0, 0.0};
                    for (int j = 0; R.cells && j < 3; j++) pr[j] = p[j * R.nAA + k];
                    Cell tc = cell_at(R.L.q2, R.L.g2, R.nblk_d, R.cells, d, load_cell(R, a.pos, sg.count, k, g),
                                      load_cell(R, a.pos, sg.count, k, v), pr);
                    if (shares) {
                        const CellRec &rec = W.cell.at(W.rank.at((size_t)word) + __builtin_popcountll(W.bits[word] & (m - 1)));
                        if (rec.k != k || rec.pos != a.pos || rec.row != i || rec.flags >> 8 != sg.h) g_viol++;
                        shared_at(R, rec, v, nu, p, tc);
                    }
                    for (int o = 0; o < 4; o++) { t.at(a.pos + o * sg.count) = tc.ab[o]; pap += tc.ab[o] * tc.ab[o]; }
                    t.at(R.nAB + k) = tc.aa;
                    t.at(R.nAB + R.nAA + k) = tc.bb;
                    pap += tc.aa * tc.aa + tc.bb * tc.bb;
                } else if (sg.kind == RK_LIST_AB) {
                    const AbRec a = W.ab.at((size_t)i);
                    keep(a.pos, rec_expl_ab(R, a, p) + AbVals(R, a, v).gram(R, a) + (nu[a.m0] + nu[a.m1]));
                } else if (sg.kind == XS_D1) {
                    keep(sg.start + i, group([&](int l) { return atu_d1_wave<false, true>(R.L, sg, i, l, p) +
                                                                gram_d1(R, sg.sub, sg.h, i, l, v, nu); }));
                }
            }
        struct Ms { const Vec &p; int64_t o; double operator[](int64_t i) const { return p[o + i]; } } pm{p, ms0};
        for (int k = 0; k < R.nM; k++) {
            const int g0 = R.nM / 2, o = k / g0, e = k % g0;
            const double self = group([&](int l) { return ms_row_self(R, o, e, l, d, s, v, nu); });
            const double gr = group([&](int l) { return ms_row_gram(R, o, e, l, pm); });
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
        std::map<int64_t, std::vector<double>> by_pos, by_cell;
        std::vector<double> rs((size_t)R.nS);
        // the records of the listed entries give the rows that the general code gives
        for (const AbRec &rec : W.ab) {
            const AbVals o(R, rec, u);
            by_pos[rec.pos] = {o.q2(), o.g1(), o.g2() - (mu[rec.m0] + mu[rec.m1]), o.x0, o.x0, o.ga(rec), o.gb(rec)};
            for (int b = 0; b < R.nblk_d; b++) by_pos[rec.pos].push_back(o.d200(R, rec, b));
        }
        for (const CellRec &rec : W.cell) {
            const int64_t ga = R.L.gems_aa[rec.flags >> 8], cc = ga * ga;
            const Cell x = load_cell(R, rec.pos, cc, rec.k, u);
            by_cell[rec.k] = {x.aa + shared_q2(R, rec, 0, u), x.bb + shared_q2(R, rec, 1, u)};
            for (int o = 0; o < 4; o++) {
                const SharedAt q(R, rec, o, u, mu);
                const double s2 = o == 1 || o == 2 ? 1.0 : -1.0, a0 = x.ab[o];
                by_pos[rec.pos + o * cc] = {a0 + q.q2, q.g1 - a0, q.g2 - a0, a0, a0, s2 * x.aa + q.g1, s2 * x.bb + q.gb};
                for (int b = 0; b < R.nblk_d; b++) {
                    double cf[4];
                    d200_coef(b, R.L.singlet, false, false, cf);
                    by_pos[rec.pos + o * cc].push_back(cf[0] * x.ab[o] + cf[1] * x.ab[o ^ 1] + cf[2] * x.ab[o ^ 2] + cf[3] * x.ab[o ^ 3]);
                }
            }
        }
        each_self(u, mu, [&](int64_t sl, int64_t, double dx, double pmv) {
            for (int f = 0; f < kSfAb; f++) {
                if (R.soff[f] < 0 || sl < R.soff[f] || sl >= R.soff[f] + R.nAB) continue;
                auto it2 = by_pos.find(sl - R.soff[f]);
                if (it2 != by_pos.end() && std::fabs(it2->second[f] - (dx - pmv)) > 1e-12 * (1.0 + std::fabs(dx))) g_viol++;
            }
            for (int sp = 0; sp < 2 && R.L.q2; sp++) {
                auto it2 = by_cell.find(sl - R.soff[SF_Q2AA + sp]);
                if (sl >= R.soff[SF_Q2AA + sp] && sl < R.soff[SF_Q2AA + sp] + R.nAA && it2 != by_cell.end() &&
                    std::fabs(it2->second[sp] - dx) > 1e-12 * (1.0 + std::fabs(dx))) g_viol++;
            }
        });
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
