// redlayout.cc -- compact offsets and work lists of the reduced CG (redcg.hpp).
#include "redcg.hpp"

namespace v2g {

bool make_red_layout(const Layout &Lt, const DevLayout &dev, RedLayout &R, RedWork &w)
{
    if (!Lt.xsegs_t2.empty()) return false;
    R.L = dev;
    for (int b = 0; b < XB_COUNT; b++)
        for (int h = 0; h < kMaxIrrep; h++) R.L.xoff[b][h] = -1;
    for (int f = 0; f < RF_COUNT; f++)
        for (int s = 0; s < 6; s++)
            for (int h = 0; h < kMaxIrrep; h++) R.L.rowoff[f][s][h] = -1;
    for (int f = 0; f < SF_COUNT; f++)
        for (int h = 0; h < kMaxIrrep; h++) R.soff[f][h] = -1;
    const bool q2 = Lt.q2_plain(), g2 = Lt.g2_plain();
    R.nblk_d = Lt.opt.spin ? (Lt.singlet ? 1 : 4) : 0;
    R.nM = Lt.opt.spin && g2 ? 2 * Lt.gems_ab[0] : 0;

    auto seg = [](std::vector<Segment> &v, int kind, int sub, int h, int dim, int64_t start,
                  int64_t count, int64_t aux, int mode) {
        if (count <= 0) return;
        Segment s{};
        s.kind = kind;
        s.sub = sub;
        s.h = h;
        s.dim = dim;
        s.start = start;
        s.count = count;
        s.aux = aux;
        s.wave = mode;
        v.push_back(s);
    };
    auto sq = [](int64_t n) { return n * n; };

    // D2 / D1 entries
    int64_t o = 0;
    std::vector<Segment> ab, aa, d1;
    for (int h = 0; h < Lt.nirrep; h++) {
        R.L.xoff[XB_D2AB][h] = o;
        seg(ab, XS_D2AB, 0, h, Lt.gems_ab[h], o, sq(Lt.gems_ab[h]), 0, 0);
        o += sq(Lt.gems_ab[h]);
    }
    for (int s = 0; s < 2; s++)
        for (int h = 0; h < Lt.nirrep; h++) {
            R.L.xoff[s ? XB_D2BB : XB_D2AA][h] = o;
            seg(aa, XS_D2AA, s, h, Lt.gems_aa[h], o, sq(Lt.gems_aa[h]), 0, 0);
            o += sq(Lt.gems_aa[h]);
        }
    for (int s = 0; s < 2; s++)
        for (int h = 0; h < Lt.nirrep; h++) {
            const int64_t n = Lt.opt.amopi[h];
            R.L.xoff[s ? XB_D1B : XB_D1A][h] = o;
            seg(d1, XS_D1, s, h, (int)n, o, sq(n), 0, 1);
            o += sq(n);
        }
    R.nD = o;

    // self slots
    o = 0;
    for (int f = 0; f < SF_COUNT; f++) {
        bool on = true;
        if (f == SF_Q2AB || f == SF_Q2AA || f == SF_Q2BB) on = q2;
        else if (f >= SF_G2AB && f <= SF_G2B) on = g2;
        else if (f >= SF_D0 && f <= SF_D3) on = f - SF_D0 < R.nblk_d;
        if (!on) continue;
        for (int h = 0; h < Lt.nirrep; h++) {
            R.soff[f][h] = o;
            o += f < kSfAb ? sq(Lt.gems_ab[h])
                           : f <= SF_Q2BB ? sq(Lt.gems_aa[h]) : sq(Lt.opt.amopi[h]);
        }
    }
    R.nS = o;

    // explicit rows, in the order of the full layout; the long rows lead the
    // residual pass (a workgroup for a trace, a wavefront for a contraction)
    o = 0;
    std::vector<Segment> lng, rest;
    for (const Segment &s : Lt.rowsegs) {
        switch (s.kind) {
        case RF_TRACE: case RF_S2: case RF_CONTR: case RF_SPIN_D1: case RF_SPIN_D2:
        case RF_SPIN_ANTI: case RF_MAXSPIN: break;
        default: continue;
        }
        R.L.rowoff[s.kind][s.sub][s.h] = o;
        const int mode = s.kind == RF_TRACE || s.kind == RF_S2 ? 2 : s.kind == RF_CONTR ? 1 : 0;
        seg(mode ? lng : rest, s.kind, s.sub, s.h, s.dim, o, s.count,
            dev.rowoff[s.kind][s.sub][s.h], mode);
        o += s.count;
    }
    R.nR = o;

    // passes
    auto cat = [](std::vector<Segment> &a, const std::vector<Segment> &b) { a.insert(a.end(), b.begin(), b.end()); };
    cat(w.p, d1);
    if (R.nM)
        for (int k = 0; k < 2; k++)
            seg(w.p, RK_MS, k, 0, Lt.gems_ab[0], R.L.rowoff[RF_MAXSPIN][k][0], Lt.gems_ab[0], 0, 1);
    cat(w.p, ab);
    cat(w.p, aa);
    seg(w.p, RK_ROWS, 0, 0, 0, 0, R.nR, 0, 0);
    seg(w.p, RK_MVEC, 0, 0, 0, 0, R.nM, 0, 0);
    cat(w.r, lng);
    cat(w.r, rest);
    seg(w.r, RK_DVEC, 0, 0, 0, 0, R.nD, 0, 0);
    seg(w.r, RK_MVEC, 0, 0, 0, 0, R.nM, 0, 0);
    cat(w.n, ab);
    cat(w.n, aa);
    for (Segment s : d1) {
        s.wave = 0;
        w.n.push_back(s);
    }
    return true;
}

}  // namespace v2g
