// redlayout.cc -- compact offsets and work lists of the reduced CG (redcg.hpp).
#include "redcg.hpp"

namespace v2g {

bool make_red_layout(const Layout &Lt, const DevLayout &dev, RedLayout &R, RedWork &w, bool records)
{
    if (!Lt.xsegs_t2.empty() || Lt.dimx >= ((int64_t)1 << 30)) return false;
    R.L = dev;
    for (int b = 0; b < XB_COUNT; b++)
        for (int h = 0; h < kMaxIrrep; h++) R.L.xoff[b][h] = -1;
    for (int f = 0; f < RF_COUNT; f++)
        for (int s = 0; s < 6; s++)
            for (int h = 0; h < kMaxIrrep; h++) R.L.rowoff[f][s][h] = -1;
    const bool q2 = Lt.q2_plain(), g2 = Lt.g2_plain();
    R.nblk_d = Lt.opt.spin ? (Lt.singlet ? 1 : 4) : 0;
    R.nM = Lt.opt.spin && g2 ? 2 * Lt.gems_ab[0] : 0;
    R.lanes = Lt.amo <= 16 ? 16 : Lt.amo <= 32 ? 32 : 64;
    R.cells = Lt.opt.spin && Lt.singlet ? 1 : 0;

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
    int64_t o = 0, k = 0;
    for (int h = 0; h < kMaxIrrep; h++) {
        const int64_t ga = h < Lt.nirrep ? Lt.gems_aa[h] : 0;
        R.ab0[h] = o;
        R.aa0[h] = k;
        o += 4 * sq(ga);
        k += sq(ga);
    }
    const int64_t ndiag = (int64_t)Lt.amo * Lt.gems_ab[0];
    R.dA = o;
    R.dB = o + ndiag;
    R.nAB = o + 2 * ndiag;
    R.nAA = k;
    o = R.nAB + 2 * R.nAA;
    std::vector<Segment> d1;
    for (int s = 0; s < 2; s++)
        for (int h = 0; h < Lt.nirrep; h++) {
            const int64_t n = Lt.opt.amopi[h];
            R.L.xoff[s ? XB_D1B : XB_D1A][h] = o;
            seg(d1, XS_D1, s, h, (int)n, o, sq(n), 0, 1);
            o += sq(n);
        }
    R.nD = o;
    const int64_t nd1 = R.nD1 = (R.nD - R.nAB - 2 * R.nAA) / 2;

    // self slots
    o = 0;
    for (int f = 0; f < SF_COUNT; f++) {
        bool on = true;
        if (f == SF_Q2AB || f == SF_Q2AA || f == SF_Q2BB) on = q2;
        else if (f >= SF_G2AB && f <= SF_G2B) on = g2;
        else if (f >= SF_D0 && f <= SF_D3) on = f - SF_D0 < R.nblk_d;
        R.soff[f] = on ? o : -1;
        if (on) o += f < kSfAb ? R.nAB : f <= SF_Q2BB ? R.nAA : nd1;
    }
    R.nS = o;

    // explicit rows: those aligned with cells, then the others in the order of the
    // full layout; a workgroup for a trace, a wavefront for a contraction
    o = R.cells ? 3 * R.nAA : 0;
    const int64_t rest0 = o;
    std::vector<Segment> lng, rest;
    for (const Segment &s : Lt.rowsegs) {
        switch (s.kind) {
        case RF_TRACE: case RF_S2: case RF_CONTR: case RF_SPIN_D1: case RF_MAXSPIN: break;
        default: continue;
        }
        R.L.rowoff[s.kind][s.sub][s.h] = o;
        const int mode = s.kind == RF_TRACE || s.kind == RF_S2 ? 2 : s.kind == RF_CONTR ? 1 : 0;
        seg(mode ? lng : rest, s.kind, s.sub, s.h, s.dim, o, s.count,
            dev.rowoff[s.kind][s.sub][s.h], mode);
        o += s.count;
    }
    R.nR = o;
    // contraction rows are looked up by their D1 entry's place: the first irrep's offset
    // is their base also when it has no orbitals
    for (int sub = 0; sub < 6; sub++)
        for (int h = 1; h < Lt.nirrep; h++)
            if (R.L.rowoff[RF_CONTR][sub][0] < 0 && R.L.rowoff[RF_CONTR][sub][h] >= 0)
                R.L.rowoff[RF_CONTR][sub][0] =
                    R.L.rowoff[RF_CONTR][sub][h] - (R.L.xoff[XB_D1A][h] - R.L.xoff[XB_D1A][0]);

    // the listed cells (pairs that share an orbital) and the D2ab entries outside cells
    auto first = [](int pr) { return pr & 0xffff; };
    auto second = [](int pr) { return pr >> 16; };
    std::vector<Segment> bulk;
    RedLayout H = R;   // with the tables of this side
    H.L.sym = Lt.sym.data();
    H.L.gab = Lt.gab.data();
    H.L.gaa = Lt.gaa.data();
    for (int h = 0; h < Lt.nirrep; h++) {
        const int *b = Lt.baa.data() + Lt.baa_off[h];
        const size_t word = w.bits.size();
        seg(bulk, RK_CELLS, 0, h, Lt.gems_aa[h], 0, sq(Lt.gems_aa[h]), (int64_t)word, 0);
        w.bits.resize(word + (size_t)((sq(Lt.gems_aa[h]) + 63) / 64), 0);
        // the pairs of each orbital, ascending: the cells of a pair that share one are the
        // union of two lists (a look at all 0.77 million cells of H50 took half of the plan)
        std::vector<std::vector<int>> with(Lt.amo);
        for (int K = 0; K < Lt.gems_aa[h]; K++) {
            with[first(b[K])].push_back(K);
            with[second(b[K])].push_back(K);
        }
        size_t listed = w.cell_key.size();
        for (int I = 0; I < Lt.gems_aa[h]; I++) listed += with[first(b[I])].size() + with[second(b[I])].size() - 1;
        w.cell_key.reserve(listed);
        if (records) w.cell.reserve(listed);
        for (int I = 0; I < Lt.gems_aa[h]; I++) {
            const int p = first(b[I]), q = second(b[I]);
            const auto &u = with[p], &v = with[q];
            for (size_t i = 0, j = 0; i < u.size() || j < v.size();) {
                const int K = j == v.size() || (i < u.size() && u[i] < v[j]) ? u[i] : v[j];
                i += i < u.size() && u[i] == K;
                j += j < v.size() && v[j] == K;
                const int64_t c = (int64_t)I * Lt.gems_aa[h] + K;
                w.bits[word + c / 64] |= (uint64_t)1 << (c % 64);
                w.cell_key.push_back(RedKey::of(p, q, first(b[K]), second(b[K])));
                if (records) w.cell.push_back(rows::make_cell_rec(H, p, q, first(b[K]), second(b[K])));
            }
        }
    }
    const int *b0 = Lt.bab.data() + Lt.bab_off[0];
    w.ab_key.reserve((size_t)(2 * ndiag));
    for (int d = 0; d < Lt.amo; d++)
        for (int n = 0; n < Lt.gems_ab[0]; n++) {
            const int p = first(b0[n]), q = second(b0[n]);
            w.ab_key.push_back(RedKey::of(d, d, p, q));
            if (p != q) w.ab_key.push_back(RedKey::of(p, q, d, d));
        }
    if (records)
        for (const uint32_t key : w.ab_key) {
            const RedKey k(key);
            w.ab.push_back(rows::make_ab_rec(H, k.p, k.q, k.r, k.s));
        }
    const int64_t nout = (int64_t)w.ab_key.size();
    // listed cells before each word's first
    w.rank.resize(w.bits.size());
    for (size_t i = 0, n = 0; i < w.bits.size(); i++) {
        w.rank[i] = (uint32_t)n;
        n += (size_t)__builtin_popcountll(w.bits[i]);
    }

    // the places of the full layout's rows
    const int amo = Lt.amo;
    w.rowtab.assign((size_t)RT_COUNT * amo * amo, 0);
    for (int x = 0; x < amo; x++)
        for (int y = 0; y < amo; y++) {
            const int h = Lt.sym[x] ^ Lt.sym[y];
            const int64_t n = Lt.gab[x * amo + y], g = Lt.gems_ab[h];
            auto put = [&](int tab, int64_t row, int64_t len, int64_t i) {
                if (row < 0) return true;
                const int64_t v = row + i * len;
                w.rowtab[((size_t)tab * amo + x) * amo + y] = (int32_t)v;
                return v <= INT32_MAX - 2 * g;
            };
            const auto &ro = dev.rowoff;
            if (!put(RT_AB, 0, 1, n) || !put(RT_GG, 0, 1, g + n) || !put(RT_Q2, ro[RF_Q2AB][0][h], g, n) ||
                !put(RT_G2AB, ro[RF_G2AB][0][h], g, n) || !put(RT_G2BA, ro[RF_G2AB][1][h], g, n) ||
                !put(RT_GA, ro[RF_G2AA][0][h], 2 * g, n) || !put(RT_GB, ro[RF_G2AA][0][h], 2 * g, g + n) ||
                !put(RT_D0, ro[Lt.singlet ? RF_SPIN_D200 : RF_SPIN_D200_4][0][h], Lt.singlet ? g : 2 * g, n) ||
                !put(RT_D1, ro[RF_SPIN_D200_4][0][h], 2 * g, g + n))
                return false;
        }

    // passes: the long rows first, so that no workgroup is left with one at the end
    auto cat = [](std::vector<Segment> &a, const std::vector<Segment> &b) { a.insert(a.end(), b.begin(), b.end()); };
    std::vector<Segment> ms;
    if (R.nM)
        for (int m = 0; m < 2; m++)
            seg(ms, RK_MS, m, 0, Lt.gems_ab[0], R.L.rowoff[RF_MAXSPIN][m][0], Lt.gems_ab[0],
                dev.rowoff[RF_MAXSPIN][m][0], 1);
    cat(w.start, d1);
    cat(w.start, ms);
    for (int h = 0; h < Lt.nirrep; h++)
        seg(w.start, RK_AB, 0, h, Lt.gems_aa[h], R.ab0[h], 4 * sq(Lt.gems_aa[h]), 0, 0);
    seg(w.start, RK_DIAG, 0, 0, 0, R.dA, 2 * ndiag, 0, 0);
    for (int h = 0; h < Lt.nirrep; h++)
        seg(w.start, RK_AA, 0, h, Lt.gems_aa[h], R.aa0[h], sq(Lt.gems_aa[h]), 0, 0);
    seg(w.start, RK_DVEC, 0, 0, 0, 0, R.nD, 0, 0);
    seg(w.start, RK_RVEC, 0, 0, 0, 0, R.nR, 0, 0);
    seg(w.start, RK_MVEC, 0, 0, 0, 0, R.nM, 0, 0);
    // rows summed over the orbitals take a full wavefront only where the orbitals fill it
    auto grouped = [](std::vector<Segment> v) {
        for (Segment &x : v)
            if (x.wave == 1) x.wave = 3;
        return v;
    };
    cat(w.dir, grouped(d1));
    cat(w.dir, grouped(ms));
    seg(w.dir, RK_LIST_AB, 0, 0, 0, 0, nout, 0, 0);
    cat(w.dir, bulk);
    seg(w.dir, RK_ROWS, 0, 0, 0, rest0, R.nR - rest0, 0, 0);
    seg(w.dir, RK_MVEC, 0, 0, 0, 0, R.nM, 0, 0);
    cat(w.res, grouped(lng));
    cat(w.res, rest);
    seg(w.res, RK_STEP, 0, 0, 0, R.dA, 2 * ndiag, 0, 0);
    seg(w.res, RK_STEP, 0, 0, 0, R.nAB + 2 * R.nAA, 2 * nd1, 0, 0);
    cat(w.res, bulk);
    seg(w.res, RK_MVEC, 0, 0, 0, 0, R.nM, 0, 0);
    for (Segment s : d1) {
        s.kind = RK_D1;
        s.wave = 0;
        w.norm.push_back(s);
    }
    seg(w.norm, RK_LIST_AB, 0, 0, 0, 0, nout, 0, 0);
    const int64_t ncell = (int64_t)w.cell_key.size();
    seg(w.norm, RK_SHARED, 0, 0, (int)ncell, 0, 4 * ncell, 0, 0);
    cat(w.norm, bulk);
    return true;
}

}  // namespace v2g
