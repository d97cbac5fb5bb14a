// emu_t2.cc -- the T2 rows by column lists (csrc/t2rows.hpp) on the host, every index
// checked, for the CPU tests: A.x and A^T.y with all other rows by rowterms.hpp.
#include <cstring>
#include <vector>

#include "../../v2rdm_casscf_amd/csrc/devlayout.hpp"
#include "../../v2rdm_casscf_amd/csrc/layout.hpp"
#include "../../v2rdm_casscf_amd/csrc/rowterms.hpp"
#include "../../v2rdm_casscf_amd/csrc/t2rows.hpp"

using namespace v2g;

namespace {

struct Sink {
    const double *x;
    double *val;
    int n;
    int64_t dimx;
    long long *viol;
    void operator()(int c, int64_t col, double coef)
    {
        if (c < 0 || c >= n || col < 0 || col >= dimx) { (*viol)++; return; }
        val[c] += coef * x[col];
    }
};

struct Rows {
    const double *y;
    const std::vector<char> *t2;   // the T2 rows, the only ones to be read
    long long *viol;
    double operator[](int64_t i) const
    {
        if (i < 0 || i >= (int64_t)t2->size() || !(*t2)[i]) { (*viol)++; return 0.0; }
        return y[i];
    }
};

}  // namespace

extern "C" {

// Ax and ATy of the T2 rows alone, into zeroed outputs; returns the number of violations:
// columns or rows out of range, units that do not tile the rows
long long emu_t2(int nirrep, const int *amopi, int na, int nb, int mult, int t1, int sz, const double *x,
                 double *Ax, const double *y, double *ATy, long long dimx, long long ncon)
{
    Options op;
    op.nirrep = nirrep;
    for (int h = 0; h < 8; h++) op.amopi[h] = h < nirrep ? amopi[h] : 0;
    op.nalpha = na;
    op.nbeta = nb;
    op.multiplicity = mult;
    op.t2 = true;
    op.t1 = t1;
    op.sz = sz;
    Layout L(op);
    if (dimx != L.dimx || ncon != L.ncon) return -1;
    const DevLayout D = make_dev_layout(L, {L.sym.data(), L.gab.data(), L.gaa.data(), L.bab.data(),
                                            L.baa.data(), L.baab.data(), L.baba.data(),
                                            L.baaa.data(), L.b00.data()});
    T2Lists t;
    make_t2_lists(L, t);
    const T2Tab tab{t.seg.data(), t.chunk.data(), t.ptr.data(), t.item.data(), t.aab.data(), t.aba.data(),
                    (int)t.seg.size(), t.units};
    long long viol = 0;
    std::vector<char> seen(ncon, 0);
    std::vector<double> val(kT2Chunk);
    for (int64_t u = 0; u < t.units; u++) {
        int row;
        T2Chunk ch;
        const T2Seg &sg = rows::t2_unit(tab, u, row, ch);
        if (row < 0 || row >= sg.dim || ch.n < 1 || ch.n > kT2Chunk) { viol++; continue; }
        const int64_t e0 = rows::t2_first(D, sg, row, ch);
        for (int c = 0; c < ch.n; c++) {
            const int64_t r = sg.row0 + e0 + c, i = sg.x0 + e0 + c;
            if (r < 0 || r >= ncon || i < 0 || i >= dimx || seen[r]++) { viol++; continue; }
            val[c] = -x[i];
            ATy[i] -= y[r];
        }
        for (int lane = 0; lane < 3; lane++) {   // three lanes: the shares tile the lists
            Sink f{x, val.data(), ch.n, dimx, &viol};
            rows::t2_unit_terms(D, tab, sg, row, ch, lane, 3, f, [] {});
        }
        for (int c = 0; c < ch.n; c++) Ax[sg.row0 + e0 + c] = val[c];
    }
    const Rows Y{y, &seen, &viol};
    for (int h = 0; h < L.nirrep; h++) {
        for (int64_t e = 0; e < (int64_t)L.gems_ab[h] * L.gems_ab[h]; e++) {
            const int b = L.bab[L.bab_off[h] + e / L.gems_ab[h]], k = L.bab[L.bab_off[h] + e % L.gems_ab[h]];
            for (int sp = 0; sp < 2; sp++)
                for (int o = 0; o < L.amo; o++)
                    ATy[L.xoff[XB_D2AB][h] + e] += rows::t2_at_ab(D, tab, sp, o, rows::P0(b), rows::P1(b), rows::P0(k), rows::P1(k), Y);
        }
        for (int64_t e = 0; e < (int64_t)L.gems_aa[h] * L.gems_aa[h]; e++) {
            const int b = L.baa[L.baa_off[h] + e / L.gems_aa[h]], k = L.baa[L.baa_off[h] + e % L.gems_aa[h]];
            for (int sp = 0; sp < 2; sp++)   // the aa pairs are stored larger orbital first
                for (int o = 0; o < L.amo; o++)
                    ATy[L.xoff[sp ? XB_D2BB : XB_D2AA][h] + e] += rows::t2_at_aa(D, tab, sp, o, rows::P1(b), rows::P0(b), rows::P1(k), rows::P0(k), Y);
        }
        const int n = op.amopi[h];
        for (int e = 0; e < n * n; e++)
            for (int sp = 0; sp < 2; sp++)
                for (int ij = 0; ij < L.amo * L.amo; ij++)
                    ATy[L.xoff[sp ? XB_D1B : XB_D1A][h] + e] +=
                        rows::t2_at_d1(D, tab, sp, ij / L.amo, ij % L.amo, e / n + L.poff[h], e % n + L.poff[h], Y);
    }
    // the units cover exactly the T2 rows
    for (const Segment &s : L.rowsegs)
        for (int64_t k = 0; k < s.count; k++) {
            const bool t2 = s.kind == RF_T2AAB || s.kind == RF_T2BIG;
            if ((seen[s.start + k] != 0) != t2) viol++;
        }
    return viol;
}

// which rows are T2 rows
void emu_t2_rows(int nirrep, const int *amopi, int na, int nb, int mult, int t1, int sz, char *is)
{
    Options op;
    op.nirrep = nirrep;
    for (int h = 0; h < 8; h++) op.amopi[h] = h < nirrep ? amopi[h] : 0;
    op.nalpha = na;
    op.nbeta = nb;
    op.multiplicity = mult;
    op.t2 = true;
    op.t1 = t1;
    op.sz = sz;
    Layout L(op);
    for (const Segment &s : L.rowsegs)
        std::memset(is + s.start, s.kind == RF_T2AAB || s.kind == RF_T2BIG, (size_t)s.count);
}

}  // extern "C"
