// t2lists.cc -- the column lists of the T2 rows (t2rows.hpp).
#include "t2rows.hpp"

#include <algorithm>
#include <stdexcept>

namespace v2g {

void make_t2_lists(const Layout &L, T2Lists &out)
{
    out = T2Lists{};
    const int amo = L.amo;
    if (amo > 255) throw std::invalid_argument("at most 255 active orbitals");
    int first[kMaxIrrep] = {}, naab[kMaxIrrep] = {}, nall[kMaxIrrep] = {};
    std::vector<std::vector<uint32_t>> by(3 * (size_t)amo);
    for (int h = 0; h < L.nirrep; h++) {
        first[h] = (int)out.chunk.size();
        for (int aba = 0; aba < 2; aba++) {
            const int cols = aba ? L.trip_aba[h] : L.trip_aab[h];
            const int *trip = aba ? L.baba.data() + L.baba_off[h] : L.baab.data() + L.baab_off[h];
            const int nc = (cols + kT2Chunk - 1) / kT2Chunk, size = nc ? (cols + nc - 1) / nc : 0;
            for (int c0 = 0; c0 < cols; c0 += size) {
                const int n = std::min(size, cols - c0);
                for (auto &v : by) v.clear();
                for (int c = 0; c < n; c++) {
                    const uint32_t p = (uint32_t)trip[c0 + c];
                    const uint32_t l = p & 255, m = p >> 8 & 255, o = p >> 16 & 255;
                    by[l].push_back((uint32_t)c | m << 10 | o << 18);
                    by[amo + m].push_back((uint32_t)c | l << 10 | o << 18);
                    by[2 * amo + o].push_back((uint32_t)c | l << 10 | m << 18);
                }
                out.chunk.push_back({c0, n, aba, (int32_t)out.ptr.size()});
                for (const auto &v : by) {
                    out.ptr.push_back((int32_t)out.item.size());
                    out.item.insert(out.item.end(), v.begin(), v.end());
                }
                out.ptr.push_back((int32_t)out.item.size());
            }
            if (!aba) naab[h] = (int)out.chunk.size() - first[h];
        }
        nall[h] = (int)out.chunk.size() - first[h];
    }
    out.aab.assign((size_t)amo * amo * amo, 0);
    out.aba.assign((size_t)amo * amo * amo, 0);
    auto place = [&](int p) { return ((size_t)(p & 255) * amo + (p >> 8 & 255)) * amo + (p >> 16 & 255); };
    for (int h = 0; h < L.nirrep; h++) {
        for (int c = 0; c < L.trip_aab[h]; c++) out.aab[place(L.baab[L.baab_off[h] + c])] = c;
        for (int c = 0; c < L.trip_aba[h]; c++) out.aba[place(L.baba[L.baba_off[h] + c])] = c;
    }
    for (const Segment &s : L.xsegs_t2) {
        if (s.kind != RF_T2AAB && s.kind != RF_T2BIG) continue;
        const int nc = s.kind == RF_T2AAB ? naab[s.h] : nall[s.h];
        out.seg.push_back({s.kind, s.sub, s.h, s.dim, first[s.h], nc, out.units, s.start, s.aux});
        out.units += (int64_t)s.dim * nc;
    }
}

}  // namespace v2g
