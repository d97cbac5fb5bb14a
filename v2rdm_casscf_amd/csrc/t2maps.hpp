// t2maps.hpp -- A.x and A^T.y of the T2 rows by column lists (t2rows.hpp)
#pragma once
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels.hpp"
#include "t2rows.hpp"

namespace v2g {

// a workgroup's share of A^T.y: n rows (i0 ..) of column k of a D2 block (sg), one D1 entry
// (i0), or n entries of a T2 block from i0 on (copied from row sg.aux + i0)
struct T2Tile {
    Segment sg;
    int64_t i0;
    int32_t k, n;
};

class T2Maps {
public:
    // the T2 rows of one layout (L.opt.t2); dlay: its device view
    void build(const Layout &L, const DevLayout *dlay);
    int au_blocks() const { return blocks_; }                  // partial sums of au()
    int atu_blocks() const { return (int)tiles_.n; }           // partial sums of atu()
    // the T2 rows of A.x; rowpart (optional): partial sums of dotv . Ax.  fz: as launch_au,
    // its partial sums from place `part0` on
    void au(const double *x, double *Ax, const double *done, const double *dotv, double *rowpart, CgFuse fz,
            int64_t part0, hipStream_t st) const;
    // A^T.y of the T2 blocks and, with all their other terms, of the D2 and D1 blocks;
    // sqpart (optional): partial sums of their squares
    void atu(const double *y, double *ATy, const double *done, double *sqpart, hipStream_t st) const;

private:
    const DevLayout *dlay_ = nullptr;
    int blocks_ = 0;
    DevBuf<T2Tile> tiles_;
    T2Tab tab_{};
    DevBuf<T2Seg> seg_;
    DevBuf<T2Chunk> chunk_;
    DevBuf<int32_t> ptr_;
    DevBuf<uint32_t> item_;
    DevBuf<int32_t> aab_, aba_;
};

}  // namespace v2g
