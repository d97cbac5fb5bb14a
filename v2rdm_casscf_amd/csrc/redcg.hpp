// redcg.hpp -- the plain CG in its reduced form (redrows.hpp): host plan,
// buffers and launch wrappers (redcg.hip).
#pragma once
#include <cstdint>
#include <vector>

#include "redrows.hpp"

namespace v2g {

// segment kinds of the reduced kernels beside XS_D1 and RowFam
enum RedKind : int {
    RK_AB = 100,     // the D2ab entries of an irrep's cells, in position order
    RK_DIAG,         // the D2ab entries with p == q or r == s
    RK_AA,           // the cells of an irrep (both like-spin blocks)
    RK_LIST_AB,      // the D2ab entries with p == q or r == s, by their records
    RK_CELLS,        // the cells of an irrep
    RK_ROWS,         // explicit rows not aligned with cells, elementwise
    RK_DVEC, RK_RVEC, RK_MVEC,   // whole vectors, elementwise
    RK_SHARED,       // the cells with a CellRec (Segment::dim of them), one orientation an item
    RK_STEP,         // D entries outside the cells, elementwise
    RK_D1,           // D1 entries one by one (XS_D1 is a RowFam's number)
    RK_MS            // maximal-spin rows, one wavefront each (direction side)
};

// work lists of one problem.  Segment::wave: 0 one thread per item, 1 one
// wavefront, 2 one workgroup, 3 RedLayout::lanes threads; Segment::start: first entry of the compact vector;
// Segment::aux: first row of the full vector
struct RedWork {
    // start and end of a solve, direction, residual, norms
    std::vector<Segment> start, dir, res, norm;
    // the orbitals of the listed D2ab entries and cells (RedKey), in order, and their records
    std::vector<uint32_t> ab_key, cell_key;
    std::vector<AbRec> ab;
    std::vector<CellRec> cell;
    std::vector<uint64_t> bits;             // one a cell, set for those with a CellRec; every
                                            // irrep starts on a word (Segment::aux of RK_CELLS)
    std::vector<int32_t> rowtab;            // RedLayout::rowtab
    std::vector<uint32_t> rank;             // CellRecs before each word's first
};

// (pq|rs) of a listed entry or cell, eight bits an orbital (at most 255, layout.cc)
struct RedKey {
    static V2G_HD uint32_t of(int p, int q, int r, int s) { return (uint32_t)p | (uint32_t)q << 8 | (uint32_t)r << 16 | (uint32_t)s << 24; }
    int p, q, r, s;
    explicit V2G_HD RedKey(uint32_t k) : p(k & 255), q(k >> 8 & 255), r(k >> 16 & 255), s(k >> 24) {}
};

// false: the layout has rows the reduced form does not cover (T1, T2,
// spin-adapted Q2 / G2), or sizes beyond its 32-bit places.  R.rowtab is left to the caller.  dev: the layout's
// device view (tables of either side).  records = false: RedWork::ab and cell stay empty
bool make_red_layout(const Layout &Lt, const DevLayout &dev, RedLayout &R, RedWork &w, bool records = true);

#if defined(__HIPCC__)

// a tile of a work list: a workgroup's share of a segment, with the segment beside
// it (one read instead of a search)
struct RedTile {
    Segment sg;
    int64_t first;      // first item of the tile
};

// one problem of the plan, in device memory.  Offsets place its share of the
// concatenated vectors; [b0, b0 + nb) are the workgroups that work on it
struct RedProb {
    RedLayout R;
    const DevLayout *full;              // the full layout: rows of rhs and y
    int64_t oD, oR, oS, oM;
    const RedTile *tile[4];             // RedWork's lists, cut into tiles
    int ntile[4];
    AbRec *ab;
    CellRec *cell;
    const uint64_t *bits;
    const uint32_t *rank;
    int b0, nb;
    const uint32_t *ab_key, *cell_key;  // where the records come from
    int nab, ncell;
};

// the vectors of a solve (concatenated over the problems); pairs are indexed by the
// iteration parity
struct RedBufs {
    double *g, *t, *w, *u[2], *v[2];    // nD + 1 each (the last one zero)
    double *r, *p[2];                   // nR + 1 each
    double *s;                          // nS
    double *mu[2], *nu[2], *om, *ams;   // nM + 1 each
    double *part;                       // kRedParts per workgroup
    double *scal;                       // kRedScal per problem
};

// per-problem scalars.  A slots (direction pass) and B slots (residual pass) are
// ping-pong pairs indexed by the iteration parity; the rest is read by the host
enum RedSlot : int {
    RS_A = 0,        // + 6 parity: done, r.z, d, p.p as in kRedParts, iterations begun
    RS_B = 12,       // + 2 parity: c, e
    RS_DONE = 18, RS_NRM = 20, RS_ITER = 21, RS_TOL = 25, RS_MAXIT = 26, RS_NRM0 = 29
};
constexpr int kRedScal = 32;
// squares of A^T p; r.r of the explicit rows and the self rows that maximal-spin rows read;
// r.r, r.p and p.p of the other self rows
constexpr int kRedParts = 5;

class RedCG {
public:
    RedCG() = default;
    RedCG(const RedCG &) = delete;
    RedCG &operator=(const RedCG &) = delete;
    ~RedCG();
    // problems in order; dev[q] is problem q's device view with its offsets in the
    // batch, d_dev its copy in device memory.  False: some layout is not covered
    bool build(const std::vector<const Layout *> &L, const std::vector<DevLayout> &dev,
               const DevLayout *d_dev);
    bool ok() const { return d_prob_ != nullptr; }
    int64_t doubles() const;            // scratch of one solve, in doubles
    RedBufs carve(double *base) const;
    // A^T y, the first residual, A^T of its self part; tol / maxiter per problem
    // from tolv (null: tol) and active (null: all)
    void start(const RedBufs &B, const double *rhs, const double *y, double tol, const double *tolv,
               const int *active, int maxiter, hipStream_t st) const;
    // n (even) iterations, then the convergence test of the last one; y's
    // explicit rows are updated as they go
    void iterate(const RedBufs &B, double *y, int n, hipStream_t st) const;
    // y's self rows
    void finish(const RedBufs &B, double *y, const int *active, hipStream_t st) const;

private:
    RedProb *d_prob_ = nullptr;
    int *d_blk_ = nullptr;              // problem of each workgroup
    void *d_work_ = nullptr;            // tiles, lists and tables
    int np_ = 0, nblk_ = 0;
    bool full_ = true;
    int64_t nD_ = 0, nR_ = 0, nS_ = 0, nM_ = 0;
};

#endif  // __HIPCC__

}  // namespace v2g
