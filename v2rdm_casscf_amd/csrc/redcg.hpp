// redcg.hpp -- the plain CG in its reduced form (redrows.hpp): host plan,
// buffers and launch wrappers (redcg.hip).
#pragma once
#include <cstdint>
#include <vector>

#include "redrows.hpp"

namespace v2g {

// segment kinds of the reduced kernels beside XSegKind / RowFam
enum RedKind : int {
    RK_ROWS = 100,   // all explicit rows, elementwise (search direction)
    RK_DVEC,         // all D2 / D1 entries, elementwise
    RK_MVEC,         // the maximal-spin coefficients, elementwise
    RK_MS            // maximal-spin rows, one wavefront each (direction side)
};

// work lists of one problem.  Segment::wave: 0 one thread per item, 1 one
// wavefront, 2 one workgroup; Segment::start: first entry of the compact vector;
// Segment::aux: first row of the full vector (explicit rows)
struct RedWork {
    std::vector<Segment> p, r, n;   // direction, residual and norm passes
};

// false: the layout has rows the reduced form does not cover (T1, T2,
// spin-adapted Q2 / G2).  dev: the layout's device view (tables of either side)
bool make_red_layout(const Layout &Lt, const DevLayout &dev, RedLayout &R, RedWork &w);

#if defined(__HIPCC__)

// one problem of the plan, in device memory.  Offsets place its share of the
// concatenated vectors; [b0, b0 + nb) are the workgroups that work on it
struct RedProb {
    RedLayout R;
    const DevLayout *full;              // the full layout: rows of rhs and y
    int64_t oD, oR, oS, oM;
    const Segment *seg[3];              // direction, residual, norm pass
    const int64_t *tile0[3];            // tile prefix of each list (nseg + 1 entries)
    int nseg[3];
    int b0, nb;
};

// the vectors of a solve (concatenated over the problems)
struct RedBufs {
    double *g, *u, *w, *v[2], *t;       // nD each
    double *r, *p[2];                   // nR each
    double *s;                          // nS
    double *mu, *nu[2], *om, *ams;      // nM each
    double *part;                       // kRedParts per workgroup
    double *scal;                       // kRedScal per problem
};

// per-problem scalars.  A slots (direction pass) and B slots (residual pass) are
// ping-pong pairs indexed by the iteration parity; the rest is read by the host
enum RedSlot : int {
    RS_A = 0,        // + 6 parity: done, r.z, d, ||p_self||^2, iterations begun
    RS_B = 12,       // + 3 parity: c, e, alpha
    RS_DONE = 18, RS_NRM = 20, RS_ITER = 21, RS_TOL = 25, RS_MAXIT = 26, RS_NRM0 = 29
};
constexpr int kRedScal = 32;
constexpr int kRedParts = 5;            // ||t||^2, explicit r.r, self r.r, r.p, p.p

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
    void *d_work_ = nullptr;            // segments and tile prefixes
    int np_ = 0, nblk_ = 0;
    int64_t nD_ = 0, nR_ = 0, nS_ = 0, nM_ = 0;
};

#endif  // __HIPCC__

}  // namespace v2g
