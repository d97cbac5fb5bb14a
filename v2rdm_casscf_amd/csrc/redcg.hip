// redcg.hip -- the plain CG on A A^T y = rhs in its reduced form (redrows.hpp).
//
// The recurrence, the stopping rule and the iteration count are CGSolver::solve's
// (cg_solver.cc:125-177).  On the self rows (26.5 of 28.8 million at (50e,50o))
// the residual, the direction and the correction of y are
//     r = c s + B2 u - P mu,   p = d s + B2 v - P nu,   y - y0 = e s + B2 w - P om,
// so an iteration updates three numbers and vectors of D2 / D1 length (4.6 million)
// instead of streaming r, p, A^T p and y.  What still needs the self rows is the
// residual norm: it is summed row by row from c s + B2 u - P mu, never expanded
// into products of its parts, whose difference would lose the digits of a small
// residual.  Three launches make an iteration:
//   direction   beta from the last norms; v, nu, p; ||A^T p||^2
//   residual    alpha; u, w, mu, om; explicit rows of r and y
//   norms       r.r, r.p and p.p of the self rows, one read of s
// ||p_self||^2 of the next direction follows from the three norms (p' = r + beta p) on the
// rows whose own entry of A^T p is +-p alone.  The G2ba rows that maximal-spin rows read have
// p_self - P p_ms there, squared entry by entry in the direction pass: on a direction that A^T
// maps to zero the two cancel, and the squares written out would leave eps ||p||^2 of either
// sign where the recurrence has (eps ||p||)^2 (a solve that goes on past its last digit then
// took steps of any size, to NaN within some 40 iterations).
//
// What bounds it: at (50e,50o) memory traffic.  By the HBM counters the three passes move
// 334, 377 and 470 MB in 86, 83 and 82 us (3.9, 4.5 and 5.7 TB/s; a large copy has 4.5): 1.18
// GB an iteration where its vectors are 0.80, lines of listed cells being fetched twice.
// 255 us an iteration against 590 us with the entries in block order (index chains and a
// divergent branch for every D1 term) and 796 us for the general form; 58 against 74 us at
// (24e,24o) without symmetry; 23 us at (10e,8o), three dependent launches.
// Norms and residual are two launches because together they need more registers than
// four workgroups a CU leave (200 us in one, spilling or at three a CU).  Every
// workgroup re-sums the partials of the pass before (at most kRedMaxBlocks of them, in
// one order), so alpha and beta are the same bits everywhere without a grid barrier or
// a launch of their own.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <stdexcept>

#include "common.hpp"
#include "redcg.hpp"

namespace v2g {

namespace {

using namespace rows;

constexpr int kNT = 256;                 // threads per workgroup
constexpr int kWaves = kNT / 64;
// workgroups of one launch: four per CU, what the registers of the passes allow
constexpr int kRedMaxBlocks = 1024;
constexpr int kXcds = 8;

enum : int { P_TT = 0, P_RR1, P_RR2, P_RP, P_PP };

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// sum over an aligned group of g lanes (16, 32 or 64)
__device__ __forceinline__ double group_sum(double v, int g)
{
    for (int o = g >> 1; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// sums of N values over the workgroup, in a fixed order; valid in every thread
template <int N>
__device__ __forceinline__ void block_sums(double (&v)[N], double *sh)
{
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; k++) {
        v[k] = wave_sum(v[k]);
        if ((threadIdx.x & 63) == 0) sh[k * kWaves + (threadIdx.x >> 6)] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; k++) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kWaves; w++) s += sh[k * kWaves + w];
        v[k] = s;
    }
}

// workgroup -> problem and place in it; XCD x (workgroups x, x + 8, ...) takes a
// contiguous eighth, so one L2 serves neighbouring entries
struct Place {
    const RedProb *pr;
    int prob, gb, lb, nb;
};

__device__ __forceinline__ Place place(const RedProb *prob, const int *blk)
{
    const int i = blockIdx.x, n = gridDim.x;
    const int x = i % kXcds, q = n / kXcds, rem = n % kXcds;
    Place p;
    p.gb = x * q + (x < rem ? x : rem) + i / kXcds;
    p.prob = blk[p.gb];
    p.pr = prob + p.prob;
    p.lb = p.gb - p.pr->b0;
    p.nb = p.pr->nb;
    return p;
}

// runs fn(segment, item, lane) over the tiles of list k that belong to this
// workgroup: elementwise items one per thread, wavefront items one per wave (all
// 64 lanes), workgroup items one per tile (all threads)
// Both orders are fixed, and so are the sums.
template <class F>
__device__ __forceinline__ void for_tiles(const Place &pl, int k, F fn)
{
    // an iteration's lists lead with latency-bound items and end with the cells' streams:
    // every other workgroup goes through its tiles backwards, so that a CU has both at a
    // time.  The start list's tiles share lines of rhs and y with their neighbours: all go
    // forwards (H50, the four passes 1.17 -> 1.11 ms)
    const int nt = pl.pr->ntile[k], mine = pl.lb < nt ? (nt - 1 - pl.lb) / pl.nb + 1 : 0;
    const RedTile *tiles = pl.pr->tile[k];
    for (int m = 0; m < mine; m++) {
        const RedTile &tl = tiles[pl.lb + (pl.lb & 1 && k > 0 ? mine - 1 - m : m) * pl.nb];
        const Segment &sg = tl.sg;
        if (sg.wave == 0) {
            const int64_t i = tl.first + threadIdx.x;
            if (i < sg.count) fn(sg, i, 0);
        } else if (sg.wave == 1) {
            const int64_t i = tl.first + (threadIdx.x >> 6);
            if (i < sg.count) fn(sg, i, (int)(threadIdx.x & 63));
        } else if (sg.wave == 3) {
            const int g = pl.pr->R.lanes;
            const int64_t i = tl.first + threadIdx.x / g;
            if (i < sg.count) fn(sg, i, (int)(threadIdx.x % g));
        } else {
            fn(sg, tl.first, (int)threadIdx.x);
        }
    }
}

// the vectors of one problem in an iteration of parity par: u0, v0, p0, mu0, nu0 as
// the iteration before left them, u1, ... as this one leaves them
struct View {
    double *g, *t, *w, *u0, *u1, *v0, *v1, *r, *p0, *p1, *s, *mu0, *mu1, *nu0, *nu1, *om, *ams, *scal;
};

__device__ __forceinline__ View view(const RedBufs &B, const RedProb &p, int prob, int par)
{
    const int o = par ^ 1;
    return {B.g + p.oD, B.t + p.oD, B.w + p.oD, B.u[o] + p.oD, B.u[par] + p.oD, B.v[o] + p.oD,
            B.v[par] + p.oD, B.r + p.oR, B.p[o] + p.oR, B.p[par] + p.oR, B.s + p.oS, B.mu[o] + p.oM,
            B.mu[par] + p.oM, B.nu[o] + p.oM, B.nu[par] + p.oM, B.om + p.oM, B.ams + p.oM,
            B.scal + (int64_t)prob * kRedScal};
}

__device__ __forceinline__ double *part(const RedBufs &B, int k, int gb)
{
    return B.part + (int64_t)k * kRedMaxBlocks + gb;
}

// a + b y, element by element, as an indexable vector
struct Axpy {
    const double *__restrict__ a;
    const double *__restrict__ y;
    double b;
    __device__ __forceinline__ double operator[](int64_t i) const { return fma(b, y[i], a[i]); }
};

struct Sum {
    Axpy a, b;
    __device__ __forceinline__ double operator[](int64_t i) const { return a[i] + b[i]; }
};

struct Ptr {
    const double *__restrict__ a;
    __device__ __forceinline__ double operator[](int64_t i) const { return a[i]; }
};

__device__ __forceinline__ double cell_sq(const Cell &t)
{
    return ((t.ab[0] * t.ab[0] + t.ab[1] * t.ab[1]) + (t.ab[2] * t.ab[2] + t.ab[3] * t.ab[3])) +
           (t.aa * t.aa + t.bb * t.bb);
}

// The cells of one irrep, one per thread: bases that every thread shares (scalar
// registers) and one 32-bit byte offset (fewer than 2^30 / 6 cells, redlayout.cc), which
// spares a 64-bit address per load.
__device__ __forceinline__ double ld(const double *__restrict__ b, uint32_t off)
{
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(b) + off);
}

__device__ __forceinline__ void st(double *__restrict__ b, uint32_t off, double v)
{
    *reinterpret_cast<double *>(reinterpret_cast<char *>(b) + off) = v;
}

struct CellAt {
    int64_t ab, aa, bb, cc;   // first D2ab / D2aa / D2bb entry of the irrep, cells of the irrep
    uint32_t off;
    __device__ __forceinline__ Cell load(const double *__restrict__ x) const
    {
        Cell c;
#pragma unroll
        for (int o = 0; o < 4; o++) c.ab[o] = ld(x + ab + o * cc, off);
        c.aa = ld(x + aa, off);
        c.bb = ld(x + bb, off);
        return c;
    }
    __device__ __forceinline__ void store(double *__restrict__ x, const Cell &c) const
    {
#pragma unroll
        for (int o = 0; o < 4; o++) st(x + ab + o * cc, off, c.ab[o]);
        st(x + aa, off, c.aa);
        st(x + bb, off, c.bb);
    }
};

// a + f b
__device__ __forceinline__ Cell cell_axpy(double f, const Cell &b, const Cell &a)
{
    Cell c;
#pragma unroll
    for (int o = 0; o < 4; o++) c.ab[o] = fma(f, b.ab[o], a.ab[o]);
    c.aa = fma(f, b.aa, a.aa);
    c.bb = fma(f, b.bb, a.bb);
    return c;
}

__device__ __forceinline__ Cell cell_add(const Cell &a, const Cell &b) { return cell_axpy(1.0, b, a); }

// the record of cell i of an irrep, if its pairs share an orbital (one bit a cell, a
// wavefront's in one word)
__device__ __forceinline__ const CellRec *shared_cell(const RedProb &p, const Segment &sg, int64_t i)
{
    const int64_t w = sg.aux + __builtin_amdgcn_readfirstlane((int)(i >> 6));
    const uint64_t b = p.bits[w], m = (uint64_t)1 << (i & 63);
    return b & m ? p.cell + p.rank[w] + __popcll(b & (m - 1)) : nullptr;
}

// an entry of the start list's RK_AB / RK_DIAG segments; false: no entry
__device__ __forceinline__ bool start_entry(const RedLayout &R, const Segment &sg, int64_t i, AbEntry &a)
{
    if (sg.kind == RK_DIAG) return diag_ab(R, i, a);
    a = cell_ab(R, sg.h, i);
    return true;
}

__device__ __forceinline__ bool is_ab(const Segment &sg) { return sg.kind == RK_AB || sg.kind == RK_DIAG; }

// slot of a D1 + Q1 row's Q1 part
__device__ __forceinline__ int64_t q1_slot(const RedLayout &R, const Segment &sg, int64_t i)
{
    return R.soff[sg.sub ? SF_Q1B : SF_Q1A] + (sg.start - R.L.xoff[sg.sub ? XB_D1B : XB_D1A][0]) + i;
}

// the full rows of the explicit rows aligned with cell k of irrep h
__device__ __forceinline__ int64_t cell_row(const RedLayout &R, const DevLayout &Lo, int j, int h, int64_t k)
{
    return (j ? Lo.rowoff[RF_SPIN_ANTI][j - 1][h] : Lo.rowoff[RF_SPIN_D2][0][h]) + (k - R.aa0[h]);
}

// what the norms of the iteration before say: the stopping rule and the next direction
struct Eval {
    bool done;
    double rr, nrm, beta, pp2, iter;
};

__device__ __forceinline__ Eval evaluate(const RedBufs &B, const Place &pl, const double *scal,
                                         const double *a, double *sh)
{
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i = threadIdx.x; i < pl.nb; i += kNT) {
        v[0] += *part(B, P_RR1, pl.pr->b0 + i);
        v[1] += *part(B, P_RR2, pl.pr->b0 + i);
        v[2] += *part(B, P_RP, pl.pr->b0 + i);
        v[3] += *part(B, P_PP, pl.pr->b0 + i);
    }
    block_sums<4>(v, sh);
    Eval e;
    e.rr = v[0] + v[1];
    e.nrm = sqrt(e.rr);
    const double begun = a[4];
    if (begun == 0.0) {          // the first direction is the first residual
        e.beta = 0.0;
        e.pp2 = v[1];
        e.iter = 0.0;
        e.done = scal[RS_MAXIT] <= 0.0;
        return e;
    }
    e.beta = e.rr / a[1];
    e.pp2 = v[1] + 2.0 * e.beta * v[2] + e.beta * e.beta * v[3];
    const bool conv = e.nrm < scal[RS_TOL];
    e.iter = conv ? begun - 1.0 : begun;
    e.done = conv || begun >= scal[RS_MAXIT];
    return e;
}

// ---- plan -------------------------------------------------------------------
// The records of the listed entries and cells from their orbitals: on the host, with the
// upload, they were most of the plan (H50: 1.5 of 1.9 ms).
__global__ void __launch_bounds__(kNT)
k_red_records(const RedProb *__restrict__ prob)
{
    const RedProb &p = prob[blockIdx.y];
    const int first = blockIdx.x * kNT + threadIdx.x, step = gridDim.x * kNT;
    for (int i = first; i < p.nab; i += step) {
        const RedKey k(p.ab_key[i]);
        p.ab[i] = make_ab_rec(p.R, k.p, k.q, k.r, k.s);
    }
    for (int i = first; i < p.ncell; i += step) {
        const RedKey k(p.cell_key[i]);
        p.cell[i] = make_cell_rec(p.R, k.p, k.q, k.r, k.s);
    }
}

// ---- start of a solve -------------------------------------------------------
// These passes and the last one, k_red_y, meet the full rows of rhs and y, where the rows of
// neighbouring entries lie apart: lines that several wavefronts touch bound them (H50: 258, 345,
// 150 and 357 us; 349, 394, 179 and 445 with the rows' places from the geminal tables).  The
// entries by blocks of 8 x 8 orbitals, or an entry's rows all loaded before the first
// store, change nothing.

// t = (A^T y)_D from the full rows; u, v, w, p, mu, nu, om = 0 and the scalars
__global__ void __launch_bounds__(kNT, 4)
k_red_aty(const RedProb *__restrict__ prob, const int *__restrict__ blk, RedBufs B,
          const double *__restrict__ y, double tol, const double *__restrict__ tolv,
          const int *__restrict__ active, int maxiter)
{
    const Place pl = place(prob, blk);
    const View V = view(B, *pl.pr, pl.prob, 0);
    if (active && !active[pl.prob]) {
        if (pl.lb == 0 && threadIdx.x == 0) {
            V.scal[RS_A] = V.scal[RS_A + 6] = V.scal[RS_DONE] = 1.0;
            V.scal[RS_ITER] = V.scal[RS_NRM] = 0.0;
        }
        return;
    }
    const RedLayout &R = pl.pr->R;
    const DevLayout &Lo = *pl.pr->full;
    for_tiles(pl, 0, [&](const Segment &sg, int64_t i, int lane) {
        if (is_ab(sg)) {
            AbEntry a;
            if (start_entry(R, sg, i, a)) V.t[a.pos] = full_at_ab(R, Lo, a, y);
        } else if (sg.kind == RK_AA) {
            const AbEntry a = cell_entry(R, sg.h, i);
            for (int sp = 0; sp < 2; sp++) V.t[R.nAB + sp * R.nAA + sg.start + i] = full_at_aa(Lo, sp, a, y);
        } else if (sg.kind == XS_D1) {
            const double a = wave_sum(atu_d1_wave(Lo, sg, i, lane, y));
            if (lane == 0) V.t[sg.start + i] = a;
        } else if (sg.kind == RK_DVEC) {
            V.u0[i] = V.v0[i] = V.w[i] = V.u1[i] = V.v1[i] = 0.0;
        } else if (sg.kind == RK_RVEC) {
            V.p0[i] = 0.0;
        } else if (sg.kind == RK_MVEC) {
            V.mu0[i] = V.nu0[i] = V.om[i] = 0.0;
        }
    });
    if (pl.lb == 0 && threadIdx.x == 0) {
        // the zero that indices without an entry point at
        V.u0[R.nD] = V.u1[R.nD] = V.v0[R.nD] = V.v1[R.nD] = 0.0;
        V.r[R.nR] = V.p0[R.nR] = V.p1[R.nR] = 0.0;
        V.mu0[R.nM] = V.mu1[R.nM] = V.nu0[R.nM] = V.nu1[R.nM] = 0.0;
        double *a = V.scal + RS_A + 6;      // as left by an iteration of parity 1
        a[0] = 0.0;                         // done
        a[1] = 1.0;                         // r.z (the first beta is 0)
        a[2] = 0.0;                         // d
        a[3] = 0.0;
        a[4] = 0.0;                         // iterations begun
        double *b = V.scal + RS_B + 2;
        b[0] = 1.0;                         // c
        b[1] = 0.0;                         // e
        V.scal[RS_DONE] = 0.0;
        V.scal[RS_NRM] = 0.0;
        V.scal[RS_ITER] = 0.0;
        V.scal[RS_TOL] = tolv ? tolv[pl.prob] : tol;
        V.scal[RS_MAXIT] = (double)maxiter;
    }
}

// visits the self rows of a start-list item: fn(slot, full row, D2 / D1 part of x
// minus the maximal-spin part of m, whether a maximal-spin row reads it)
template <class X, class M, class F>
__device__ __forceinline__ void self_slots(const RedLayout &R, const DevLayout &Lo, const Segment &sg,
                                           int64_t i, int lane, const X &x, const M &m, F fn)
{
    if (is_ab(sg)) {
        AbEntry a;
        if (!start_entry(R, sg, i, a)) return;
        auto one = [&](int f, double o, bool ms = false) { fn(R.soff[f] + a.pos, self_row_ab(R, f, a), o, ms); };
        const SelfAb<X> o(R, a, x);
        if (R.L.q2) one(SF_Q2AB, o.q2);
        if (R.L.g2) {
            one(SF_G2AB, o.g1);
            one(SF_G2BA, o.g2 - ms_part(R, a.p, a.q, a.r, a.s, m), ms_reads(R, a.p, a.q, a.r, a.s));
            one(SF_G2X, o.x);
            one(SF_G2Y, o.x);
            one(SF_G2A, o.ga);
            one(SF_G2B, o.gb);
        }
        if (R.nblk_d) {
            const D200Ab<X> d(R, a, x);
            for (int k = 0; k < R.nblk_d; k++) one(SF_D0 + k, d.row(R, a, k));
        }
    } else if (sg.kind == RK_AA) {
        if (!R.L.q2) return;
        const AbEntry a = cell_entry(R, sg.h, i);
        for (int sp = 0; sp < 2; sp++)
            fn(R.soff[SF_Q2AA + sp] + sg.start + i, Lo.rowoff[RF_Q2AA][sp][sg.h] + i, self_row_aa(R, sp, a, x), false);
    } else if (sg.kind == XS_D1 && lane == 0) {
        fn(q1_slot(R, sg, i), self_row_d1(Lo, sg.sub, sg.h, i), x[sg.start + i], false);
    }
}

// s = rhs - y - B2 t + P y_ms on the self rows, and the sums of its squares
__global__ void __launch_bounds__(kNT, 4)
k_red_self(const RedProb *__restrict__ prob, const int *__restrict__ blk, RedBufs B,
           const double *__restrict__ rhs, const double *__restrict__ y)
{
    __shared__ double sh[2 * kWaves];
    const Place pl = place(prob, blk);
    const View V = view(B, *pl.pr, pl.prob, 0);
    if (V.scal[RS_DONE] != 0.0) return;
    const RedLayout &R = pl.pr->R;
    const DevLayout &Lo = *pl.pr->full;
    const Ptr t{V.t}, ms{y + (R.nM ? Lo.rowoff[RF_MAXSPIN][0][0] : 0)};
    double ss[2] = {0.0, 0.0};
    for_tiles(pl, 0, [&](const Segment &sg, int64_t i, int lane) {
        self_slots(R, Lo, sg, i, lane, t, ms, [&](int64_t slot, int64_t row, double o, bool ms) {
            const double v = rhs[row] - y[row] - o;
            V.s[slot] = v;
            ss[0] += ms ? 0.0 : v * v;
            ss[1] += ms ? v * v : 0.0;
        });
    });
    block_sums<2>(ss, sh);
    if (threadIdx.x == 0) {
        *part(B, P_RR2, pl.gb) = ss[0];
        *part(B, P_RR1, pl.gb) = ss[1];
    }
}

// g = B2^T s, and r = rhs - A (A^T y) on the explicit rows
__global__ void __launch_bounds__(kNT, 4)
k_red_expl(const RedProb *__restrict__ prob, const int *__restrict__ blk, RedBufs B,
           const double *__restrict__ rhs, const double *__restrict__ y)
{
    __shared__ double sh[kWaves];
    const Place pl = place(prob, blk);
    const View V = view(B, *pl.pr, pl.prob, 0);
    if (V.scal[RS_DONE] != 0.0) return;
    const RedLayout &R = pl.pr->R;
    const DevLayout &Lo = *pl.pr->full;
    const Ptr s{V.s}, t{V.t}, ms{y + (R.nM ? Lo.rowoff[RF_MAXSPIN][0][0] : 0)};
    double rr[1] = {0.0};
    auto row = [&](int64_t k, int64_t full, double at) {
        const double ri = rhs[full] - at;
        V.r[k] = ri;
        rr[0] += ri * ri;
    };
    for_tiles(pl, 0, [&](const Segment &sg, int64_t i, int lane) {
        if (is_ab(sg)) {
            AbEntry a;
            if (start_entry(R, sg, i, a)) V.g[a.pos] = self_at_ab(R, a, s);
        } else if (sg.kind == RK_AA) {
            const AbEntry a = cell_entry(R, sg.h, i);
            const int64_t k = sg.start + i;
            for (int sp = 0; sp < 2; sp++) V.g[R.nAB + sp * R.nAA + k] = self_at_aa(R, sp, sg.h, a, s);
            if (R.cells) {
                double at[3];
                cell_rows(load_cell(R, a.pos, sg.count, k, t), at);
                for (int j = 0; j < 3; j++) row(j * R.nAA + k, cell_row(R, Lo, j, sg.h, k), at[j]);
            }
        } else if (sg.kind == XS_D1) {
            const double a = wave_sum(self_at_d1(R, sg.sub, sg.h, i, lane, s));
            if (lane == 0) V.g[sg.start + i] = a;
        } else if (sg.kind == RK_MS) {
            // sum_i of A^T y over the row's G2ba entries: P^T P y_ms - P^T y_self
            const int pr = R.L.bab[R.L.bab_off[0] + i], k = P0(pr), l = P1(pr);
            double v = lane < R.lanes ? ms_row_gram(R, sg.sub, (int)i, lane, ms) : 0.0;
            for (int j = lane; j < R.L.amo; j += 64) {
                const AbEntry a{sg.sub ? l : j, sg.sub ? j : k, sg.sub ? j : l, sg.sub ? k : j, 0};
                v -= y[self_row_ab(R, SF_G2BA, a)];
            }
            v = wave_sum(v);
            if (lane == 0) row(sg.start + i, sg.aux + i, v);
        }
    });
    for_tiles(pl, 2, [&](const Segment &sg, int64_t i, int lane) {
        if (sg.kind == RF_SPIN_D1) {
            row(sg.start + i, sg.aux + i, t[R.L.xoff[XB_D1A][sg.h] + i] - t[R.L.xoff[XB_D1B][sg.h] + i]);
        } else if (sg.kind == RF_CONTR) {
            const double v = group_sum(long_row(R, sg, i, lane, R.lanes, t), R.lanes);
            if (lane == 0) row(sg.start + i, sg.aux + i, v);
        } else if (sg.wave == 2) {
            double v[1] = {long_row(R, sg, i, lane, kNT, t)};
            block_sums<1>(v, sh);
            if (lane == 0) row(sg.start + i, sg.aux + i, v[0]);
        }
    });
    block_sums<1>(rr, sh);
    if (threadIdx.x == 0) {
        *part(B, P_RR1, pl.gb) += rr[0];
        *part(B, P_RP, pl.gb) = 0.0;
        *part(B, P_PP, pl.gb) = 0.0;
    }
}

// ---- one iteration ----------------------------------------------------------

// direction: beta and the stopping rule; v, nu, p; ||A^T p||^2 (t = A^T p is kept where
// it is gathered from: listed entries and D1) and the maximal-spin rows of A A^T p
// FULL: every problem is a singlet with Q2, G2 and spin rows, so no load hides behind a
// branch; else the flags of each layout decide
template <bool FULL>
__global__ void __launch_bounds__(kNT, 4)
k_red_dir(const RedProb *__restrict__ prob, const int *__restrict__ blk, RedBufs B, int par)
{
    __shared__ double sh[4 * kWaves];
    const Place pl = place(prob, blk);
    const View V = view(B, *pl.pr, pl.prob, par);
    double *a1 = V.scal + RS_A + 6 * par;
    const double *a0 = V.scal + RS_A + 6 * (par ^ 1), *b0 = V.scal + RS_B + 2 * (par ^ 1);
    if (a0[0] != 0.0) {
        if (pl.lb == 0 && threadIdx.x == 0) a1[0] = 1.0;
        return;
    }
    const Eval ev = evaluate(B, pl, V.scal, a0, sh);
    const double d = b0[0] + ev.beta * a0[2];
    if (pl.lb == 0 && threadIdx.x == 0) {
        if (ev.done) {
            V.scal[RS_DONE] = 1.0;
            V.scal[RS_NRM] = a0[4] > 0.0 ? ev.nrm : 0.0;
            V.scal[RS_ITER] = ev.iter;
        }
        a1[0] = ev.done ? 1.0 : 0.0;
        a1[1] = ev.rr;
        a1[2] = d;
        a1[3] = ev.pp2;
        a1[4] = a0[4] + 1.0;
        if (a0[4] == 0.0) V.scal[RS_NRM0] = ev.nrm;
    }
    if (ev.done) return;
    const RedLayout &R = pl.pr->R;
    const bool q2 = FULL || R.L.q2, g2 = FULL || R.L.g2, cells = FULL || R.cells;
    const int nd = FULL ? 1 : R.nblk_d;
    const Axpy v{V.u0, V.v0, ev.beta}, p{V.r, V.p0, ev.beta}, nu{V.mu0, V.nu0, ev.beta};
    double tt[1] = {0.0};
    auto keep = [&](int64_t k, double t) {
        V.t[k] = t;
        V.v1[k] = v[k];
        tt[0] += t * t;
    };
    for_tiles(pl, 1, [&](const Segment &sg, int64_t i, int lane) {
        if (sg.kind == RK_CELLS) {
            const CellRec *rec = shared_cell(*pl.pr, sg, i);
            const int64_t k0 = R.aa0[sg.h];
            const CellAt at{R.ab0[sg.h], R.nAB + k0, R.nAB + R.nAA + k0, sg.count, (uint32_t)i * 8u};
            const Cell u = at.load(V.u0), v0 = at.load(V.v0), g = at.load(V.g);
            double pr[3] = {0.0, 0.0, 0.0};
            if (cells)
#pragma unroll
                for (int j = 0; j < 3; j++)
                    pr[j] = fma(ev.beta, ld(V.p0 + j * R.nAA + k0, at.off), ld(V.r + j * R.nAA + k0, at.off));
            const Cell vc = cell_axpy(ev.beta, v0, u);
            Cell t = cell_at(q2, g2, nd, cells, d, g, vc, pr);
            if (rec) {
                shared_at(R, *rec, v, nu, p, t);
                at.store(V.t, t);
            }
            tt[0] += cell_sq(t);
            at.store(V.v1, vc);
            if (cells)
#pragma unroll
                for (int j = 0; j < 3; j++) st(V.p1 + j * R.nAA + k0, at.off, pr[j]);
        } else if (sg.kind == RK_LIST_AB) {
            const AbRec a = pl.pr->ab[i];
            const double t = fma(d, V.g[a.pos], rec_expl_ab(R, a, p)) +
                             (AbVals(R, a, v).gram(R, a) + (nu[a.m0] + nu[a.m1]));
            keep(a.pos, t);
        } else if (sg.kind == XS_D1) {
            const int64_t k = sg.start + i;
            const double t = group_sum(atu_d1_wave<false, true>(R.L, sg, i, lane, p) +
                                           gram_d1(R, sg.sub, sg.h, i, lane, v, nu), R.lanes) + d * V.g[k];
            if (lane == 0) keep(k, t);
        } else if (sg.kind == RK_ROWS) {
            V.p1[sg.start + i] = p[sg.start + i];
        } else if (sg.kind == RK_MVEC) {
            V.nu1[i] = nu[i];
        } else {
            // maximal-spin row: (A A^T p) = P^T (P p_ms - p_self), the sum of A^T p over its
            // G2ba entries, and their squares
            const int64_t m0 = R.L.rowoff[RF_MAXSPIN][0][0];
            const Sum m{nu, Axpy{V.r + m0, V.p0 + m0, ev.beta}};
            const double a = group_sum(ms_row_self(R, sg.sub, (int)i, lane, d, Ptr{V.s}, v, m, tt), R.lanes);
            if (lane == 0) V.ams[sg.sub * (R.nM / 2) + i] = -a;
        }
    });
    block_sums<1>(tt, sh);
    if (threadIdx.x == 0) *part(B, P_TT, pl.gb) = tt[0];
}

// residual: alpha; u, w, mu, om, c, e; the explicit rows of r and y
__global__ void __launch_bounds__(kNT, 4)
k_red_res(const RedProb *__restrict__ prob, const int *__restrict__ blk, RedBufs B,
          double *__restrict__ y, int par)
{
    __shared__ double sh[kWaves];
    const Place pl = place(prob, blk);
    const View V = view(B, *pl.pr, pl.prob, par);
    const double *a = V.scal + RS_A + 6 * par, *b0 = V.scal + RS_B + 2 * (par ^ 1);
    double *b1 = V.scal + RS_B + 2 * par;
    if (a[0] != 0.0) {
        if (pl.lb == 0 && threadIdx.x == 0) { b1[0] = b0[0]; b1[1] = b0[1]; }
        return;
    }
    double tt[1] = {0.0};
    for (int i = threadIdx.x; i < pl.nb; i += kNT) tt[0] += *part(B, P_TT, pl.pr->b0 + i);
    block_sums<1>(tt, sh);
    const double alpha = a[1] / (tt[0] + a[3]), d = a[2];
    if (pl.lb == 0 && threadIdx.x == 0) {
        b1[0] = fma(-alpha, d, b0[0]);
        b1[1] = fma(alpha, d, b0[1]);
    }
    const RedLayout &R = pl.pr->R;
    const DevLayout &Lo = *pl.pr->full;
    const Ptr t{V.t};
    double rr[1] = {0.0};
    auto row = [&](int64_t k, int64_t full, double at) {
        const double yn = fma(alpha, V.p1[k], y[full]), rn = fma(-alpha, at, V.r[k]);
        y[full] = yn;
        V.r[k] = rn;
        rr[0] = fma(rn, rn, rr[0]);
    };
    for_tiles(pl, 2, [&](const Segment &sg, int64_t i, int lane) {
        if (sg.kind == RK_CELLS) {
            const CellRec *rec = shared_cell(*pl.pr, sg, i);
            const int64_t k0 = R.aa0[sg.h];
            const CellAt at{R.ab0[sg.h], R.nAB + k0, R.nAB + R.nAA + k0, sg.count, (uint32_t)i * 8u};
            // every load before the first store, so that none waits for another
            const Cell vc = at.load(V.v1), g = at.load(V.g), u = at.load(V.u0), w = at.load(V.w);
            double pr[3] = {0.0, 0.0, 0.0}, r[3], yy[3];
            if (R.cells)
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    pr[j] = ld(V.p1 + j * R.nAA + k0, at.off);
                    r[j] = ld(V.r + j * R.nAA + k0, at.off);
                    yy[j] = ld(y + cell_row(R, Lo, j, sg.h, k0), at.off);
                }
            Cell tc = cell_at(R.L.q2, R.L.g2, R.nblk_d, R.cells, d, g, vc, pr);
            if (rec) tc = at.load(V.t);
            at.store(V.u1, cell_axpy(-alpha, cell_add(vc, tc), u));
            at.store(V.w, cell_axpy(alpha, vc, w));
            if (R.cells) {
                double ct[3];
                cell_rows(tc, ct);
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    const double rn = fma(-alpha, ct[j], r[j]);
                    rr[0] = fma(rn, rn, rr[0]);
                    st(V.r + j * R.nAA + k0, at.off, rn);
                    st(y + cell_row(R, Lo, j, sg.h, k0), at.off, fma(alpha, pr[j], yy[j]));
                }
            }
        } else if (sg.kind == RK_STEP) {
            const int64_t k = sg.start + i;
            const double v = V.v1[k], u = fma(-alpha, v + V.t[k], V.u0[k]), w = fma(alpha, v, V.w[k]);
            V.u1[k] = u;
            V.w[k] = w;
        } else if (sg.kind == RK_MVEC) {
            const double v = V.nu1[i], m = V.mu0[i], o = V.om[i];
            V.mu1[i] = fma(-alpha, v + V.p1[R.L.rowoff[RF_MAXSPIN][0][0] + i], m);
            V.om[i] = fma(alpha, v, o);
        } else if (sg.kind == RF_MAXSPIN) {
            row(sg.start + i, sg.aux + i, V.ams[sg.sub * (R.nM / 2) + i]);
        } else if (sg.kind == RF_SPIN_D1) {
            row(sg.start + i, sg.aux + i, t[R.L.xoff[XB_D1A][sg.h] + i] - t[R.L.xoff[XB_D1B][sg.h] + i]);
        } else if (sg.kind == RF_CONTR) {
            const double at = group_sum(long_row(R, sg, i, lane, R.lanes, t), R.lanes);
            if (lane == 0) row(sg.start + i, sg.aux + i, at);
        } else if (sg.wave == 2) {
            double at[1] = {long_row(R, sg, i, lane, kNT, t)};
            block_sums<1>(at, sh);
            if (lane == 0) row(sg.start + i, sg.aux + i, at[0]);
        }
    });
    block_sums<1>(rr, sh);
    if (threadIdx.x == 0) *part(B, P_RR1, pl.gb) = rr[0];
}

// norms: r.r, r.p, p.p of the self rows, r of this iteration and p its direction
template <bool FULL>
__global__ void __launch_bounds__(kNT, 4)
k_red_norm(const RedProb *__restrict__ prob, const int *__restrict__ blk, RedBufs B, int par)
{
    __shared__ double sh[4 * kWaves];
    const Place pl = place(prob, blk);
    const View V = view(B, *pl.pr, pl.prob, par);
    if (V.scal[RS_A + 6 * par] != 0.0) return;
    const double c = V.scal[RS_B + 2 * par], d = V.scal[RS_A + 6 * par + 2];
    const RedLayout &R = pl.pr->R;
    const bool q2 = FULL || R.L.q2, g2 = FULL || R.L.g2;
    const int nd = FULL ? 1 : R.nblk_d;
    const Ptr u{V.u1}, v{V.v1}, mu{V.mu1}, nu{V.nu1};
    double n[4] = {0.0, 0.0, 0.0, 0.0};
    const double rr1 = *part(B, P_RR1, pl.gb);   // of the residual pass
    auto self = [&](double s, double ru, double pv) {
        const double r = fma(c, s, ru), p = fma(d, s, pv);
        n[0] = fma(r, r, n[0]);
        n[1] = fma(r, p, n[1]);
        n[2] = fma(p, p, n[2]);
    };
    // a G2ba row; ms: a maximal-spin row reads it
    auto g2ba = [&](bool ms, double s, double ru, double pv) {
        const double r = fma(c, s, ru), p = fma(d, s, pv), rr = r * r;
        n[0] += ms ? 0.0 : rr;
        n[1] += ms ? 0.0 : r * p;
        n[2] += ms ? 0.0 : p * p;
        n[3] += ms ? rr : 0.0;
    };
    for_tiles(pl, 3, [&](const Segment &sg, int64_t i, int) {
        if (sg.kind == RK_CELLS) {
            const CellRec *rec = shared_cell(*pl.pr, sg, i);
            const int64_t k0 = R.aa0[sg.h], cc = sg.count;
            const CellAt at{R.ab0[sg.h], R.nAB + k0, R.nAB + R.nAA + k0, cc, (uint32_t)i * 8u};
            const uint32_t off = at.off;
            const Cell uc = at.load(V.u1), vc = at.load(V.v1);
            const double *s = V.s + at.ab;
            // rows that a shared orbital does not touch
            if (g2) {
#pragma unroll
                for (int o = 0; o < 4; o++) {
                    self(ld(s + o * cc + R.soff[SF_G2X], off), uc.ab[o], vc.ab[o]);
                    self(ld(s + o * cc + R.soff[SF_G2Y], off), uc.ab[o], vc.ab[o]);
                }
            }
            for (int b = 0; b < nd; b++) {
                double cf[4];
                d200_coef(b, FULL || R.L.singlet, false, false, cf);
#pragma unroll
                for (int o = 0; o < 4; o++)
                    self(ld(s + R.soff[SF_D0 + b] + o * cc, off),
                         cf[0] * uc.ab[o] + cf[1] * uc.ab[o ^ 1] + cf[2] * uc.ab[o ^ 2] + cf[3] * uc.ab[o ^ 3],
                         cf[0] * vc.ab[o] + cf[1] * vc.ab[o ^ 1] + cf[2] * vc.ab[o ^ 2] + cf[3] * vc.ab[o ^ 3]);
            }
            if (!rec) {
                if (q2) {
#pragma unroll
                    for (int o = 0; o < 4; o++) self(ld(s + R.soff[SF_Q2AB] + o * cc, off), uc.ab[o], vc.ab[o]);
                    self(ld(V.s + R.soff[SF_Q2AA] + k0, off), uc.aa, vc.aa);
                    self(ld(V.s + R.soff[SF_Q2BB] + k0, off), uc.bb, vc.bb);
                }
                if (g2) {
#pragma unroll
                    for (int o = 0; o < 4; o++) {
                        const double *so = s + o * cc;
                        const double x = uc.ab[o], z = vc.ab[o], sg2 = o == 1 || o == 2 ? 1.0 : -1.0;
                        self(ld(so + R.soff[SF_G2AB], off), -x, -z);
                        self(ld(so + R.soff[SF_G2BA], off), -x, -z);
                        self(ld(so + R.soff[SF_G2A], off), sg2 * uc.aa, sg2 * vc.aa);
                        self(ld(so + R.soff[SF_G2B], off), sg2 * uc.bb, sg2 * vc.bb);
                    }
                }
            }
        } else if (sg.kind == RK_SHARED) {
            // the other rows of a cell whose pairs share an orbital, one orientation a thread
            const int64_t nc = sg.dim;
            const int o = (int)(i / nc);
            const CellRec a = pl.pr->cell[i - o * nc];
            const int64_t ga = R.L.gems_aa[a.flags >> 8], e = a.pos + o * ga * ga, k = a.k;
            const double f = o == 1 || o == 2 ? 1.0 : -1.0;
            const SharedAt su(R, a, o, u, mu), sv(R, a, o, v, nu);
            const double x = u[e], z = v[e], xa = u[R.nAB + k], za = v[R.nAB + k], xb = u[R.nAB + R.nAA + k],
                         zb = v[R.nAB + R.nAA + k];
            if (q2) {
                self(V.s[R.soff[SF_Q2AB] + e], x + su.q2, z + sv.q2);
                if (o < 2)
                    self(V.s[R.soff[SF_Q2AA + o] + k], (o ? xb : xa) + shared_q2(R, a, o, u),
                         (o ? zb : za) + shared_q2(R, a, o, v));
            }
            if (g2) {
                self(V.s[R.soff[SF_G2AB] + e], su.g1 - x, sv.g1 - z);
                g2ba(shared_ms(R, a, o), V.s[R.soff[SF_G2BA] + e], su.g2 - x, sv.g2 - z);
                self(V.s[R.soff[SF_G2A] + e], fma(f, xa, su.g1), fma(f, za, sv.g1));
                self(V.s[R.soff[SF_G2B] + e], fma(f, xb, su.gb), fma(f, zb, sv.gb));
            }
        } else if (sg.kind == RK_LIST_AB) {
            const AbRec a = pl.pr->ab[i];
            const AbVals su(R, a, u), sv(R, a, v);
            auto one = [&](int f, double ru, double pv) { self(V.s[R.soff[f] + a.pos], ru, pv); };
            if (q2) one(SF_Q2AB, su.q2(), sv.q2());
            if (g2) {
                one(SF_G2AB, su.g1(), sv.g1());
                g2ba(a.m0 != R.nM || a.m1 != R.nM, V.s[R.soff[SF_G2BA] + a.pos],
                     su.g2() - (mu[a.m0] + mu[a.m1]), sv.g2() - (nu[a.m0] + nu[a.m1]));
                one(SF_G2X, su.x0, sv.x0);
                one(SF_G2Y, su.x0, sv.x0);
                one(SF_G2A, su.ga(a), sv.ga(a));
                one(SF_G2B, su.gb(a), sv.gb(a));
            }
            for (int b = 0; b < nd; b++) one(SF_D0 + b, su.d200(R, a, b), sv.d200(R, a, b));
        } else {   // the D1 + Q1 rows
            self(V.s[q1_slot(R, sg, i)], u[sg.start + i], v[sg.start + i]);
        }
    });
    block_sums<4>(n, sh);
    if (threadIdx.x == 0) {
        *part(B, P_RR2, pl.gb) = n[0];
        *part(B, P_RP, pl.gb) = n[1];
        *part(B, P_PP, pl.gb) = n[2];
        *part(B, P_RR1, pl.gb) = rr1 + n[3];
    }
}

// the host's view after an even number of iterations: done, ||r||, iteration count
__global__ void __launch_bounds__(kNT)
k_red_status(const RedProb *__restrict__ prob, RedBufs B)
{
    __shared__ double sh[4 * kWaves];
    Place pl;
    pl.prob = blockIdx.x;
    pl.pr = prob + pl.prob;
    pl.gb = pl.lb = 0;
    pl.nb = pl.pr->nb;
    double *scal = B.scal + (int64_t)pl.prob * kRedScal;
    if (scal[RS_DONE] != 0.0) return;
    const double *a = scal + RS_A + 6;
    const Eval ev = evaluate(B, pl, scal, a, sh);
    if (threadIdx.x == 0) {
        scal[RS_NRM] = a[4] > 0.0 ? ev.nrm : 0.0;
        scal[RS_ITER] = ev.iter;
        scal[RS_DONE] = ev.done ? 1.0 : 0.0;
    }
}

// y += e s + B2 w - P om on the self rows
__global__ void __launch_bounds__(kNT, 4)
k_red_y(const RedProb *__restrict__ prob, const int *__restrict__ blk, RedBufs B,
        double *__restrict__ y, const int *__restrict__ active)
{
    const Place pl = place(prob, blk);
    if (active && !active[pl.prob]) return;
    const View V = view(B, *pl.pr, pl.prob, 0);
    // no iterations: y keeps every bit (0 times a residual that is not finite is no zero,
    // and -0 + 0 is not -0)
    if (V.scal[RS_MAXIT] <= 0.0) return;
    const double e = V.scal[RS_B + 2 + 1];
    const RedLayout &R = pl.pr->R;
    const DevLayout &Lo = *pl.pr->full;
    const Ptr w{V.w}, om{V.om};
    for_tiles(pl, 0, [&](const Segment &sg, int64_t i, int lane) {
        self_slots(R, Lo, sg, i, lane, w, om, [&](int64_t slot, int64_t row, double o, bool) {
            y[row] += fma(e, V.s[slot], o);
        });
    });
}

}  // namespace

RedCG::~RedCG()
{
    if (d_prob_) (void)hipFree(d_prob_);
    if (d_blk_) (void)hipFree(d_blk_);
    if (d_work_) (void)hipFree(d_work_);
}

bool RedCG::build(const std::vector<const Layout *> &L, const std::vector<DevLayout> &dev,
                  const DevLayout *d_dev)
{
    np_ = (int)L.size();
    if (np_ > kRedMaxBlocks) return false;
    std::vector<RedProb> prob(np_);
    std::vector<RedWork> work(np_);
    std::vector<int64_t> tiles(np_);
    int64_t total = 0;
    for (int q = 0; q < np_; q++) {
        RedProb &p = prob[q];
        if (!make_red_layout(*L[q], dev[q], p.R, work[q], false)) return false;
        p.full = d_dev + q;
        full_ = full_ && p.R.L.q2 && p.R.L.g2 && p.R.cells;
        p.oD = nD_;
        p.oR = nR_;
        p.oS = nS_;
        p.oM = nM_;
        nD_ += p.R.nD + 1;
        nR_ += p.R.nR + 1;
        nS_ += p.R.nS;
        nM_ += p.R.nM + 1;
    }
    // the tiles of every problem's four lists, in one array
    std::vector<RedTile> tl;
    std::vector<size_t> to(4 * np_);
    auto list = [&](int q, int k) -> const std::vector<Segment> & {
        return k == 0 ? work[q].start : k == 1 ? work[q].dir : k == 2 ? work[q].res : work[q].norm;
    };
    auto items = [&](int q, const Segment &s) -> int64_t {
        return s.wave == 0 ? kNT : s.wave == 1 ? kWaves : s.wave == 3 ? kNT / prob[q].R.lanes : 1;
    };
    size_t ntl = 0;
    for (int q = 0; q < np_; q++)
        for (int k = 0; k < 4; k++)
            for (const Segment &s : list(q, k)) ntl += (size_t)((s.count + items(q, s) - 1) / items(q, s));
    tl.reserve(ntl);
    for (int q = 0; q < np_; q++) {
        tiles[q] = 1;
        for (int k = 0; k < 4; k++) {
            to[4 * q + k] = tl.size();
            for (const Segment &s : list(q, k)) {
                const int64_t per = items(q, s);
                for (int64_t i = 0; i < s.count; i += per) tl.push_back({s, i});
            }
            prob[q].ntile[k] = (int)(tl.size() - to[4 * q + k]);
            tiles[q] = std::max<int64_t>(tiles[q], prob[q].ntile[k]);
        }
        total += tiles[q];
    }
    // workgroups in proportion to the tiles, at least one a problem
    std::vector<int> blk;
    for (int q = 0; q < np_; q++) {
        const int64_t share = total <= kRedMaxBlocks ? tiles[q] : tiles[q] * (kRedMaxBlocks - np_) / total;
        prob[q].b0 = (int)blk.size();
        prob[q].nb = (int)std::max<int64_t>(1, std::min(share, tiles[q]));
        blk.insert(blk.end(), prob[q].nb, q);
    }
    nblk_ = (int)blk.size();
    if (nblk_ > kRedMaxBlocks) throw std::logic_error("reduced CG: more workgroups than partial sums");
    // one allocation, regions on 256-byte boundaries: the tiles, then what is uploaded beside
    // them in one piece, then the records
    auto room = [](size_t n) { return (n + 255) / 256 * 256; };
    const size_t tb = room(sizeof(RedTile) * tl.size());
    size_t sb = 0, nb = 0;
    auto bytes = [](const auto &v) { return sizeof(v[0]) * v.size(); };
    for (int q = 0; q < np_; q++) {
        const RedWork &w = work[q];
        sb += room(bytes(w.ab_key)) + room(bytes(w.cell_key)) + room(bytes(w.bits)) + room(bytes(w.rank)) +
              room(bytes(w.rowtab));
        nb += room(sizeof(AbRec) * w.ab_key.size()) + room(sizeof(CellRec) * w.cell_key.size());
    }
    HIPCHK(hipMalloc(&d_work_, tb + sb + nb));
    char *const base = static_cast<char *>(d_work_);
    std::vector<char> stage(sb);
    size_t at = 0;
    auto put = [&](const auto &v) {
        using T = std::decay_t<decltype(v[0])>;
        if (!v.empty()) std::memcpy(stage.data() + at, v.data(), bytes(v));
        const T *p = reinterpret_cast<const T *>(base + tb + at);
        at += room(bytes(v));
        return p;
    };
    char *rec = base + tb + sb;
    for (int q = 0; q < np_; q++) {
        RedProb &p = prob[q];
        const RedWork &w = work[q];
        for (int k = 0; k < 4; k++) p.tile[k] = reinterpret_cast<const RedTile *>(base) + to[4 * q + k];
        p.ab_key = put(w.ab_key);
        p.cell_key = put(w.cell_key);
        p.bits = put(w.bits);
        p.rank = put(w.rank);
        p.R.rowtab = put(w.rowtab);
        p.nab = (int)w.ab_key.size();
        p.ncell = (int)w.cell_key.size();
        p.ab = reinterpret_cast<AbRec *>(rec);
        rec += room(sizeof(AbRec) * p.nab);
        p.cell = reinterpret_cast<CellRec *>(rec);
        rec += room(sizeof(CellRec) * p.ncell);
    }
    HIPCHK(hipMemcpy(base, tl.data(), sizeof(RedTile) * tl.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(base + tb, stage.data(), sb, hipMemcpyHostToDevice));
    HIPCHK(hipMalloc(&d_blk_, sizeof(int) * blk.size()));
    HIPCHK(hipMemcpy(d_blk_, blk.data(), sizeof(int) * blk.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMalloc(&d_prob_, sizeof(RedProb) * prob.size()));
    HIPCHK(hipMemcpy(d_prob_, prob.data(), sizeof(RedProb) * prob.size(), hipMemcpyHostToDevice));
    // (the solves' streams do not wait for this one)
    hipLaunchKernelGGL(k_red_records, dim3(std::max(1, kRedMaxBlocks / np_), np_), dim3(kNT), 0, nullptr, d_prob_);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(nullptr));
    return true;
}

namespace {
// regions start on 256-byte boundaries
int64_t up(int64_t n) { return (n + 31) / 32 * 32; }
}  // namespace

int64_t RedCG::doubles() const
{
    return 7 * up(nD_) + 3 * up(nR_) + up(nS_) + 6 * up(nM_) + kRedParts * kRedMaxBlocks +
           up((int64_t)np_ * kRedScal);
}

RedBufs RedCG::carve(double *s) const
{
    RedBufs B;
    auto take = [&](int64_t n) { double *p = s; s += up(n); return p; };
    B.s = take(nS_);
    for (double **p : {&B.g, &B.t, &B.w, &B.u[0], &B.u[1], &B.v[0], &B.v[1]}) *p = take(nD_);
    for (double **p : {&B.r, &B.p[0], &B.p[1]}) *p = take(nR_);
    for (double **p : {&B.mu[0], &B.mu[1], &B.nu[0], &B.nu[1], &B.om, &B.ams}) *p = take(nM_);
    B.part = take(kRedParts * kRedMaxBlocks);
    B.scal = take((int64_t)np_ * kRedScal);
    return B;
}

void RedCG::start(const RedBufs &B, const double *rhs, const double *y, double tol, const double *tolv,
                  const int *active, int maxiter, hipStream_t st) const
{
    hipLaunchKernelGGL(k_red_aty, dim3(nblk_), dim3(kNT), 0, st, d_prob_, d_blk_, B, y, tol, tolv,
                       active, maxiter);
    hipLaunchKernelGGL(k_red_self, dim3(nblk_), dim3(kNT), 0, st, d_prob_, d_blk_, B, rhs, y);
    hipLaunchKernelGGL(k_red_expl, dim3(nblk_), dim3(kNT), 0, st, d_prob_, d_blk_, B, rhs, y);
}

void RedCG::iterate(const RedBufs &B, double *y, int n, hipStream_t st) const
{
    for (int k = 0; k < n; k++) {
        hipLaunchKernelGGL(full_ ? k_red_dir<true> : k_red_dir<false>, dim3(nblk_), dim3(kNT), 0, st,
                           d_prob_, d_blk_, B, k & 1);
        hipLaunchKernelGGL(k_red_res, dim3(nblk_), dim3(kNT), 0, st, d_prob_, d_blk_, B, y, k & 1);
        hipLaunchKernelGGL(full_ ? k_red_norm<true> : k_red_norm<false>, dim3(nblk_), dim3(kNT), 0, st,
                           d_prob_, d_blk_, B, k & 1);
    }
    hipLaunchKernelGGL(k_red_status, dim3(np_), dim3(kNT), 0, st, d_prob_, B);
}

void RedCG::finish(const RedBufs &B, double *y, const int *active, hipStream_t st) const
{
    hipLaunchKernelGGL(k_red_y, dim3(nblk_), dim3(kNT), 0, st, d_prob_, d_blk_, B, y, active);
}

}  // namespace v2g
