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
//   direction   beta from the last norms; v, nu, p; t = A^T p on the D entries
//   residual    alpha from ||A^T p||^2; u, w, mu, om; explicit rows of r and y
//   norms       one read of s: r.r, r.p and p.p of the self rows
// ||p_self||^2 of the next direction follows from the three norms (p' = r + beta p).
//
// What bounds it: the norm pass reads s once (212 MB at (50e,50o)); the D2 vectors
// are read through L2 and the memory-side cache.  Every workgroup re-sums the
// partials of the pass before (at most kRedMaxBlocks of them, in one order), so
// alpha and beta are the same bits everywhere without a grid barrier or a launch
// of their own.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <stdexcept>

#include "common.hpp"
#include "redcg.hpp"

namespace v2g {

namespace {

using namespace rows;

constexpr int kNT = 512;                 // threads per workgroup
constexpr int kWaves = kNT / 64;
// workgroups of one launch: four per CU
constexpr int kRedMaxBlocks = 1024;
constexpr int kXcds = 8;

enum : int { P_TT = 0, P_RR1, P_RR2, P_RP, P_PP };

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
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

__device__ __forceinline__ int find_segment(const int64_t *__restrict__ t0, int nseg, int64_t b)
{
    int lo = 0, hi = nseg;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (t0[mid] <= b) lo = mid;
        else hi = mid;
    }
    return lo;
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
template <class F>
__device__ __forceinline__ void for_tiles(const Place &pl, int k, F fn)
{
    const int nseg = pl.pr->nseg[k];
    const int64_t *t0 = pl.pr->tile0[k];
    const int64_t nt = t0[nseg];
    for (int64_t t = pl.lb; t < nt; t += pl.nb) {
        const int si = find_segment(t0, nseg, t);
        const Segment sg = pl.pr->seg[k][si];
        const int64_t l = t - t0[si];
        if (sg.wave == 0) {
            const int64_t i = l * kNT + threadIdx.x;
            if (i < sg.count) fn(sg, i, 0);
        } else if (sg.wave == 1) {
            const int64_t i = l * kWaves + (threadIdx.x >> 6);
            if (i < sg.count) fn(sg, i, (int)(threadIdx.x & 63));
        } else {
            fn(sg, l, (int)threadIdx.x);
        }
    }
}

// the vectors of one problem
struct View {
    double *g, *u, *w, *v0, *v1, *t, *r, *p0, *p1, *s, *mu, *nu0, *nu1, *om, *ams, *scal;
};

__device__ __forceinline__ View view(const RedBufs &B, const RedProb &p, int prob, int par)
{
    // v0 / p0 / nu0: the direction before this iteration, v1 / p1 / nu1: its own
    return {B.g + p.oD, B.u + p.oD, B.w + p.oD, B.v[par ^ 1] + p.oD, B.v[par] + p.oD, B.t + p.oD,
            B.r + p.oR, B.p[par ^ 1] + p.oR, B.p[par] + p.oR, B.s + p.oS, B.mu + p.oM,
            B.nu[par ^ 1] + p.oM, B.nu[par] + p.oM, B.om + p.oM, B.ams + p.oM,
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

struct Ptr {
    const double *__restrict__ a;
    __device__ __forceinline__ double operator[](int64_t i) const { return a[i]; }
};

struct GatherD {
    const double *__restrict__ x;
    double acc;
    __device__ __forceinline__ void operator()(int64_t col, double c) { acc += c * x[col]; }
};

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

// ---- start of a solve -------------------------------------------------------

// t = (A^T y)_D from the full rows, u = w = v = 0 and the scalars
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
    const DevLayout &Lo = *pl.pr->full;
    for_tiles(pl, 0, [&](const Segment &sg, int64_t i, int lane) {
        if (sg.kind == XS_D1) {
            const double a = wave_sum(atu_d1_wave(Lo, sg, i, lane, y));
            if (lane == 0) {
                V.t[sg.start + i] = a;
                V.u[sg.start + i] = V.w[sg.start + i] = V.v0[sg.start + i] = 0.0;
            }
        } else if (sg.kind == XS_D2AB || sg.kind == XS_D2AA) {
            V.t[sg.start + i] = sg.kind == XS_D2AB ? atu_d2ab(Lo, sg, i, y) : atu_d2aa(Lo, sg, i, y);
            V.u[sg.start + i] = V.w[sg.start + i] = V.v0[sg.start + i] = 0.0;
        } else if (sg.kind == RK_ROWS) {
            V.p0[i] = 0.0;
        } else if (sg.kind == RK_MVEC) {
            V.mu[i] = V.om[i] = V.nu0[i] = 0.0;
        }
    });
    if (pl.lb == 0 && threadIdx.x == 0) {
        double *a = V.scal + RS_A + 6;      // as left by an iteration of parity 1
        a[0] = 0.0;                         // done
        a[1] = 1.0;                         // r.z (the first beta is 0)
        a[2] = 0.0;                         // d
        a[3] = 0.0;
        a[4] = 0.0;                         // iterations begun
        double *b = V.scal + RS_B + 3;
        b[0] = 1.0;                         // c
        b[1] = 0.0;                         // e
        b[2] = 0.0;
        V.scal[RS_DONE] = 0.0;
        V.scal[RS_NRM] = 0.0;
        V.scal[RS_ITER] = 0.0;
        V.scal[RS_TOL] = tolv ? tolv[pl.prob] : tol;
        V.scal[RS_MAXIT] = (double)maxiter;
    }
}

// visits the self rows of one D entry: fn(slot, full row, D2 / D1 part of x minus the
// maximal-spin part of m)
template <class X, class M, class F>
__device__ __forceinline__ void self_slots(const RedLayout &R, const DevLayout &Lo, const Segment &sg,
                                           int64_t i, const X &x, const M &m, F fn)
{
    if (sg.kind == XS_D2AB) {
        const AbEntry a = ab_entry(R.L, sg.h, i);
        auto one = [&](int f, double o) { fn(R.soff[f][sg.h] + i, self_row_ab(Lo, f, a), o); };
        const SelfAb<X> o(R, a, x);
        if (R.L.q2) one(SF_Q2AB, o.q2);
        if (R.L.g2) {
            one(SF_G2AB, o.g1);
            one(SF_G2BA, o.g2 - ms_part(R, a.p, a.q, a.r, a.s, m));
            one(SF_G2X, o.x);
            one(SF_G2Y, o.x);
            one(SF_G2A, o.ga);
            one(SF_G2B, o.gb);
        }
        if (R.nblk_d) {
            const D200Ab<X> d(R, a, x);
            for (int k = 0; k < R.nblk_d; k++) one(SF_D0 + k, d.row(R, a, k));
        }
    } else if (sg.kind == XS_D2AA) {
        if (R.L.q2)
            fn(R.soff[sg.sub ? SF_Q2BB : SF_Q2AA][sg.h] + i, Lo.rowoff[RF_Q2AA][sg.sub][sg.h] + i,
               self_row_aa(R, sg.sub, sg.h, i, x));
    } else {
        fn(R.soff[sg.sub ? SF_Q1B : SF_Q1A][sg.h] + i, self_row_d1(Lo, sg.sub, sg.h, i), x[sg.start + i]);
    }
}

// s = rhs - y - B2 t + P y_ms on the self rows, and the sum of its squares
__global__ void __launch_bounds__(kNT, 4)
k_red_self(const RedProb *__restrict__ prob, const int *__restrict__ blk, RedBufs B,
           const double *__restrict__ rhs, const double *__restrict__ y)
{
    __shared__ double sh[kWaves];
    const Place pl = place(prob, blk);
    const View V = view(B, *pl.pr, pl.prob, 0);
    if (V.scal[RS_DONE] != 0.0) return;
    const RedLayout &R = pl.pr->R;
    const DevLayout &Lo = *pl.pr->full;
    const Ptr t{V.t}, ms{y + (R.nM ? Lo.rowoff[RF_MAXSPIN][0][0] : 0)};
    double ss[1] = {0.0};
    for_tiles(pl, 2, [&](const Segment &sg, int64_t i, int) {
        self_slots(R, Lo, sg, i, t, ms, [&](int64_t slot, int64_t row, double o) {
            const double v = rhs[row] - y[row] - o;
            V.s[slot] = v;
            ss[0] += v * v;
        });
    });
    block_sums<1>(ss, sh);
    if (threadIdx.x == 0) *part(B, P_RR2, pl.gb) = ss[0];
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
    const Ptr s{V.s}, ms{y + (R.nM ? Lo.rowoff[RF_MAXSPIN][0][0] : 0)};
    double rr[1] = {0.0};
    for_tiles(pl, 0, [&](const Segment &sg, int64_t i, int lane) {
        if (sg.kind == XS_D2AB) {
            V.g[sg.start + i] = self_at_ab(R, ab_entry(R.L, sg.h, i), s);
        } else if (sg.kind == XS_D2AA) {
            V.g[sg.start + i] = self_at_aa(R, sg.sub, sg.h, i, s);
        } else if (sg.kind == XS_D1) {
            const double a = wave_sum(self_at_d1(R, sg.sub, sg.h, i, lane, s));
            if (lane == 0) V.g[sg.start + i] = a;
        } else if (sg.kind == RK_MS) {
            // sum_i of A^T y over the row's G2ba entries: P^T P y_ms - P^T y_self
            const int pr = R.L.bab[R.L.bab_off[0] + i], k = P0(pr), l = P1(pr);
            double v = ms_row_gram(R, sg.sub, (int)i, lane, ms);
            for (int j = lane; j < R.L.amo; j += 64) {
                AbEntry a{};
                a.q = sg.sub ? j : k;
                a.r = sg.sub ? j : l;
                a.s = sg.sub ? k : j;
                a.p = sg.sub ? l : j;
                v -= y[self_row_ab(Lo, SF_G2BA, a)];
            }
            v = wave_sum(v);
            if (lane == 0) {
                const double ri = rhs[Lo.rowoff[RF_MAXSPIN][sg.sub][0] + i] - v;
                V.r[sg.start + i] = ri;
                rr[0] += ri * ri;
            }
        }
    });
    for_tiles(pl, 1, [&](const Segment &sg, int64_t i, int lane) {
        if (sg.kind >= RK_ROWS || sg.kind == RF_MAXSPIN) return;
        GatherD f{V.t, 0.0};
        if (sg.wave == 0) {
            elem_terms(R.L, sg, i, f);
        } else if (sg.wave == 1) {
            wave_terms(R.L, sg, i, lane, f);
            f.acc = wave_sum(f.acc);
        } else {
            wave_terms(R.L, sg, i, lane, f, kNT);
            double a[1] = {f.acc};
            block_sums<1>(a, sh);
            f.acc = a[0];
        }
        if (sg.wave == 0 || lane == 0) {
            const double ri = rhs[sg.aux + i] - f.acc;
            V.r[sg.start + i] = ri;
            rr[0] += ri * ri;
        }
    });
    block_sums<1>(rr, sh);
    if (threadIdx.x == 0) {
        *part(B, P_RR1, pl.gb) = rr[0];
        *part(B, P_RP, pl.gb) = 0.0;
        *part(B, P_PP, pl.gb) = 0.0;
    }
}

// ---- one iteration ----------------------------------------------------------

// direction: beta and the stopping rule; v, nu, p; t = A^T p on the D entries, the
// maximal-spin rows of A A^T p, and the sum of t.t and their cross terms
__global__ void __launch_bounds__(kNT, 4)
k_red_dir(const RedProb *__restrict__ prob, const int *__restrict__ blk, RedBufs B, int par)
{
    __shared__ double sh[4 * kWaves];
    const Place pl = place(prob, blk);
    const View V = view(B, *pl.pr, pl.prob, par);
    double *a1 = V.scal + RS_A + 6 * par;
    const double *a0 = V.scal + RS_A + 6 * (par ^ 1), *b0 = V.scal + RS_B + 3 * (par ^ 1);
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
    const Axpy v{V.u, V.v0, ev.beta}, p{V.r, V.p0, ev.beta}, nu{V.mu, V.nu0, ev.beta};
    double tt[1] = {0.0};
    for_tiles(pl, 0, [&](const Segment &sg, int64_t i, int lane) {
        if (sg.kind == XS_D2AB) {
            const int64_t k = sg.start + i;
            const double t = fma(d, V.g[k], atu_d2ab<false, true>(R.L, sg, i, p)) +
                             gram_ab(R, ab_entry(R.L, sg.h, i), v, nu);
            V.t[k] = t;
            V.v1[k] = v[k];
            tt[0] += t * t;
        } else if (sg.kind == XS_D2AA) {
            const int64_t k = sg.start + i;
            const double t = fma(d, V.g[k], atu_d2aa<false, true>(R.L, sg, i, p)) +
                             gram_aa(R, sg.sub, sg.h, i, v);
            V.t[k] = t;
            V.v1[k] = v[k];
            tt[0] += t * t;
        } else if (sg.kind == XS_D1) {
            const int64_t k = sg.start + i;
            const double t = wave_sum(atu_d1_wave<false, true>(R.L, sg, i, lane, p) +
                                      gram_d1(R, sg.sub, sg.h, i, lane, v, nu)) + d * V.g[k];
            if (lane == 0) {
                V.t[k] = t;
                V.v1[k] = v[k];
                tt[0] += t * t;
            }
        } else if (sg.kind == RK_ROWS) {
            V.p1[i] = p[i];
        } else if (sg.kind == RK_MVEC) {
            V.nu1[i] = nu[i];
        } else {
            // maximal-spin row: (A A^T p) = P^T P p_ms - P^T p_self, and its share
            // of ||A^T p||^2 beyond ||p_self||^2
            const Axpy ps{V.r + R.L.rowoff[RF_MAXSPIN][0][0], V.p0 + R.L.rowoff[RF_MAXSPIN][0][0], ev.beta};
            const double self = wave_sum(ms_row_self(R, sg.sub, (int)i, lane, d, Ptr{V.s}, v, nu));
            const double gr = wave_sum(ms_row_gram(R, sg.sub, (int)i, lane, ps));
            if (lane == 0) {
                const int64_t k = sg.sub * (R.nM / 2) + i;
                V.ams[k] = gr - self;
                tt[0] += ps[k] * (gr - 2.0 * self);
            }
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
    const double *a = V.scal + RS_A + 6 * par, *b0 = V.scal + RS_B + 3 * (par ^ 1);
    double *b1 = V.scal + RS_B + 3 * par;
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
        b1[2] = alpha;
    }
    const RedLayout &R = pl.pr->R;
    double rr[1] = {0.0};
    for_tiles(pl, 1, [&](const Segment &sg, int64_t i, int lane) {
        if (sg.kind == RK_DVEC) {
            const double vi = V.v1[i];
            V.u[i] = fma(-alpha, vi + V.t[i], V.u[i]);
            V.w[i] = fma(alpha, vi, V.w[i]);
            return;
        }
        if (sg.kind == RK_MVEC) {
            const double vi = V.nu1[i];
            V.mu[i] = fma(-alpha, vi + V.p1[R.L.rowoff[RF_MAXSPIN][0][0] + i], V.mu[i]);
            V.om[i] = fma(alpha, vi, V.om[i]);
            return;
        }
        double at;
        if (sg.kind == RF_MAXSPIN) {
            at = V.ams[sg.sub * (R.nM / 2) + i];
        } else {
            GatherD f{V.t, 0.0};
            if (sg.wave == 0) {
                elem_terms(R.L, sg, i, f);
                at = f.acc;
            } else if (sg.wave == 1) {
                wave_terms(R.L, sg, i, lane, f);
                at = wave_sum(f.acc);
            } else {
                wave_terms(R.L, sg, i, lane, f, kNT);
                double s[1] = {f.acc};
                block_sums<1>(s, sh);
                at = s[0];
            }
        }
        if (sg.wave == 0 || lane == 0) {
            const int64_t k = sg.start + i;
            y[sg.aux + i] = fma(alpha, V.p1[k], y[sg.aux + i]);
            const double rn = fma(-alpha, at, V.r[k]);
            V.r[k] = rn;
            rr[0] = fma(rn, rn, rr[0]);
        }
    });
    block_sums<1>(rr, sh);
    if (threadIdx.x == 0) *part(B, P_RR1, pl.gb) = rr[0];
}

// norms: r.r, r.p, p.p of the self rows, r of this iteration and p its direction
__global__ void __launch_bounds__(kNT, 4)
k_red_norm(const RedProb *__restrict__ prob, const int *__restrict__ blk, RedBufs B, int par)
{
    __shared__ double sh[3 * kWaves];
    const Place pl = place(prob, blk);
    const View V = view(B, *pl.pr, pl.prob, par);
    if (V.scal[RS_A + 6 * par] != 0.0) return;
    const double c = V.scal[RS_B + 3 * par], d = V.scal[RS_A + 6 * par + 2];
    const RedLayout &R = pl.pr->R;
    const Ptr u{V.u}, v{V.v1}, mu{V.mu}, nu{V.nu1};
    double n[3] = {0.0, 0.0, 0.0};
    auto add = [&](double s, double ru, double pv) {
        const double r = fma(c, s, ru), p = fma(d, s, pv);
        n[0] = fma(r, r, n[0]);
        n[1] = fma(r, p, n[1]);
        n[2] = fma(p, p, n[2]);
    };
    for_tiles(pl, 2, [&](const Segment &sg, int64_t i, int) {
        if (sg.kind == XS_D2AB) {
            const AbEntry a = ab_entry(R.L, sg.h, i);
            SelfAb<Ptr> su(R, a, u), sv(R, a, v);
            const double *s = V.s + i;
            auto one = [&](int f, double ru, double pv) { add(s[R.soff[f][sg.h]], ru, pv); };
            if (R.L.q2) one(SF_Q2AB, su.q2, sv.q2);
            if (R.L.g2) {
                one(SF_G2AB, su.g1, sv.g1);
                one(SF_G2BA, su.g2 - ms_part(R, a.p, a.q, a.r, a.s, mu),
                    sv.g2 - ms_part(R, a.p, a.q, a.r, a.s, nu));
                one(SF_G2X, su.x, sv.x);
                one(SF_G2Y, su.x, sv.x);
                one(SF_G2A, su.ga, sv.ga);
                one(SF_G2B, su.gb, sv.gb);
            }
            if (R.nblk_d) {
                const D200Ab<Ptr> du(R, a, u), dv(R, a, v);
                for (int k = 0; k < R.nblk_d; k++) one(SF_D0 + k, du.row(R, a, k), dv.row(R, a, k));
            }
        } else if (sg.kind == XS_D2AA) {
            if (R.L.q2)
                add(V.s[R.soff[sg.sub ? SF_Q2BB : SF_Q2AA][sg.h] + i],
                    self_row_aa(R, sg.sub, sg.h, i, u), self_row_aa(R, sg.sub, sg.h, i, v));
        } else {
            add(V.s[R.soff[sg.sub ? SF_Q1B : SF_Q1A][sg.h] + i], u[sg.start + i], v[sg.start + i]);
        }
    });
    block_sums<3>(n, sh);
    if (threadIdx.x == 0) {
        *part(B, P_RR2, pl.gb) = n[0];
        *part(B, P_RP, pl.gb) = n[1];
        *part(B, P_PP, pl.gb) = n[2];
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
    const double e = V.scal[RS_B + 3 + 1];
    const RedLayout &R = pl.pr->R;
    const DevLayout &Lo = *pl.pr->full;
    const Ptr w{V.w}, om{V.om};
    for_tiles(pl, 2, [&](const Segment &sg, int64_t i, int) {
        self_slots(R, Lo, sg, i, w, om, [&](int64_t slot, int64_t row, double o) {
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
        if (!make_red_layout(*L[q], dev[q], p.R, work[q])) return false;
        p.full = d_dev + q;
        p.oD = nD_;
        p.oR = nR_;
        p.oS = nS_;
        p.oM = nM_;
        nD_ += p.R.nD;
        nR_ += p.R.nR;
        nS_ += p.R.nS;
        nM_ += p.R.nM;
    }
    // segments and tile prefixes of every problem's three lists, in one array each
    std::vector<Segment> segs;
    std::vector<int64_t> t0;
    std::vector<size_t> so(3 * np_), to(3 * np_);
    for (int q = 0; q < np_; q++) {
        tiles[q] = 1;
        for (int k = 0; k < 3; k++) {
            const auto &v = k == 0 ? work[q].p : k == 1 ? work[q].r : work[q].n;
            so[3 * q + k] = segs.size();
            to[3 * q + k] = t0.size();
            prob[q].nseg[k] = (int)v.size();
            int64_t t = 0;
            for (const Segment &s : v) {
                t0.push_back(t);
                const int64_t per = s.wave == 0 ? kNT : s.wave == 1 ? kWaves : 1;
                t += (s.count + per - 1) / per;
                segs.push_back(s);
            }
            t0.push_back(t);
            tiles[q] = std::max(tiles[q], t);
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
    const size_t sb = sizeof(Segment) * segs.size(), tb = sizeof(int64_t) * t0.size();
    HIPCHK(hipMalloc(&d_work_, sb + tb));
    const Segment *ds = static_cast<const Segment *>(d_work_);
    const int64_t *dt = reinterpret_cast<const int64_t *>(static_cast<char *>(d_work_) + sb);
    HIPCHK(hipMemcpy(d_work_, segs.data(), sb, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(static_cast<char *>(d_work_) + sb, t0.data(), tb, hipMemcpyHostToDevice));
    for (int q = 0; q < np_; q++)
        for (int k = 0; k < 3; k++) {
            prob[q].seg[k] = ds + so[3 * q + k];
            prob[q].tile0[k] = dt + to[3 * q + k];
        }
    HIPCHK(hipMalloc(&d_blk_, sizeof(int) * blk.size()));
    HIPCHK(hipMemcpy(d_blk_, blk.data(), sizeof(int) * blk.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMalloc(&d_prob_, sizeof(RedProb) * prob.size()));
    HIPCHK(hipMemcpy(d_prob_, prob.data(), sizeof(RedProb) * prob.size(), hipMemcpyHostToDevice));
    return true;
}

namespace {
// regions start on 256-byte boundaries
int64_t up(int64_t n) { return (n + 31) / 32 * 32; }
}  // namespace

int64_t RedCG::doubles() const
{
    return 6 * up(nD_) + 3 * up(nR_) + up(nS_) + 5 * up(nM_) + kRedParts * kRedMaxBlocks +
           up((int64_t)np_ * kRedScal);
}

RedBufs RedCG::carve(double *s) const
{
    RedBufs B;
    auto take = [&](int64_t n) { double *p = s; s += up(n); return p; };
    B.s = take(nS_);
    for (double **p : {&B.g, &B.u, &B.w, &B.v[0], &B.v[1], &B.t}) *p = take(nD_);
    for (double **p : {&B.r, &B.p[0], &B.p[1]}) *p = take(nR_);
    for (double **p : {&B.mu, &B.nu[0], &B.nu[1], &B.om, &B.ams}) *p = take(nM_);
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
        hipLaunchKernelGGL(k_red_dir, dim3(nblk_), dim3(kNT), 0, st, d_prob_, d_blk_, B, k & 1);
        hipLaunchKernelGGL(k_red_res, dim3(nblk_), dim3(kNT), 0, st, d_prob_, d_blk_, B, y, k & 1);
        hipLaunchKernelGGL(k_red_norm, dim3(nblk_), dim3(kNT), 0, st, d_prob_, d_blk_, B, k & 1);
    }
    hipLaunchKernelGGL(k_red_status, dim3(np_), dim3(kNT), 0, st, d_prob_, B);
}

void RedCG::finish(const RedBufs &B, double *y, const int *active, hipStream_t st) const
{
    hipLaunchKernelGGL(k_red_y, dim3(nblk_), dim3(kNT), 0, st, d_prob_, d_blk_, B, y, active);
}

}  // namespace v2g
