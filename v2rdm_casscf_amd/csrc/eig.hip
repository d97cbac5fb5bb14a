// eig.hip -- the per-block positive / negative split of Update_xz
// (v2rdm_solver.cc:3216-3289) on CDNA4, in FP64.
//
// For every block of the primal vector: M = sym(A^T y - c + mu x); M = V L V^T;
// x = V max(L,0)/mu V^T; z = mu x - M  (= -V min(L,0) V^T).
//
// Eigensolver: two-sided block Jacobi.  A block of dimension n is padded to
// N (a multiple of 64, zero rows / columns never couple) and cut into N/32
// column blocks.  Each round pairs the column blocks (circle method); a
// workgroup diagonalizes each 64x64 pair sub-matrix in LDS by parallel
// cyclic Jacobi, and a second kernel applies the pair rotations to A
// (tile-wise Q_P^T A_PR Q_R on FP64 MFMA) and to V.  Sweeps repeat until a
// full sweep applies no rotation above tol = 2e-14 ||M||_F (64 / N times that
// when the split must converge; blocks n <= 64: 1e-15 ||M||_F).
//
// Warm start: the eigenvectors of the previous Update_xz stay on the device;
// the next call starts from V^T M V, which is nearly diagonal once the BPSDP
// iteration settles, so most pairs need no rotation and are skipped.
// Blocks with n <= 64 are solved completely by one workgroup (no warm start).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "eig.hpp"

namespace v2g {

namespace {

constexpr int kT = 256;      // threads per workgroup
constexpr int kP = 64;       // pair sub-problem size
constexpr int kLd = 65;      // LDS row pitch (breaks bank conflicts on columns)

typedef double v4d __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void circle_pair(int m, int r, int k, int &a, int &b)
{
    // round r of the circle method on m players (m even): k = 0 pairs the
    // fixed player m-1 with r; k >= 1 pairs (r+k) and (r-k) mod (m-1)
    if (k == 0) { a = m - 1; b = r; return; }
    const int mm = m - 1;
    a = (r + k) % mm;
    b = (r - k + mm) % mm;
}

// Jacobi rotation (c, s) that annihilates apq.  t = tan(theta), the smaller
// root: the textbook t = sgn(th) / (|th| + sqrt(th^2 + 1)), th = d / e with
// d = aqq - app, e = 2 apq, multiplied through by |e|, gives
// t = sgn(d) e / (|d| + sqrt(d^2 + e^2)); c = 1 / sqrt(1 + t^2), s = t c.
// A step of the pair problems waits for this chain.  The root and the quotient are the
// hardware estimates (better than 2^-20), one third-order step and one correction by the
// residual each, which rounds as the library's do but without their scaling for the ends
// of the range (those take the library's); c is the estimate and two Newton steps.
__device__ __forceinline__ void jacobi_rotation(double app, double aqq, double apq, double &c,
                                                double &s)
{
    const double d = aqq - app, e = 2.0 * apq;
    const double h = fma(d, d, e * e);
    double t;
    if (h > 1e-280 && h < 1e280) {
        double y = __builtin_amdgcn_rsq(h);
        const double f = fma(-(h * y), y, 1.0);
        y = fma(y * f, fma(0.375, f, 0.5), y);
        const double r0 = h * y, r = fma(fma(-r0, r0, h), 0.5 * y, r0);
        const double den = fabs(d) + r, num = d >= 0.0 ? e : -e;
        double w = __builtin_amdgcn_rcp(den);
        const double g = fma(-den, w, 1.0);
        w = fma(w, fma(g, g, g), w);
        const double q = num * w;
        t = fma(fma(-den, q, num), w, q);
    } else {
        const double r = sqrt(h);
        if (r > 0.0 && r <= 1.79e308) {
            t = (d >= 0.0 ? e : -e) / (fabs(d) + r);
        } else {   // d^2 + e^2 under- or overflows: the textbook form
            const double th = d / e;
            t = (th >= 0.0 ? 1.0 : -1.0) / (fabs(th) + sqrt(fma(th, th, 1.0)));
        }
    }
    const double x = fma(t, t, 1.0), hx = 0.5 * x;
    double y = __builtin_amdgcn_rsq(x);
    y = fma(y, fma(-hx * y, y, 0.5), y);
    y = fma(y, fma(-hx * y, y, 0.5), y);
    c = y;
    s = t * y;
}

// R_P^T B R_R for one 2 x 2 block B = [b00 b01; b10 b11] with R = [c s; -s c]
// (rows by (cp, sp), columns by (cr, sr)).  Every product and sum is spelled
// out with fma(), so the rounding does not depend on how the compiler
// schedules a particular kernel: each launch shape of the eigen split makes
// the same rotations bit for bit.
__device__ __forceinline__ void rot2x2(double cp, double sp, double cr, double sr, double b00,
                                       double b01, double b10, double b11, double (&o)[4])
{
    // rows: R_P^T B
    const double u00 = fma(cp, b00, -(sp * b10)), u01 = fma(cp, b01, -(sp * b11));
    const double u10 = fma(sp, b00, cp * b10), u11 = fma(sp, b01, cp * b11);
    // columns: (R_P^T B) R_R
    o[0] = fma(cr, u00, -(sr * u01));
    o[1] = fma(sr, u00, cr * u01);
    o[2] = fma(cr, u10, -(sr * u11));
    o[3] = fma(sr, u10, cr * u11);
}

// Parallel Jacobi in one workgroup, for the pair sub-problems of the large blocks
// (k_pair_eig) and for whole small blocks (k_small).  m = 2 h indices, h slots; step r
// rotates one pair of indices a slot:
//  * cyclic order (the circle method): slot 0 holds (r, m - 1), slot k (r + k, r - k)
//    modulo m - 1; m - 1 steps visit every pair once;
//  * cross order (CROSS, m = 64): slot k holds (k, 32 + (k + r) mod 32); 32 steps rotate
//    every pair with one index in each half once and no pair inside a half.  A split's
//    sweep uses it after its first round: that round's cyclic order has already rotated
//    the pairs inside every column block (each block takes part in every round), so the
//    sweep still visits every pair, in 31 fewer dependent steps per later round.
// A step is a chain: the pair's elements -> rotation -> update of S = R^T S R and Q <- Q R
// -> the next step's elements.  What bounds a pair problem is that chain's latency (a few
// hundred workgroups of one CU each), so the next step's rotations are formed beside
// this step's update instead of after it: a lane of wave 0 owns the 2 x 2 block of S that
// holds its next pair (blocks {k - 1, k + 1} of the cyclic order, {k, k + 1} of the cross
// order), updates it first, and goes on to the rotation, the pair's new diagonal and the
// publication of (c, s) while the other threads update the other blocks.  One barrier a
// step.  24 orbitals, blocks up to 1 152: 46 -> 26 us a launch beside the tile updates (1 400 -> about 500 ns
// a step); every index is computed, not looked up, so the reads of S need not wait.
//  * S keeps its upper triangle (element (i, j) lives at (min, max)), 66 (MAXN + 2) doubles
//    a row: the accesses of a step walk diagonals and anti-diagonals, whose strides (67, 65)
//    are odd;
//  * Q lives in registers.  Cyclic order: a lane holds one column, rows of its wave; the
//    partner column is fetched by lane shuffles.  Cross order: a lane holds one row, its
//    wave the columns of a few slots, rotated in place; then the second half's columns
//    move on by one slot (a register move; one column a wave goes through LDS).
// From NT = 8 MAXN on, S lies with the first half of the waves and Q with the other: where a
// launch has a few hundred problems.  256 threads for 64 indices do the same work in fewer
// instructions, for many small problems at once (bond scans).
template <int NT, int MAXN, bool CROSS> struct JacobiShape {
    static constexpr int kH = MAXN / 2, kLd = MAXN + 2;
    static constexpr bool kSplit = NT >= 8 * MAXN;
    static constexpr int kST = kSplit ? NT / 2 : NT;                   // threads of S: the first
    static constexpr int kU = (kH * (kH - 3) / 2 + kH + kST - 1) / kST;   // blocks of S a thread
    static constexpr int kQ0 = kSplit ? NT / 2 : 0, kQT = NT - kQ0;       // threads of Q
    static constexpr int kQ = MAXN * MAXN / kQT;                       // entries of Q a thread
    static constexpr int kXw = CROSS ? kQT / 64 : 0;
    static_assert(!CROSS || MAXN == 64, "the cross order is for 64 indices");
    struct Lds {
        double2 rot[2][kH];       // (c, s) of the slots, by step parity
        int any[2];               // whether the step rotates at all
        double xch[CROSS ? 2 * kXw * 64 : 1];
    };
};

// the slot at place c of the cycle 0, 1, 3, 5, .., 4, 2 in which the cyclic order's next
// pairs join neighbours
__device__ __forceinline__ int cycle_slot(int c, int h)
{
    const int odd = h / 2;
    return c == 0 ? 0 : c <= odd ? 2 * c - 1 : 2 * (h - c);
}

// Returns whether anything was rotated.  q: see JacobiShape::kQ; on return (CROSS) lane =
// row, q[s] column s0 + s, q[kQ / 2 + s] column 32 + s0 + s, s0 = kQ / 2 times the wave of Q;
// else thread t of Q holds column t % MAXN, rows kQ (t / MAXN) ..
template <int NT, int MAXN, bool CROSS>
__device__ __forceinline__ bool jacobi(double *S, double (&q)[JacobiShape<NT, MAXN, CROSS>::kQ], int m, double tol,
                                       int maxsweeps, typename JacobiShape<NT, MAXN, CROSS>::Lds &sh)
{
    using Sh = JacobiShape<NT, MAXN, CROSS>;
    constexpr int kLd = Sh::kLd, kH = Sh::kH, kU = Sh::kU, kQ = Sh::kQ;
    const int tid = threadIdx.x, h = m / 2, mm = m - 1, nsteps = CROSS ? h : mm;
    const bool lead = tid < h;      // a lane of wave 0 that forms the rotations of slot tid
    const bool ofS = tid < Sh::kST, ofQ = tid >= Sh::kQ0;
    // the two indices of a slot at step 0, and one step on
    auto first = [&](int k) { return CROSS ? k : k == 0 ? mm : k; };
    auto second = [&](int k) { return CROSS ? kH + k : k == 0 ? 0 : mm - k; };
    auto next1 = [&](int x) { return CROSS ? x : x == mm ? mm : x + 1 == mm ? 0 : x + 1; };
    auto next2 = [&](int x) { return CROSS ? kH + ((x + 1) & (kH - 1)) : x + 1 == mm ? 0 : x + 1; };
    auto at = [](int i, int j) { return i < j ? i * kLd + j : j * kLd + i; };
    // this thread's blocks (P < R): slots and their current indices
    int P[kU], R[kU], p1[kU], p2[kU], r1[kU], r2[kU];
    bool have[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) {
        const int id = u * Sh::kST + tid - kH;
        int a, b;
        if (id < 0) {
            a = CROSS ? tid : max(tid - 1, 0);
            b = CROSS ? (tid + 1) & (kH - 1) : min(tid + 1, h - 1);
            have[u] = lead && h > 1;
        } else {
            const int delta = 2 + id / h, c = id % h, c2 = c + delta < h ? c + delta : c + delta - h;
            have[u] = ofS && (2 * delta < h || (2 * delta == h && c < delta));
            a = CROSS ? c : cycle_slot(c, h);
            b = CROSS ? c2 : cycle_slot(c2, h);
        }
        P[u] = have[u] ? min(a, b) : 0;
        R[u] = have[u] ? max(a, b) : 0;
        p1[u] = first(P[u]);
        p2[u] = second(P[u]);
        r1[u] = first(R[u]);
        r2[u] = second(R[u]);
    }
    // wave 0: the pair of slot tid
    int l1 = first(lead ? tid : 0), l2 = second(lead ? tid : 0);
    auto publish = [&](int buf, double app, double aqq, double apq) {
        bool rot = false;
        if (lead) {
            double c = 1.0, s = 0.0;
            const int p = min(l1, l2), r = max(l1, l2);
            if (fabs(apq) > tol) {
                jacobi_rotation(app, aqq, apq, c, s);
                rot = true;
                double o[4];
                rot2x2(c, s, c, s, app, apq, apq, aqq, o);
                S[p * kLd + p] = o[0];
                S[p * kLd + r] = o[2];
                S[r * kLd + r] = o[3];
            }
            sh.rot[buf][tid] = make_double2(c, s);
        }
        const unsigned long long b = __ballot(rot);
        if (tid == 0) sh.any[buf] = b != 0;
    };
    if (tid < 64) {
        const int p = min(l1, l2), r = max(l1, l2);
        publish(0, S[p * kLd + p], S[r * kLd + r], S[p * kLd + r]);
        __builtin_amdgcn_s_setprio(3);
    }
    // Q: cyclic order: this lane's column and its distance from the step number
    const int qlane = tid % MAXN, qwave = (tid - Sh::kQ0) / 64;
    int dist = qlane, partner_r = 0;    // (qlane - r) mod mm; r
    bool first_step = true, total = false;
    int buf = 0;
    __syncthreads();
    for (int sweep = 0; sweep < maxsweeps; sweep++) {
        bool swept = false;
        for (int r = 0; r < nsteps; r++) {
            const bool any = sh.any[buf] != 0, last = sweep + 1 == maxsweeps && r + 1 == nsteps;
            swept |= any;
            if (ofS && !last) {
                int n1 = 0, n2 = 0;
                double app = 0.0, aqq = 0.0, apq = 0.0;
                if (tid < 64) {
                    n1 = next1(l1);
                    n2 = next2(l2);
                    l1 = n1;
                    l2 = n2;
                    app = S[n1 * kLd + n1];
                    aqq = S[n2 * kLd + n2];
                    if (n1 > n2) { const double t = app; app = aqq; aqq = t; }
                    apq = S[at(n1, n2)];
                }
                if (any) {
                    int ad[kU][4];
                    double bv[kU][4];
                    double2 cp[kU], cr[kU];
#pragma unroll
                    for (int u = 0; u < kU; u++) {
                        cp[u] = sh.rot[buf][P[u]];
                        cr[u] = sh.rot[buf][R[u]];
                        const int pl = min(p1[u], p2[u]), ph = max(p1[u], p2[u]);
                        const int rl = min(r1[u], r2[u]), rh = max(r1[u], r2[u]);
                        ad[u][0] = at(pl, rl);
                        ad[u][1] = at(pl, rh);
                        ad[u][2] = at(ph, rl);
                        ad[u][3] = at(ph, rh);
                    }
#pragma unroll
                    for (int u = 0; u < kU; u++)
#pragma unroll
                        for (int e = 0; e < 4; e++) bv[u][e] = S[ad[u][e]];
#pragma unroll
                    for (int u = 0; u < kU; u++) {
                        if (!have[u] || (cp[u].y == 0.0 && cr[u].y == 0.0)) continue;
                        double o[4];
                        rot2x2(cp[u].x, cp[u].y, cr[u].x, cr[u].y, bv[u][0], bv[u][1], bv[u][2], bv[u][3], o);
#pragma unroll
                        for (int e = 0; e < 4; e++) S[ad[u][e]] = o[e];
                        if (u == 0 && lead) {
                            const int w = at(n1, n2);
                            apq = w == ad[u][0] ? o[0] : w == ad[u][1] ? o[1] : w == ad[u][2] ? o[2] : o[3];
                        }
                    }
                }
                if (tid < 64) publish(buf ^ 1, app, aqq, apq);
#pragma unroll
                for (int u = 0; u < kU; u++) {
                    p1[u] = next1(p1[u]);
                    p2[u] = next2(p2[u]);
                    r1[u] = next1(r1[u]);
                    r2[u] = next2(r2[u]);
                }
            }
            if (ofQ) {
                if constexpr (CROSS) {
                    constexpr int kS = kQ / 2, kW = Sh::kXw;
                    if (!first_step) q[kQ - 1] = sh.xch[((buf ^ 1) * kW + (qwave + 1) % kW) * 64 + (tid & 63)];
                    if (any) {
#pragma unroll
                        for (int s = 0; s < kS; s++) {
                            const double2 cs = sh.rot[buf][qwave * kS + s];
                            const double a = q[s], b = q[kS + s];
                            q[s] = fma(cs.x, a, -cs.y * b);
                            q[kS + s] = fma(cs.x, b, cs.y * a);
                        }
                    }
                    sh.xch[(buf * kW + qwave) * 64 + (tid & 63)] = q[kS];
#pragma unroll
                    for (int s = 0; s + 1 < kS; s++) q[kS + s] = q[kS + s + 1];
                    first_step = false;
                } else {
                    if (any && (tid - Sh::kQ0) / MAXN * kQ < m) {   // rows from m on stay zero
                        const bool in = qlane < m;
                        int pl = qlane, slot = 0;
                        if (in) {
                            pl = qlane == mm ? partner_r : dist == 0 ? mm : partner_r - dist + (partner_r < dist ? mm : 0);
                            slot = qlane == mm ? 0 : dist < h ? dist : mm - dist;
                        }
                        const double2 cs = sh.rot[buf][slot];
                        const double c = in ? cs.x : 1.0, sn = in ? (qlane < pl ? -cs.y : cs.y) : 0.0;
                        // all shuffles first, then the arithmetic: one wait for the batch
                        double o[kQ];
#pragma unroll
                        for (int i = 0; i < kQ; i++) o[i] = __shfl(q[i], pl, MAXN);
#pragma unroll
                        for (int i = 0; i < kQ; i++) q[i] = fma(c, q[i], sn * o[i]);
                    }
                    dist = dist == 0 ? mm - 1 : dist - 1;
                    partner_r = partner_r + 1 == mm ? 0 : partner_r + 1;
                }
            }
            buf ^= 1;
            __syncthreads();
        }
        total |= swept;
        if (!swept) break;
    }
    if constexpr (CROSS) {
        if (ofQ && !first_step)
            q[kQ - 1] = sh.xch[((buf ^ 1) * Sh::kXw + (qwave + 1) % Sh::kXw) * 64 + (tid & 63)];
    }
    if (tid < 64) __builtin_amdgcn_s_setprio(0);
    return total;
}

// One block (n <= 64) a workgroup.  LDS holds S alone (34 KB; Q lives in registers, M is
// formed again at the end), so four workgroups share a CU where
// S, Q and M in LDS let in one: a bond scan has a thousand such blocks at once.
template <int NT, int MAXN>
__global__ void __launch_bounds__(NT, 4)   // waves a SIMD
k_small(const EigBlock *__restrict__ blocks, const double *__restrict__ aty,
        const double *__restrict__ c, double *__restrict__ x, double *__restrict__ z, double mu0,
        EigBatch eb)
{
    using Shape = JacobiShape<NT, MAXN, false>;
    // 16-column strips of the matrix go to the first waves, kEl elements a thread
    constexpr int kLd = Shape::kLd, kWav = NT / 64, kRowB = MAXN / 16, kSw = kWav < kRowB ? kWav : kRowB;
    constexpr int kStrips = kRowB / kSw, kEl = 4 * kRowB * kStrips, kSmallRows = Shape::kQ;
    __shared__ double S[MAXN * kLd];
    __shared__ double lam[MAXN], red[kWav];
    __shared__ typename Shape::Lds sh;
    const EigBlock B = blocks[blockIdx.x];
    if (eb.active && !eb.active[B.prob]) return;
    const double mu = eb.mus ? eb.mus[B.prob] : mu0;
    const int n = B.n, m = (n + 1) & ~1;
    const int64_t o = B.xoff;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
    // this thread's elements: the layout of the MFMA results of the wave's column
    // strips (row 16 b + 4 r + lk, column 16 strip + li)
    auto row_of = [&](int e) { return 16 * (e / 4 % kRowB) + 4 * (e & 3) + lk; };
    auto col_of = [&](int e) { return 16 * (wave * kStrips + e / (4 * kRowB)) + li; };
    auto element = [&](int e) -> double {
        const int row = row_of(e), col = col_of(e);
        if (row >= n || col >= n) return 0.0;
        const int64_t ipq = o + (int64_t)row * n + col, iqp = o + (int64_t)col * n + row;
        return 0.5 * ((aty[ipq] - c[ipq] + mu * x[ipq]) + (aty[iqp] - c[iqp] + mu * x[iqp]));
    };
    double fro = 0.0;
    if (wave < kSw)
#pragma unroll
        for (int e = 0; e < kEl; e++) {
            const double v = element(e);
            S[row_of(e) * kLd + col_of(e)] = v;
            fro += v * v;
        }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) fro += __shfl_xor(fro, off, 64);
    if (lane == 0) red[wave] = fro;
    __syncthreads();
    double tot = 0.0;
    for (int i = 0; i < kWav; i++) tot += red[i];
    const double tol = 1e-15 * sqrt(tot) + 1e-300;
    const bool ofQ = (int)threadIdx.x >= Shape::kQ0;
    const int qc = threadIdx.x % MAXN, qr = ((int)threadIdx.x - Shape::kQ0) / MAXN * kSmallRows;
    double q[kSmallRows];
#pragma unroll
    for (int i = 0; i < kSmallRows; i++) q[i] = (qr + i == qc) ? 1.0 : 0.0;
    if (n > 1) jacobi<NT, MAXN, false>(S, q, m, tol, 60, sh);
    __syncthreads();
    if (threadIdx.x < MAXN) {
        const double l = S[threadIdx.x * kLd + threadIdx.x];
        lam[threadIdx.x] = threadIdx.x < m && l > 0.0 ? l / mu : 0.0;
    }
    __syncthreads();   // the diagonal has been read: S takes Q
    if (ofQ)
#pragma unroll
        for (int i = 0; i < kSmallRows; i++) S[(qr + i) * kLd + qc] = q[i];
    // M once more, before x is overwritten: the registers held through the solve would spill
    double Mv[kEl];
    if (wave < kSw)
#pragma unroll
        for (int e = 0; e < kEl; e++) Mv[e] = element(e);
    __syncthreads();
    if (wave >= kSw) return;
    // x = Q diag(lam) Q^T, one or two 16-column strips a wave
#pragma unroll
    for (int st = 0; st < kStrips; st++) {
        v4d acc[kRowB];
#pragma unroll
        for (int b = 0; b < kRowB; b++) acc[b] = v4d{0.0, 0.0, 0.0, 0.0};
        const int col = 16 * (wave * kStrips + st) + li;
        for (int k0 = 0; k0 < m; k0 += 4) {
            const int k = k0 + lk;
            const double l = lam[k], bv = S[col * kLd + k];
#pragma unroll
            for (int b = 0; b < kRowB; b++)
                if (16 * b < n)
                    acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(S[(16 * b + li) * kLd + k] * l, bv, acc[b], 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 4 * kRowB; e++) {
            const int row = 16 * (e >> 2) + 4 * (e & 3) + lk;
            if (row < n && col < n) {
                const int64_t i = o + (int64_t)row * n + col;
                const double xv = acc[e >> 2][e & 3];
                x[i] = xv;
                z[i] = mu * xv - Mv[st * 4 * kRowB + e];
            }
        }
    }
}

// ---- large blocks -----------------------------------------------------------
// M = sym(A^T y - c + mu x) into the padded N x N workspace, one 64 x 64 tile
// pair (P, R), P <= R, per workgroup: both tiles are read with coalesced rows,
// the transpose goes through LDS, and the (R, P) tile is written as the
// transpose of the (P, R) one.  Cold calls also set A = M, V = I.
__global__ void __launch_bounds__(kT)
k_build_m(const EigBlock *__restrict__ blocks, const double *__restrict__ aty,
          const double *__restrict__ c, const double *__restrict__ x, double mu0,
          double *__restrict__ Mw, double *__restrict__ Aw, double *__restrict__ Vw, int cold,
          EigBatch eb)
{
    __shared__ double S[kP * kLd];
    const EigBlock B = blocks[blockIdx.y];
    if (eb.active && !eb.active[B.prob]) return;
    const double mu = eb.mus ? eb.mus[B.prob] : mu0;
    const int nt = B.N / kP;
    int64_t rem = blockIdx.x;
    if (rem >= (int64_t)nt * (nt + 1) / 2) return;
    int P = 0;
    while (rem >= nt - P) { rem -= nt - P; P++; }
    const int R = P + (int)rem;
    const int n = B.n;
    const int j = threadIdx.x & (kP - 1), i0 = threadIdx.x / kP;
    constexpr int kU = kP * kP / kT;
    auto g = [&](int p, int q) -> double {
        if (p >= n || q >= n) return 0.0;
        const int64_t i = B.xoff + (int64_t)p * n + q;
        return aty[i] - c[i] + mu * x[i];
    };
    // (R, P) tile into LDS, (P, R) tile into registers
    double v[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) {
        const int i = i0 + u * (kT / kP);
        S[i * kLd + j] = g(R * kP + i, P * kP + j);
        v[u] = g(P * kP + i, R * kP + j);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kU; u++) {
        const int i = i0 + u * (kT / kP);
        v[u] = 0.5 * (v[u] + S[j * kLd + i]);
    }
    auto put = [&](int p, int q, double val) {
        const int64_t w = B.woff + (int64_t)p * B.N + q;
        Mw[w] = val;
        if (cold) {
            Aw[w] = val;
            Vw[w] = (p == q) ? 1.0 : 0.0;
        }
    };
#pragma unroll
    for (int u = 0; u < kU; u++) put(P * kP + i0 + u * (kT / kP), R * kP + j, v[u]);
    if (P == R) return;
    __syncthreads();   // every thread has read S
#pragma unroll
    for (int u = 0; u < kU; u++) S[(i0 + u * (kT / kP)) * kLd + j] = v[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kU; u++) {
        const int i = i0 + u * (kT / kP);
        put(R * kP + i, P * kP + j, S[j * kLd + i]);
    }
}

constexpr int kFroParts = 64;

// partial squared Frobenius norms: block y, part x
__global__ void __launch_bounds__(kT)
k_fro_part(const EigBlock *__restrict__ blocks, const double *__restrict__ Mw,
           double *__restrict__ part, EigBatch eb)
{
    __shared__ double red[kT / 64];
    const EigBlock B = blocks[blockIdx.y];
    if (eb.active && !eb.active[B.prob]) return;
    const int64_t NN = (int64_t)B.N * B.N;
    double s = 0.0;
    for (int64_t w = blockIdx.x * (int64_t)kT + threadIdx.x; w < NN; w += (int64_t)kFroParts * kT) {
        const double v = Mw[B.woff + w];
        s += v * v;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int i = 0; i < kT / 64; i++) t += red[i];
        part[blockIdx.y * kFroParts + blockIdx.x] = t;
    }
}

// rotation threshold of block b: 2e-14 ||M||_F, scaled by 64 / N for a split
// that must converge (its off-diagonal remainder then stays at the level of
// one 64-wide block's however large the block is)
__global__ void k_fro_fin(const EigBlock *__restrict__ blocks, int nblocks,
                          const double *__restrict__ part, double *__restrict__ tol, int tight)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nblocks) return;
    double t = 0.0;
    for (int i = 0; i < kFroParts; i++) t += part[b * kFroParts + i];
    const double scale = tight ? 64.0 / (double)blocks[b].N : 1.0;
    tol[b] = 2e-14 * scale * sqrt(t) + 1e-300;
}

// index of the 64 pair rows: first column block a (32 indices), then b
__device__ __forceinline__ int pair_index(int a, int b, int i)
{
    return i < 32 ? a * 32 + i : b * 32 + (i - 32);
}

// the column blocks of pair k in round r, lower block first: the rotated
// matrix A is kept as its upper triangle of 32 x 32 sub-blocks (sub-block
// (u, v) with u > v is stale; it is the transpose of (v, u)), and with a < b
// the off-diagonal sub-block of every pair problem is a stored one
__device__ __forceinline__ void ordered_pair(int m, int r, int k, int &a, int &b)
{
    circle_pair(m, r, k, a, b);
    if (a > b) { const int t = a; a = b; b = t; }
}

template <int NT, bool CROSS>
__global__ void __launch_bounds__(NT, NT == 256 ? 4 : 1)
k_pair_eig(const EigBlock *__restrict__ blocks, int round, const double *__restrict__ Aw,
           double *__restrict__ Qbuf, int *__restrict__ active, const double *__restrict__ tol,
           int *__restrict__ counter, int inner_sweeps, EigBatch eb)
{
    using Shape = JacobiShape<NT, kP, CROSS>;
    constexpr int kLd = Shape::kLd, kQ = Shape::kQ;
    __shared__ double S[kP * kLd];
    __shared__ typename Shape::Lds sh;
    __shared__ int sh_big;
    const EigBlock B = blocks[blockIdx.y];
    const int nbk = B.N / 32;
    const int k = blockIdx.x;
    if (k >= nbk / 2 || round >= nbk - 1) return;
    if (eb.active && !eb.active[B.prob]) {   // a problem left out: no rotation
        if (threadIdx.x == 0) active[B.poff + k] = 0;
        return;
    }
    int a, b;
    ordered_pair(nbk, round, k, a, b);
    const double *A = Aw + B.woff;
    const double tl = tol[blockIdx.y];
    if (threadIdx.x == 0) sh_big = 0;
    int big = 0;
    // thread (i0, j) loads rows i0, i0 + NT / kP, ... of column j, all
    // loads in flight at once
    // the upper triangle of the pair matrix is all that is used: its
    // (b, a) sub-block is stale in A and is not loaded
    const int j = threadIdx.x & (kP - 1), i0 = threadIdx.x / kP;
    {
        const int64_t colj = pair_index(a, b, j);
        double v[kP * kP / NT];
#pragma unroll
        for (int u = 0; u < kP * kP / NT; u++) {
            const int i = i0 + u * (NT / kP);
            v[u] = (i >= 32 && j < 32) ? 0.0 : A[(int64_t)pair_index(a, b, i) * B.N + colj];
        }
#pragma unroll
        for (int u = 0; u < kP * kP / NT; u++) {
            const int i = i0 + u * (NT / kP);
            S[i * kLd + j] = v[u];
            big |= (i < j && fabs(v[u]) > tl);
        }
    }
    __syncthreads();
    if (big) sh_big = 1;
    __syncthreads();
    if (!sh_big) {   // uniform; already diagonal to tolerance: identity rotation
        if (threadIdx.x == 0) active[B.poff + k] = 0;
        return;
    }
    const int lane = threadIdx.x & 63, qw = ((int)threadIdx.x - Shape::kQ0) >> 6;
    double q[kQ];
#pragma unroll
    for (int i = 0; i < kQ; i++) {
        // cross order: lane = row, entry i a column; cyclic: lane = column, entry i a row
        const int other = CROSS ? (i < kQ / 2 ? qw * (kQ / 2) + i : 32 + qw * (kQ / 2) + i - kQ / 2) : qw * kQ + i;
        q[i] = other == lane ? 1.0 : 0.0;
    }
    const bool rot = jacobi<NT, kP, CROSS>(S, q, kP, tl, inner_sweeps, sh);
    if (threadIdx.x == 0) {
        active[B.poff + k] = rot;
        if (rot) atomicAdd(counter, 1);
    }
    if (!rot) return;
    double *Qo = Qbuf + B.qoff + (int64_t)k * kP * kP;
    if (!CROSS) {
        if (qw >= 0)
#pragma unroll
            for (int i = 0; i < kQ; i++) Qo[(qw * kQ + i) * kP + lane] = q[i];
        return;
    }
    // through S, which nothing needs any more, into rows of 512 bytes
    if (qw >= 0)
#pragma unroll
        for (int i = 0; i < kQ / 2; i++) {
            S[lane * kLd + qw * (kQ / 2) + i] = q[i];
            S[lane * kLd + 32 + qw * (kQ / 2) + i] = q[kQ / 2 + i];
        }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kP * kP / NT; u++) {
        const int i = i0 + u * (NT / kP);
        Qo[i * kP + j] = S[i * kLd + j];
    }
}

// A_PR <- Q_P^T A_PR Q_R for the pair tiles with P <= R (A is symmetric and
// kept as its upper triangle of 32 x 32 sub-blocks); V[:, R] <- V[:, R] Q_R.
// Four waves per SIMD: the LDS tile allows four workgroups per CU, and the
// bound keeps the registers within that (122 VGPRs).  FP64 MFMA
// v_mfma_f64_16x16x4f64: A[i][k] from lane i + 16k, B[k][j] from lane
// j + 16k, D[i][j] in lane j + 16 (i % 4), element i / 4.
__global__ void __launch_bounds__(kT, 4)
k_apply(const EigBlock *__restrict__ blocks, int nblocks, const int64_t *__restrict__ tile_start, int round,
        double *__restrict__ Aw, double *__restrict__ Vw, const double *__restrict__ Qbuf,
        const int *__restrict__ active, EigBatch eb)
{
    // only the tile lives in LDS; the pair rotations Q_P, Q_R are read from
    // global memory (L2-resident: each one serves a row of tiles), which
    // halves the LDS footprint and doubles the workgroups per CU
    __shared__ double T[kP * kLd];
    // the tiles of all blocks in one line: a grid of the largest block's by the number of
    // blocks is three quarters empty workgroups at H50
    int lo = 0, hi = nblocks;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (tile_start[mid] <= (int64_t)blockIdx.x) lo = mid;
        else hi = mid;
    }
    const EigBlock B = blocks[lo];
    const int nbk = B.N / 32, np = nbk / 2;
    if (eb.active && !eb.active[B.prob]) return;
    const int64_t ntA = (int64_t)np * (np + 1) / 2;
    const int64_t t = (int64_t)blockIdx.x - tile_start[lo];
    const bool isA = t < ntA;
    int P = -1, R, rt = 0;
    if (isA) {
        // t -> (P, R) with P <= R, row-major over the upper triangle
        int64_t rem = t;
        P = 0;
        while (rem >= np - P) { rem -= np - P; P++; }
        R = P + (int)rem;
    } else {
        rt = (int)((t - ntA) / np);
        R = (int)((t - ntA) % np);
    }
    const bool actP = isA && active[B.poff + P];
    const bool actR = active[B.poff + R];
    if (!actP && !actR) return;
    int pa = 0, pb = 0, ra, rb;
    if (isA) ordered_pair(nbk, round, P, pa, pb);
    ordered_pair(nbk, round, R, ra, rb);
    double *M = isA ? Aw + B.woff : Vw + B.woff;
    const int j = threadIdx.x & (kP - 1), i0 = threadIdx.x / kP;
    const int64_t colj = pair_index(ra, rb, j);
    // A tiles move as four 32 x 32 sub-blocks (u, v), u in {pa, pb}, v in
    // {ra, rb}: a stored one (u <= v) directly, a stale one (u > v) as the
    // transpose of (v, u); thread t moves stored rows t / 32 + 8 k, column
    // t % 32 of each (coalesced 256-byte rows either way).  Each unordered
    // pair of column blocks belongs to one tile of the round, so every
    // stored sub-block is written once; in a diagonal tile (P == R) the
    // (pb, pa) sub-block duplicates (pa, pb) and is not written back.
    const int sr0 = threadIdx.x >> 5, sc = threadIdx.x & 31;
    auto sub_addr = [&](int ub, int vb, int k, int &ti, int &tj) -> int64_t {
        const int u = ub ? pb : pa, v = vb ? rb : ra, sr = sr0 + 8 * k;
        if (u <= v) {
            ti = ub * 32 + sr;
            tj = vb * 32 + sc;
            return (int64_t)(u * 32 + sr) * B.N + v * 32 + sc;
        }
        ti = ub * 32 + sc;
        tj = vb * 32 + sr;
        return (int64_t)(v * 32 + sr) * B.N + u * 32 + sc;
    };
    if (isA) {
        double v[16];
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int k = 0; k < 4; k++) {
                int ti, tj;
                v[s * 4 + k] = M[sub_addr(s >> 1, s & 1, k, ti, tj)];
            }
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int k = 0; k < 4; k++) {
                int ti, tj;
                (void)sub_addr(s >> 1, s & 1, k, ti, tj);
                T[ti * kLd + tj] = v[s * 4 + k];
            }
    } else {
        // V tiles: thread (i0, j) moves rows i0, i0 + 4, ... of column j, all
        // 16 loads issued before the first LDS write
        double v[kP * kP / kT];
#pragma unroll
        for (int u = 0; u < kP * kP / kT; u++)
            v[u] = M[(int64_t)(rt * kP + i0 + u * (kT / kP)) * B.N + colj];
#pragma unroll
        for (int u = 0; u < kP * kP / kT; u++) T[(i0 + u * (kT / kP)) * kLd + j] = v[u];
    }
    // The tile passes through LDS once.  Wave w forms the 64 x 16 column strip
    // w of U = T Q_R (A operand T from LDS, B operand Q_R from global memory)
    // in its MFMA accumulators: accumulator register r of row block bi holds
    // U[16 bi + 4 r + lane / 16][16 w + lane % 16], which is exactly the B
    // operand layout of the k-step 16 bi + 4 r of the next product, so the
    // strip of Q_P^T U is formed from registers.  Stored sub-blocks are then
    // written from registers (four 128-byte row pieces per store); stale
    // (transposed) ones go through LDS for coalesced writes.
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int li = lane & 15, lk = lane >> 4;
    const int jc = 16 * wave + li;
    v4d u[4];
    if (actR) {
        const double *QR = Qbuf + B.qoff + (int64_t)R * kP * kP;
#pragma unroll
        for (int bi = 0; bi < 4; bi++) u[bi] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int k0 = 0; k0 < kP; k0 += 4) {
            const double bv = QR[(k0 + lk) * kP + jc];
#pragma unroll
            for (int bi = 0; bi < 4; bi++) {
                const double av = T[(16 * bi + li) * kLd + k0 + lk];
                u[bi] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, u[bi], 0, 0, 0);
            }
        }
    } else {
#pragma unroll
        for (int bi = 0; bi < 4; bi++)
#pragma unroll
            for (int r = 0; r < 4; r++) u[bi][r] = T[(16 * bi + 4 * r + lk) * kLd + jc];
    }
    v4d o[4];
    if (actP) {
        const double *QP = Qbuf + B.qoff + (int64_t)P * kP * kP;
#pragma unroll
        for (int bi = 0; bi < 4; bi++) o[bi] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int kb = 0; kb < 4; kb++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int k = 16 * kb + 4 * r + lk;
                const double bv = u[kb][r];
#pragma unroll
                for (int bi = 0; bi < 4; bi++) {
                    const double av = QP[k * kP + 16 * bi + li];   // (Q_P^T)[row][k]
                    o[bi] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, o[bi], 0, 0, 0);
                }
            }
    } else {
#pragma unroll
        for (int bi = 0; bi < 4; bi++) o[bi] = u[bi];
    }
    if (!isA) {
        const int64_t col = pair_index(ra, rb, jc);
#pragma unroll
        for (int bi = 0; bi < 4; bi++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                M[(int64_t)(rt * kP + 16 * bi + 4 * r + lk) * B.N + col] = o[bi][r];
        return;
    }
    __syncthreads();   // every wave has read T
    const int vb = wave >> 1, vv = vb ? rb : ra;
#pragma unroll
    for (int ub = 0; ub < 2; ub++) {
        const int uu = ub ? pb : pa;
        if (P == R && ub == 1 && vb == 0) continue;   // (pb, pa) of a diagonal tile
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int bi = 2 * ub + h;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = 16 * bi + 4 * r + lk;
                if (uu <= vv)
                    M[(int64_t)(uu * 32 + i - 32 * ub) * B.N + vv * 32 + jc - 32 * vb] = o[bi][r];
                else
                    T[i * kLd + jc] = o[bi][r];
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int ub = s >> 1, vb2 = s & 1;
        const int uu = ub ? pb : pa, v2 = vb2 ? rb : ra;
        if (uu <= v2 || (P == R && s == 2)) continue;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int sr = sr0 + 8 * k;
            M[(int64_t)(v2 * 32 + sr) * B.N + uu * 32 + sc] = T[(ub * 32 + sc) * kLd + vb2 * 32 + sr];
        }
    }
}
// The columns of V that x is made of, lambda_j = A[j][j] > 0: their indices in order (cols),
// sqrt(lambda_j / mu) (scale, 0 for the padding) and how many, rounded up to the depth of a
// GEMM panel (count).  About half of a block's eigenvalues are positive, so the
// reconstruction has half the work.
__global__ void __launch_bounds__(kT)
k_positive(const EigBlock *__restrict__ blocks, const double *__restrict__ Aw, int *__restrict__ cols,
           double *__restrict__ scale, int *__restrict__ count, double mu0, EigBatch eb)
{
    __shared__ int wcnt[kT / 64];
    const EigBlock B = blocks[blockIdx.x];
    if (eb.active && !eb.active[B.prob]) return;
    const double mu = eb.mus ? eb.mus[B.prob] : mu0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int done = 0;
    for (int j0 = 0; j0 < B.N; j0 += kT) {
        const int j = j0 + threadIdx.x;
        const double l = j < B.N ? Aw[B.woff + (int64_t)j * (B.N + 1)] : 0.0;
        const unsigned long long b = __ballot(l > 0.0);
        if (lane == 0) wcnt[wave] = __popcll(b);
        __syncthreads();
        int pos = done + __popcll(b & ((1ull << lane) - 1));
        for (int w = 0; w < kT / 64; w++) {
            if (w < wave) pos += wcnt[w];
            done += wcnt[w];
        }
        if (l > 0.0) {
            cols[B.coff + pos] = j;
            scale[B.coff + pos] = sqrt(l / mu);
        }
        __syncthreads();
    }
    const int padded = (done + kGemmK - 1) / kGemmK * kGemmK;
    if (done + (int)threadIdx.x < padded) {
        cols[B.coff + done + threadIdx.x] = 0;
        scale[B.coff + done + threadIdx.x] = 0.0;
    }
    if (threadIdx.x == 0) count[blockIdx.x] = padded;
}

constexpr int kScaleRows = 8;

// T[:, i] = V[:, cols[i]] scale[i], i < count; kScaleRows rows a workgroup.  H50: 332 us
// with all columns, the diagonal read again for every entry; below 60 now.
__global__ void __launch_bounds__(kT)
k_scale_vecs(const EigBlock *__restrict__ blocks, const double *__restrict__ Vw, const int *__restrict__ cols,
             const double *__restrict__ scale, const int *__restrict__ count, double *__restrict__ Tw, EigBatch eb)
{
    const EigBlock B = blocks[blockIdx.y];
    const int row0 = blockIdx.x * kScaleRows;
    if (row0 >= B.N || (eb.active && !eb.active[B.prob])) return;
    const double *V = Vw + B.woff + (int64_t)row0 * B.N;
    double *T = Tw + B.woff + (int64_t)row0 * B.N;
    for (int i = threadIdx.x; i < count[blockIdx.y]; i += kT) {
        const int j = cols[B.coff + i];
        const double s = scale[B.coff + i];
        double v[kScaleRows];
#pragma unroll
        for (int r = 0; r < kScaleRows; r++) v[r] = V[(int64_t)r * B.N + j];
#pragma unroll
        for (int r = 0; r < kScaleRows; r++) T[(int64_t)r * B.N + i] = s > 0.0 ? v[r] * s : 0.0;
    }
}

__global__ void __launch_bounds__(kT)
k_z(const EigBlock *__restrict__ blocks, const double *__restrict__ x,
    const double *__restrict__ Mw, double *__restrict__ z, double mu0, EigBatch eb)
{
    const EigBlock B = blocks[blockIdx.y];
    if (eb.active && !eb.active[B.prob]) return;
    const double mu = eb.mus ? eb.mus[B.prob] : mu0;
    const int n = B.n;
    const int64_t nn = (int64_t)n * n;
    for (int64_t w = blockIdx.x * (int64_t)kT + threadIdx.x; w < nn; w += (int64_t)gridDim.x * kT) {
        const int p = (int)(w / n), q = (int)(w % n);
        z[B.xoff + w] = mu * x[B.xoff + w] - Mw[B.woff + (int64_t)p * B.N + q];
    }
}

}  // namespace

namespace {
// Blocks of 33 to 64 take 1024 threads each up to this many in a launch, 256 beyond.  One
// workgroup of 1024 fits a CU (80 registers a thread), four of 256 do.  Up to 256 blocks, one
// a CU, a launch waits for one block's latency: blocks of 50 indices 365 us against 565 with
// 256 threads, of 64 513 against 731.  Above 512 the throughput counts, which 256 threads
// have: 520 blocks of 50 1052 against 837 us, 550 of 64 1528 against 1213.  Between them it
// depends on the sizes: the 400 or so of 64 chains, 33 to 64 mixed and the largest first, 715
// against 786 us, but 400 equal blocks of 50 726 against 622, 350 of 64 1024 against 920.
// Blocks up to 32 take 256 threads at any count (128 chains: 201 against 328 us with a
// wavefront each).
constexpr int kFewMid = 512;
}

int eig_order_small(std::vector<EigBlock> &small)
{
    std::stable_sort(small.begin(), small.end(), [](const EigBlock &a, const EigBlock &b) {
        const bool ta = a.n <= kTinyN, tb = b.n <= kTinyN;
        return ta != tb ? ta : a.n > b.n;
    });
    int n = 0;
    for (const auto &b : small) n += b.n <= kTinyN;
    return n;
}

void eig_small(const EigBlock *blocks, int nblocks, int ntiny, const double *aty, const double *c, double *x,
               double *z, double mu, hipStream_t st, EigBatch eb)
{
    const int nmid = nblocks - ntiny;
    if (ntiny > 0)
        hipLaunchKernelGGL((k_small<256, 32>), dim3(ntiny), dim3(256), 0, st, blocks, aty, c, x, z, mu, eb);
    if (nmid > 0)
        hipLaunchKernelGGL((nmid <= kFewMid ? k_small<1024, 64> : k_small<256, 64>), dim3(nmid),
                           dim3(nmid <= kFewMid ? 1024 : 256), 0, st, blocks + ntiny, aty, c, x, z, mu, eb);
}

void eig_build_m(const EigBlock *blocks, int nblocks, int max_N, const double *aty, const double *c,
                 const double *x, double mu, double *Mw, double *Aw, double *Vw, int cold,
                 hipStream_t st, EigBatch eb)
{
    const int nt = max_N / kP;
    hipLaunchKernelGGL(k_build_m, dim3(nt * (nt + 1) / 2, nblocks), dim3(kT), 0, st, blocks, aty, c,
                       x, mu, Mw, Aw, Vw, cold, eb);
}

void eig_tol(const EigBlock *blocks, int nblocks, const double *Mw, double *tol, double *part,
             int tight, hipStream_t st, EigBatch eb)
{
    hipLaunchKernelGGL(k_fro_part, dim3(kFroParts, nblocks), dim3(kT), 0, st, blocks, Mw, part, eb);
    hipLaunchKernelGGL(k_fro_fin, dim3((nblocks + 63) / 64), dim3(64), 0, st, blocks, nblocks, part,
                       tol, tight);
}

void eig_pairs(const EigBlock *blocks, int nblocks, int maxpairs, int round, const double *Aw,
               double *Qbuf, int *active, const double *tol, int *counter, int inner_sweeps,
               int wide, int bip, hipStream_t st, EigBatch eb)
{
    auto *k = wide ? (bip ? k_pair_eig<1024, true> : k_pair_eig<1024, false>)
                   : (bip ? k_pair_eig<256, true> : k_pair_eig<256, false>);
    hipLaunchKernelGGL(k, dim3(maxpairs, nblocks), dim3(wide ? 1024 : 256), 0, st, blocks, round, Aw, Qbuf,
                       active, tol, counter, inner_sweeps, eb);
}

void eig_apply(const EigBlock *blocks, int nblocks, const int64_t *tile_start, int64_t ntiles, int round,
               double *Aw, double *Vw, const double *Qbuf, const int *active, hipStream_t st, EigBatch eb)
{
    hipLaunchKernelGGL(k_apply, dim3((unsigned)ntiles), dim3(kT), 0, st, blocks, nblocks, tile_start, round, Aw,
                       Vw, Qbuf, active, eb);
}

void eig_scale(const EigBlock *blocks, int nblocks, int max_N, const double *Aw, const double *Vw, double *Tw,
               int *cols, double *scale, int *count, double mu, hipStream_t st, EigBatch eb)
{
    hipLaunchKernelGGL(k_positive, dim3(nblocks), dim3(kT), 0, st, blocks, Aw, cols, scale, count, mu, eb);
    hipLaunchKernelGGL(k_scale_vecs, dim3(max_N / kScaleRows, nblocks), dim3(kT), 0, st, blocks, Vw, cols, scale,
                       count, Tw, eb);
}

void eig_z(const EigBlock *blocks, int nblocks, const double *x, const double *Mw, double *z,
           double mu, hipStream_t st, EigBatch eb)
{
    hipLaunchKernelGGL(k_z, dim3(256, nblocks), dim3(kT), 0, st, blocks, x, Mw, z, mu, eb);
}

}  // namespace v2g
