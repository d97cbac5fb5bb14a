// t2maps.hip -- A.x and A^T.y of the T2 rows, a wavefront a unit (t2rows.hpp).
#include "t2maps.hpp"

#include <algorithm>

namespace v2g {

namespace {

using namespace rows;

constexpr int kBlock = 256, kWaves = kBlock / 64, kPer = kT2Chunk / 64;

__device__ __forceinline__ void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

struct AddTo {
    double *acc;
    const double *__restrict__ x;
    __device__ __forceinline__ void operator()(int c, int64_t col, double coef) { acc[c] += coef * x[col]; }
};

// The sums of a unit's lists are formed in LDS while its own entries are on their way (12
// orbitals, with the residual update: 162 us with the entries streamed in first, 87 us; a
// row a thread of rowterms.hpp, without the update: 168 us; the bytes 75 us).  The lists
// follow each other in program order within the wavefront, so the sums have one order.  A
// list is a chain of item, pair tables and D2 entry: latency, hence four workgroups a CU,
// what the sums' 32 KB of LDS allow.
__global__ void __launch_bounds__(kBlock, 4)
k_t2_au(const DevLayout *__restrict__ Lp, T2Tab T, const double *__restrict__ x, double *__restrict__ Ax,
        const double *__restrict__ done, const double *__restrict__ dotv, double *__restrict__ rowpart, CgFuse fz,
        int64_t part0)
{
    __shared__ double sh[kWaves][kT2Chunk];
    __shared__ double red[3][kWaves];
    if (done && done[0] != 0.0) return;
    const DevLayout &L = *Lp;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t unit = (int64_t)blockIdx.x * kWaves + wave;
    const double alpha = fz.r ? fz.scal[CG_ALPHA] : 0.0;
    double sum[3] = {0.0, 0.0, 0.0};
    if (unit < T.units) {
        int row;
        T2Chunk ch;
        const T2Seg &sg = t2_unit(T, unit, row, ch);
        const int64_t e0 = t2_first(L, sg, row, ch);
        const double *own = x + sg.x0 + e0;
        const int64_t r0 = sg.row0 + e0;
        double *acc = sh[wave];
        double v[kPer];   // in flight while the lists are walked
#pragma unroll
        for (int u = 0; u < kPer; u++) v[u] = u * 64 + lane < ch.n ? own[u * 64 + lane] : 0.0;
#pragma unroll
        for (int u = 0; u < kPer; u++) acc[u * 64 + lane] = 0.0;
        wave_fence();
        AddTo f{acc, x};
        t2_unit_terms(L, T, sg, row, ch, lane, 64, f, wave_fence);
        if (fz.r) {
            double ro[kPer];
#pragma unroll
            for (int u = 0; u < kPer; u++) ro[u] = u * 64 + lane < ch.n ? fz.r[r0 + u * 64 + lane] : 0.0;
#pragma unroll
            for (int u = 0; u < kPer; u++) {
                const int c = u * 64 + lane;
                if (c >= ch.n) break;
                const double rn = ro[u] - alpha * (acc[c] - v[u]);
                fz.r[r0 + c] = rn;
                const double zn = fz.minv ? fz.minv[r0 + c] * rn : rn;
                sum[0] += rn * zn;
                sum[1] += rn * rn;
                sum[2] += ro[u] * zn;
            }
        } else {
#pragma unroll
            for (int u = 0; u < kPer; u++) {
                const int c = u * 64 + lane;
                if (c >= ch.n) break;
                const double a = acc[c] - v[u];
                Ax[r0 + c] = a;
                if (dotv) sum[0] += a * dotv[r0 + c];
            }
        }
    }
    if (!rowpart && !fz.r) return;
#pragma unroll
    for (int k = 0; k < 3; k++) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) sum[k] += __shfl_xor(sum[k], o, 64);
        if (lane == 0) red[k][wave] = sum[k];
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        double s = 0.0;
        for (int w = 0; w < kWaves; w++) s += red[threadIdx.x][w];
        if (fz.r) fz.part[threadIdx.x * fz.ntiles + part0 + blockIdx.x] = s;
        else if (threadIdx.x == 0) rowpart[blockIdx.x] = s;
    }
}

constexpr int kATut = 1024, kEntries = 128, kParts = kATut / kEntries, kCopy = 8 * kATut;

// A D2 column's entries go one to a thread in eight parts of the orbitals' sum: neighbours
// share the T2 rows they read or their lines.  The copies of the T2 blocks follow (by turns
// with the sums, at 512 threads, two workgroups a CU: 7 % slower).  12 orbitals (14 million T2
// rows): 98 us, the copies' bytes 50 us; with one row a thread and FP64 atomics instead
// 148 us (6 million atomics on 30 000 entries), and a second pass over D2, which also kept
// the CG from its fused form.
__global__ void __launch_bounds__(kATut)
k_t2_atu(const DevLayout *__restrict__ Lp, T2Tab T, const T2Tile *__restrict__ tiles,
         const double *__restrict__ y, double *__restrict__ ATy, const double *__restrict__ done,
         double *__restrict__ sqpart)
{
    __shared__ double sh[kParts][kEntries];
    __shared__ double red[kATut / 64];
    if (done && done[0] != 0.0) return;
    const DevLayout &L = *Lp;
    const T2Tile &tl = tiles[blockIdx.x];
    const Segment &sg = tl.sg;
    const int tid = threadIdx.x, lane = tid & 63;
    double sq = 0.0;
    if (sg.kind == XS_SELF) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int i = u * kATut + tid;
            v[u] = i < tl.n ? -y[sg.aux + tl.i0 + i] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int i = u * kATut + tid;
            if (i < tl.n) ATy[sg.start + tl.i0 + i] = v[u];
            sq += v[u] * v[u];
        }
    } else if (sg.kind == XS_D1) {
        const int n = (int)(tl.i0 / sg.dim) + L.poff[sg.h], k = (int)(tl.i0 % sg.dim) + L.poff[sg.h];
        double v = 0.0;
        if (tid < 64) v = atu_d1_wave(L, sg, tl.i0, lane, y);
        for (int ij = tid; ij < L.amo * L.amo; ij += kATut) v += t2_at_d1(L, T, sg.sub, ij / L.amo, ij % L.amo, n, k, y);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if (lane == 0) red[tid >> 6] = v;
        __syncthreads();
        if (tid == 0) {
            v = 0.0;
            for (int w = 0; w < kATut / 64; w++) v += red[w];
            ATy[sg.start + tl.i0] = v;
            sq = v * v;
        }
        __syncthreads();
    } else {
        const int e = tid % kEntries, part = tid / kEntries;
        double v = 0.0;
        if (e < tl.n) {
            const bool ab = sg.kind == XS_D2AB;
            const int *pairs = ab ? L.bab + L.bab_off[sg.h] : L.baa + L.baa_off[sg.h];
            const int b = pairs[tl.i0 + e], k = pairs[tl.k];
            if (ab) {
                for (int u = part; u < 2 * L.amo; u += kParts)
                    v += t2_at_ab(L, T, u & 1, u >> 1, P0(b), P1(b), P0(k), P1(k), y);
            } else {   // the aa pairs are stored larger orbital first
                for (int u = part; u < L.amo; u += kParts)
                    v += t2_at_aa(L, T, sg.sub, u, P1(b), P0(b), P1(k), P0(k), y);
            }
            if (part == kParts - 1) {
                const int64_t i = (tl.i0 + e) * sg.dim + tl.k;
                v += ab ? atu_d2ab(L, sg, i, y) : atu_d2aa(L, sg, i, y);
            }
        }
        sh[part][e] = v;
        __syncthreads();
        if (part == 0 && e < tl.n) {
            for (int w = 1; w < kParts; w++) v += sh[w][e];
            ATy[sg.start + (tl.i0 + e) * sg.dim + tl.k] = v;
            sq = v * v;
        }
    }
    if (!sqpart) return;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o, 64);
    if (lane == 0) red[tid >> 6] = sq;
    __syncthreads();
    if (tid == 0) {
        double s = 0.0;
        for (int w = 0; w < kATut / 64; w++) s += red[w];
        sqpart[blockIdx.x] = s;
    }
}

}  // namespace

void T2Maps::build(const Layout &L, const DevLayout *dlay)
{
    T2Lists t;
    make_t2_lists(L, t);
    dlay_ = dlay;
    seg_.upload(t.seg);
    chunk_.upload(t.chunk);
    ptr_.upload(t.ptr);
    item_.upload(t.item);
    aab_.upload(t.aab);
    aba_.upload(t.aba);
    tab_ = {seg_.p, chunk_.p, ptr_.p, item_.p, aab_.p, aba_.p, (int)t.seg.size(), t.units};
    // the D2 and D1 entries, then the T2 blocks' own
    std::vector<T2Tile> tl;
    for (const Segment &s : L.xsegs) {
        if (s.kind == XS_D1) {
            for (int64_t i = 0; i < s.count; i++) tl.push_back({s, i, 0, 1});
        } else if (s.kind == XS_D2AB || s.kind == XS_D2AA) {
            const int nc = (s.dim + kEntries - 1) / kEntries, size = (s.dim + nc - 1) / nc;
            for (int k = 0; k < s.dim; k++)
                for (int i = 0; i < s.dim; i += size) tl.push_back({s, i, k, std::min(size, s.dim - i)});
        }
    }
    for (Segment s : L.xsegs_t2) {
        if (s.kind != RF_T2AAB && s.kind != RF_T2BIG) continue;
        s.kind = XS_SELF;
        for (int64_t i = 0; i < s.count; i += kCopy)
            tl.push_back({s, i, 0, (int32_t)std::min<int64_t>(kCopy, s.count - i)});
    }
    tiles_.upload(tl);
    blocks_ = (int)((t.units + kWaves - 1) / kWaves);
}

void T2Maps::au(const double *x, double *Ax, const double *done, const double *dotv, double *rowpart,
                CgFuse fz, int64_t part0, hipStream_t st) const
{
    if (blocks_ > 0)
        hipLaunchKernelGGL(k_t2_au, dim3(blocks_), dim3(kBlock), 0, st, dlay_, tab_, x, Ax, done, dotv, rowpart, fz,
                           part0);
}

void T2Maps::atu(const double *y, double *ATy, const double *done, double *sqpart, hipStream_t st) const
{
    if (tiles_.n > 0)
        hipLaunchKernelGGL(k_t2_atu, dim3((unsigned)tiles_.n), dim3(kATut), 0, st, dlay_, tab_, tiles_.p, y, ATy,
                           done, sqpart);
}

}  // namespace v2g
