// gemm.hip -- batched FP64 GEMM C = op(A) op(B) for the eigen split
// (warm-start transform V^T M V and the reconstruction x = W W^T).
// 64 x 64 output tile per workgroup, 32-deep K panels staged in LDS, the next
// panel prefetched into registers while the current one is multiplied; each
// wave computes a 32 x 32 sub-tile with v_mfma_f64_16x16x4f64 (A[i][k] from
// lane i + 16k, B[k][j] from lane j + 16k, D[i][j] in lane j + 16 (i % 4),
// element i / 4).  A descriptor with sym = 1 declares C symmetric: only the
// tiles on and above the diagonal are computed, and each is also written
// transposed.
//
// Operands are whole padded workspaces (eig.hpp), so the panels are read without bounds
// checks, 16 bytes a load, from scalar bases with 32-bit offsets.  H50 (two blocks padded to
// 2 560, eight to 1 280, eight to 640; 105 GFLOP for M V): 2.36 ms with panels whose LDS
// reads and transposed writes met in the same banks, which kept the LDS pipe as busy as the
// matrix cores; 2.00 ms (52 TFLOP/s) with the layout below.  The order of the tiles over
// the XCDs gives the symmetric products another 10 %.
#include <hip/hip_runtime.h>

#include "eig.hpp"

namespace v2g {

namespace {

constexpr int kT = 256, kTile = 64, kK = kGemmK;
constexpr int kXcds = 8, kBand = 8;
constexpr int kPieces = kK * kTile / 2 / kT;   // 16-byte pieces of a panel one thread moves
// a panel lies in LDS the way it lies in memory: as 32 k rows of 64 entries, odd rows with
// bit 4 of the column flipped, or as 64 rows of 32 + 2: both kinds of operand reads (32
// lanes: 16 entries by 2 k) and the 16-byte writes are then free of bank conflicts
constexpr int kPitch = kK + 2;
typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

// a panel of one operand: KMAJOR: 32 k rows of 64 entries; else 64 rows of 32 k entries
template <bool KMAJOR>
struct Panel {
    static constexpr int kDoubles = KMAJOR ? kK * kTile : kTile * kPitch;
    static __device__ __forceinline__ int at(int k, int i)
    {
        return KMAJOR ? k * kTile + (i ^ (k & 1) << 4) : i * kPitch + k;
    }
    const char *base;       // first entry of the tile's first panel
    uint32_t off[kPieces];  // byte offsets of this thread's pieces
    uint32_t step;          // bytes from one panel to the next
    v2d v[kPieces];
    __device__ __forceinline__ Panel(const double *p, int ld, int tile0)
    {
        const double *b = KMAJOR ? p + tile0 : p + (int64_t)tile0 * ld;
        base = reinterpret_cast<const char *>(b);
        step = KMAJOR ? (uint32_t)(kK * ld * 8) : (uint32_t)(kK * 8);
#pragma unroll
        for (int u = 0; u < kPieces; u++) {
            const int w = threadIdx.x + u * kT;
            const int row = KMAJOR ? w / (kTile / 2) : w / (kK / 2), c = KMAJOR ? w % (kTile / 2) : w % (kK / 2);
            off[u] = (uint32_t)(row * ld + 2 * c) * 8u;
        }
    }
    __device__ __forceinline__ void fetch()
    {
#pragma unroll
        for (int u = 0; u < kPieces; u++) v[u] = *reinterpret_cast<const v2d *>(base + off[u]);
        base += step;
    }
    __device__ __forceinline__ void stash(double *s) const
    {
#pragma unroll
        for (int u = 0; u < kPieces; u++) {
            const int w = threadIdx.x + u * kT;
            const int row = KMAJOR ? w / (kTile / 2) : w / (kK / 2), c = KMAJOR ? w % (kTile / 2) : w % (kK / 2);
            *reinterpret_cast<v2d *>(s + (KMAJOR ? at(row, 2 * c) : at(2 * c, row))) = v[u];
        }
    }
};

// The output tile of workgroup blockIdx.x (gridDim.x is a multiple of 8, so blockIdx.x % 8
// is its XCD): each XCD takes one contiguous run of the tiles, in bands of kBand tile rows
// walked column by column, so the tiles it computes at one time share their panels in its L2.
__device__ __forceinline__ bool tile_of(const GemmDesc &d, int &tm, int &tn)
{
    const int rows = (d.M + kTile - 1) / kTile, cols = (d.N + kTile - 1) / kTile;
    const int total = d.sym ? rows * (rows + 1) / 2 : rows * cols, run = (total + kXcds - 1) / kXcds;
    const int i = blockIdx.x / kXcds;
    int t = blockIdx.x % kXcds * run + i;
    if (i >= run || t >= total) return false;
    for (int r0 = 0;; r0 += kBand) {
        const int h = min(kBand, rows - r0);                 // tile rows r0 .. r0 + h - 1
        const int head = d.sym ? h * (h + 1) / 2 : 0;        // the band's triangle at the diagonal
        const int count = head + h * (d.sym ? cols - r0 - h : cols);
        if (t >= count) {
            t -= count;
            continue;
        }
        if (t < head) {
            tn = 0;
            while (t > tn) t -= ++tn;
            tm = r0 + t;
            tn += r0;
        } else {
            t -= head;
            tm = r0 + t % h;
            tn = (d.sym ? r0 + h : 0) + t / h;
        }
        return true;
    }
}

// four waves per SIMD (the LDS panels allow four workgroups per CU)
template <bool TA, bool TB>
__global__ void __launch_bounds__(kT, 4)
k_gemm(const GemmDesc *__restrict__ descs)
{
    __shared__ __align__(16) double As[Panel<TA>::kDoubles];
    __shared__ __align__(16) double Bs[Panel<!TB>::kDoubles];
    const GemmDesc d = descs[blockIdx.y];
    int tm, tn;
    if (!tile_of(d, tm, tn)) return;
    const int m0 = tm * kTile, n0 = tn * kTile;
    const int K = d.kcount ? *d.kcount : d.K;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32, li = lane & 15, lk = lane >> 4;

    Panel<TA> pa(d.A, d.lda, m0);       // op(A)[m][k] = A[k][m] when transposed
    Panel<!TB> pb(d.B, d.ldb, n0);      // op(B)[k][n] = B[n][k] when transposed
    v4d acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) acc[a][b] = v4d{0.0, 0.0, 0.0, 0.0};
    if (K > 0) {
        pa.fetch();
        pb.fetch();
    }
    for (int k0 = 0; k0 < K; k0 += kK) {
        pa.stash(As);
        pb.stash(Bs);
        __syncthreads();
        if (k0 + kK < K) {   // next panel in flight during the MFMAs
            pa.fetch();
            pb.fetch();
        }
#pragma unroll
        for (int k4 = 0; k4 < kK; k4 += 4) {
            const double av[2] = {As[Panel<TA>::at(k4 + lk, wr + li)], As[Panel<TA>::at(k4 + lk, wr + li + 16)]};
            const double bv[2] = {Bs[Panel<!TB>::at(k4 + lk, wc + li)], Bs[Panel<!TB>::at(k4 + lk, wc + li + 16)]};
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int b = 0; b < 2; b++)
                    acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[a], bv[b], acc[a][b], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int gm = m0 + wr + a * 16 + 4 * r + lk, gn = n0 + wc + b * 16 + li;
                if (gm < d.M && gn < d.N) {
                    d.C[(int64_t)gm * d.ldc + gn] = acc[a][b][r];
                    if (d.sym && tm != tn) d.C[(int64_t)gn * d.ldc + gm] = acc[a][b][r];
                }
            }
}

}  // namespace

void gemm_batched(const GemmDesc *descs, int ndesc, int max_m, int max_n, int ta, int tb, hipStream_t st)
{
    if (ndesc <= 0) return;
    const int tiles = ((max_m + kTile - 1) / kTile) * ((max_n + kTile - 1) / kTile);
    const int grid = (tiles + kXcds - 1) / kXcds * kXcds;
    auto *k = ta ? (tb ? k_gemm<true, true> : k_gemm<true, false>) : (tb ? k_gemm<false, true> : k_gemm<false, false>);
    hipLaunchKernelGGL(k, dim3(grid, ndesc), dim3(kT), 0, st, descs);
}

}  // namespace v2g
