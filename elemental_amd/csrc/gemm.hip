// C := beta*C + alpha * op(A) * op(B), FP64, op(A) m x k, op(B) k x n
// (column-major), optionally restricted to the lower or the upper triangle
// of a square C, with triangular operand masks.
//
// Uses:
//  * Elemental's LocalTrrk / Trrk(LOWER, TRANSPOSE, NORMAL, ...)
//    (src/blas-like/Trrk/Local.hpp:733-775 and :931-976, leaf kernels
//    :452-536), the triangular rank-k update of the DistMatrix route of the
//    blocked Cholesky (include/elemental/lapack-like/Cholesky/LVar3Square.hpp).
//    The reference recurses by halves down to 64x64 leaves and then does full
//    square GEMMs plus AxpyTriangle; on the GPU the lower tiles are simply
//    enumerated and diagonal tiles mask their upper part, which gives the same
//    lower trapezoid.
//  * elem::Gemm (include/elemental/blas-like/level3/Gemm.hpp) in every
//    orientation, and the products with a triangular factor or its inverse
//    (Trmm-like) of the HPD inverse, the triangular inverse and the
//    two-sided reductions: a masked operand reads as zero outside its
//    triangle (and as one on a unit diagonal), so the other triangle of the
//    stored matrix is never used.
//
// 64 x 64 tiles (tile64_dev.hpp) of eight waves, two chunks of 16 along k on
// their way.  Global loads follow the stored layout: an operand whose m or n
// index runs down the columns is read 64 rows at a time, one whose k index
// does (A transposed, B not) as 16 consecutive k of four columns.  Several
// products that do not depend on each other go into one launch (GemmJobs): a
// step of the HPD inverse at n = 3000 has products of 2 to 700 tiles, and
// alone each took 43 us in 128 x 128 tiles; the two launches of a step now
// take 25 us on average.  1024^3: 200 us, now 60; 256^3: 53 and 18.
#include "common.hpp"
#include "kernels.hpp"
#include "syrk_dev.hpp"
#include "tile64_dev.hpp"

namespace elemamd {

constexpr int kGemmKC = 16, kGemmNW = 8, kGemmDepth = 2;
constexpr int kGemmLd = tile64::kTile + 17;  // 16 k of a column go to as many banks

// Stored element (r, c) of a masked operand (kGemmShape*).
__device__ __forceinline__ double gemm_mask(double v, int r, int c, int shape) {
    if (shape == kGemmShapeFull) return v;
    const bool lower = shape == kGemmShapeLower || shape == kGemmShapeLowerUnit;
    const bool unit = shape == kGemmShapeLowerUnit || shape == kGemmShapeUpperUnit;
    if (r == c) return unit ? 1.0 : v;
    return (lower ? r > c : r < c) ? v : 0.0;
}

// One operand tile of 64 (m or n) x 16 (k) into registers, then LDS s[l][x] =
// op(M)(x0 + x, l) with x the m (A) or n (B) index; loads without branches, as
// in tile64::RowLoader.  KDOWN: the stored matrix holds k down its columns
// (element (l, x) at M[l + x ld]); otherwise element (x, l) at M[x + l ld].
template <bool KDOWN>
struct GemmLoader {
    static constexpr int kDepth = kGemmDepth, kW = kGemmNW, kQ = 16 / kGemmNW;
    const double* p[kQ];  // this thread's elements of the chunk to load next
    i64 step;
    int k, x0, shape, l[kQ], xt[kQ];  // l: within the chunk; xt: within the tile
    int next;                          // first k of the chunk to load next
    double g[kDepth][kQ];
    __device__ __forceinline__ GemmLoader(const double* M, i64 ld, int ext, int k_, int x0_, int shape_)
        : step(k_ > 0 ? (KDOWN ? kGemmKC : kGemmKC * ld) : 0), k(k_), x0(x0_), shape(shape_), next(0) {
        const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int q = 0; q < kQ; ++q) {
            l[q] = KDOWN ? lane & 15 : w + kGemmNW * q;
            xt[q] = KDOWN ? 4 * (w + kGemmNW * q) + (lane >> 4) : lane;
            const int x = min(x0 + xt[q], ext - 1), lc = max(min(l[q], k - 1), 0);
            p[q] = k > 0 ? M + (KDOWN ? lc + x * ld : x + lc * ld) : (const double*)tile64::kNoColumn;
        }
    }
    __device__ __forceinline__ void load(int d) {
        next += kGemmKC;
#pragma unroll
        for (int q = 0; q < kQ; ++q) {
            g[d][q] = *p[q];
            p[q] += next + l[q] < k ? step : 0;
        }
    }
    template <typename Row>
    __device__ __forceinline__ void store(Row* s, double scale, int k0, int d) const {
#pragma unroll
        for (int q = 0; q < kQ; ++q) {
            double v = g[d][q];
            const int x = x0 + xt[q], kk = k0 + l[q];
            if (shape != kGemmShapeFull) v = KDOWN ? gemm_mask(v, kk, x, shape) : gemm_mask(v, x, kk, shape);
            s[l[q]][xt[q]] = kk < k ? scale * v : 0.0;
        }
    }
};

typedef tile64::Smem<double, kGemmKC, kGemmLd> GemmSmem;

template <bool TA, bool TB>
__device__ __forceinline__ void gemm_tile(GemmSmem& sm, const GemmJob& g, int i0, int j0) {
    GemmLoader<TA> la(g.A, g.lda, g.m, g.k, i0, g.ashape);   // op(A) = A^T: stored k x m
    GemmLoader<!TB> lb(g.B, g.ldb, g.n, g.k, j0, g.bshape);  // op(B) = B: stored k x n
    tile64::tile<false>(sm, la, lb, i0, j0, g.m, g.n, g.k, g.alpha, g.beta, g.C, g.ldc, g.tri);
}

// tri: 0 every tile; 1 the lower triangle (tiles ti >= tj, j <= i); 2 the
// upper triangle (tiles ti <= tj, i <= j)
__global__ __launch_bounds__(64 * kGemmNW, 4) void gemm_f64_kernel(GemmJobs jobs, const int* __restrict__ info) {
    __shared__ GemmSmem sm;
    if (info != nullptr && *info != 0) return;  // an earlier step failed
    int t = blockIdx.x, q = 0;
    while (t >= jobs.job[q].tiles) t -= jobs.job[q++].tiles;  // (the grid is the sum of the jobs' tiles)
    const GemmJob& g = jobs.job[q];
    int ti, tj;
    if (g.tri == 1) tri_tile(t, ti, tj);
    else if (g.tri == 2) tri_tile(t, tj, ti);
    else {
        const int tm = (g.m + tile64::kTile - 1) / tile64::kTile;
        ti = t % tm;
        tj = t / tm;
    }
    const int i0 = ti * tile64::kTile, j0 = tj * tile64::kTile;
    if (g.ta) {
        if (g.tb) gemm_tile<true, true>(sm, g, i0, j0);
        else gemm_tile<true, false>(sm, g, i0, j0);
    } else {
        if (g.tb) gemm_tile<false, true>(sm, g, i0, j0);
        else gemm_tile<false, false>(sm, g, i0, j0);
    }
}

// ------------------------------------------------ large products
// 128 x 128 tiles, four waves of 64 x 64, double-buffered chunks of 16.
// From 1024 such tiles on (four a CU) these tiles' halved L2 traffic pays for
// what the last round of them leaves idle: 4096^3 (NN / NT) 2.59 and 2.36 ms,
// with 64 x 64 tiles 2.51 to 2.70 and 2.52 to 2.59; 6144 x 6144 x 1024 1.42 and
// 1.51, 1.42 and 1.44; but 3072^3 1.49 and 1.76, 1.06 and 1.08; 1024^3 0.20,
// 0.06.
constexpr i64 kGemmBigTiles = 1024;
constexpr int kGemmTile = 128;
constexpr int kGemmLdp = kGemmTile + 16;

// One operand tile of 128 (m or n) x 16 (k) into registers, then LDS s[l][x]
// = op(M)(x0 + x, l) with x the m (A) or n (B) index.  KCONTIG: the stored
// matrix holds k down its columns (element (l, x) at M[l + x*ld]); otherwise
// element (x, l) at M[x + l*ld].
template <bool KCONTIG>
struct GemmBigLoader {
    const double* M;
    i64 ld;
    int ext, k, x0, shape;
    int tid;
    double g[8];
    __device__ __forceinline__ void load(int kc0) {
        if constexpr (KCONTIG) {
            const int x = tid >> 1, lh = (tid & 1) * 8;
            const bool xin = (x0 + x) < ext;
            const double* p = M + (i64)(x0 + x) * ld;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int l = kc0 + lh + q;
                const double v = (xin && l < k) ? p[l] : 0.0;
                g[q] = gemm_mask(v, l, x0 + x, shape);  // stored (row l, column x)
            }
        } else {
            const int l = kc0 + (tid >> 4), xb = (tid & 15) * 8;
            const bool lin = l < k;
            const double* p = M + (i64)l * ld + x0 + xb;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int x = x0 + xb + q;
                const double v = (lin && x < ext) ? p[q] : 0.0;
                g[q] = gemm_mask(v, x, l, shape);  // stored (row x, column l)
            }
        }
    }
    __device__ __forceinline__ void store(double (*s)[kGemmLdp]) const {
        if constexpr (KCONTIG) {
            const int x = tid >> 1, lh = (tid & 1) * 8;
#pragma unroll
            for (int q = 0; q < 8; ++q) s[lh + q][x] = g[q];
        } else {
            const int l = tid >> 4, xb = (tid & 15) * 8;
#pragma unroll
            for (int q = 0; q < 8; ++q) s[l][xb + q] = g[q];
        }
    }
};

template <bool TA, bool TB>
__global__ __launch_bounds__(256, 2) void gemm_big_f64_kernel(int m, int n, int k, double alpha, const double* A,
                                                          i64 lda, int ashape, const double* B, i64 ldb, int bshape,
                                                          double beta, double* C, i64 ldc, int tri,
                                                          const int* __restrict__ info) {
    __shared__ double sA[2][kGemmKC][kGemmLdp];  // sA[l][i] = op(A)(i0+i, l)
    __shared__ double sB[2][kGemmKC][kGemmLdp];  // sB[l][j] = op(B)(l, j0+j)
    if (info != nullptr && *info != 0) return;   // an earlier step failed
    // tri: 0 every tile; 1 the lower triangle (tiles ti >= tj, j <= i);
    // 2 the upper triangle (tiles ti <= tj, i <= j)
    int ti, tj;
    if (tri == 1) {
        tri_tile(blockIdx.x, ti, tj);
    } else if (tri == 2) {
        tri_tile(blockIdx.x, tj, ti);
    } else {
        ti = blockIdx.x;
        tj = blockIdx.y;
    }
    const int i0 = ti * kGemmTile, j0 = tj * kGemmTile;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wj = (w >> 1) * 64, wi = (w & 1) * 64;
    const bool skip = (ti == tj) && ((tri == 1 && wj > wi) || (tri == 2 && wi > wj));

    // op(A) = A^T: A stored k x m (k down the columns); op(B) = B: B stored k x n
    GemmBigLoader<TA> la{A, lda, m, k, i0, ashape, tid, {}};
    GemmBigLoader<!TB> lb{B, ldb, n, k, j0, bshape, tid, {}};
    d4_t acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = (d4_t){0.0, 0.0, 0.0, 0.0};
    la.load(0);
    lb.load(0);
    la.store(sA[0]);
    lb.store(sB[0]);
    __syncthreads();
    const int nchunks = (int)ceil_div(k, kGemmKC);
    for (int c = 0; c < nchunks; ++c) {
        const int buf = c & 1;
        const bool more = (c + 1) < nchunks;
        if (more) {
            la.load((c + 1) * kGemmKC);
            lb.load((c + 1) * kGemmKC);
        }
        if (!skip) {
#pragma unroll
            for (int ks = 0; ks < kGemmKC / 4; ++ks) {
                const int kr = ks * 4 + (lane >> 4);
                double fa[4], fb[4];
#pragma unroll
                for (int mb = 0; mb < 4; ++mb) fa[mb] = sB[buf][kr][wj + 16 * mb + (lane & 15)];
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) fb[nb] = sA[buf][kr][wi + 16 * nb + (lane & 15)];
#pragma unroll
                for (int mb = 0; mb < 4; ++mb)
#pragma unroll
                    for (int nb = 0; nb < 4; ++nb)
                        acc[mb][nb] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[mb], fb[nb], acc[mb][nb], 0, 0, 0);
            }
        }
        if (more) {
            la.store(sA[buf ^ 1]);
            lb.store(sB[buf ^ 1]);
        }
        __syncthreads();
    }
    if (skip) return;
    // dependent zero-operand MFMAs before the accumulators are read (the
    // compiler's wait states after a loop back edge are short for FP64 MFMA)
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb)
            acc[mb][nb] = __builtin_amdgcn_mfma_f64_16x16x4f64(0.0, 0.0, acc[mb][nb], 0, 0, 0);
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            const int i = i0 + wi + 16 * nb + (lane & 15);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int j = j0 + wj + 16 * mb + (lane >> 4) + 4 * v;  // f64 MFMA: row = lane/16 + 4*v
                if (i < m && j < n && (tri == 0 || (tri == 1 ? j <= i : i <= j))) {
                    double* p = C + (i64)i + (i64)j * ldc;
                    const double upd = alpha * acc[mb][nb][v];
                    *p = (beta == 0.0) ? upd : beta * (*p) + upd;
                }
            }
        }
}

void GemmJobs::add(bool ta, bool tb, int m, int n, int k, double alpha, const double* A, i64 lda, int ashape,
                   const double* B, i64 ldb, int bshape, double beta, double* C, i64 ldc, int tri) {
    if (m <= 0 || n <= 0) return;
    const i64 Tm = ceil_div(m, tile64::kTile), Tn = ceil_div(n, tile64::kTile);
    job[count++] = GemmJob{A, B, C, lda, ldb, ldc, alpha, beta, m, n, k < 0 ? 0 : k,
                           (int)(tri != 0 ? Tm * (Tm + 1) / 2 : Tm * Tn), ashape, bshape, ta ? 1 : 0, tb ? 1 : 0, tri};
}

hipError_t launch_gemm_jobs_f64(const GemmJobs& jobs, const int* info, hipStream_t s) {
    unsigned tiles = 0;
    for (int q = 0; q < jobs.count; ++q) tiles += (unsigned)jobs.job[q].tiles;
    if (tiles == 0) return hipSuccess;
    hipLaunchKernelGGL(gemm_f64_kernel, dim3(tiles), dim3(64 * kGemmNW), 0, s, jobs, info);
    return hipGetLastError();
}

hipError_t launch_gemm_f64(bool ta, bool tb, int m, int n, int k, double alpha, const double* A, i64 lda, int ashape,
                           const double* B, i64 ldb, int bshape, double beta, double* C, i64 ldc, int tri,
                           const int* info, hipStream_t s, bool in_place) {
    if (m <= 0 || n <= 0) return hipSuccess;
    if (tri != 0 && m != n) return hipErrorInvalidValue;
    const i64 Tm = ceil_div(m, kGemmTile), Tn = ceil_div(n, kGemmTile), tiles = tri != 0 ? Tm * (Tm + 1) / 2 : Tm * Tn;
    if (tiles >= kGemmBigTiles || in_place) {
        const dim3 grid = tri != 0 ? dim3((unsigned)tiles) : dim3((unsigned)Tm, (unsigned)Tn);
        auto kernel = ta ? (tb ? gemm_big_f64_kernel<true, true> : gemm_big_f64_kernel<true, false>)
                         : (tb ? gemm_big_f64_kernel<false, true> : gemm_big_f64_kernel<false, false>);
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, m, n, k < 0 ? 0 : k, alpha, A, lda, ashape, B, ldb, bshape, beta,
                           C, ldc, tri, info);
        return hipGetLastError();
    }
    GemmJobs jobs;
    jobs.add(ta, tb, m, n, k, alpha, A, lda, ashape, B, ldb, bshape, beta, C, ldc, tri);
    return launch_gemm_jobs_f64(jobs, info, s);
}

hipError_t launch_gemm_tn_f64(int m, int n, int k, double alpha, const double* A, i64 lda, const double* B, i64 ldb,
                              double beta, double* C, i64 ldc, int tri, hipStream_t s, bool in_place) {
    return launch_gemm_f64(true, false, m, n, k, alpha, A, lda, kGemmShapeFull, B, ldb, kGemmShapeFull, beta, C, ldc,
                           tri, nullptr, s, in_place);
}

}  // namespace elemamd
