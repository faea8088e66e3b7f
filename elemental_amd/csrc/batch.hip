// Batched HPD factor-and-solve for many independent matrices of uneven size
// (no reference counterpart: Elemental factors one matrix per call).
//
// Each matrix is the same computation as the single-matrix path: LVar3 with
// block size nb (the same potrf / panel-solve / trailing-update device code,
// so a matrix gives the same result alone and inside a batch), then the
// forward and backward solves (batch_solve.hip).  Matrices are processed in
// order of decreasing size; step j of the factorization of every matrix that has a step j runs in
// one launch per kernel type, and a workgroup finds its (matrix, tile) from a
// per-step prefix sum of work counts, so small and large matrices share
// launches without idle workgroups.  The whole sequence is captured in a
// hipGraph by the host driver and replayed as one submission.
//
// Layout: matrix i is column-major with ld = n_i at element offset a_off[i] of
// one buffer; its right-hand sides (n_i x k_i, ld = n_i) at b_off[i].
#include <algorithm>

#include "batch.hpp"
#include "common.hpp"
#include "diag16_dev.hpp"
#include "kernels.hpp"
#include "panel16_dev.hpp"
#include "syrk_dev.hpp"
#include "tile64_dev.hpp"

namespace elemamd {

// index p with prefix[p] <= w < prefix[p+1]
__device__ inline int find_item(const int* prefix, int cnt, int w) {
    int lo = 0, hi = cnt;  // prefix[0] = 0 <= w < prefix[cnt]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (prefix[mid] <= w) lo = mid;
        else hi = mid;
    }
    return lo;
}

// ---------------------------------------------------------- factorization
// One workgroup per matrix: 30 us per 128-column step of 1024 matrices
// (n = 16 ... 1024) where a column-by-column factor through LDS took 84.
template <typename T>
__global__ __launch_bounds__(diag16::kThreads, 4) void batch_potrf_kernel(BatchArgs a, T* A, int step, int nb) {
    __shared__ diag16::Lds<false> sh;
    const int p = blockIdx.x;
    const int n = a.n[p];
    const int c0 = step * nb;
    if (c0 >= n) return;
    if (a.skip != nullptr && a.skip[p]) return;
    const int* info = a.info + p;
    if (step > 0 && *info != 0 && *info <= c0) return;  // an earlier block failed: this one was not updated
    const int b = min(nb, n - c0);
    diag16::factor_block<T, false>(sh, b, A + a.a_off[p] + c0 + (i64)c0 * n, n, nullptr, a.info + p, c0);
}

template <typename T>
__global__ __launch_bounds__(256) void batch_trsm_kernel(BatchArgs a, T* A, int step, int nb, const int* prefix,
                                                         int cnt) {
    __shared__ panel16::Lds sh;
    const int p = find_item(prefix, cnt, blockIdx.x);
    const int rb = blockIdx.x - prefix[p];
    const int n = a.n[p];
    const int c0 = step * nb;
    const int m = n - c0 - nb;
    if (m <= 0) return;  // (prefix gives such matrices no workgroups)
    if (a.skip != nullptr && a.skip[p]) return;
    const int* info = a.info + p;
    if (*info != 0 && *info <= c0 + nb) return;
    T* L = A + a.a_off[p] + c0 + (i64)c0 * n;
    panel16::slab<T>(sh, m, nb, L, n, L + nb, n, L + nb, n, rb);
}

// MODE 0, 1 (FP64, FP32): 64 x 64 tiles, as in the single matrix's update (in
// the persistent launch, where one workgroup has all of a matrix's tiles, 128
// x 128; each entry's operations are the same).  Most tiles of a batch belong
// to updates of a few hundred rows, where 128 x 128 ones leave half of the
// diagonal tiles' work and most CUs unused: 1024 matrices (n = 16 ... 1024),
// seven steps of 128: FP64 1.15 ms with 128 x 128 tiles, 0.88 now, FP32 0.79
// and 0.54.
template <typename T, int MODE>
__global__ __launch_bounds__(256, MODE == 2 ? 2 : 4) void batch_syrk_kernel(BatchArgs a, T* A, int step, int nb,
                                                                            const int* prefix, int cnt) {
    const int p = find_item(prefix, cnt, blockIdx.x);
    const int t = blockIdx.x - prefix[p];
    const int n = a.n[p];
    const int c0 = step * nb;
    const int m = n - c0 - nb;
    if (m <= 0) return;
    if (a.skip != nullptr && a.skip[p]) return;
    const int* info = a.info + p;
    if (*info != 0 && *info <= c0 + nb) return;
    int ti, tj;
    tri_tile(t, ti, tj);
    const T* P = A + a.a_off[p] + (c0 + nb) + (i64)c0 * n;
    T* C = A + a.a_off[p] + (c0 + nb) + (i64)(c0 + nb) * n;
    if constexpr (MODE == 2) {
        syrk_tile_bf16x3(m, m, nb, -1.0f, (const float*)P, n, (const float*)P, n, 1.0f, (float*)C, n, ti, tj);
    } else {
        constexpr int KC = MODE == 0 ? 16 : 32;
        __shared__ tile64::Smem<T, KC> sm;
        const int i0 = ti * tile64::kTile, j0 = tj * tile64::kTile;
        tile64::RowLoader<T, KC> li(P, n, m, nb, i0), lj(P, n, m, nb, j0);
        tile64::tile<sizeof(T) == 8>(sm, li, lj, i0, j0, m, m, nb, T(-1), T(1), C, n, 1);
    }
}

// ------------------------------------------------------ persistent launch
// One launch per size bucket: every workgroup takes the bucket's matrices in
// processing order (largest first) from a counter and factors each one whole
// with the device code of the stepwise launches above -- the diagonal block
// (256 threads, the same operation order), the register
// panel solve, the trailing tiles in the same K order -- so a matrix's
// factor is the same bit for bit in either form.  Workgroups never wait on
// each other.  The phases share one LDS arena (they never overlap), so two
// workgroups fit on a CU.
constexpr int kArenaPanel = sizeof(panel16::Lds);
constexpr int kArenaSyrk64 = 2 * 2 * kSyrkKC64 * kSyrkLdp * 8;
constexpr int kArenaSyrk32 = 2 * 2 * kSyrkKC * kSyrkLdpF * 4;
constexpr int kArenaBf16 = 4 * kSyrkTile * kBfLd * 2;
constexpr int cmax(int x, int y) { return x > y ? x : y; }
constexpr int kArenaBytes =
    cmax(cmax(cmax(kArenaPanel, kArenaSyrk64), cmax(kArenaSyrk32, kArenaBf16)), (int)sizeof(diag16::Lds<false>));

// The phases are separate (not inlined) functions: each gets the registers
// it needs on its own (inlined together they spilled).
template <typename T>
__device__ __noinline__ void persist_factor_block(int b, T* L, int n, int* info, int c0, char* arena) {
    diag16::factor_block<T, false, 4>(*reinterpret_cast<diag16::Lds<false>*>(arena), b, L, n, nullptr, info, c0);
}

// (NT: eight tiles spill, 64 columns do with four: 1024 matrices of n = 16 ...
// 1024 in blocks of 64, FP64: 7.3 ms, 11.0 with eight)
template <typename T, int NT>
__device__ __noinline__ void persist_panel(int m, int b, T* L, int n, char* arena) {
    for (int rb = 0; rb < (m + 63) / 64; ++rb) {
        panel16::slab<T, unsigned, false, NT>(*reinterpret_cast<panel16::Lds*>(arena), m, b, L, n, L + b, n, L + b, n, rb);
        __syncthreads();
    }
}

template <typename T, int MODE>
__device__ __noinline__ void persist_trailing(int m, int b, const T* P, T* C, int n, char* arena) {
    const int nt = (m + 127) / 128;
    for (int tt = 0; tt < nt * (nt + 1) / 2; ++tt) {
        int ti, tj;
        tri_tile(tt, ti, tj);
        if constexpr (MODE == 0) {
            auto sI = reinterpret_cast<double(*)[kSyrkKC64][kSyrkLdp]>(arena);
            auto sJ = reinterpret_cast<double(*)[kSyrkKC64][kSyrkLdp]>(arena + kArenaSyrk64 / 2);
            syrk_tile_f64_lds(m, m, b, -1.0, (const double*)P, n, (const double*)P, n, 1.0, (double*)C, n, ti, tj,
                              sI, sJ);
        } else if constexpr (MODE == 1) {
            auto sI = reinterpret_cast<float(*)[kSyrkKC][kSyrkLdpF]>(arena);
            auto sJ = reinterpret_cast<float(*)[kSyrkKC][kSyrkLdpF]>(arena + kArenaSyrk32 / 2);
            syrk_tile_f32_lds(m, m, b, -1.0f, (const float*)P, n, (const float*)P, n, 1.0f, (float*)C, n, ti, tj,
                              sI, sJ);
        } else {
            constexpr int q = kArenaBf16 / 4;
            auto s0 = reinterpret_cast<unsigned short(*)[kBfLd]>(arena);
            auto s1 = reinterpret_cast<unsigned short(*)[kBfLd]>(arena + q);
            auto s2 = reinterpret_cast<unsigned short(*)[kBfLd]>(arena + 2 * q);
            auto s3 = reinterpret_cast<unsigned short(*)[kBfLd]>(arena + 3 * q);
            syrk_tile_bf16x3_lds(m, m, b, -1.0f, (const float*)P, n, (const float*)P, n, 1.0f, (float*)C, n, ti, tj,
                                 s0, s1, s2, s3);
        }
        __syncthreads();
    }
}

template <typename T, int MODE>
__global__ __launch_bounds__(256, 2) void batch_persistent_kernel(BatchArgs a, T* A, int nb, int* counter) {
    __shared__ __align__(16) char arena[kArenaBytes];
    __shared__ int s_p;
    for (;;) {
        __syncthreads();  // every thread is done with the previous matrix
        if (threadIdx.x == 0) s_p = atomicAdd(counter, 1);
        __syncthreads();
        const int p = s_p;
        if (p >= a.count) return;
        const int n = a.n[p];
        T* M = A + a.a_off[p];
        int* info = a.info + p;
        for (int c0 = 0; c0 < n; c0 += nb) {
            const int b = min(nb, n - c0);
            T* L = M + c0 + (i64)c0 * n;
            persist_factor_block<T>(b, L, n, info, c0, arena);
            __syncthreads();  // the block and info are written (same CU: visible)
            if (*info != 0) break;
            const int m = n - c0 - b;
            if (m <= 0) break;
            if (b <= 64) {
                persist_panel<T, panel16::kTiles / 2>(m, b, L, n, arena);
            } else {
                int width = b;  // (opaque: FP32 lost 7 % at 128 columns with the range known inside)
                asm volatile("" : "+s"(width));
                persist_panel<T, panel16::kTiles>(m, width, L, n, arena);
            }
            persist_trailing<T, MODE>(m, b, L + b, M + (c0 + b) + (i64)(c0 + b) * n, n, arena);
        }
    }
}

// -------------------------------------------------- refinement helpers
// R_i := B_i - A_i X_i (A_i symmetric, lower triangle read), FP64.  Work
// items are 64-row blocks of every matrix (prefix sums over the bucket); a
// workgroup streams the 64x64 tiles of its block row of the symmetric matrix
// (tiles above the diagonal are read transposed from the stored lower
// triangle), with the right-hand sides in chunks of 8 columns.  Per-matrix
// maxima -- ||A||_inf (row sums of |A|), ||r_c||_inf, ||x_c||_inf,
// ||b_c||_inf -- are reduced per wave and merged with integer atomic max on
// the bit patterns of the non-negative doubles, which is order independent.
// red[p] layout: [0] ||A||_inf, [1 + c] r, [1 + kmax + c] x, [1 + 2 kmax + c] b.
__device__ inline double wave_max(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double u = __shfl_xor(v, o);
        v = (u > v || u != u) ? u : v;
    }
    return v;
}

__device__ inline void atomic_max_nonneg(double* p, double v) {
    atomicMax(reinterpret_cast<unsigned long long*>(p), (unsigned long long)__double_as_longlong(v));
}

// FIRST: X is zero and not read (R = B, the norms as above), and the tiles on
// and below the diagonal also go to S as float.
// What bounds it: reading A, each tile once in either orientation by the
// workgroups of its two block rows.  A thread keeps its 16 entries of a tile in
// registers and multiplies them by all columns (X by LDS broadcasts); only the
// tiles above the diagonal are turned through LDS.  1024 matrices, n = 16 ...
// 1024, up to 8 columns (1.03 GB read): 198 us (5.2 TB/s), with S 267; with all
// tiles and X read from LDS for two columns a thread 304, and 201 more for S.
template <bool FIRST>
__global__ __launch_bounds__(256) void batch_symv_residual_kernel(BatchArgs a, const double* A, const double* X,
                                                                  const double* Bin, double* R, const int* prefix,
                                                                  int cnt, double* red, int kmax, float* S) {
    __shared__ double sM[64][65];  // a tile to be turned; at the end the waves' sums
    __shared__ __align__(16) double sX[64][8];
    const int p = find_item(prefix, cnt, blockIdx.x);
    const int I = blockIdx.x - prefix[p];
    if (a.skip != nullptr && a.skip[p]) return;
    const int n = a.n[p], k = a.k[p];
    const double* Ap = A + a.a_off[p];
    const double* Xp = X + a.b_off[p];
    const double* Bp = Bin + a.b_off[p];
    double* Rp = R + a.b_off[p];
    double* rd = red + (i64)p * (1 + 3 * kmax);
    const int t = threadIdx.x, r = t & 63, w = t >> 6;
    const int r0 = I * 64;
    const int nT = (n + 63) / 64;
    const int row = r0 + r;
    const bool in = row < n;
    for (int c0 = 0; c0 < k; c0 += 8) {
        const int kc = min(8, k - c0);
        double acc[8] = {}, asum = 0.0;
        for (int J = 0; J < nT; ++J) {
            const int q0 = J * 64;
            // stored tile A(r0 + r, q0 + y) up to the diagonal (its lower part,
            // mirrored below), else Asym(r0 + y, q0 + r) = A(q0 + r, r0 + y),
            // y = w + 4 s; lanes along rows, clamped addresses
            const int rb = J <= I ? r0 : q0, cb = J <= I ? q0 : r0;
            double g[16];
            if (rb + 64 <= n && J != I) {  // (cb < rb)
                const double* e = Ap + (rb + r) + (i64)(cb + w) * n;
#pragma unroll
                for (int s = 0; s < 16; ++s, e += 4 * (i64)n) g[s] = *e;
            } else {
#pragma unroll
                for (int s = 0; s < 16; ++s) {
                    const int y = w + 4 * s;
                    const bool ok = rb + r < n && cb + y < n && (J != I || r >= y);
                    const double v = Ap[ok ? (rb + r) + (i64)(cb + y) * n : 0];
                    g[s] = ok ? v : 0.0;
                }
            }
            double x[2];
            if constexpr (!FIRST)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int c = w + 4 * u;
                    const bool ok = q0 + r < n && c < kc;
                    const double v = Xp[ok ? (q0 + r) + (i64)(c0 + c) * n : 0];
                    x[u] = ok ? v : 0.0;
                }
            if constexpr (FIRST)
                if (c0 == 0 && J <= I && in) {
                    float* Sp = S + a.a_off[p] + row + (i64)(q0 + w) * n;
#pragma unroll
                    for (int s = 0; s < 16; ++s, Sp += 4 * (i64)n)
                        if (J < I || r >= w + 4 * s) *Sp = (float)g[s];
                }
            __syncthreads();  // the tile before is done with sM and sX
            if (J > I) {
#pragma unroll
                for (int s = 0; s < 16; ++s) sM[r][w + 4 * s] = g[s];  // sM[q][row]
            } else if (J == I) {
#pragma unroll
                for (int s = 0; s < 16; ++s) {
                    const int y = w + 4 * s;
                    if (r >= y) sM[y][r] = sM[r][y] = g[s];
                }
            }
            if constexpr (!FIRST)
#pragma unroll
                for (int u = 0; u < 2; ++u) sX[r][w + 4 * u] = x[u];
            __syncthreads();
            if (J >= I)
#pragma unroll
                for (int s = 0; s < 16; ++s) g[s] = sM[w + 4 * s][r];
#pragma unroll
            for (int s = 0; s < 16; ++s) {  // g[s] = Asym(r0 + r, q0 + w + 4 s)
                asum += fabs(g[s]);
                if constexpr (!FIRST)
#pragma unroll
                    for (int c = 0; c < 8; ++c) acc[c] = fma(g[s], sX[w + 4 * s][c], acc[c]);
            }
        }
        // the four waves' sums of row r, [wave][8] and [32 + wave]
        __syncthreads();
        if constexpr (!FIRST)
#pragma unroll
            for (int c = 0; c < 8; ++c) sM[r][8 * w + c] = acc[c];
        sM[r][32 + w] = asum;
        __syncthreads();
        if (c0 == 0 && w == 0) {
            const double am = wave_max(in ? (sM[r][32] + sM[r][33]) + (sM[r][34] + sM[r][35]) : 0.0);
            if (r == 0) atomic_max_nonneg(&rd[0], am);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int c = w + 4 * u;
            double rv = 0.0, xv = 0.0, bv = 0.0;
            if (in && c < kc) {
                const i64 e = row + (i64)(c0 + c) * n;
                bv = Bp[e];
                rv = bv;
                if constexpr (!FIRST) {
                    xv = Xp[e];
                    rv -= (sM[r][c] + sM[r][8 + c]) + (sM[r][16 + c] + sM[r][24 + c]);
                }
                Rp[e] = rv;
            }
            const double rm = wave_max(fabs(rv)), xm = wave_max(fabs(xv)), bm = wave_max(fabs(bv));
            if (r == 0 && c < kc) {
                atomic_max_nonneg(&rd[1 + c0 + c], rm);
                atomic_max_nonneg(&rd[1 + kmax + c0 + c], xm);
                atomic_max_nonneg(&rd[1 + 2 * kmax + c0 + c], bm);
            }
        }
    }
}

// eta_i = max_c ||r_c||_inf / (||A_i||_inf ||x_c||_inf + ||b_c||_inf) (a NaN
// or an infinite ratio gives +inf), rscale_i(c) = ||r_c||_inf.
__global__ void batch_eta_kernel(BatchArgs a, const double* red, double* eta, double* rscale, int kmax) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.count) return;
    if (a.skip != nullptr && a.skip[p]) return;
    const double* rd = red + (i64)p * (1 + 3 * kmax);
    const double anorm = rd[0];
    double e = 0.0;
    for (int c = 0; c < a.k[p]; ++c) {
        const double rm = rd[1 + c], xm = rd[1 + kmax + c], bm = rd[1 + 2 * kmax + c];
        e = fmax(e, column_backward_error(rm, anorm, xm, bm));
        if (rscale != nullptr) rscale[(i64)p * kmax + c] = rm;
    }
    eta[p] = e;
}

__global__ void batch_fill_kernel(double* p, double v, i64 count) {
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (i64)gridDim.x * blockDim.x) p[i] = v;
}

// refinement bookkeeping: mark converged matrices, scale residuals to float
__global__ void batch_ir_prepare_kernel(BatchArgs a, const double* eta, double tol, const double* R,
                                        const double* rscale, float* Rf, int kmax, int* iters) {
    const int p = blockIdx.x;
    if (a.skip[p]) return;
    if (eta[p] <= tol) {  // uniform across the workgroup
        if (threadIdx.x == 0) a.skip[p] = 1;
        return;
    }
    if (threadIdx.x == 0) iters[p] += 1;
    const int n = a.n[p], k = a.k[p];
    for (int c = 0; c < k; ++c) {
        const double sc = rscale[(i64)p * kmax + c];
        for (int i = threadIdx.x; i < n; i += blockDim.x) {
            const i64 e = a.b_off[p] + i + (i64)c * n;
            Rf[e] = (float)(sc > 0.0 ? R[e] / sc : 0.0);
        }
    }
}

__global__ void batch_ir_update_kernel(BatchArgs a, const float* D, const double* rscale, double* X, int kmax) {
    const int p = blockIdx.x;
    if (a.skip[p]) return;
    const int n = a.n[p], k = a.k[p];
    for (int c = 0; c < k; ++c) {
        const double sc = rscale[(i64)p * kmax + c];
        for (int i = threadIdx.x; i < n; i += blockDim.x) {
            const i64 e = a.b_off[p] + i + (i64)c * n;
            X[e] += sc * (double)D[e];
        }
    }
}

// dst_i := src_i (FP64), fdst_i := float(src_i), or dst_i := 0 when src is null
__global__ void batch_copy_kernel(BatchArgs a, const double* src, double* dst, float* fdst) {
    const int p = blockIdx.x;
    const int n = a.n[p], k = a.k[p];
    const i64 o = a.b_off[p];
    for (i64 e = threadIdx.x; e < (i64)n * k; e += blockDim.x) {
        if (src == nullptr) dst[o + e] = 0.0;
        else if (fdst != nullptr) fdst[o + e] = (float)src[o + e];
        else dst[o + e] = src[o + e];
    }
}

// ------------------------------------------------------------ launchers
hipError_t batch_potrf(const BatchArgs& a, void* A, bool f32, int step, int nb, int cnt, hipStream_t s) {
    if (cnt <= 0) return hipSuccess;
    if (f32) hipLaunchKernelGGL(batch_potrf_kernel<float>, dim3(cnt), dim3(512), 0, s, a, (float*)A, step, nb);
    else hipLaunchKernelGGL(batch_potrf_kernel<double>, dim3(cnt), dim3(512), 0, s, a, (double*)A, step, nb);
    return hipGetLastError();
}

hipError_t batch_trsm(const BatchArgs& a, void* A, bool f32, int step, int nb, const int* prefix, int cnt, int wgs,
                      hipStream_t s) {
    if (wgs <= 0) return hipSuccess;
    if (f32)
        hipLaunchKernelGGL(batch_trsm_kernel<float>, dim3(wgs), dim3(256), 0, s, a, (float*)A, step, nb, prefix, cnt);
    else
        hipLaunchKernelGGL(batch_trsm_kernel<double>, dim3(wgs), dim3(256), 0, s, a, (double*)A, step, nb, prefix,
                           cnt);
    return hipGetLastError();
}

hipError_t batch_syrk(const BatchArgs& a, void* A, int mode, int step, int nb, const int* prefix, int cnt, int wgs,
                      hipStream_t s) {
    if (wgs <= 0) return hipSuccess;
    if (mode == 0)
        hipLaunchKernelGGL((batch_syrk_kernel<double, 0>), dim3(wgs), dim3(256), 0, s, a, (double*)A, step, nb, prefix,
                           cnt);
    else if (mode == 1)
        hipLaunchKernelGGL((batch_syrk_kernel<float, 1>), dim3(wgs), dim3(256), 0, s, a, (float*)A, step, nb, prefix,
                           cnt);
    else
        hipLaunchKernelGGL((batch_syrk_kernel<float, 2>), dim3(wgs), dim3(256), 0, s, a, (float*)A, step, nb, prefix,
                           cnt);
    return hipGetLastError();
}

hipError_t batch_persistent(const BatchArgs& a, void* F, int mode, int nb, int* counter, int grid, hipStream_t s) {
    if (a.count <= 0) return hipSuccess;
    if (nb < 1 || nb > kPersistMaxNb || grid < 1) return hipErrorInvalidValue;
    const dim3 g((unsigned)std::min(grid, a.count));
    if (mode == 0)
        hipLaunchKernelGGL((batch_persistent_kernel<double, 0>), g, dim3(256), 0, s, a, (double*)F, nb, counter);
    else if (mode == 1)
        hipLaunchKernelGGL((batch_persistent_kernel<float, 1>), g, dim3(256), 0, s, a, (float*)F, nb, counter);
    else
        hipLaunchKernelGGL((batch_persistent_kernel<float, 2>), g, dim3(256), 0, s, a, (float*)F, nb, counter);
    return hipGetLastError();
}

hipError_t batch_residual(const BatchArgs& a, const double* A, const double* X, const double* B, double* R,
                          const int* prefix, int wgs, double* red, double* eta, double* rscale, int kmax,
                          hipStream_t s, float* S) {
    if (a.count <= 0 || wgs <= 0) return hipSuccess;
    const i64 nred = (i64)a.count * (1 + 3 * kmax);
    hipLaunchKernelGGL(batch_fill_kernel, dim3((unsigned)std::min<i64>(ceil_div(nred, 256), 1024)), dim3(256), 0, s,
                       red, 0.0, nred);
    auto kernel = S != nullptr ? batch_symv_residual_kernel<true> : batch_symv_residual_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(256), 0, s, a, A, X, B, R, prefix, a.count, red, kmax, S);
    hipLaunchKernelGGL(batch_eta_kernel, dim3((unsigned)ceil_div(a.count, 256)), dim3(256), 0, s, a, red, eta, rscale,
                       kmax);
    return hipGetLastError();
}

hipError_t batch_ir_prepare(const BatchArgs& a, const double* eta, double tol, const double* R, const double* rscale,
                            float* Rf, int kmax, int* iters, hipStream_t s) {
    if (a.count <= 0) return hipSuccess;
    hipLaunchKernelGGL(batch_ir_prepare_kernel, dim3(a.count), dim3(256), 0, s, a, eta, tol, R, rscale, Rf, kmax,
                       iters);
    return hipGetLastError();
}

hipError_t batch_ir_update(const BatchArgs& a, const float* D, const double* rscale, double* X, int kmax,
                           hipStream_t s) {
    if (a.count <= 0) return hipSuccess;
    hipLaunchKernelGGL(batch_ir_update_kernel, dim3(a.count), dim3(256), 0, s, a, D, rscale, X, kmax);
    return hipGetLastError();
}

hipError_t batch_copy_rhs(const BatchArgs& a, const double* src, double* dst, float* fdst, hipStream_t s) {
    if (a.count <= 0) return hipSuccess;
    hipLaunchKernelGGL(batch_copy_kernel, dim3(a.count), dim3(256), 0, s, a, src, dst, fdst);
    return hipGetLastError();
}

}  // namespace elemamd
