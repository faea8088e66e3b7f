// Products and updates in 64 x 64 tiles of C, four waves of 32 x 32, K in
// chunks of KC staged through LDS.
//
// What bounds them: with few tiles every chunk waits out a memory latency
// (about 1 us), so small tiles spread the work over the CUs and a chunk's
// loads are all issued at once, under the MFMAs of the chunk before.  With
// many tiles the FP64 MFMA pipe (64 cycles per 16x16x4): several workgroups
// share a CU (20 KB of LDS and about 100 registers each) and fill each
// other's load, store and barrier phases.  Addresses cost no vector work
// inside the loop: rows past the edge are clamped once (their products fall
// on entries of C that are not stored), the k tail alone is masked.
#pragma once

#include "common.hpp"
#include "solve_dev.hpp"

namespace elemamd {
namespace tile64 {

constexpr int kTile = 64;
constexpr int kLd = kTile + 16;  // LDS row stride of a chunk [k][row]: an MFMA operand's k rows start on other banks

template <typename T, int KC>
struct Smem {
    T I[KC][kLd], J[KC][kLd];
};

// One operand, rows x0 .. x0 + 63 of an ext x k matrix with element (x, l) at
// M[x + l ld], KC columns per chunk.
template <typename T, int KC>
struct RowLoader {
    const T* p;  // this thread's row (clamped), first column
    i64 ld;
    int k, l0;
    T g[KC / 4];
    __device__ __forceinline__ RowLoader(const T* M, i64 ld_, int ext, int k_, int x0)
        : ld(ld_), k(k_), l0(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) {
        const int x = x0 + (int)(threadIdx.x & 63);
        p = M + (x < ext ? x : ext - 1);
    }
    __device__ __forceinline__ void load(int k0) {
        if (k0 >= k) return;  // (k = 0: nothing may be read)
        if (k0 + KC <= k) {
#pragma unroll
            for (int q = 0; q < KC / 4; ++q) g[q] = p[(i64)(k0 + l0 + 4 * q) * ld];
        } else {
#pragma unroll
            for (int q = 0; q < KC / 4; ++q) {
                const int l = k0 + l0 + 4 * q;
                const T v = p[(i64)(l < k ? l : 0) * ld];
                g[q] = l < k ? v : T(0);
            }
        }
    }
    __device__ __forceinline__ void store(T (*s)[kLd], T scale) const {
#pragma unroll
        for (int q = 0; q < KC / 4; ++q) s[l0 + 4 * q][threadIdx.x & 63] = scale * g[q];
    }
};

// Tile (i0, j0) of C := beta C + alpha I J^T by the calling 256-thread
// workgroup (C m x n).  tri: 0 the whole tile, 1 entries j <= i, 2 entries
// i <= j.  beta == 1 (the factorizations): C is read under the first chunk's
// loads, and in FP64 the accumulators start from it (in FP32 they start from
// zero and C is added at the end: fewer roundings at C's size); beta == 0: C
// is not read.
template <typename T, int KC, typename LI, typename LJ>
__device__ __forceinline__ void tile(Smem<T, KC>& sm, LI& li, LJ& lj, int i0, int j0, int m, int n, int k, T alpha,
                                     T beta, T* __restrict__ C, i64 ldc, int tri) {
    typedef typename Acc4<T>::type acc_t;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c16 = lane & 15, g = lane >> 4;
    const int wj = (w >> 1) * 32, wi = (w & 1) * 32;
    const bool skip = i0 == j0 && ((tri == 1 && wj > wi) || (tri == 2 && wi > wj));
    constexpr bool kFromC = sizeof(T) == 8;
    const bool acc_c = beta == T(1);
    auto in = [&](int i, int j) { return i < m && j < n && (tri == 0 || (tri == 1 ? j <= i : i <= j)); };
    li.load(0);
    lj.load(0);
    acc_t acc[2][2], pre[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = i0 + wi + 16 * b + c16, j = j0 + wj + 16 * a + mfma_row<T>(lane, v);
                pre[a][b][v] = (acc_c && !skip && in(i, j)) ? C[i + (i64)j * ldc] : T(0);
                acc[a][b][v] = kFromC ? pre[a][b][v] : T(0);
            }
    const T scale = (kFromC && acc_c) ? alpha : T(1);
    for (int k0 = 0; k0 < k; k0 += KC) {
        li.store(sm.I, T(1));
        lj.store(sm.J, scale);
        __syncthreads();
        if (k0 + KC < k) {
            li.load(k0 + KC);
            lj.load(k0 + KC);
        }
        if (!skip) {
#pragma unroll
            for (int ks = 0; ks < KC / 4; ++ks) {
                const int kr = 4 * ks + g;
                T fa[2], fb[2];
#pragma unroll
                for (int a = 0; a < 2; ++a) fa[a] = sm.J[kr][wj + 16 * a + c16];
#pragma unroll
                for (int b = 0; b < 2; ++b) fb[b] = sm.I[kr][wi + 16 * b + c16];
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int b = 0; b < 2; ++b) acc[a][b] = mfma16(fa[a], fb[b], acc[a][b]);
            }
        }
        __syncthreads();
    }
    if (skip) return;
    // dependent zero-operand MFMAs before the accumulators are read (the
    // compiler's wait states after a loop back edge are short for FP64 MFMA)
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = mfma16(T(0), T(0), acc[a][b]);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = i0 + wi + 16 * b + c16, j = j0 + wj + 16 * a + mfma_row<T>(lane, v);
                if (!in(i, j)) continue;
                T* p = C + i + (i64)j * ldc;
                if (acc_c) *p = kFromC ? acc[a][b][v] : pre[a][b][v] + alpha * acc[a][b][v];
                else *p = beta == T(0) ? alpha * acc[a][b][v] : beta * *p + alpha * acc[a][b][v];
            }
}

}  // namespace tile64
}  // namespace elemamd
