// Products and updates in 64 x 64 tiles of C, four waves of 32 x 32 or eight
// of 32 x 16, K in chunks of KC staged through LDS.
//
// What bounds them: with few tiles every chunk waits out a memory latency
// (about 1 us), so small tiles spread the work over the CUs and a chunk's
// loads are all issued at once, under the MFMAs of the chunk before.  With
// many tiles the FP64 MFMA pipe (64 cycles per 16x16x4): several workgroups
// share a CU (20 KB of LDS and about 100 registers each) and fill each
// other's load, store and barrier phases.  Addresses cost no vector work
// inside the loop: rows past the edge are clamped once (their products fall
// on entries of C that are not stored), and loads step from column to column.
#pragma once

#include "common.hpp"
#include "solve_dev.hpp"

namespace elemamd {
namespace tile64 {

constexpr int kTile = 64;
constexpr int kLd = kTile + 16;  // LDS row stride of a chunk [k][row]: an MFMA operand's k rows start on other banks

template <typename T, int KC, int LD = kLd>
struct Smem {
    T I[KC][LD], J[KC][LD];
};

// What an operand without columns reads in their place.
static __device__ double kNoColumn[1] = {};

// One operand, rows x0 .. x0 + 63 of an ext x k matrix with element (x, l) at
// M[x + l ld], KC columns per chunk, DEPTH chunks on their way, loaded by NW
// waves.  load() has no branches (columns past k repeat an earlier one), so the
// compiler waits for the chunk it needs and not for the ones behind it.
template <typename T, int KC, int DEPTH = 1, int NW = 4>
struct RowLoader {
    static constexpr int kDepth = DEPTH, kW = NW;
    const T* p;  // this thread's row (clamped), the column to load next
    i64 step;
    int k, l0, next;
    T g[DEPTH][KC / NW];
    __device__ __forceinline__ RowLoader(const T* M, i64 ld, int ext, int k_, int x0)
        : step(NW * ld), k(k_), l0(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)), next(l0) {
        const int x = x0 + (int)(threadIdx.x & 63);
        p = k > 0 ? M + (x < ext ? x : ext - 1) + (i64)min(l0, k - 1) * ld : (const T*)kNoColumn;
    }
    __device__ __forceinline__ void load(int d = 0) {  // the next chunk, into slot d
#pragma unroll
        for (int q = 0; q < KC / NW; ++q) {
            g[d][q] = *p;
            next += NW;
            p += next < k ? step : 0;
        }
    }
    template <typename Row>
    __device__ __forceinline__ void store(Row* s, T scale, int k0, int d = 0) const {
        if (k0 + KC <= k) {
#pragma unroll
            for (int q = 0; q < KC / NW; ++q) s[l0 + NW * q][threadIdx.x & 63] = scale * g[d][q];
        } else {
#pragma unroll
            for (int q = 0; q < KC / NW; ++q)
                s[l0 + NW * q][threadIdx.x & 63] = k0 + l0 + NW * q < k ? scale * g[d][q] : T(0);
        }
    }
};

// Tile (i0, j0) of C := beta C + alpha I J^T by the calling workgroup of the
// loaders' NW waves (C m x n).  tri: 0 the whole tile, 1 entries j <= i, 2
// entries i <= j.  beta == 1: C is read under the first chunk's loads, and with
// FROM_C (the FP64 factorizations) the accumulators start from it; otherwise
// they start from zero and C is added at the end (fewer roundings at C's size:
// the n = 3000 inverse's error against 64 bits is 4.4 times larger with it).
// beta == 0: C is not read.
template <bool FROM_C, typename T, int KC, int LD, typename LI, typename LJ>
__device__ __forceinline__ void tile(Smem<T, KC, LD>& sm, LI& li, LJ& lj, int i0, int j0, int m, int n, int k, T alpha,
                                     T beta, T* __restrict__ C, i64 ldc, int tri) {
    typedef typename Acc4<T>::type acc_t;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c16 = lane & 15, g = lane >> 4;
    constexpr int NW = LI::kW, NA = 8 / NW;  // waves, 16-column tiles of a wave
    const int wj = (w >> 1) * 16 * NA, wi = (w & 1) * 32;
    const bool skip = i0 == j0 && ((tri == 1 && wj >= wi + 32) || (tri == 2 && wi >= wj + 16 * NA));
    const bool acc_c = beta == T(1);
    // the thread's entries: rows i + 16 b, columns j + 16 a + jv v; a whole tile
    // off the diagonal needs no masks
    const int i = i0 + wi + c16, j = j0 + wj + mfma_row<T>(lane, 0), jv = mfma_row<T>(0, 1);
    T* const Ct = C + i + (i64)j * ldc;
    const bool whole = i0 + kTile <= m && j0 + kTile <= n && (tri == 0 || i0 != j0);
    auto in = [&](int a, int b, int v) __attribute__((always_inline)) {
        const int r = i + 16 * b, c = j + 16 * a + jv * v;
        return r < m && c < n && (tri == 0 || (tri == 1 ? c <= r : r <= c));
    };
    constexpr int DEPTH = LI::kDepth;
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        li.load(d);
        lj.load(d);
    }
    acc_t acc[NA][2], pre[NA][2] = {};
    if (acc_c && whole) {
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const T* c = Ct + (i64)(16 * a + jv * v) * ldc;
#pragma unroll
                for (int b = 0; b < 2; ++b) pre[a][b][v] = c[16 * b];
            }
    } else if (acc_c && !skip) {
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int b = 0; b < 2; ++b)
                    if (in(a, b, v)) pre[a][b][v] = Ct[16 * b + (i64)(16 * a + jv * v) * ldc];
    }
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[a][b][v] = FROM_C ? pre[a][b][v] : T(0);
    const T scale = (FROM_C && acc_c) ? alpha : T(1);
    for (int k1 = 0; k1 < k; k1 += DEPTH * KC) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            const int k0 = k1 + d * KC;
            if (k0 >= k) break;
            li.store(sm.I, T(1), k0, d);
            lj.store(sm.J, scale, k0, d);
            __syncthreads();
            li.load(d);
            lj.load(d);
            if (!skip) {
#pragma unroll
                for (int ks = 0; ks < KC / 4; ++ks) {
                    const int kr = 4 * ks + g;
                    T fa[NA], fb[2];
#pragma unroll
                    for (int a = 0; a < NA; ++a) fa[a] = sm.J[kr][wj + 16 * a + c16];
#pragma unroll
                    for (int b = 0; b < 2; ++b) fb[b] = sm.I[kr][wi + 16 * b + c16];
#pragma unroll
                    for (int a = 0; a < NA; ++a)
#pragma unroll
                        for (int b = 0; b < 2; ++b) acc[a][b] = mfma16(fa[a], fb[b], acc[a][b]);
                }
            }
            __syncthreads();
        }
    }
    if (skip) return;
    // dependent zero-operand MFMAs before the accumulators are read (the
    // compiler's wait states after a loop back edge are short for FP64 MFMA)
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = mfma16(T(0), T(0), acc[a][b]);
    if (acc_c) {
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if constexpr (!FROM_C) acc[a][b][v] = pre[a][b][v] + alpha * acc[a][b][v];
        if (whole) {
#pragma unroll
            for (int a = 0; a < NA; ++a)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    T* c = Ct + (i64)(16 * a + jv * v) * ldc;
#pragma unroll
                    for (int b = 0; b < 2; ++b) c[16 * b] = acc[a][b][v];
                }
        } else {
#pragma unroll
            for (int a = 0; a < NA; ++a)
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int b = 0; b < 2; ++b)
                        if (in(a, b, v)) Ct[16 * b + (i64)(16 * a + jv * v) * ldc] = acc[a][b][v];
        }
        return;
    }
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                if (!in(a, b, v)) continue;
                T* c = Ct + 16 * b + (i64)(16 * a + jv * v) * ldc;
                *c = beta == T(0) ? alpha * acc[a][b][v] : beta * *c + alpha * acc[a][b][v];
            }
}

}  // namespace tile64
}  // namespace elemamd
