// The panel solve B := B L11^{-T} of the blocked factorizations (single
// matrix FP64, batched; panel_f64.hip describes the method).
#pragma once

#include "common.hpp"
#include "solve_chain_dev.hpp"
#include "solve_dev.hpp"

namespace elemamd {
namespace panel16 {

constexpr int kTiles = 8;  // 16-column tiles of a panel of up to 128 columns (kTiles / 2: of up to 64)

struct Lds {
    double M[kTiles][16][16];  // [tile][k][c]: multipliers l_ck / l_kk (k < c, else 0); [15]: 1 / l_cc
    double X[4][16][16];       // wave w: a tile, [row][column ^ row]
};

// a[v] -= (lane K of the 16-lane row's a[v]) m[K] for K = 0 .. 14
template <int K>
struct TileColumn {
    static __device__ __forceinline__ void run(double (&a)[4], const double (&m)[15]) {
#pragma unroll
        for (int v = 0; v < 4; ++v) chain::self_step<K>(a[v], m[K]);
        if constexpr (K < 14) TileColumn<K + 1>::run(a, m);
    }
};

// Rows [64 slab, 64 slab + 64) of X := B L^{-T} (m x b, b <= 128; X may be B)
// by the calling 256-thread workgroup, storage T (double, or float computed in
// double).  Off: what holds the offset of three columns in bytes.  IDENT: B
// is the identity.  NT: tiles (b <= 16 NT).
template <typename T, typename Off = unsigned, bool IDENT = false, int NT = kTiles>
__device__ __forceinline__ void slab(Lds& sh, int m, int b, const T* __restrict__ L, i64 ldl, const T* B, i64 ldb, T* X,
                                     i64 ldx, int slab) {
    const int t = threadIdx.x, lane = t & 63, c = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int np = (b + 15) / 16;
    // Every load has its address clamped into the matrix and no branch around
    // it, so the compiler waits for exactly the loads it needs.  What is read
    // past b stays in columns past b, which are not stored.
    // The addresses of a full panel's loads and stores are steps from one to
    // the next (a wave alone on its SIMD pays 4 to 8 cycles for every scalar
    // or vector instruction: with a product and clamps per load, loading took
    // 14000 of 36000 cycles).
    const bool full = b == 16 * NT;
    // row c of the diagonal tile w or, of eight and for lanes with g > 1, w + 4
    const int d0 = 16 * (NT > 4 ? w + 4 * (g >> 1) : w), dr = min(d0 + c, b - 1);
    double lm[15];
    {
        T raw[15];
        if (full) {
            const T* p = L + dr + (i64)d0 * ldl;
#pragma unroll
            for (int k = 0; k < 15; ++k, p += ldl) raw[k] = *p;
        } else {
#pragma unroll
            for (int k = 0; k < 15; ++k) raw[k] = L[dr + (i64)min(d0 + k, b - 1) * ldl];
        }
#pragma unroll
        for (int k = 0; k < 15; ++k) lm[k] = (double)raw[k];
    }
    const double dd = (double)L[dr + (i64)dr * ldl];
    const int rw = 64 * slab + 16 * w;  // this wave's first row
    const int last = np - 1;
    // an element at a (32-bit) offset from a scalar address: no vector work
    auto at = [](const T* base, Off offset) __attribute__((always_inline)) {
        return *(const T*)((const char*)base + offset * (Off)sizeof(T));
    };
    // The rows, 16 of them by 4 columns per load (128-byte lines; with lanes
    // along columns every lane is an access of its own, 64 cycles a load), then
    // turned through LDS into lane (c, g): rows g + 4 v of column c.
    const T* Bw = B + min(rw, m - 1);
    const Off rowc = (Off)min(c, max(m - 1 - rw, 0));
    T raw[NT][4];
    if constexpr (IDENT) {
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) raw[q][v] = rw + c == 16 * q + g + 4 * v ? T(1) : T(0);
    } else if (full) {
        const T* p = Bw;
        const Off off = (Off)g * (Off)ldb + rowc;
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v, p += 4 * ldb) raw[q][v] = at(p, off);
    } else {
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                // (a partial tile's last column again in the place of missing ones)
                const int q0 = 16 * min(q, last), end = q < last ? 15 : b - 1 - 16 * last, v0 = 4 * min(v, end / 4);
                raw[q][v] = at(Bw + (i64)(q0 + v0) * ldb, (Off)min(g, end - v0) * (Off)ldb + rowc);
            }
    }
    // operands of the update of tile p by tile q: L(16 p + c, 16 q + 4 ks + g)
    // (a tile that updates others is full)
    const i64 ls = b >= 16 ? ldl : 0;
    Off rowp[NT - 1];
#pragma unroll
    for (int p = 1; p < NT; ++p) rowp[p - 1] = (Off)g * (Off)ls + (Off)min(16 * p + c, b - 1);
    double y[NT - 1][4];
    auto load_y = [&](int p, int q) __attribute__((always_inline)) {
        const T* Lq = L + (i64)(16 * q + 16 <= b ? 16 * q : 0) * ls;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) y[p - 1][ks] = (double)at(Lq + 4 * ks * ls, rowp[p - 1]);
    };
#pragma unroll
    for (int p = 1; p < NT; ++p) load_y(p, 0);
    {
        const double r = 1.0 / dd;
        chain::Multipliers<double, 0>::run(lm, r, c);
        if (NT > 4 ? (g & 1) == 0 : g == 0) {
            double(*M)[16] = sh.M[NT > 4 ? w + 4 * (g >> 1) : w];
#pragma unroll
            for (int k = 0; k < 15; ++k) M[k][c] = lm[k];
            M[15][c] = r;
        }
    }
    d4_t a[NT];
    double(*sx)[16] = sh.X[w];  // (LDS serves a wave's accesses in order; the barriers keep the compiler's)
#pragma unroll
    for (int q = 0; q < NT; ++q) {
#pragma unroll
        for (int v = 0; v < 4; ++v) sx[c][(g + 4 * v) ^ c] = (double)raw[q][v];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int v = 0; v < 4; ++v) a[q][v] = sx[g + 4 * v][c ^ (g + 4 * v)];
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NT; ++q) {
        if (q >= np) break;
        double mk[15], x[4] = {a[q][0], a[q][1], a[q][2], a[q][3]};
#pragma unroll
        for (int k = 0; k < 15; ++k) mk[k] = sh.M[q][k][c];
        const double r = sh.M[q][15][c];
        // (the copies above end two wait states before the first DPP read)
        asm volatile("s_nop 1" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]));
        TileColumn<0>::run(x, mk);
#pragma unroll
        for (int v = 0; v < 4; ++v) a[q][v] = x[v] * r;
        // into MFMA operand order, which is also the order of the stores
#pragma unroll
        for (int v = 0; v < 4; ++v) sx[g + 4 * v][c ^ (g + 4 * v)] = a[q][v];
        __builtin_amdgcn_wave_barrier();
        double fa[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) fa[ks] = sx[c][(4 * ks + g) ^ c];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int v = 0; v < 4; ++v) raw[q][v] = (T)fa[v];
        if (q + 1 >= np) break;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            fa[ks] = -fa[ks];
            asm volatile("" : "+v"(fa[ks]));  // (made once)
        }
#pragma unroll
        for (int p = q + 1; p < NT; ++p) {
            if (p < np) mfma_tile(a[p], fa, y[p - 1]);
            if (p > q + 1) load_y(p, q + 1);
        }
    }
    // (all stores at the end: a load behind a store waits for both)
    if (full && rw + 16 <= m) {
        T* p = X + rw;
        const Off off = (Off)g * (Off)ldx + (Off)c;
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v, p += 4 * ldx) *(T*)((char*)p + off * (Off)sizeof(T)) = raw[q][v];
    } else {
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = rw + c, col = 16 * q + g + 4 * v;
                if (r < m && col < b) X[r + (i64)col * ldx] = raw[q][v];
            }
    }
}

}  // namespace panel16
}  // namespace elemamd
