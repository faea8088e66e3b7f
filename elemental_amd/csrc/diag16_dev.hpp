// Cholesky of a diagonal block of up to 128 columns by one workgroup, in
// 16-column pieces held in registers: the diagonal factor of the blocked
// factorizations (LVar3Unb's role in cholesky::LVar3,
// include/elemental/lapack-like/Cholesky/LVar3.hpp:83-123).
//
// What bounds it: the chain of 128 pivots, each a reciprocal square root, a
// scaling and the next column's update, and one wave's issue rate (measured
// cycles from one wave: FP64 FMA 5, dependent 8, with a DPP operand 8,
// reciprocal root 20, FP64 MFMA 16x16x4 64, so MFMA has no more throughput
// than FMA here).  A piece takes about 5500 cycles: 3500 for its 16 columns,
// 1200 for the tiles below, 700 for the next diagonal tile.  So the columns
// of a piece are factored without leaving one wave's registers, and
// everything else of the block runs beside that wave:
//  * wave w owns tile row w of the block, 16 x 16 tiles t[J] (J <= w) in the
//    FP64 MFMA accumulator layout: lane (c, g) = (lane % 16, lane / 16) holds
//    rows g + 4v (v = 0..3) of column c;
//  * wave p holds piece p's diagonal tile by rows (lane i of each 16-lane row:
//    row i, all 16 columns).  A rank-1 update's broadcast operand comes from a
//    lane of the same 16-lane row, which v_fmac_f64 reads through DPP
//    row_newbcast: one instruction per column, no LDS and no lane reads;
//  * the waves below then solve their tile of the piece (the same broadcast,
//    64 instructions), the solved tiles go through LDS into MFMA operand
//    order, and wave p + 1 updates its diagonal tile and goes on with piece
//    p + 1 while the others update theirs.  Two barriers a piece.
// The pivot's reciprocal root is the hardware estimate with a third-order
// correction, exact for powers of four (integer problems stay exact).
//
// A pivot that is not a positive finite number sends its piece through
// piece_careful(), which follows LVar3Unb's columns in LDS with real square
// roots and divisions: +infinity goes on as in the reference loop, and a
// failing column leaves the reference's state (columns before it factored,
// the trailing triangle updated by them).  So does every piece of a
// block that holds an infinity or NaN off its diagonal tiles: the tiles'
// substitution would let it into the row's earlier columns (zero times
// infinity).  The waves look for one while the first piece is factored.
#pragma once

#include "common.hpp"
#include "solve_dev.hpp"

namespace elemamd {
namespace diag16 {

constexpr int kWaves = 8;             // tile rows of a 128-column block
constexpr int kThreads = 64 * kWaves;
constexpr int kXLd = 130;             // LDS column stride of the solved tiles (rows of the block)

template <bool INV>
struct Lds {
    static constexpr int kV = INV ? kWaves : 2;  // without the inverses two diagonal tiles alternate
    double X[16][kXLd];        // the piece's solved tiles, [column of the piece][row of the block]
    double D[16][18];          // the diagonal tile before its factorization, by rows
    double M[16][18];          // [c][k]: l_ck / l_kk for c > k, else 0 (the piece's multipliers)
    double V[kV][16][17];      // wave w, [w % kV]: its diagonal tile's unscaled columns [column][row]; then its inverse (INV)
    int bad;                   // bit 0: this piece goes through piece_careful(), bit 1: every piece
};

// acc -= (lane N of the 16-lane row's x) * l.  The DPP operand needs two wait
// states after its last write; callers keep that distance.
template <int N>
__device__ __forceinline__ void fnma_bcast(double& acc, double x, double l) {
    asm volatile("v_fmac_f64_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                 : "+v"(acc)
                 : "v"(x), "v"(l), "n"(N));
}
// acc[v] -= (lane N of acc[v]) * l for the wave's tile
template <int N>
__device__ __forceinline__ void fnma_bcast_self(double& acc, double l) {
    asm volatile("v_fmac_f64_dpp %0, -%0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(l), "n"(N));
}
template <int N, bool WAIT = true>
__device__ __forceinline__ double bcast(double x) {
    double r;
    if constexpr (WAIT)
        asm volatile("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
                     : "=v"(r)
                     : "v"(x), "n"(N));
    else  // two instructions lie between the write of x and this
        asm volatile("v_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(r) : "v"(x), "n"(N));
    return r;
}

// 1 / sqrt(d): hardware estimate (2^-24 or so), third-order correction, one
// instruction per step.  The steps are volatile so that they stay where the
// column loop puts them, between the updates that hide their latency (left to
// itself the compiler runs them one after the other behind all updates).  A
// transcendental's result needs one instruction before its use.
__device__ __forceinline__ double rsq_estimate(double d) {
    double y;
    asm volatile("v_rsq_f64 %0, %1" : "=v"(y) : "v"(d));
    return y;
}
__device__ __forceinline__ double rsqrt_full(double d) {
    const double y = __builtin_amdgcn_rsq(d);
    const double h = fma(-(d * y), y, 1.0);
    return fma(y * h, fma(h, 0.375, 0.5), y);
}
__device__ __forceinline__ double mul_here(double a, double b) {
    double r;
    asm volatile("v_mul_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double fnma_one_here(double a, double b) {  // 1 - a b
    double r;
    asm volatile("v_fma_f64 %0, -%1, %2, 1.0" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double fnma_here(double a, double c) {  // c - a a
    double r;
    asm volatile("v_fma_f64 %0, -%1, %1, %2" : "=v"(r) : "v"(a), "v"(c));
    return r;
}
__device__ __forceinline__ double fma_half_here(double a, double b) {  // a b + 1/2
    double r;
    asm volatile("v_fma_f64 %0, %1, %2, 0.5" : "=v"(r) : "v"(a), "s"(b));
    return r;
}
__device__ __forceinline__ double fma_here(double a, double b, double c) {
    double r;
    asm volatile("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// d[C] -= l_C l of the diagonal tile, C = FROM .. TO - 1 (below 16).
template <int FROM, int TO>
__device__ __forceinline__ void update_cols(double (&d)[16], double l) {
    if constexpr (FROM < TO && FROM < 16) {
        fnma_bcast<FROM>(d[FROM], l, l);
        update_cols<FROM + 1, TO>(d, l);
    }
}

// Columns K .. 15 of the piece; r is pivot K's reciprocal root.  The chain
// from one root to the next does not wait for the columns' updates: pivot
// K + 1 is z - (x r)^2 with x = a_(K+1,K) and z = a_(K+1,K+1) broadcast
// beforehand (the same operations, and bits, as lane K + 1's own update).
// The unscaled column and the multipliers go to LDS as they appear, so no
// column stays in registers once it is applied.
template <int K>
struct Column {
    static __device__ __forceinline__ void run(double (&d)[16], double r, int i, bool& good, double (*M)[18],
                                               double (*V)[17]) {
        V[K][i] = d[K];
        if constexpr (K < 15) {
            const double x = bcast<K + 1, false>(d[K]);
            const double z = bcast<K + 1, false>(d[K + 1]);
            const double l = mul_here(d[K], r);
            const double xr = mul_here(x, r);
            const double lr = mul_here(l, r);
            const double next = fnma_here(xr, z);
            fnma_bcast<K + 1>(d[K + 1], l, l);
            const double y = rsq_estimate(next);
            good = good && __builtin_amdgcn_class(next, 0x180);  // positive, not infinite, not NaN
            update_cols<K + 2, K + 5>(d, l);
            const double ty = mul_here(next, y);
            update_cols<K + 5, K + 7>(d, l);
            const double h = fnma_one_here(ty, y);
            update_cols<K + 7, K + 9>(d, l);
            const double e = mul_here(y, h);
            const double q = fma_half_here(h, 0.375);
            update_cols<K + 9, K + 11>(d, l);
            const double rn = fma_here(e, q, y);
            update_cols<K + 11, 16>(d, l);
            int k = K;  // opaque: 15 hoisted lane masks would not fit the scalar registers
            asm volatile("" : "+s"(k));
            M[i][K] = i > k ? lr : 0.0;
            Column<K + 1>::run(d, rn, i, good, M, V);
        }
    }
};

// The wave's tile of the piece, a := a L^{-T} up to the scaling by the
// reciprocal diagonal: column K's entries, times the multipliers m[K], from
// the later columns.
template <int K>
struct TileColumn {
    static __device__ __forceinline__ void run(double (&a)[4], const double (&m)[16]) {
        fnma_bcast_self<K>(a[0], m[K]);
        fnma_bcast_self<K>(a[1], m[K]);
        fnma_bcast_self<K>(a[2], m[K]);
        fnma_bcast_self<K>(a[3], m[K]);
        if constexpr (K < 14) TileColumn<K + 1>::run(a, m);
    }
};

// Inverse of the 16 x 16 factor held by rows (d, reciprocal diagonal rv):
// lane c ends with column c in x[0..15].
template <int I, int M>
struct InvRest {
    static __device__ __forceinline__ void run(double (&x)[16], const double (&d)[16]) {
        fnma_bcast<M>(x[M], d[I], x[I]);
        InvRest<I, M + 1>::run(x, d);
    }
};
template <int I>
struct InvRest<I, 16> {
    static __device__ __forceinline__ void run(double (&)[16], const double (&)[16]) {}
};
template <int I>
struct InvCol {
    static __device__ __forceinline__ void run(double (&x)[16], const double (&d)[16], double rv) {
        x[I] *= bcast<I>(rv);
        InvRest<I, I + 1>::run(x, d);
        InvCol<I + 1>::run(x, d, rv);
    }
};
template <>
struct InvCol<16> {
    static __device__ __forceinline__ void run(double (&)[16], const double (&)[16], double) {}
};

// Piece p once more, by LVar3Unb's columns: the diagonal tile (sh.D) and the
// rows below it (already stored unsolved in sh.X), all threads.  Returns the
// 0-based failing column of the piece, or 16.  On return sh.X holds the
// piece's columns (the diagonal tile's rows among them), columns from the
// failing one on as they stood when it failed.
template <bool INV>
__device__ __forceinline__ int piece_careful(Lds<INV>& sh, int p, int nrows) {
#pragma clang fp contract(off)
    const int t = threadIdx.x, r0 = 16 * p, row = r0 + t;
    if (t < 16)
#pragma unroll 1
        for (int c = 0; c < 16; ++c) sh.X[c][row] = sh.D[t][c];
    __syncthreads();
#pragma unroll 1
    for (int k = 0; k < 16; ++k) {
        const double ajj = sh.X[k][r0 + k];
        if (!(ajj > 0.0)) return k;
        const double alpha = sqrt(ajj);
        __syncthreads();
        if (row < nrows && t >= k) sh.X[k][row] = t == k ? alpha : sh.X[k][row] / alpha;
        __syncthreads();
        if (row < nrows)
#pragma unroll 1
            for (int c = k + 1; c < 16 && c <= t; ++c) sh.X[c][row] = sh.X[c][row] - sh.X[k][row] * sh.X[k][r0 + c];
        __syncthreads();
    }
    return 16;
}

// The b x b (b <= 128) block at A, lower triangle, by the calling workgroup
// of 64 NW threads; storage T, arithmetic FP64.  NW = 4: wave w owns the tile
// rows w and w + 4, with the same operations (and bits) as NW = 8.  A failing pivot records
// col_offset + column (1-based) in *info.  INV: the inverses of the block's
// 32 x 32 diagonal pieces also go to Xd (4 x 32 x 32, row-major).
template <typename T, bool INV, int NW = kWaves>
__device__ __forceinline__ void factor_block(Lds<INV>& sh, int b, T* __restrict__ A, i64 lda, float* __restrict__ Xd,
                                             int* __restrict__ info, int col_offset) {
    static_assert(NW == kWaves || (2 * NW == kWaves && !INV), "tile rows per wave");
    constexpr int NR = kWaves / NW;  // tile rows of a wave: w0, w0 + NW
    const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
    const int w0 = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int np = (b + 15) / 16;
    const bool full = b == 16 * kWaves;
    if (tid == 0) sh.bad = 0;
    if (np > 1) __syncthreads();  // (before another wave sets it)
    // tile row w, tiles 0 .. w (zero past b, the padded diagonal one; the
    // diagonal tile whole, mirrored).  16 rows by 4 columns per load, whole
    // lines (with lanes along columns every lane is an access of its own, 64
    // cycles a load, 7 us in all), then turned through the wave's part of sh.X.
    d4_t t[NR][kWaves];  // (row r has no tiles from NW (r + 1) on)
    {
        T raw[NR][kWaves][4];
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int w = w0 + NW * r;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = 16 * w + g + 4 * v, j = 16 * w + c;
                const int row = min(max(i, j), b - 1), col = min(min(i, j), b - 1);
                raw[r][kWaves - 1][v] = A[row + (i64)col * lda];
            }
            if (full) {  // addresses by steps
                const T* q = A + 16 * w + c + (i64)g * lda;
#pragma unroll
                for (int J = 0; J < NW * (r + 1) - 1; ++J)
                    if (J < w)
#pragma unroll
                        for (int v = 0; v < 4; ++v, q += 4 * lda) raw[r][J][v] = *q;
            } else {
#pragma unroll
                for (int J = 0; J < NW * (r + 1) - 1; ++J)
                    if (J < w)
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            raw[r][J][v] = A[min(16 * w + c, b - 1) + (i64)min(16 * J + g + 4 * v, b - 1) * lda];
            }
        }
        double(*sx)[16] = reinterpret_cast<double(*)[16]>(&sh.X[0][0] + 256 * w0);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int w = w0 + NW * r;
#pragma unroll
            for (int J = 0; J < NW * (r + 1); ++J) {
                if (J < w && J < NW * (r + 1) - 1) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) sx[c][(g + 4 * v) ^ c] = (double)raw[r][J][v];
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int v = 0; v < 4; ++v) t[r][J][v] = sx[g + 4 * v][c ^ (g + 4 * v)];
                    __builtin_amdgcn_wave_barrier();
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v) t[r][J][v] = (double)raw[r][kWaves - 1][v];
                }
            }
        }
    }
    if (b < 16 * kWaves)
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
            for (int J = 0; J < NW * (r + 1); ++J)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int i = 16 * (w0 + NW * r) + g + 4 * v, j = 16 * J + c;
                    if (i >= b || j >= b) t[r][J][v] = i == j ? 1.0 : 0.0;
                }
    bool odd = false;
    if (np > 1) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
            for (int J = 0; J < NW * (r + 1) - 1; ++J)
                if (J < w0 + NW * r)
#pragma unroll
                    for (int v = 0; v < 4; ++v) odd = odd | __builtin_amdgcn_class(t[r][J][v], 0x207);
    }
    if (__ballot(odd) != 0 && lane == 0) atomicOr(&sh.bad, 2);
    if (w0 == 0) {
#pragma unroll
        for (int v = 0; v < 4; ++v) sh.D[g + 4 * v][c] = t[0][0][v];
        __builtin_amdgcn_wave_barrier();
    }
    // tile (w, q) of the factor, from its rows of sh.X
    auto store_tile = [&](int w, int q) __attribute__((always_inline)) {
        // (opaque lane: the addresses are made here, not kept in registers
        // across the loop)
        int lv = lane;
        asm volatile("" : "+v"(lv));
        const int cs = lv & 15, gs = lv >> 4, row = 16 * w + cs;
        if (full) {
            T* to = A + row + (i64)(16 * q + gs) * lda;
#pragma unroll
            for (int v = 0; v < 4; ++v, to += 4 * lda) *to = (T)sh.X[gs + 4 * v][row];
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int col = 16 * q + gs + 4 * v;
                if (row < b && col < b) A[row + (i64)col * lda] = (T)sh.X[gs + 4 * v][row];
            }
        }
    };
    int failed = 0;  // 1-based failing column of the block
    for (int p = 0; p < np; ++p) {
        const bool mine = w0 == p % NW;  // piece p's diagonal tile is this wave's
        if (mine) {
            __builtin_amdgcn_s_setprio(3);
            int lv = lane;  // (opaque, as in store_tile)
            asm volatile("" : "+v"(lv));
            const int c = lv & 15;
            double d[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) d[q] = sh.D[c][q];
            const double piv = bcast<0>(d[0]);
            bool good = __builtin_amdgcn_class(piv, 0x180);
            Column<0>::run(d, rsqrt_full(piv), c, good, sh.M, sh.V[p % Lds<INV>::kV]);
            if (!good && lane == 0) atomicOr(&sh.bad, 1);
            __builtin_amdgcn_s_setprio(2);
        }
        if (p > 0)  // t[r][0]: this piece's tile
#pragma unroll
            for (int r = 0; r < NR; ++r)
#pragma unroll
                for (int J = 0; J + 1 < NW * (r + 1); ++J) t[r][J] = t[r][J + 1];
        __syncthreads();
        int kend = 16;  // columns of the piece that were factored
        const bool careful = sh.bad != 0;
        if (!careful) {
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const int w = w0 + NW * r;
                if (w > p && w < np) {
                    double m[16], a[4] = {t[r][0][0], t[r][0][1], t[r][0][2], t[r][0][3]};
#pragma unroll
                    for (int k = 0; k < 16; ++k) m[k] = sh.M[c][k];  // (the last one is not used)
                    const double rv = rsqrt_full(sh.V[p % Lds<INV>::kV][c][c]);
                    // (the copies above end two wait states before the first DPP read)
                    asm volatile("s_nop 1" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]));
                    TileColumn<0>::run(a, m);
#pragma unroll
                    for (int v = 0; v < 4; ++v) sh.X[c][16 * w + g + 4 * v] = a[v] * rv;
                }
            }
            __syncthreads();
        } else {
#pragma unroll
            for (int r = 0; r < NR; ++r)
                if (w0 + NW * r > p)
#pragma unroll
                    for (int v = 0; v < 4; ++v) sh.X[c][16 * (w0 + NW * r) + g + 4 * v] = t[r][0][v];
            if (mine && p > 0) store_tile(p, p - 1);
            // (with INV, tile (p, p-1), whose rows piece_careful() takes, comes
            // back afterwards, since the end needs it; sh.M is free here)
            int lk = lane;  // (opaque, as in store_tile)
            asm volatile("" : "+v"(lk));
            if (INV && mine)
#pragma unroll 1
                for (int q = lk >> 4; q < 16; q += 4) sh.M[q][lk & 15] = sh.X[q][16 * p + (lk & 15)];
            __syncthreads();
            if (tid == 0) atomicAnd(&sh.bad, 2);
            kend = piece_careful(sh, p, 16 * np);
            if (kend < 16) failed = 16 * p + kend + 1;
            if (mine) {
#pragma unroll 1
                for (int q = 0; q < 16; ++q) sh.V[p % Lds<INV>::kV][q][c] = sh.X[q][16 * p + c];
                __builtin_amdgcn_wave_barrier();
                if (INV && !failed)  // (a failing piece's pivot may still be read; nothing needs the tile then)
#pragma unroll 1
                    for (int q = lk >> 4; q < 16; q += 4) sh.X[q][16 * p + (lk & 15)] = sh.M[q][lk & 15];
            }
            if (failed) {
                for (int w = w0; w < np; w += NW)
                    if (w > p) store_tile(w, p);
                __syncthreads();
                // columns from the failing one on update nothing
                if (tid < 128)
#pragma unroll 1
                    for (int q = kend; q < 16; ++q) sh.X[q][tid] = 0.0;
            }
            __syncthreads();
        }
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int w = w0 + NW * r;
            if (w > p && w < np) {
                double fa[4];
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) fa[ks] = -sh.X[4 * ks + g][16 * w + c];
#pragma unroll
                for (int j = 1; j < NW * (r + 1); ++j)
                    if (p + j <= w) {
                        double fb[4];
#pragma unroll
                        for (int ks = 0; ks < 4; ++ks) fb[ks] = sh.X[4 * ks + g][16 * (p + j) + c];
                        mfma_tile(t[r][j], fa, fb);
                    }
                // the solved tile (unsolved columns as they stand); the wave of
                // p + 1 has the next piece to factor first and stores its tile
                // afterwards
                if (w != p + 1 && !failed) store_tile(w, p);
            }
        }
        if (mine) {
            if (p > 0 && !careful) store_tile(p, p - 1);
            // the diagonal tile's columns, scaled by the reciprocal roots; l_kk
            // is the root itself, pivot * r with one correction
            int lv = lane;  // (opaque, as in store_tile)
            asm volatile("" : "+v"(lv));
            const int c = lv & 15, g = lv >> 4;
            double pv = sh.V[p % Lds<INV>::kV][c][c], rv = 1.0;
            if (kend == 16 && !careful) {
                rv = rsqrt_full(pv);
                const double s = pv * rv;
                pv = fma(fma(-s, s, pv), 0.5 * rv, s);
            }
            double l[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = g + 4 * v;
                l[v] = r == c ? pv : sh.V[p % Lds<INV>::kV][c][r] * rv;
                const int row = 16 * p + r, col = 16 * p + c;
                if (row < b && c <= r) A[row + (i64)col * lda] = (T)l[v];
            }
            if constexpr (INV) {
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int v = 0; v < 4; ++v) sh.V[p % Lds<INV>::kV][c][g + 4 * v] = l[v];
            }
        }
        if (failed) {
            // the rest of the block as the failing column left it
            int lv = lane;  // (opaque, as in store_tile)
            asm volatile("" : "+v"(lv));
            const int c = lv & 15, g = lv >> 4;
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const int w = w0 + NW * r;
                if (w > p && w < np)
#pragma unroll
                    for (int J = 1; J < NW * (r + 1); ++J)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const int row = 16 * w + g + 4 * v, col = 16 * (p + J) + c;
                            if (p + J <= w && row < b && col <= row) A[row + (i64)col * lda] = (T)t[r][J][v];
                        }
            }
            if (tid == 0 && info != nullptr) *info = col_offset + failed;
            return;
        }
#pragma unroll
        for (int r = 0; r < NR; ++r)
            if (w0 + NW * r == p + 1) {
#pragma unroll
                for (int v = 0; v < 4; ++v) sh.D[g + 4 * v][c] = t[r][1][v];
                __builtin_amdgcn_wave_barrier();
            }
    }
    if constexpr (INV) {
        const int w = w0;
        __syncthreads();
        // wave w: the inverse of its diagonal tile (the identity past b), then
        // X21 = -X22 (L21 X11) of each 32 x 32 piece by the odd waves
        double x[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) x[q] = q == c ? 1.0 : 0.0;
        if (w < np) {
            double d[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) d[q] = sh.V[w][q][c];
            InvCol<0>::run(x, d, 1.0 / sh.V[w][c][c]);
        }
        __builtin_amdgcn_wave_barrier();
        if (lane < 16)
#pragma unroll
            for (int q = 0; q < 16; ++q) sh.V[w][q][c] = x[q];
        __syncthreads();
        float* Xp = Xd + 1024 * (w >> 1);
        const int h = 16 * (w & 1);
#pragma unroll
        for (int v = 0; v < 4; ++v)
            Xp[(h + g + 4 * v) * 32 + h + c] = (float)sh.V[w][g + 4 * v][c];
        d4_t y = {0.0, 0.0, 0.0, 0.0};
        if ((w & 1) && w < np) {
            // L21 = tile (w, w-1): its rows of sh.X still hold it (a later piece
            // wrote only later rows, or put them back)
            d4_t z = {0.0, 0.0, 0.0, 0.0};
            double fa[4], fb[4];
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) fa[ks] = sh.X[4 * ks + g][16 * w + c], fb[ks] = sh.V[w - 1][4 * ks + g][c];
            mfma_tile(z, fa, fb);
            // the accumulator layout is the operand layout of the next product
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) fa[ks] = -sh.V[w][c][4 * ks + g], fb[ks] = z[ks];
            mfma_tile(y, fa, fb);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if (w & 1) Xp[(16 + g + 4 * v) * 32 + c] = (float)y[v];
            else Xp[(g + 4 * v) * 32 + 16 + c] = 0.0f;
        }
    }
}

}  // namespace diag16
}  // namespace elemamd
