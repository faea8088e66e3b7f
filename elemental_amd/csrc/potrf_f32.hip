// Panel step of the low-precision (float-storage) factorization: the
// diagonal block L11 = chol(A11) of cholesky::LVar3
// (include/elemental/lapack-like/Cholesky/LVar3.hpp:83-123, LVar3Unb at :19-49)
// and the panel solve L21 := A21 L11^{-T}.  Two kernels:
//
// potrf_f32_kernel -- one workgroup, the block in FP64 registers
//   (diag16_dev.hpp), stored back as float with the inverses of its 32 x 32
//   diagonal pieces.
// panel_f32_kernel -- one 64-row slab per workgroup, with the inverses of
//   the four 32 x 32 diagonal pieces of L11 (by the diagonal-block kernel):
//   each wave solves its 16 rows block by block,
//       X_p = (A_p - sum_{q<p} X_q L_pq^T) inv(L_pp)^T   (FP32 MFMA),
//   with no further synchronisation (the rows are independent).  Products
//   with the 32 x 32 inverses replace the 128-step substitution per row; the
//   refinement absorbs their larger rounding error (this factor only
//   preconditions).  With planes requested the result is also written as
//   bf16 hi/lo planes for the split-BF16x3 updates.
#include "common.hpp"
#include "diag16_dev.hpp"
#include "kernels.hpp"
#include "solve_dev.hpp"

namespace elemamd {

constexpr int kPiLd = 132;  // LDS row stride (floats): MFMA operand reads are conflict-free

// acc[nt] (16 x 16 each) += P (16 x 32) Q^T, nt < 2: rows pr.. of P from column
// pc, rows 16 nt .. of Q, both row-major in LDS; all 24 operand loads are in
// flight together, then the 16 MFMA steps.
template <int LP, int LQ>
__device__ inline void tile_ab_t(f4_t (&acc)[2], const float (*P)[LP], int pr, int pc, const float (*Q)[LQ], int m,
                                 int g) {
    float pa[8], qb[2][8];
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        pa[ks] = P[pr + m][pc + 4 * ks + g];
        qb[0][ks] = Q[m][4 * ks + g];
        qb[1][ks] = Q[16 + m][4 * ks + g];
    }
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
        mfma_acc(acc[0], pa[ks], qb[0][ks]);
        mfma_acc(acc[1], pa[ks], qb[1][ks]);
    }
}

// One b x b (b <= 128) diagonal block at A (float storage): L11 overwrites
// its lower triangle, the inverses of its four 32 x 32 diagonal pieces go to
// Xd (4 x 32 x 32 floats, row-major).  A failing pivot records
// col_offset + column in *info.  b = 128: 25.0 us alone, 36 us beside the
// trailing update at n = 16384; the form before it (the block as float in
// LDS, 32-column pieces through LDS, 94 KB) took 56 and 70 us.
__global__ __launch_bounds__(diag16::kThreads, 4) void potrf_f32_kernel(int b, float* __restrict__ A, i64 lda,
                                                                     float* __restrict__ Xd, int* __restrict__ info,
                                                                     int col_offset) {
    __shared__ diag16::Lds<true> sh;
    // the factorization's chain: its waves issue ahead of the trailing
    // update's waves sharing the SIMD (wave priority, not queue priority)
    __builtin_amdgcn_s_setprio(2);
    if (info != nullptr && *info != 0 && *info <= col_offset) return;
    diag16::factor_block<float, true>(sh, b, A, lda, Xd, info, col_offset);
}

// Rows rw .. rw+15 of a panel slab (staged in sB) -= P_slab P_top^T: the
// update of the block column from the group's earlier panels, which these
// rows have not received yet.  upd points at the planes' row of the block's
// first (diagonal) row, so P_top = upd rows 0 .. b-1 and the slab's rows are
// upd rows b + r0 + rw + i; K = kk columns (the planes are zero-padded to a
// multiple of 32 columns).  One wave, split-bf16 products (all plane pairs
// p + q < NP), fragments loaded straight from the planes into registers,
// the next 32-wide chunk loading while the current one multiplies.
template <int NP>
__device__ __forceinline__ void panel_slab_update(float (*sB)[kPiLd], const unsigned short* __restrict__ upd, i64 ps,
                                                  i64 ldk, int kk, int b, int m, i64 r0, int rw, int m16, int g) {
    const i64 rows = (i64)b + m;  // rows of the planes block
    const i64 ra = b + r0 + rw + m16 < rows ? b + r0 + rw + m16 : rows - 1;  // clamped; its outputs are dropped
    const unsigned short* a_p = upd + ra * ldk + 8 * g;
    const s8_t neg = {(short)0x8000, (short)0x8000, (short)0x8000, (short)0x8000,
                      (short)0x8000, (short)0x8000, (short)0x8000, (short)0x8000};
    const int nchunks = (kk + 31) / 32;
    // two passes over 64 columns each keep the fragments in few registers
    // (this kernel must stay small enough to be placed beside the trailing
    // update's workgroups)
    for (int h = 0; h < 2; ++h) {
        if (64 * h >= b) break;
        f4_t acc[4];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[nt][v] = sB[rw + 4 * g + v][64 * h + 16 * nt + m16];
        constexpr int kR = 3;  // chunks in flight: the loads are L2-latency bound
        s8_t fa[kR][NP], fb[kR][4][NP];  // [buffer][plane], [buffer][column tile][plane]
        auto load = [&](int buf, int kc) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < NP; ++p) fa[buf][p] = *reinterpret_cast<const s8_t*>(a_p + p * ps + kc) ^ neg;
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                const int c = 64 * h + 16 * nt + m16;
                const i64 rb = (i64)(c < b ? c : b - 1) * ldk + 8 * g + kc;
#pragma unroll
                for (int p = 0; p < NP; ++p) fb[buf][nt][p] = *reinterpret_cast<const s8_t*>(upd + p * ps + rb);
            }
        };
        auto step = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
            for (int nt = 0; nt < 4; ++nt)
#pragma unroll
                for (int o = NP - 1; o >= 0; --o)  // term order o = p + q, smallest first
#pragma unroll
                    for (int p = o; p >= 0; --p) mfma_acc_bf16(acc[nt], fa[buf][p], fb[buf][nt][o - p]);
        };
        // chunk c lives in buffer c % kR; chunk c + kR - 1 loads while chunk c multiplies
#pragma unroll
        for (int c = 0; c < kR - 1; ++c)
            if (c < nchunks) load(c, 32 * c);
        for (int c0 = 0; c0 < nchunks; c0 += kR) {
#pragma unroll
            for (int u = 0; u < kR; ++u) {
                const int c = c0 + u;
                if (c >= nchunks) break;
                if (c + kR - 1 < nchunks) load((u + kR - 1) % kR, 32 * (c + kR - 1));
                step(u);
            }
        }
        mfma_retire();
        // columns past b stay zero (the padding the solve relies on)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (64 * h + 16 * nt + m16 < b) sB[rw + 4 * g + v][64 * h + 16 * nt + m16] = acc[nt][v];
    }
}

// The same update for two planes with P_top staged through LDS: the four
// waves share each 32-column chunk of P_top's planes (16 KB) instead of
// each loading all of it (the update is bound by that traffic), and chunk
// c + 2's global loads are in flight while chunk c multiplies.  sP: two
// chunk buffers, [buffer][plane][row 0..127][32 columns] bf16 (32 KB).
// All threads of the workgroup call it (it synchronises the workgroup).
__device__ __forceinline__ void panel_slab_update_lds(float (*sB)[kPiLd], unsigned short* sP,
                                                      const unsigned short* __restrict__ upd, i64 ps, i64 ldk, int kk,
                                                      int b, int m, i64 r0, int t, int w, int m16, int g) {
    constexpr int NP = 2, kR = 3;
    const int rw = 16 * w;
    const i64 rows = (i64)b + m;
    const i64 ra = b + r0 + rw + m16 < rows ? b + r0 + rw + m16 : rows - 1;  // clamped; its outputs are dropped
    const unsigned short* a_p = upd + ra * ldk + 8 * g;
    const s8_t neg = {(short)0x8000, (short)0x8000, (short)0x8000, (short)0x8000,
                      (short)0x8000, (short)0x8000, (short)0x8000, (short)0x8000};
    // staging: thread t carries 16-byte segments 2 (t / 128) and 2 (t / 128) + 1
    // of P_top row t % 128 (rows past b repeat row b - 1; their outputs are dropped)
    const int sr = t & 127, sseg = (t >> 7) * 2;
    const unsigned short* s_src = upd + (i64)(sr < b ? sr : b - 1) * ldk + 8 * sseg;
    s8_t st[kR][NP][2], fa[kR][NP];
    auto gload = [&](int slot, int kc) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
#pragma unroll
            for (int h = 0; h < 2; ++h) st[slot][p][h] = *reinterpret_cast<const s8_t*>(s_src + p * ps + kc + 8 * h);
            fa[slot][p] = *reinterpret_cast<const s8_t*>(a_p + p * ps + kc) ^ neg;
        }
    };
    auto sstore = [&](int slot, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                *reinterpret_cast<s8_t*>(sP + ((buf * NP + p) * 128 + sr) * 32 + 8 * (sseg + h)) = st[slot][p][h];
    };
    f4_t acc[8];
#pragma unroll
    for (int nt = 0; nt < 8; ++nt)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[nt][v] = sB[rw + 4 * g + v][16 * nt + m16];
    const int nchunks = (kk + 31) / 32;
#pragma unroll
    for (int c = 0; c < kR - 1; ++c)
        if (c < nchunks) gload(c, 32 * c);
    for (int c0 = 0; c0 < nchunks; c0 += kR) {
#pragma unroll
        for (int u = 0; u < kR; ++u) {
            const int c = c0 + u;  // chunk c: registers slot u, LDS buffer c % 2
            if (c >= nchunks) break;
            const int buf = c & 1;
            sstore(u, buf);
            // chunk c is staged, and every wave is done with chunk c - 2,
            // the last user of this buffer
            __syncthreads();
            if (c + kR - 1 < nchunks) gload((u + kR - 1) % kR, 32 * (c + kR - 1));
#pragma unroll
            for (int nt = 0; nt < 8; ++nt) {
                s8_t fb[NP];
#pragma unroll
                for (int p = 0; p < NP; ++p)
                    fb[p] = *reinterpret_cast<const s8_t*>(sP + ((buf * NP + p) * 128 + 16 * nt + m16) * 32 + 8 * g);
#pragma unroll
                for (int o = NP - 1; o >= 0; --o)  // term order o = p + q, smallest first
#pragma unroll
                    for (int p = o; p >= 0; --p) mfma_acc_bf16(acc[nt], fa[u][p], fb[o - p]);
            }
        }
    }
    mfma_retire();
    // columns past b stay zero (the padding the solve relies on)
#pragma unroll
    for (int nt = 0; nt < 8; ++nt)
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (16 * nt + m16 < b) sB[rw + 4 * g + v][16 * nt + m16] = acc[nt][v];
}

// B (m x b, b <= 128) := B L11^{-T}, L11 the b x b float factor at L; one
// 64-row slab per workgroup (n = 4000, no pending update: 10.2 us a launch,
// 15.1 with an address made anew for every load), the result staged through LDS so the
// column-major stores are contiguous.  With NPU > 0 the slab first takes the
// block column's pending update from the group's earlier panels (NPU planes
// at upd, uk columns; panel_slab_update), so no separate kernel has to
// update the rows below the diagonal block before this one runs.
template <int NPU>
__global__ __launch_bounds__(256) void panel_f32_kernel(int m, int b, const float* __restrict__ L, i64 ldl,
                                                        const float* __restrict__ Xd, float* __restrict__ B, i64 ldb,
                                                        const int* __restrict__ info, int limit,
                                                        unsigned short* __restrict__ planes, int np, i64 ps,
                                                        i64 ldk, const unsigned short* __restrict__ upd, int uk) {
    // LDS kept under half a CU (80 KB) so workgroups of this kernel fit beside
    // two of the trailing update's: L11 only as its six 32 x 32 blocks below
    // the diagonal pieces (block (p, q), q < p, at p (p - 1) / 2 + q; zero
    // outside the b x b block, whose padding is the identity) and the
    // inverses of its four 32 x 32 diagonal pieces, in one area that first
    // stages the slab's pending update
    __shared__ __align__(16) float sU[10 * 32 * 36];
    float(*sLb)[32][36] = reinterpret_cast<float(*)[32][36]>(sU);
    float(*sXd)[32][36] = reinterpret_cast<float(*)[32][36]>(sU + 6 * 32 * 36);
    __shared__ float sB[64][kPiLd];
    __builtin_amdgcn_s_setprio(3);  // chain kernel (see potrf_f32_kernel)
    if (info != nullptr && *info != 0 && *info <= limit) return;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, m16 = lane & 15, g = lane >> 4;
    const i64 r0 = (i64)blockIdx.x * 64;
    const int rw = 16 * w;
    // Addresses of whole slabs and blocks are steps from one load to the next
    // (a wave alone on its SIMD pays 4 to 8 cycles for every instruction).
    const bool whole = r0 + 64 <= m, full = b == 128;
    float v[32];
    {  // the slab: row t % 64, columns t / 64 + 4q
        const int rs = t & 63, c_lo = t >> 6;
        if (whole && full) {
            const float* src = B + r0 + rs + (i64)c_lo * ldb;
#pragma unroll
            for (int q = 0; q < 32; ++q, src += 4 * ldb) v[q] = *src;
#pragma unroll
            for (int q = 0; q < 32; ++q) sB[rs][c_lo + 4 * q] = v[q];
        } else {
            const i64 rb = r0 + rs < m ? r0 + rs : m - 1;
#pragma unroll
            for (int q = 0; q < 32; ++q) {
                const int c = c_lo + 4 * q;
                v[q] = B[rb + (i64)(c < b ? c : b - 1) * ldb];
            }
#pragma unroll
            for (int q = 0; q < 32; ++q) {
                const int c = c_lo + 4 * q;
                sB[rs][c] = (r0 + rs < m && c < b) ? v[q] : 0.0f;
            }
        }
    }
    // the slab's pending update: wave w on rows 16w .. 16w+15
    if constexpr (NPU > 0) {
        __syncthreads();
        if constexpr (NPU == 2)
            panel_slab_update_lds(sB, reinterpret_cast<unsigned short*>(sU), upd, ps, ldk, uk, b, m, r0, t, w, m16, g);
        else
            panel_slab_update<NPU>(sB, upd, ps, ldk, uk, b, m, r0, rw, m16, g);
        __syncthreads();  // the staging area becomes L11's blocks
    }
    // block q / 4: row t % 32 (lanes along the column), column t / 32 + 8 (q % 4)
    // (clamped loads, then select)
    {
        const int rr = t & 31, c0 = t >> 5;
        if (full) {
            const float* src = L + rr + (i64)c0 * ldl;
#pragma unroll
            for (int q = 0; q < 24; ++q) {
                const int blk = q >> 2, p = blk < 1 ? 1 : blk < 3 ? 2 : 3, qb = blk - p * (p - 1) / 2;
                v[q] = src[32 * p + (i64)(32 * qb + 8 * (q & 3)) * ldl];
            }
#pragma unroll
            for (int q = 0; q < 24; ++q) sLb[q >> 2][rr][c0 + 8 * (q & 3)] = v[q];
        } else {
#pragma unroll
            for (int q = 0; q < 24; ++q) {
                const int blk = q >> 2, p = blk < 1 ? 1 : blk < 3 ? 2 : 3, qb = blk - p * (p - 1) / 2;
                const int r = 32 * p + rr, c = 32 * qb + c0 + 8 * (q & 3);
                v[q] = L[(r < b ? r : b - 1) + (i64)(c < b ? c : b - 1) * ldl];
            }
#pragma unroll
            for (int q = 0; q < 24; ++q) {
                const int blk = q >> 2, p = blk < 1 ? 1 : blk < 3 ? 2 : 3, qb = blk - p * (p - 1) / 2;
                const int r = 32 * p + rr, c = 32 * qb + c0 + 8 * (q & 3);
                sLb[blk][rr][c0 + 8 * (q & 3)] = (r < b && c < b) ? v[q] : 0.0f;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)  // (the rows of sXd are 16-byte aligned)
        *reinterpret_cast<f4_t*>(&sXd[q][t >> 3][4 * (t & 7)]) = *reinterpret_cast<const f4_t*>(Xd + 1024 * q + 4 * t);
    __syncthreads();
    // wave w: rows 16w .. 16w+15 of the slab, pieces p = 0..3 in order (no
    // other wave touches these rows)
    for (int p = 0; p < 4; ++p) {
        f4_t acc[2] = {};
        for (int q = 0; q < p; ++q) {  // S = sum_q X_q L_pq^T
            const float(*Lpq)[36] = sLb[p * (p - 1) / 2 + q];
            tile_ab_t(acc, sB, rw, 32 * q, Lpq, m16, g);
        }
        mfma_retire();
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int v = 0; v < 4; ++v) sB[rw + 4 * g + v][32 * p + 16 * nt + m16] -= acc[nt][v];
        // X_p = T inv(L_pp)^T (T = the updated columns, this wave's rows only)
        f4_t x[2] = {};
        tile_ab_t(x, sB, rw, 32 * p, sXd[p], m16, g);
        mfma_retire();
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
            for (int v = 0; v < 4; ++v) sB[rw + 4 * g + v][32 * p + 16 * nt + m16] = x[nt][v];
    }
    __syncthreads();
    if (whole && full) {
        float* dst = B + r0 + (t & 63) + (i64)(t >> 6) * ldb;
#pragma unroll
        for (int q = 0; q < 32; ++q, dst += 4 * ldb) *dst = sB[t & 63][(t >> 6) + 4 * q];
    } else {
        for (int idx = t; idx < 64 * 128; idx += 256) {
            const int r = idx & 63, c = idx >> 6;
            if (r0 + r < m && c < b) B[r0 + r + (i64)c * ldb] = sB[r][c];
        }
    }
    if (planes != nullptr) {  // bf16 planes of the result: thread = (row, 8 columns), 16-byte stores
        for (int e = t; e < 64 * 16; e += 256) {
            const int r = e >> 4, c = 8 * (e & 15);
            if (r0 + r >= m || c >= b) continue;
            float x[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) x[q] = (c + q < b) ? sB[r][c + q] : 0.0f;
            for (int p = 0; p < np; ++p) {
                s8_t h;
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const unsigned short hb = f32_to_bf16_rne(x[q]);
                    h[q] = (short)hb;
                    x[q] -= bf16_to_f32(hb);
                }
                *reinterpret_cast<s8_t*>(planes + p * ps + (r0 + r) * ldk + c) = h;
            }
        }
    }
}

hipError_t launch_potrf_f32(int b, float* A, i64 lda, float* Xd, int* info, int col_offset, hipStream_t s) {
    if (b <= 0) return hipSuccess;
    hipLaunchKernelGGL(potrf_f32_kernel, dim3(1), dim3(diag16::kThreads), 0, s, b, A, lda, Xd, info, col_offset);
    return hipGetLastError();
}

hipError_t launch_panel_f32(int m, int b, const float* L, i64 ldl, const float* Xd, float* B, i64 ldb,
                            const int* info, int limit, unsigned short* planes, int np, i64 ps, i64 ldk,
                            hipStream_t s, const unsigned short* upd, int uk) {
    if (m <= 0 || b <= 0) return hipSuccess;
    const dim3 grid((unsigned)ceil_div(m, 64));
    if (upd == nullptr || uk <= 0)
        hipLaunchKernelGGL(panel_f32_kernel<0>, grid, dim3(256), 0, s, m, b, L, ldl, Xd, B, ldb, info, limit, planes,
                           np, ps, ldk, upd, 0);
    else if (np == 2)
        hipLaunchKernelGGL(panel_f32_kernel<2>, grid, dim3(256), 0, s, m, b, L, ldl, Xd, B, ldb, info, limit, planes,
                           np, ps, ldk, upd, uk);
    else if (np == 3)
        hipLaunchKernelGGL(panel_f32_kernel<3>, grid, dim3(256), 0, s, m, b, L, ldl, Xd, B, ldb, info, limit, planes,
                           np, ps, ldk, upd, uk);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace elemamd
