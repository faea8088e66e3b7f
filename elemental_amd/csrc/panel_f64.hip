// Panel solve of the FP64 blocked factorization, B := B L11^{-T}: the
// Trsm(RIGHT, LOWER, ADJOINT, NON_UNIT, 1, A11, A21) of cholesky::LVar3
// (include/elemental/lapack-like/Cholesky/LVar3.hpp:113), which the
// reference hands to dtrsm_('R','L','T','N') (src/core/imports/blas.cpp:1203-1210).
//
// One 64-row slab per workgroup, 16 rows per wave; a wave never waits for
// another after the diagonal tiles' multipliers are in LDS.  The rows stay in
// registers in the FP64 MFMA accumulator layout (lane (c, g) = (lane % 16,
// lane / 16) holds rows g + 4v, v = 0..3, of column c of a 16-column tile),
// eight tiles for 128 columns.  Tile by tile, right-looking:
//   * substitution inside the tile by DPP row broadcasts (the column's owner
//     is lane k of every 16-lane row): b_c -= b_k (l_ck / l_kk), one
//     instruction per column and register, then a scaling by 1 / l_cc;
//   * the solved tile goes through a 2 KB wave-private LDS buffer into MFMA
//     operand order and updates every later tile at once, B_p -= X_q L_pq^T
//     (FP64 MFMA 16x16x4, the accumulators are the rows); the L_pq operands
//     come straight from memory (L2), each loaded a tile ahead, as soon as
//     its registers are free.
// Exact on integer problems with power-of-two diagonals; not bit-identical to
// the reference loop (the bit-exact column sweep is trsm_rlt_kernel).
//
// What bounds it: per wave 112 FP64 MFMAs (64 cycles each) and 480 DPP FMAs
// (5 cycles), and, a wave being alone on its SIMD, 4 to 8 cycles for each other
// instruction: 30000 cycles a slab, of which 8000 go to loading, 1300 to
// turning, 9000 to the substitutions and 11000 to the updates.  12.6 us a
// launch at n = 2048 (128 columns); 30 with 32-column pieces whose broadcasts
// were four instructions, whose loads ran along columns (every lane an access
// of its own) and whose addresses were made anew for each.  The
// factorization and solve at n = 2048: 1.53 -> 1.27 ms.
// 24 KB of LDS fit beside four workgroups of the trailing update; its 234
// registers take the place of one that leaves.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "panel16_dev.hpp"

namespace elemamd {

template <typename Off>
__global__ __launch_bounds__(256) void panel_f64_kernel(int m, int b, const double* __restrict__ L, i64 ldl,
                                                        double* __restrict__ B, i64 ldb, const int* __restrict__ info,
                                                        int limit) {
    __shared__ panel16::Lds sh;
    // the factorization's chain: its waves issue ahead of the trailing
    // update's waves sharing the SIMD (wave priority, not queue priority)
    __builtin_amdgcn_s_setprio(3);
    if (info != nullptr && *info != 0 && *info <= limit) return;
    panel16::slab<double, Off>(sh, m, b, L, ldl, B, ldb, B, ldb, blockIdx.x);
}

hipError_t launch_panel_f64(int m, int b, const double* L, i64 ldl, double* B, i64 ldb, const int* info, int limit,
                            hipStream_t s) {
    if (m <= 0 || b <= 0) return hipSuccess;
    if (b > 128) return hipErrorInvalidValue;
    // three columns' bytes in 32 bits
    auto kernel = std::max(ldl, ldb) < (i64)1 << 27 ? panel_f64_kernel<unsigned> : panel_f64_kernel<unsigned long long>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div(m, 64)), dim3(256), 0, s, m, b, L, ldl, B, ldb, info, limit);
    return hipGetLastError();
}

// X := B L^{-T} (m x b) and R := L^{-T} (b x b, zero below the diagonal) in one
// launch: the panel of the HPD inverse and its diagonal block's inverse,
// transposed.
template <typename Off>
__global__ __launch_bounds__(256) void panel_inverse_kernel(int m, int b, const double* __restrict__ L, i64 ldl,
                                                            const double* B, i64 ldb, double* X, i64 ldx, double* R,
                                                            i64 ldr, const int* __restrict__ info) {
    __shared__ panel16::Lds sh;
    if (info != nullptr && *info != 0) return;
    const int ns = (b + 63) / 64;
    if ((int)blockIdx.x < ns)
        panel16::slab<double, Off, true>(sh, b, b, L, ldl, nullptr, 0, R, ldr, blockIdx.x);
    else
        panel16::slab<double, Off>(sh, m, b, L, ldl, B, ldb, X, ldx, blockIdx.x - ns);
}

hipError_t launch_panel_inverse_f64(int m, int b, const double* L, i64 ldl, const double* B, i64 ldb, double* X, i64 ldx,
                                    double* R, i64 ldr, const int* info, hipStream_t s) {
    if (b <= 0) return hipSuccess;
    if (b > 128) return hipErrorInvalidValue;
    const i64 ld = std::max(std::max(ldl, ldb), std::max(ldx, ldr));
    auto kernel = ld < (i64)1 << 27 ? panel_inverse_kernel<unsigned> : panel_inverse_kernel<unsigned long long>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(ceil_div(b, 64) + (m > 0 ? ceil_div(m, 64) : 0))), dim3(256), 0, s, m, b, L,
                       ldl, B, ldb, X, ldx, R, ldr, info);
    return hipGetLastError();
}

}  // namespace elemamd
