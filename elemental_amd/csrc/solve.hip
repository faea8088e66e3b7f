// Inverses of the 64 x 64 diagonal blocks of the low-precision factor, and
// the sizes of the triangular solves' scratch.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "solve_dev.hpp"

namespace elemamd {

// ------------------------------------------------ inverse of diagonal blocks
// Dinv + I*64*64 (column-major, ld 64) := inv(L(I*64.., I*64..)), upper part 0.
// Column c is built row by row: W(i,c) = -(sum_{c<=k<i} L(i,k) W(k,c)) / L(i,i),
// the dot product split over four thread groups and reduced in LDS.
__global__ __launch_bounds__(256) void trtri_diag64_kernel(int n, int I0, const float* __restrict__ L, i64 ldl,
                                                           float* __restrict__ Dinv) {
    __shared__ float sL[kSB][kSLd];  // sL[i][k]
    __shared__ float sW[kSB][kSLd];  // sW[k][c]
    __shared__ float red[4][kSB];
    const int I = I0 + blockIdx.x, t = threadIdx.x;
    const i64 r0 = (i64)I * kSB;
    const int bs = (int)min<i64>(kSB, n - r0);
    for (int idx = t; idx < kSB * kSB; idx += 256) {
        const int i = idx % kSB, k = idx / kSB;
        sL[i][k] = (i < bs && k < bs && k <= i) ? L[r0 + i + (r0 + k) * ldl] : (i == k ? 1.0f : 0.0f);
        sW[i][k] = 0.0f;
    }
    __syncthreads();
    const int c = t & 63, part = t >> 6;
    if (part == 0) sW[c][c] = 1.0f / sL[c][c];
    __syncthreads();
    for (int i = 1; i < kSB; ++i) {
        float s = 0.0f;
        if (c < i)
            for (int k = c + part; k < i; k += 4) s += sL[i][k] * sW[k][c];
        red[part][c] = s;
        __syncthreads();
        if (part == 0 && c < i) sW[i][c] = -(red[0][c] + red[1][c] + red[2][c] + red[3][c]) / sL[i][i];
        __syncthreads();
    }
    float* out = Dinv + (i64)I * kSB * kSB;
    for (int idx = t; idx < kSB * kSB; idx += 256) {
        const int i = idx % kSB, k = idx / kSB;
        out[idx] = (i < bs && k < bs) ? sW[i][k] : 0.0f;
    }
}

hipError_t launch_trtri_diag64_range(int n, int I0, int I1, const float* L, i64 ldl, float* Dinv, hipStream_t s) {
    I1 = (int)std::min<i64>(I1, ceil_div(n, kSB));
    if (n <= 0 || I0 >= I1) return hipSuccess;
    hipLaunchKernelGGL(trtri_diag64_kernel, dim3((unsigned)(I1 - I0)), dim3(256), 0, s, n, I0, L, ldl, Dinv);
    return hipGetLastError();
}

// Solve scratch in ints: the chain solve's tickets and flags, then (256-byte
// aligned) its n x kc partial sums (room for doubles).
size_t solve_ctrl_count(int n, int kc) {
    const size_t flags = ((chain_ctrl_count(n, kc) * sizeof(int) + 255) & ~(size_t)255) / sizeof(int);
    return flags + (size_t)n * kc * 2 + 64;
}
size_t solve_dinv_count(int n) { return (size_t)ceil_div(n, kSB) * kSB * kSB; }

}  // namespace elemamd
