// The solves of a batch: one workgroup per matrix, forward then backward, as
// the chain of 16-row tiles of solve_chain.hip.
//
// What bounds it: the serial chain (about 3.5 us per 64 rows and direction)
// up to n = 1000, and beyond that one CU's stream of L (32 KB per 64 x 64
// block in FP64).  A batch fills the chip with matrices, so each one stays in
// one workgroup: the band waves take every block before the last one (no
// helpers), with L two blocks ahead in registers, and read the solved blocks
// from LDS, where those of a matrix up to about 2000 (FP64, up to 4 columns),
// 1280 (up to 8; FP32: 16) or 770 rows (16) fit; older ones come back from memory.
// One launch takes all matrices, the largest first, so that the small ones
// fill the CUs that the large ones leave.
// Measured (1024 matrices, n = 16 ... 1024, up to 8 columns): 2.73 ms in six
// launches of a kernel that staged every block between two barriers and
// substituted 64 rows by wave broadcasts, 0.39 ms now; FP32 (four sweeps)
// 6.81 and 0.66 ms.
#include <algorithm>

#include "batch.hpp"
#include "common.hpp"
#include "solve_chain_dev.hpp"

namespace elemamd {

namespace chain {

// solved blocks kept in LDS, and blocks that the other waves work ahead
template <typename T, int NV>
struct LocalShape {
    static constexpr int R = sizeof(T) == 4 ? 20 : NV == 1 ? 32 : NV == 2 ? 20 : 12;
    static constexpr int RB = sizeof(T) == 8 && NV == 4 ? 2 : 3;
};

// Band wave w of a matrix that has no helpers: rows 16 w of every block, sums
// over the solved blocks q <= pos - 2.
template <typename T, bool TRANS, bool CONTIG, typename S>
__device__ __forceinline__ void local_band(S& sh, const Rows<T, TRANS, CONTIG>& L, int w, int lane, int nT, int kcl,
                                           const T* B, i64 ldb, long limit) {
    typedef typename Acc4<T>::type acc_t;
    constexpr int NB = 2;  // blocks of L in registers (three spill)
    const int c16 = lane & 15, g = lane >> 4;
    acc_t acc = {};
    for (int pos = 0; pos < min(nT, 2); ++pos) hand_over<T>(sh, pos, w, lane, acc, limit);
    if (nT < 3) return;
    T o[NB][4][4];
    int pos = 2, q = 0, ppos = 2, pq = 0;  // the block multiplied, the block loaded
    const T* row = L.row(2);
    auto load_next = [&](T(&x)[4][4]) __attribute__((always_inline)) {
#pragma unroll
        for (int tq = 0; tq < 4; ++tq) L.load4(x[tq], row, (i64)pq * kSB + 16 * tq, L.cs);
        if (++pq > ppos - 2) {
            ppos = min(ppos + 1, nT - 1);  // (past the end: loaded, not used)
            pq = 0;
            row = L.row(ppos);
        }
    };
#pragma unroll
    for (int u = 0; u < NB; ++u) load_next(o[u]);
    while (pos < nT) {
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            if (pos >= nT) break;
            if (q > pos - S::R) {
                await(&sh.seq, 4 * (q + 1), limit, &sh.err);
#pragma unroll
                for (int tq = 0; tq < 4; ++tq) product(acc, sh.Y[q % S::R], tq, o[u][tq], c16, g);
            } else {  // its place in LDS may have been taken: from memory
                await(&sh.out[q & 1], q / 2 + 1, limit, &sh.err);
                T y[4][4];
#pragma unroll
                for (int tq = 0; tq < 4; ++tq)
#pragma unroll
                    for (int ks = 0; ks < 4; ++ks)
                        y[tq][ks] = __hip_atomic_load(
                            &B[L.phys((i64)q * kSB + 16 * tq + 4 * g + ks) + (i64)min(c16, kcl - 1) * ldb],
                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
                for (int tq = 0; tq < 4; ++tq)
#pragma unroll
                    for (int ks = 0; ks < 4; ++ks) acc = mfma16(y[tq][ks], o[u][tq][ks], acc);
            }
            load_next(o[u]);
            if (++q > pos - 2) {
                acc = mfma16(T(0), T(0), acc);  // (as in the chain)
                hand_over<T>(sh, pos, w, lane, acc, limit);
                acc = {};
                q = 0;
                ++pos;
            }
        }
    }
}

template <bool TRANS, bool CONTIG, int NV, typename T, typename S>
__device__ __forceinline__ void local_solve(S& sh, int n, int kcl, const T* A, T* B, int wave, int lane) {
    const int w = wave & 3, nT = (int)ceil_div(n, kSB);
    const Rows<T, TRANS, CONTIG> rows(n, A, n, false, w, lane);
    if (wave < 4) {
        __builtin_amdgcn_s_setprio(2);
        solve_tiles<NV>(sh, rows, w, lane, nT, kSpinLimit);
        __builtin_amdgcn_s_setprio(0);
    } else if (wave < 8) {
        local_band(sh, rows, w, lane, nT, kcl, B, (i64)n, kSpinLimit);
    } else if (wave < 10) {
        fetch_blocks(sh, rows, wave - 8, lane, nT, kcl, (const T*)B, (i64)n, false, kSpinLimit,
                     [](int, i64, T(&)[S::KC]) {});
    } else {
        publish_blocks<false>(sh, rows, wave - 10, lane, nT, kcl, B, (i64)n, kSpinLimit,
                              [&](int pos) __attribute__((always_inline)) { post(&sh.out[pos & 1], pos / 2 + 1); });
    }
}

}  // namespace chain

template <typename T, bool BACK, int NV>
__global__ __launch_bounds__(chain::kThreads) void batch_solve_kernel(BatchArgs a, const T* L_all, T* B_all,
                                                                      int slab0) {
    using namespace chain;
    typedef LocalShape<T, NV> Shape;
    typedef Lds<T, columns<T>(NV), Shape::R, Shape::RB> S;
    __shared__ S sh;
    const int p = blockIdx.x;
    if (a.info[p] != 0) return;
    if (a.skip != nullptr && a.skip[p]) return;
    const int n = a.n[p], k = a.k[p];
    const T* A = L_all + a.a_off[p];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const i64 c0 = (i64)(slab0 + blockIdx.y) * S::KC;
    if (c0 >= k) return;
    if (threadIdx.x == 0) sh.reset();
    __syncthreads();
    local_solve<BACK, BACK, NV>(sh, n, min(S::KC, k - (int)c0), A, B_all + a.b_off[p] + c0 * n, wave, lane);
    if (lane == 0 && sh.err != 0) a.info[p] = -1;
}

template <typename T, int NV>
static hipError_t solve_both(const BatchArgs& a, const void* L, void* B, int kmax, hipStream_t s) {
    const int slabs = (int)ceil_div(kmax, chain::columns<T>(NV));
    const dim3 block(chain::kThreads);
    for (int first = 0; first < slabs; first += 32768) {  // (a grid's y stays below 65536)
        const dim3 grid(a.count, std::min(slabs - first, 32768));
        hipLaunchKernelGGL((batch_solve_kernel<T, false, NV>), grid, block, 0, s, a, (const T*)L, (T*)B, first);
        hipLaunchKernelGGL((batch_solve_kernel<T, true, NV>), grid, block, 0, s, a, (const T*)L, (T*)B, first);
    }
    return hipGetLastError();
}

hipError_t batch_solve(const BatchArgs& a, const void* L, void* B, bool f32, int kmax, hipStream_t s) {
    if (a.count <= 0) return hipSuccess;
    if (f32) return solve_both<float, 4>(a, L, B, kmax, s);
    // (as few registers on the chain as the right-hand sides need)
    if (kmax > 8) return solve_both<double, 4>(a, L, B, kmax, s);
    return kmax > 4 ? solve_both<double, 2>(a, L, B, kmax, s) : solve_both<double, 1>(a, L, B, kmax, s);
}

}  // namespace elemamd
