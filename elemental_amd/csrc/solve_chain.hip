// Triangular solves with the Cholesky factor as a chain plus helpers, one
// launch per direction:
//   forward  B := inv(L) B     (Trsm(LEFT, LOWER, NORMAL,  NON_UNIT) -> dtrsm_('L','L','N','N'))
//   backward B := inv(L^T) B   (Trsm(LEFT, LOWER, ADJOINT, NON_UNIT) -> dtrsm_('L','L','T','N'))
// as used by cholesky::SolveAfter (include/elemental/lapack-like/Cholesky/SolveAfter.hpp:20-75).
//
// Rows are taken in solve order (the backward solve's from the last row up),
// so that every form is one lower triangular solve: logical row i's
// coefficient of row k < i sits at base[i rs + k cs].  They are cut into
// 64-row blocks (positions pos = 0, 1, ...; only the last one may be short)
// and each block into four 16-row tiles.
//
// What bounds it: the chain of n / 16 tiles, each a substitution and the
// product that brings it into the next tile.  So nothing else is on that
// chain:
// * One chain workgroup per 16-column slab of right-hand sides.  Wave w (w <
//   4) solves the tiles 4 pos + w.  It holds the tile transposed (right-hand
//   sides as rows) in the MFMA accumulator layout, and substitutes in
//   registers with DPP row broadcasts: a_c -= a_k (l_ck / l_kk), then a
//   scaling by the reciprocal diagonal (exact on integer problems with
//   power-of-two diagonals; a tile that this does not serve, because a
//   multiplier over- or underflows or a row is not finite, is solved again
//   as the reference's loop does it, solve_tile_careful).  A solved tile is written to LDS with a sequence
//   number behind it (the LDS unit serves a wave's accesses in order); the
//   other waves poll that number, so no barrier holds the waves together.
//   The products with the block before and with the own block's earlier tiles
//   are made as their tiles appear, in the three tile times in which the
//   other waves are on the chain, with operands of L loaded a block ahead
//   straight into MFMA operand layout.  These loads are the same ones in
//   every step (addresses clamped, no branch around them, nothing else of
//   these waves goes to memory), so that the compiler waits for exactly the
//   one it needs.
// * Waves 4-7 apply the blocks at distance 2 and 3 (the band), waves 8 and 9
//   fetch the right-hand sides and a helper's partial sum of the older blocks
//   and make the substitutions' multipliers, all into LDS ahead of their use;
//   waves 10 and 11 publish solved blocks (two waves each, in turn: a block's
//   round trips to memory take longer than a block on the chain).  Memory
//   latency is theirs, not the chain's.
// * One helper workgroup per (pos >= D + 1, slab) accumulates
//   sum_{q <= pos - D - 1} M(pos, q) Y_q as the chain publishes those blocks
//   and hands the partial sum to the chain: waves 0-3 the products (16 rows
//   each), waves 8 and 9 bring the blocks into LDS, in turn.
// Measured (FP64, n = 8192, 16 columns): 3.6 us per 64-row block forward, 4.0
// backward (there every lane of an operand load reads another row, 64 cycles a
// load, and the block's 120 loads of eight waves set the pace); 3.4 and 4.0
// with 8 columns.  A chain paced by workgroup barriers with one load phase per
// block was 20.7 us (6.2 and 7.5 with products by inverted diagonal blocks in
// the substitutions' place).
// Both solves with an n = 8192 factor: 5.43 ms before, 1.00 ms now; the same
// chain with conditional loads, whose waits the compiler cannot count: 1.35.
// Cross-workgroup data (solved blocks, partial sums, flags) moves only
// through device-coherent loads and stores; a writer waits for the
// acknowledgement of its stores before it raises a flag (solve_dev.hpp).
// Workgroups take tickets in launch order: the chains first, then helpers by
// increasing position, so every wait is on a workgroup that is running or
// done, or (a chain's) on the next helper to be dispatched, for which
// chain_slabs() leaves CUs as long as no more than four such launches run at a
// time, one for each hardware queue.  Every wait is bounded (spin_limit polls,
// then an error in ctrl[1], which the caller clears once per solve, so a wait
// that gave up in the forward solve is still reported after the backward one).
#include <algorithm>

#include "chain_slabs.hpp"
#include "common.hpp"
#include "kernels.hpp"
#include "runtime.hpp"
#include "solve_chain_dev.hpp"

namespace elemamd {

namespace chain {

constexpr int D = 3;          // blocks before its own that the chain workgroup applies (a helper the older ones)
constexpr int RH = 4;         // helper: blocks of solved rows in LDS
// R = 5: the band, the current block, the one being published
template <typename T, int NV>
struct Shared : Lds<T, columns<T>(NV), 5, 3> {
    int have[2];  // helper: blocks brought by waves 8, 9 (counting each one's own)
    int used[4];  // helper: blocks multiplied by waves 0-3
    int done, ord;
};

}  // namespace chain

// unit: the diagonal is taken as one and never used (Trsm's UNIT diag).  NV:
// accumulator registers that hold right-hand sides.  epoch: the value that
// raises a flag in this launch (flags keep the values of earlier launches);
// tickets start at `base`.  TRANS, CONTIG, upper: see chain::Rows.
template <typename T, bool TRANS, bool CONTIG, int NV>
__global__ __launch_bounds__(chain::kThreads) void trsm_chain_kernel(int n, int kc, const T* __restrict__ L, i64 ldl,
                                                                     T* __restrict__ B, i64 ldb,
                                                                     int* __restrict__ ctrl, int* __restrict__ flags,
                                                                     T* __restrict__ part,
                                                                     const int* __restrict__ info, long spin_limit,
                                                                     int upper, int unit, int epoch, int base) {
    using namespace chain;
    typedef typename Acc4<T>::type acc_t;
    typedef Shared<T, NV> S;
    constexpr int KC = S::KC;
    __shared__ S sh;
    if (info != nullptr && *info != 0) return;
    const int t = threadIdx.x, lane = t & 63, c16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int w = wave & 3;  // rows 16 w of a block (waves 0-3: the chain, 4-7: the band)
    const int nT = (int)ceil_div(n, kSB);
    const int CY = (int)ceil_div(kc, kSC);
    if (t == 0) {
        sh.ord = atomicAdd(&ctrl[0], 1) - base;
        sh.reset();
        sh.done = 0;
        for (int v = 0; v < 2; ++v) sh.have[v] = 0;
        for (int v = 0; v < 4; ++v) sh.used[v] = 0;
    }
    __syncthreads();
    const int ord = __builtin_amdgcn_readfirstlane(sh.ord);
    int* flagsX = flags;            // by position: solved block published
    int* flagsP = flags + nT * CY;  // by position: helper's partial sum published
    const Rows<T, TRANS, CONTIG> rows(n, L, ldl, upper != 0, w, lane);
    // a wave's end: waits that gave up are recorded for the caller
    auto report = [&]() __attribute__((always_inline)) {
        if (lane == 0 && sh.err != 0) atomicOr(&ctrl[1], 1);
    };

    if (ord >= CY) {
        // ------------------------------------------------------------ helper
        const int h = ord - CY;
        const int pos = h / CY + D + 1, cy = h % CY;
        const int c_base = cy * kSC, kcl = min(kSC, kc - c_base);
        const int nJ = pos - D;  // positions 0 .. pos - D - 1
        if (wave >= 4) {
            if (wave != 8 && wave != 9) return;
            // blocks u, u + 2, ... into LDS (slot q % RH) as they are published
            const int u = wave - 8;
            int seen = 0;  // blocks known to be published
            for (int q = u; q < nJ; q += 2) {
                if (q >= seen) {
                    long spins = 0;
                    for (;;) {
                        const int f = seen + lane < nJ ? coherent_load(&flagsX[(seen + lane) * CY + cy]) : 0;
                        const unsigned long long msk = __ballot(f >= epoch);
                        seen += (~msk == 0ull) ? 64 : (int)__builtin_ctzll(~msk);
                        if (q < seen) break;
                        if (++spins > spin_limit) {
                            sh.err = 1;
                            seen = nJ;
                            break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                    }
                }
                const i64 row = rows.phys((i64)q * kSB + lane);
                T y[KC];
#pragma unroll
                for (int c = 0; c < KC; ++c) y[c] = coherent_load(&B[row + (i64)(c_base + min(c, kcl - 1)) * ldb]);
                for (int v = 0; v < 4; ++v) await(&sh.used[v], q - RH + 1, spin_limit, &sh.err);
#pragma unroll
                for (int c = 0; c < KC; ++c) sh.Y[q % RH][lane][c] = y[c];
                post(&sh.have[u], q / 2 + 1);
            }
            report();
            return;
        }
        acc_t acc = {};
        const T* row = rows.row(pos);
        T o[2][4][4];
#pragma unroll
        for (int tq = 0; tq < 4; ++tq) rows.load4(o[0][tq], row, 16 * tq, rows.cs);
        // (two blocks per pass: the buffers' indices stay fixed at compile time)
        for (int q0 = 0; q0 < nJ; q0 += 2) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int q = q0 + u;
                if (q >= nJ) break;
                const i64 kn = (i64)min(q + 1, nJ - 1) * kSB;
#pragma unroll
                for (int tq = 0; tq < 4; ++tq) rows.load4(o[u ^ 1][tq], row, kn + 16 * tq, rows.cs);
                await(&sh.have[u], q / 2 + 1, spin_limit, &sh.err);
#pragma unroll
                for (int tq = 0; tq < 4; ++tq) product(acc, sh.Y[q % RH], tq, o[u][tq], c16, g);
                post(&sh.used[w], q + 1);
            }
        }
        acc = mfma16(T(0), T(0), acc);  // (as in the chain)
        const i64 i = (i64)pos * kSB + 16 * w + c16;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int c = mfma_row<T>(lane, v);
            if (i < n && c < kcl) coherent_store(&part[i + (i64)(c_base + c) * n], acc[v]);
        }
        report();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (lane == 0 && atomicAdd(&sh.done, 1) == 3) coherent_store(&flagsP[pos * CY + cy], epoch);
        return;
    }

    const int cy = ord;
    const int c_base = cy * kSC, kcl = min(kSC, kc - c_base);
    T* Bc = B + (i64)c_base * ldb;
    if (wave == 8 || wave == 9) {
        fetch_blocks(sh, rows, wave - 8, lane, nT, kcl, (const T*)Bc, ldb, unit != 0, spin_limit,
                     [&](int pos, i64 i, T(&b)[KC]) __attribute__((always_inline)) {
                         if (pos <= D) return;
                         long spins = 0;
                         while (coherent_load(&flagsP[pos * CY + cy]) < epoch) {
                             __builtin_amdgcn_s_sleep(1);
                             if (++spins > spin_limit) {
                                 sh.err = 1;
                                 break;
                             }
                         }
                         asm volatile("" ::: "memory");
                         T h[KC];
#pragma unroll
                         for (int c = 0; c < KC; ++c) h[c] = coherent_load(&part[i + (i64)(c_base + min(c, kcl - 1)) * n]);
                         pin(h);
#pragma unroll
                         for (int c = 0; c < KC; ++c) b[c] -= h[c];
                     });
    } else if (wave >= 10) {
        publish_blocks<true>(sh, rows, wave - 10, lane, nT, kcl, Bc, ldb, spin_limit,
                             [&](int pos) __attribute__((always_inline)) {
                                 if (lane == 0) coherent_store(&flagsX[pos * CY + cy], epoch);
                             });
    } else if (wave >= 4) {
        // ---------------------------------------------------------- band waves
        T o[2][4][4];  // distance 3, distance 2
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int tq = 0; tq < 4; ++tq) rows.load4(o[u][tq], rows.row(0), 16 * tq, rows.cs64);
        for (int pos = 0; pos < nT; ++pos) {
            const T* row = rows.row(min(pos + 1, nT - 1));
            acc_t acc = {};
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int q = pos - 3 + u;
                if (q >= 0) {
                    await(&sh.seq, 4 * (q + 1), spin_limit, &sh.err);
#pragma unroll
                    for (int tq = 0; tq < 4; ++tq) product(acc, sh.Y[q % S::R], tq, o[u][tq], c16, g);
                }
                // the next position's operands, under the rest of this one
                const i64 kn = (i64)max(q + 1, 0) * kSB;
#pragma unroll
                for (int tq = 0; tq < 4; ++tq) rows.load4(o[u][tq], row, kn + 16 * tq, rows.cs64);
            }
            acc = mfma16(T(0), T(0), acc);  // (as in the chain)
            hand_over<T>(sh, pos, w, lane, acc, spin_limit);
        }
    } else {
        __builtin_amdgcn_s_setprio(2);
        solve_tiles<NV>(sh, rows, w, lane, nT, spin_limit);
    }
    report();
}

size_t chain_ctrl_count(int n, int kc) { return 2 + 2 * (size_t)ceil_div(n, kSB) * ceil_div(kc, kSC); }

template <typename T, bool TRANS, bool CONTIG, typename... Args>
static void chain_launch(unsigned grid, hipStream_t s, int n, int kc, Args... args) {
    // FP64: each accumulator register holds four right-hand sides, so few
    // right-hand sides need fewer instructions on the chain (n = 8192: 473 us
    // for one, 487 for 16 or 32; FP32's registers interleave the columns)
    auto kernel = sizeof(T) == 4 || kc > 8 ? trsm_chain_kernel<T, TRANS, CONTIG, 4>
                  : kc > 4                 ? trsm_chain_kernel<T, TRANS, CONTIG, sizeof(T) == 4 ? 4 : 2>
                                           : trsm_chain_kernel<T, TRANS, CONTIG, sizeof(T) == 4 ? 4 : 1>;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(chain::kThreads), 0, s, n, kc, args...);
}

template <typename T>
hipError_t launch_trsm_chain(bool forward, bool backward, int n, int kc, const T* L, i64 ldl, T* B, i64 ldb, int* ctrl,
                             T* part, const int* info, hipStream_t s, bool upper, bool unit) {
    if (n <= 0 || kc <= 0) return hipSuccess;
    // tickets (ctrl[0]), the error word (ctrl[1]) and the flags start at zero
    // once: the backward launches raise flags to 2 and their tickets go on
    // from the forward ones'
    hipError_t e = launch_fill_int(ctrl, 0, (int)chain_ctrl_count(n, kc), s);
    if (e != hipSuccess) return e;
    const long spin = solve_spin_limit();
    const int nT = (int)ceil_div(n, kSB);
    const int cus = device_cus();
    if (cus <= 0) return hipErrorInvalidDevice;
    const int helpers = std::max(0, nT - chain::D - 1), slabs = chain_slabs(helpers, cus);
    int base = 0, epoch = 0;
    for (int dir = 0; dir < 2; ++dir) {
        if (dir == 0 ? !forward : !backward) continue;
        ++epoch;
        for (int c0 = 0; c0 < kc; c0 += slabs * kSC) {
            const int k = std::min(kc - c0, slabs * kSC), CY = (int)ceil_div(k, kSC);
            const unsigned grid = (unsigned)(CY + CY * helpers);
            int* flags = ctrl + 2 + 2 * nT * (c0 / kSC);
            T* Bc = B + (i64)c0 * ldb;
            T* pc = part + (i64)c0 * n;
            const bool contig = (dir == 1) != upper;
#define ELEMAMD_CHAIN(TRANS, CONTIG)                                                                          \
    chain_launch<T, TRANS, CONTIG>(grid, s, n, k, L, ldl, Bc, ldb, ctrl, flags, pc, info, spin, (int)upper, \
                                   (int)unit, epoch, base)
            if (dir == 0) {
                if (contig) ELEMAMD_CHAIN(false, true);
                else ELEMAMD_CHAIN(false, false);
            } else {
                if (contig) ELEMAMD_CHAIN(true, true);
                else ELEMAMD_CHAIN(true, false);
            }
#undef ELEMAMD_CHAIN
            e = hipGetLastError();
            if (e != hipSuccess) return e;
            base += (int)grid;
        }
    }
    return hipSuccess;
}

template hipError_t launch_trsm_chain<double>(bool, bool, int, int, const double*, i64, double*, i64, int*, double*,
                                              const int*, hipStream_t, bool, bool);
template hipError_t launch_trsm_chain<float>(bool, bool, int, int, const float*, i64, float*, i64, int*, float*,
                                             const int*, hipStream_t, bool, bool);

}  // namespace elemamd
