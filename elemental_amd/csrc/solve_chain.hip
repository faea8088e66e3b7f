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
//   power-of-two diagonals).  A solved tile is written to LDS with a sequence
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
// Measured (FP64, n = 8192, 16 columns): 3.3 us per 64-row block forward, 3.9
// backward, of which the substitutions are 4 x 0.35; a chain paced by
// workgroup barriers with one load phase per block was 20.7 us (6.2 and 7.5
// with products by inverted diagonal blocks in the substitutions' place).
// Both solves with an n = 8192 factor: 5.43 ms before, 1.00 ms now; the same
// chain with conditional loads, whose waits the compiler cannot count: 1.35.
// Cross-workgroup data (solved blocks, partial sums, flags) moves only
// through device-coherent loads and stores; a writer waits for the
// acknowledgement of its stores before it raises a flag (solve_dev.hpp).
// Workgroups take tickets in launch order: the chains first, then helpers by
// increasing position, so every wait is on a workgroup that is running or
// done.  Every wait is bounded (spin_limit polls, then an error in ctrl[1],
// which the caller clears once per solve, so a wait that gave up in the
// forward solve is still reported after the backward one).
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "runtime.hpp"
#include "solve_dev.hpp"

namespace elemamd {

namespace chain {

constexpr int D = 3;      // blocks before its own that the chain workgroup applies (a helper the older ones)
constexpr int R = 5;      // solved blocks kept in LDS (the band, the current one, what is being published)
constexpr int RB = 3;     // blocks of right-hand sides, multipliers and band sums ahead of the chain
constexpr int RH = 4;     // helper: blocks of Y in LDS
constexpr int kWaves = 12, kThreads = 64 * kWaves;
constexpr int kMaxSlabs = 8;  // slabs per launch: more right-hand sides take several launches

template <typename T>
struct Lds {
    T Y[R][kSB][kSC + 1];   // chain: solved blocks [row][rhs]; helper: blocks of Y
    T Bv[RB][kSB][kSC + 1]; // chain: right-hand sides less the helper's sum
    T Sb[RB][kSB][kSC + 1]; // chain: the band's sums
    T M[RB][kSB][kSC + 1];  // chain: multipliers [row][column in the tile], [15]: reciprocal diagonal
    int seq;                // chain: tiles solved
    int fetched[2];         // chain: blocks in Bv and M (counting each fetching wave's own)
    int taken[2];           // chain: blocks read out of Y (counting each publishing wave's own)
    int band[4];            // chain: blocks in Sb, rows of wave w
    int have[2];            // helper: blocks brought by waves 8, 9 (counting each one's own)
    int used[4];            // helper: blocks multiplied by waves 0-3
    int done, ord, err;
};

__device__ __forceinline__ int peek(const int* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
__device__ __forceinline__ void post(int* p, int v) {
    asm volatile("" ::: "memory");  // the data before it (LDS serves a wave's accesses in order)
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ i64 lesser(i64 a, i64 b) { return a < b ? a : b; }

// Until *p >= v (LDS), at most `limit` polls.
__device__ __forceinline__ void await(const int* p, int v, long limit, int* err) {
    long spins = 0;
    while (peek(p) < v) {
        if (++spins > limit) {
            *err = 1;
            break;
        }
    }
    asm volatile("" ::: "memory");
}

// The values are formed here: the compiler neither delays their making (onto
// the chain) nor splits their loads.
template <typename T, int N>
__device__ __forceinline__ void pin(T (&x)[N]) {
#pragma unroll
    for (int k = 0; k < N; ++k) asm volatile("" : "+v"(x[k]));
}

// a -= (lane K of the 16-lane row's a) * m, with the DPP operand's two wait
// states after its last write: the other accumulators' instructions lie
// between, `gap` fills up.
template <int K>
__device__ __forceinline__ void self_step(double& a, double m) {
    asm volatile("v_fmac_f64_dpp %0, -%0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "+v"(a) : "v"(m), "n"(K));
}
template <int K>
__device__ __forceinline__ void self_step(float& a, float m) {
    asm volatile("v_fmac_f32_dpp %0, -%0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "+v"(a) : "v"(m), "n"(K));
}
template <int NV>
__device__ __forceinline__ void gap() {
    if constexpr (NV == 1) asm volatile("s_nop 1");
    else if constexpr (NV == 2) asm volatile("s_nop 0");
}
template <typename T, int NV, int K>
struct Substitute {
    static __device__ __forceinline__ void run(T (&a)[NV], const T (&m)[15]) {
        gap<NV>();
#pragma unroll
        for (int v = 0; v < NV; ++v) self_step<K>(a[v], m[K]);
        if constexpr (K < 14) Substitute<T, NV, K + 1>::run(a, m);
    }
};

// The tile's multipliers: m[k] := l_ck / l_kk for k < c, else 0 (lane c of
// every 16-lane row holds row c's coefficients in m; r its reciprocal
// diagonal).
template <int K>
__device__ __forceinline__ double row_lane(double x) {
    double y;
    asm volatile("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
                 : "=v"(y)
                 : "v"(x), "n"(K));
    return y;
}
template <int K>
__device__ __forceinline__ float row_lane(float x) {
    float y;
    asm volatile("s_nop 1\n\tv_mov_b32_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
                 : "=v"(y)
                 : "v"(x), "n"(K));
    return y;
}
template <typename T, int K>
struct Multipliers {
    static __device__ __forceinline__ void run(T (&m)[15], T r, int c) {
        const T rk = row_lane<K>(r);
        m[K] = K < c ? m[K] * rk : T(0);
        if constexpr (K < 14) Multipliers<T, K + 1>::run(m, r, c);
    }
};

}  // namespace chain

// TRANS: the backward direction.  upper: the factor is stored in the upper
// triangle (L = U^T, element (i, j) of L at (j, i)).  CONTIG: a row's
// coefficients are known to be contiguous (TRANS != upper) and n >= 16, so
// that a group of four exists in every row.  unit: the diagonal is
// taken as one and never used (Trsm's UNIT diag).  NV: accumulator registers
// that hold right-hand sides (FP64: four columns each).  epoch: the value that
// raises a flag in this launch (flags keep the values of earlier launches);
// tickets start at `base`.
template <typename T, bool TRANS, bool CONTIG, int NV>
__global__ __launch_bounds__(chain::kThreads) void trsm_chain_kernel(int n, int kc, const T* __restrict__ L, i64 ldl,
                                                                     T* __restrict__ B, i64 ldb,
                                                                     int* __restrict__ ctrl, int* __restrict__ flags,
                                                                     T* __restrict__ part,
                                                                     const int* __restrict__ info, long spin_limit,
                                                                     int upper, int unit, int epoch, int base) {
    using namespace chain;
    const bool read_t = CONTIG || TRANS != (upper != 0);  // the coefficient (i, k) is stored at (k, i)
    constexpr int sgn = TRANS ? -1 : 1;
    typedef typename Acc4<T>::type acc_t;
    __shared__ Lds<T> sh;
    if (info != nullptr && *info != 0) return;
    const int t = threadIdx.x, lane = t & 63, c16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int w = wave & 3;  // rows 16 w of a block (waves 0-3: the chain, 4-7: the band)
    const int nT = (int)ceil_div(n, kSB);
    const int CY = (int)ceil_div(kc, kSC);
    if (t == 0) {
        sh.ord = atomicAdd(&ctrl[0], 1) - base;
        sh.seq = sh.done = sh.err = 0;
        for (int v = 0; v < 2; ++v) sh.fetched[v] = sh.taken[v] = sh.have[v] = 0;
        for (int v = 0; v < 4; ++v) sh.used[v] = sh.band[v] = 0;
    }
    __syncthreads();
    const int ord = __builtin_amdgcn_readfirstlane(sh.ord);
    int* flagsX = flags;            // by position: solved block published
    int* flagsP = flags + nT * CY;  // by position: helper's partial sum published
    auto phys = [&](i64 i) -> i64 { return TRANS ? n - 1 - i : i; };  // stored row of logical row i
    const T* Lb = TRANS ? L + (i64)(n - 1) * (1 + ldl) : L;
    // (columns past the slab's last repeat that one: they are solved and dropped)
    const i64 rs = sgn * (read_t ? ldl : 1);
    const i64 cs = read_t ? sgn : sgn * ldl;
    // rows past n (in the last block) repeat row n - 1: nothing of them is used
    auto row_ptr = [&](int pos) -> const T* {
        return Lb + lesser((i64)pos * kSB + 16 * w + c16, n - 1) * rs;
    };
    // MFMA operand: this lane's row, columns k0 + 4 g + ks, ks < 4
    auto load4 = [&](T (&o)[4], const T* row, i64 k0, i64 step) __attribute__((always_inline)) {
        const T* p = row + (k0 + 4 * g) * step;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) o[ks] = CONTIG ? p[sgn * ks] : p[ks * step];
    };
    auto product = [&](acc_t& acc, const T (*Y)[kSC + 1], int tq, const T (&o)[4]) __attribute__((always_inline)) {
        T y[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) y[ks] = Y[16 * tq + 4 * g + ks][c16];
        pin(y);  // (all four reads in flight together)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) acc = mfma16(y[ks], o[ks], acc);
    };
    // the same with a tile that may still be on its way: the sequence number
    // and the tile are read together (LDS serves a wave's reads in order, so a
    // tile read after a sufficient number is complete)
    auto product_when = [&](int need, acc_t& acc, const T (*Y)[kSC + 1], int tq, const T (&o)[4])
                            __attribute__((always_inline)) {
        T y[4];
        long spins = 0;
        for (;;) {
            const int have = peek(&sh.seq);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) y[ks] = Y[16 * tq + 4 * g + ks][c16];
            pin(y);
            if (have >= need) break;
            if (++spins > spin_limit) {
                sh.err = 1;
                break;
            }
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) acc = mfma16(y[ks], o[ks], acc);
    };
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
                const i64 row = phys((i64)q * kSB + lane);
                T y[kSC];
#pragma unroll
                for (int c = 0; c < kSC; ++c) y[c] = coherent_load(&B[row + (i64)(c_base + min(c, kcl - 1)) * ldb]);
                for (int v = 0; v < 4; ++v) await(&sh.used[v], q - RH + 1, spin_limit, &sh.err);
#pragma unroll
                for (int c = 0; c < kSC; ++c) sh.Y[q % RH][lane][c] = y[c];
                post(&sh.have[u], q / 2 + 1);
            }
            report();
            return;
        }
        acc_t acc = {};
        const T* row_p = row_ptr(pos);
        T o[2][4][4];
#pragma unroll
        for (int tq = 0; tq < 4; ++tq) load4(o[0][tq], row_p, 16 * tq, cs);
        // (two blocks per pass: the buffers' indices stay fixed at compile time)
        for (int q0 = 0; q0 < nJ; q0 += 2) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int q = q0 + u;
                if (q >= nJ) break;
                const i64 kn = (i64)min(q + 1, nJ - 1) * kSB;
#pragma unroll
                for (int tq = 0; tq < 4; ++tq) load4(o[u ^ 1][tq], row_p, kn + 16 * tq, cs);
                await(&sh.have[u], q / 2 + 1, spin_limit, &sh.err);
#pragma unroll
                for (int tq = 0; tq < 4; ++tq) product(acc, sh.Y[q % RH], tq, o[u][tq]);
                post(&sh.used[w], q + 1);
            }
        }
        // dependent zero-operand MFMA before the accumulator is read (the
        // compiler's wait states after a loop back edge are short for FP64 MFMA)
        acc = mfma16(T(0), T(0), acc);
        const i64 i = (i64)pos * kSB + 16 * w + c16;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
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
    if (wave == 8 || wave == 9) {
        // ------------------------------------------------------ fetching waves
        for (int pos = wave - 8; pos < nT; pos += 2) {
            const i64 i = (i64)pos * kSB + lane;
            const bool in = i < n;
            const i64 ic = in ? i : n - 1, t0 = ic - (ic & 15);  // (clamped) row, its tile's first row
            T m[15], b[kSC];
#pragma unroll
            for (int k = 0; k < 15; ++k) m[k] = Lb[ic * rs + lesser(t0 + k, ic) * cs];
            const T dd = Lb[ic * rs + ic * cs];
            const i64 row = phys(ic);
#pragma unroll
            for (int c = 0; c < kSC; ++c) b[c] = B[row + (i64)(c_base + min(c, kcl - 1)) * ldb];
            // multipliers l_ck / l_kk of the tile's earlier columns
            const T r = in && !unit ? T(1) / dd : T(1);
            Multipliers<T, 0>::run(m, r, in ? c16 : 0);
            if (pos > D) {
                long spins = 0;
                while (coherent_load(&flagsP[pos * CY + cy]) < epoch) {
                    __builtin_amdgcn_s_sleep(1);
                    if (++spins > spin_limit) {
                        sh.err = 1;
                        break;
                    }
                }
                asm volatile("" ::: "memory");
                T h[kSC];
#pragma unroll
                for (int c = 0; c < kSC; ++c) h[c] = coherent_load(&part[ic + (i64)(c_base + min(c, kcl - 1)) * n]);
                pin(h);
#pragma unroll
                for (int c = 0; c < kSC; ++c) b[c] -= h[c];
            }
            await(&sh.seq, 4 * (pos - RB + 1), spin_limit, &sh.err);  // the slot's last block is solved
#pragma unroll
            for (int c = 0; c < kSC; ++c) sh.Bv[pos % RB][lane][c] = b[c];
#pragma unroll
            for (int k = 0; k < 15; ++k) sh.M[pos % RB][lane][k] = m[k];
            sh.M[pos % RB][lane][15] = r;
            post(&sh.fetched[pos & 1], pos / 2 + 1);
        }
        report();
        return;
    }
    if (wave >= 10) {
        // ---------------------------------------------------- publishing waves
        for (int pos = wave - 10; pos < nT; pos += 2) {
            await(&sh.seq, 4 * (pos + 1), spin_limit, &sh.err);
            T y[kSC];
#pragma unroll
            for (int c = 0; c < kSC; ++c) y[c] = sh.Y[pos % R][lane][c];
            pin(y);
            post(&sh.taken[pos & 1], pos / 2 + 1);
            const i64 i = (i64)pos * kSB + lane, row = phys(i);
#pragma unroll
            for (int c = 0; c < kSC; ++c)
                if (i < n && c < kcl) coherent_store(&B[row + (i64)(c_base + c) * ldb], y[c]);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (lane == 0) coherent_store(&flagsX[pos * CY + cy], epoch);
        }
        report();
        return;
    }
    // The loads of each step must exist for every n: with fewer columns than
    // they span they all read their row's first one (nothing of it is used).
    const i64 cs64 = n >= kSB ? cs : 0, cs16 = n >= 16 ? cs : 0;
    if (wave >= 4) {
        // ---------------------------------------------------------- band waves
        T o[2][4][4];  // distance 3, distance 2
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int tq = 0; tq < 4; ++tq) load4(o[u][tq], Lb, 16 * tq, cs64);
        for (int pos = 0; pos < nT; ++pos) {
            const T* row_p = row_ptr(min(pos + 1, nT - 1));
            acc_t acc = {};
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int q = pos - 3 + u;
                if (q >= 0) {
                    await(&sh.seq, 4 * (q + 1), spin_limit, &sh.err);
#pragma unroll
                    for (int tq = 0; tq < 4; ++tq) product(acc, sh.Y[q % R], tq, o[u][tq]);
                }
                // the next position's operands, under the rest of this one
                const i64 kn = (i64)max(q + 1, 0) * kSB;
#pragma unroll
                for (int tq = 0; tq < 4; ++tq) load4(o[u][tq], row_p, kn + 16 * tq, cs64);
            }
            acc = mfma16(T(0), T(0), acc);  // (as in the helper)
            await(&sh.seq, 4 * (pos - RB) + w + 1, spin_limit, &sh.err);  // the slot's last sums have been taken
#pragma unroll
            for (int v = 0; v < 4; ++v) sh.Sb[pos % RB][16 * w + c16][mfma_row<T>(lane, v)] = acc[v];
            post(&sh.band[w], pos + 1);
        }
        report();
        return;
    }

    // ----------------------------------------------------------------- chain
    __builtin_amdgcn_s_setprio(2);
    T far[4][4], near[3][4];
    // operands for position `next`: tile tq of the block before it (all full
    // blocks), tile tq of its own (a tile past n is not used)
    auto load_far = [&](const T* row, int next, int tq) __attribute__((always_inline)) {
        load4(far[tq], row, (i64)max(next - 1, 0) * kSB + 16 * tq, cs64);
    };
    auto load_near = [&](const T* row, int next, int tq) __attribute__((always_inline)) {
        load4(near[tq], row, lesser((i64)next * kSB + 16 * tq, max(n - 16, 0)), cs16);
    };
    {
        const T* row_p = row_ptr(0);
#pragma unroll
        for (int tq = 0; tq < 4; ++tq) load_far(row_p, 0, tq);
#pragma unroll
        for (int tq = 0; tq < 3; ++tq) load_near(row_p, 0, tq);
    }
    for (int pos = 0; pos < nT; ++pos) {
        const int next = min(pos + 1, nT - 1);
        const T* row_p = row_ptr(next);
        const bool in = (i64)pos * kSB + 16 * w + c16 < n;  // whether this lane's row exists
        acc_t acc = {};
        const T(*Yp)[kSC + 1] = sh.Y[(pos + R - 1) % R];
        // tile tq of the block before; its operand is then reloaded
        auto before = [&](int tq) __attribute__((always_inline)) {
            if (pos > 0) product_when(4 * (pos - 1) + tq + 1, acc, Yp, tq, far[tq]);
            load_far(row_p, next, tq);
        };
        before(0);
        before(1);
        before(2);
        // what was made elsewhere: multipliers, right-hand sides, band sums
        await(&sh.fetched[pos & 1], pos / 2 + 1, spin_limit, &sh.err);
        await(&sh.band[w], pos + 1, spin_limit, &sh.err);
        // (the slot's last block has been published)
        if (pos >= R) await(&sh.taken[(pos - R) & 1], (pos - R) / 2 + 1, spin_limit, &sh.err);
        T m[15], bv[4];
        const T(*Ms)[kSC + 1] = sh.M[pos % RB];
#pragma unroll
        for (int k = 0; k < 15; ++k) m[k] = Ms[16 * w + c16][k];
        const T r = Ms[16 * w + c16][15];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int c = mfma_row<T>(lane, v);
            bv[v] = sh.Bv[pos % RB][16 * w + c16][c] - sh.Sb[pos % RB][16 * w + c16][c];
        }
        pin(m);
        pin(bv);
        before(3);
        // the block's own tiles
        const T(*Y)[kSC + 1] = sh.Y[pos % R];
#pragma unroll
        for (int tq = 0; tq < 3; ++tq) {
            if (tq < w) product_when(4 * pos + tq + 1, acc, Y, tq, near[tq]);
            load_near(row_p, next, tq);
        }
        acc = mfma16(T(0), T(0), acc);  // (as in the helper)
        T a[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) a[v] = in ? bv[v] - acc[v] : T(0);
#pragma unroll
        for (int v = 0; v < NV; ++v) asm volatile("s_nop 0" : "+v"(a[v]));  // all written, two states before the first DPP read
        if constexpr (NV == 1) asm volatile("s_nop 0");
        Substitute<T, NV, 0>::run(a, m);
#pragma unroll
        for (int v = 0; v < 4; ++v) sh.Y[pos % R][16 * w + c16][mfma_row<T>(lane, v)] = v < NV ? a[v < NV ? v : 0] * r : T(0);
        post(&sh.seq, 4 * pos + w + 1);
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
    int base = 0, epoch = 0;
    for (int dir = 0; dir < 2; ++dir) {
        if (dir == 0 ? !forward : !backward) continue;
        ++epoch;
        for (int c0 = 0; c0 < kc; c0 += chain::kMaxSlabs * kSC) {
            const int k = std::min(kc - c0, chain::kMaxSlabs * kSC), CY = (int)ceil_div(k, kSC);
            const unsigned grid = (unsigned)(CY + CY * std::max(0, nT - chain::D - 1));
            int* flags = ctrl + 2 + 2 * nT * (c0 / kSC);
            T* Bc = B + (i64)c0 * ldb;
            T* pc = part + (i64)c0 * n;
            // (n < 16: rows with fewer than four coefficients are read one by one)
            const bool contig = (dir == 1) != upper && n >= 16;
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
