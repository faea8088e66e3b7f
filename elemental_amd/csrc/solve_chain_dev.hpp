// The parts of a triangular solve as a chain of 16-row tiles (solve_chain.hip
// explains the whole): the waves that one workgroup needs for one 64-row block
// after another.  The solves with one factor (solve_chain.hip) add helper
// workgroups; the batched ones (batch.hip) keep a matrix in one workgroup.
#pragma once

#include "common.hpp"
#include "solve_dev.hpp"

namespace elemamd {
namespace chain {

constexpr int kWaves = 12, kThreads = 64 * kWaves;

// Right-hand sides of a workgroup with NV accumulator registers that hold
// some (FP64: a register holds four columns; FP32's interleave 16).
template <typename T>
constexpr int columns(int nv) {
    return sizeof(T) == 8 ? 4 * nv : kSC;
}

// KC: columns; R: solved blocks kept; RB: blocks of right-hand sides,
// multipliers and sums ahead of the chain.
template <typename T, int KC_, int R_, int RB_>
struct Lds {
    typedef T value;
    static constexpr int KC = KC_, R = R_, RB = RB_;
    T Y[R][kSB][KC + 1];    // solved blocks [row][column]
    T Bv[RB][kSB][KC + 1];  // right-hand sides less the sums made elsewhere
    T Sb[RB][kSB][KC + 1];  // the band's sums
    // multipliers [row][column in the tile], [15]: reciprocal diagonal; for a
    // tile with one that is not an ordinary number the coefficients themselves
    // and NaN in [15]; [16]: the reciprocal diagonal in either case
    T M[RB][kSB][17];
    int seq;                // tiles solved
    int fetched[2];         // blocks in Bv and M (counting each fetching wave's own)
    int taken[2];           // blocks read out of Y (counting each publishing wave's own)
    int out[2];             // blocks written to memory (the same)
    int band[4];            // blocks in Sb, rows of wave w
    int err;                // a wait gave up
    __device__ __forceinline__ void reset() {
        seq = err = 0;
        for (int v = 0; v < 2; ++v) fetched[v] = taken[v] = out[v] = 0;
        for (int v = 0; v < 4; ++v) band[v] = 0;
    }
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

// Classes of v_cmp_class: normal numbers, infinities, infinities and NaN.
constexpr int kNormal = 0x108, kInfinite = 0x204, kNotFinite = 0x207;
__device__ __forceinline__ bool is_class(double x, int c) { return __builtin_amdgcn_class(x, c); }
__device__ __forceinline__ bool is_class(float x, int c) { return __builtin_amdgcn_classf(x, c); }

// Whether all of m are normal numbers, from their leading bits x: 2 x less the
// least normal number's is below the bound for these alone (zeros and
// subnormal numbers wrap around to the top, where infinities and NaN are).
__device__ __forceinline__ unsigned leading_bits(double x) { return (unsigned)__double2hiint(x); }
__device__ __forceinline__ unsigned leading_bits(float x) { return (unsigned)__float_as_int(x); }
template <typename T>
__device__ __forceinline__ bool all_normal(const T (&m)[15]) {
    constexpr unsigned least = sizeof(T) == 8 ? 0x00200000u : 0x01000000u, bound = 0u - 2 * least;
    unsigned worst = 0;
#pragma unroll
    for (int k = 0; k < 15; ++k) worst = max(worst, (leading_bits(m[k]) << 1) - least);
    return worst < bound;
}

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
    // m := l_ck / l_kk without the mask
    static __device__ __forceinline__ void products(T (&m)[15], const T (&l)[15], T r) {
        m[K] = l[K] * row_lane<K>(r);
        if constexpr (K < 14) Multipliers<T, K + 1>::products(m, l, r);
    }
};


// What rows with fewer than 16 coefficients read in a group's place: nothing
// of it is used.
static __device__ double kNoRow[8] = {};

// The factor's rows in solve order.  TRANS: the backward direction.  upper:
// the factor is stored in the upper triangle.  CONTIG: a row's coefficients
// are contiguous (TRANS != upper).
template <typename T, bool TRANS, bool CONTIG>
struct Rows {
    static constexpr int sgn = TRANS ? -1 : 1;
    int n, w, c16, g;
    const T* L;
    i64 rs, cs;
    // Loads of a step must exist for every n: with fewer columns than they
    // span they all read their row's first one (nothing of it is used).
    i64 cs64, cs16;
    __device__ __forceinline__ Rows(int n_, const T* L_, i64 ldl, bool upper, int w_, int lane)
        : n(n_), w(w_), c16(lane & 15), g(lane >> 4), L(TRANS ? L_ + (i64)(n_ - 1) * (1 + ldl) : L_) {
        const bool read_t = CONTIG || TRANS != upper;  // the coefficient (i, k) is stored at (k, i)
        rs = sgn * (read_t ? ldl : 1);
        cs = read_t ? sgn : sgn * ldl;
        cs64 = n >= kSB ? cs : 0;
        cs16 = n >= 16 ? cs : 0;
    }
    __device__ __forceinline__ i64 phys(i64 i) const { return TRANS ? n - 1 - i : i; }  // stored row of row i
    // rows past n (in the last block) repeat row n - 1: nothing of them is used
    __device__ __forceinline__ const T* row(int pos) const {
        return n >= 16 ? L + lesser((i64)pos * kSB + 16 * w + c16, n - 1) * rs : (const T*)kNoRow + 4;
    }
    // MFMA operand: this lane's row, columns k0 + 4 g + ks, ks < 4
    __device__ __forceinline__ void load4(T (&o)[4], const T* r, i64 k0, i64 step) const {
        const T* p = r + (k0 + 4 * g) * step;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) o[ks] = CONTIG ? p[sgn * ks] : p[ks * step];
    }
};

// acc += tile tq of a solved block times the operand o
template <typename T, int LD, typename A>
__device__ __forceinline__ void product(A& acc, const T (*Y)[LD], int tq, const T (&o)[4], int c16, int g) {
    const int c = LD - 1 < 16 ? min(c16, LD - 2) : c16;
    T y[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) y[ks] = Y[16 * tq + 4 * g + ks][c];
    pin(y);  // (all four reads in flight together)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) acc = mfma16(y[ks], o[ks], acc);
}
// the same with a tile that may still be on its way: the sequence number and
// the tile are read together (LDS serves a wave's reads in order, so a tile
// read after a sufficient number is complete)
template <typename S, typename T, int LD, typename A>
__device__ __forceinline__ void product_when(S& sh, int need, A& acc, const T (*Y)[LD], int tq, const T (&o)[4],
                                             int c16, int g, long limit) {
    const int c = LD - 1 < 16 ? min(c16, LD - 2) : c16;
    T y[4];
    long spins = 0;
    for (;;) {
        const int have = peek(&sh.seq);
        asm volatile("" ::: "memory");
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) y[ks] = Y[16 * tq + 4 * g + ks][c];
        pin(y);
        if (have >= need) break;
        if (++spins > limit) {
            sh.err = 1;
            break;
        }
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) acc = mfma16(y[ks], o[ks], acc);
}

// Fetching wave u (of two): right-hand sides and multipliers of the blocks u,
// u + 2, ... into LDS.  B: the slab's first column; kcl: its columns (columns
// past it repeat the last one: they are solved and dropped).  less(pos, i, b):
// subtracts what was summed elsewhere from row i's right-hand sides.
template <typename T, bool TRANS, bool CONTIG, typename S, typename F>
__device__ __forceinline__ void fetch_blocks(S& sh, const Rows<T, TRANS, CONTIG>& L, int u, int lane, int nT, int kcl,
                                             const T* B, i64 ldb, bool unit, long limit, F less) {
    constexpr int KC = S::KC, RB = S::RB;
    for (int pos = u; pos < nT; pos += 2) {
        const i64 i = (i64)pos * kSB + lane;
        const bool in = i < L.n;
        const i64 ic = in ? i : L.n - 1, t0 = ic - (ic & 15);  // (clamped) row, its tile's first row
        T m[15], l[15], b[KC];
#pragma unroll
        for (int k = 0; k < 15; ++k) l[k] = L.L[ic * L.rs + lesser(t0 + k, ic) * L.cs];
        const T dd = L.L[ic * L.rs + ic * L.cs];
        const i64 row = L.phys(ic);
#pragma unroll
        for (int c = 0; c < KC; ++c) b[c] = B[row + (i64)min(c, kcl - 1) * ldb];
        // multipliers l_ck / l_kk of the tile's earlier columns
        const T r = in && !unit ? T(1) / dd : T(1);
        const int c16 = in ? lane & 15 : 0;
        Multipliers<T, 0>::products(m, l, r);
        // (a first look at all exponents; tiles with a zero take the second)
        bool careful = false;
        if (__ballot(!all_normal(m)) != 0) {
            // a multiplier that is not a normal number, of a coefficient other
            // than zero, has lost its value; an infinite one with l_kk = 0 has not
            bool lost = r != r;
#pragma unroll 1
            for (int k = 0; k < 15; ++k) {
                const T lk = L.L[ic * L.rs + lesser(t0 + k, ic) * L.cs], rk = __shfl(r, (lane & 48) + k);
                lost = lost | ((k < c16) & (lk != T(0)) & !is_class(lk * rk, kNormal) & !is_class(rk, kInfinite));
            }
            // the whole tile takes the coefficients then
            careful = (__ballot(lost) >> (lane & 48) & 0xffff) != 0;
            if (careful)
#pragma unroll
                for (int k = 0; k < 15; ++k) m[k] = l[k];
        }
#pragma unroll
        for (int k = 0; k < 15; ++k) m[k] = k < c16 ? m[k] : T(0);
        less(pos, ic, b);
        await(&sh.seq, 4 * (pos - RB + 1), limit, &sh.err);  // the slot's last block is solved
#pragma unroll
        for (int c = 0; c < KC; ++c) sh.Bv[pos % RB][lane][c] = b[c];
#pragma unroll
        for (int k = 0; k < 15; ++k) sh.M[pos % RB][lane][k] = m[k];
        sh.M[pos % RB][lane][15] = careful ? T(__builtin_nan("")) : r;
        sh.M[pos % RB][lane][16] = r;
        post(&sh.fetched[u], pos / 2 + 1);
    }
}

// Publishing wave u (of two): the solved blocks u, u + 2, ... to B; done(pos)
// once a block is in memory.  COHERENT: other workgroups read it.
template <bool COHERENT, typename T, bool TRANS, bool CONTIG, typename S, typename F>
__device__ __forceinline__ void publish_blocks(S& sh, const Rows<T, TRANS, CONTIG>& L, int u, int lane, int nT, int kcl,
                                               T* B, i64 ldb, long limit, F done) {
    constexpr int KC = S::KC, R = S::R;
    for (int pos = u; pos < nT; pos += 2) {
        await(&sh.seq, 4 * (pos + 1), limit, &sh.err);
        T y[KC];
#pragma unroll
        for (int c = 0; c < KC; ++c) y[c] = sh.Y[pos % R][lane][c];
        pin(y);
        post(&sh.taken[u], pos / 2 + 1);
        const i64 i = (i64)pos * kSB + lane, row = L.phys(i);
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            if (i < L.n && c < kcl) {
                if constexpr (COHERENT) coherent_store(&B[row + (i64)c * ldb], y[c]);
                else B[row + (i64)c * ldb] = y[c];
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        done(pos);
    }
}

// The band's sums of position pos are taken over by the chain.
template <typename T, typename S, typename A>
__device__ __forceinline__ void hand_over(S& sh, int pos, int w, int lane, const A& acc, long limit) {
    await(&sh.seq, 4 * (pos - S::RB) + w + 1, limit, &sh.err);  // the slot's last sums have been taken
#pragma unroll
    for (int v = 0; v < (S::KC + 3) / 4; ++v) sh.Sb[pos % S::RB][16 * w + (lane & 15)][mfma_row<T>(lane, v)] = acc[v];
    post(&sh.band[w], pos + 1);
}

// A tile once more, row by row as the reference's loop: x_k = a_k r_k, then
// a_c -= l_ck x_k for the later rows only.  The substitution in registers lets
// a row that is not finite into the tile's earlier rows (zero times infinity),
// and its multipliers l_ck / l_kk may overflow or vanish where x_k does not;
// the chain comes here when a result is not finite, which the NaN of a tile
// kept as coefficients sees to.  The rows pass through their places in sh.Y.
// n = 4096, 16 columns, forward: 253 us, 1130 with every tile solved here; the
// tests alone cost little (n = 8192, both solves: 1008 us with and without
// them; 20000 matrices of n = 8 ... 16, FP64, 0.97 and 1.00 ms).
template <int NV, typename S, typename A>
__device__ __forceinline__ void solve_tile_careful(S& sh, int pos, int w, int lane, bool in, const A& acc) {
    typedef typename S::value T;
    const int c16 = lane & 15, row = 16 * w + c16;
    const T(*Ms)[17] = sh.M[pos % S::RB];
    T(*Y)[S::KC + 1] = sh.Y[pos % S::R];
    const bool coefficients = Ms[row][15] != Ms[row][15];
    T a[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int c = mfma_row<T>(lane, v);
        a[v] = in ? sh.Bv[pos % S::RB][row][c] - sh.Sb[pos % S::RB][row][c] - acc[v] : T(0);
    }
#pragma unroll 1
    for (int k = 0; k < 15; ++k) {
        const T m = Ms[row][k], rk = Ms[16 * w + k][16];
#pragma unroll
        for (int v = 0; v < NV; ++v) Y[row][mfma_row<T>(lane, v)] = a[v];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            // (m has l_ck's zeros and, but for r_k's, its sign)
            const T ak = Y[16 * w + k][mfma_row<T>(lane, v)], xk = ak * rk;
            const bool far = !coefficients & is_class(xk, kNotFinite);
            const T f = far & (rk < T(0)) ? -m : m, x = coefficients | far ? xk : ak;
            if (in & (c16 > k)) a[v] = fma(-f, x, a[v]);
        }
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) Y[row][mfma_row<T>(lane, v)] = a[v] * Ms[row][16];
}

// Chain wave w: solves the tiles 4 pos + w.
template <int NV, typename T, bool TRANS, bool CONTIG, typename S>
__device__ __forceinline__ void solve_tiles(S& sh, const Rows<T, TRANS, CONTIG>& L, int w, int lane, int nT, long limit) {
    typedef typename Acc4<T>::type acc_t;
    constexpr int R = S::R, RB = S::RB, LD = S::KC + 1;
    const int c16 = lane & 15, g = lane >> 4, n = L.n;
    T far[4][4], near[3][4];
    // operands for position `next`: tile tq of the block before it (all full
    // blocks), tile tq of its own (a tile past n is not used)
    auto load_far = [&](const T* row, int next, int tq) __attribute__((always_inline)) {
        L.load4(far[tq], row, (i64)max(next - 1, 0) * kSB + 16 * tq, L.cs64);
    };
    auto load_near = [&](const T* row, int next, int tq) __attribute__((always_inline)) {
        L.load4(near[tq], row, lesser((i64)next * kSB + 16 * tq, max(n - 16, 0)), L.cs16);
    };
    {
        const T* row = L.row(0);
#pragma unroll
        for (int tq = 0; tq < 4; ++tq) load_far(row, 0, tq);
#pragma unroll
        for (int tq = 0; tq < 3; ++tq) load_near(row, 0, tq);
    }
    for (int pos = 0; pos < nT; ++pos) {
        const int next = min(pos + 1, nT - 1);
        const T* row = L.row(next);
        const bool in = (i64)pos * kSB + 16 * w + c16 < n;  // whether this lane's row exists
        acc_t acc = {};
        const T(*Yp)[LD] = sh.Y[(pos + R - 1) % R];
        // tile tq of the block before; its operand is then reloaded
        auto before = [&](int tq) __attribute__((always_inline)) {
            if (pos > 0) product_when(sh, 4 * (pos - 1) + tq + 1, acc, Yp, tq, far[tq], c16, g, limit);
            load_far(row, next, tq);
        };
        before(0);
        before(1);
        before(2);
        // what was made elsewhere: multipliers, right-hand sides, band sums
        await(&sh.fetched[pos & 1], pos / 2 + 1, limit, &sh.err);
        await(&sh.band[w], pos + 1, limit, &sh.err);
        // (the slot's last block has been published)
        if (pos >= R) await(&sh.taken[(pos - R) & 1], (pos - R) / 2 + 1, limit, &sh.err);
        T m[15], bv[NV];
        const T(*Ms)[17] = sh.M[pos % RB];
#pragma unroll
        for (int k = 0; k < 15; ++k) m[k] = Ms[16 * w + c16][k];
        const T r = Ms[16 * w + c16][15];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int c = mfma_row<T>(lane, v);
            bv[v] = sh.Bv[pos % RB][16 * w + c16][c] - sh.Sb[pos % RB][16 * w + c16][c];
        }
        pin(m);
        pin(bv);
        before(3);
        // the block's own tiles
        const T(*Y)[LD] = sh.Y[pos % R];
#pragma unroll
        for (int tq = 0; tq < 3; ++tq) {
            if (tq < w) product_when(sh, 4 * pos + tq + 1, acc, Y, tq, near[tq], c16, g, limit);
            load_near(row, next, tq);
        }
        // dependent zero-operand MFMA before the accumulator is read (the
        // compiler's wait states after a loop back edge are short for FP64 MFMA)
        acc = mfma16(T(0), T(0), acc);
        T a[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) a[v] = in ? bv[v] - acc[v] : T(0);
#pragma unroll
        for (int v = 0; v < NV; ++v) asm volatile("s_nop 0" : "+v"(a[v]));  // all written, two states before the first DPP read
        if constexpr (NV == 1) asm volatile("s_nop 0");
        Substitute<T, NV, 0>::run(a, m);
        bool lost = false;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            a[v] *= r;
            sh.Y[pos % R][16 * w + c16][mfma_row<T>(lane, v)] = a[v];
            lost = lost | is_class(a[v], kNotFinite);
        }
        if (__ballot(lost) != 0) solve_tile_careful<NV>(sh, pos, w, lane, in, acc);
        post(&sh.seq, 4 * pos + w + 1);
    }
}

}  // namespace chain
}  // namespace elemamd
