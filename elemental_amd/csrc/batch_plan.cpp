// Host side of the batched HPD factor-and-solve: the plan (size buckets,
// processing order, per-step work prefix sums, device descriptors), the
// launch sequence, its hipGraph capture and replay, and per-matrix results.
#include "batch.hpp"

#include <algorithm>
#include <cmath>
#include <new>
#include <numeric>
#include <vector>

#include "kernels.hpp"

namespace elemamd {

namespace {

template <typename T>
hipError_t upload(T** dst, const std::vector<T>& v) {
    hipError_t e = hipMalloc(dst, sizeof(T) * std::max<size_t>(v.size(), 1));
    if (e != hipSuccess) return e;
    if (!v.empty()) e = hipMemcpy(*dst, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice);
    return e;
}

inline size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

// descriptors of the positions [first, first + count)
BatchArgs plan_args(const BatchPlan* P, int first, int count, bool with_skip) {
    return BatchArgs{count,
                     P->d_n + first,
                     P->d_k + first,
                     P->d_aoff + first,
                     P->d_boff + first,
                     P->d_info + first,
                     with_skip ? P->d_skip + first : nullptr};
}
BatchArgs plan_args(const BatchPlan* P, bool with_skip) { return plan_args(P, 0, P->count, with_skip); }

// The runs and their steps' work prefix sums, from the buckets and their
// launch forms.  Buckets with the same block size share their steps' launches
// (each of which lasts as long as its largest matrix's chain): 1024 matrices
// of n = 16 ... 1024 in six buckets take 10 block steps instead of 17.  On
// failure the plan keeps the runs and the table that it has.
int plan_runs(BatchPlan* P) {
    std::vector<BatchRun> runs;
    for (const BatchBucket& bk : P->buckets) {
        BatchRun* last = runs.empty() ? nullptr : &runs.back();
        if (last != nullptr && bk.grid == 0 && last->grid == 0 && last->nb == bk.nb) {
            last->count += bk.count;
            continue;
        }
        BatchRun r;
        r.nb = bk.nb;
        r.grid = bk.grid;
        r.first = bk.first;
        r.count = bk.count;
        runs.push_back(r);
    }
    const int tile = P->precision == 2 ? 128 : 64;  // of the trailing update
    std::vector<int> prefix;
    auto size = [&](int p) { return P->n[P->order[p]]; };
    for (BatchRun& r : runs) {
        if (r.grid > 0) continue;
        const int nb = r.nb, steps = (size(r.first) + nb - 1) / nb;
        for (int j = 0; j < steps; ++j) {
            BatchRun::Step st;
            st.active = 0;
            while (st.active < r.count && size(r.first + st.active) > j * nb) ++st.active;
            std::vector<int> pt(st.active + 1, 0), ps(st.active + 1, 0);
            for (int q = 0; q < st.active; ++q) {
                const int m = size(r.first + q) - (j + 1) * nb;
                const i64 T = m > 0 ? (m + tile - 1) / tile : 0;
                pt[q + 1] = pt[q] + (m > 0 ? (m + 63) / 64 : 0);  // panel: 64 rows per workgroup
                ps[q + 1] = ps[q] + (int)(T * (T + 1) / 2);       // trailing: lower tiles
            }
            st.trsm_wgs = pt[st.active];
            st.syrk_wgs = ps[st.active];
            st.trsm_prefix_off = (int)prefix.size();
            prefix.insert(prefix.end(), pt.begin(), pt.end());
            st.syrk_prefix_off = (int)prefix.size();
            prefix.insert(prefix.end(), ps.begin(), ps.end());
            r.step.push_back(st);
        }
    }
    std::vector<int> pr(P->count + 1, 0);
    for (int q = 0; q < P->count; ++q) pr[q + 1] = pr[q] + (size(q) + 63) / 64;
    const int res_off = (int)prefix.size();
    prefix.insert(prefix.end(), pr.begin(), pr.end());
    int* table = nullptr;
    if (upload(&table, prefix) != hipSuccess) {
        if (table != nullptr) (void)hipFree(table);
        return kErrHip;
    }
    if (P->d_prefix != nullptr) (void)hipFree(P->d_prefix);  // (waits for work that still reads it)
    P->d_prefix = table;
    P->runs.swap(runs);
    P->res_wgs = pr[P->count];
    P->res_prefix_off = res_off;
    return kOk;
}

}  // namespace

BatchPlan::~BatchPlan() {
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    if (capture_stream) (void)hipStreamDestroy(capture_stream);
    if (d_prefix) (void)hipFree(d_prefix);
    for (void* p : dev_allocs) (void)hipFree(p);
}

int batch_plan_create(int count, const int* n, const int* k, int precision, int nbuckets, const int* bucket_max_n,
                      const int* bucket_nb, BatchPlan** out) {
    if (out == nullptr) return kErrArg;
    *out = nullptr;
    if (count < 0 || (count > 0 && (n == nullptr || k == nullptr))) return kErrArg;
    if (precision < 0 || precision > 2) return kErrArg;
    if (nbuckets < 1 || bucket_max_n == nullptr || bucket_nb == nullptr) return kErrArg;
    for (int b = 0; b < nbuckets; ++b) {
        if (bucket_nb[b] < 1 || bucket_nb[b] > 128) return kErrArg;
        if (b > 0 && bucket_max_n[b] <= bucket_max_n[b - 1]) return kErrArg;
    }
    for (int i = 0; i < count; ++i)
        if (n[i] < 1 || k[i] < 1) return kErrArg;
    auto* P = new BatchPlan();
    P->count = count;
    P->precision = precision;
    P->n.assign(n, n + count);
    P->k.assign(k, k + count);
    // packed layout in the caller's order
    P->a_off.resize(count);
    P->b_off.resize(count);
    i64 ao = 0, bo = 0;
    for (int i = 0; i < count; ++i) {
        P->a_off[i] = ao;
        P->b_off[i] = bo;
        ao += (i64)P->n[i] * P->n[i];
        bo += (i64)P->n[i] * P->k[i];
        P->kmax = std::max(P->kmax, P->k[i]);
    }
    P->a_total = ao;
    P->b_total = bo;
    // bucket of each matrix; processing order = by decreasing size, so that
    // the matrices still active at step j form a prefix and each bucket is a
    // range
    std::vector<int> bk(count);
    for (int i = 0; i < count; ++i) {
        int b = 0;
        while (b < nbuckets - 1 && P->n[i] > bucket_max_n[b]) ++b;
        bk[i] = b;
    }
    P->order.resize(count);
    std::iota(P->order.begin(), P->order.end(), 0);
    std::stable_sort(P->order.begin(), P->order.end(),
                     [&](int a, int b) { return P->n[a] > P->n[b]; });
    std::vector<int> ns(count), ks(count);
    std::vector<i64> aos(count), bos(count);
    for (int p = 0; p < count; ++p) {
        const int i = P->order[p];
        ns[p] = P->n[i];
        ks[p] = P->k[i];
        aos[p] = P->a_off[i];
        bos[p] = P->b_off[i];
    }
    int pos = 0;
    for (int b = nbuckets - 1; b >= 0; --b) {
        BatchBucket B;
        B.index = b;
        B.nb = bucket_nb[b];
        B.first = pos;
        while (pos < count && bk[P->order[pos]] == b) ++pos;
        B.count = pos - B.first;
        if (B.count > 0) P->buckets.push_back(B);
    }
    int *d_n = nullptr, *d_k = nullptr, *d_ints = nullptr;
    i64 *d_ao = nullptr, *d_bo = nullptr;
    double* d_dbl = nullptr;
    bool ok = upload(&d_n, ns) == hipSuccess;
    if (d_n) P->dev_allocs.push_back(d_n);
    ok = ok && upload(&d_k, ks) == hipSuccess;
    if (d_k) P->dev_allocs.push_back(d_k);
    ok = ok && upload(&d_ao, aos) == hipSuccess;
    if (d_ao) P->dev_allocs.push_back(d_ao);
    ok = ok && upload(&d_bo, bos) == hipSuccess;
    if (d_bo) P->dev_allocs.push_back(d_bo);
    ok = ok && plan_runs(P) == kOk;
    ok = ok && hipMalloc(&d_ints, sizeof(int) * (size_t)(3 * count + nbuckets)) == hipSuccess;
    if (d_ints) P->dev_allocs.push_back(d_ints);
    // eta, rscale (kmax per matrix), reduction scratch (1 + 3 kmax per matrix)
    ok = ok && hipMalloc(&d_dbl, sizeof(double) * (size_t)std::max(count * (2 + 4 * P->kmax), 1)) == hipSuccess;
    if (d_dbl) P->dev_allocs.push_back(d_dbl);
    if (!ok) {
        delete P;
        return kErrHip;
    }
    P->d_n = d_n;
    P->d_k = d_k;
    P->d_aoff = d_ao;
    P->d_boff = d_bo;
    P->d_info = d_ints;
    P->d_skip = d_ints + count;
    P->d_iters = d_ints + 2 * count;
    P->d_counters = d_ints + 3 * count;
    P->d_eta = d_dbl;
    P->d_rscale = d_dbl + count;
    P->d_red = d_dbl + (size_t)count * (1 + P->kmax);
    *out = P;
    return kOk;
}

int batch_set_launch(BatchPlan* P, const int* bucket_grid) {
    if (P == nullptr || bucket_grid == nullptr) return kErrArg;
    for (const BatchBucket& bk : P->buckets)
        if (bucket_grid[bk.index] < 0 || (bucket_grid[bk.index] > 0 && bk.nb > kPersistMaxNb)) return kErrArg;
    std::vector<BatchBucket> before;
    int rc = kErrHip;
    try {  // (no exception leaves the C interface)
        before = P->buckets;
        bool same = true;
        for (BatchBucket& bk : P->buckets) {
            same = same && bk.grid == bucket_grid[bk.index];
            bk.grid = bucket_grid[bk.index];
        }
        if (same) return kOk;
        rc = plan_runs(P);
    } catch (const std::bad_alloc&) {
    }
    if (rc != kOk) {
        if (!before.empty()) P->buckets.swap(before);
        return rc;
    }
    if (P->graph_exec) {  // captured with the previous launch forms and table
        (void)hipGraphExecDestroy(P->graph_exec);
        P->graph_exec = nullptr;
    }
    return kOk;
}

size_t batch_workspace_bytes(const BatchPlan* P) {
    if (P->precision == 0) return 0;
    // float copy of every A (the factor), FP64 iterate and residual, float correction
    return al256(sizeof(float) * P->a_total) + 2 * al256(sizeof(double) * P->b_total) +
           al256(sizeof(float) * P->b_total);
}

// The launch sequence: kernels only, fixed shapes, so it can be captured.
static int enqueue(BatchPlan* P, double* A, double* B, void* work, hipStream_t s) {
    if (P->count == 0) return kOk;
    // info, skip, iters, the persistent launches' counters
    ELEMAMD_HIP_TRY(launch_fill_int(P->d_info, 0, 3 * P->count + (int)P->runs.size(), s));
    const bool f32 = P->precision != 0;
    const int mode = P->precision;  // trailing update: 0 FP64, 1 FP32, 2 BF16x3
    float* S = nullptr;
    double *X = nullptr, *R = nullptr;
    float* Rf = nullptr;
    if (f32) {
        char* w = (char*)work;
        S = (float*)w;
        w += al256(sizeof(float) * P->a_total);
        X = (double*)w;
        w += al256(sizeof(double) * P->b_total);
        R = (double*)w;
        w += al256(sizeof(double) * P->b_total);
        Rf = (float*)w;
    }
    const BatchArgs a = plan_args(P, false);
    const BatchArgs ai = plan_args(P, true);
    const int* res_prefix = P->d_prefix + P->res_prefix_off;
    // the refinement's first residual (X = 0) reads all of A: the float copy
    // to factor is made on the way
    if (f32)
        ELEMAMD_HIP_TRY(batch_residual(ai, A, X, B, R, res_prefix, P->res_wgs, P->d_red, P->d_eta, P->d_rscale,
                                       P->kmax, s, S));
    void* F = f32 ? (void*)S : (void*)A;
    for (const BatchRun& r : P->runs) {
        const BatchArgs ar = plan_args(P, r.first, r.count, false);
        if (r.grid > 0)  // the whole factorization in one launch
            ELEMAMD_HIP_TRY(batch_persistent(ar, F, mode, r.nb, P->d_counters + (&r - P->runs.data()), r.grid, s));
        for (size_t j = 0; j < r.step.size(); ++j) {
            const BatchRun::Step& st = r.step[j];
            ELEMAMD_HIP_TRY(batch_potrf(ar, F, f32, (int)j, r.nb, st.active, s));
            ELEMAMD_HIP_TRY(
                batch_trsm(ar, F, f32, (int)j, r.nb, P->d_prefix + st.trsm_prefix_off, st.active, st.trsm_wgs, s));
            ELEMAMD_HIP_TRY(
                batch_syrk(ar, F, mode, (int)j, r.nb, P->d_prefix + st.syrk_prefix_off, st.active, st.syrk_wgs, s));
        }
    }
    if (!f32) {
        ELEMAMD_HIP_TRY(batch_solve(a, A, B, false, P->kmax, s));
        return kOk;
    }
    // low-precision factor + FP64-residual refinement from X = 0: a fixed
    // number of sweeps (the sequence is replayable); a converged matrix is
    // skipped by every kernel of the remaining sweeps
    ELEMAMD_HIP_TRY(batch_copy_rhs(a, nullptr, X, nullptr, s));  // X := 0
    for (int it = 0; it < P->ir_sweeps; ++it) {
        if (it > 0)
            ELEMAMD_HIP_TRY(batch_residual(ai, A, X, B, R, res_prefix, P->res_wgs, P->d_red, P->d_eta, P->d_rscale,
                                           P->kmax, s));
        ELEMAMD_HIP_TRY(batch_ir_prepare(ai, P->d_eta, P->tol, R, P->d_rscale, Rf, P->kmax, P->d_iters, s));
        ELEMAMD_HIP_TRY(batch_solve(ai, S, Rf, true, P->kmax, s));
        ELEMAMD_HIP_TRY(batch_ir_update(ai, Rf, P->d_rscale, X, P->kmax, s));
    }
    // backward error of every matrix, then X -> B
    ELEMAMD_HIP_TRY(batch_residual(a, A, X, B, R, res_prefix, P->res_wgs, P->d_red, P->d_eta, nullptr, P->kmax, s));
    ELEMAMD_HIP_TRY(batch_copy_rhs(a, X, B, nullptr, s));
    return kOk;
}

int batch_hpd_solve(BatchPlan* P, double* A, double* B, void* work, size_t work_bytes, bool use_graph,
                    hipStream_t s) {
    if (P == nullptr || (P->count > 0 && (A == nullptr || B == nullptr))) return kErrArg;
    if (work_bytes < batch_workspace_bytes(P) || (P->precision != 0 && work == nullptr)) return kErrWorkspace;
    if (!use_graph) return enqueue(P, A, B, work, s);
    if (P->graph_exec == nullptr || P->g_A != A || P->g_B != B || P->g_work != work) {
        if (P->graph_exec) {
            ELEMAMD_HIP_TRY(hipGraphExecDestroy(P->graph_exec));
            P->graph_exec = nullptr;
        }
        // capture on a private stream (the caller's may be the default
        // stream, which cannot be captured); the graph is launched on `s`
        if (P->capture_stream == nullptr)
            ELEMAMD_HIP_TRY(hipStreamCreateWithFlags(&P->capture_stream, hipStreamNonBlocking));
        hipStream_t cs = P->capture_stream;
        hipGraph_t g = nullptr;
        ELEMAMD_HIP_TRY(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
        const int rc = enqueue(P, A, B, work, cs);
        const hipError_t e = hipStreamEndCapture(cs, &g);
        if (rc != kOk) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        ELEMAMD_HIP_TRY(e);
        const hipError_t ei = hipGraphInstantiate(&P->graph_exec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (ei != hipSuccess) {
            P->graph_exec = nullptr;
            return kErrHip;
        }
        P->g_A = A;
        P->g_B = B;
        P->g_work = work;
    }
    ELEMAMD_HIP_TRY(hipGraphLaunch(P->graph_exec, s));
    return kOk;
}

int batch_results(const BatchPlan* P, int* info, double* eta, int* iters, hipStream_t s) {
    if (P == nullptr) return kErrArg;
    if (P->count == 0) return kOk;
    std::vector<int> hi(3 * (size_t)P->count);
    std::vector<double> he(P->count);
    ELEMAMD_HIP_TRY(hipMemcpyAsync(hi.data(), P->d_info, sizeof(int) * hi.size(), hipMemcpyDeviceToHost, s));
    ELEMAMD_HIP_TRY(hipMemcpyAsync(he.data(), P->d_eta, sizeof(double) * he.size(), hipMemcpyDeviceToHost, s));
    ELEMAMD_HIP_TRY(hipStreamSynchronize(s));
    for (int p = 0; p < P->count; ++p) {
        const int i = P->order[p];
        if (info) info[i] = hi[p];
        if (iters) iters[i] = hi[2 * (size_t)P->count + p];
        if (eta) eta[i] = P->precision == 0 ? NAN : he[p];
    }
    return kOk;
}

int batch_backward_error(const BatchPlan* P, const double* A, const double* X, const double* B, double* R,
                         double* eta, hipStream_t s) {
    if (P == nullptr || eta == nullptr) return kErrArg;
    if (P->count == 0) return kOk;
    ELEMAMD_HIP_TRY(batch_residual(plan_args(P, false), A, X, B, R, P->d_prefix + P->res_prefix_off, P->res_wgs,
                                   P->d_red, P->d_eta, nullptr, P->kmax, s));
    std::vector<double> he(P->count);
    ELEMAMD_HIP_TRY(hipMemcpyAsync(he.data(), P->d_eta, sizeof(double) * he.size(), hipMemcpyDeviceToHost, s));
    ELEMAMD_HIP_TRY(hipStreamSynchronize(s));
    for (int p = 0; p < P->count; ++p) eta[P->order[p]] = he[p];
    return kOk;
}

}  // namespace elemamd
