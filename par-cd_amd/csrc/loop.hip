// The refinement loop of main.cpp:226-266 kept on the device.
//
// One pass (compress, metric, stop rule, then a propagation step or a
// merging step, with the statistics update) is captured once as a hipGraph
// per step kind and replayed in the order of the schedule: -s 0 propagates
// every pass, -s 1 merges every pass, -s 2 alternates, starting with
// propagation (main.cpp:247-258); every rule, WCC once the graph's
// triangles are counted.  The pass number, the previous score and the
// stop rule (main.cpp:241-242, -n, the iteration cap) live in a device
// record; the captured step reads its step number from it, so every
// replay is the next pass.  When the rule fires, or the requested number of
// passes is reached, the pass freezes the record and keeps a copy of the
// compressed labels and the renumbered statistics; from then on the step
// number is -1, so further replays select no vertex and change nothing.
// The host launches a few replays at a time and reads the record once per
// batch of replays, never once per pass; at the end it puts the kept copy
// back.  The result equals pcd_iterate called pass by pass.
//
// Under modularity and CPM with -s 0 a pass takes the fused form: its
// compression, metric, rule and bookkeeping share launches (fused_compress_dev),
// and no copy is kept, since what the replays after the stop leave is the
// stopped pass's own result: a compression of compressed labels changes
// nothing and no vertex moves.
#include <algorithm>
#include <chrono>
#include <cstring>

#include "../host/hostutil.hpp"
#include "prims.h"

namespace pcd {

__global__ void k_loop_rule(LoopState *s, const double *score, const int32_t *dk, LoopParams p) {
    loop_rule(s, *score, *dk, p);
}

__global__ void k_loop_snapshot(const LoopState *s, int n, const int32_t *labels, const CommStats *stats,
                                int32_t *snap_labels, CommStats *snap_stats) {
    if (!s->just) return;
    const int k = s->k_freeze;
    const int stride = gridDim.x * blockDim.x;
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride) snap_labels[v] = labels[v];
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < k; c += stride) snap_stats[c] = stats[c];
}

__global__ void k_loop_next(LoopState *s) { loop_next(s); }

// a pass that stopped after its propagation had run: no vertex moves
__global__ void k_loop_drop(const LoopState *s, int n, const int32_t *labels, int32_t *next) {
    if (!s->just) return;
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) next[v] = labels[v];
}

enum PassKind { PASS_PROPAGATE = 0, PASS_MERGE = 1 };

// step kind of pass `it` under schedule `strategy` (main.cpp:247-258)
static int pass_kind(int strategy, int it) {
    if (strategy == 0) return PASS_PROPAGATE;
    if (strategy == 1) return PASS_MERGE;
    return it % 2 == 0 ? PASS_PROPAGATE : PASS_MERGE;
}

// What a captured pass depends on: the buffers, the tuning and the job.
struct PassKey {
    const void *ptrs[4] = {nullptr, nullptr, nullptr, nullptr};
    int64_t alloc_gen = -1, tune_gen = -1;
    pcd_rule rule{};
    double cc = 0;  // clustering coefficient, which WCC's gains hold
    double frac = 0, threshold = 0;
    uint64_t seed = 0;
    int tie = 0, max_iter = 0, cap = 0;
    int rounds = 0;      // of a merging pass; 0 for a propagation pass
    bool fused = false;  // a propagation pass in its fused form: no copy is kept

    bool operator==(const PassKey &o) const {
        return std::equal(ptrs, ptrs + 4, o.ptrs) && alloc_gen == o.alloc_gen && tune_gen == o.tune_gen &&
               rule.kind == o.rule.kind && rule.lambda == o.rule.lambda && cc == o.cc && frac == o.frac &&
               threshold == o.threshold && seed == o.seed && tie == o.tie && max_iter == o.max_iter && cap == o.cap && rounds == o.rounds &&
               fused == o.fused;
    }
};

// The captured passes, each with its own key (schedules -s 0, 1 and 2 share
// the two slots, and a call recaptures only the kinds it replays), and their
// state.
struct Loop {
    hipGraphExec_t exec[2] = {nullptr, nullptr};  // by PassKind
    PassKey key[2];
    LoopState *d_state = nullptr, *h_state = nullptr;
    int32_t *snap_labels = nullptr;
    CommStats *snap_stats = nullptr;
    bool broken = false;  // capture failed once: this context runs pass by pass
};

static Loop *loop_of(pcd_ctx *ctx) { return (Loop *)ctx->loop; }

void loop_release(pcd_ctx *ctx) {
    Loop *L = loop_of(ctx);
    if (!L) return;
    for (hipGraphExec_t &e : L->exec)
        if (e) (void)hipGraphExecDestroy(e);
    if (L->h_state) (void)hipHostFree(L->h_state);
    // device buffers belong to the context's allocation list
    delete L;
    ctx->loop = nullptr;
}

static PassKey pass_key(pcd_ctx *ctx, const pcd_job *job, int cap, int kind, int rounds, bool fused) {
    PassKey k;
    const void *p[4] = {ctx->d_labels, ctx->d_labels_alt, ctx->d_stats, ctx->d_stats_alt};
    std::copy(p, p + 4, k.ptrs);
    k.alloc_gen = ctx->alloc_gen;
    k.tune_gen = ctx->tune_gen;
    k.rule = job->rule;
    k.cc = ctx->cc;
    k.frac = job->frac;
    k.threshold = job->threshold;
    k.seed = job->seed;
    k.tie = job->tie;
    k.max_iter = job->max_iter;
    k.cap = cap;
    k.rounds = kind == PASS_MERGE ? rounds : 0;
    k.fused = fused;
    return k;
}

// Everything the passes of `kinds` (bit per PassKind) may otherwise allocate
// lazily: no allocation may happen while the stream captures, nor between two
// captures (it would make the first one's key stale).
static int reserve_passes(pcd_ctx *ctx, Loop *L, unsigned kinds, bool fused) {
    PCD_TRY(ensure_scan_parts(ctx, (int64_t)ctx->n + ctx->num_stat_items + 64));
    if ((kinds >> PASS_MERGE) & 1) PCD_TRY(merge_rows_reserve(ctx));
    if (!L->d_state) PCD_TRY(dev_alloc_t(ctx, &L->d_state, 1));
    if (!L->h_state && hipHostMalloc((void **)&L->h_state, sizeof(LoopState), hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        L->h_state = nullptr;
        return fail(PCD_E_NOMEM, "pinned loop state");
    }
    if (!fused && !L->snap_labels) PCD_TRY(dev_alloc_t(ctx, &L->snap_labels, ctx->n + 1));
    if (!fused && !L->snap_stats) PCD_TRY(dev_alloc_t(ctx, &L->snap_stats, ctx->n + 1));
    return PCD_OK;
}

// Captures one pass of step kind `kind`.  Nothing runs: the host
// bookkeeping is put back as it was after the capture.  Any failure leaves
// no graph behind.
static int capture_pass(pcd_ctx *ctx, Loop *L, const pcd_job *job, int cap, int kind, int rounds, bool fused) {
    hipGraphExec_t &exec = L->exec[kind];
    if (exec) {
        (void)hipGraphExecDestroy(exec);
        exec = nullptr;
    }
    // host bookkeeping as it stands (a pass changes it while capturing)
    const bool s_timing = ctx->timing, s_counters = ctx->counters, s_comp = ctx->labels_compressed,
               s_has = ctx->has_stats, s_pend = ctx->stats_pending, s_new = ctx->labels_have_new,
               s_kdef = ctx->k_deferred;
    const int s_bound = ctx->label_bound, s_k = ctx->k;
    const void *p0[4] = {ctx->d_labels, ctx->d_labels_alt, ctx->d_stats, ctx->d_stats_alt};
    ctx->timing = false;
    ctx->counters = false;
    ctx->label_bound = ctx->n;
    const pcd_rule rule = job->rule;
    LoopParams lp{job->max_iter, cap, job->threshold};
    PCD_HIP(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    ctx->capturing = true;
    ctx->graph_step = &L->d_state->step;
    int rc = PCD_OK;
    if (fused) {
        ctx->fused = L->d_state;
        rc = fused_compress_dev(ctx, rule, lp, L->d_state);
        if (rc == PCD_OK) rc = propagation_launch(ctx, rule, job->frac, job->seed, 0, job->tie);
        if (rc == PCD_OK) rc = propagation_commit(ctx);
        ctx->fused = nullptr;
    } else {
        rc = compress_labels_dev(ctx, true);
        // Under WCC the metric's internal-triangle pass takes about as long
        // as the propagation and neither reads the other: it runs beside it
        // on the metric stream, and a pass that turns out to be the last
        // drops its step (Chung-Lu, 1 M vertices: 0.27 of a pass's 0.72 ms).
        // A pass with two branches costs more to capture and replay, so graphs
        // below wcc_beside_min_edges keep the metric in line (8 passes and the
        // clustering before them, which makes them captured anew, on Chung-Lu
        // graphs, beside / in line: 0.17 M edges 2.75 / 2.32 ms, 0.32 M 2.71 /
        // 2.49, 0.47 M 2.91 / 2.69, 0.64 M 3.39 / 3.73, 1.7 M 4.08 / 4.46, 7.4 M
        // 7.41 / 8.42; replayed only: 0.47 M 1.78 / 1.75, 0.64 M 1.94 / 2.27).
        const bool beside = kind == PASS_PROPAGATE && rule.kind == PCD_RULE_WCC &&
                            ctx->m >= ctx->tune.wcc_beside_min_edges && ctx->mstream && ctx->ev_mfork && ctx->ev_metric;
        hipStream_t main_stream = ctx->stream;
        if (rc == PCD_OK && beside) {
            if (hipEventRecord(ctx->ev_mfork, ctx->stream) != hipSuccess ||
                hipStreamWaitEvent(ctx->mstream, ctx->ev_mfork, 0) != hipSuccess)
                rc = fail(PCD_E_HIP, "loop capture: metric stream");
            else
                ctx->stream = ctx->mstream;
        }
        if (rc == PCD_OK) rc = metric_enqueue(ctx, rule);
        if (ctx->stream != main_stream) {
            // joined on every path: a capture does not end with an open branch
            if (hipEventRecord(ctx->ev_metric, ctx->mstream) != hipSuccess) rc = fail(PCD_E_HIP, "loop capture: event");
            ctx->stream = main_stream;
            if (rc == PCD_OK) rc = propagation_launch(ctx, rule, job->frac, job->seed, 0, job->tie);
            if (hipStreamWaitEvent(ctx->stream, ctx->ev_metric, 0) != hipSuccess)
                rc = fail(PCD_E_HIP, "loop capture: join");
        }
        if (rc == PCD_OK) {
            hipLaunchKernelGGL(k_loop_rule, dim3(1), dim3(1), 0, ctx->stream, L->d_state, ctx->d_result, ctx->d_k, lp);
            hipLaunchKernelGGL(k_loop_snapshot, dim3(grid_for(ctx, ctx->n + 1, 256, 8)), dim3(256), 0, ctx->stream,
                               L->d_state, ctx->n, ctx->d_labels, ctx->d_stats, L->snap_labels, L->snap_stats);
            if (beside)
                hipLaunchKernelGGL(k_loop_drop, dim3(grid_for(ctx, ctx->n, 256, 8)), dim3(256), 0, ctx->stream,
                                   L->d_state, ctx->n, ctx->d_labels, ctx->d_labels_alt);
            else if (kind == PASS_PROPAGATE)
                rc = propagation_launch(ctx, rule, job->frac, job->seed, 0, job->tie);
            if (rc == PCD_OK && kind == PASS_PROPAGATE) rc = propagation_commit(ctx);
            if (kind == PASS_MERGE) rc = merging_dev(ctx, rule, rounds, job->seed, 0, job->tie);
        }
    }
    if (rc == PCD_OK && !fused) hipLaunchKernelGGL(k_loop_next, dim3(1), dim3(1), 0, ctx->stream, L->d_state);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(ctx->stream, &g);
    ctx->capturing = false;
    ctx->graph_step = nullptr;
    const bool same_ptrs = p0[0] == ctx->d_labels && p0[1] == ctx->d_labels_alt && p0[2] == ctx->d_stats &&
                           p0[3] == ctx->d_stats_alt;
    ctx->timing = s_timing;
    ctx->counters = s_counters;
    ctx->labels_compressed = s_comp;
    ctx->has_stats = s_has;
    ctx->stats_pending = s_pend;
    ctx->labels_have_new = s_new;
    ctx->k_deferred = s_kdef;
    ctx->label_bound = s_bound;
    ctx->k = s_k;
    (void)hipGetLastError();
    if (rc == PCD_OK && (e != hipSuccess || !g)) rc = fail(PCD_E_HIP, std::string("loop capture: ") + hipGetErrorString(e));
    if (rc == PCD_OK && !same_ptrs) rc = fail(PCD_E_STATE, "loop capture: the pass does not return its buffers");
    if (rc == PCD_OK && hipGraphInstantiate(&exec, g, nullptr, nullptr, 0) != hipSuccess) {
        (void)hipGetLastError();
        exec = nullptr;
        rc = fail(PCD_E_HIP, "loop graph instantiation");
    }
    if (g) (void)hipGraphDestroy(g);
    if (rc != PCD_OK) return rc;
    L->key[kind] = pass_key(ctx, job, cap, kind, rounds, fused);
    return PCD_OK;
}

// Passes [it, it + count) on the device; see pcd_iterate_many.
static int device_passes(pcd_ctx *ctx, Loop *L, int strategy, bool fused, int it, int count, double prev_score,
                         int *passes, double *score, int *num_labels, int *done) {
    LoopState &h = *L->h_state;
    std::memset(&h, 0, sizeof(h));
    h.it = it;
    h.step = it;
    h.it_end = it + count;
    h.prev = prev_score;
    h.prev_k = ctx->k;
    PCD_HIP(hipMemcpyAsync(L->d_state, &h, sizeof(LoopState), hipMemcpyHostToDevice, ctx->stream));
    if (fused) PCD_TRY(fused_prepare(ctx));
    // replays per read of the record: about half a millisecond of passes
    // (one pass at a time for large graphs), never beyond the first pass
    // that can freeze
    int per = 1;
    double pass_ms = -1.0;
    for (;;) {
        const int left = h.it_end - h.it + 1;  // the pass at it_end freezes
        const int c = std::max(1, std::min(per, left));
        const auto t0 = std::chrono::steady_clock::now();
        // replay r of this batch is pass h.it + r (once frozen, a replay
        // of either kind changes nothing)
        for (int r = 0; r < c; r++) PCD_HIP(hipGraphLaunch(L->exec[pass_kind(strategy, h.it + r)], ctx->stream));
        PCD_HIP(hipMemcpyAsync(&h, L->d_state, sizeof(LoopState), hipMemcpyDeviceToHost, ctx->stream));
        PCD_HIP(hipStreamSynchronize(ctx->stream));
        if (h.frozen) break;
        const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count() / c;
        pass_ms = pass_ms < 0 ? ms : std::min(pass_ms, ms);
        per = std::max(1, std::min(32, (int)(0.5 / std::max(pass_ms, 1e-3))));
    }
    // the labels and statistics of the frozen pass back in place
    if (!fused) {
        PCD_HIP(hipMemcpyAsync(ctx->d_labels, L->snap_labels, sizeof(int32_t) * (size_t)ctx->n,
                               hipMemcpyDeviceToDevice, ctx->stream));
        if (h.k_freeze > 0)
            PCD_HIP(hipMemcpyAsync(ctx->d_stats, L->snap_stats, sizeof(CommStats) * (size_t)h.k_freeze,
                                   hipMemcpyDeviceToDevice, ctx->stream));
    }
    PCD_HIP(hipStreamSynchronize(ctx->stream));
    ctx->k = h.k_freeze;
    ctx->label_bound = h.k_freeze;
    ctx->k_deferred = false;
    ctx->labels_compressed = true;
    ctx->has_stats = true;
    ctx->stats_pending = false;
    ctx->labels_have_new = false;
    if (h.done) {
        *passes = h.it - it + 1;
        *score = h.score_done;
        *num_labels = h.k_freeze;
        *done = 1;
    } else {
        *passes = h.it - it;
        *score = h.prev;
        *num_labels = h.prev_k;
        *done = 0;
    }
    return PCD_OK;
}

}  // namespace pcd

using namespace pcd;

// passes of [it, it + count) that -n and the iteration cap leave, at least one
static int last_passes(const pcd_job *job, int cap, int it, int count) {
    int64_t end = std::min<int64_t>((int64_t)it + count, (int64_t)cap + 1);
    if (job->max_iter != -1) end = std::min<int64_t>(end, (int64_t)job->max_iter + 1);
    return (int)std::max<int64_t>(1, end - it);
}

extern "C" int pcd_iterate_many(pcd_ctx *ctx, const pcd_job *job, int strategy, int rounds, int it, int count,
                                double prev_score, int *passes, double *score, int *num_labels, int *done) {
    if (!ctx || !job || !passes || !score || !num_labels || !done) return fail(PCD_E_INVALID, "null argument");
    if (count <= 0) return fail(PCD_E_INVALID, "count must be positive");
    if (strategy < 0 || strategy > 2) return fail(PCD_E_INVALID, "strategy must be 0, 1 or 2");
    if (job->rule.kind < PCD_RULE_MODULARITY || job->rule.kind > PCD_RULE_CONDUCTANCE)
        return fail(PCD_E_INVALID, "unknown rule kind " + std::to_string(job->rule.kind));
    if (strategy != 1 && !(job->frac > 0.0)) return fail(PCD_E_INVALID, "frac must be > 0");
    if (strategy != 0 && rounds <= 0) return fail(PCD_E_INVALID, "rounds must be positive");
    if (job->tie != PCD_TIE_RANDOM && job->tie != PCD_TIE_LOWEST) return fail(PCD_E_INVALID, "unknown tie order");
    if (!ctx->has_graph) return fail(PCD_E_STATE, "no graph uploaded");
    if (!ctx->has_labels) return fail(PCD_E_STATE, "no labels uploaded");
    if (it < 0 || (int64_t)it + count > INT32_MAX / 2) return fail(PCD_E_INVALID, "pass range out of range");
    *passes = 0;
    *done = 0;
    *score = prev_score;
    *num_labels = 0;
    const int cap = job->iter_cap > 0 ? job->iter_cap : 1000;
    double prev = prev_score;
    int run = 0;
    if (ctx->tune.graph_loop && ctx->tune.solo_loop && ctx->tune.inc_stats &&
        2 * (int64_t)ctx->m >= ctx->tune.graph_loop_min_entries && !ctx->counters && !ctx->timing &&
        solo_fits(ctx, job, strategy, last_passes(job, cap, it, count))) {
        // a small graph: the passes in one launch, up to SOLO_MAX_PASSES at a time
        PCD_HIP(hipSetDevice(ctx->device));
        while (run < count && !*done) {
            SoloResult r;
            PCD_TRY(solo_passes(ctx, job, cap, it + run, std::min(count - run, SOLO_MAX_PASSES), prev, &r));
            run = r.it - it + (r.done ? 1 : 0);
            prev = r.score;
            *passes = run;
            *score = r.score;
            *num_labels = r.last_k;
            *done = r.done;
        }
        return PCD_OK;
    }
    // pass by pass until the statistics follow the labels (the first pass
    // of labels from outside counts them in full), or for the rules and
    // strategies the captured pass does not cover
    // captured step kinds the schedule replays (bit per PassKind); merging
    // is captured in its community-row form
    const unsigned kinds = strategy == 0 ? 1u : strategy == 1 ? 2u : 3u;
    for (;;) {
        const bool device_ok = (strategy == 0 || !ctx->tune.merge_sort) &&
                               (job->rule.kind != PCD_RULE_WCC || ctx->has_triangles) &&
                               ctx->tune.graph_loop && ctx->tune.inc_stats && ctx->ev_metric && ctx->has_labels &&
                               (ctx->stats_pending || ctx->has_stats) &&
                               2 * (int64_t)ctx->m >= ctx->tune.graph_loop_min_entries &&
                               !(loop_of(ctx) && loop_of(ctx)->broken) && count - run >= 2;
        if (run >= count || device_ok) break;
        int d = 0, k = 0;
        double s = 0.0;
        PCD_TRY(pcd_iterate(ctx, job, strategy, rounds, it + run, prev, &s, &k, &d));
        run++;
        prev = s;
        *passes = run;
        *score = s;
        *num_labels = k;
        if (d) {
            *done = 1;
            return PCD_OK;
        }
    }
    if (run >= count) return PCD_OK;
    PCD_HIP(hipSetDevice(ctx->device));
    if (!ctx->loop) ctx->loop = new Loop();
    Loop *L = loop_of(ctx);
    const bool fused = strategy == 0 && ctx->tune.fused_pass &&
                       (job->rule.kind == PCD_RULE_MODULARITY || job->rule.kind == PCD_RULE_CPM);
    int rc = reserve_passes(ctx, L, kinds, fused);
    for (int kd = 0; kd < 2 && rc == PCD_OK; kd++) {
        if (!((kinds >> kd) & 1u)) continue;
        if (!L->exec[kd] || !(L->key[kd] == pass_key(ctx, job, cap, kd, rounds, fused)))
            rc = capture_pass(ctx, L, job, cap, kd, rounds, fused);
    }
    if (rc != PCD_OK) {
        // this context runs pass by pass from now on
        L->broken = true;
        int p2 = 0, d2 = 0, k2 = 0;
        double s2 = 0.0;
        PCD_TRY(pcd_iterate_many(ctx, job, strategy, rounds, it + run, count - run, prev, &p2, &s2, &k2, &d2));
        *passes = run + p2;
        *score = p2 ? s2 : *score;
        *num_labels = p2 ? k2 : *num_labels;
        *done = d2;
        return PCD_OK;
    }
    int p2 = 0, d2 = 0, k2 = 0;
    double s2 = 0.0;
    PCD_TRY(device_passes(ctx, L, strategy, fused, it + run, count - run, prev, &p2, &s2, &k2, &d2));
    if (kinds & 2u) PCD_TRY(merge_rows_check(ctx));
    *passes = run + p2;
    if (p2) {
        *score = s2;
        *num_labels = k2;
    }
    *done = d2;
    return PCD_OK;
}
