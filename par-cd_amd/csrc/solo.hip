// The refinement loop of main.cpp:226-266 on a small graph, in one launch of
// one workgroup.
//
// A pass over a few thousand entries is a few microseconds of work; as some
// twenty kernels it costs 75 us, each of them at the floor of a launch.  Here
// one workgroup runs every pass (compression, statistics, metric, stop rule,
// propagation, statistics update) between barriers, with the labels, the
// community records and the totals in LDS, and the host reads one record at
// the end.  What bounds it is the chain of dependent reads and barriers of a
// pass and, with growing rows, the instruction rate of one CU, so it serves
// graphs of at most SOLO_MAX_N vertices and SOLO_MAX_E entries, and of those the jobs
// that solo_pays picks; the others run their passes over the whole chip
// (loop.hip).  Every label, statistic and score is
// the one those passes give: the sums are integers, and ties have a total
// order.
#include <algorithm>

#include "lp.h"

namespace pcd {

constexpr int SOLO_NT = 1024, SOLO_W = SOLO_NT / WAVE;
constexpr int SOLO_N = SOLO_MAX_N, SOLO_PER = SOLO_N / SOLO_NT;
constexpr int SOLO_TW = 512, SOLO_TWAVES = 8;  // degrees 65-256: wave tables, held by eight waves

struct SoloArgs {
    LPArgs lp;  // indices, adj, order, rule, seed, tie, f
    int n, m, kind;
    int start[NUM_BINS + 1];
    int32_t *labels;
    CommStats *stats;
    int has_stats;    // `stats` holds the records of `labels` (NEW_LABEL vertices left out)
    int it, it_end, max_iter, cap;
    double threshold, prev;
    SoloResult *out;
    int32_t *dk;
};

struct SoloTables {
    int keys[SOLO_TWAVES][SOLO_TW], cnts[SOLO_TWAVES][SOLO_TW];
    uint16_t occ[SOLO_TWAVES][SOLO_TW / 2];
    int nocc[SOLO_TWAVES];
};
union SoloScratch {
    struct {
        int first[SOLO_N], newid[SOLO_N];
    } c;
    SoloTables w;
    BlockTable<SOLO_NT, 2 * SOLO_N, false, uint16_t> b;
};

struct SoloLds {
    int cur[SOLO_N], nxt[SOLO_N];       // labels before and after a step
    int size[SOLO_N], iv[SOLO_N], ev[SOLO_N], tot[SOLO_N];
    int list[SOLO_W][WAVE];
    int part[SOLO_W];
    long long sums[3][SOLO_W];
    int k, stop;
    double score;
};

// exclusive prefix of x over the workgroup; *total receives the sum
__device__ inline int solo_scan(int x, int *part, int *total) {
    const int lane = __lane_id(), w = threadIdx.x / WAVE;
    const int inc = wave_incl_scan(x);
    if (lane == WAVE - 1) part[w] = inc;
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < SOLO_W; i++) {
        const int t = part[i];
        if (i < w) base += t;
        tot += t;
    }
    *total = tot;
    return base + inc - x;
}

// positions [p0, p1) of one small bin over the workgroup's waves, starting at
// wave `at`; units of two groups' rows, for about half the vertices are active
template <int G, unsigned KM>
__device__ inline int solo_small(const LPArgs &a, int p0, int p1, int at, SoloLds &s) {
    if (p1 <= p0) return at;
    constexpr int CP = std::min(WAVE, 2 * WAVE / G);
    const RangeSrc src{p0, p1, CP, a};
    const int w = threadIdx.x / WAVE;
    lp_small<G, CP, false, KM>(src, __builtin_amdgcn_readfirstlane((w - at) & (SOLO_W - 1)), SOLO_W, s.list[w]);
    return (at + src.units()) & (SOLO_W - 1);
}

template <unsigned KM>
__global__ __launch_bounds__(SOLO_NT) void k_solo_loop(SoloArgs a) {
    __shared__ SoloLds s;
    __shared__ SoloScratch x;
    const int tid = threadIdx.x, w = tid / WAVE, lane = __lane_id(), n = a.n;
    for (int v = tid; v < n; v += SOLO_NT) {
        s.cur[v] = a.labels[v];
        if (a.has_stats) {
            const CommStats c = a.stats[v];  // ids below n
            s.size[v] = c.size;
            s.iv[v] = c.int_vol;
            s.ev[v] = c.ext_vol;
        }
    }
    int it = a.it, prev_k = 0;
    double prev = a.prev;
    bool counted = a.has_stats != 0;
    LPArgs lp = a.lp;
    lp.labels = s.cur;
    lp.new_labels = s.nxt;
    lp.tot = s.tot;
    lp.counters = nullptr;
    lp.step_ptr = nullptr;
    for (;;) {
        // compress_labels (framework.cpp:146-170): first occurrences, new ids
        // in their order, records moved with them
        __syncthreads();
        for (int c = tid; c < n; c += SOLO_NT) x.c.first[c] = INT32_MAX;
        __syncthreads();
        for (int v = tid; v < n; v += SOLO_NT)
            if (s.cur[v] >= 0) atomicMin(&x.c.first[s.cur[v]], v);
        __syncthreads();
        const int per = (n + SOLO_NT - 1) / SOLO_NT, v0 = min(n, tid * per), v1 = min(n, v0 + per);
        int flags = 0;
        for (int v = v0; v < v1; v++) flags += s.cur[v] < 0 || x.c.first[s.cur[v]] == v;
        int k;
        int id = solo_scan(flags, s.part, &k);
        int rs[SOLO_PER], ri[SOLO_PER], re[SOLO_PER], at[SOLO_PER];
#pragma unroll
        for (int j = 0; j < SOLO_PER; j++) {
            const int v = v0 + j;
            at[j] = -1;
            if (v >= v1) continue;
            const int l = s.cur[v];
            if (l >= 0 && x.c.first[l] != v) continue;
            at[j] = id++;
            if (l >= 0) x.c.newid[l] = at[j];
            if (!counted) continue;
            rs[j] = l < 0 ? 1 : s.size[l];
            ri[j] = l < 0 ? 0 : s.iv[l];
            re[j] = l < 0 ? lp.indices[v + 1] - lp.indices[v] : s.ev[l];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < SOLO_PER; j++) {
            const int v = v0 + j;
            if (v >= v1) continue;
            const int l = s.cur[v];
            s.cur[v] = l < 0 ? at[j] : x.c.newid[l];
            if (at[j] >= 0 && counted) {
                s.size[at[j]] = rs[j];
                s.iv[at[j]] = ri[j];
                s.ev[at[j]] = re[j];
            }
        }
        if (!counted) {
            // collect_statistics (framework.cpp:103-143), eight lanes a row
            for (int c = tid; c < n; c += SOLO_NT) s.size[c] = s.iv[c] = s.ev[c] = 0;
            __syncthreads();
            for (int v = tid / 8; v < n; v += SOLO_NT / 8) {
                const int b = lp.indices[v], e = lp.indices[v + 1], l = s.cur[v];
                int same = 0;
                for (int j = b + (tid & 7); j < e; j += 8) same += s.cur[lp.adj[j]] == l;
#pragma unroll
                for (int d = 4; d > 0; d >>= 1) same += __shfl_xor(same, d, WAVE);
                if ((tid & 7) == 0) {
                    atomicAdd(&s.size[l], 1);
                    atomicAdd(&s.iv[l], same);
                    atomicAdd(&s.ev[l], e - b - same);
                }
            }
            counted = true;
        }
        __syncthreads();
        // Rule::calculate (rules.cpp:9-22, 121-129) and the totals the gains read
        long long ti = 0, tv = 0, ts = 0;
        for (int c = tid; c < k; c += SOLO_NT) {
            const long long vol = (long long)s.iv[c] + s.ev[c];
            ti += s.iv[c];
            tv += vol * vol;
            ts += (long long)s.size[c] * (s.size[c] - 1);
            s.tot[c] = KM == RK_MOD ? s.iv[c] + s.ev[c] : s.size[c];
        }
        ti = wave_sum64(ti);
        tv = wave_sum64(tv);
        ts = wave_sum64(ts);
        if (lane == 0) {
            s.sums[0][w] = ti;
            s.sums[1][w] = tv;
            s.sums[2][w] = ts;
        }
        // the labels after the step start as those before it
        for (int v = tid; v < n; v += SOLO_NT) s.nxt[v] = s.cur[v];
        __syncthreads();
        if (tid == 0) {
            long long A = 0, B = 0, C = 0;
            for (int i = 0; i < SOLO_W; i++) {
                A += s.sums[0][i];
                B += s.sums[1][i];
                C += s.sums[2][i];
            }
            const double sc = score_of_sums(A, B, C, a.kind, a.lp.rule.lambda, a.m);
            // main.cpp:241-242, -n, the iteration cap; the pass at it_end only compresses
            const bool over = it >= a.it_end;
            const bool known = (a.max_iter != -1 && it >= a.max_iter) || it >= a.cap;
            const bool done =
                !over && (known || (a.max_iter == -1 && prev > 0 && sc > 0 && sc / prev - 1 <= a.threshold));
            s.score = sc;
            s.stop = done || over;
            if (s.stop) {
                *a.out = SoloResult{it, done ? 1 : 0, k, done ? k : prev_k, done ? sc : prev};
                *a.dk = k;
            }
        }
        __syncthreads();
        if (s.stop) {
            s.k = k;
            break;
        }
        // one propagation step (refinement.cpp:114-182)
        lp.step = it;
        if (a.start[BIN_HUB] < a.start[BIN_W256]) {  // degrees above 256: the workgroup takes a row at a time
            const RangeSrc src{a.start[BIN_HUB], a.start[BIN_W256], 1, lp};
            lp_block<SOLO_NT, 2 * SOLO_N, KM, RangeSrc, false, 4, uint16_t>(src, 0, 1, x.b);
            __syncthreads();
        }
        if (w < SOLO_TWAVES && a.start[BIN_W256] < a.start[BIN_G64]) {
            const RangeSrc src{a.start[BIN_W256], a.start[BIN_G64], 1, lp};
            lp_wave<SOLO_TW, KM, RangeSrc, false, 4>(src, __builtin_amdgcn_readfirstlane(w), SOLO_TWAVES, x.w.keys[w],
                                                     x.w.cnts[w], nullptr, x.w.occ[w], &x.w.nocc[w]);
        }
        int from = SOLO_TWAVES;  // the waves without a table start on the small rows
        from = solo_small<64, KM>(lp, a.start[BIN_G64], a.start[BIN_G32], from, s);
        from = solo_small<32, KM>(lp, a.start[BIN_G32], a.start[BIN_G16], from, s);
        from = solo_small<16, KM>(lp, a.start[BIN_G16], a.start[BIN_G8], from, s);
        from = solo_small<8, KM>(lp, a.start[BIN_G8], a.start[BIN_G4], from, s);
        solo_small<4, KM>(lp, a.start[BIN_G4], a.start[NUM_BINS], from, s);
        __syncthreads();
        // the statistics follow the moved vertices' rows (see k_delta_all): a
        // pair whose other end kept its label counts twice
        for (int v = tid / 8; v < n; v += SOLO_NT / 8) {
            const int lo = s.cur[v], ln = s.nxt[v];
            if (lo == ln) continue;
            const int b = lp.indices[v], deg = lp.indices[v + 1] - b;
            int ca = 0, cb = 0;
            for (int j = tid & 7; j < deg; j += 8) {
                const int u = lp.adj[b + j];
                const int lu = s.cur[u], nu = s.nxt[u], f = lu != nu ? 1 : 2;
                ca += lu == lo ? f : 0;
                cb += nu == ln ? f : 0;
            }
#pragma unroll
            for (int d = 4; d > 0; d >>= 1) {
                ca += __shfl_xor(ca, d, WAVE);
                cb += __shfl_xor(cb, d, WAVE);
            }
            if ((tid & 7) == 0) {
                atomicAdd(&s.size[lo], -1);
                atomicAdd(&s.iv[lo], -ca);
                atomicAdd(&s.ev[lo], ca - deg);
                if (ln >= 0) {
                    atomicAdd(&s.size[ln], 1);
                    atomicAdd(&s.iv[ln], cb);
                    atomicAdd(&s.ev[ln], deg - cb);
                }
            }
        }
        __syncthreads();
        for (int v = tid; v < n; v += SOLO_NT) s.cur[v] = s.nxt[v];
        prev = s.score;
        prev_k = k;
        it++;
    }
    for (int v = tid; v < n; v += SOLO_NT) a.labels[v] = s.cur[v];
    const int k = s.k;
    for (int c = tid; c < k; c += SOLO_NT) a.stats[c] = CommStats{s.size[c], s.iv[c], s.ev[c], 0};
}

// Whether the passes of a job (at most `passes` of them) are faster on one
// workgroup than replayed over the whole chip.  A pass here takes about 11 us
// and, per 1,000, 1.2 us for entries, 1.6 us for entries of active rows and
// 3.2 us for active vertices, and 3.2 us for each active row above 256 entries,
// which the whole workgroup takes by itself (least squares over 250 to 4,000
// vertices, 4,000 to 32,000 entries, 0 to 24 such rows, half of the vertices
// and all of them active; the largest error up to 16,000 entries is 7 us).  A replayed
// pass takes 45-48 us at all these sizes, after some 120 us for a first pass of
// single launches and the capture.  Runs of 20 passes, one workgroup / replayed:
// 1,000 vertices of 8,000 entries 0.53 / 0.95 ms, of 16,000 0.96 / 0.97, of
// 24,000 1.30 / 0.94; 60 rows of 265 entries 3.6 / 0.98.
static bool solo_pays(const pcd_ctx *ctx, const pcd_job *job, int passes) {
    const double f = std::min(job->frac, 1.0), e = 2e-3 * ctx->m, n = 1e-3 * ctx->n;
    const int long_rows = ctx->bins.start[BIN_W256] - ctx->bins.start[BIN_HUB];
    const double pass = 11.0 + e * (1.2 + 1.6 * f) + 3.2 * f * (n + long_rows);
    return pass <= 46.0 + 120.0 / passes;
}

bool solo_fits(const pcd_ctx *ctx, const pcd_job *job, int strategy, int passes) {
    return strategy == 0 && (job->rule.kind == PCD_RULE_MODULARITY || job->rule.kind == PCD_RULE_CPM) &&
           ctx->n <= SOLO_N && 2 * (int64_t)ctx->m <= SOLO_MAX_E && ctx->label_bound <= ctx->n &&
           (ctx->tune.solo_loop == 2 || solo_pays(ctx, job, passes));
}

int solo_passes(pcd_ctx *ctx, const pcd_job *job, int cap, int it, int count, double prev, SoloResult *res) {
    if (!ctx->d_solo) PCD_TRY(dev_alloc_t(ctx, &ctx->d_solo, 1));
    SoloArgs a{};
    a.lp.indices = ctx->d_indices;
    a.lp.adj = ctx->d_adj;
    a.lp.order = ctx->d_order;
    a.lp.rule = make_rule(ctx, job->rule);
    a.lp.seed = job->seed;
    a.lp.tie = job->tie;
    a.lp.f = (int)((job->frac < 1.0 ? job->frac : 1.0) * 2147483647.0);  // refinement.cpp:116
    a.n = ctx->n;
    a.m = ctx->m;
    a.kind = job->rule.kind;
    for (int b = 0; b <= NUM_BINS; b++) a.start[b] = ctx->bins.start[b];
    a.labels = ctx->d_labels;
    a.stats = ctx->d_stats;
    a.has_stats = ctx->stats_pending || ctx->has_stats;
    a.it = it;
    a.it_end = it + count;
    a.max_iter = job->max_iter;
    a.cap = cap;
    a.threshold = job->threshold;
    a.prev = prev;
    a.out = ctx->d_solo;
    a.dk = ctx->d_k;
    if (a.kind == PCD_RULE_MODULARITY)
        hipLaunchKernelGGL(k_solo_loop<RK_MOD>, dim3(1), dim3(SOLO_NT), 0, ctx->stream, a);
    else
        hipLaunchKernelGGL(k_solo_loop<RK_CPM>, dim3(1), dim3(SOLO_NT), 0, ctx->stream, a);
    PCD_HIP(hipGetLastError());
    SoloResult *h = (SoloResult *)(ctx->h_small + 16);
    PCD_HIP(hipMemcpyAsync(h, ctx->d_solo, sizeof(SoloResult), hipMemcpyDeviceToHost, ctx->stream));
    PCD_HIP(hipStreamSynchronize(ctx->stream));
    *res = *h;
    ctx->k = h->k;
    ctx->label_bound = h->k;
    ctx->k_deferred = false;
    ctx->labels_compressed = true;
    ctx->has_stats = true;
    ctx->stats_pending = false;
    ctx->labels_have_new = false;
    return PCD_OK;
}

}  // namespace pcd
