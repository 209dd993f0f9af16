// Partition phases on the device: label compression, community statistics
// and the metric evaluation of modularity / CPM / conductance.
#include "prims.h"

namespace pcd {

// ------------------------------------------------------------ compression
// framework.cpp:146-170 numbers labels in order of first occurrence over v.
// Here: first[l] = min v with label l (atomicMin), a vertex is a "first" if
// it is the minimum of its label or has NEW_LABEL, and the exclusive scan of
// those flags over v is exactly the reference's running counter.

// A plain read of first[l] skips the atomic when it already holds a smaller
// vertex: the value only decreases, so a stale read costs at most an
// atomic, and large communities do not serialise every member's update.
// The table's start: the vertex the last compression found first for label
// c, if it still has label c (an upper bound of the new first occurrence, so
// most members' reads skip their atomic, large communities included), else
// INT32_MAX.  firstv holds vertex ids or -1.
__global__ void k_first_init(int bound, const int32_t *labels, const int32_t *firstv, int32_t *first) {
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < bound; c += gridDim.x * blockDim.x) {
        const int w = firstv[c];
        first[c] = (w >= 0 && labels[w] == c) ? w : INT32_MAX;
    }
}

// The least vertex of every label.  A workgroup keeps the labels it meets
// first in LDS (as StatsAcc does) and sends each one's least vertex to
// memory at its end, so the members of a large community neither read its
// word of `first` nor queue on it; other labels go to memory (R-MAT-20 under
// a partition of hub neighbourhoods: 0.29 -> 0.05 ms; R-MAT-22 from many
// small communities unchanged).  What bounds it is then the labels' read and
// one random read per vertex of a small community.  A small table and four
// vertices a thread: the flush of a full table costs as much as the reads it
// saved.
constexpr int FO_LOG = 7, FO_NT = 512;
__global__ __launch_bounds__(FO_NT) void k_first_occurrence(int n, const int32_t *labels, int32_t *first) {
    __shared__ int key[1 << FO_LOG], low[1 << FO_LOG];
    for (int i = threadIdx.x; i < (1 << FO_LOG); i += FO_NT) {
        key[i] = EMPTY_KEY;
        low[i] = INT32_MAX;
    }
    __syncthreads();
    for (int v = blockIdx.x * FO_NT + threadIdx.x; v < n; v += gridDim.x * FO_NT) {
        const int l = labels[v];
        if (l < 0) continue;
        const int h = (int)(((uint32_t)l * 0x9E3779B1u) >> (32 - FO_LOG));
        int k = __hip_atomic_load(&key[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (k == EMPTY_KEY) {
            k = atomicCAS(&key[h], EMPTY_KEY, l);
            if (k == EMPTY_KEY) k = l;
        }
        if (k == l) atomicMin(&low[h], v);
        else if (first[l] > v) atomicMin(&first[l], v);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < (1 << FO_LOG); i += FO_NT) {
        const int l = key[i];
        if (l != EMPTY_KEY && first[l] > low[i]) atomicMin(&first[l], low[i]);
    }
}

struct FirstFlag {
    const int32_t *labels, *first;
    __device__ int operator()(int64_t v) const {
        int l = labels[v];
        return (l < 0 || first[l] == (int)v) ? 1 : 0;
    }
};
// Each first occurrence gets its new id.  With st_in set, the statistics
// move to the new ids as well: st_out[new id] = st_in[old label], and a
// NEW_LABEL vertex opens its singleton record {1, 0, deg}.
struct FirstStore {
    const int32_t *labels;
    int32_t *out, *newid;
    const CommStats *st_in;
    CommStats *st_out;
    const int32_t *indices;
    int32_t *firstv;  // firstv[new id] = its first vertex
    __device__ void operator()(int64_t v, int ex, int flag) const {
        if (!flag) return;
        int l = labels[v];
        firstv[ex] = (int)v;
        if (l < 0) out[v] = ex;
        else newid[l] = ex;
        if (st_in) st_out[ex] = l < 0 ? CommStats{1, 0, indices[v + 1] - indices[v], 0} : st_in[l];
    }
};

__global__ void k_relabel(int n, const int32_t *labels, const int32_t *newid, int32_t *out) {
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
        int l = labels[v];
        if (l >= 0) out[v] = newid[l];
    }
}

__global__ void k_copy_i32(int32_t *dst, const int32_t *src) { *dst = *src; }

// the first *kp community records of src into dst
__global__ void k_copy_stats(const int32_t *kp, const CommStats *src, CommStats *dst) {
    const int k = *kp;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < k; c += gridDim.x * blockDim.x) dst[c] = src[c];
}

// slot of the pinned scratch ints that receives a deferred k
constexpr int K_SLOT = 8;

void resolve_k(pcd_ctx *ctx) {
    if (!ctx->k_deferred) return;
    ctx->k = ctx->h_small[K_SLOT];
    ctx->label_bound = ctx->k;
    ctx->k_deferred = false;
}

int compress_labels_dev(pcd_ctx *ctx, bool defer_k) {
    const int n = ctx->n;
    kt_begin(ctx, KS_COMPRESS);
    if (ctx->label_bound > 0 && ctx->label_bound <= n + 1)
        hipLaunchKernelGGL(k_first_init, dim3(grid_for(ctx, ctx->label_bound, 256)), dim3(256), 0, ctx->stream,
                           ctx->label_bound, ctx->d_labels, ctx->d_firstv, ctx->d_first);
    else if (ctx->label_bound > 0)
        PCD_TRY(fill_i32(ctx, ctx->d_first, INT32_MAX, ctx->label_bound));
    hipLaunchKernelGGL(k_first_occurrence, dim3(grid_for(ctx, n, FO_NT * 4, 4)), dim3(FO_NT), 0, ctx->stream, n,
                       ctx->d_labels, ctx->d_first);
    // statistics of these labels (full count, or updated by the last
    // propagation step) are renumbered with them
    const bool renumber = ctx->stats_pending || ctx->has_stats;
    int32_t *total = nullptr;
    PCD_TRY(device_scan(ctx, n, FirstFlag{ctx->d_labels, ctx->d_first},
                        FirstStore{ctx->d_labels, ctx->d_labels_alt, ctx->d_newid, renumber ? ctx->d_stats : nullptr,
                                   ctx->d_stats_alt, ctx->d_indices, ctx->d_firstv},
                        &total));
    hipLaunchKernelGGL(k_relabel, dim3(grid_for(ctx, n, 256)), dim3(256), 0, ctx->stream, n, ctx->d_labels,
                       ctx->d_newid, ctx->d_labels_alt);
    hipLaunchKernelGGL(k_copy_i32, dim3(1), dim3(1), 0, ctx->stream, ctx->d_k, total);
    kt_end(ctx, KS_COMPRESS);
    PCD_HIP(hipGetLastError());
    if (ctx->capturing) {
        // a captured pass: k stays on the device, and the renumbered
        // statistics move back in place so that the replayed pass always
        // reads and writes the same buffers
        ctx->k_deferred = true;
        if (renumber)
            hipLaunchKernelGGL(k_copy_stats, dim3(grid_for(ctx, n + 1, 256, 8)), dim3(256), 0, ctx->stream,
                               ctx->d_k, ctx->d_stats_alt, ctx->d_stats);
    } else if (defer_k) {
        PCD_HIP(hipMemcpyAsync(ctx->h_small + K_SLOT, ctx->d_k, sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
        ctx->k_deferred = true;
    } else {
        PCD_HIP(hipMemcpyAsync(ctx->h_small, ctx->d_k, sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
        PCD_HIP(hipStreamSynchronize(ctx->stream));
        ctx->k = ctx->h_small[0];
        ctx->label_bound = ctx->k;
        ctx->k_deferred = false;
    }
    std::swap(ctx->d_labels, ctx->d_labels_alt);
    if (renumber && !ctx->capturing) std::swap(ctx->d_stats, ctx->d_stats_alt);
    ctx->labels_compressed = true;
    ctx->has_stats = renumber;
    ctx->stats_pending = false;
    return PCD_OK;
}

// ------------------------------------------------------------ the fused pass
// What follows the numbering, elementwise: the new labels (into both label
// buffers: the step's result starts as a copy), the records back in place,
// the total each gain reads, and the metric's sums; the workgroup that adds
// its sums last scores the partition and applies the stop rule.
struct PassTail {
    int n, m, kind;
    double lambda;
    const int32_t *total;  // k
    const int32_t *newid;
    int32_t *labels;       // before the compression; the copy
    int32_t *out;          // compressed
    const CommStats *st_in;
    CommStats *st;
    int32_t *tot, *dk;
    unsigned long long *acc;  // zero between passes
    LoopState *state;
    LoopParams rule;
};
constexpr int TAIL_NT = 512;
__global__ __launch_bounds__(TAIL_NT) void k_pass_tail(PassTail a) {
    __shared__ long long lds[3][TAIL_NT / WAVE];
    const int k = *a.total;
    const int stride = gridDim.x * TAIL_NT, t0 = blockIdx.x * TAIL_NT + threadIdx.x;
    long long s0 = 0, s1 = 0, s2 = 0;
    for (int c = t0; c < k; c += stride) {
        const CommStats r = a.st_in[c];
        const int v = r.int_vol + r.ext_vol;
        a.st[c] = r;
        a.tot[c] = a.kind == PCD_RULE_MODULARITY ? v : r.size;
        const long long vol = (long long)r.int_vol + r.ext_vol;
        s0 += r.int_vol;
        s1 += vol * vol;
        s2 += (long long)r.size * (r.size - 1);
    }
    for (int v = t0; v < a.n; v += stride) {
        const int l = a.labels[v];
        const int x = l < 0 ? a.out[v] : a.newid[l];
        a.out[v] = x;
        a.labels[v] = x;
    }
    s0 = wave_sum64(s0);
    s1 = wave_sum64(s1);
    s2 = wave_sum64(s2);
    const int w = threadIdx.x / WAVE;
    if (__lane_id() == 0) {
        lds[0][w] = s0;
        lds[1][w] = s1;
        lds[2][w] = s2;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int i = 1; i < TAIL_NT / WAVE; i++) {
        s0 += lds[0][i];
        s1 += lds[1][i];
        s2 += lds[2][i];
    }
    atomicAdd(&a.acc[0], (unsigned long long)s0);
    atomicAdd(&a.acc[1], (unsigned long long)s1);
    atomicAdd(&a.acc[2], (unsigned long long)s2);
    __threadfence();
    if (atomicAdd(&a.state->arrived, 1) != (int)gridDim.x - 1) return;
    __threadfence();
    // atomics read what the others added, and leave zeros for the next pass
    const long long x0 = (long long)atomicExch(&a.acc[0], 0ULL), x1 = (long long)atomicExch(&a.acc[1], 0ULL),
                    x2 = (long long)atomicExch(&a.acc[2], 0ULL);
    a.state->arrived = 0;
    *a.dk = k;
    loop_rule(a.state, score_of_sums(x0, x1, x2, a.kind, a.lambda, a.m), k, a.rule);
}

int fused_prepare(pcd_ctx *ctx) {
    if (ctx->label_bound > 0)
        hipLaunchKernelGGL(k_first_init, dim3(grid_for(ctx, ctx->label_bound, 256)), dim3(256), 0, ctx->stream,
                           ctx->label_bound, ctx->d_labels, ctx->d_firstv, ctx->d_first);
    PCD_TRY(fill_u64(ctx, (uint64_t *)ctx->d_acc, 0, 4));
    PCD_HIP(hipGetLastError());
    return PCD_OK;
}

int fused_compress_dev(pcd_ctx *ctx, pcd_rule rule, const LoopParams &p, LoopState *state) {
    const int n = ctx->n;
    hipLaunchKernelGGL(k_first_occurrence, dim3(grid_for(ctx, n, FO_NT * 4, 4)), dim3(FO_NT), 0, ctx->stream, n,
                       ctx->d_labels, ctx->d_first);
    const FirstFlag flag{ctx->d_labels, ctx->d_first};
    const FirstStore store{ctx->d_labels, ctx->d_labels_alt, ctx->d_newid, ctx->d_stats,
                           ctx->d_stats_alt, ctx->d_indices, ctx->d_firstv};
    int32_t *total = ctx->d_scan_part;
    if (n <= SCAN_DIRECT_N)
        hipLaunchKernelGGL((k_scan_direct<FirstFlag, FirstStore>), dim3((n + SCAN_DIRECT_NT - 1) / SCAN_DIRECT_NT),
                           dim3(SCAN_DIRECT_NT), 0, ctx->stream, n, flag, store, total);
    else
        PCD_TRY(device_scan(ctx, n, flag, store, &total));
    const PassTail t{n, ctx->m, rule.kind, rule.lambda, total, ctx->d_newid, ctx->d_labels, ctx->d_labels_alt,
                     ctx->d_stats_alt, ctx->d_stats, ctx->d_tot, ctx->d_k, (unsigned long long *)ctx->d_acc, state, p};
    // up to two workgroups per CU: each adds its sums with three atomics
    hipLaunchKernelGGL(k_pass_tail, dim3(grid_for(ctx, n, TAIL_NT, 2)), dim3(TAIL_NT), 0, ctx->stream, t);
    PCD_HIP(hipGetLastError());
    std::swap(ctx->d_labels, ctx->d_labels_alt);
    ctx->k_deferred = true;
    ctx->labels_compressed = true;
    ctx->has_stats = true;
    ctx->stats_pending = false;
    return PCD_OK;
}

// ------------------------------------------------------------ statistics
// framework.cpp:69-143: per vertex, count neighbours with the same label;
// sizes[l] += 1, int_volume[l] += same, ext_volume[l] += deg - same.


__global__ void k_clear_stats(CommStats *st, const int32_t *kp) {
    const int k = *kp;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < k; c += gridDim.x * blockDim.x)
        st[c] = CommStats{0, 0, 0, 0};
}

// The whole recount in one launch: every wave takes work items {v, begin,
// end, first} of the long rows (each lane PF gathers in flight), then its
// share of the small bins, G lanes per vertex.  The labels of vertices
// [0, ncache) are staged in LDS (ids are degree-descending: the most frequent
// gather targets), and the sums go through the workgroup's accumulators, for
// large communities' records are what the pass waited for: a recount of
// R-MAT-20 (31 M entries) under a partition of hub neighbourhoods took 2.5 ms
// with an atomic pair per row and takes 0.17 ms; from singletons, where the
// label gathers bound it, R-MAT-22 (128 M entries) takes 0.62 ms either way.
struct StatsRows {
    int start[6];  // small bins G64..G4: positions [start[b], start[b + 1])
    int nitems, ncache;
    const int4 *items;
    const int32_t *order, *indices, *adj, *labels;
    CommStats *st;
};
constexpr int STATS_NT = 1024, STATS_LOG = 9;  // 64 + 8 KB of LDS: two workgroups per CU

// A label from LDS or memory without a branch: both reads are issued (lanes
// served by LDS all read word 0 in memory), so a row's gathers stay in flight
// together.
struct HotLabels {
    const int32_t *hot, *labels;
    int n;
    __device__ int operator()(int v) const {
        const bool in = v < n;
        const int32_t g = labels[in ? 0 : v], h = hot[in ? v : 0];
        return in ? h : g;
    }
};

template <int G>
__device__ inline void stats_small(const StatsRows &r, int b, int wave_g, int nwaves, const HotLabels &label,
                                   StatsAcc<STATS_LOG> &acc) {
    const int lane = __lane_id(), glane = lane & (G - 1);
    constexpr int per_wave = WAVE / G;
    const int p0 = r.start[b], count = r.start[b + 1] - p0;
    for (int base = wave_g * per_wave; base < count; base += nwaves * per_wave) {
        const int gi = base + lane / G;
        const bool has = gi < count;
        int start = 0, deg = 0, l = 0;
        if (has) {
            const int v = r.order ? r.order[p0 + gi] : p0 + gi;
            start = r.indices[v];
            deg = r.indices[v + 1] - start;
            l = r.labels[v];
        }
        int same = 0;
        for (int j = glane; j < deg; j += G) same += label(r.adj[start + j]) == l ? 1 : 0;
#pragma unroll
        for (int d = G / 2; d > 0; d >>= 1) same += __shfl_xor(same, d, WAVE);
        if (has && glane == 0) acc.add(r.st, l, 1, same, deg - same);
    }
}

__global__ __launch_bounds__(STATS_NT) void k_stats_rows(StatsRows r) {
    constexpr int PF = 8;
    __shared__ int32_t hot[STATS_CACHE];
    __shared__ StatsAcc<STATS_LOG> acc;
    for (int i = threadIdx.x; i < r.ncache; i += STATS_NT) hot[i] = r.labels[i];
    acc.init();
    __syncthreads();
    const HotLabels label{hot, r.labels, r.ncache};
    const int lane = __lane_id();
    const int wave_g = (blockIdx.x * STATS_NT + threadIdx.x) / WAVE;
    const int nwaves = gridDim.x * STATS_NT / WAVE;
    for (int it = wave_g; it < r.nitems; it += nwaves) {
        const int4 w = r.items[it];
        const int l = r.labels[w.x];
        int same = 0;
        for (int j0 = w.y + lane; j0 < w.z; j0 += PF * WAVE) {
            int nb[PF];
#pragma unroll
            for (int e = 0; e < PF; e++) {
                const int j = j0 + e * WAVE;
                nb[e] = j < w.z ? r.adj[j] : -1;
            }
            int lab[PF];
#pragma unroll
            for (int e = 0; e < PF; e++) lab[e] = nb[e] < 0 ? -2 : label(nb[e]);
#pragma unroll
            for (int e = 0; e < PF; e++) same += lab[e] == l ? 1 : 0;
        }
        same = wave_sum(same);
        if (lane == 0) acc.add(r.st, l, w.w ? 1 : 0, same, (w.z - w.y) - same);
    }
    stats_small<64>(r, 0, wave_g, nwaves, label, acc);
    stats_small<32>(r, 1, wave_g, nwaves, label, acc);
    stats_small<16>(r, 2, wave_g, nwaves, label, acc);
    stats_small<8>(r, 3, wave_g, nwaves, label, acc);
    stats_small<4>(r, 4, wave_g, nwaves, label, acc);
    __syncthreads();
    acc.flush(r.st);
}

int collect_statistics_dev(pcd_ctx *ctx) {
    const BinLayout &b = ctx->bins;
    hipLaunchKernelGGL(k_clear_stats, dim3(grid_for(ctx, ctx->k, 256)), dim3(256), 0, ctx->stream, ctx->d_stats,
                       ctx->d_k);
    StatsRows r;
    for (int i = 0; i < 6; i++) r.start[i] = b.start[BIN_G64 + i];
    r.nitems = ctx->num_stat_items;
    r.ncache = ctx->tune.stats_cache ? std::min(ctx->n, STATS_CACHE) : 0;
    r.items = ctx->d_stat_items;
    r.order = ctx->d_order;
    r.indices = ctx->d_indices;
    r.adj = ctx->d_adj;
    r.labels = ctx->d_labels;
    r.st = ctx->d_stats;
    // two workgroups per CU, at most one per 8192 entries: each stages its
    // own copy of the cached labels
    kt_begin(ctx, KS_STATS_ITEMS);
    const int grid = std::max(grid_for(ctx, 2 * (int64_t)ctx->m, 8192, 2), grid_for(ctx, ctx->n, STATS_NT, 2) / 4);
    hipLaunchKernelGGL(k_stats_rows, dim3(std::max(grid, 1)), dim3(STATS_NT), 0, ctx->stream, r);
    kt_end(ctx, KS_STATS_ITEMS);
    PCD_HIP(hipGetLastError());
    ctx->has_stats = true;
    return PCD_OK;
}

// ------------------------------------------------------------ statistics after a propagation step
// The counts of framework.cpp:69-143, brought from the labels before a
// propagation step (L) to those after it (N) through the rows of the
// vertices that moved.  Moving v from lo = L(v) to ln = N(v) touches the
// records of lo and ln alone.  For each neighbour w of v, the ordered pair
// (v, w) -- and (w, v) too when w kept its label, weight f = 2 -- was
// internal to lo when L(w) = lo and is internal to ln when N(w) = ln; a
// pair whose ends both moved is counted once from each end's row.  The
// volume moves by deg(v), and ext = volume - int.  A vertex with NEW_LABEL
// only leaves lo here: compression opens its singleton record.  The sums are
// exact integer additions, so the records equal a full recount.

// One list of the moved vertices, built by an exclusive scan of "moved"
// flags over index t: t < nsmall is small-bin position s[0] + t (its entry
// is the vertex), t in [nsmall, nsmall + nitems) is long-row item
// t - nsmall (its entry is the item index), and a last index with flag 0
// closes the list.  The scan keeps position order, so the small bins'
// moved vertices come out grouped by bin; bounds[b] (b < 5) is where bin b
// starts, bounds[5] where the items start and bounds[6] the total; bounds[7]
// starts k_moved_bits' count at 0.
struct MovedArgs {
    int s[6];  // small bins G64..G4: positions [s[b], s[b+1])
    int nitems;
    const int32_t *order;
    const int4 *items;
    const int32_t *L, *N;
};

struct MovedFlag {
    MovedArgs a;
    __device__ int operator()(int64_t t) const {
        const int nsmall = a.s[5] - a.s[0];
        int v;
        if (t < nsmall) {
            const int p = a.s[0] + (int)t;
            v = a.order ? a.order[p] : p;
        } else if (t < nsmall + a.nitems) {
            v = a.items[t - nsmall].x;
        } else {
            return 0;
        }
        return a.L[v] != a.N[v] ? 1 : 0;
    }
};

struct MovedStore {
    MovedArgs a;
    int32_t *bounds, *list;
    __device__ void operator()(int64_t t, int ex, int flag) const {
        const int nsmall = a.s[5] - a.s[0];
#pragma unroll
        for (int b = 0; b < 5; b++)
            if (t == a.s[b] - a.s[0]) bounds[b] = ex;
        if (t == nsmall) bounds[5] = ex;
        if (t == nsmall + a.nitems) {
            bounds[6] = ex;
            bounds[7] = 0;
        }
        if (!flag) return;
        if (t < nsmall) {
            const int p = a.s[0] + (int)t;
            list[ex] = a.order ? a.order[p] : p;
        } else {
            list[ex] = (int)(t - nsmall);
        }
    }
};

// Moved bitmap: bit v of M is set when vertex v's label changed in the step
// (L[v] != N[v]).  One wave writes one 64-bit word.
// With dk set (a captured pass) it also starts the next compression's
// first-occurrence table, as k_first_init does.  Every CROWD_SAMPLE-th
// workgroup counts the moved vertices that share the old or the new community
// of another of their wave: *crowd tells crowded steps (see
// k_delta_crowded).
constexpr int CROWD_SAMPLE = 16;
__global__ __launch_bounds__(256) void k_moved_bits(int n, const int32_t *L, const int32_t *N, uint64_t *M,
                                                    const int32_t *dk, const int32_t *firstv, int32_t *first,
                                                    int32_t *crowd) {
    const bool sample = blockIdx.x % CROWD_SAMPLE == 0;
    int shared = 0;
    if (dk) {
        const int k = *dk;
        for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < k; c += gridDim.x * blockDim.x) {
            const int w = firstv[c];
            first[c] = N[w] == c ? w : INT32_MAX;
        }
    }
    const int lane = __lane_id();
    const int nwords = (n + WAVE - 1) / WAVE;
    const int wave_g = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
    const int nwaves = gridDim.x * blockDim.x / WAVE;
    for (int wd = wave_g; wd < nwords; wd += nwaves) {
        const int v = wd * WAVE + lane;
        const int lo = v < n ? L[v] : 0, ln = v < n ? N[v] : 0;
        const uint64_t bits = __ballot(lo != ln);
        if (lane == 0) M[wd] = bits;
        if (sample && bits) {
            const int one = __builtin_ctzll(bits);
            shared += __popcll(__ballot(lo != ln && lo == __builtin_amdgcn_readlane(lo, one))) - 1;
            if (__builtin_amdgcn_readlane(ln, one) >= 0)  // leaving vertices join nothing
                shared += __popcll(__ballot(lo != ln && ln == __builtin_amdgcn_readlane(ln, one))) - 1;
        }
    }
    if (sample && lane == 0 && shared) atomicAdd(crowd, shared);
}

// A neighbour's label before the step is its label after the step (already
// gathered) unless the bitmap says it moved, so unmoved neighbours cost one
// random gather instead of two (the bitmap itself stays in L2).

// Moved vertices of one small bin, G lanes each.  The first `left` lanes hold
// one vertex's row and labels each; the wave runs through them two groups of
// 64 / G at a time.  What bounds it is the chain of dependent loads per row,
// which this shortens from five to two for two rows.
constexpr int DELTA_BATCH = 16, DELTA_LOG = 7;
struct DeltaArgs {
    const int32_t *indices, *adj, *L, *N;
    const uint64_t *M;  // moved bitmap, or nullptr: L is read for every neighbour
    CommStats *st;
};
__device__ inline int label_before(const DeltaArgs &a, int w, int after) {
    return !a.M || ((a.M[w >> 6] >> (w & 63)) & 1) ? a.L[w] : after;
}
struct DirectSums {  // no accumulators between a row and the records
    __device__ void add(CommStats *st, int l, int size, int same, int e) { add_stats(st, l, size, same, e); }
};
struct PlainLabels {
    const int32_t *labels;
    __device__ int operator()(int v) const { return labels[v]; }
};
template <int G, class After, class Sums>
__device__ inline void delta_batch(const DeltaArgs &d, int left, int v, const After &after, Sums &acc) {
    const int lane = __lane_id(), glane = lane & (G - 1);
    constexpr int per_wave = WAVE / G;
    int bstart = 0, bdeg = 0, blo = 0, bln = 0;
    if (lane < left) {
        blo = d.L[v];
        bln = d.N[v];
        bstart = d.indices[v];
        bdeg = d.indices[v + 1] - bstart;
    }
    for (int g0 = 0; g0 < left; g0 += 2 * per_wave) {
        int deg[2], lo[2], ln[2], w[2], nw[2], lw[2], a[2], b[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int gi = g0 + t * per_wave + lane / G;
            const int src = gi < left ? gi : 0;
            const int start = __shfl(bstart, src, WAVE);
            deg[t] = __shfl(bdeg, src, WAVE);
            lo[t] = __shfl(blo, src, WAVE);
            ln[t] = __shfl(bln, src, WAVE);
            if (gi >= left) deg[t] = 0;
            w[t] = glane < deg[t] ? d.adj[start + glane] : -1;  // a row of the bin has at most G entries
        }
#pragma unroll
        for (int t = 0; t < 2; t++) nw[t] = w[t] < 0 ? -2 : after(w[t]);
#pragma unroll
        for (int t = 0; t < 2; t++) lw[t] = w[t] < 0 ? -2 : label_before(d, w[t], nw[t]);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int f = lw[t] != nw[t] ? 1 : 2;
            a[t] = w[t] >= 0 && lw[t] == lo[t] ? f : 0;
            b[t] = w[t] >= 0 && nw[t] == ln[t] ? f : 0;
#pragma unroll
            for (int x = G / 2; x > 0; x >>= 1) {
                a[t] += __shfl_xor(a[t], x, WAVE);
                b[t] += __shfl_xor(b[t], x, WAVE);
            }
            if (g0 + t * per_wave + lane / G < left && glane == 0) {
                acc.add(d.st, lo[t], -1, -a[t], a[t] - deg[t]);
                if (ln[t] >= 0) acc.add(d.st, ln[t], 1, b[t], deg[t] - b[t]);
            }
        }
    }
}
// a wave takes up to DELTA_BATCH entries of the bin's list at once
template <int G, class After, class Sums>
__device__ inline void delta_small(const DeltaArgs &d, int wave_g, int nwaves, const int32_t *list, int cnt,
                                   const After &after, Sums &acc) {
    constexpr int per_wave = WAVE / G;
    const int lane = __lane_id();
    // entries per batch: a multiple of per_wave that leaves no wave idle
    const int share = (cnt + nwaves - 1) / nwaves;
    const int batch = min(max(per_wave, DELTA_BATCH), (share + per_wave - 1) / per_wave * per_wave);
    for (int base = wave_g * batch; base < cnt; base += nwaves * batch) {
        const int left = min(batch, cnt - base);
        delta_batch<G>(d, left, lane < left ? list[base + lane] : 0, after, acc);
    }
}

// One long-row item {v, begin, end, first} of a moved vertex, the whole wave
template <class After, class Sums>
__device__ inline void delta_item(const DeltaArgs &d, const int4 &w, int lo, int ln, const After &after, Sums &acc) {
    constexpr int PF = 8;
    const int lane = __lane_id();
    int a = 0, b = 0;
    for (int j0 = w.y + lane; j0 < w.z; j0 += PF * WAVE) {
        int nb[PF];
#pragma unroll
        for (int e = 0; e < PF; e++) {
            const int j = j0 + e * WAVE;
            nb[e] = j < w.z ? d.adj[j] : -1;
        }
        int lw[PF], nw[PF];
#pragma unroll
        for (int e = 0; e < PF; e++) nw[e] = nb[e] < 0 ? -2 : after(nb[e]);
#pragma unroll
        for (int e = 0; e < PF; e++) lw[e] = nb[e] < 0 ? -2 : label_before(d, nb[e], nw[e]);
#pragma unroll
        for (int e = 0; e < PF; e++) {
            if (nb[e] < 0) continue;
            const int f = lw[e] != nw[e] ? 1 : 2;
            a += lw[e] == lo ? f : 0;
            b += nw[e] == ln ? f : 0;
        }
    }
    a = wave_sum(a);
    b = wave_sum(b);
    if (lane == 0) {
        const int len = w.z - w.y;
        acc.add(d.st, lo, w.w ? -1 : 0, -a, a - len);
        if (ln >= 0) acc.add(d.st, ln, w.w ? 1 : 0, b, len - b);
    }
}

// Moved items, one wave each: workgroup wg of nwg takes list entries wg,
// wg + nwg, ..., its waves whichever comes next (rows differ 30-fold in
// length), and the next item's records are on their way while one is counted.
template <class After, class Sums>
__device__ inline void delta_items(const DeltaArgs &d, int wg, int nwg, int *next, const int32_t *list, int cnt,
                                   const int4 *items, const After &after, Sums &acc) {
    const int lane = __lane_id();
    int4 wn = make_int4(0, 0, 0, 0);
    int lon = 0, lnn = 0;
    auto fetch = [&]() {
        int j = 0;
        if (lane == 0) j = atomicAdd(next, 1);
        j = __builtin_amdgcn_readfirstlane(j);
        const int64_t i = wg + (int64_t)j * nwg;
        if (i >= cnt) return false;
        wn = items[list[i]];
        lon = d.L[wn.x];
        lnn = d.N[wn.x];
        return true;
    };
    bool more = fetch();
    while (more) {
        const int4 w = wn;
        const int lo = lon, ln = lnn;
        more = fetch();
        delta_item(d, w, lo, ln, after, acc);
    }
}

// All six moved lists in one launch, so that the lists' short chains of
// dependent loads overlap.  Every workgroup reads the list bounds and computes
// the same split of the grid into ranges, one per list, in proportion to the
// lists' entries (a long-row item as DELTA_ITEM_COST), at least one workgroup
// for a list that is not empty.  The sums go to the records directly, and small
// workgroups finish unevenly and leave room to the next (modularity from
// singletons, steps 1 to 6: R-MAT-18 38 24 18 15 13 12 us, R-MAT-22 670 330 177
// 103 64 46; as k_delta_crowded 66 43 34 25 21 18 and 642 354 200 132 100 77).
// Crowded steps are left to k_delta_crowded.
constexpr int DELTA_NT = 256, DELTA_ITEM_COST = 512, DELTA_PER_CU = 24;
// Moved vertices that share a community with another of their wave, among the
// sampled, up to which a step is not crowded.  Steps that both kernels took:
// counts up to 1, 38 us direct and 51 with accumulators (R-MAT-18, modularity),
// 101 and 141 (R-MAT-22); 2 and 3, 64 and 46, 48 and 39 (Chung-Lu graphs, WCC);
// from 4 on, 62 and 51 to 1465 and 120.
constexpr int CROWDED = 2;
__global__ __launch_bounds__(DELTA_NT) void k_delta_all(const int32_t *list, const int32_t *bounds, const int4 *items,
                                                        DeltaArgs d) {
    int bd[8];
#pragma unroll
    for (int i = 0; i < 8; i++) bd[i] = bounds[i];
    if (bd[0] == bd[6] || bd[7] > CROWDED) return;
    // this workgroup's list, and its place among the list's workgroups
    constexpr int cost[6] = {64, 32, 16, 8, 4, DELTA_ITEM_COST};
    float total = 0.0f, before = 0.0f;
    int nonempty = 0, at = 0, mine = -1, wg = 0, nwg = 1;
#pragma unroll
    for (int i = 0; i < 6; i++) {
        total += (float)(bd[i + 1] - bd[i]) * cost[i];
        nonempty += bd[i + 1] > bd[i];
    }
    const float per = (float)((int)gridDim.x - nonempty) / total;
#pragma unroll
    for (int i = 0; i < 6; i++) {
        if (bd[i + 1] == bd[i]) continue;
        const float upto = before + (float)(bd[i + 1] - bd[i]) * cost[i];
        const int count = 1 + ((int)(upto * per) - (int)(before * per));
        if ((int)blockIdx.x >= at && (int)blockIdx.x < at + count) {
            mine = i;
            wg = (int)blockIdx.x - at;
            nwg = count;
        }
        at += count;
        before = upto;
    }
    if (mine < 0) return;  // beyond the last range
    __shared__ int next;
    if (threadIdx.x == 0) next = 0;
    __syncthreads();
    const int wave_g = wg * (DELTA_NT / WAVE) + (int)threadIdx.x / WAVE, nwaves = nwg * (DELTA_NT / WAVE);
    const PlainLabels after{d.N};
    DirectSums sums;
    switch (mine) {
    case 0: delta_small<64>(d, wave_g, nwaves, list + bd[0], bd[1] - bd[0], after, sums); break;
    case 1: delta_small<32>(d, wave_g, nwaves, list + bd[1], bd[2] - bd[1], after, sums); break;
    case 2: delta_small<16>(d, wave_g, nwaves, list + bd[2], bd[3] - bd[2], after, sums); break;
    case 3: delta_small<8>(d, wave_g, nwaves, list + bd[3], bd[4] - bd[3], after, sums); break;
    case 4: delta_small<4>(d, wave_g, nwaves, list + bd[4], bd[5] - bd[4], after, sums); break;
    default: delta_items(d, wg, nwg, &next, list + bd[5], bd[6] - bd[5], items, after, sums); break;
    }
}

// The same for a crowded step, one that moves many vertices into or out of few
// communities: the atomics on those communities' records are the bound, so the
// sums go through the workgroup's accumulators (first step of CPM 0.01 on
// R-MAT-20, 15.7 M entries: 1.28 ms without, 0.22 with).  Every wave takes its
// share of each list in turn, from a place in the list that differs by list.
// One resident round of workgroups: every workgroup pays the accumulators'
// start and flush (0.34 ms with 2,048 workgroups of 256 threads).
constexpr int CROWD_NT = 1024, DELTA_HOT_ITEMS = 2;
constexpr int64_t DELTA_ONE = 1 << 18;
__global__ __launch_bounds__(CROWD_NT) void k_delta_crowded(int n, int least, const int32_t *list,
                                                            const int32_t *bounds, const int4 *items, DeltaArgs d,
                                                            LoopState *state) {
    if (state && blockIdx.x == 0 && threadIdx.x == 0) loop_next(state);  // a captured pass ends here
    int bd[8];  // read at once: a read per list would lengthen every wave's chain
#pragma unroll
    for (int i = 0; i < 8; i++) bd[i] = bounds[i];
    if (bd[0] == bd[6] || bd[7] <= least) return;
    __shared__ int32_t hot[STATS_CACHE];
    __shared__ StatsAcc<DELTA_LOG> acc;
    __shared__ int next;
    const int nwaves = gridDim.x * CROWD_NT / WAVE;
    // with several long-row items a wave, the labels of the most frequent
    // neighbours are staged in LDS (as in k_stats_rows)
    const HotLabels after{hot, d.N, bd[6] - bd[5] >= DELTA_HOT_ITEMS * nwaves ? min(n, STATS_CACHE) : 0};
    for (int i = threadIdx.x; i < after.n; i += CROWD_NT) hot[i] = d.N[i];
    if (threadIdx.x == 0) next = 0;
    acc.init();
    __syncthreads();
    const int wave_g = (blockIdx.x * CROWD_NT + threadIdx.x) / WAVE;
    auto place = [&](int i) {
        const int w = wave_g + i * (nwaves / 6);
        return w < nwaves ? w : w - nwaves;
    };
    delta_items(d, blockIdx.x, gridDim.x, &next, list + bd[5], bd[6] - bd[5], items, after, acc);
    delta_small<64>(d, place(1), nwaves, list + bd[0], bd[1] - bd[0], after, acc);
    delta_small<32>(d, place(2), nwaves, list + bd[1], bd[2] - bd[1], after, acc);
    delta_small<16>(d, place(3), nwaves, list + bd[2], bd[3] - bd[2], after, acc);
    delta_small<8>(d, place(4), nwaves, list + bd[3], bd[4] - bd[3], after, acc);
    delta_small<4>(d, place(5), nwaves, list + bd[4], bd[5] - bd[4], after, acc);
    __syncthreads();
    acc.flush(d.st);
}

// The same without lists, in one launch, for graphs whose rows are looked at
// sooner than the lists are made: a wave takes 64 positions of a small bin at
// a time and runs through the moved ones, then its share of the items.  Also
// starts the next compression's first-occurrence table (see k_first_init) and
// closes a captured pass.
// Refinement of 20 passes, lists / direct: block models of 10,000 and 40,000
// vertices 1.40 / 1.01 and 1.47 / 1.38 ms, Chung-Lu graphs of 20,000 and 65,000
// vertices 1.99 / 1.84 and 2.38 / 2.24, R-MAT-16 2.72 / 2.29; the line is on the
// safe side, direct was ahead as far as it was measured (R-MAT-18, 174,000
// vertices, 3.97 / 3.54).
constexpr int DIRECT_MAX_N = 1 << 16, DIRECT_NT = 512;
template <int G>
__device__ inline void delta_positions(const DeltaArgs &d, const MovedArgs &m, int b, int wave_g, int nwaves, int *list,
                                       StatsAcc<DELTA_LOG> &acc) {
    const int lane = __lane_id();
    // no wider than the bin leaves every wave busy
    const int count = m.s[b + 1] - m.s[b];
    const int share = min(WAVE, max(2 * WAVE / G, (count + nwaves - 1) / nwaves));
    for (int base = wave_g * share; base < count; base += nwaves * share) {
        const int p = m.s[b] + base + lane;
        const bool in = lane < share && base + lane < count;
        const int v = in ? (m.order ? m.order[p] : p) : 0;
        const bool moved = in && d.L[v] != d.N[v];
        const uint64_t mm = __ballot(moved);
        if (!mm) continue;
        if (moved) list[__popcll(mm & ((1ULL << lane) - 1))] = v;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int left = __popcll(mm);
        delta_batch<G>(d, left, lane < left ? list[lane] : 0, PlainLabels{d.N}, acc);
        __builtin_amdgcn_wave_barrier();
    }
}
__global__ __launch_bounds__(DIRECT_NT) void k_delta_direct(MovedArgs m, DeltaArgs d, const int32_t *dk,
                                                            const int32_t *firstv, int32_t *first, LoopState *state) {
    __shared__ int s_list[DIRECT_NT / WAVE][WAVE];
    __shared__ StatsAcc<DELTA_LOG> acc;
    if (blockIdx.x == 0 && threadIdx.x == 0) loop_next(state);
    const int k = *dk;
    for (int c = blockIdx.x * DIRECT_NT + threadIdx.x; c < k; c += gridDim.x * DIRECT_NT) {
        const int w = firstv[c];
        first[c] = d.N[w] == c ? w : INT32_MAX;
    }
    acc.init();
    __syncthreads();
    const int w = threadIdx.x / WAVE;
    const int nwaves = gridDim.x * DIRECT_NT / WAVE, wave_g = blockIdx.x * DIRECT_NT / WAVE + w;
    auto place = [&](int i) { return (wave_g + i * (nwaves / 6)) % nwaves; };
    for (int i = wave_g; i < m.nitems; i += nwaves) {
        const int4 it = m.items[i];
        const int lo = d.L[it.x], ln = d.N[it.x];
        if (lo != ln) delta_item(d, it, lo, ln, PlainLabels{d.N}, acc);
    }
    delta_positions<64>(d, m, 0, place(1), nwaves, s_list[w], acc);
    delta_positions<32>(d, m, 1, place(2), nwaves, s_list[w], acc);
    delta_positions<16>(d, m, 2, place(3), nwaves, s_list[w], acc);
    delta_positions<8>(d, m, 3, place(4), nwaves, s_list[w], acc);
    delta_positions<4>(d, m, 4, place(5), nwaves, s_list[w], acc);
    __syncthreads();
    acc.flush(d.st);
}

int statistics_delta_dev(pcd_ctx *ctx, const int32_t *before, const int32_t *after) {
    const BinLayout &b = ctx->bins;
    kt_begin(ctx, KS_STATS_DELTA);
    MovedArgs m;
    for (int i = 0; i < 6; i++) m.s[i] = b.start[BIN_G64 + i];
    m.nitems = ctx->num_stat_items;
    m.order = ctx->d_order;
    m.items = ctx->d_stat_items;
    m.L = before;
    m.N = after;
    const DeltaArgs d{ctx->d_indices, ctx->d_adj, before, after, ctx->d_moved_bits, ctx->d_stats};
    if (ctx->fused && ctx->n <= DIRECT_MAX_N) {
        DeltaArgs dd = d;
        dd.M = nullptr;
        const int64_t rows = std::max<int64_t>(m.s[5] - m.s[0], (int64_t)m.nitems * 16);
        hipLaunchKernelGGL(k_delta_direct, dim3(grid_for(ctx, rows, 64, 4)), dim3(DIRECT_NT), 0, ctx->stream, m, dd,
                           ctx->d_k, ctx->d_firstv, ctx->d_first, ctx->fused);
        kt_end(ctx, KS_STATS_DELTA);
        PCD_HIP(hipGetLastError());
        return PCD_OK;
    }
    int32_t *bounds = ctx->d_moved;
    int32_t *list = ctx->d_moved + 8;
    const int64_t len = (int64_t)(m.s[5] - m.s[0]) + m.nitems + 1;
    PCD_TRY(device_scan(ctx, len, MovedFlag{m}, MovedStore{m, bounds, list}, nullptr));
    hipLaunchKernelGGL(k_moved_bits, dim3(grid_for(ctx, (ctx->n + WAVE - 1) / WAVE, 4, 8)), dim3(256), 0, ctx->stream,
                       ctx->n, before, after, ctx->d_moved_bits, ctx->fused ? ctx->d_k : nullptr, ctx->d_firstv,
                       ctx->d_first, bounds + 7);
    // one of the two has work; fewer workgroups for small graphs, and of graphs
    // below DELTA_ONE entries the second takes every step: a launch more is
    // what they would notice (R-MAT-12, 97,000 entries: 27 to 22 us a step
    // either way)
    const int64_t E = 2 * (int64_t)ctx->m;
    const bool one = E < DELTA_ONE;
    if (!one)
        hipLaunchKernelGGL(k_delta_all, dim3(std::max(8, grid_for(ctx, E, 1024, DELTA_PER_CU))), dim3(DELTA_NT), 0,
                           ctx->stream, list, bounds, ctx->d_stat_items, d);
    hipLaunchKernelGGL(k_delta_crowded, dim3(std::max(8, grid_for(ctx, E, 2048, 2))), dim3(CROWD_NT), 0, ctx->stream,
                       ctx->n, one ? -1 : CROWDED, list, bounds, ctx->d_stat_items, d, ctx->fused);
    kt_end(ctx, KS_STATS_DELTA);
    PCD_HIP(hipGetLastError());
    return PCD_OK;
}

// ------------------------------------------------------------ metric
// Modularity (rules.cpp:9-22) and CPM (rules.cpp:121-129) depend on the
// statistics only through sum(int), sum(vol^2) and sum(size*(size-1)),
// which are accumulated exactly in int64 (order independent); the final
// double arithmetic runs on the device.  Conductance (rules.cpp:58-70) is
// an FP64 sum in a fixed two-level order.

__global__ __launch_bounds__(256) void k_metric_sums(const CommStats *st, const int32_t *kp,
                                                     unsigned long long *acc) {
    __shared__ long long lds[3][256 / WAVE];
    const int k = *kp;
    long long a = 0, b = 0, c = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < k; i += gridDim.x * blockDim.x) {
        CommStats s = st[i];
        long long vol = (long long)s.int_vol + s.ext_vol;
        a += s.int_vol;
        b += vol * vol;
        c += (long long)s.size * (s.size - 1);
    }
    a = wave_sum64(a); b = wave_sum64(b); c = wave_sum64(c);
    const int w = threadIdx.x / WAVE;
    if (__lane_id() == 0) { lds[0][w] = a; lds[1][w] = b; lds[2][w] = c; }
    __syncthreads();
    if (threadIdx.x < 3) {
        long long t = 0;
        for (int i = 0; i < 256 / WAVE; i++) t += lds[threadIdx.x][i];
        atomicAdd(&acc[threadIdx.x], (unsigned long long)t);
    }
}

__global__ void k_metric_final(const unsigned long long *acc, int kind, double lambda, int m, double *out) {
    *out = score_of_sums((long long)acc[0], (long long)acc[1], (long long)acc[2], kind, lambda, m);
}

constexpr int FSUM_BLOCKS = 1024;

__global__ __launch_bounds__(256) void k_cond_partial(const CommStats *st, const int32_t *kp, double *part) {
    __shared__ double lds[256 / WAVE];
    const int k = *kp;
    double acc = 0;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < k; c += gridDim.x * blockDim.x) {
        CommStats s = st[c];
        acc += s.size * (s.int_vol / (double)(s.int_vol + s.ext_vol));
    }
    acc = wave_sum_f64(acc);
    if (__lane_id() == 0) lds[threadIdx.x / WAVE] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int i = 0; i < 256 / WAVE; i++) t += lds[i];
        part[blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(256) void k_sum_partials(const double *part, int np, double div, double *out) {
    __shared__ double lds[256 / WAVE];
    double acc = 0;
    for (int i = threadIdx.x; i < np; i += blockDim.x) acc += part[i];
    acc = wave_sum_f64(acc);
    if (__lane_id() == 0) lds[threadIdx.x / WAVE] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int i = 0; i < 256 / WAVE; i++) t += lds[i];
        *out = t / div;
    }
}

int metric_dev(pcd_ctx *ctx, pcd_rule rule, double *out) {
    if (rule.kind == PCD_RULE_WCC) return wcc_metric_dev(ctx, out);
    PCD_TRY(metric_enqueue(ctx, rule));
    PCD_HIP(hipStreamSynchronize(ctx->stream));
    *out = ctx->h_result[0];
    return PCD_OK;
}

int metric_enqueue(pcd_ctx *ctx, pcd_rule rule) {
    if (rule.kind == PCD_RULE_WCC) return wcc_metric_enqueue(ctx);
    kt_begin(ctx, KS_METRIC);
    if (rule.kind == PCD_RULE_CONDUCTANCE) {
        hipLaunchKernelGGL(k_cond_partial, dim3(FSUM_BLOCKS), dim3(256), 0, ctx->stream, ctx->d_stats, ctx->d_k,
                           ctx->d_dacc);
        // rules.cpp:69 divides the sum by n
        hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, ctx->stream, ctx->d_dacc, FSUM_BLOCKS,
                           (double)ctx->n, ctx->d_result);
    } else {
        PCD_TRY(fill_u64(ctx, (uint64_t *)ctx->d_acc, 0, 4));
        // the kernel reads k from d_k; a deferred k is bounded by n + 1
        const int kg = ctx->k_deferred ? ctx->n + 1 : ctx->k;
        hipLaunchKernelGGL(k_metric_sums, dim3(grid_for(ctx, kg, 256 * 8, 2)), dim3(256), 0, ctx->stream,
                           ctx->d_stats, ctx->d_k, (unsigned long long *)ctx->d_acc);
        hipLaunchKernelGGL(k_metric_final, dim3(1), dim3(1), 0, ctx->stream, (const unsigned long long *)ctx->d_acc,
                           rule.kind, rule.lambda, ctx->m, ctx->d_result);
    }
    kt_end(ctx, KS_METRIC);
    PCD_HIP(hipGetLastError());
    if (!ctx->capturing)
        PCD_HIP(hipMemcpyAsync(ctx->h_result, ctx->d_result, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    return PCD_OK;
}

}  // namespace pcd
