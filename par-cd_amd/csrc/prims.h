// Device-wide primitives written for CDNA4 wave64: exclusive scan with
// user load/store functors, and wave/block reductions.
#ifndef PARCD_PRIMS_H
#define PARCD_PRIMS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "internal.h"

namespace pcd {

// Community statistics update: size and int_vol are adjacent 32-bit fields,
// so one 64-bit atomic adds both (neither field can carry past 2^31).
// Adds (size, same, ext) to record l; size and same share one 64-bit
// atomic.  The deltas may be negative: the packed word changes by
// same * 2^32 + size mod 2^64, so a transient borrow between the halves is
// undone by the later additions and the final halves are exact.
__device__ inline void add_stats(CommStats *st, int l, int size, int same, int ext) {
    atomicAdd((unsigned long long *)&st[l].size,
              (unsigned long long)((long long)same * 4294967296LL + (long long)size));
    if (ext) atomicAdd(&st[l].ext_vol, ext);
}

// Workgroup-local accumulators of add_stats, so that the members of a large
// community cost one pair of memory atomics per workgroup instead of one per
// member: atomics on one address are served one after another (about 10 ns
// each on MI355X, the bound of a statistics pass over a partition with a few
// large communities).  A slot is taken by the first label that hashes to it
// and kept until the flush; a label whose two slots are taken by others goes
// to memory directly, so communities that are small or many lose two LDS
// reads and nothing else.  Call init, then a barrier, add from any lane, a
// barrier, flush.  The sums are integers: their order does not matter.
template <int LOG>
struct StatsAcc {
    int key[1 << LOG];
    int ext[1 << LOG];
    unsigned long long si[1 << LOG];  // size and int_volume, packed as in CommStats

    __device__ void init() {
        for (int i = threadIdx.x; i < (1 << LOG); i += blockDim.x) {
            key[i] = EMPTY_KEY;
            ext[i] = 0;
            si[i] = 0;
        }
    }
    // the slot of label l, or -1
    __device__ int slot(int l) {
        const uint32_t x = (uint32_t)l * 0x9E3779B1u;
        int h = (int)(x >> (32 - LOG));
#pragma unroll
        for (int t = 0; t < 2; t++) {
            int k = __hip_atomic_load(&key[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (k == EMPTY_KEY) {
                k = atomicCAS(&key[h], EMPTY_KEY, l);
                if (k == EMPTY_KEY) k = l;
            }
            if (k == l) return h;
            h = (int)((x >> 3) & ((1u << LOG) - 1));
        }
        return -1;
    }
    __device__ void add(CommStats *st, int l, int size, int same, int e) {
        const int h = slot(l);
        if (h < 0) {
            add_stats(st, l, size, same, e);
            return;
        }
        atomicAdd(&si[h], (unsigned long long)((long long)same * 4294967296LL + (long long)size));
        if (e) atomicAdd(&ext[h], e);
    }
    __device__ void flush(CommStats *st) {
        for (int i = threadIdx.x; i < (1 << LOG); i += blockDim.x) {
            const int l = key[i];
            if (l == EMPTY_KEY) continue;
            if (si[i]) atomicAdd((unsigned long long *)&st[l].size, si[i]);
            if (ext[i]) atomicAdd(&st[l].ext_vol, ext[i]);
        }
    }
};

// rules.cpp:9-22 (modularity) and rules.cpp:121-129 (CPM) from the exact sums of
// int_volume, volume^2 and size (size - 1)
__device__ inline double score_of_sums(long long a, long long b, long long c, int kind, double lambda, int m) {
    const double two_m = 2.0 * m;
    if (kind == PCD_RULE_MODULARITY) return a / two_m - (double)b / (two_m * two_m);
    return (a - lambda * (double)c) / (double)(2 * m);
}

// main.cpp:241-242, -n and the iteration cap for the pass the state stands at
__device__ inline void loop_rule(LoopState *s, double sc, int k, const LoopParams &p) {
    if (s->frozen) return;
    const int it = s->it;
    if (it >= s->it_end) {
        s->frozen = 1;
        s->just = 1;
        s->k_freeze = k;
        s->step = -1;
        return;
    }
    const bool known = (p.max_iter != -1 && it >= p.max_iter) || it >= p.cap;
    const bool d = known || (p.max_iter == -1 && s->prev > 0 && sc > 0 && sc / s->prev - 1 <= p.threshold);
    s->cur = sc;
    s->cur_k = k;
    if (d) {
        s->frozen = 1;
        s->done = 1;
        s->just = 1;
        s->k_freeze = k;
        s->score_done = sc;
        s->step = -1;
    } else {
        s->step = it;
    }
}

// closes the pass; the next one's step number (a propagation that runs beside
// its metric starts before the rule has seen the score)
__device__ inline void loop_next(LoopState *s) {
    if (!s->frozen) {
        s->prev = s->cur;
        s->prev_k = s->cur_k;
        s->it++;
        s->step = s->it;
    }
    s->just = 0;
}

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ROUNDS = 16;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ROUNDS;

__device__ inline int lane_id() { return __lane_id(); }

__device__ inline int wave_incl_scan(int x) {
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        int y = __shfl_up(x, d, WAVE);
        if (lane_id() >= d) x += y;
    }
    return x;
}

__device__ inline int wave_sum(int x) {
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) x += __shfl_xor(x, d, WAVE);
    return x;
}

__device__ inline long long wave_sum64(long long x) {
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) x += __shfl_xor(x, d, WAVE);
    return x;
}

__device__ inline double wave_sum_f64(double x) {
#pragma unroll
    for (int d = WAVE / 2; d > 0; d >>= 1) x += __shfl_xor(x, d, WAVE);
    return x;
}

// Block-wide exclusive scan of one value per thread (blockDim == SCAN_THREADS);
// returns the exclusive prefix, *total receives the block sum.
__device__ inline int block_excl_scan(int x, int *total, int *lds /* >= SCAN_THREADS/WAVE + 1 */) {
    const int lane = lane_id(), w = threadIdx.x / WAVE;
    int inc = wave_incl_scan(x);
    if (lane == WAVE - 1) lds[w] = inc;
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < SCAN_THREADS / WAVE; i++) {
        int t = lds[i];
        if (i < w) base += t;
        tot += t;
    }
    __syncthreads();
    *total = tot;
    return base + inc - x;
}

// Block-wide exclusive scan for a block of NT threads (all threads call).
template <int NT>
__device__ inline int block_excl_scan_n(int x, int *total, int *lds /* >= NT/WAVE */) {
    const int lane = lane_id(), w = threadIdx.x / WAVE;
    int inc = wave_incl_scan(x);
    __syncthreads();
    if (lane == WAVE - 1) lds[w] = inc;
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NT / WAVE; i++) {
        int t = lds[i];
        if (i < w) base += t;
        tot += t;
    }
    __syncthreads();
    *total = tot;
    return base + inc - x;
}

// Phase 1: per-tile sums (a tile is `rounds` x SCAN_THREADS values).
template <class Load>
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_tiles(int64_t n, Load load, int32_t *parts, int rounds) {
    __shared__ int lds[SCAN_THREADS / WAVE + 1];
    const int64_t base = (int64_t)blockIdx.x * rounds * SCAN_THREADS;
    int acc = 0;
#pragma unroll 4
    for (int r = 0; r < rounds; r++) {
        int64_t i = base + (int64_t)r * SCAN_THREADS + threadIdx.x;
        if (i < n) acc += load(i);
    }
    acc = wave_sum(acc);
    if (lane_id() == 0) lds[threadIdx.x / WAVE] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        int s = 0;
        for (int i = 0; i < SCAN_THREADS / WAVE; i++) s += lds[i];
        parts[blockIdx.x] = s;
    }
}

// Phase 2: exclusive scan of the tile sums by one block; parts[nparts] = total.
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_parts(int nparts, int32_t *parts);

// Phase 3: rescan each tile with its offset; store(i, exclusive, value).
template <class Load, class Store>
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_apply(int64_t n, Load load, Store store, const int32_t *parts,
                                                             int rounds) {
    __shared__ int lds[SCAN_THREADS / WAVE + 1];
    const int64_t base = (int64_t)blockIdx.x * rounds * SCAN_THREADS;
    int run = parts[blockIdx.x];
    for (int r = 0; r < rounds; r++) {
        int64_t i = base + (int64_t)r * SCAN_THREADS + threadIdx.x;
        int x = i < n ? load(i) : 0;
        int tot;
        int ex = block_excl_scan(x, &tot, lds);
        if (i < n) store(i, run + ex, x);
        run += tot;
    }
}

// The scan in one launch: every workgroup sums the values before its tile
// itself, which for up to SCAN_DIRECT_N values costs less than the two
// launches and their gaps that a scan of tile sums takes (first occurrences
// of 10,000 labels: 7 us instead of 9 and two gaps; of 60,000 it costs 8 us
// more).  *total receives the sum.
constexpr int SCAN_DIRECT_N = 20480, SCAN_DIRECT_NT = 1024;
template <class Load, class Store>
__global__ __launch_bounds__(SCAN_DIRECT_NT) void k_scan_direct(int n, Load load, Store store, int32_t *total) {
    __shared__ int lds[SCAN_DIRECT_NT / WAVE];
    const int tile = blockIdx.x * SCAN_DIRECT_NT;
    int before = 0;
#pragma unroll 8
    for (int v = threadIdx.x; v < tile; v += SCAN_DIRECT_NT) before += load(v);
    int run;
    block_excl_scan_n<SCAN_DIRECT_NT>(before, &run, lds);
    const int v = tile + threadIdx.x;
    const int x = v < n ? load(v) : 0;
    int tot;
    const int ex = block_excl_scan_n<SCAN_DIRECT_NT>(x, &tot, lds);
    if (v < n) store(v, run + ex, x);
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *total = run + tot;
}

// Rounds per scan tile for n values: of 16, 8, 4, 2 and 1, the one whose
// tile count is nearest (by ratio) to scan_tiles_per_cu tiles per CU, the
// smaller on a tie (a small n is one tile whatever the rounds).  A scan is then a few short rounds on many workgroups
// rather than 16 serial rounds on a few (its time is latency, not work),
// without so many tiles that the one-workgroup scan of their sums grows.
inline int scan_rounds(const pcd_ctx *ctx, int64_t n) {
    const double want = (double)ctx->tune.scan_tiles_per_cu * ctx->cu_count;
    int best = SCAN_ROUNDS;
    double best_d = 1e300;
    for (int r = SCAN_ROUNDS; r >= 1; r /= 2) {
        const int64_t tiles = (n + (int64_t)r * SCAN_THREADS - 1) / ((int64_t)r * SCAN_THREADS);
        const double ratio = tiles > 0 ? (double)tiles / want : 1e-300;
        const double d = ratio >= 1.0 ? ratio : 1.0 / ratio;
        if (d <= best_d) {
            best_d = d;
            best = r;
        }
    }
    return best;
}

// Exclusive scan over [0, n): load(i) gives the value, store(i, prefix,
// value) consumes it.  The total lands in ctx->d_scan_part[num_tiles].
// Returns the device address of the total.
template <class Load, class Store>
int device_scan(pcd_ctx *ctx, int64_t n, Load load, Store store, int32_t **total_dev) {
    PCD_TRY(ensure_scan_parts(ctx, n));
    const int rounds = scan_rounds(ctx, n);
    int64_t tiles = (n + (int64_t)rounds * SCAN_THREADS - 1) / ((int64_t)rounds * SCAN_THREADS);
    if (tiles < 1) tiles = 1;
    if (tiles + 1 > ctx->scan_part_cap) return fail(PCD_E_STATE, "scan tile sums exceed their buffer");
    hipLaunchKernelGGL(k_scan_tiles<Load>, dim3((unsigned)tiles), dim3(SCAN_THREADS), 0, ctx->stream, n, load,
                       ctx->d_scan_part, rounds);
    hipLaunchKernelGGL(k_scan_parts, dim3(1), dim3(SCAN_THREADS), 0, ctx->stream, (int)tiles, ctx->d_scan_part);
    hipLaunchKernelGGL((k_scan_apply<Load, Store>), dim3((unsigned)tiles), dim3(SCAN_THREADS), 0, ctx->stream, n,
                       load, store, ctx->d_scan_part, rounds);
    PCD_HIP(hipGetLastError());
    if (total_dev) *total_dev = ctx->d_scan_part + tiles;
    return PCD_OK;
}

}  // namespace pcd

#endif
