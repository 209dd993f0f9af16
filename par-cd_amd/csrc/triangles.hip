// Triangle counting (Graph::count_triangles, graph.cpp:107-175) and the
// internal-triangle pass of WCCRule::calculate (rules.cpp:150-235).
//
// For each vertex v and each neighbour u < v, the reference intersects
// N(v) ∩ [0,u) with N(u) ∩ [0,u), and for every common w adds one to the
// entry counters of (v,w), (u,w) and (v,u); then every entry (x,y), y < x,
// with a positive counter adds it to both ends' totals and one edge to both
// ends' degrees.  Here v's prefix (its neighbours below v) goes into an LDS
// hash table and the entries of N(u) ∩ [0,u) are looked up in it, one LDS
// read for most that are not there.  The counters of (v,·) live beside the
// table, and they give every vertex total: the triangles of (v,p), v the
// highest corner, add two to p each and two to v each.  Of (u,w) only "some
// triangle uses this entry" matters, so a hit stores a flag byte instead of
// adding to a counter in memory.  R-MAT-18 (3.8 M edges, 660 M lookups):
// 6.4 ms with binary searches, an atomic per hit and a pass that summed the
// counters with two atomics per edge; 1.1 ms so, 600 G lookups/s, bound by the
// instructions and LDS reads of a lookup.  With labels given, only edges and triangles inside one
// community count (rules.cpp:172,185): neighbours of other communities are
// left out of the prefix.
#include <algorithm>

#include "prims.h"

namespace pcd {

// prefixes of at most TRI_WAVE entries: one wave per vertex; longer ones,
// listed once per graph: one workgroup per vertex
constexpr int TRI_WAVE = 64, TRI_WAVE_LOG = 9;
constexpr int TRI_BLOCK_LOG = 11, TRI_CHUNK = 1 << (TRI_BLOCK_LOG - 1);
// vertices whose totals a workgroup sums in LDS: the lowest ids are the
// highest degrees, and their words are what the additions queue on
constexpr int TRI_HOT = 1024;
constexpr int TRI_PF = 3;  // row entries a lane looks up at once

// lowpos[v] = number of neighbours of v with a smaller id, and, where `list` is
// given, the vertices whose prefix exceeds one table, in any order (there are
// few: *listed starts at 0)
__global__ void k_lowpos(int n, const int32_t *indices, const int32_t *adj, int32_t *lowpos, int32_t *list,
                         int32_t *listed) {
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
        int lo = indices[v], hi = indices[v + 1];
        while (lo < hi) {
            int mid = (lo + hi) >> 1;
            if (adj[mid] < v) lo = mid + 1;
            else hi = mid;
        }
        lo -= indices[v];
        lowpos[v] = lo;
        if (list && lo > TRI_CHUNK) list[atomicAdd(listed, 1)] = v;
    }
}

struct TriArgs {
    int n;
    const int32_t *indices, *adj, *lowpos, *labels;
    const int32_t *list, *listed;  // vertices with longer prefixes, their number
    uint8_t *flag;                 // per entry (x,y), y < x: some counted triangle uses it
    int32_t *tri;
};

struct LongPrefix {
    const int32_t *lowpos;
    __device__ int operator()(int64_t v) const { return lowpos[v] > TRI_WAVE ? 1 : 0; }
};
struct LongStore {
    int32_t *list, *listed;
    int64_t n;
    __device__ void operator()(int64_t v, int ex, int flag) const {
        if (flag) list[ex] = (int)v;
        if (v == n - 1) *listed = ex + flag;
    }
};

__device__ inline void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Table of at least 8 slots per entry (2 at the cap): what is not there is
// then mostly told by one read (R-MAT-18: 1.46 ms at 4 slots, 1.23 at 8).
__device__ inline int tri_log(int len) { return max(6, 32 - __clz(8 * len - 1)); }

__device__ inline int tri_insert(int *keys, int log, int x) {
    const int mask = (1 << log) - 1;
    int h = (int)(((uint32_t)x * 0x9E3779B1u) >> (32 - log));
    while (atomicCAS(&keys[h], EMPTY_KEY, x) != EMPTY_KEY) h = (h + 1) & mask;  // the keys of a row differ
    return h;
}

// slot of x, or -1, given the key k of its first slot h; a table is never full
__device__ inline int tri_probe(const int *keys, int log, int x, int h, int k) {
    const int mask = (1 << log) - 1;
    while (k != x && k != EMPTY_KEY) {
        h = (h + 1) & mask;
        k = keys[h];
    }
    return k == x ? h : -1;
}
__device__ inline int tri_find(const int *keys, int log, int x) {
    const int h = (int)(((uint32_t)x * 0x9E3779B1u) >> (32 - log));
    return tri_probe(keys, log, x, h, keys[h]);
}

// W lanes look the entries [s, s + len) up, PF a lane in flight; returns
// this lane's hits
template <int W, int PF>
__device__ inline int tri_row(const TriArgs &a, const int *keys, int *cnts, int log, int s, int len, int glane) {
    int found = 0;
    for (int y = glane; y < len; y += PF * W) {
        int x[PF], k[PF];
#pragma unroll
        for (int e = 0; e < PF; e++) x[e] = a.adj[s + min(y + e * W, len - 1)];
#pragma unroll
        for (int e = 0; e < PF; e++) k[e] = keys[((uint32_t)x[e] * 0x9E3779B1u) >> (32 - log)];
#pragma unroll
        for (int e = 0; e < PF; e++) {
            if (y + e * W >= len || k[e] == EMPTY_KEY) continue;
            const int h = tri_probe(keys, log, x[e], (int)(((uint32_t)x[e] * 0x9E3779B1u) >> (32 - log)), k[e]);
            if (h >= 0) {
                found++;
                atomicAdd(&cnts[h], 1);
                a.flag[s + y + e * W] = 1;
            }
        }
    }
    return found;
}

__device__ inline void tri_add(const TriArgs &a, int *hot, int x, int c) {
    if (x < TRI_HOT) atomicAdd(&hot[x], c);
    else atomicAdd(&a.tri[x], c);
}

template <int NT>
__device__ inline void tri_flush(const TriArgs &a, const int *hot) {
    __syncthreads();
    for (int i = threadIdx.x; i < TRI_HOT; i += NT)
        if (hot[i]) atomicAdd(&a.tri[i], hot[i]);
}

// A wave looks at `per` vertices at once (eight, fewer where the graph has too
// few vertices for all waves), eight lanes each, and takes those with at least
// two (same-label) neighbours below them one by one.  Rows
// u are read 64 lanes wide, or four at a time 16 lanes wide where they are
// short on average (Chung-Lu rows hold 30-60 entries, R-MAT rows 150-190).
// A wave's vertices follow one another, or with `spread` lie the number of
// waves apart: ids descend by degree, so the dear ones stand together, and up
// to TRI_SPREAD_N vertices there are too few waves to even that out
// (consecutive / spread: Chung-Lu graphs of 60,000 vertices 334 / 168 us, of
// 200,000 568 / 491, of 400,000 872 / 869; where only the internal triangles
// of small communities count, reading the extents is most of it: 44 / 45 us,
// 75 / 81, 101 / 108).
constexpr int TRI_SPREAD_N = 1 << 18;
__global__ __launch_bounds__(256) void k_triangles_wave(TriArgs a, int per, bool spread) {
    __shared__ int s_keys[256 / WAVE][1 << TRI_WAVE_LOG], s_cnts[256 / WAVE][1 << TRI_WAVE_LOG];
    __shared__ int s_row[256 / WAVE][3][TRI_WAVE];
    __shared__ int hot[TRI_HOT];
    for (int i = threadIdx.x; i < TRI_HOT; i += 256) hot[i] = 0;
    __syncthreads();
    const int lane = __lane_id(), w = threadIdx.x / WAVE, oct = lane & 7;
    const uint64_t below = (1ULL << lane) - 1;
    int *keys = s_keys[w], *cnts = s_cnts[w];
    int *rsu = s_row[w][0], *rlen = s_row[w][1], *rcnt = s_row[w][2];
    const int wave_g = (blockIdx.x * 256 + threadIdx.x) / WAVE;
    const int nwaves = gridDim.x * (256 / WAVE);
    const int step = spread ? nwaves : 1;
    for (int64_t base = spread ? wave_g : (int64_t)wave_g * per; base < a.n; base += (int64_t)nwaves * per) {
        const int64_t vl = base + (int64_t)(lane / 8) * step;
        const int vo = (int)min((int64_t)a.n - 1, vl);
        int plen = lane / 8 < per && vl < a.n ? a.lowpos[vo] : 0;
        if (plen > TRI_WAVE) plen = 0;
        const int pstart = a.indices[vo], plab = a.labels ? a.labels[vo] : 0;
        int mine = plen;
        if (a.labels) {
            mine = 0;
            for (int i = oct; i < plen; i += 8) mine += a.labels[a.adj[pstart + i]] == plab;
#pragma unroll
            for (int d = 4; d > 0; d >>= 1) mine += __shfl_xor(mine, d, WAVE);
        }
        uint64_t todo = __ballot(oct == 0 && mine >= 2);
        while (todo) {
            const int src = __builtin_ctzll(todo);
            todo &= todo - 1;
            const int v = (int)(base + (int64_t)(src / 8) * step);
            const int len = __builtin_amdgcn_readlane(plen, src), sv = __builtin_amdgcn_readlane(pstart, src);
            const int lab = __builtin_amdgcn_readlane(plab, src);
            const int log = tri_log(len);
            for (int i = lane; i < (1 << log); i += WAVE) {
                keys[i] = EMPTY_KEY;
                cnts[i] = 0;
            }
            int u = -1, su = 0, lu = 0, slot = 0;
            if (lane < len) {
                u = a.adj[sv + lane];
                if (a.labels && a.labels[u] != lab) u = -1;
                if (u >= 0) {
                    su = a.indices[u];
                    lu = a.lowpos[u];
                }
            }
            wave_sync_lds();
            if (u >= 0) slot = tri_insert(keys, log, u);
            if (lane == 0) lu = 0;  // no neighbour lies below the lowest
            wave_sync_lds();
            uint64_t rows = __ballot(lu > 0);
            const int nrows = __popcll(rows), total = wave_sum(lu);
            int found = 0;  // of this lane's row
            if (total > 32 * nrows) {
                while (rows) {
                    const int r = __builtin_ctzll(rows);
                    rows &= rows - 1;
                    const int f = wave_sum(tri_row<WAVE, TRI_PF>(a, keys, cnts, log, __builtin_amdgcn_readlane(su, r),
                                                         __builtin_amdgcn_readlane(lu, r), lane));
                    if (lane == r) found = f;
                }
            } else {
                const int at = __popcll(rows & below);
                if (lu > 0) {
                    rsu[at] = su;
                    rlen[at] = lu;
                }
                wave_sync_lds();
                for (int i = lane / 16; i < nrows; i += WAVE / 16) {
                    int f = tri_row<16, 2>(a, keys, cnts, log, rsu[i], rlen[i], lane & 15);
#pragma unroll
                    for (int d = 8; d > 0; d >>= 1) f += __shfl_xor(f, d, WAVE);
                    if ((lane & 15) == 0) rcnt[i] = f;
                }
                wave_sync_lds();
                if (lu > 0) found = rcnt[at];
            }
            wave_sync_lds();
            const int c = u >= 0 ? cnts[slot] + found : 0;
            if (c) {
                a.flag[sv + lane] = 1;
                tri_add(a, hot, u, 2 * c);
            }
            const int tv = wave_sum(c);
            if (lane == 0 && tv) tri_add(a, hot, v, tv);
            wave_sync_lds();
        }
    }
    tri_flush<256>(a, hot);
}

// [first entry >= lo, first entry > hi) of the ascending entries [s, s + len):
// what of a row can be in a table of the ids lo..hi.  Rows shorter than one
// step of a wave are kept or left out as a whole.
__device__ inline void tri_clip(const TriArgs &a, int lo, int hi, int &s, int &len) {
    if (a.adj[s + len - 1] < lo || a.adj[s] > hi) {
        len = 0;
        return;
    }
    if (len <= TRI_PF * WAVE) return;
    const int e = s + len;
    int b = s, t = e;
    while (b < t) {
        const int mid = b + (t - b) / 2;
        if (a.adj[mid] < lo) b = mid + 1;
        else t = mid;
    }
    s = b;
    t = e;
    while (b < t) {
        const int mid = b + (t - b) / 2;
        if (a.adj[mid] <= hi) b = mid + 1;
        else t = mid;
    }
    len = b - s;
}

// One workgroup per listed vertex: its prefix goes into the table, and the
// waves take the rows behind its first entry (64 rows' extents loaded at once,
// one lane each).  Prefixes of more than TRI_CHUNK entries, the hubs of graphs
// whose ids do not descend by degree, go in by chunks, and of a row only the
// entries within the chunk's ids are looked up in it, not every entry once per
// chunk (a hub after the 200,000 vertices of its wheel 179 -> 8 ms).  They have
// a list and a launch of their own: the parts below are then counted over them
// alone (R-MAT-19 with shuffled ids, clipped, 57 -> 18 ms), and the clipping in
// one kernel with the others cost these 10 % (R-MAT-20 3.5 -> 3.9 ms).  Where
// the list is short, up to TRI_PARTS workgroups share a vertex, each with its
// own table and a part of the rows: the rows of one wave are a serial chain.
// With that and the smaller units of k_triangles_wave a repeated call takes 100
// us for R-MAT-11, 172 for R-MAT-13 (237 and 332 without, 142 and 270 with a
// binary search per lookup); R-MAT-18 is unchanged.
constexpr int TRI_PARTS = 16, TRI_BLOCK_NT = 256;
template <bool CHUNKS>
__global__ __launch_bounds__(TRI_BLOCK_NT) void k_triangles_block(TriArgs a, const int32_t *list,
                                                                  const int32_t *listed) {
    constexpr int NT = TRI_BLOCK_NT, NW = NT / WAVE;
    __shared__ int keys[1 << TRI_BLOCK_LOG], cnts[1 << TRI_BLOCK_LOG];
    __shared__ int hot[TRI_HOT];
    const int nlist = *listed;
    if (nlist == 0) return;
    for (int i = threadIdx.x; i < TRI_HOT; i += NT) hot[i] = 0;
    const int lane = __lane_id(), w = threadIdx.x / WAVE;
    const int parts = max(1, min(TRI_PARTS, (int)gridDim.x / nlist));
    const int64_t items = (int64_t)nlist * parts;
    for (int64_t it = blockIdx.x; it < items; it += gridDim.x) {
        const int v = list[it / parts];
        const int first = (int)(it % parts) * NW + w, step = parts * NW;  // this wave's rows
        const int sv = a.indices[v], len = a.lowpos[v], lab = a.labels ? a.labels[v] : 0;
        if (!CHUNKS && len > TRI_CHUNK) continue;
        int tv = 0;
        for (int c0 = 0; c0 < len; c0 += TRI_CHUNK) {
            const int c1 = min(len, c0 + TRI_CHUNK);
            const int log = min(TRI_BLOCK_LOG, tri_log(c1 - c0));
            for (int i = threadIdx.x; i < (1 << log); i += NT) {
                keys[i] = EMPTY_KEY;
                cnts[i] = 0;
            }
            __syncthreads();
            for (int i = c0 + threadIdx.x; i < c1; i += NT) {
                const int u = a.adj[sv + i];
                if (!a.labels || a.labels[u] == lab) tri_insert(keys, log, u);
            }
            __syncthreads();
            for (int r0 = c0 + 1 + first; r0 < len; r0 += step * WAVE) {
                const int r = r0 + step * lane;
                int u = -1, su = 0, lu = 0;
                if (r < len) {
                    u = a.adj[sv + r];
                    if (!a.labels || a.labels[u] == lab) {
                        su = a.indices[u];
                        lu = a.lowpos[u];
                        if (CHUNKS && lu > 0) tri_clip(a, a.adj[sv + c0], a.adj[sv + c1 - 1], su, lu);
                    }
                }
                int found = 0;
                uint64_t rows = __ballot(lu > 0);
                while (rows) {
                    const int i = __builtin_ctzll(rows);
                    rows &= rows - 1;
                    const int f = wave_sum(tri_row<WAVE, TRI_PF>(a, keys, cnts, log, __builtin_amdgcn_readlane(su, i),
                                                         __builtin_amdgcn_readlane(lu, i), lane));
                    if (lane == i) found = f;
                }
                if (found) {
                    a.flag[sv + r] = 1;
                    tri_add(a, hot, u, 2 * found);
                    tv += found;
                }
            }
            __syncthreads();
            for (int i = threadIdx.x; i < (1 << log); i += NT) {
                const int c = cnts[i];
                if (c) {
                    tri_add(a, hot, keys[i], 2 * c);
                    tv += c;
                }
            }
            for (int i = c0 + threadIdx.x; i < c1; i += NT) {
                const int x = tri_find(keys, log, a.adj[sv + i]);
                if (x >= 0 && cnts[x]) a.flag[sv + i] = 1;
            }
            __syncthreads();
        }
        tv = wave_sum(tv);
        if (lane == 0 && tv) tri_add(a, hot, v, tv);
    }
    tri_flush<NT>(a, hot);
}

// Each flagged entry (v,u) counts one edge at both ends (graph.cpp:146-159,
// rules.cpp:197-211): eight lanes per vertex, one wave per listed vertex.
constexpr int TDEG_NT = 1024, TDEG_HOT = 4096;
__global__ __launch_bounds__(TDEG_NT) void k_tri_degrees(TriArgs a, int32_t *tdeg) {
    __shared__ int hot[TDEG_HOT];
    for (int i = threadIdx.x; i < TDEG_HOT; i += TDEG_NT) hot[i] = 0;
    __syncthreads();
    const int lane = __lane_id();
    auto add = [&](int x, int c) {
        if (x < TDEG_HOT) atomicAdd(&hot[x], c);
        else atomicAdd(&tdeg[x], c);
    };
    auto entries = [&](int s, int len, int first, int step) {
        int c = 0;
        for (int i = first; i < len; i += step)
            if (a.flag[s + i]) {
                c++;
                add(a.adj[s + i], 1);
            }
        return c;
    };
    const int64_t g = ((int64_t)blockIdx.x * TDEG_NT + threadIdx.x) / 8, ng = (int64_t)gridDim.x * TDEG_NT / 8;
    for (int64_t v = g; v < a.n; v += ng) {  // the lanes of a group share v
        const int len = a.lowpos[v];
        int c = len <= TRI_WAVE ? entries(a.indices[v], len, lane & 7, 8) : 0;
#pragma unroll
        for (int d = 4; d > 0; d >>= 1) c += __shfl_xor(c, d, WAVE);
        if ((lane & 7) == 0 && c) add((int)v, c);
    }
    const int nlist = *a.listed;
    for (int it = (blockIdx.x * TDEG_NT + threadIdx.x) / WAVE; it < nlist; it += gridDim.x * TDEG_NT / WAVE) {
        const int v = a.list[it];
        const int c = wave_sum(entries(a.indices[v], a.lowpos[v], lane, WAVE));
        if (lane == 0 && c) add(v, c);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < TDEG_HOT; i += TDEG_NT)
        if (hot[i]) atomicAdd(&tdeg[i], hot[i]);
}

// flags of E entries (padded to words) and both totals, cleared
__global__ void k_tri_clear(int64_t words, uint32_t *flag, int n, int32_t *tri, int32_t *tdeg) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x, t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (int64_t i = t; i < words; i += stride) flag[i] = 0;
    for (int64_t i = t; i < n; i += stride) {
        tri[i] = 0;
        tdeg[i] = 0;
    }
}

constexpr int TSUM_BLOCKS = 1024;

// graph.cpp:161-169: cc = sum over v with deg > 1 of (tri/(deg(deg-1)))/n
__global__ __launch_bounds__(256) void k_cc_partial(int n, const int32_t *indices, const int32_t *tri, double *part) {
    __shared__ double lds[256 / WAVE];
    double acc = 0;
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
        int deg = indices[v + 1] - indices[v];
        if (deg > 1) acc += (tri[v] / (deg * (deg - 1.0))) / n;
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

// rules.cpp:213-228
__global__ __launch_bounds__(256) void k_wcc_partial(int n, const int32_t *labels, const CommStats *st,
                                                     const int32_t *tri, const int32_t *tdeg, const int32_t *it,
                                                     const int32_t *itd, double *part) {
    __shared__ double lds[256 / WAVE];
    double acc = 0;
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) {
        int t = tri[v];
        if (t > 0) {
            int size = st[labels[v]].size;
            int dt = tdeg[v];
            double a = it[v] / (double)t;
            double b = dt / (double)(size - 1 + dt - itd[v]);
            acc += (a * b) / n;
        }
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

// (with `count` set, out[1] receives it: one copy brings both to the host)
__global__ __launch_bounds__(256) void k_sum_partials_plain(const double *part, int np, double *out,
                                                            const int32_t *count) {
    __shared__ double lds[256 / WAVE];
    double acc = 0;
    for (int i = threadIdx.x; i < np; i += blockDim.x) acc += part[i];
    acc = wave_sum_f64(acc);
    if (__lane_id() == 0) lds[threadIdx.x / WAVE] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int i = 0; i < 256 / WAVE; i++) t += lds[i];
        *out = t;
        if (count) out[1] = *count;
    }
}

// The arrays of the counts.  A user counts a graph once, and seven allocations
// and three launches for the list were 12 of the 100 us that call takes on up to
// some 10,000 entries: up to TRI_ONE_ALLOC words share one allocation (cut at 64
// words).  Larger arrays have one each; together they took longer to allocate
// (1 M vertices, 15 M entries: the first count 2.6 ms in one, 2.1 in seven).
constexpr int64_t TRI_ONE_ALLOC = 1 << 19;
static int ensure_tri_buffers(pcd_ctx *ctx) {
    if (ctx->d_tri) return PCD_OK;
    const int64_t E = (int64_t)2 * ctx->m;
    // prefixes above 64 entries: at most E / 65 vertices, and their number
    const int64_t cap = std::min<int64_t>(ctx->n, E / (TRI_WAVE + 1)) + 1;
    // and those above one table's
    const int64_t chunked = ctx->max_degree > TRI_CHUNK ? std::min<int64_t>(ctx->n, E / (TRI_CHUNK + 1)) + 1 : 0;
    constexpr int ARRAYS = 8;
    const int64_t n1 = (int64_t)ctx->n + 1, none = chunked ? chunked + 1 : 0;
    const int64_t words[ARRAYS] = {n1, n1, n1, n1, n1, E / 4 + 1, cap + 1, none};
    int64_t total = 0;
    for (int64_t w : words) total += (w + 63) & ~(int64_t)63;
    int32_t *array[ARRAYS] = {}, *block = nullptr;
    if (total <= TRI_ONE_ALLOC) PCD_TRY(dev_alloc_t(ctx, &block, total));
    for (int i = 0; i < ARRAYS; i++) {
        if (words[i] == 0) continue;
        if (block) {
            array[i] = block;
            block += (words[i] + 63) & ~(int64_t)63;
            continue;
        }
        const int rc = dev_alloc_t(ctx, &array[i], words[i]);
        if (rc == PCD_OK) continue;
        for (int k = 0; k < i; k++) dev_free(ctx, array[k]);
        return rc;
    }
    ctx->d_tri_deg = array[1];
    ctx->d_lowpos = array[2];
    ctx->d_it = array[3];
    ctx->d_itd = array[4];
    ctx->d_tri_flag = (uint8_t *)array[5];
    ctx->d_tri_list = array[6];
    ctx->d_tri_chunked = array[7];
    ctx->tri_chunked = -1;
    if (chunked) PCD_TRY(fill_i32(ctx, ctx->d_tri_chunked, 0, 1));
    hipLaunchKernelGGL(k_lowpos, dim3(grid_for(ctx, ctx->n, 256)), dim3(256), 0, ctx->stream, ctx->n, ctx->d_indices,
                       ctx->d_adj, ctx->d_lowpos, chunked ? ctx->d_tri_chunked + 1 : nullptr, ctx->d_tri_chunked);
    // in the order of the ids, which descend by degree: the listed vertices'
    // work then falls off along the list (R-MAT-16 0.49 ms, in any order 0.51)
    const LongPrefix is_long{ctx->d_lowpos};
    const LongStore store{ctx->d_tri_list + 1, ctx->d_tri_list, ctx->n};
    if (ctx->n <= SCAN_DIRECT_N)
        hipLaunchKernelGGL((k_scan_direct<LongPrefix, LongStore>), dim3((ctx->n + SCAN_DIRECT_NT - 1) / SCAN_DIRECT_NT),
                           dim3(SCAN_DIRECT_NT), 0, ctx->stream, ctx->n, is_long, store, ctx->d_tri_list);
    else
        PCD_TRY(device_scan(ctx, ctx->n, is_long, store, nullptr));
    PCD_HIP(hipGetLastError());
    ctx->d_tri = array[0];  // set last: the others are there
    return PCD_OK;
}

// Runs the counting pass (labels: nullptr for all triangles) and leaves the
// per-vertex totals in (t, td).
static int count_pass(pcd_ctx *ctx, const int32_t *labels, int32_t *t, int32_t *td) {
    const int n = ctx->n;
    const int64_t E = (int64_t)2 * ctx->m;
    const TriArgs a{n,      ctx->d_indices,      ctx->d_adj,      ctx->d_lowpos,   labels,
                    ctx->d_tri_list + 1, ctx->d_tri_list, ctx->d_tri_flag, t};
    kt_begin(ctx, KS_TRIANGLES);
    const int64_t words = (E + 3) / 4;
    hipLaunchKernelGGL(k_tri_clear, dim3(grid_for(ctx, std::max<int64_t>(words, n), 256 * 4)), dim3(256), 0,
                       ctx->stream, words, (uint32_t *)ctx->d_tri_flag, n, t, td);
    // several rounds of workgroups: vertices differ a hundredfold in work
    const int64_t listed = std::min<int64_t>(n, E / (TRI_WAVE + 1)) + 1;  // at most
    const dim3 grid((unsigned)std::min<int64_t>(ctx->cu_count * 24, listed * TRI_PARTS)), block(TRI_BLOCK_NT);
    if (ctx->d_tri_chunked && ctx->tri_chunked != 0)  // unknown (-1) until the first count is read back
        hipLaunchKernelGGL(k_triangles_block<true>, grid, block, 0, ctx->stream, a, ctx->d_tri_chunked + 1,
                           ctx->d_tri_chunked);
    hipLaunchKernelGGL(k_triangles_block<false>, grid, block, 0, ctx->stream, a, a.list, a.listed);
    const int per = std::min(8, (n + ctx->cu_count * 32 - 1) / (ctx->cu_count * 32));
    hipLaunchKernelGGL(k_triangles_wave, dim3(grid_for(ctx, n, 4 * per, 24)), dim3(256), 0, ctx->stream, a, per,
                       n <= TRI_SPREAD_N);
    hipLaunchKernelGGL(k_tri_degrees, dim3(grid_for(ctx, n, TDEG_NT / 8, 2)), dim3(TDEG_NT), 0, ctx->stream, a, td);
    kt_end(ctx, KS_TRIANGLES);
    PCD_HIP(hipGetLastError());
    return PCD_OK;
}

int triangles_dev(pcd_ctx *ctx) {
    PCD_TRY(ensure_tri_buffers(ctx));
    PCD_TRY(count_pass(ctx, nullptr, ctx->d_tri, ctx->d_tri_deg));
    hipLaunchKernelGGL(k_cc_partial, dim3(TSUM_BLOCKS), dim3(256), 0, ctx->stream, ctx->n, ctx->d_indices, ctx->d_tri,
                       ctx->d_dacc);
    hipLaunchKernelGGL(k_sum_partials_plain, dim3(1), dim3(256), 0, ctx->stream, ctx->d_dacc, TSUM_BLOCKS,
                       ctx->d_result, ctx->d_tri_chunked);
    PCD_HIP(hipGetLastError());
    PCD_HIP(hipMemcpyAsync(ctx->h_result, ctx->d_result, 2 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    PCD_HIP(hipStreamSynchronize(ctx->stream));
    ctx->cc = ctx->h_result[0];
    if (ctx->d_tri_chunked) ctx->tri_chunked = (int)ctx->h_result[1];
    ctx->has_triangles = true;
    return PCD_OK;
}

// WCCRule::calculate (rules.cpp:150-235) into d_result; the triangles of
// the graph must be counted.  The score is copied to the host unless a pass
// is being captured.
int wcc_metric_enqueue(pcd_ctx *ctx) {
    if (!ctx->has_triangles) return fail(PCD_E_STATE, "WCC metric needs the triangle counts");
    PCD_TRY(count_pass(ctx, ctx->d_labels, ctx->d_it, ctx->d_itd));
    hipLaunchKernelGGL(k_wcc_partial, dim3(TSUM_BLOCKS), dim3(256), 0, ctx->stream, ctx->n, ctx->d_labels,
                       ctx->d_stats, ctx->d_tri, ctx->d_tri_deg, ctx->d_it, ctx->d_itd, ctx->d_dacc);
    hipLaunchKernelGGL(k_sum_partials_plain, dim3(1), dim3(256), 0, ctx->stream, ctx->d_dacc, TSUM_BLOCKS,
                       ctx->d_result, (const int32_t *)nullptr);
    PCD_HIP(hipGetLastError());
    if (!ctx->capturing)
        PCD_HIP(hipMemcpyAsync(ctx->h_result, ctx->d_result, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    return PCD_OK;
}

int wcc_metric_dev(pcd_ctx *ctx, double *out) {
    if (!ctx->has_triangles) PCD_TRY(triangles_dev(ctx));
    PCD_TRY(wcc_metric_enqueue(ctx));
    PCD_HIP(hipStreamSynchronize(ctx->stream));
    *out = ctx->h_result[0];
    return PCD_OK;
}

}  // namespace pcd
