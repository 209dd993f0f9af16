// compress_labels (framework.cpp:146-170) on caller-owned device arrays,
// without any device allocation: the first-occurrence table, the new-id
// table, the scan partials and the error flag live in one file-scope
// device array.  For callers that cannot allocate: code under HIP graph
// capture, serving loops, harnesses that forbid hipMalloc.
//
// Up to NA_SOLO labels take one launch: one workgroup whose first-occurrence
// table, then new-id table, is in LDS.  Larger arrays use
// the algorithm of the context path (partition.hip): first[l] = the least
// vertex with label l (atomicMin), a vertex is a "first" if it holds its
// label's first[] or NEW_LABEL, and the exclusive scan of those flags over
// v is the reference's running counter.  The output is bit-identical.
//
// Calls above NA_SOLO labels share their device's array and overwrite what the
// last one left there; those that overlap in time on one device race.
#include <algorithm>
#include <mutex>

#include "../host/hostutil.hpp"
#include "prims.h"

namespace pcd {
namespace {

constexpr int64_t NA_MAX = PCD_NOALLOC_MAX_VERTICES;
constexpr int64_t NA_TILES = 1024;  // at most (see na_rounds)
// word offsets inside the scratch array
constexpr int64_t NA_FIRST = 0;                      // first[l], l < n
constexpr int64_t NA_NEWID = NA_MAX;                 // newid[l]
constexpr int64_t NA_PARTS = 2 * NA_MAX;             // tile sums, then their scan and the total
constexpr int64_t NA_FLAGS = NA_PARTS + NA_TILES + 64;  // [0] = a label outside [-1, n)
constexpr int64_t NA_WORDS = NA_FLAGS + 64;

static __device__ __align__(256) int32_t scratch[NA_WORDS];

__global__ void k_na_clear(int n, int32_t *first, int32_t *flags) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) first[i] = INT32_MAX;
    if (blockIdx.x == 0 && threadIdx.x == 0) flags[0] = 0;
}

// atomicMin of the first vertex per label, the labels a workgroup meets first
// combined in LDS (as k_first_occurrence); labels outside [-1, n) set the flag
// and are left out of every table
constexpr int NF_NT = 512, NF_LOG = 7;
__global__ __launch_bounds__(NF_NT) void k_na_first(int n, const int32_t *labels, int32_t *first, int32_t *flags) {
    __shared__ int key[1 << NF_LOG], low[1 << NF_LOG];
    for (int i = threadIdx.x; i < (1 << NF_LOG); i += NF_NT) {
        key[i] = EMPTY_KEY;
        low[i] = INT32_MAX;
    }
    __syncthreads();
    for (int v = blockIdx.x * NF_NT + threadIdx.x; v < n; v += gridDim.x * NF_NT) {
        const int l = labels[v];
        if (l < -1 || l >= n) {
            flags[0] = 1;
            continue;
        }
        if (l < 0) continue;
        const int h = (int)(((uint32_t)l * 0x9E3779B1u) >> (32 - NF_LOG));
        int k = __hip_atomic_load(&key[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (k == EMPTY_KEY) {
            k = atomicCAS(&key[h], EMPTY_KEY, l);
            if (k == EMPTY_KEY) k = l;
        }
        if (k == l) atomicMin(&low[h], v);
        else if (first[l] > v) atomicMin(&first[l], v);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < (1 << NF_LOG); i += NF_NT) {
        const int l = key[i];
        if (l != EMPTY_KEY && first[l] > low[i]) atomicMin(&first[l], low[i]);
    }
}

// The whole compression of up to CH * 1024 labels by one workgroup: each wave
// holds CH chunks of 64 consecutive labels in registers, read at once.  The
// table in LDS holds the least vertex of every label, then the complement of
// its new id (negative, so a later test for "am I the least" stays false).
// Seven launches take 20-24 us whatever the labels, most of it their floors;
// one takes 6 us for 4,000 labels in many communities, 12 for 20,000, 17 for
// 28,000 and 24 for 36,000, the most its table in LDS holds.  Labels that fall
// into one community queue on its word: 7, 27, 37 and 48 us.  A build costs what
// it has registers for (4,096 labels in the builds for 4, 8, 12, 20, 28 and 36
// thousand: 5.8, 6.0, 6.4, 8.5, 10.6 and 14.7 us), so there are six.
constexpr int NA_CH = 36, NA_SOLO = NA_CH * 1024;
template <int CH>
__global__ __launch_bounds__(1024) void k_na_solo(int n, const int32_t *labels, int32_t *out, int32_t *num_labels) {
    constexpr int NW = 1024 / WAVE;
    __shared__ int first[CH * 1024];
    __shared__ int part[NW], bad;
    const int tid = threadIdx.x, w = tid / WAVE, lane = __lane_id();
    const int chunks = (n + 1023) / 1024;  // chunks of 64 per wave
    const int v0 = w * chunks * WAVE + lane;
    int l[CH];
#pragma unroll
    for (int c = 0; c < CH; c++) l[c] = c < chunks && v0 + c * WAVE < n ? labels[v0 + c * WAVE] : INT32_MIN;
    for (int i = tid; i < n; i += 1024) first[i] = INT32_MAX;
    if (tid == 0) bad = 0;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int v = v0 + c * WAVE;
        if (c >= chunks || v >= n) continue;
        if (l[c] < -1 || l[c] >= n) {
            bad = 1;
            out[v] = -1;  // out of contract: reported through k = -1
            l[c] = INT32_MIN;
        } else if (l[c] >= 0) {
            atomicMin(&first[l[c]], v);
        }
    }
    __syncthreads();
    int mine = 0;
#pragma unroll
    for (int c = 0; c < CH; c++)
        mine += __popcll(__ballot(l[c] == -1 || (l[c] >= 0 && first[l[c]] == v0 + c * WAVE)));
    if (lane == 0) part[w] = mine;
    __syncthreads();
    int id = 0, total = 0;
#pragma unroll
    for (int i = 0; i < NW; i++) {
        if (i < w) id += part[i];
        total += part[i];
    }
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int v = v0 + c * WAVE;
        const bool head = l[c] == -1 || (l[c] >= 0 && first[l[c]] == v);
        const uint64_t m = __ballot(head);
        const int rank = id + __popcll(m & ((1ULL << lane) - 1));
        id += __popcll(m);
        if (!head) continue;
        if (l[c] < 0) out[v] = rank;
        else first[l[c]] = ~rank;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CH; c++)
        if (l[c] >= 0) out[v0 + c * WAVE] = ~first[l[c]];
    if (tid == 0) *num_labels = bad ? -1 : total;
}

struct NaFlag {
    int n;
    const int32_t *labels, *first;
    __device__ int operator()(int64_t v) const {
        const int l = labels[v];
        if (l < -1 || l >= n) return 0;
        return (l < 0 || first[l] == (int)v) ? 1 : 0;
    }
};

struct NaStore {
    const int32_t *labels;
    int32_t *out, *newid;
    __device__ void operator()(int64_t v, int ex, int flag) const {
        if (!flag) return;
        const int l = labels[v];
        if (l < 0) out[v] = ex;
        else newid[l] = ex;
    }
};

// the new labels; *num_labels receives k
__global__ void k_na_relabel(int n, const int32_t *labels, const int32_t *newid, int32_t *out, const int32_t *total,
                             const int32_t *flags, int32_t *num_labels) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *num_labels = flags[0] ? -1 : *total;
    const int stride = gridDim.x * blockDim.x;
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride) {
        const int l = labels[v];
        if (l >= 0 && l < n) out[v] = newid[l];
        else if (l != -1) out[v] = -1;  // out of contract: reported through k = -1
    }
}

// rounds per scan tile: as few as leave at most NA_TILES tiles
inline int na_rounds(int64_t n) {
    int r = 1;
    while ((n + (int64_t)r * SCAN_THREADS - 1) / ((int64_t)r * SCAN_THREADS) > NA_TILES) r *= 2;
    return r;
}

// the device address of `scratch` on each device, taken once per device
std::mutex g_mu;
int32_t *g_ptr[64] = {nullptr};

int scratch_ptr(int32_t **out) {
    int dev = -1;
    PCD_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return fail(PCD_E_INVALID, "device index out of range");
    std::lock_guard<std::mutex> lk(g_mu);
    if (!g_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            (void)hipGetLastError();
            return fail(PCD_E_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        }
        g_ptr[dev] = (int32_t *)p;
    }
    *out = g_ptr[dev];
    return PCD_OK;
}

}  // namespace
}  // namespace pcd

using namespace pcd;

extern "C" int pcd_compress_labels_noalloc(int n, const int32_t *labels, int32_t *out_labels, int32_t *num_labels,
                                           void *stream) {
    if (n < 0) return fail(PCD_E_INVALID, "n must be >= 0");
    if (n > NA_MAX)
        return fail(PCD_E_INVALID, "n = " + std::to_string(n) + " exceeds the allocation-free maximum of " +
                                       std::to_string(NA_MAX) + " vertices");
    if (!num_labels || (n > 0 && (!labels || !out_labels)))
        return fail(PCD_E_INVALID, "null device pointer");
    if (n > 0 && labels == out_labels) return fail(PCD_E_INVALID, "labels and out_labels must not be the same array");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) {
        (void)hipGetLastError();
        return fail(PCD_E_NODEVICE, "no HIP device available");
    }
    hipStream_t s = (hipStream_t)stream;
    if (n <= NA_SOLO) {  // no shared table in memory
        const auto kernel = n <= 4096 ? k_na_solo<4>
                            : n <= 8192  ? k_na_solo<8>
                            : n <= 12288 ? k_na_solo<12>
                            : n <= 20480 ? k_na_solo<20>
                            : n <= 28672 ? k_na_solo<28>
                                         : k_na_solo<NA_CH>;
        hipLaunchKernelGGL(kernel, dim3(1), dim3(1024), 0, s, n, labels, out_labels, num_labels);
        PCD_HIP(hipGetLastError());
        return PCD_OK;
    }
    int32_t *base = nullptr;
    PCD_TRY(scratch_ptr(&base));
    int32_t *first = base + NA_FIRST, *newid = base + NA_NEWID, *parts = base + NA_PARTS, *flags = base + NA_FLAGS;
    const int grid = (int)std::min<int64_t>((n + 255) / 256, 2048);
    hipLaunchKernelGGL(k_na_clear, dim3(grid), dim3(256), 0, s, n, first, flags);
    hipLaunchKernelGGL(k_na_first, dim3(std::min((n + NF_NT * 4 - 1) / (NF_NT * 4), 1024)), dim3(NF_NT), 0, s, n, labels,
                       first, flags);
    const NaFlag load{n, labels, first};
    const NaStore store{labels, out_labels, newid};
    const int rounds = na_rounds(n);
    const int tiles = (int)((n + (int64_t)rounds * SCAN_THREADS - 1) / ((int64_t)rounds * SCAN_THREADS));
    hipLaunchKernelGGL(k_scan_tiles<NaFlag>, dim3(tiles), dim3(SCAN_THREADS), 0, s, (int64_t)n, load, parts, rounds);
    hipLaunchKernelGGL(k_scan_parts, dim3(1), dim3(SCAN_THREADS), 0, s, tiles, parts);
    hipLaunchKernelGGL((k_scan_apply<NaFlag, NaStore>), dim3(tiles), dim3(SCAN_THREADS), 0, s, (int64_t)n, load, store,
                       parts, rounds);
    hipLaunchKernelGGL(k_na_relabel, dim3(grid), dim3(256), 0, s, n, labels, newid, out_labels,
                       parts + tiles, flags, num_labels);
    PCD_HIP(hipGetLastError());
    return PCD_OK;
}
