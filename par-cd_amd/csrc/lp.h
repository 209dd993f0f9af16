// Device code of one propagation or merging row: candidates, label tables and
// the per-row kernels' bodies (G lanes, one wave or one workgroup per vertex).
#ifndef PARCD_LP_H
#define PARCD_LP_H

#include <type_traits>

#include "work.h"

namespace pcd {

struct Cand {
    double s;
    uint32_t key;
    int label;
};

__device__ inline Cand cand_none() { return Cand{-__builtin_inf(), 0xFFFFFFFFu, INT32_MAX}; }

__device__ inline bool cand_better(const Cand &a, const Cand &b) {
    if (a.s > b.s) return true;
    if (a.s < b.s) return false;
    if (a.key != b.key) return a.key < b.key;
    return a.label < b.label;
}

// x of lane ^ J, every lane of the wave active: a DPP quad permute for
// J = 1 and 2 (no LDS access), ds_swizzle's bit mode (and 0x1f, xor J,
// within 32 lanes; no address register) for J = 4..16, ds_bpermute for 32.
template <int J>
__device__ inline int xor_shfl(int x) {
    static_assert(J >= 1 && J <= 32 && (J & (J - 1)) == 0, "lane distance");
    if constexpr (J == 1) return __builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, false);       // quad_perm [1,0,3,2]
    else if constexpr (J == 2) return __builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, false);  // quad_perm [2,3,0,1]
    else if constexpr (J <= 16) return __builtin_amdgcn_ds_swizzle(x, 0x1F | (J << 10));
    else return __shfl_xor(x, J, WAVE);
}

// x of lane - 1 (DPP wave_shr:1, every lane active); lane 0's result is
// undefined
__device__ inline int prev_lane(int x) { return __builtin_amdgcn_mov_dpp(x, 0x138, 0xF, 0xF, false); }

template <int J>
__device__ inline Cand cand_xor(const Cand &c) {
    Cand o;
    const long long b = __double_as_longlong(c.s);
    const int lo = xor_shfl<J>((int)(uint32_t)b), hi = xor_shfl<J>((int)(b >> 32));
    o.s = __longlong_as_double((long long)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo));
    o.key = (uint32_t)xor_shfl<J>((int)c.key);
    o.label = xor_shfl<J>(c.label);
    return o;
}

// best candidate and largest own count over aligned groups of 2D lanes
template <int D>
__device__ inline void group_reduce_cand(Cand &c, int &own_cnt) {
    const Cand o = cand_xor<D>(c);
    if (cand_better(o, c)) c = o;
    own_cnt = max(own_cnt, xor_shfl<D>(own_cnt));
    if constexpr (D > 1) group_reduce_cand<D / 2>(c, own_cnt);
}

// bitonic sort of each aligned group of G lanes, ascending: one
// compare-exchange per step, the lane keeping the smaller or the larger of
// its value and its partner's (lane ^ J)
template <int G, int K = 2, int J = 1>
__device__ inline int group_sort(int x, int glane) {
    const bool take_min = ((glane & K) == 0) == ((glane & J) == 0);
    const int y = xor_shfl<J>(x);
    x = take_min ? min(x, y) : max(x, y);
    if constexpr (J > 1) return group_sort<G, K, J / 2>(x, glane);
    else if constexpr (K < G) return group_sort<G, 2 * K, K>(x, glane);
    else return x;
}

// partial result of one hub partition
struct HubPartial {
    Cand c;
    int own_cnt;
    int distinct;
};
static_assert(sizeof(HubPartial) <= HUB_PARTIAL_BYTES, "hub partial record size");

// Community record as the gains see it.  With aux: modularity reads
// int_volume + ext_volume (= aux + 0), CPM reads size (= aux).
__device__ inline CommStats comm_of(const LPArgs &a, int label, int aux) {
    if (a.use_aux) return CommStats{aux, aux, 0, 0};
    return a.stats[label];
}

// Kernel builds for the batch read the 16-byte community records (a batch
// keeps no per-community totals); an extra bit of the rule-kind mask.
constexpr unsigned RK_REC = 1u << 8;
constexpr unsigned RK_BATCH = RK_MOD | RK_CPM | RK_REC;

// Builds for the merging step (MergingRefinement::refine,
// refinement.cpp:185-288): a row is a community l, its entries are the
// labels of its members' neighbours (gathered into the row once per step),
// its own label is l, a candidate is another community not yet matched,
// scored by score_merge and accepted from 0 up, and the row's result is its
// best partner or -1.  They read the community records, whose pad word
// holds the community's "matched" flag during a merging step (one gather
// per candidate brings both).
constexpr unsigned RK_MERGE = 1u << 9;
constexpr unsigned RK_MERGE_REC = RK_MERGE | RK_REC;

template <unsigned KM>
__device__ inline bool lp_active(const LPArgs &a, int v) {
    if constexpr ((KM & RK_MERGE) != 0) {
        // a replayed merging pass whose loop has stopped (step -1) merges nothing
        if (a.step_ptr && *a.step_ptr < 0) return false;
        // refinement.cpp:224-226: matched communities, and those whose chosen
        // partner is still unmatched, sit the round out
        if (a.found[v]) return false;
        const int b = a.new_labels[v];
        return b == -1 || a.found[b] != 0;
    } else {
        return lp_selected(a, v);
    }
}

// label of a neighbour entry (merging rows hold labels already) and of the row
template <unsigned KM>
__device__ inline int entry_label(const LPArgs &a, int nb) {
    if constexpr ((KM & RK_MERGE) != 0) return nb;
    else return a.labels[nb];
}
template <unsigned KM>
__device__ inline int own_label(const LPArgs &a, int v) {
    if constexpr ((KM & RK_MERGE) != 0) return v;
    else return a.labels[v];
}

// Score of a candidate label other than the row's own, and whether it is a
// candidate at all: score_join > 0 (refinement.cpp:152-166), or for a
// merging row score_merge >= 0 (refinement.cpp:247-260: a zero score ties
// with "no partner" and is taken).  A merging caller has already dropped
// matched communities.
template <unsigned KM>
__device__ inline bool cand_score(const LPArgs &a, int deg, const CommStats &own_rec, const CommStats &rec, int cnt,
                                  double &sc) {
    if constexpr ((KM & RK_MERGE) != 0) {
        sc = score_merge<KM & RK_ALL>(a.rule, own_rec, rec, cnt);
        return sc >= 0.0;
    } else {
        sc = score_join<KM>(a.rule, deg, rec, cnt);
        return sc > 0;
    }
}

// merging row's result (refinement.cpp:262): the best partner, or -1
__device__ inline int merge_partner(const Cand &c) { return c.label != INT32_MAX ? c.label : -1; }

// Community record of `label` as the gains read it.  Builds for modularity
// or CPM alone read the 4-byte per-community total the step built (one
// random read into a 4x smaller array than the records); the others read
// the record.
template <unsigned KM>
__device__ inline CommStats comm_rec(const LPArgs &a, int label) {
    if constexpr ((KM & (RK_WCC | RK_COND | RK_REC)) == 0) {
        const int x = a.tot[label];
        return CommStats{x, x, 0, 0};
    } else {
        return a.stats[label];
    }
}

// refinement.cpp:169-179: best_score (0 if no join candidate beat 0) plus
// score_leave decides between moving, leaving to a new singleton, staying.
template <unsigned KM>
__device__ inline int lp_decide(const LPArgs &a, int deg, int own, int own_aux, int own_cnt, const Cand &best) {
    double leave = score_leave<KM>(a.rule, deg, comm_of(a, own, own_aux), own_cnt);
    double bs = best.label != INT32_MAX ? best.s : 0.0;
    bs += leave;
    if (bs > 0 && bs > leave) return best.label;
    if (leave > 0) return PCD_NEW_LABEL;
    return own;
}

template <unsigned KM>
__device__ inline int lp_decide_rec(const LPArgs &a, int deg, int own, const CommStats &own_rec, int own_cnt,
                                    const Cand &best) {
    double leave = score_leave<KM>(a.rule, deg, own_rec, own_cnt);
    double bs = best.label != INT32_MAX ? best.s : 0.0;
    bs += leave;
    if (bs > 0 && bs > leave) return best.label;
    if (leave > 0) return PCD_NEW_LABEL;
    return own;
}

template <unsigned KM>
__device__ inline int lp_decide_stats(const LPArgs &a, int deg, int own, int own_cnt, const Cand &best) {
    return lp_decide_rec<KM>(a, deg, own, comm_rec<KM>(a, own), own_cnt, best);
}

__device__ inline void count3(const LPArgs &a, long long act, long long ent, long long dist) {
    atomicAdd(&a.counters[0], (unsigned long long)act);
    atomicAdd(&a.counters[1], (unsigned long long)ent);
    atomicAdd(&a.counters[2], (unsigned long long)dist);
}

__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ------------------------------------------------------------- G lanes / vertex
template <int G, int CP, bool AUX, unsigned KM, class Src>
__device__ inline void lp_small(const Src &src, int wave_g, int nwaves, int *list) {
    const int lane = __lane_id(), glane = lane & (G - 1);
    const uint64_t lt = lane == 0 ? 0ULL : (~0ULL >> (64 - lane));
    const int per_wave = WAVE / G;
    const int nunits = src.units();
    for (int u = wave_g; u < nunits; u += nwaves) {
        LPArgs a;
        int q0, q1;
        if (!src.unit(u, a, q0, q1)) continue;
        // compaction of the active vertices among (at most CP) consecutive positions
        int p = q0 + lane;
        bool valid = lane < CP && p < q1;
        int v = valid ? vertex_at(a, p) : 0;
        bool act = valid && lp_active<KM>(a, v);
        uint64_t am = __ballot(act);
        int nact = __popcll(am);
        if (act) list[__popcll(am & lt)] = v;
        wave_sync();
        // the row, own label and own community record of every active vertex
        // of the unit, one lane each, loaded together (nact <= CP <= 64);
        // each group takes its vertices' values by shuffle
        int pu = 0, pstart = 0, pdeg = 0, pown = 0, paux = 0;
        CommStats pst{0, 0, 0, 0};
        uint64_t ptb = 0;  // the vertex's tie-key base (one hash per vertex, not per pass)
        if (lane < nact) {
            pu = list[lane];
            pstart = a.indices[pu];
            pdeg = a.indices[pu + 1] - pstart;
            if constexpr (AUX) {
                const int2 o = a.lv[pu];
                pown = o.x;
                paux = o.y;
            } else {
                pown = own_label<KM>(a, pu);
                pst = comm_rec<KM>(a, pown);
            }
            if (a.tie != PCD_TIE_LOWEST) ptb = tie_base(a.seed, step_of(a), pu);
        }
        for (int gb = 0; gb < nact; gb += per_wave) {
            int gi = gb + lane / G;
            bool has = gi < nact;
            const int sl = has ? gi : 0;
            int u = __shfl(pu, sl, WAVE), start = __shfl(pstart, sl, WAVE), deg = __shfl(pdeg, sl, WAVE);
            const uint64_t tb = ((uint64_t)(uint32_t)__shfl((int)(ptb >> 32), sl, WAVE) << 32) |
                                (uint32_t)__shfl((int)(uint32_t)ptb, sl, WAVE);
            int2 own = make_int2(__shfl(pown, sl, WAVE), __shfl(paux, sl, WAVE));
            const CommStats own_rec{__shfl(pst.size, sl, WAVE), __shfl(pst.int_vol, sl, WAVE),
                                    __shfl(pst.ext_vol, sl, WAVE), 0};
            if (!has) {
                u = start = deg = 0;
                own = make_int2(0, 0);
            }
            int2 r = make_int2(INT32_MAX, 0);
            if (has && glane < deg) {
                int nb = a.adj[start + glane];
                r = AUX ? a.lv[nb] : make_int2(entry_label<KM>(a, nb), 0);
            }
            int x = r.x, xa = r.y;
            if constexpr (AUX) {
#pragma unroll
                for (int k = 2; k <= G; k <<= 1) {
#pragma unroll
                    for (int j = k >> 1; j > 0; j >>= 1) {
                        const bool take_min = ((glane & k) == 0) == ((glane & j) == 0);
                        const int y = __shfl_xor(x, j, WAVE), ya = __shfl_xor(xa, j, WAVE);
                        const bool other = take_min ? (y < x) : (y > x);
                        x = other ? y : x;
                        xa = other ? ya : xa;
                    }
                }
            } else {
                x = group_sort<G>(x, glane);
            }
            const int prev = prev_lane(x);  // read only where glane > 0
            bool head = x != INT32_MAX && (glane == 0 || x != prev);
            uint64_t heads = __ballot(head);
            Cand c = cand_none();
            int own_cnt = 0;
            if (head) {
                uint64_t above = lane == 63 ? 0ULL : (heads >> (lane + 1));
                int nxt = above ? lane + 1 + __builtin_ctzll(above) : WAVE;
                int gend = (lane & ~(G - 1)) + deg;
                int cnt = min(nxt, gend) - lane;
                if (x == own.x) {
                    own_cnt = cnt;
                } else {
                    const CommStats xr = AUX ? CommStats{xa, xa, 0, 0} : comm_rec<KM>(a, x);
                    if ((KM & RK_MERGE) == 0 || !xr.pad) {  // merging: matched communities are no candidates
                        double sc;
                        if (cand_score<KM>(a, deg, own_rec, xr, cnt, sc)) c = Cand{sc, tie_key(a.tie, tb, x), x};
                    }
                }
            }
            group_reduce_cand<G / 2>(c, own_cnt);
            if (has && glane == 0) {
                if constexpr ((KM & RK_MERGE) != 0) a.new_labels[u] = merge_partner(c);
                else a.new_labels[u] = AUX ? lp_decide<KM>(a, deg, own.x, own.y, own_cnt, c)
                                           : lp_decide_rec<KM>(a, deg, own.x, own_rec, own_cnt, c);
            }
            if (a.counters) {
                // every lane votes: a wave holds up to 64 / G active vertices
                const int act = __popcll(__ballot(has && glane == 0));
                int ent = wave_sum((has && glane < deg) ? 1 : 0);
                if (lane == 0) count3(a, act, ent, __popcll(heads));
            }
        }
        wave_sync();
    }
}

// ------------------------------------------------------------- LDS hash table
// Hub partition tables: T slots (any multiple of 64), linear probing from
// (hash * T) >> 32.
__device__ inline int tslot(int key, int T) {
    return (int)(((uint64_t)((uint32_t)key * 0x9E3779B1u) * (uint32_t)T) >> 32);
}

// Listed-slot scans read SB slots at a time so that their community-record
// gathers overlap.
constexpr int SB = 4;

__device__ inline void wave_reduce_cand(Cand &c, int &own_cnt) { group_reduce_cand<WAVE / 2>(c, own_cnt); }

template <int NT>
__device__ inline void block_reduce_cand(Cand &c, int &own_cnt, int &distinct, Cand *s_c, int *s_i) {
    const int lane = __lane_id(), w = threadIdx.x / WAVE;
    wave_reduce_cand(c, own_cnt);
    distinct = wave_sum(distinct);
    if (lane == 0) { s_c[w] = c; s_i[w] = own_cnt; s_i[NT / WAVE + w] = distinct; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < NT / WAVE; i++) {
            if (cand_better(s_c[i], c)) c = s_c[i];
            own_cnt = max(own_cnt, s_i[i]);
            distinct += s_i[NT / WAVE + i];
        }
    }
    __syncthreads();
}

__device__ inline int round64(int x) { return (x + 63) & ~63; }

// ------------------------------------------------------------- label tables
// Tables of the per-vertex kernels hold nextpow2(2 deg) slots, more than the
// row's distinct labels, so probing always ends at a free or matching slot.
__device__ inline uint32_t pslot(int key, int log_t) { return ((uint32_t)key * 0x9E3779B1u) >> (32 - log_t); }

// Counts of a table: 32-bit, or 16-bit where a row's degree bounds them
// below 2^16.  A 16-bit count is incremented by a 32-bit LDS atomic on the
// word holding it (the other half cannot carry into it); it is read and
// cleared with 16-bit accesses.
__device__ inline void count_add(int *cnts, uint32_t h) { atomicAdd(&cnts[h], 1); }
__device__ inline void count_add(uint16_t *cnts, uint32_t h) {
    atomicAdd((unsigned *)(cnts + (h & ~1u)), 1u << ((h & 1u) * 16));
}

// Inserts `key` (with AUX its aux, stored by the lane that claims the slot)
// with count 1; returns true when this lane claimed a free slot, whose
// index lands in `slot`.
template <bool AUX, class CT = int>
__device__ inline bool pinsert(int *keys, CT *cnts, int *auxs, int mask, int log_t, int key, int aux, int &slot) {
    uint32_t h = pslot(key, log_t);
    while (true) {
        int old = atomicCAS(&keys[h], EMPTY_KEY, key);
        if (AUX && old == EMPTY_KEY) auxs[h] = aux;
        if (old == EMPTY_KEY || old == key) {
            count_add(cnts, h);
            slot = (int)h;
            return old == EMPTY_KEY;
        }
        h = (h + 1) & mask;
    }
}

// Appends the slots this wave's lanes claimed to the table's slot list
// (one LDS atomic per wave).  Called by every lane of the wave.
__device__ inline void occ_append(bool claimed, int slot, uint16_t *occ, int *nocc) {
    const uint64_t cm = __ballot(claimed);
    if (!cm) return;
    const int lane = __lane_id();
    const int leader = __builtin_ctzll(cm);
    int base = 0;
    if (lane == leader) base = atomicAdd(nocc, __popcll(cm));
    base = __builtin_amdgcn_readlane(base, leader);
    if (claimed) occ[base + __popcll(cm & ((1ULL << lane) - 1))] = (uint16_t)slot;
}

// Gathers the labels (with AUX the {label, aux} records: one 8-byte gather
// brings what the gains read, and aux lands in the table) of row entries
// base + lo + e * stride, PF at a time (independent loads in flight), and
// inserts them; claimed slots go to the slot list.  A merging row (its
// entries are labels) leaves out its own label, which is never a
// candidate.  The loop bounds are the same for every lane of the workgroup.
template <int PF, unsigned KM, bool AUX = false, class CT = int>
__device__ inline void insert_labels(const LPArgs &a, int *keys, CT *cnts, int *auxs, uint16_t *occ, int *nocc,
                                     int mask, int log_t, int start, int deg, int lo, int stride, int own) {
    constexpr bool MERGE = (KM & RK_MERGE) != 0;
    for (int base = 0; base < deg; base += PF * stride) {
        int nb[PF];
#pragma unroll
        for (int e = 0; e < PF; e++) {
            int j = base + lo + e * stride;
            nb[e] = j < deg ? a.adj[start + j] : -1;
        }
        int2 rec[PF];
#pragma unroll
        for (int e = 0; e < PF; e++)
            rec[e] = nb[e] < 0 ? make_int2(EMPTY_KEY, 0)
                               : (AUX ? a.lv[nb[e]] : make_int2(entry_label<KM>(a, nb[e]), 0));
#pragma unroll
        for (int e = 0; e < PF; e++) {
            bool claimed = false;
            int slot = 0;
            if (rec[e].x != EMPTY_KEY && (!MERGE || rec[e].x != own))
                claimed = pinsert<AUX, CT>(keys, cnts, auxs, mask, log_t, rec[e].x, rec[e].y, slot);
            occ_append(claimed, slot, occ, nocc);
        }
    }
}

// Scans the D listed slots [lo, D) with stride `stride` for candidates, SB
// at a time so that their community-record gathers overlap, and clears each
// slot it read (the table is empty again for the next row).
template <bool AUX, unsigned KM, class CT = int>
__device__ inline void scan_listed(const LPArgs &a, int *keys, CT *cnts, const int *auxs, const uint16_t *occ, int D,
                                   int lo, int stride, int deg, int own, uint64_t tb, Cand &c, int &own_cnt) {
    constexpr bool MERGE = (KM & RK_MERGE) != 0;
    CommStats orec{0, 0, 0, 0};
    if constexpr (MERGE) orec = a.stats[own];
    for (int i0 = lo; i0 < D; i0 += SB * stride) {
        int key[SB], cnt[SB];
        CommStats st[SB];
#pragma unroll
        for (int e = 0; e < SB; e++) {
            const int i = i0 + e * stride;
            key[e] = EMPTY_KEY;
            cnt[e] = 0;
            if (i < D) {
                const int h = occ[i];
                key[e] = keys[h];
                cnt[e] = cnts[h];
                if (AUX) {
                    const int x = auxs[h];
                    st[e] = CommStats{x, x, 0, 0};
                }
                keys[h] = EMPTY_KEY;
                cnts[h] = 0;
            }
        }
        if (!AUX) {
#pragma unroll
            for (int e = 0; e < SB; e++)
                if (key[e] != EMPTY_KEY && key[e] != own) st[e] = comm_rec<KM>(a, key[e]);
        }
#pragma unroll
        for (int e = 0; e < SB; e++) {
            if (key[e] == EMPTY_KEY) continue;
            if (MERGE && key[e] != own && st[e].pad) continue;  // matched: no candidate
            if (key[e] == own) {
                own_cnt = cnt[e];
            } else {
                double sc;
                if (cand_score<KM>(a, deg, orec, st[e], cnt[e], sc)) {
                    Cand o{sc, tie_key(a.tie, tb, key[e]), key[e]};
                    if (cand_better(o, c)) c = o;
                }
            }
        }
    }
}

__device__ inline int ceil_log2(int x) { return x <= 1 ? 0 : 32 - __clz(x - 1); }

// ------------------------------------------------------------- wave / vertex
// The table starts empty and each row's scan clears the slots it used.
// One wave per vertex over the units of src, with this wave's LDS table
// (TW slots of keys, counts and aux, a slot list of TW / 2 entries).
template <int TW, unsigned KM, class Src, bool AUX, int PF, class CT = int>
__device__ inline void lp_wave(const Src &src, int wave_g, int nwaves, int *keys, CT *cnts, int *auxs, uint16_t *occ,
                               int *nocc) {
    const int lane = __lane_id();
    for (int i = lane; i < TW; i += WAVE) {
        keys[i] = EMPTY_KEY;
        cnts[i] = 0;
    }
    if (lane == 0) *nocc = 0;
    wave_sync();
    const int nunits = src.units();
    for (int u = wave_g; u < nunits; u += nwaves) {
      LPArgs a;
      int q0, q1;
      if (!src.unit(u, a, q0, q1)) continue;
      for (int p = q0; p < q1; p++) {
        int v = vertex_at(a, p);
        if (!lp_active<KM>(a, v)) continue;
        int start = a.indices[v], deg = a.indices[v + 1] - start;
        int2 ownr = AUX ? a.lv[v] : make_int2(own_label<KM>(a, v), 0);
        int own = ownr.x;
        int log_t = max(6, ceil_log2(2 * deg));
        insert_labels<PF, KM, AUX, CT>(a, keys, cnts, auxs, occ, nocc, (1 << log_t) - 1, log_t, start, deg, lane, WAVE,
                                       own);
        wave_sync();
        const int D = *nocc;
        uint64_t tb = a.tie == PCD_TIE_LOWEST ? 0 : tie_base(a.seed, step_of(a), v);
        Cand c = cand_none();
        int own_cnt = 0;
        scan_listed<AUX, KM, CT>(a, keys, cnts, auxs, occ, D, lane, WAVE, deg, own, tb, c, own_cnt);
        wave_reduce_cand(c, own_cnt);
        if (lane == 0) {
            if constexpr ((KM & RK_MERGE) != 0) a.new_labels[v] = merge_partner(c);
            else a.new_labels[v] = AUX ? lp_decide<KM>(a, deg, own, ownr.y, own_cnt, c)
                                       : lp_decide_stats<KM>(a, deg, own, own_cnt, c);
            if (a.counters) count3(a, 1, deg, D);
            *nocc = 0;
        }
        wave_sync();
      }
    }
}

// ------------------------------------------------------------- workgroup / vertex
// LDS of a workgroup that counts one row at a time in a table of
// nextpow2(2 deg) slots, at most TB.
// CT = uint16_t needs rows below 2^16 entries (the table's counts).
template <int NT, int TB, bool AUX = false, class CT = int>
struct BlockTable {
    int keys[TB];
    __align__(16) CT cnts[TB];
    int auxs[AUX ? TB : 1];
    uint16_t occ[TB / 2];
    int nocc;
    Cand c[NT / WAVE];
    int i[2 * NT / WAVE];
};

template <int NT, int TB, unsigned KM, class Src, bool AUX, int PF, class CT>
__device__ inline void lp_block(const Src &src, int wg, int nwg, BlockTable<NT, TB, AUX, CT> &t) {
    for (int i = threadIdx.x; i < TB; i += NT) {
        t.keys[i] = EMPTY_KEY;
        t.cnts[i] = 0;
    }
    if (threadIdx.x == 0) t.nocc = 0;
    __syncthreads();
    const int nunits = src.units();
    for (int u = wg; u < nunits; u += nwg) {
      LPArgs a;
      int q0, q1;
      if (!src.unit(u, a, q0, q1)) continue;
      for (int p = q0; p < q1; p++) {
        int v = vertex_at(a, p);
        if (!lp_active<KM>(a, v)) continue;
        int start = a.indices[v], deg = a.indices[v + 1] - start;
        int2 ownr = AUX ? a.lv[v] : make_int2(own_label<KM>(a, v), 0);
        int own = ownr.x;
        int log_t = max(6, ceil_log2(2 * deg));
        insert_labels<PF, KM, AUX, CT>(a, t.keys, t.cnts, t.auxs, t.occ, &t.nocc, (1 << log_t) - 1, log_t, start, deg,
                                      threadIdx.x, NT, own);
        __syncthreads();
        const int D = t.nocc;
        uint64_t tb = a.tie == PCD_TIE_LOWEST ? 0 : tie_base(a.seed, step_of(a), v);
        Cand c = cand_none();
        int own_cnt = 0, distinct = 0;
        scan_listed<AUX, KM, CT>(a, t.keys, t.cnts, t.auxs, t.occ, D, threadIdx.x, NT, deg, own, tb, c, own_cnt);
        block_reduce_cand<NT>(c, own_cnt, distinct, t.c, t.i);
        if (threadIdx.x == 0) {
            if constexpr ((KM & RK_MERGE) != 0) a.new_labels[v] = merge_partner(c);
            else a.new_labels[v] = AUX ? lp_decide<KM>(a, deg, own, ownr.y, own_cnt, c)
                                       : lp_decide_stats<KM>(a, deg, own, own_cnt, c);
            if (a.counters) count3(a, 1, deg, D);
            t.nocc = 0;
        }
        __syncthreads();
      }
    }
}

}  // namespace pcd

#endif
