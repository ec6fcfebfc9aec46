// ft_query.hip -- gfx950 neighbour-query kernels over a built TreeSoA:
//   self_knn_query / self_knn_query_subset / knn_query (src/hlbvh.hpp:1057-1983)
//   range_query (src/hlbvh.hpp:2006-2136) and a CSR range query.
//
// Two traversal families:
//  * per-lane DFS (one query per lane, 64-entry stack in LDS): the reference's
//    algorithm -- pop, node d2, prune, leaf push or two child d2 with the
//    farther child pushed first while sp < 62 (src/hlbvh.hpp:1545-1628).  Heap
//    tiers: a canonical register top-k (k <= 32) and an LDS max-heap per lane
//    (any k), the latter also in the reference's exact heap mechanics.
//  * packet traversal (one wavefront of 64 SFC-adjacent queries shares one
//    stack; node boxes are wave-uniform loads; small subtrees are scanned as
//    contiguous leaf buckets).  Canonical results only.
//
// Canonical results: the k smallest (d2, returned index) pairs in ascending
// order -- a unique answer, independent of traversal order.
#include "ft_traverse.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace ft {

int scratch_ensure_public(Scratch &S, size_t n);
int radix_sort_u64(hipStream_t s, Scratch &S, const uint64_t *keys_in, size_t n,
                   uint64_t *sorted_out, int key_bits);


// ===========================================================================
// Query positions.  A "slot" is a position in the launch's query order; the
// query it holds is order[slot] (external queries sorted along the curve) or
// the slot itself.  Results are written at the query's own row.  A direct pass
// appends the slots it leaves unanswered to a list that a listed pass takes.
// ===========================================================================
struct QueryMap {
    const uint32_t *order;  // slot -> query (null: identity)
    int32_t *list;          // direct passes: slots left to the listed pass, appended;
                            // LISTED: the slots to run
    uint32_t *count;        // [0] list entries, [1] queries of the packets left whole
                            // (where the caller counts)
    int32_t *packets;       // direct passes of cut keys: per packet, 1 if left whole
};

// Appends the slots of the lanes in `left` (a wave mask), one atomic per wave.
// Called by whole waves.
__device__ inline void append_slots(const QueryMap &qm, uint64_t left, int slot) {
    if (!left) return;
    const int lane = threadIdx.x & 63;
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(&qm.count[0], (uint32_t)__popcll(left));
    base = (uint32_t)uni((int)base);
    if ((left >> lane) & 1)
        qm.list[base + __builtin_amdgcn_mbcnt_hi((uint32_t)(left >> 32),
                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)left, 0u))] = slot;
}

// Leaves packet blk, whose queries are the lanes in `act`, to the exact pass.  A
// flag per packet, not a list: appending 15,600 packets of a lattice took 300 us
// of atomics on one word, and a list loses the packets' order along the curve.
__device__ inline void leave_packet(const QueryMap &qm, int blk, uint64_t act, bool counting) {
    if ((threadIdx.x & 63) != 0) return;
    qm.packets[blk] = 1;
    if (counting) atomicAdd(&qm.count[1], (uint32_t)__popcll(act));
}

__device__ inline int slot_query(const QueryMap &qm, int slot) {
    return qm.order ? (int)qm.order[slot] : slot;
}

// ===========================================================================
// Per-lane DFS with the canonical register top-k (k <= M <= 32): the
// reference's grouped self-kNN / knn_query_small_k walk on wave64 lanes, with
// the reference's 64-entry stack.  A query whose walk would need more is left
// to the listed pass.
// ===========================================================================
template <typename T, int M, bool GROUPED, int MK>
__global__ __launch_bounds__(LANE_BLOCK) void lane_knn_reg_kernel(
    DTree<T> t, QSrc<T> qs, int nq, int k, int excl, QueryMap qm, uint64_t *__restrict__ res,
    typename CoordTraits<T>::D *__restrict__ dists, uint64_t *__restrict__ stats) {
    using D = typename CoordTraits<T>::D;
    __shared__ int32_t stk[STACK_DEPTH * LANE_BLOCK];
    const int lane = threadIdx.x;
    uint64_t visits = 0, inserts = 0;
    const int slot = xcd_block() * LANE_BLOCK + lane;
    const bool active = slot < nq;
    const int q = active ? slot_query(qm, slot) : 0;
    T px = T(0), py = T(0), pz = T(0);
    int self = -1;
    if (active) load_query(t, qs, q, px, py, pz, self);
    if (!excl) self = -1;
    TopK<D, M> h;
    h.init(k, dist_max<D>());
    const bool ovf = lane_reg_walk<T, M, GROUPED, STACK_DEPTH, MK>(
        t, active, px, py, pz, self, h, stk, LANE_BLOCK, lane, visits, inserts);
    if (active && !ovf) h.store(k, res, dists, (size_t)q);
    append_slots(qm, __ballot(active && ovf), slot);
    wave_add_stats(stats, 0, visits);
    wave_add_stats(stats, 4, inserts);
}

// Per-lane DFS with an LDS heap row per lane (LocalMaxHeap, src/maxheap.hpp:340-478):
// REF = the reference's mechanics (ties as the reference picks them, 64-entry
// stack with its silent drop), else canonical (direct passes flag overflowing
// walks; LISTED re-runs use 128 entries).
template <typename T, bool REF, bool GROUPED, bool LISTED, int MK>
__global__ __launch_bounds__(LANE_BLOCK) void lane_knn_lds_kernel(
    DTree<T> t, QSrc<T> qs, int nq, int k, int excl, int lanes, QueryMap qm,
    uint64_t *__restrict__ res, typename CoordTraits<T>::D *__restrict__ dists,
    uint64_t *__restrict__ stats) {
    using D = typename CoordTraits<T>::D;
    constexpr int DEPTH = (LISTED && !REF) ? LANE_STACK_CANON : STACK_DEPTH;
    extern __shared__ __align__(16) unsigned char lds[];
    D *hd = (D *)lds;                                   // [k][lanes]
    int32_t *hi = (int32_t *)(hd + (size_t)k * lanes);  // [k][lanes]
    int32_t *stk = hi + (size_t)k * lanes;              // [DEPTH][lanes]
    const int lane = threadIdx.x;
    const bool lane_ok = lane < lanes;
    const int nlist = LISTED ? (int)qm.count[0] : nq;
    uint64_t visits = 0, drops = 0, inserts = 0;
    for (int base = (LISTED ? (int)blockIdx.x : xcd_block()) * lanes; base < nlist;
         base += (LISTED ? gridDim.x * lanes : nlist)) {
        const int pos = base + lane;
        const bool active = lane_ok && pos < nlist;
        const int slot = active ? (LISTED ? qm.list[pos] : pos) : 0;
        const int q = active ? slot_query(qm, slot) : 0;
        T px = T(0), py = T(0), pz = T(0);
        int self = -1;
        if (active) load_query(t, qs, q, px, py, pz, self);
        if (!excl) self = -1;
        LdsHeap<D, REF> h{hd, hi, lanes, lane, 0};
        const bool ovf = lane_heap_walk<T, REF, GROUPED, DEPTH, MK>(
            t, k, active, px, py, pz, self, h, stk, lanes, lane, visits, drops, inserts);
        const bool left = active && !REF && !LISTED && ovf;
        if (active) {
            if (!left) {
                h.sort();
                const size_t o = (size_t)q * k;
                for (int s = 0; s < k; ++s) {
                    const bool ok = s < h.count && h.ii(s) >= 0;
                    res[o + s] = ok ? (uint64_t)(uint32_t)h.ii(s) : ~0ull;
                    dists[o + s] = ok ? h.dd(s) : missing_dist<D>();
                }
            }
        }
        if constexpr (!REF && !LISTED) append_slots(qm, __ballot(left), slot);
        if (!LISTED) break;
    }
    wave_add_stats(stats, 0, visits);
    wave_add_stats(stats, 2, drops);
    wave_add_stats(stats, 4, inserts);
}

// ===========================================================================
// knn_query k > 32 in the reference's mechanics: one workgroup per query,
// lane 0 walks the stack, every leaf is merged through a 32-entry stage and a
// full bitonic network over the sorted list (SortedMergeHeap and
// local_bitonic_sort, src/maxheap.hpp:193-324; knn_query_large_k,
// src/hlbvh.hpp:1232-1387).  The network is data-oblivious, so running its
// compare-exchange stages across 64 lanes gives the reference's tie order.
// ===========================================================================
template <typename D>
__device__ inline void lds_bitonic(D *d, int32_t *ix, int n) {
    for (int kk = 2; kk <= n; kk <<= 1) {
        for (int j = kk >> 1; j > 0; j >>= 1) {
            for (int i = threadIdx.x; i < n; i += blockDim.x) {
                const int l = i ^ j;
                const bool asc = (i & kk) == 0;
                if (l > i && l < n) {
                    if ((d[i] > d[l]) == asc) {
                        D td = d[i]; d[i] = d[l]; d[l] = td;
                        int32_t ti = ix[i]; ix[i] = ix[l]; ix[l] = ti;
                    }
                }
            }
            __syncthreads();
        }
    }
}

template <typename T>
__global__ __launch_bounds__(64) void merge_knn_kernel(DTree<T> t, QSrc<T> qs, int nq, int k,
                                                       int cap, uint64_t *__restrict__ res,
                                                       typename CoordTraits<T>::D *__restrict__ dists,
                                                       uint64_t *__restrict__ stats) {
    using D = typename CoordTraits<T>::D;
    extern __shared__ __align__(16) unsigned char lds[];
    D *sd = (D *)lds;                                  // [cap]
    int32_t *si = (int32_t *)(sd + cap);               // [cap]
    D *gd = (D *)(si + cap + (cap & 1));               // [32] stage
    int32_t *gi = (int32_t *)(gd + 32);                // [32]
    int32_t *stk = gi + 32;                            // [64]
    __shared__ int s_count, s_sp, s_node;
    const int q = blockIdx.x;
    const int n = t.n;
    T px, py, pz;
    int self;
    load_query(t, qs, q, px, py, pz, self);
    for (int i = threadIdx.x; i < cap; i += blockDim.x) {
        sd[i] = dist_max<D>();
        si[i] = -1;
    }
    if (threadIdx.x == 0) {
        s_count = 0;
        s_sp = 1;
        stk[0] = 0;
    }
    __syncthreads();
    uint64_t visits = 0, drops = 0;
    while (true) {
        if (threadIdx.x == 0) s_node = s_sp > 0 ? stk[--s_sp] : -1;
        __syncthreads();
        const int node = s_node;
        __syncthreads();
        if (node < 0) break;
        ++visits;
        const D d2 = node_d2(t, px, py, pz, node);
        if (s_count >= k && d2 >= sd[k - 1]) continue;  // should_prune
        if (node >= n - 1 || n == 1) {
            // merge_batch: lane 0's candidate plus 31 empty entries
            if (threadIdx.x < 32) {
                const bool mine = threadIdx.x == 0;
                gd[threadIdx.x] = mine ? d2 : dist_max<D>();
                gi[threadIdx.x] = mine ? ((n == 1) ? 0 : ret_index(t, node)) : -1;
            }
            __syncthreads();
            lds_bitonic(gd, gi, 32);
            const int cnt = s_count;
            if (threadIdx.x < 32) {
                const int dst = cnt + threadIdx.x;
                if (dst < cap) {
                    sd[dst] = gd[threadIdx.x];
                    si[dst] = gi[threadIdx.x];
                }
            }
            __syncthreads();
            const int nc = min(cnt + 32, cap);
            int p2 = 1;
            while (p2 < nc) p2 <<= 1;
            for (int i = nc + threadIdx.x; i < p2 && i < cap; i += blockDim.x) {
                sd[i] = dist_max<D>();
                si[i] = -1;
            }
            __syncthreads();
            lds_bitonic(sd, si, p2);
            if (threadIdx.x == 0) s_count = min(min(nc, cap), k);
            __syncthreads();
        } else {
            if (threadIdx.x == 0) {
                const int l = t.left[node], r = t.right[node];
                const D ld = node_d2(t, px, py, pz, l);
                const D rd = node_d2(t, px, py, pz, r);
                if (s_sp < STACK_DEPTH - 2) {
                    if (ld <= rd) {
                        stk[s_sp++] = r;
                        stk[s_sp++] = l;
                    } else {
                        stk[s_sp++] = l;
                        stk[s_sp++] = r;
                    }
                } else {
                    ++drops;
                }
            }
            __syncthreads();
        }
    }
    const size_t o = (size_t)q * k;
    for (int i = threadIdx.x; i < k; i += blockDim.x) {
        const bool ok = si[i] >= 0;
        res[o + i] = ok ? (uint64_t)(uint32_t)si[i] : ~0ull;
        dists[o + i] = ok ? sd[i] : missing_dist<D>();
    }
    if (stats && threadIdx.x == 0) {
        atomicAdd((unsigned long long *)&stats[0], (unsigned long long)visits);
        if (drops) atomicAdd((unsigned long long *)&stats[2], (unsigned long long)drops);
    }
}


// ===========================================================================
// Packet traversal: a wavefront of 64 queries (consecutive slots) shares one
// DFS (packet_walk).  Results are canonical.
// SEEDED: each lane's k-th distance starts at its seed bound; a lane that ends
// with fewer than k neighbours inside the seed leaves its slot for an exact
// re-run.  PACKED: 64-bit (d2, index) keys; queries the packed form cannot
// order exactly are left too, and so are all queries of a packet whose walk
// passes its budget.  The listed pass (launch_listed) answers the slots left,
// unseeded and lexicographic, so exact.
// ===========================================================================
struct PacketArgs {
    int nq, k, excl, bucket, ibits;
    int width;   // queries per packet (16, 32 or 64): lanes at or above it idle
    int full;    // passes of 32: a row with a slot left empty goes to the listed pass
    uint32_t stop;  // leaves a packet may scan before its queries are handed over
    int window;  // self queries over all leaves: leaves pre-scanned on each side
    uint64_t *stats;
};

// MULTI (register tier, packed keys, k > M): ceil(k / M) passes, a separate
// instantiation so that the single-pass kernels keep their register budget.
// ===========================================================================
// Wave-per-query canonical tier (FT_ALGO_WAVE): one wavefront per query, its
// sorted list of C = 64 S entries spread over the lanes and candidates merged
// 64 leaves at a time by cross-lane bitonic networks (WaveList, wave_walk) --
// the canonical counterpart of knn_query_large_k's SortedMergeHeap
// (src/hlbvh.hpp:1232-1387, src/maxheap.hpp:226-324).  Exact in one walk for
// k up to 1024.  Four queries per 256-thread block; self and subset queries
// anchor their first leaves at their own rank, external ones at the leaf a
// greedy descent reaches.
//
// LISTED: the slots that a direct pass left (qm.list, qm.count[0] of them);
// the waves take list entries in turn.
// ===========================================================================
template <typename T, int S, int MK, bool LISTED = false>
__global__ __launch_bounds__(256) void wave_knn_kernel(DTree<T> t, QSrc<T> qs, int nq, int k,
                                                       int excl, uint64_t cap, QueryMap qm,
                                                       uint64_t *__restrict__ res,
                                                       typename CoordTraits<T>::D *__restrict__ dists,
                                                       uint64_t *__restrict__ stats) {
    __shared__ WaveBuf wbuf[4];
    const int lane = threadIdx.x & 63;
    const int wave = uni(xcd_block() * 4 + (int)(threadIdx.x >> 6));
    WaveCounters c;
    auto answer = [&](int slot) {
        const int q = uni(slot_query(qm, slot));
        T px = T(0), py = T(0), pz = T(0);
        int rank = -1;
        load_query(t, qs, q, px, py, pz, rank);
        const int self = excl ? rank : -1;
        const int anchor = rank >= 0 ? rank : descend_rank_v<T, MK>(t, px, py, pz);
        WaveList<S> L;
        // (integer distances and k above 128 have no cap: constant there)
        const uint64_t top = CoordTraits<T>::fp && S <= 2 ? cap : ~0ull;
        L.init(k, top);
        wave_walk<T, S, MK>(t, px, py, pz, self, anchor, L, c, &wbuf[threadIdx.x >> 6], top);
        L.store(k, res, dists, (size_t)q, lane);
    };
    if constexpr (LISTED) {
        const int cnt = (int)qm.count[0];
        for (int e = wave; e < cnt; e += (int)gridDim.x * 4) answer(uni(qm.list[e]));
    } else if (wave < nq) {
        answer(wave);
    }
    if (stats) {  // one atomic per block and counter: a wave per query would contend
        __shared__ unsigned long long s_st[3];
        if (threadIdx.x < 3) s_st[threadIdx.x] = 0;
        __syncthreads();
        if (lane == 0) {
            atomicAdd(&s_st[0], (unsigned long long)c.nodes);
            atomicAdd(&s_st[1], (unsigned long long)c.leaves);
            atomicAdd(&s_st[2], (unsigned long long)c.inserts);
        }
        __syncthreads();
        if (threadIdx.x < 3 && s_st[threadIdx.x])
            atomicAdd((unsigned long long *)&stats[threadIdx.x == 2 ? 4 : threadIdx.x],
                      s_st[threadIdx.x]);
    }
}

// Packed-key packets: at least 4 waves per SIMD (128 VGPRs), 11 % faster than
// 3 at k = 32.  With the walk's counters in 32 bits the k = 32 kernel spills
// nothing (72 bytes a lane before: 10M clustered points 16.9 -> 16.7 ms).  The
// passes of 32 spill a little (integers up to 52 bytes, doubles up to 80) and
// are faster so than at 3 waves (k = 64 subset of 20M doubles 30.8 against 35.5
// ms).  Exact pairs of doubles run 3 waves (k = 32: 172 registers, two waves,
// without the bound: a rounded lattice of 1M 4.2 against 3.5 ms).
//
// CUT keys (double coordinates, TopKFp): a packet whose queries have many
// distances that agree above the cut -- rounded grids -- is left whole to the
// LISTED instantiation, which takes the packets flagged in qm.packets and keeps
// exact (d, index) pairs.  It is found out by its fill (equal neighbours among
// the k curve neighbours of a quarter of the lanes), by its first run of leaves
// where there is no fill, or at the end (a quarter of the lanes tied).  Exact
// pairs for every packet, as before there were packed keys, against now, us:
// rounded lattice of 1M, self k = 8 / 16 / 32 879 / 1546 / 3475 against 923 /
// 1514 / 3515; 400k external queries on its points 1258 / 1863 / 3501 against
// 1468 / 2048 / 3754; 250k of its leaves 741 / 1053 / 2181 against 711 / 1041 /
// 2217.  Packets whose points are on a coarse enough grid (KeyGrid) need none of
// it: lattice of 1M, spacing 1, 1035 / 1557 / 3474 against 849 / 1027 / 1723.
template <typename T, int M, bool HEAP, bool SEEDED, bool PACKED, int MK, bool MULTI = false,
          bool LISTED = false>
__global__ __launch_bounds__(64, PACKED ? 4 : (MULTI ? 2 : 3)) void packet_knn_kernel(
    DTree<T> t, QSrc<T> qs, PacketArgs a, QueryMap qm,
    const typename CoordTraits<T>::D *__restrict__ seed, uint64_t *__restrict__ res,
    typename CoordTraits<T>::D *__restrict__ dists) {
    using D = typename CoordTraits<T>::D;
    using H = typename std::conditional<HEAP, TopKHeapLds<M>,
                                        typename TopKSel<T, M, PACKED>::type>::type;
    static_assert(!HEAP || (PACKED && !CoordTraits<T>::fp), "LDS heap tier needs packed integer keys");
    constexpr bool FPK = PACKED && CoordTraits<T>::fp;
    static_assert(HEAP || M <= 32, "register tiers hold at most 32 entries");
    __shared__ int32_t stk[PK_STACK];
    [[maybe_unused]] uint64_t *heap_mem = nullptr;
    if constexpr (HEAP) {
        __shared__ uint64_t heap[M * 64];
        heap_mem = heap;
    }
    const int lane = threadIdx.x;
    const int k = a.k;
    PacketCounters c;
    const int blk = xcd_block();
    const int W = a.width;
    if (blk * W >= a.nq) return;  // padding block of the XCD-ordered grid
    if constexpr (LISTED) {
        if (!uni(qm.packets[blk])) return;
    }
    const int slot = blk * W + lane;
    const bool active = lane < W && slot < a.nq;
    const int q = active ? slot_query(qm, slot) : 0;
    T px = T(0), py = T(0), pz = T(0);
    int self = -1;
    if (active) load_query(t, qs, q, px, py, pz, self);
    const int rank = self;  // the query's leaf rank (self queries), else -1
    if (!a.excl) self = -1;
    // Which queries are left to the listed pass is kept as masks of the wave, voted
    // outside divergent branches.  Which side of the walk the mask of the packet's
    // queries is voted on decides what it spills: self k = 32 of 10M points unseeded
    // 16.01 ms before it and 15.60 after, seeded 15.79 and 16.00.
    [[maybe_unused]] const uint64_t act0 = SEEDED ? __ballot(active) : 0ull;
    const int tie_min = W / 4;  // tied lanes that make a packet a tied one
    KeyGrid kg;
    [[maybe_unused]] bool grid = false;  // every point so far is on kg's grid
    // (not in passes, whose registers it would spill: k = 64 of 20M doubles 2 %)
    if constexpr (FPK && H::kRankKeys && !MULTI) {
        const bool in = px >= t.mnx[0] && px <= t.mxx[0] && py >= t.mny[0] && py <= t.mxy[0] &&
                        pz >= t.mnz[0] && pz <= t.mxz[0];
        grid = !t.orig_indices && kg.init(t, a.ibits) &&
               !__any(active && !(in && kg.on(px, py, pz)));
    }
    // Window pre-scan.  Self queries over all leaves: the packet is leaf ranks
    // [r0, r0 + 64), so its neighbours along the curve are the leaves on
    // either side.  Subset and external queries (Morton-ordered, so a
    // packet's queries are neighbours): the run of 64 leaves around the
    // middle lane's leaf rank, or around the leaf a greedy descent reaches
    // for the middle lane's point.
    int wlo = 0, whi = 0;
    int r0 = blk * W;
    if (a.window > 0) {
        const int src = (blk * W + W / 2 < a.nq) ? W / 2 : 0;
        if (qs.qx) r0 = run_start(descend_rank<T, MK>(t, rl(px, src), rl(py, src), rl(pz, src)), t.n);
        else if (qs.leaf_ids) r0 = run_start(uni(__shfl(rank, src, 64)), t.n);
        wlo = r0 - a.window > 0 ? r0 - a.window : 0;
        whi = r0 + 64 + a.window < t.n ? r0 + 64 + a.window : t.n;
    }
    static_assert(!MULTI || !HEAP, "passes need the register tier");
    if constexpr (MULTI) {
        // k above M (register tier): ceil(k / M) passes, each taking the M
        // nearest (d2, index) above the previous pass's last one, stored in
        // place.
        uint64_t redo = 0;  // lanes left to the listed pass
        [[maybe_unused]] uint64_t few = 0;  // of them: those whose seed held too few
        bool whole = false;
        typename H::Floor lo = H::no_floor();
        for (int base = 0; base < k; base += M) {
            const int kk = k - base < M ? k - base : M;
            H h;
            // The seed is read again in every pass (an opaque copy of q keeps
            // the load in the loop): holding it across the passes would cost
            // the kernel two registers.
            int qv = q;
            asm volatile("" : "+v"(qv));
            const D bound = (SEEDED && active) ? seed[qv] : dist_max<D>();
            if constexpr (PACKED) h.init(kk, bound, a.ibits);
            else h.init(kk, bound);
            // one walk instance for every pass (the first with no floor)
            const bool ties =
                packet_walk<T, H, MK, true>(t, a.bucket, active, px, py, pz, self, h, stk, c, wlo,
                                            whi, r0, lo, 0, 0, a.stop, base ? 0 : kk, tie_min, kg,
                                            grid);
            const uint64_t act = SEEDED ? act0 : __ballot(active);
            bool r = false;
            if constexpr (FPK) r = !grid & h.tied();
            else if constexpr (PACKED) r = h.needs_exact(kk);
            else r = (SEEDED || a.full) && h.unfilled();
            redo |= (ties ? ~0ull : __ballot(r)) & act;
            if constexpr (FPK)
                if (SEEDED || a.full) few |= __ballot(h.unfilled()) & act;
            const bool row = ((act & ~redo) >> lane) & 1;
            if constexpr (FPK) {
                volatile int32_t *bad = stk + lane;  // (the walk's stack is free again)
                *bad = 0;
                if (row)
                    h.template store_row<MK>(kk, res, dists, (size_t)q, k, base, t, px, py, pz, bad);
                redo |= act & __ballot(*bad != 0);
            } else if (row) {
                h.store_part(kk, res, dists, (size_t)q, k, base);
            }
            lo = h.next_floor();
            if constexpr (H::kRankKeys) {
                whole = ties || __popcll(redo) >= tie_min;
                if (whole) break;
            }
        }
        const uint64_t act = SEEDED ? act0 : __ballot(active);
        const bool over = c.leaves >= a.stop;
        if (H::kRankKeys && whole && !over) leave_packet(qm, blk, act, a.stats);
        else append_slots(qm, over ? act : redo | few, slot);
        // (its packet has counted the query already)
        if (LISTED && lane == 0 && redo && a.stats) atomicSub(&qm.count[1], (uint32_t)__popcll(redo));
    } else {
        H h;
        if constexpr (HEAP) h.key = heap_mem;
        const D bound = (SEEDED && active) ? seed[q] : dist_max<D>();
        if constexpr (PACKED) h.init(k, bound, a.ibits);
        else h.init(k, bound);
        int flo = 0, fhi = 0;
        int tie_k = k;  // (0: the fill has looked for ties)
        bool ties = false;
        if constexpr (H::kSortFill) {
            // self queries over all leaves: lane = leaf rank r0 + lane; the
            // window (>= 32 leaves on each side) covers every filled rank
            if (!qs.qx && !qs.leaf_ids && a.window >= 32) {
                __shared__ FillStage<T> fst;
                c.inserts += (uint32_t)fill_from_run<T, MK>(t, h, k, active, self >= 0, rank, px,
                                                            py, pz, r0, &fst, flo, fhi, kg, grid);
                tie_k = 0;
                if constexpr (H::kRankKeys)
                    ties = !grid && __popcll(__ballot(active && h.agreeing(k))) >= tie_min;
            }
        }
        // (a packet tied by its fill still enters the walk, which ends at the root: a
        // way out here, with its store before the walk's loads, made those vector
        // loads, 5 % of k = 16 of 2M points)
        ties |= packet_walk<T, H, MK>(t, a.bucket, active, px, py, pz, self, h, stk, c,
                                      ties ? 0 : wlo, ties ? 0 : whi, r0, H::no_floor(), flo, fhi,
                                      ties ? 0u : a.stop, tie_k, tie_min, kg, grid);
        const uint64_t act = SEEDED ? act0 : __ballot(active);
        const bool over = c.leaves >= a.stop;
        bool r = false;
        if constexpr (FPK) r = !grid & h.tied();
        else if constexpr (PACKED) r = h.needs_exact(k);
        else if constexpr (SEEDED) r = h.unfilled();
        uint64_t left = (over || ties ? ~0ull : __ballot(r)) & act;
        const bool row = ((act & ~left) >> lane) & 1;
        if constexpr (FPK) {
            volatile int32_t *bad = stk + lane;  // (the walk's stack is free)
            *bad = 0;
            if (row) h.template store_row<MK>(k, res, dists, (size_t)q, k, 0, t, px, py, pz, bad);
            left |= act & __ballot(*bad != 0);
        } else if (row) {
            h.store(k, res, dists, (size_t)q);
        }
        if (H::kRankKeys && !over && (ties || __popcll(left) >= tie_min)) {
            leave_packet(qm, blk, act, a.stats);
        } else {
            // (seeds that were too small do not make a packet a tied one)
            if constexpr (FPK && SEEDED) left |= __ballot(h.unfilled()) & act;
            append_slots(qm, left, slot);
        }
    }
    if (lane == 0 && a.stats) {
        atomicAdd((unsigned long long *)&a.stats[0], (unsigned long long)c.nodes);
        atomicAdd((unsigned long long *)&a.stats[1], (unsigned long long)c.leaves);
        if (c.overflow) atomicAdd((unsigned long long *)&a.stats[2], (unsigned long long)c.overflow);
        atomicAdd((unsigned long long *)&a.stats[5], (unsigned long long)c.rounds);
        atomicAdd((unsigned long long *)&a.stats[6], (unsigned long long)c.chains);
    }
    wave_add_stats(a.stats, 4, c.inserts);
}

// Range query, 64 queries per wave on one shared DFS (range_query,
// src/hlbvh.hpp:2006-2136), with the reference's results exactly:
//  * The reference's per-query DFS pushes right then left, so every query
//    meets its hits in ascending leaf rank; the shared walk is left-first too,
//    and each lane appends its hits in the order the walk meets them.
//  * The reference pushes a node's children only while its stack holds fewer
//    than 62 entries.  When it pops node v its stack holds the right siblings
//    pending along v's path, one per left turn, so that count -- the same for
//    every query that reaches v -- decides: the shared walk carries each
//    node's left turns and does not descend below a node with 62.
//  * A subtree of at most 64 leaves is tested leaf by leaf without
//    descending (its nodes add at most cnt - 1 left turns, so this is done
//    only when the reference could not have stopped inside it).
//  * A node is skipped only when no lane needs it (exact box distance, or the
//    conservative float32 form for integer periodic metrics); every leaf is
//    tested exactly: r_min^2 <= d2 <= r_max^2.
// Queries are taken in the order `order` (slot -> query; Morton order of the
// points inside the root box), so a wave's 64 queries are neighbours.
//
// Leaf test.  A float32 squared distance from coordinates relative to the
// packet's middle query, or another where that is not finite (fpf_*, whose error
// bound then follows the packet's extent instead of the box's), tells most pairs
// apart: surely inside, surely outside, and a few for the exact test.  Rounded relative coordinates q, x of
// a pair at gap g: |x| <= |q| + g, so the float gap is within (1 + 2u) g +
// 2u |q|, which fpf_upper / fpf_lower cover with E = 2.02 u max|q| and the
// doubles' own rounding.  Periodic boxes use it while every query is within a
// quarter period, less its radius, of the middle one: then no pair within a
// radius is wrapped, and a pair beyond half a period is outside either way.
// Float coordinates have no relative form; their exact distances are floats.
// 11 VALU a leaf (an LDS broadcast, a distance, two compares) where the exact
// test of doubles took 35.
//
// A dense region makes one wave's walk long (thousands of leaves), so each
// level costs one round trip to memory: both children's boxes, ranges and
// links are loaded together and the stack holds them; a row that is full is
// only counted.  Counts and CSR of 5M clustered doubles (60 hits a query) 30.5
// -> 16.5 ms, long rows by waves; 200k queries of 3M 64-bit points (at most 64
// hits kept) 8.5 -> 4.2 ms; runs of at most 32 / 48 / 64 leaves 20.1 / 18.5 /
// 18.1 ms before the long rows.
constexpr int RANGE_DROP_DEPTH = STACK_DEPTH - 2;  // 62

// Where a range query's hits go: counts, fixed-stride rows, CSR rows.
struct RangeOut {
    int32_t *res, *counts;
    int max_res;
    const int64_t *row_ptr;
    int32_t *cols;
    int64_t col_cap;
};
template <typename T> struct RangeSrc {
    const T *x, *y, *z, *rmin, *rmax;
};

// Squared radii of query q.
template <typename T>
__device__ inline void range_radii(const Metric &m, const RangeSrc<T> &s, int q,
                                   typename CoordTraits<T>::D &lo, typename CoordTraits<T>::D &hi) {
    if constexpr (CoordTraits<T>::fp) {
        const double a = (double)s.rmin[q], b = (double)s.rmax[q];
        lo = a * a;
        hi = b * b;
    } else {
        const uint64_t a = (uint64_t)s.rmin[q] >> m.dshift, b = (uint64_t)s.rmax[q] >> m.dshift;
        lo = a * a;
        hi = b * b;
    }
}

__device__ inline float wave_max_f32(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// A node's leaf range and children (uniform across the wave); node 0 of a
// one-leaf tree is that leaf.
struct RangeNode {
    int first, cnt, left, right;
};
template <typename T> __device__ inline RangeNode range_node(const DTree<T> &t, int v) {
    const int off = t.n - 1;
    if (t.n == 1) return RangeNode{0, 1, 0, 0};
    const int i = v < off ? v : 0;  // (a leaf has no entry: any will do)
    const int f = uni(t.rfirst[i]), l = uni(t.rlast[i]);
    const int lc = uni(t.left[i]), rc = uni(t.right[i]);
    return v < off ? RangeNode{f, l - f + 1, lc, rc} : RangeNode{v - off, 1, 0, 0};
}

template <typename T, int MK>
__global__ __launch_bounds__(64) void range_packet_kernel(DTree<T> t, RangeSrc<T> src, int nq,
                                                          const uint32_t *__restrict__ order,
                                                          RangeOut out) {
    using D = typename CoordTraits<T>::D;
    constexpr bool F32 = std::is_same<T, float>::value && MK != MK_ANY;
    constexpr bool REL = !std::is_same<T, float>::value && MK != MK_ANY;
    __shared__ int4 stk[PK_STACK];
    __shared__ uint8_t stk_lt[PK_STACK];
    [[maybe_unused]] __shared__ float4 s_leaf[64];
    const int lane = threadIdx.x;
    const int blk = xcd_block();
    if (blk * 64 >= nq) return;  // padding block of the XCD-ordered grid
    const int slot = blk * 64 + lane;
    const bool active = slot < nq;
    const int q = active ? (int)order[slot] : 0;
    const int n = t.n;
    const int off = n - 1;
    T px = T(0), py = T(0), pz = T(0);
    D rm2 = D(0), RM2 = D(0);
    if (active) {
        px = src.x[q]; py = src.y[q]; pz = src.z[q];
        range_radii<T>(t.m, src, q, rm2, RM2);
    }
    constexpr bool PRE = !CoordTraits<T>::fp && MK == MK_WRAP;
    [[maybe_unused]] const int wsh = PRE ? 32 - t.m.bits : 0;
    [[maybe_unused]] uint32_t qxs = 0, qys = 0, qzs = 0;
    [[maybe_unused]] T qmx = px, qmy = py, qmz = pz;
    [[maybe_unused]] float RM2f = 0.f;
    if constexpr (PRE) {
        qxs = (uint32_t)px << wsh;
        qys = (uint32_t)py << wsh;
        qzs = (uint32_t)pz << wsh;
        if constexpr (sizeof(T) >= 8) {
            const T mask = (T)((T(1) << t.m.bits) - T(1));
            qmx = px & mask;
            qmy = py & mask;
            qmz = pz & mask;
        }
        RM2f = wrap_filter_bound_pre((uint64_t)RM2, wsh);
    }
    // Leaf filter (RangeFilter).
    [[maybe_unused]] T cx = T(0), cy = T(0), cz = T(0);
    [[maybe_unused]] float fx = 0.f, fy = 0.f, fz = 0.f;
    [[maybe_unused]] float f_in = 0.f, f_out = 0.f, g_in = -1.f, g_out = -1.f;
    bool filter = F32;
    if constexpr (F32) {
        fx = px; fy = py; fz = pz;
        // exact: the float distances within [rm2, RM2]
        f_out = __double2float_rd(RM2);
        g_out = __double2float_ru(rm2);
    } else if constexpr (REL) {
        const int mid = centre_lane<T>(active, px, py, pz, blk * 64 + 32 < nq ? 32 : 0);
        cx = rl(px, mid); cy = rl(py, mid); cz = rl(pz, mid);
        if (active) {
            fx = rel_coord<T, MK>(t.m, px, cx);
            fy = rel_coord<T, MK>(t.m, py, cy);
            fz = rel_coord<T, MK>(t.m, pz, cz);
        }
        const float ext = wave_max_f32(fmaxf(fabsf(fx), fmaxf(fabsf(fy), fabsf(fz))));
        const float rad = wave_max_f32((float)sqrt((double)RM2) * (1.0f + 0x1p-20f));
        const double E = rel_err<T, MK>(t.m, ext, cx, cy, cz);
        const float period = CoordTraits<T>::fp ? (float)t.m.box : (float)(1ull << t.m.bits);
        filter = (MK == MK_WRAP ? ext + rad < 0.249f * period : true) && rad < 1.0e18f && ext < 1.0e18f;
        const RangeFilter rf = range_filter<D>(rm2, RM2, E);
        f_in = rf.f_in; f_out = rf.f_out; g_in = rf.g_in; g_out = rf.g_out;
    }
    const bool inner = __any(!(rm2 <= D(0)));
    auto node_near = [&](int nd) -> bool {
        if (!active) return false;
        if constexpr (PRE) {
            const float gx = wrap_box_gap_pre<T>(qmx, qxs, t.mnx[nd], t.mxx[nd], wsh);
            const float gy = wrap_box_gap_pre<T>(qmy, qys, t.mny[nd], t.mxy[nd], wsh);
            const float gz = wrap_box_gap_pre<T>(qmz, qzs, t.mnz[nd], t.mxz[nd], wsh);
            float d = gx * gx;
            d = __builtin_fmaf(gy, gy, d);
            d = __builtin_fmaf(gz, gz, d);
            return d <= RM2f;
        } else {
            return node_d2_k<T, MK>(t, px, py, pz, nd) <= RM2;
        }
    };
    const int64_t w0 = (active && out.row_ptr) ? out.row_ptr[q] : 0;
    int count = 0;
    // Tests leaf ranks [first, first + cnt) (cnt <= 64): lane j loads leaf j.
    auto scan = [&](int first, int cnt) {
        T bx = T(0), by = T(0), bz = T(0);
        int32_t bo = 0;
        if (lane < cnt) {
            bx = t.mnx[off + first + lane];
            by = t.mny[off + first + lane];
            bz = t.mnz[off + first + lane];
            bo = ret_index(t, off + first + lane);
        }
        auto exact = [&](T x, T y, T z) -> bool {
            const D d = leaf_d2_k<T, MK>(t.m, px, py, pz, x, y, z);
            return d >= rm2 && d <= RM2;
        };
        uint64_t hit = 0;
        // bit j of the mask = test(j), leaves taken last to first
        auto mask = [&](auto &&test) -> uint64_t {
            uint32_t lo = 0, hi = 0;
            const int c0 = cnt < 32 ? cnt : 32;
#pragma unroll 4
            for (int j = cnt - 1; j >= 32; --j) hi = (hi << 1) | (test(s_leaf[j]) ? 1u : 0u);
#pragma unroll 4
            for (int j = c0 - 1; j >= 0; --j) lo = (lo << 1) | (test(s_leaf[j]) ? 1u : 0u);
            return ((uint64_t)hi << 32) | lo;
        };
        if (filter) {
            if constexpr (F32) {
                s_leaf[lane] = make_float4(bx, by, bz, 0.f);
                hit = mask([&](const float4 &e) {
                    const float d = leaf_f32<MK>(t.m, px, py, pz, e.x, e.y, e.z);
                    return d <= f_out && d >= g_out;
                });
            } else if constexpr (REL) {
                s_leaf[lane] = make_float4(rel_coord<T, MK>(t.m, bx, cx), rel_coord<T, MK>(t.m, by, cy),
                                           rel_coord<T, MK>(t.m, bz, cz), 0.f);
                auto dist = [&](const float4 &e) { return fpf_sq(fx - e.x, fy - e.y, fz - e.z); };
                uint64_t unsure;
                {
                    uint32_t slo = 0, shi = 0, ulo = 0, uhi = 0;
                    const int c0 = cnt < 32 ? cnt : 32;
#pragma unroll 4
                    for (int j = cnt - 1; j >= 32; --j) {
                        const float d = dist(s_leaf[j]);
                        shi = (shi << 1) | (d < f_in ? 1u : 0u);
                        uhi = (uhi << 1) | (d <= f_out ? 1u : 0u);
                    }
#pragma unroll 4
                    for (int j = c0 - 1; j >= 0; --j) {
                        const float d = dist(s_leaf[j]);
                        slo = (slo << 1) | (d < f_in ? 1u : 0u);
                        ulo = (ulo << 1) | (d <= f_out ? 1u : 0u);
                    }
                    hit = ((uint64_t)shi << 32) | slo;
                    unsure = ((uint64_t)uhi << 32) | ulo;
                }
                if (inner) {  // only packets with an inner radius pay for it
                    hit &= ~mask([&](const float4 &e) { return dist(e) <= g_in; });
                    unsure &= ~mask([&](const float4 &e) { return dist(e) < g_out; });
                }
                unsure = active ? unsure & ~hit : 0ull;
                while (__any(unsure != 0)) {
                    const bool has = unsure != 0;
                    const int j = has ? __ffsll((long long)unsure) - 1 : 0;
                    const bool in = exact(shfl_any(bx, j), shfl_any(by, j), shfl_any(bz, j));
                    hit |= (has && in) ? (1ull << j) : 0ull;
                    unsure &= unsure - 1;
                }
            }
        } else {
            for (int j = 0; j < cnt; ++j)
                hit |= exact(rl(bx, j), rl(by, j), rl(bz, j)) ? (1ull << j) : 0ull;
        }
        if (!active) hit = 0;
        // a full row (or none): the rest is only counted
        if (!out.cols && count >= (out.res ? out.max_res : 0)) {
            count += __popcll(hit);
            hit = 0;
        }
        while (__any(hit != 0)) {  // one hit per lane per round, ascending rank
            const bool has = hit != 0;
            const int j = has ? __ffsll((long long)hit) - 1 : 0;
            hit &= hit - 1;
            const int32_t ri = t.orig_indices ? shfl_any(bo, j) : first + j;
            if (has) {
                if (out.res && count < out.max_res) out.res[(size_t)q * out.max_res + count] = ri;
                if (out.cols && w0 + count < out.col_cap) out.cols[w0 + count] = ri;
                ++count;
            }
        }
    };
    // The boxes and the ranges and links of both children are loaded together,
    // so a level costs one round trip to memory; the stack holds what was
    // loaded.  A Karras tree is less than 97 levels deep: it never overflows.
    int sp = 0, lt = 0;
    RangeNode v = range_node(t, 0);
    bool have = __any(node_near(0));
    while (have) {
        have = false;
        if (v.cnt == 1 || (v.cnt <= 64 && lt + v.cnt - 1 < RANGE_DROP_DEPTH)) {
            scan(v.first, v.cnt);
        } else if (lt < RANGE_DROP_DEPTH) {  // (the reference stops there)
            const RangeNode l = range_node(t, v.left), r = range_node(t, v.right);
            const bool nl = node_near(v.left), nr = node_near(v.right);
            const bool gl = __any(nl), gr = __any(nr);
            if (gl && gr) {
                stk[sp] = make_int4(r.first, r.cnt, r.left, r.right);
                stk_lt[sp] = (uint8_t)lt;
                ++sp;
            }
            have = gl || gr;
            v = gl ? l : r;
            lt += gl ? 1 : 0;
        }
        if (!have && sp > 0) {
            --sp;
            const int4 e = stk[sp];
            v = RangeNode{uni(e.x), uni(e.y), uni(e.z), uni(e.w)};
            lt = uni((int)stk_lt[sp]);
            have = true;
        }
    }
    if (active && out.counts) out.counts[q] = count;
}

// Range query, one wave per query: for queries that share too little of their
// walks for a packet (few, or far apart).  Both children of a node are tested
// in one vector pass, a run of at most 64 leaves one leaf per lane, and a
// run's hits leave in one store, ascending.  The same results, including the
// reference's stop at 62 left turns.  Bound by the latency of its walk: 3,000
// queries of 3M points 9.0 ms in packets, 0.87 ms here.  (The packet's way of
// loading both children's links early loads the scalar unit more and was 10 %
// slower here.)
// LISTED: the listed slots (the CSR query's long rows).
template <typename T, int MK, bool LISTED>
__global__ __launch_bounds__(256) void range_wave_kernel(DTree<T> t, RangeSrc<T> src, int nq,
                                                         QueryMap qm, RangeOut out) {
    using D = typename CoordTraits<T>::D;
    __shared__ int32_t s_node[4][PK_STACK];
    __shared__ uint8_t s_lt[4][PK_STACK];
    const int lane = threadIdx.x & 63;
    int32_t *stk = s_node[threadIdx.x >> 6];
    uint8_t *stk_lt = s_lt[threadIdx.x >> 6];
    const int wave = uni(xcd_block() * 4 + (int)(threadIdx.x >> 6));
    const int n = t.n, off = n - 1;
    auto answer = [&](int slot) {
        const int q = uni(slot_query(qm, slot));
        const T px = src.x[q], py = src.y[q], pz = src.z[q];
        D rm2, RM2;
        range_radii<T>(t.m, src, q, rm2, RM2);
        const int64_t w0 = out.row_ptr ? out.row_ptr[q] : 0;
        int count = 0;
        auto scan = [&](int first, int cnt) {
            const int leaf = off + first + (lane < cnt ? lane : 0);
            const D d = leaf_d2_k<T, MK>(t.m, px, py, pz, t.mnx[leaf], t.mny[leaf], t.mnz[leaf]);
            const bool in = lane < cnt && d >= rm2 && d <= RM2;
            const uint64_t m = __ballot(in);
            if (in && (out.res || out.cols)) {
                const int at = count + (int)__builtin_amdgcn_mbcnt_hi(
                                           (uint32_t)(m >> 32),
                                           __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                const int32_t ri = ret_index(t, leaf);
                if (out.res && at < out.max_res) out.res[(size_t)q * out.max_res + at] = ri;
                if (out.cols && w0 + at < out.col_cap) out.cols[w0 + at] = ri;
            }
            count += __popcll(m);
        };
        int sp = 0, v = 0, lt = 0;
        bool have = __any(node_d2_k<T, MK>(t, px, py, pz, 0) <= RM2);
        while (have) {
            have = false;
            int first = 0, cnt = 1;
            if (n > 1) {
                if (v >= off) {
                    first = v - off;
                } else {
                    first = uni(t.rfirst[v]);
                    cnt = uni(t.rlast[v]) - first + 1;
                }
            }
            if (cnt == 1 || (cnt <= 64 && lt + cnt - 1 < RANGE_DROP_DEPTH)) {
                scan(first, cnt);
            } else if (lt < RANGE_DROP_DEPTH) {
                const int l = uni(t.left[v]), r = uni(t.right[v]);
                const D d = node_d2_k<T, MK>(t, px, py, pz, (lane & 1) ? r : l);
                const uint64_t near = __ballot(d <= RM2);
                const bool gl = near & 1, gr = near & 2;
                if (gl && gr) {
                    stk[sp] = r;
                    stk_lt[sp] = (uint8_t)lt;
                    ++sp;
                }
                have = gl || gr;
                v = gl ? l : r;
                lt += gl ? 1 : 0;
            }
            if (!have && sp > 0) {
                --sp;
                v = uni(stk[sp]);
                lt = uni((int)stk_lt[sp]);
                have = true;
            }
        }
        if (lane == 0 && out.counts) out.counts[q] = count;
    };
    if constexpr (LISTED) {
        const int cnt = (int)qm.count[0];
        for (int e = wave; e < cnt; e += (int)gridDim.x * 4) answer(uni(qm.list[e]));
    } else if (wave < nq) {
        answer(wave);
    }
}

// Exclusive scan of int32 counts into int64 offsets (Q+1 entries), one block
// per 1024 counts, then block totals, then a fix-up pass.
__global__ __launch_bounds__(256) void scan_block_kernel(const int32_t *__restrict__ c, int nq,
                                                         int64_t *__restrict__ out,
                                                         int64_t *__restrict__ block_sums) {
    __shared__ int64_t wsum[4];
    const int base = blockIdx.x * 1024;
    int64_t v[4];
    int64_t s = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int i = base + threadIdx.x * 4 + j;
        v[j] = (i < nq) ? (int64_t)c[i] : 0;
        s += v[j];
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int64_t x = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int64_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    int64_t add = 0;
    for (int q = 0; q < w; ++q) add += wsum[q];
    int64_t run = x - s + add;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int i = base + threadIdx.x * 4 + j;
        if (i < nq) out[i] = run;
        run += v[j];
    }
    if (threadIdx.x == 255) block_sums[blockIdx.x] = run;
}

// Block totals -> exclusive offsets in place, and the grand total into
// out[nq]: one 1024-thread block, each thread taking a contiguous run of
// ceil(nb / 1024) totals (a single lane walking 20k totals took 2 ms).
__global__ __launch_bounds__(1024) void scan_totals_kernel(int64_t *block_sums, int nb,
                                                           int64_t *out, int nq) {
    __shared__ int64_t wsum[16];
    const int per = (nb + 1023) / 1024;
    const int b0 = (int)threadIdx.x * per;
    const int b1 = b0 + per < nb ? b0 + per : nb;
    int64_t s = 0;
    for (int b = b0; b < b1; ++b) s += block_sums[b];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int64_t x = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int64_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    int64_t run = x - s;
    for (int q = 0; q < w; ++q) run += wsum[q];
    for (int b = b0; b < b1; ++b) {
        const int64_t v = block_sums[b];
        block_sums[b] = run;
        run += v;
    }
    if (threadIdx.x == 1023) out[nq] = run;
}

__global__ __launch_bounds__(256) void scan_add_kernel(int64_t *out, int nq,
                                                       const int64_t *block_sums) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nq) out[i] += block_sums[i / 1024];
}

// ===========================================================================
// Query order for packet launches: external points by their Morton code (21
// bits per axis) inside the tree's root box, subset leaf ranks by rank, so a
// wavefront's 64 queries are neighbours whatever order the caller used.
// ===========================================================================
template <typename T>
__global__ __launch_bounds__(256) void query_key_kernel(DTree<T> t, QSrc<T> qs, int nq,
                                                        uint64_t *__restrict__ keys) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nq) return;
    if (!qs.qx) {
        keys[i] = (uint64_t)(uint32_t)qs.leaf_ids[i];
        return;
    }
    constexpr int QB = 21;
    const double side = (double)((1u << QB) - 1);
    auto quant = [&](T v, T lo, T hi) -> uint64_t {
        const double ext = (double)hi - (double)lo;
        double u = ext > 0.0 ? ((double)v - (double)lo) / ext : 0.0;
        u = u < 0.0 ? 0.0 : (u > 1.0 ? 1.0 : u);
        return (uint64_t)(u * side);
    };
    const uint64_t ix = quant(qs.qx[i], t.mnx[0], t.mxx[0]);
    const uint64_t iy = quant(qs.qy[i], t.mny[0], t.mxy[0]);
    const uint64_t iz = quant(qs.qz[i], t.mnz[0], t.mxz[0]);
    uint64_t m = 0;
    for (int b = 0; b < QB; ++b) {
        m |= ((ix >> b) & 1ull) << (3 * b + 2);
        m |= ((iy >> b) & 1ull) << (3 * b + 1);
        m |= ((iz >> b) & 1ull) << (3 * b);
    }
    keys[i] = m;
}

// ===========================================================================
// Host dispatch
// ===========================================================================
static inline unsigned blocks_for(size_t n, int per) {
    size_t g = (n + per - 1) / per;
    return (unsigned)(g ? g : 1);
}

// Lanes per block for an LDS heap of k entries with a DEPTH-entry stack: as
// many as fit 64 KiB.
template <typename T> static int lds_lanes(int k, int depth, size_t &lds) {
    using D = typename CoordTraits<T>::D;
    const size_t per_lane = (size_t)k * (sizeof(D) + 4) + (size_t)depth * 4;
    int lanes = 64;
    const size_t budget = 64 * 1024;
    while (lanes > 1 && (size_t)lanes * per_lane > budget) lanes >>= 1;
    lds = (size_t)lanes * per_lane;
    return lds <= budget ? lanes : 0;
}

// Per-stream work buffers of the query paths: the slot list of a direct pass
// and its counts, and the query-order sort buffers.  Each stream has its own set, grown on
// demand, so queries on different streams do not share memory; a stream's
// set is released by ft_stream_destroy / ft_stream_release.
//
// A graph captured on a stream holds the raw addresses of that stream's
// buffers.  While any such graph lives, a buffer that grows, or a set that is
// released, is not freed: its block joins the set's retired list, freed when
// the stream's last graph is destroyed, so a replay never touches freed
// memory.
struct RerunBuf {
    int32_t *list = nullptr;
    uint32_t *count = nullptr;
    int32_t *packets = nullptr;  // one entry per packet of 16 queries or more
    size_t cap = 0;
    void *block = nullptr;
};
struct QueryOrderBuf {
    Scratch S;
    uint64_t *keys = nullptr, *sorted = nullptr;
    size_t cap = 0;
};
struct StreamBufs {
    RerunBuf rr;
    QueryOrderBuf qo;
    int graphs = 0;               // live graphs captured on the stream
    bool released = false;        // out of the map, kept for its graphs
    std::vector<void *> retired;  // blocks replaced while graphs > 0
};
static std::mutex g_bufs_mu;
static std::unordered_map<hipStream_t, StreamBufs *> g_bufs;
static std::unordered_map<void *, StreamBufs *> g_graph_bufs;

static StreamBufs &stream_bufs(hipStream_t s) {
    std::lock_guard<std::mutex> lk(g_bufs_mu);
    auto it = g_bufs.find(s);
    if (it != g_bufs.end()) return *it->second;
    StreamBufs *b = new StreamBufs();
    g_bufs.emplace(s, b);
    return *b;
}

// Frees block p of stream s's set b after s's pending work, or keeps it on
// the retired list while a graph captured on s may still use it.
static int drop_block(StreamBufs &b, hipStream_t s, void *p) {
    if (!p) return FT_OK;
    {
        std::lock_guard<std::mutex> lk(g_bufs_mu);
        if (b.graphs > 0) {
            b.retired.push_back(p);
            return FT_OK;
        }
    }
    FT_HIP(hipStreamSynchronize(s));  // this stream's launches may still use it
    (void)hipFree(p);
    return FT_OK;
}

static void free_set(StreamBufs *b) {
    if (b->rr.block) (void)hipFree(b->rr.block);
    if (b->qo.keys) (void)hipFree(b->qo.keys);
    if (b->qo.S.block) (void)hipFree(b->qo.S.block);
    for (void *p : b->retired) (void)hipFree(p);
    for (auto &e : b->qo.S.ev)
        if (e) (void)hipEventDestroy(e);
    delete b;
}

// Frees the work buffers of stream s (after its pending work).  A set that a
// live graph uses leaves the map (the stream's next query makes a new one)
// and is freed with that graph.
int release_stream_bufs(hipStream_t s) {
    StreamBufs *b = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_bufs_mu);
        auto it = g_bufs.find(s);
        if (it == g_bufs.end()) return FT_OK;
        b = it->second;
        g_bufs.erase(it);
        if (b->graphs > 0) {
            b->released = true;
            return FT_OK;
        }
    }
    (void)hipStreamSynchronize(s);
    free_set(b);
    return FT_OK;
}

// A graph exec captured on stream s now holds s's buffers.
void graph_attach(hipStream_t s, void *exec) {
    StreamBufs &b = stream_bufs(s);
    std::lock_guard<std::mutex> lk(g_bufs_mu);
    ++b.graphs;
    g_graph_bufs[exec] = &b;
}

// The graph exec is destroyed: when it was its stream's last, the retired
// blocks (and a released set) are freed once the device is idle, since the
// graph may have been launched on any stream.
void graph_detach(void *exec) {
    StreamBufs *b = nullptr;
    std::vector<void *> old;
    bool drop_set = false;
    {
        std::lock_guard<std::mutex> lk(g_bufs_mu);
        auto it = g_graph_bufs.find(exec);
        if (it == g_graph_bufs.end()) return;
        b = it->second;
        g_graph_bufs.erase(it);
        if (--b->graphs > 0) return;
        old.swap(b->retired);
        drop_set = b->released;
    }
    if (old.empty() && !drop_set) return;
    (void)hipDeviceSynchronize();
    for (void *p : old) (void)hipFree(p);
    if (drop_set) free_set(b);
}

static int rerun_ensure(hipStream_t s, size_t n) {
    StreamBufs &sb = stream_bufs(s);
    RerunBuf &g_rerun = sb.rr;
    if (n <= g_rerun.cap && g_rerun.block) return FT_OK;
    FT_TRY(drop_block(sb, s, g_rerun.block));
    g_rerun.block = nullptr;
    g_rerun.cap = 0;
    const size_t cap = n + n / 2 + 1024;
    auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t bytes = al(cap * 4) + 256 + al((cap / 16 + 1) * 4);
    void *p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) return fail(FT_ENOMEM, "re-run buffer allocation failed");
    char *c = (char *)p;
    g_rerun.block = p;
    g_rerun.list = (int32_t *)c;
    g_rerun.count = (uint32_t *)(c + al(cap * 4));
    g_rerun.packets = (int32_t *)(c + al(cap * 4) + 256);
    g_rerun.cap = cap;
    return FT_OK;
}

// Starts a direct pass's list (QueryMap::count) and clears its packets' flags.
__global__ __launch_bounds__(256) void zero_counts_kernel(uint32_t *count, int32_t *packets, int np) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < 2) count[i] = 0;
    if (i < np) packets[i] = 0;
}
__global__ void add_count_kernel(uint64_t *stats, const uint32_t *count) { stats[3] += count[0] + count[1]; }

static inline int bit_length(uint64_t v) {
    int b = 0;
    while (v) {
        ++b;
        v >>= 1;
    }
    return b;
}

// Runs the statement with M = the register tier width for k (1, 4, 8, 16, 32).
#define FT_BY_M(K, ...)                                        \
    do {                                                       \
        if ((K) <= 1) { constexpr int M = 1; __VA_ARGS__; }         \
        else if ((K) <= 4) { constexpr int M = 4; __VA_ARGS__; }    \
        else if ((K) <= 8) { constexpr int M = 8; __VA_ARGS__; }    \
        else if ((K) <= 16) { constexpr int M = 16; __VA_ARGS__; }  \
        else { constexpr int M = 32; __VA_ARGS__; }                 \
    } while (0)

// Answers the slots that a direct pass left, exactly: up to k = 128 one wave
// per listed query (the wave-per-query tier), above that the per-lane heap
// walk with a 128-entry stack.  One lane per listed query left the 0.2 % of a
// seeded 10M-query pass latency-bound on a few hundred waves (1.7 ms against
// 0.3 ms with one wave each).
template <typename T, int MK>
static int launch_listed(hipStream_t s, const DTree<T> &dt, const QSrc<T> &qs, int nq, int k,
                         int excl, uint64_t cap, const QueryMap &qm, uint64_t *res,
                         typename CoordTraits<T>::D *d, uint64_t *stats) {
    if (k <= 128) {
        const dim3 g(xcd_grid(std::min<unsigned>(blocks_for(nq, 4), 2048u))), b(256);
        if (k <= 64)
            hipLaunchKernelGGL((wave_knn_kernel<T, 1, MK, true>), g, b, 0, s, dt, qs, nq, k, excl,
                               cap, qm, res, d, stats);
        else
            hipLaunchKernelGGL((wave_knn_kernel<T, 2, MK, true>), g, b, 0, s, dt, qs, nq, k, excl,
                               cap, qm, res, d, stats);
    } else {
        size_t lds = 0;
        const int lanes = lds_lanes<T>(k, LANE_STACK_CANON, lds);
        if (!lanes) return fail(FT_ELDS, "k too large for local memory: reduce k");
        const unsigned g = std::min<unsigned>(blocks_for(nq, lanes), 4096u);
        hipLaunchKernelGGL((lane_knn_lds_kernel<T, false, true, true, MK>), dim3(g),
                           dim3(LANE_BLOCK), lds, s, dt, qs, nq, k, excl, lanes, qm, res, d,
                           stats);
    }
    FT_CHECK_LAUNCH();
    return FT_OK;
}

// Top-k container of the packet kernels: packed keys, but for floating-point
// coordinates' shortest list.  Self-kNN of 3M clustered points, exact pairs
// against packed keys: double (periodic) k = 8 / 16 / 32 3.15 / 5.12 / 11.1
// against 2.69 / 3.54 / 5.75 ms, float 2.38 / 3.93 / 9.82 against 1.88 / 2.43 /
// 4.35 ms; 20 % of 20M doubles, k = 64 in passes, 97 against 31 ms.
template <typename T, int M> constexpr bool packs_keys() { return !CoordTraits<T>::fp || M >= 4; }

template <typename T, int M, bool HEAP, bool SEEDED, bool PACKED, int MK>
static void launch_pk(hipStream_t s, const DTree<T> &dt, const QSrc<T> &qs, const PacketArgs &a,
                      const QueryMap &qm, const typename CoordTraits<T>::D *seed, uint64_t *res,
                      typename CoordTraits<T>::D *d) {
    const dim3 g(xcd_grid(blocks_for(a.nq, a.width)));
    if constexpr (!HEAP && M == 32) {
        if (a.k > M) {
            hipLaunchKernelGGL((packet_knn_kernel<T, M, HEAP, SEEDED, PACKED, MK, true>), g,
                               dim3(64), 0, s, dt, qs, a, qm, seed, res, d);
            return;
        }
    }
    hipLaunchKernelGGL((packet_knn_kernel<T, M, HEAP, SEEDED, PACKED, MK>), g, dim3(64), 0, s, dt,
                       qs, a, qm, seed, res, d);
}

// The packets that a pass of cut keys left whole, with exact (d, index) pairs.
template <typename T, int MK>
static void launch_packets_listed(hipStream_t s, const DTree<T> &dt, const QSrc<T> &qs,
                                  const PacketArgs &a, const QueryMap &qm, uint64_t *res,
                                  typename CoordTraits<T>::D *d) {
    const dim3 g(xcd_grid(blocks_for(a.nq, a.width)));
#define FT_LISTED(M_, MULTI_)                                                                     \
    hipLaunchKernelGGL((packet_knn_kernel<T, M_, false, false, false, MK, MULTI_, true>), g,      \
                       dim3(64), 0, s, dt, qs, a, qm, (const double *)nullptr, res, d)
    if (a.k <= 4) FT_LISTED(4, false);
    else if (a.k <= 8) FT_LISTED(8, false);
    else if (a.k <= 16) FT_LISTED(16, false);
    else if (a.k <= 32) FT_LISTED(32, false);
    else FT_LISTED(32, true);
#undef FT_LISTED
}

template <typename T, int M, bool HEAP, int MK>
static void launch_packet_m(hipStream_t s, const DTree<T> &dt, const QSrc<T> &qs,
                            const PacketArgs &a, const QueryMap &qm,
                            const typename CoordTraits<T>::D *seed, uint64_t *res,
                            typename CoordTraits<T>::D *d) {
    constexpr bool PACKED = packs_keys<T, M>();
    if (seed) launch_pk<T, M, HEAP, true, PACKED, MK>(s, dt, qs, a, qm, seed, res, d);
    else launch_pk<T, M, HEAP, false, PACKED, MK>(s, dt, qs, a, qm, seed, res, d);
}

// Whether a call's queries are so few that a wave for each of them finishes
// before packets of 64 do.  A packet's walk is one wave's serial work (0.2 to
// 1 ms, more where its queries lie far apart, as few queries of many points
// do) and few packets leave the chip idle; a wave per query costs 5 to 13 ns of
// the whole chip.  The line is where both took the same time over trees of 20k
// to 10M points (packets against waves, us): 30k points k = 8 30k queries
// 580 / 476, 100k 481 / 1186; 300k points 30k 899 / 374, 100k 821 / 849; 10M
// points 200k 3003 / 2785, 500k 3039 / 6308; k = 32 of 10M points 200k
// 5412 / 3282, 500k 5861 / 7408.  1,000 queries k = 32 of 10M points took 21 ms
// in packets.
static bool few_queries(int64_t nq, int64_t n, int k) {
    const double f = k <= 4 ? 0.8 : (k <= 16 ? 1.0 : (k <= 32 ? 1.7 : 5.0));
    return (double)nq <= 900.0 * f * std::cbrt((double)n);
}

// Wave-tier queries up to this many run in the caller's order: sorting them
// along the curve costs 60 us of launches and gains nothing while the waves in
// flight hold most of them (10M points, k = 32, ordered / unordered: 1k queries
// 196 / 150 us, 20k 575 / 532, 40k 924 / 938, 80k 1544 / 1794).
constexpr int UNORDERED_WAVES = 24576;

// Queries per packet: 64, one per lane, or 32 while the packets of 64 would be
// fewer than about two and a half per SIMD (build + self-kNN of 100k doubles,
// k = 4 / 8 / 16 / 32: uniform 373 / 436 / 503 / 681 us with 64, 362 / 418 /
// 481 / 667 with 32; clustered 565 / 638 / 746 / 1174 and 521 / 594 / 703 /
// 1079; at 400k points 64 are 10 % faster).
constexpr int WIDE_PACKETS_FROM = 150000;

// Leaves a packet may scan before its queries go to one wave each, so that the
// few packets whose queries lie far apart do not set the time.  A hand-over
// costs 60 to 100 us however few the queries, so the limits lie above what
// packets of uniform points need (2,000 in packets of 64 cost k = 16 of 100k
// uniform doubles 40 us of 500).  Self-kNN of 300k clustered floats k = 8 /
// 16 / 32: 885 / 1145 / 1591 us without, 476 / 579 / 959 with; above 600k
// points packets are enough to cover the slow ones (2M points 3 % slower with
// 4,000).  Other queries share less of their walks the sparser they are
// (k = 32, 1M queries of 2M doubles 4.77 ms without, 3.81 with 4,000; of 10M
// points 7.25 without, 14.6 with 4,000).
static uint32_t packet_leaf_limit(int64_t nq, int64_t n, int k, int width, bool all_leaves,
                                  bool fp) {
    if (k > 32 && !fp) return ~0u;  // the integers' passes have no limit (packet_walk)
    const int64_t passes = (k + 31) / 32;
    if (!all_leaves) return (uint32_t)std::min<int64_t>(passes * (3000 + 1000 * (n / nq)), 1 << 30);
    if (n > 600000) return ~0u;
    const int64_t per_pass = width == 64 ? (k <= 16 ? 3000 : 4000)
                                         : (k <= 8 ? 2000 : (k <= 16 ? 2500 : 3000));
    return (uint32_t)(passes * per_pass);
}

// One canonical query launch: a direct pass, and where it can leave slots
// unanswered (packed keys that saturate, seeds that were too small, per-lane
// stacks that would overflow) the listed pass over the slots it appended.  No
// host round trip.  The wave tier answers every query itself.
template <typename T, int MK>
static int run_canonical(hipStream_t s, const DTree<T> &dt, const QSrc<T> &qs, int nq, int k,
                         int excl, int algo, bool automatic, int bucket, int topk, int window,
                         int width, const uint32_t *order,
                         const typename CoordTraits<T>::D *seed, uint64_t *res,
                         typename CoordTraits<T>::D *d, uint64_t *stats, const RerunBuf *rr) {
    constexpr bool INTD = !CoordTraits<T>::fp;
    // (the listed pass's wave tier is the one of k <= 128)
    const uint32_t stop = algo == FT_ALGO_PACKET && !seed && topk != FT_TOPK_LDS_HEAP
                              ? packet_leaf_limit(nq, dt.n, k, width, !qs.qx && !qs.leaf_ids, !INTD)
                              : ~0u;
    // Neighbours at an infinite distance, or at none (a NaN coordinate): the packet
    // tier has none, the wave tier puts them after the finite ones.  Which of the
    // two a call shows follows from its algorithm and k alone, not from the tier
    // that its numbers of queries and leaves lead to: the automatic choice shows
    // none up to k = 32 and all above, an explicit one its tier's (exact re-runs of
    // seeded queries and of full stacks: the wave tier's).
    const bool none = !INTD && !seed && (automatic ? k <= 32 : algo == FT_ALGO_PACKET);
    const uint64_t cap = none ? 0x7fefffffffffffffull : ~0ull;  // (the bits of DBL_MAX)
    const bool full = !INTD && automatic && k > 32 && algo == FT_ALGO_PACKET;
    // (float coordinates' keys are exact: nothing to leave without a seed)
    const bool cuts = INTD || (std::is_same<T, double>::value && k > 1);
    const bool leaves_slots = algo == FT_ALGO_PACKET ? (cuts || seed || full || stop != ~0u)
                                                     : algo != FT_ALGO_WAVE;
    if (!rr) {  // the stream's own buffers, grown to nq (also where this call leaves
                // nothing: see query_order_ensure)
        FT_TRY(rerun_ensure(s, (size_t)nq));
        rr = &stream_bufs(s).rr;
    }
    if (leaves_slots) {
        const bool flags = algo == FT_ALGO_PACKET && std::is_same<T, double>::value;
        const int np = flags ? (int)blocks_for(nq, width) : 0;
        hipLaunchKernelGGL(zero_counts_kernel, dim3(blocks_for(std::max(np, 2), 256)), dim3(256), 0,
                           s, rr->count, rr->packets, np);
    }
    const QueryMap qm{order, leaves_slots ? rr->list : nullptr, leaves_slots ? rr->count : nullptr,
                      leaves_slots ? rr->packets : nullptr};
    if (algo == FT_ALGO_PACKET) {
        PacketArgs a{};
        a.nq = nq;
        a.k = k;
        a.excl = excl;
        a.bucket = bucket;
        a.width = width;
        a.ibits = bit_length((uint64_t)dt.n);
        // A subset packet's leaves spread over about n / nq times more ranks:
        // its window grows with that spread, up to 4x (a 20 % subset of 20M
        // clustered points at k = 64: windows of 128 / 256 / 512 / 1024 took
        // 114.7 / 112.7 / 111.9 / 113.8 ms).
        const int spread = qs.leaf_ids ? (int)std::min<int64_t>(4, std::max<int64_t>(1, dt.n / std::max(nq, 1))) : 1;
        a.window = window * spread;
        a.full = full;
        a.stop = stop;
        a.stats = stats;
        // k above 32 with integer coordinates: multi-pass register tier by
        // default, LDS heap tiers on request.
        const bool heap = INTD && topk == FT_TOPK_LDS_HEAP;
        if (!heap) {
            FT_BY_M(k, (launch_packet_m<T, M, false, MK>(s, dt, qs, a, qm, seed, res, d)));
            if constexpr (std::is_same<T, double>::value) {
                a.stop = ~0u;
                if (k > 1) launch_packets_listed<T, MK>(s, dt, qs, a, qm, res, d);
            }
        } else if constexpr (INTD) {
            if (k <= 32) launch_packet_m<T, 32, true, MK>(s, dt, qs, a, qm, seed, res, d);
            else if (k <= 64) launch_packet_m<T, 64, true, MK>(s, dt, qs, a, qm, seed, res, d);
            else if (k <= 128) launch_packet_m<T, 128, true, MK>(s, dt, qs, a, qm, seed, res, d);
            else return fail(FT_EINVAL, "packet traversal: k above the heap tiers");
        }
    } else if (algo == FT_ALGO_WAVE) {
        const dim3 g(xcd_grid(blocks_for(nq, 4))), b(256);
#define FT_WAVE_LAUNCH(S_)                                                                      \
    hipLaunchKernelGGL((wave_knn_kernel<T, S_, MK>), g, b, 0, s, dt, qs, nq, k, excl, cap, qm, \
                       res, d, stats)
        if (k <= 64) FT_WAVE_LAUNCH(1);
        else if (k <= 128) FT_WAVE_LAUNCH(2);
        else if (k <= 256) FT_WAVE_LAUNCH(4);
        else if (k <= 512) FT_WAVE_LAUNCH(8);
        else if (k <= WAVE_MAX_K) FT_WAVE_LAUNCH(16);
        else return fail(FT_EINVAL, "wave traversal: k above 1024");
#undef FT_WAVE_LAUNCH
    } else if (k <= 32) {
        const dim3 g(xcd_grid(blocks_for(nq, LANE_BLOCK))), b(LANE_BLOCK);
        if (algo == FT_ALGO_PLAIN)
            FT_BY_M(k, hipLaunchKernelGGL((lane_knn_reg_kernel<T, M, false, MK>), g, b, 0, s,
                                          dt, qs, nq, k, excl, qm, res, d, stats));
        else
            FT_BY_M(k, hipLaunchKernelGGL((lane_knn_reg_kernel<T, M, true, MK>), g, b, 0, s,
                                          dt, qs, nq, k, excl, qm, res, d, stats));
    } else {
        size_t lds = 0;
        const int lanes = lds_lanes<T>(k, STACK_DEPTH, lds);
        if (!lanes) return fail(FT_ELDS, "k too large for local memory: reduce k");
        const dim3 g(xcd_grid(blocks_for(nq, lanes))), b(LANE_BLOCK);
        if (algo == FT_ALGO_PLAIN)
            hipLaunchKernelGGL((lane_knn_lds_kernel<T, false, false, false, MK>), g, b, lds, s, dt,
                               qs, nq, k, excl, lanes, qm, res, d, stats);
        else
            hipLaunchKernelGGL((lane_knn_lds_kernel<T, false, true, false, MK>), g, b, lds, s, dt,
                               qs, nq, k, excl, lanes, qm, res, d, stats);
    }
    FT_CHECK_LAUNCH();
    if (!leaves_slots) return FT_OK;
    if (stats) {
        hipLaunchKernelGGL(add_count_kernel, dim3(1), dim3(1), 0, s, stats,
                           (const uint32_t *)rr->count);
        FT_CHECK_LAUNCH();
    }
    // (the work of a seed's exact re-runs is not counted, only their number)
    return launch_listed<T, MK>(s, dt, qs, nq, k, excl, cap, qm, res, d, seed ? nullptr : stats);
}

// The stream's buffers for ordering nq queries.  Every call that may order its
// queries makes sure of them, also one that leaves them as they are: a call
// captured later, which may not grow a buffer, then finds them large enough
// whichever tier either of the two takes.
static int query_order_ensure(hipStream_t s, int nq) {
    StreamBufs &sb = stream_bufs(s);
    QueryOrderBuf &g_qorder = sb.qo;
    if (g_qorder.cap < (size_t)nq) {
        FT_TRY(drop_block(sb, s, g_qorder.keys));
        g_qorder.keys = nullptr;
        g_qorder.cap = 0;
        const size_t cap = (size_t)nq + (size_t)nq / 2 + 1024;
        if (hipMalloc(&g_qorder.keys, 2 * cap * 8) != hipSuccess)
            return fail(FT_ENOMEM, "query order allocation failed");
        g_qorder.sorted = g_qorder.keys + cap;
        g_qorder.cap = cap;
    }
    if ((size_t)nq > g_qorder.S.cap_n && g_qorder.S.block) {
        // the sort scratch grows: hand its block over here, so that the
        // sort's own growth allocates a new one and frees nothing
        FT_TRY(drop_block(sb, s, g_qorder.S.block));
        g_qorder.S.block = nullptr;
        g_qorder.S.cap_n = 0;
    }
    return scratch_ensure_public(g_qorder.S, (size_t)nq);
}

template <typename T>
static int query_order(hipStream_t s, const DTree<T> &dt, const QSrc<T> &qs, int nq,
                       const uint32_t *&order) {
    FT_TRY(query_order_ensure(s, nq));
    QueryOrderBuf &g_qorder = stream_bufs(s).qo;
    hipLaunchKernelGGL((query_key_kernel<T>), dim3(blocks_for(nq, 256)), dim3(256), 0, s, dt, qs,
                       nq, g_qorder.keys);
    FT_CHECK_LAUNCH();
    FT_TRY(radix_sort_u64(s, g_qorder.S, g_qorder.keys, (size_t)nq, g_qorder.sorted,
                          qs.qx ? 63 : 32));
    order = g_qorder.S.perm;
    return FT_OK;
}

template <typename T>
static int knn_dispatch(hipStream_t s, const ft_tree *tree, const QSrc<T> &qs, int nq, int k,
                        int excl, uint64_t *res, void *dists_v, const ft_query_opts *opts,
                        bool external, const RerunBuf *rr = nullptr) {
    using D = typename CoordTraits<T>::D;
    D *dists = (D *)dists_v;
    const DTree<T> dt = make_dtree<T>(*tree);
    ft_query_opts o{};
    if (opts) o = *opts;
    uint64_t *stats = o.stats;
    int algo = o.algorithm;
    const bool automatic = algo == FT_ALGO_AUTO;
    if (o.mode == FT_MODE_REFERENCE) {
        if (o.seed_bound) return fail(FT_EINVAL, "a seed bound needs canonical mode");
        if (external && k > 32) {
            // SortedMergeHeap tier, capacity next_pow2(max_k)
            int maxk = o.max_k > 0 ? o.max_k : 256;
            int cap = 1;
            while (cap < maxk) cap <<= 1;
            const size_t lds = (size_t)cap * (sizeof(D) + 4) + 8 + 32 * (sizeof(D) + 4) + STACK_DEPTH * 4 + 64;
            if (lds > 64 * 1024)
                return fail(FT_ELDS, "knn_query_large_k: k too large, local memory requirement exceeds device limit");
            hipLaunchKernelGGL((merge_knn_kernel<T>), dim3(nq), dim3(64), lds, s, dt, qs, nq, k,
                               cap, res, dists, stats);
            FT_CHECK_LAUNCH();
            return FT_OK;
        }
        size_t lds = 0;
        const int lanes = lds_lanes<T>(k, STACK_DEPTH, lds);
        if (!lanes) return fail(FT_ELDS, "k too large for local memory: reduce k");
        const QueryMap qm{nullptr, nullptr, nullptr, nullptr};
        const dim3 g(xcd_grid(blocks_for(nq, lanes))), b(LANE_BLOCK);
        if (algo == FT_ALGO_PLAIN)
            hipLaunchKernelGGL((lane_knn_lds_kernel<T, true, false, false, MK_ANY>), g, b, lds, s,
                               dt, qs, nq, k, excl, lanes, qm, res, dists, stats);
        else
            hipLaunchKernelGGL((lane_knn_lds_kernel<T, true, true, false, MK_ANY>), g, b, lds, s,
                               dt, qs, nq, k, excl, lanes, qm, res, dists, stats);
        FT_CHECK_LAUNCH();
        return FT_OK;
    }
    // Canonical mode.  Packet tiers: registers for k <= 32, passes of 32 up
    // to k = 128 where packets share their walks best: every leaf, or queries
    // at least a fifth as many as the leaves up to k = 64 (10M clustered int64
    // points, passes against the wave tier: self k = 64 / 128 43 / 93 against
    // 107 / 154 ms, a 20 % subset k = 64 19.1 against 22.6, 1M external queries
    // 19.4 against 16.1; 20M doubles: self k = 64 76 against 209 ms, a 20 %
    // subset k = 64 / 128 31 / 67 against 45 / 62).  The wave tier for the
    // others up to k = 1,024 and wherever the queries are few; above k = 1,024
    // the per-lane heap walk.
    const bool packet_ok = k <= 128;  // above 32: passes of 32
    if (algo == FT_ALGO_AUTO) {
        const bool all_leaves = !external && !qs.leaf_ids;
        const bool dense = (int64_t)nq * 5 >= (int64_t)dt.n;
        if (k > WAVE_MAX_K) algo = FT_ALGO_GROUPED;
        else if (few_queries(nq, dt.n, k)) algo = FT_ALGO_WAVE;
        else if (k <= 32 || (all_leaves && k <= 128) || (dense && k <= 64)) algo = FT_ALGO_PACKET;
        else algo = FT_ALGO_WAVE;
    }
    if (o.seed_bound && packet_ok) algo = FT_ALGO_PACKET;
    if (algo == FT_ALGO_PACKET && !packet_ok)
        algo = k <= WAVE_MAX_K ? FT_ALGO_WAVE : FT_ALGO_GROUPED;
    const D *seed = algo == FT_ALGO_PACKET ? (const D *)o.seed_bound : nullptr;
    const int bucket = o.leaf_bucket > 0 ? std::min(o.leaf_bucket, 64) : 64;
    const uint32_t *order = nullptr;
    if (algo == FT_ALGO_WAVE && k > WAVE_MAX_K) algo = FT_ALGO_GROUPED;
    if ((algo == FT_ALGO_PACKET || algo == FT_ALGO_WAVE) && (qs.qx || qs.leaf_ids) && nq > 64) {
        if (algo == FT_ALGO_WAVE && nq <= UNORDERED_WAVES) FT_TRY(query_order_ensure(s, nq));
        else FT_TRY(query_order<T>(s, dt, qs, nq, order));
    }
    // auto: 192 leaves on each side (self k = 32 at 10M clustered points: 64 /
    // 128 / 192 / 256 / 384 took 19.17 / 18.93 / 18.80 / 18.77 / 18.81 ms;
    // 192 was also as fast or faster at k = 1 to 64, for subsets and for
    // external queries)
    const int window = o.window < 0 ? 0 : (o.window == 0 ? 192 : std::min(o.window, 1 << 20));
    if (o.group_width != 0 && o.group_width != 16 && o.group_width != 32 && o.group_width != 64)
        return fail(FT_EINVAL, "group_width must be 0, 16, 32 or 64");
    const int width = o.group_width ? o.group_width : (nq < WIDE_PACKETS_FROM ? 32 : 64);
    switch (metric_kind<T>(dt.m)) {
    case MK_WRAP:
        return run_canonical<T, MK_WRAP>(s, dt, qs, nq, k, excl, algo, automatic, bucket, o.topk,
                                         window, width, order, seed, res, dists, stats, rr);
    case MK_OPEN:
        return run_canonical<T, MK_OPEN>(s, dt, qs, nq, k, excl, algo, automatic, bucket, o.topk,
                                         window, width, order, seed, res, dists, stats, rr);
    default:
        return fail(FT_EINVAL, "unsupported metric: periodic integer coordinates need B <= 31");
    }
}

// Entry points used by the C ABI layer (device pointers only).
int knn_entry(hipStream_t s, const ft_tree *tree, const void *qx, const void *qy, const void *qz,
              const int32_t *leaf_ids, int nq, int k, int excl, uint64_t *res, void *dists,
              const ft_query_opts *opts) {
    FT_DISPATCH_COORD(tree->coord_type, {
        QSrc<T> qs{(const T *)qx, (const T *)qy, (const T *)qz, leaf_ids};
        return knn_dispatch<T>(s, tree, qs, nq, k, excl, res, dists, opts, qx != nullptr);
    });
    return FT_OK;
}

// ---- non-allocating self-kNN (no reference counterpart) ----------------------
// For callers that cannot allocate (code under graph capture, serving loops):
// the canonical pipeline's slot list and its counts live in one file-scope
// device array instead of per-stream allocations.  Every call on a device
// shares that device's copy, which keeps the last call's contents; the counts
// are cleared by a kernel at the start of each call and list entries are
// written before they are read.  Calls that overlap on one device race.
constexpr size_t NA_MAX_QUERIES = (size_t)1 << 24;
constexpr size_t NA_OFF_PACKETS = NA_MAX_QUERIES * 4;
constexpr size_t NA_OFF_COUNT = NA_OFF_PACKETS + (NA_MAX_QUERIES / 16 + 64) * 4;
constexpr size_t NA_BYTES = NA_OFF_COUNT + 256;  // 68 MiB + 512 bytes
static __device__ __align__(256) uint8_t scratch[NA_BYTES];

constexpr int NA_MAX_DEVICES = 64;
static std::mutex g_na_mu;
static void *g_na_ptr[NA_MAX_DEVICES];

// The device address of `scratch` on the current device, looked up once per
// device (each device holds its own copy of the array at its own address).
static int noalloc_scratch(void **out) {
    int dev = 0;
    FT_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= NA_MAX_DEVICES) return fail(FT_EINVAL, "device index out of range");
    std::lock_guard<std::mutex> lk(g_na_mu);
    if (!g_na_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(FT_EHIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_na_ptr[dev] = p;
    }
    *out = g_na_ptr[dev];
    return FT_OK;
}

size_t noalloc_max_queries() { return NA_MAX_QUERIES; }

int knn_noalloc_entry(hipStream_t s, const ft_tree *tree, int k, int excl, uint64_t *res,
                      void *dists, const ft_query_opts *opts) {
    const size_t nq = tree->num_leaves;
    if (nq > NA_MAX_QUERIES)
        return fail(FT_ERANGE, "ft_self_knn_query_noalloc: more than 16777216 queries (its "
                               "fixed scratch size); use ft_self_knn_query");
    void *p = nullptr;
    FT_TRY(noalloc_scratch(&p));
    char *c = (char *)p;
    RerunBuf rr;
    rr.list = (int32_t *)c;
    rr.packets = (int32_t *)(c + NA_OFF_PACKETS);
    rr.count = (uint32_t *)(c + NA_OFF_COUNT);
    rr.cap = NA_MAX_QUERIES;
    FT_DISPATCH_COORD(tree->coord_type, {
        const QSrc<T> qs{nullptr, nullptr, nullptr, nullptr};
        return knn_dispatch<T>(s, tree, qs, (int)nq, k, excl, res, dists, opts, false, &rr);
    });
    return FT_OK;
}

// Whether a wave per query beats packets of 64 for nq range queries: a packet's
// serial walk against 10 to 50 ns of the whole chip per query (packets /
// waves, us, queries following the density: 3M points 30k queries 4193 / 1500,
// 100k 3341 / 3491; 1M points 30k 3099 / 2055, 100k 3043 / 5168; 300k points
// 3k 1913 / 585, 30k 1483 / 1689).
static bool few_range_queries(int64_t nq, int64_t n) {
    return (double)nq <= 400.0 * std::cbrt((double)n);
}

// Range query launch: a wave per query where the queries are few for the tree,
// else packets in Morton order of the points inside the root box.  (Packets
// that handed wide or slow walks over to waves, by leaves scanned or by the
// share of hits, were slower: 18.0 -> 20.6 ms and more on 5M doubles.)
template <typename T, int MK>
static int range_walk(hipStream_t s, const DTree<T> &dt, const RangeSrc<T> &src, int nq,
                      const RangeOut &out) {
    if (few_range_queries(nq, dt.n)) {
        FT_TRY(query_order_ensure(s, nq));
        const QueryMap qm{nullptr, nullptr, nullptr, nullptr};
        hipLaunchKernelGGL((range_wave_kernel<T, MK, false>), dim3(xcd_grid(blocks_for(nq, 4))),
                           dim3(256), 0, s, dt, src, nq, qm, out);
    } else {
        const QSrc<T> qs{src.x, src.y, src.z, nullptr};
        const uint32_t *order = nullptr;
        FT_TRY(query_order<T>(s, dt, qs, nq, order));
        hipLaunchKernelGGL((range_packet_kernel<T, MK>), dim3(xcd_grid(blocks_for(nq, 64))),
                           dim3(64), 0, s, dt, src, nq, order, out);
    }
    FT_CHECK_LAUNCH();
    return FT_OK;
}

// The statement with MK = the metric kind of tree dt.
#define FT_BY_METRIC(dt, ...)                                         \
    switch (metric_kind<T>((dt).m)) {                                 \
    case MK_WRAP: { constexpr int MK = MK_WRAP; __VA_ARGS__; } break; \
    case MK_OPEN: { constexpr int MK = MK_OPEN; __VA_ARGS__; } break; \
    default: { constexpr int MK = MK_ANY; __VA_ARGS__; } break;       \
    }

template <typename T>
static int range_launch(hipStream_t s, const ft_tree &tree, const RangeSrc<T> &src, int nq,
                        const RangeOut &out) {
    if (nq <= 0) return FT_OK;
    const DTree<T> dt = make_dtree<T>(tree);
    FT_BY_METRIC(dt, return (range_walk<T, MK>(s, dt, src, nq, out)));
    return FT_OK;
}

int range_entry(hipStream_t s, const ft_tree *tree, const void *qx, const void *qy,
                const void *qz, const void *rmin, const void *rmax, int nq, int32_t *res,
                int32_t *counts, int max_res, const int64_t *row_ptr, int32_t *cols,
                int64_t col_cap) {
    int rc = FT_OK;
    FT_DISPATCH_COORD(tree->coord_type,
                      rc = range_launch<T>(s, *tree,
                                           RangeSrc<T>{(const T *)qx, (const T *)qy, (const T *)qz,
                                                       (const T *)rmin, (const T *)rmax},
                                           nq, RangeOut{res, counts, max_res, row_ptr, cols,
                                                        col_cap}));
    return rc;
}

// ---------------------------------------------------------------------------
// CSR range query with the columns in one walk (no reference counterpart).
// The walk writes every query's hit count and its first CSR_POOL hits into a
// fixed-stride pool (the fixed-stride range_query output); after the scan of
// the counts, the pool rows are copied to their CSR rows, and only queries
// with more than CSR_POOL hits are walked again, one wave each, writing their
// whole rows (1.4 % of the rows of 5M clustered points, scattered: 8.0 ms in
// packets).
// A walk meets a query's hits in the same (ascending rank) order every time,
// so the rows equal those of a counting walk followed by a filling walk.
// ---------------------------------------------------------------------------
constexpr int CSR_POOL = 128;

// Rows of at most CSR_POOL hits from the pool into cols.  One wave per group
// of 64 rows (grid-stride over groups): the lanes load the group's counts and
// offsets in one pass, then the wave copies four rows at a time, their pool
// loads issued before their stores (one row at a time, each waiting on its
// count and offset, ran at 1.9 TB/s).
__global__ __launch_bounds__(256) void csr_copy_kernel(const int32_t *__restrict__ pool,
                                                       const int32_t *__restrict__ counts,
                                                       const int64_t *__restrict__ row_ptr, int nq,
                                                       int32_t *__restrict__ cols,
                                                       int64_t col_cap) {
    const int lane = threadIdx.x & 63;
    const int64_t w = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int64_t nw = (int64_t)gridDim.x * (blockDim.x >> 6);
    for (int64_t g = w; g * 64 < nq; g += nw) {
        const int64_t q0 = g * 64;
        const int64_t ql = q0 + lane;
        // rows past nq count 0 hits, so nothing below touches them
        const int cl = ql < nq ? counts[ql] : 0;
        const int64_t bl = ql < nq ? row_ptr[ql] : 0;
        for (int r = 0; r < 64; r += 4) {
            int32_t v0[4], v1[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int c = __shfl(cl, r + u, 64);
                const size_t off = (size_t)(q0 + r + u) * CSR_POOL;
                const bool fits = c <= CSR_POOL;
                v0[u] = (fits && lane < c) ? pool[off + lane] : 0;
                v1[u] = (fits && lane + 64 < c) ? pool[off + lane + 64] : 0;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int c = __shfl(cl, r + u, 64);
                const int64_t base = __shfl(bl, r + u, 64);
                if (c > CSR_POOL) continue;
                if (lane < c && base + lane < col_cap) cols[base + lane] = v0[u];
                if (lane + 64 < c && base + lane + 64 < col_cap) cols[base + lane + 64] = v1[u];
            }
        }
    }
}

// Lists the queries with more hits than the pool holds.
__global__ __launch_bounds__(256) void csr_overflow_kernel(const int32_t *__restrict__ counts,
                                                           int nq, QueryMap qm) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    append_slots(qm, __ballot(q < nq && counts[q] > CSR_POOL), q);
}

int scan_entry(hipStream_t s, const int32_t *counts, int nq, int64_t *row_ptr);

template <typename T>
static int range_csr_t(hipStream_t s, const ft_tree &tree, const RangeSrc<T> &src, int nq,
                       int64_t *row_ptr, int32_t *(*cols_for)(int64_t total, void *ctx), void *ctx,
                       int64_t col_cap, int64_t *total_out) {
    int32_t *counts = nullptr, *pool = nullptr;
    FT_HIP(hipMallocAsync((void **)&counts, (size_t)nq * 4, s));
    // Without room for the pool: a counting walk now and a filling walk later.
    if (hipMallocAsync((void **)&pool, (size_t)nq * CSR_POOL * 4, s) != hipSuccess) {
        (void)hipGetLastError();
        pool = nullptr;
    }
    auto release = [&]() {
        (void)hipFreeAsync(counts, s);
        if (pool) (void)hipFreeAsync(pool, s);
    };
    int rc = range_launch<T>(s, tree, src, nq,
                             RangeOut{pool, counts, pool ? CSR_POOL : 0, nullptr, nullptr, 0});
    if (rc == FT_OK) rc = scan_entry(s, counts, nq, row_ptr);
    int64_t total = 0;
    if (rc == FT_OK && hipMemcpyAsync(&total, row_ptr + nq, 8, hipMemcpyDeviceToHost, s) != hipSuccess)
        rc = fail(FT_EHIP, "CSR range query: reading the total failed");
    if (rc == FT_OK && hipStreamSynchronize(s) != hipSuccess)
        rc = fail(FT_EHIP, "CSR range query: synchronize failed");
    if (rc == FT_OK) *total_out = total;
    if (rc == FT_OK && total > col_cap)
        rc = fail(FT_ERANGE, "CSR column capacity is smaller than the number of hits");
    int32_t *cols = nullptr;
    if (rc == FT_OK) {
        cols = cols_for(total, ctx);
        if (!cols) rc = fail(FT_ENOMEM, "CSR range query: column buffer");
    }
    const RangeOut fill{nullptr, nullptr, 0, row_ptr, cols, col_cap};
    if (rc == FT_OK && !pool) {
        rc = range_launch<T>(s, tree, src, nq, fill);
    } else if (rc == FT_OK) {
        hipLaunchKernelGGL(csr_copy_kernel, dim3(std::min<unsigned>(blocks_for((nq + 63) / 64, 4), 16384u)),
                           dim3(256), 0, s, (const int32_t *)pool, (const int32_t *)counts,
                           (const int64_t *)row_ptr, nq, cols, col_cap);
        rc = rerun_ensure(s, (size_t)nq);
        if (rc == FT_OK) {
            // the longer rows, one wave per query
            const RerunBuf &rr = stream_bufs(s).rr;
            const QueryMap qm{nullptr, rr.list, rr.count, nullptr};
            const DTree<T> dt = make_dtree<T>(tree);
            hipLaunchKernelGGL(zero_counts_kernel, dim3(1), dim3(256), 0, s, rr.count,
                               (int32_t *)nullptr, 0);
            hipLaunchKernelGGL(csr_overflow_kernel, dim3(blocks_for(nq, 256)), dim3(256), 0, s,
                               (const int32_t *)counts, nq, qm);
            const dim3 g(xcd_grid(std::min<unsigned>(blocks_for(nq, 4), 2048u))), b(256);
            FT_BY_METRIC(dt, hipLaunchKernelGGL((range_wave_kernel<T, MK, true>), g, b, 0, s, dt,
                                                src, nq, qm, fill));
            if (hipGetLastError() != hipSuccess) rc = fail(FT_EHIP, "CSR range query: launch failed");
        }
    }
    release();
    return rc;
}

int range_csr_entry(hipStream_t s, const ft_tree *tree, const void *qx, const void *qy,
                    const void *qz, const void *rmin, const void *rmax, int nq, int64_t *row_ptr,
                    int32_t *(*cols_for)(int64_t total, void *ctx), void *ctx, int64_t col_cap,
                    int64_t *total) {
    int rc = FT_OK;
    FT_DISPATCH_COORD(tree->coord_type,
                      rc = range_csr_t<T>(s, *tree,
                                          RangeSrc<T>{(const T *)qx, (const T *)qy, (const T *)qz,
                                                      (const T *)rmin, (const T *)rmax},
                                          nq, row_ptr, cols_for, ctx, col_cap, total));
    return rc;
}

int scan_entry(hipStream_t s, const int32_t *counts, int nq, int64_t *row_ptr) {
    const int nb = (nq + 1023) / 1024;
    int64_t *sums = nullptr;
    FT_HIP(hipMallocAsync((void **)&sums, (size_t)(nb > 0 ? nb : 1) * 8, s));
    if (nq > 0) {
        hipLaunchKernelGGL(scan_block_kernel, dim3(nb), dim3(256), 0, s, counts, nq, row_ptr, sums);
        hipLaunchKernelGGL(scan_totals_kernel, dim3(1), dim3(1024), 0, s, sums, nb, row_ptr, nq);
        hipLaunchKernelGGL(scan_add_kernel, dim3(blocks_for(nq, 256)), dim3(256), 0, s, row_ptr,
                           nq, (const int64_t *)sums);
    } else {
        FT_HIP(hipMemsetAsync(row_ptr, 0, 8, s));
    }
    FT_CHECK_LAUNCH();
    FT_HIP(hipFreeAsync(sums, s));
    return FT_OK;
}

}  // namespace ft
