// Push levels inside one launch: what the small-frontier kernel and the
// batched BFS share.  A team of co-resident workgroups (kListBlock threads)
// runs push levels with one barrier each:
//   - a workgroup's own part of a frontier is a list of its edges in LDS
//     (PushLds); vertices with more than kListDeg out-edges, and those beyond
//     the list's capacity, go to a queue in memory that the team shares;
//   - the found vertices go to a list in memory, in per-workgroup
//     reservations, off the levels' critical path;
//   - the barrier's arrivals carry the level's three counts (found vertices,
//     their out-edges, shared-queue entries).
// The small-frontier kernel's comment has the reasons and the figures.
#pragma once
#include "dev_common.h"

// The threads of a workgroup are the including file's choice (PUSH_LIST_BLOCK);
// the list has 1 024 edges either way.
#ifndef PUSH_LIST_BLOCK
#error "PUSH_LIST_BLOCK: threads of a workgroup"
#endif

namespace {

constexpr int kListBlock = PUSH_LIST_BLOCK;
constexpr int kListWaves = kListBlock / 64;
constexpr int kListPer = 1024 / kListBlock;          // own edges per thread
constexpr int kListEdges = kListPer * kListBlock;    // edges of the LDS list
constexpr int kListDeg = 32;                         // most out-edges of a listed vertex
constexpr int kListSlack = 64, kListKeep = 32;       // see list_cap
constexpr int kSharePer = 2048 / kListBlock;         // shared-queue edges per thread and window
constexpr int kShareEdges = kSharePer * kListBlock;
constexpr int kFound = 2048;                         // found-list entries reserved at a time
static_assert(kFound >= kListEdges && kFound >= kShareEdges, "a window finds at most one reservation more");

struct PushLds {
    // the next level's own edges: entry in push_col (-1: none) and source id
    int32_t ecol[kListEdges];
    uint32_t eou[kListEdges];
    // a staged part of the shared queue
    int64_t pre[kListBlock], start[kListBlock];
    uint32_t ou[kListBlock];
    int64_t scan[kListWaves];
    // per level parity: listed edges << 32 | found; their out-edges; spilled
    unsigned long long cnt[2], edges[2], spill[2];
    unsigned long long arrive[3]; // what the workgroup's arrival carries
    unsigned long long tot[3];    // the team's sums
    int64_t chunk[2];             // found-list reservations in use, by number & 1
    int64_t reserved;             // reservations made so far
    int ok;
};

// The memory of the levels: `visited` as it was at the launch (null: the keys
// alone decide), the keys, the found list and its reservation counter.
struct PushMem {
    const uint64_t *visited;
    unsigned long long *key;
    int32_t *found;
    unsigned long long *reserve;
};

// The team's barrier: slot[set][word][workgroup], `stride` workgroups apart.
struct TeamSlots {
    unsigned long long *slot;
    unsigned int *error;
    int32_t stride, members, rank;
    uint32_t spin_limit;
};

// One edge of a lane: target position, the source's id, the filters (the
// target's visited word and its key's level) and the target's row and id.
// Every field is one register: of 64-bit entries only the half that matters
// is loaded (stored entries are fewer than 2^31).
struct PushEdge {
    bool act;
    int32_t v, start, end;
    uint32_t ou, ro, vis, level;
};

// The thread's index, opaque to the compiler: what a function below derives
// from it is computed there.  Hoisted out of the level loops, as it otherwise
// is, it fills the registers of a kernel that has other phases and is spilled
// (in the batched kernel about 70 registers, reloaded on every level).
__device__ __forceinline__ int here_tid()
{
    int t = (int)threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

__device__ __forceinline__ void list_reset(PushLds &S)
{
    if (threadIdx.x < 2) {
        S.cnt[threadIdx.x] = S.edges[threadIdx.x] = S.spill[threadIdx.x] = 0;
        S.chunk[threadIdx.x] = 0;
    }
    if (threadIdx.x == 0) {
        S.ok = 1;
        S.reserved = 0;
    }
}

__device__ __forceinline__ void edge_filters(const PushMem &M, PushEdge &e)
{
    e.vis = e.act && M.visited ? reinterpret_cast<const uint32_t *>(M.visited)[e.v >> 5] : 0u;
    e.level = e.act ? reinterpret_cast<const uint32_t *>(M.key)[2 * (int64_t)e.v + 1] : 0u;
}

__device__ __forceinline__ void edge_row(const albd_graph &g, bool act, PushEdge &e)
{
    const int32_t *ptr = reinterpret_cast<const int32_t *>(g.push_ptr);
    e.start = act ? ptr[2 * (int64_t)e.v] : 0;
    e.end = act ? ptr[2 * (int64_t)e.v + 2] : 0;
    e.ro = act ? (uint32_t)g.row_order[e.v] : 0u;
}

// Relax a window of edges (every lane of the wave calls): won lanes are their
// vertices' discoverers; f gets their numbers among the level's found.  LATE:
// the targets' rows are loaded here, for the won ones only.
template <int PER, bool LATE>
__device__ __forceinline__ void relax_edges(PushLds &S, const albd_graph &g, const PushMem &M, PushEdge (&e)[PER],
                                            uint32_t lvl, int par, int cap, unsigned long long *spill_ctr,
                                            int32_t *qb, bool (&won)[PER], uint32_t (&f)[PER], bool &spilled)
{
    const int lane = here_tid() & 63;
    uint64_t sm[PER]; // lanes whose vertex goes to the shared queue
    unsigned int spills = 0;
    // a full list stays full to the level's end
    const bool full = __builtin_amdgcn_readfirstlane((S.cnt[par] >> 32) >= (unsigned long long)cap ? 1 : 0) != 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        won[i] = false;
        // unvisited at the launch and not found at an earlier level of it
        if (e[i].act && !((e[i].vis >> (e[i].v & 31)) & 1u) && e[i].level >= lvl)
            won[i] = atomicMin(&M.key[e[i].v], ((unsigned long long)lvl << 32) | e[i].ou) == ~0ull;
    }
    if constexpr (LATE) {
#pragma unroll
        for (int i = 0; i < PER; ++i) edge_row(g, won[i], e[i]);
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const uint64_t m = __ballot(won[i]);
        f[i] = 0;
        sm[i] = 0;
        if (m == 0) continue; // wave-uniform
        const int32_t deg = won[i] ? e[i].end - e[i].start : 0;
        const bool listed = !full && deg > 0 && deg <= kListDeg;
        // exclusive prefix of the listed degrees, bit by bit
        uint32_t pre = 0, tot = 0;
        if (!full) {
#pragma unroll
            for (int b = 0; b < 6; ++b) {
                const uint64_t mb = __ballot(listed && ((deg >> b) & 1));
                pre += (uint32_t)__popcll(mb & lanemask_lt(lane)) << b;
                tot += (uint32_t)__popcll(mb) << b;
            }
        }
        static_assert(kListDeg < 64, "six bits hold a listed degree");
        const unsigned long long es = wave_sum((unsigned long long)(uint32_t)deg);
        unsigned long long base = 0;
        if (lane == 0) {
            base = atomicAdd(&S.cnt[par], ((unsigned long long)tot << 32) | (unsigned long long)__popcll(m));
            if (es) atomicAdd(&S.edges[par], es);
        }
        base = uniform64(base); // lane 0's
        f[i] = (uint32_t)base + (uint32_t)__popcll(m & lanemask_lt(lane));
        const unsigned long long e0 = (base >> 32) + pre;
        const bool fits = listed && e0 + (unsigned long long)deg <= (unsigned long long)cap;
        if (listed)
            for (int k = 0; k < deg; ++k) {
                if (e0 + k >= (unsigned long long)cap) break;
                S.ecol[e0 + k] = fits ? e[i].start + k : -1;
                S.eou[e0 + k] = e[i].ro;
            }
        sm[i] = __ballot(deg > 0 && !fits);
        spills += (unsigned int)__popcll(sm[i]);
    }
    if (spills == 0) return;
    // one reservation per wave and window: same-address atomics serialise
    unsigned long long q = 0;
    if (lane == 0) {
        q = atomicAdd(spill_ctr, (unsigned long long)spills);
        atomicAdd(&S.spill[par], (unsigned long long)spills);
    }
    q = uniform64(q); // lane 0's
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        if ((sm[i] >> lane) & 1ull) st_coherent(&qb[q + __popcll(sm[i] & lanemask_lt(lane))], e[i].v);
        q += (unsigned long long)__popcll(sm[i]);
    }
    spilled = true;
}

// the workgroup's found vertices of one window -> its reservations; F: found
// before this level (a barrier after reserve_found comes first)
template <int PER>
__device__ __forceinline__ void store_found(const PushLds &S, int32_t *found, const PushEdge (&e)[PER],
                                            const bool (&won)[PER], const uint32_t (&f)[PER], int64_t F)
{
#pragma unroll
    for (int i = 0; i < PER; ++i)
        if (won[i]) {
            const int64_t at = F + f[i];
            st_coherent(&found[S.chunk[(at / kFound) & 1] + at % kFound], e[i].v);
        }
}

// room for a window's found vertices after the first `at` (thread 0)
__device__ __forceinline__ void reserve_found(PushLds &S, const PushMem &M, int64_t at)
{
    while (S.reserved < at / kFound + 2) {
        S.chunk[S.reserved & 1] = (int64_t)atomicAdd(M.reserve, (unsigned long long)kFound);
        ++S.reserved;
    }
}

// the unused ends of the workgroup's reservations hold no vertex (F: found so
// far; the found list has room for `cap` entries)
__device__ __forceinline__ void end_found(const PushLds &S, const PushMem &M, int64_t F, int64_t cap)
{
    for (int64_t j = F + here_tid(); j < S.reserved * kFound; j += kListBlock) {
        const int64_t at = S.chunk[(j / kFound) & 1] + j % kFound;
        if (at < cap) st_coherent(&M.found[at], (int32_t)-1);
    }
}

// The team's share of the queue in memory qa[0, ns): the workgroup expands
// entries [rank * ns / T ...) in windows.  The targets' rows are loaded for
// the vertices found only: most edges of a large frontier find nothing.
__device__ __forceinline__ void push_shared(PushLds &S, const albd_graph &g, const PushMem &M, const int32_t *qa,
                                            int64_t ns, int rank, int T, uint32_t lvl, int par, int cap,
                                            unsigned long long *spill_ctr, int32_t *qb, int64_t F, bool &spilled)
{
    const int tid = here_tid();
    const int64_t per = (ns + T - 1) / T;
    const int64_t q0 = (int64_t)rank * per, q1 = q0 + per < ns ? q0 + per : ns;
    for (int64_t base = q0; base < q1; base += kListBlock) { // uniform in the workgroup
        const int cnt_e = (int)(q1 - base < kListBlock ? q1 - base : kListBlock);
        int64_t a0 = 0, a1 = 0;
        uint32_t o0 = 0;
        if (tid < cnt_e) {
            const int32_t u = ld_coherent(&qa[base + tid]);
            a0 = g.push_ptr[u];
            a1 = g.push_ptr[u + 1];
            o0 = (uint32_t)g.row_order[u];
        }
        int64_t total;
        const int64_t ex = block_scan_excl<kListBlock>(a1 - a0, &total, S.scan);
        S.pre[tid] = ex;
        S.start[tid] = a0;
        S.ou[tid] = o0;
        for (int64_t wb = 0; wb < total; wb += kShareEdges) { // uniform
            // every found of the earlier windows has its place
            __syncthreads();
            if (tid == 0) reserve_found(S, M, F + (int64_t)(S.cnt[par] & 0xffffffffull));
            __syncthreads();
            // consecutive edges per thread: one search, then a walk
            PushEdge x[kSharePer];
            int64_t en = wb + (int64_t)tid * kSharePer;
            const int64_t end = en + kSharePer < total ? en + kSharePer : total;
            int lo = 0;
            if (en < end) {
                int hi = cnt_e;
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (S.pre[mid] <= en) lo = mid;
                    else hi = mid;
                }
            }
#pragma unroll
            for (int i = 0; i < kSharePer; ++i) {
                x[i].act = en < end;
                x[i].v = 0;
                x[i].ou = 0;
                if (x[i].act) {
                    while (lo + 1 < cnt_e && S.pre[lo + 1] <= en) ++lo;
                    x[i].v = g.push_col[S.start[lo] + (en - S.pre[lo])];
                    x[i].ou = S.ou[lo];
                    ++en;
                }
            }
#pragma unroll
            for (int i = 0; i < kSharePer; ++i) edge_filters(M, x[i]);
            bool xw[kSharePer];
            uint32_t xf[kSharePer];
            relax_edges<kSharePer, true>(S, g, M, x, lvl, par, cap, spill_ctr, qb, xw, xf, spilled);
            store_found<kSharePer>(S, M.found, x, xw, xf, F);
        }
        __syncthreads(); // the staged entries are replaced
    }
}

// Load everything about the list's `count` edges but the atomic.
__device__ __forceinline__ void load_list(const PushLds &S, const albd_graph &g, const PushMem &M, int count,
                                          PushEdge (&e)[kListPer])
{
    const int tid = here_tid();
#pragma unroll
    for (int i = 0; i < kListPer; ++i) {
        const int en = i * kListBlock + tid;
        const int32_t at = en < count ? S.ecol[en] : -1;
        e[i].act = at >= 0;
        e[i].ou = e[i].act ? S.eou[en] : 0;
        e[i].v = e[i].act ? g.push_col[at] : 0;
    }
#pragma unroll
    for (int i = 0; i < kListPer; ++i) {
        edge_filters(M, e[i]);
        edge_row(g, e[i].act, e[i]);
    }
}

// edges the list takes at the next level: a workgroup that holds more than
// twice its part of the level's edges keeps half a part of what it finds next
// and shares the rest
__device__ __forceinline__ int list_cap(int64_t mine, int64_t edges, int T)
{
    const int64_t part = edges / T;
    if (mine <= 2 * part + kListSlack) return kListEdges;
    return (int)(part / 2 < kListKeep ? kListKeep : (part / 2 > kListEdges ? kListEdges : part / 2));
}

// Arrival at the barrier (three lanes of one wave): S.arrive, tagged.  The
// slots alternate between two sets by the tag: a set is written again only
// two barriers later, when every workgroup has passed the one after reading
// it; tags count up and wrap, so a stale one never equals the awaited.
__device__ __forceinline__ void team_arrive(PushLds &S, const TeamSlots &B, unsigned int tag)
{
    const int lane = here_tid() & 63;
    if (B.members == 1) {
        if (lane < 3) S.tot[lane] = S.arrive[lane]; // nobody to wait for
    } else if (lane < 3)
        st_coherent(&B.slot[((tag & 1) * 3 + lane) * B.stride + B.rank],
                    ((unsigned long long)(tag & 0xffffu) << 48) | S.arrive[lane]);
}

// wait for every workgroup's arrival with `tag`; the wave sums word `k`
__device__ __forceinline__ void team_poll(PushLds &S, const TeamSlots &B, int k, unsigned int tag)
{
    if (B.members == 1) return;
    const int lane = here_tid() & 63;
    const unsigned long long *slot = &B.slot[((tag & 1) * 3 + k) * B.stride];
    unsigned long long sum = 0;
    bool ok = true;
    for (uint32_t spins = 0;; ++spins) {
        bool all = true;
        sum = 0;
        for (int i = lane; i < B.members; i += 64) {
            const unsigned long long x = ld_coherent(&slot[i]);
            all = all && (x >> 48) == (tag & 0xffffu);
            sum += x & ((1ull << 48) - 1);
        }
        if (__ballot(!all) == 0) break;
        if (spins >= B.spin_limit || ((spins & 63) == 63 && ld_coherent(B.error) != 0)) {
            ok = false;
            break;
        }
    }
    sum = wave_sum(sum);
    if (lane == 0) {
        S.tot[k] = sum;
        if (!ok) {
            atomicOr(B.error, 1u);
            S.ok = 0;
        }
    }
}

// The barrier off the critical path: every memory operation of the workgroup
// before it is done when it arrives; x, y, z (thread 0's) are its counts.
__device__ __forceinline__ bool team_barrier(PushLds &S, const TeamSlots &B, unsigned int tag,
                                             unsigned long long x = 0, unsigned long long y = 0,
                                             unsigned long long z = 0)
{
    const int tid = here_tid(), poll = (tid >> 6) - (kListWaves - 3);
    __builtin_amdgcn_s_waitcnt(0);
    if (tid == 0) {
        S.arrive[0] = x;
        S.arrive[1] = y;
        S.arrive[2] = z;
    }
    __syncthreads();
    if (poll == 0) team_arrive(S, B, tag);
    if (poll >= 0) team_poll(S, B, poll, tag);
    __syncthreads();
    return S.ok != 0;
}

} // namespace
