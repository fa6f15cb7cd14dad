// Batched BFS: many instances (graphs and roots of uneven size) in one
// persistent launch of co-resident workgroups.  The workgroups are split into teams; a team runs the
// complete level loop of its instances one after the other, with one team
// barrier per level and the direction of every level chosen on the device
// (the reference heuristic, bfs/src/bfs_SELLCSv2.c:282-284, or the learned
// selector's MLP), so no instance ever waits for the host.
//
// Exactness, as in the small-frontier kernel: every position has a 64-bit
// key (level << 32 | parent id), all ones at rest.  A push edge u -> v at
// level L does atomicMin(key[v], L << 32 | id(u)); a pull lane that finds
// its row's first frontier neighbour u does the same.  The key keeps the
// smallest (level, parent) pair, so it holds the BFS level and the min-id
// parent no matter in which order the team's waves run, and the old value
// names the one discoverer.
//
// Push levels run as in the small-frontier kernel (push_lists.h): lists of
// edges in LDS, a shared queue (in the result arrays, which are written at the
// end only), one barrier that carries the counts, and no bitmaps.  What bounds
// the batch is its grids' thousands of levels: bitmaps set by the discoverers,
// a queue in memory with its reservations and a counting barrier cost the
// largest grid of a 24-instance mix 16.9 us a level where these take 5.2 (the
// launch 45 -> 14 ms; 96 instances 66 -> 25, 256 instances 111 -> 62 ms).
//
// The kernel has phases with nothing in common, and values that the compiler
// hoisted out of one were spilled in the others: the thread's index is taken
// anew in each (here_tid), the push levels' registers live in a loop of their
// own, the descriptor comes through scalar loads and the selector's logarithm
// is a call.  79 spilled registers -> 33 took the push levels from 5.9 to 4.5
// us and one workgroup's RMAT s20 search from 63 to 50 ms.
//
// A pull needs the frontier bitmap and the visited one: the found list since
// the last pull gives both (materialize), once per turn from push to pull.
// Bitmaps rotate over three buffers: a pull reads one, sets the next and
// clears the one before; all are clean while levels push.
#include "dev_common.h"
// 512 threads, two workgroups a CU: 1 024 take a batch of 24 from 16.9 to 15.8 ms,
// and one of 256 from 63 to 85, which then has half the teams
#define PUSH_LIST_BLOCK 512
#include "push_lists.h"
#include "select_dev.h"
#include "../../../include/albba.h"

namespace {

constexpr int kBB = kListBlock; // threads per workgroup
constexpr int kBWaves = kListWaves;

struct BLds {
    PushLds l;
    unsigned long long red[3][kBWaves];
    unsigned int s_cnt[kBWaves];
    unsigned long long s_base;
    int choice;
    float params[ALBBA_MLP_NPARAM];
    float xs[ALBBA_MLP_IN], h1[ALBBA_MLP_H1], h2[ALBBA_MLP_H2], ys[ALBBA_MLP_OUT];
};

__device__ __forceinline__ unsigned int *err_flag(const albd_batch_item &it)
{
    return reinterpret_cast<unsigned int *>(&it.ctl[2]);
}

// sums of one value per thread over the workgroup, to thread 0
__device__ __forceinline__ unsigned long long block_sum(BLds &S, int row, unsigned long long x)
{
    x = wave_sum(x);
    if (lane_id() == 0) S.red[row][threadIdx.x >> 6] = x;
    __syncthreads();
    unsigned long long t = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < kBWaves; ++i) t += S.red[row][i];
    return t;
}

// One BFS of one instance by a team of T workgroups (this one is `rank`).
// Returns false when a team barrier gave up.
__device__ bool run_instance(BLds &S, const albd_batch_item &it, int rank, int T, bool learned,
                             uint32_t spin_limit)
{
    const albd_graph &g = it.g;
    const int tid = threadIdx.x;
    const int64_t gthreads = (int64_t)T * kBB;
    // the thread's number in the team, worked out where a phase begins
    auto team_tid = [&]() -> int64_t { return (int64_t)rank * kBB + here_tid(); };
    const int64_t nwords = g.nwords;
    PushLds &L = S.l;
    const TeamSlots B{it.slot, err_flag(it), ALBD_BATCH_TEAM_MAX, T, rank, spin_limit};
    unsigned int tag = 0;
    const bool leader = rank == 0 && tid == 0;
    if (leader) st_coherent(reinterpret_cast<long long *>(&it.ctl[ALBD_RES_T0]), (long long)wall_clock64());
    for (int64_t i = team_tid(); i < nwords; i += gthreads) {
        st_coherent(&it.visited[i], (uint64_t)0);
        st_coherent(&it.bm[0][i], (uint64_t)0);
        st_coherent(&it.bm[1][i], (uint64_t)0);
        st_coherent(&it.bm[2][i], (uint64_t)0);
    }
    list_reset(L);
    // the found list's reservations: counters 0 and 1 in turn, from one
    // materialize to the next
    unsigned long long *next_reserve = &it.ctl[3];
    PushMem M{nullptr, it.key, it.found, &it.ctl[1]};
    const int64_t found_cap = (int64_t)ALBD_BATCH_FOUND(g.npos, T);
    __syncthreads();
    if (tid == 0) reserve_found(L, M, 0);
    int32_t *qa = it.level, *qb = it.parent; // the shared queues
    const int32_t rp = g.pos_of[it.root];
    const int64_t rdeg = g.push_ptr[rp + 1] - g.push_ptr[rp];
    if (leader) {
        // the root: level 0, its own parent, the queue and the found list
        st_coherent(&it.key[rp], (unsigned long long)(uint32_t)it.root);
        st_coherent(&qa[0], rp);
        st_coherent(&it.found[L.chunk[0]], rp);
    }
    int64_t F = rank == 0 ? 1 : 0; // in this workgroup's reservations
    if (!team_barrier(L, B, ++tag)) return false;

    // team-uniform loop state
    unsigned long long Fr = 1, mf = (unsigned long long)rdeg, nzw = 1, F_prev = 0;
    unsigned long long reached = 1, redges = (unsigned long long)rdeg;
    int prev_choice = ALBBA_CHOICE_PUSH;
    int64_t ns = 1;         // the shared queue's length
    int cap = kListEdges;   // edges the workgroup's list takes
    bool lists = true;      // the frontier is in the lists and the queue
    bool bitmap = false;    // it is in bcur, and visited is up to date
    bool old_dirty = false; // bold holds an older frontier
    // the bitmaps (pointers that rotate: an index into the descriptor's array
    // would put the descriptor into scratch memory)
    uint64_t *bcur = it.bm[0], *bnext = it.bm[1], *bold = it.bm[2];
    int listed = 0;         // edges of the workgroup's list
    long long pushes = 0, pulls = 0;
    const long long thr = (long long)(int)((double)g.n * 0.04);
    // Whether a level is anything but a plain push.  The heuristic pulls when
    // the frontier is large by its count.  A batched pull visits every word of
    // the instance with the team's few workgroups, so the learned selector is
    // consulted only then, or when the frontier's out-edges reach 1/16 of the
    // unexplored edges.
    auto decide = [&](unsigned long long f, unsigned long long edges, unsigned long long seen) -> bool {
        if ((long long)f > thr) return true;
        const unsigned long long unexplored = (unsigned long long)g.nnz > seen ? (unsigned long long)g.nnz - seen : 0ull;
        return learned && 16 * edges >= unexplored;
    };
    int Lv = 0;
    while (Fr > 0) {
        // direction of this level (the same in every workgroup of the team)
        int choice = (long long)Fr > thr ? ALBBA_CHOICE_PULL_SB : ALBBA_CHOICE_PUSH;
        const bool consult = learned && decide(Fr, mf, redges);
        if ((consult || choice != ALBBA_CHOICE_PUSH) && !bitmap) {
            // materialize: the vertices found since the last time into
            // visited, those of this level into the frontier bitmap
            __syncthreads(); // the reservation made since the last level
            end_found(L, M, F, found_cap);
            if (!team_barrier(L, B, ++tag)) return false;
            int64_t total = (int64_t)ld_coherent(M.reserve);
            if (total > found_cap) total = found_cap;
            unsigned long long my_w = 0;
            for (int64_t i = team_tid(); i < total; i += gthreads) {
                const int32_t v = ld_coherent(&it.found[i]);
                if (v < 0) continue;
                const uint64_t bit = 1ull << (v & 63);
                atomicOr(reinterpret_cast<unsigned long long *>(&it.visited[v >> 6]), bit);
                if ((uint32_t)(ld_coherent(&it.key[v]) >> 32) == (uint32_t)Lv)
                    my_w += atomicOr(reinterpret_cast<unsigned long long *>(&bcur[v >> 6]), bit) == 0 ? 1 : 0;
            }
            const unsigned long long w = block_sum(S, 0, my_w);
            if (!team_barrier(L, B, ++tag, w)) return false;
            nzw = uniform64(L.tot[0]);
            bitmap = true;
            // a fresh found list, by the other counter
            if (leader) st_coherent(M.reserve, 0ull);
            unsigned long long *t = M.reserve;
            M.reserve = next_reserve;
            next_reserve = t;
            F = 0;
            __syncthreads();
            if (tid == 0) {
                L.reserved = 0;
                reserve_found(L, M, 0);
            }
            __syncthreads();
        }
        if (consult) {
            if (tid < 64)
                level_features<true>(S.xs, g.n, g.nnz, nwords, Fr, mf, nzw, reached, redges, Lv,
                                     prev_choice, F_prev);
            __syncthreads();
            const int c = mlp_argmin(S.params, S.xs, S.h1, S.h2, S.ys, 0xF, &S.choice);
            if (c >= 0) choice = c;
        }
        if (choice == ALBBA_CHOICE_PUSH) {
            if (!lists) {
                // the frontier came from a pull: list its vertices from the
                // bitmap, one reservation per block step, and leave every
                // bitmap clean
                const int tid = here_tid(), lane = tid & 63, wid = tid >> 6;
                unsigned long long mine = 0; // thread 0's
                for (int64_t wb = (int64_t)rank * kBB; wb < nwords; wb += gthreads) {
                    const int64_t w = wb + tid;
                    const uint64_t word = w < nwords ? ld_coherent(&bcur[w]) : 0ull;
                    if (word) st_coherent(&bcur[w], (uint64_t)0);
                    if (old_dirty && w < nwords) st_coherent(&bold[w], (uint64_t)0);
                    unsigned long long wtot;
                    const unsigned long long ex =
                        wave_exclusive_scan<unsigned long long>((unsigned long long)__popcll(word), &wtot);
                    if (lane == 0) S.s_cnt[wid] = (unsigned int)wtot;
                    __syncthreads();
                    if (tid == 0) {
                        unsigned long long tot = 0;
                        for (int i = 0; i < kBWaves; ++i) tot += S.s_cnt[i];
                        S.s_base = tot ? atomicAdd(&it.ctl[8 + (pushes & 3)], tot) : 0ull;
                        mine += tot;
                    }
                    __syncthreads();
                    unsigned long long o = S.s_base + ex;
                    for (int i = 0; i < wid; ++i) o += S.s_cnt[i];
                    __syncthreads();
                    uint64_t kb = word;
                    while (kb) {
                        const int b = __ffsll((unsigned long long)kb) - 1;
                        kb &= kb - 1;
                        st_coherent(&qa[o++], (int32_t)(w * 64 + b));
                    }
                }
                if (!team_barrier(L, B, ++tag, mine)) return false;
                ns = (int64_t)uniform64(L.tot[0]);
                cap = kListEdges;
                listed = 0;
                lists = true;
                old_dirty = false;
            } else if (bitmap) {
                // materialized for the selector, which pushes all the same
                for (int64_t i = team_tid(); i < nwords; i += gthreads) st_coherent(&bcur[i], (uint64_t)0);
            }
            bitmap = false;
            // push levels, as long as nothing else is to be decided: the
            // edges' registers live in this loop only
            PushEdge e[kListPer];
            load_list(L, g, M, listed, e);
            do {
                const int wid = here_tid() >> 6, lane = here_tid() & 63;
                // the waves that poll: the last ones, which hold the fewest edges
                const int poll = wid - (kBWaves - 3);
                const int par = (int)(pushes & 1);
                // this push level's counter of entries put on the shared
                // queue; that of two push levels ahead, and the one of listing
                // a bitmap, are free (their last users passed a barrier) and
                // start from zero
                unsigned long long *spill_ctr = &it.ctl[4 + (pushes & 3)];
                if (leader) {
                    st_coherent(&it.ctl[4 + ((pushes + 2) & 3)], 0ull);
                    st_coherent(&it.ctl[8 + ((pushes + 2) & 3)], 0ull);
                }
                ++pushes;
                if (tid == 0) L.cnt[par ^ 1] = L.edges[par ^ 1] = L.spill[par ^ 1] = 0;
                bool won[kListPer], spilled = false;
                uint32_t f[kListPer];
                const uint32_t lvl = (uint32_t)(Lv + 1);
                relax_edges<kListPer, false>(L, g, M, e, lvl, par, cap, spill_ctr, qb, won, f, spilled);
                if (ns > 0) {
                    __syncthreads(); // the reservation made since the last level
                    store_found<kListPer>(L, it.found, e, won, f, F);
                    push_shared(L, g, M, qa, ns, rank, T, lvl, par, cap, spill_ctr, qb, F, spilled);
                }
                // the shared queue's entries and the leader's zeros are in
                // place before the arrival
                if (spilled || (rank == 0 && wid == 0)) __builtin_amdgcn_s_waitcnt(0);
                __syncthreads();
                if (poll == 0) {
                    if (lane < 3)
                        L.arrive[lane] =
                            lane == 0 ? (L.cnt[par] & 0xffffffffull) : (lane == 1 ? L.edges[par] : L.spill[par]);
                    team_arrive(L, B, tag + 1);
                }
                if (ns == 0) store_found<kListPer>(L, it.found, e, won, f, F);
                const unsigned long long mine = uniform64(L.cnt[par]);
                F += (int64_t)(mine & 0xffffffffull);
                listed = (int)((mine >> 32) < (unsigned long long)cap ? (mine >> 32) : (unsigned long long)cap);
                load_list(L, g, M, listed, e);
                if (poll >= 0) team_poll(L, B, poll, tag + 1);
                ++tag;
                __syncthreads();
                if (!L.ok) return false;
                F_prev = Fr;
                Fr = uniform64(L.tot[0]);
                mf = uniform64(L.tot[1]);
                ns = (int64_t)uniform64(L.tot[2]);
                if (tid == 0) reserve_found(L, M, F);
                cap = list_cap((int64_t)(mine >> 32), (int64_t)mf, T);
                int32_t *t = qa;
                qa = qb;
                qb = t;
                reached += Fr;
                redges += mf;
                ++Lv;
            } while (Fr > 0 && !decide(Fr, mf, redges));
            prev_choice = ALBBA_CHOICE_PUSH;
        } else {
            ++pulls;
            const int lane = here_tid() & 63, wid = here_tid() >> 6;
            unsigned long long my_f = 0, my_e = 0, my_w = 0;
            if (old_dirty)
                for (int64_t i = team_tid(); i < nwords; i += gthreads) st_coherent(&bold[i], (uint64_t)0);
            const unsigned long long lkey = (unsigned long long)(uint32_t)(Lv + 1) << 32;
            // pull: workgroup `rank` takes words [w0, w1) in runs of 64; wave
            // wid takes every kBWaves-th run.  The wave's lanes test the 64
            // words of a run at once (rows with a length, not visited), then the wave works through the words that have
            // such rows; their unvisited lanes look for their row's first
            // neighbour in B_L (rows list neighbours by ascending id)
            const int64_t per = (nwords + T - 1) / T;
            const int64_t w0 = (int64_t)rank * per, w1 = w0 + per < nwords ? w0 + per : nwords;
            for (int64_t run = w0 + (int64_t)wid * 64; run < w1; run += (int64_t)kBWaves * 64) {
                const int64_t wl = run + lane;
                uint64_t unres_l = 0;
                if (wl < w1) {
                    const uint64_t hl = g.haslen[wl];
                    if (hl) unres_l = hl & ~ld_coherent(&it.visited[wl]);
                }
                uint64_t todo_w = __ballot(unres_l != 0);
                while (todo_w) {
                    const int kw = __ffsll((unsigned long long)todo_w) - 1;
                    todo_w &= todo_w - 1;
                    const int64_t w = run + kw;
                    const uint64_t unres = __shfl(unres_l, kw, 64);
                    const int64_t p = w * 64 + lane;
                    int32_t par = -1;
                    if (it.mapping == ALBD_MAP_LANE_ROW) {
                        if ((unres >> lane) & 1ull) {
                            const int64_t r1 = g.pull_ptr[p + 1];
                            for (int64_t k = g.pull_ptr[p]; k < r1; ++k) {
                                const int32_t u = g.pull_col[k];
                                if ((ld_coherent(&bcur[u >> 6]) >> (u & 63)) & 1ull) {
                                    par = g.row_order[u];
                                    break;
                                }
                            }
                        }
                    } else {
                        // the wave scans one row at a time, 64 entries per step
                        uint64_t todo = unres;
                        while (todo) {
                            const int r = __ffsll((unsigned long long)todo) - 1;
                            todo &= todo - 1;
                            const int64_t rs = g.pull_ptr[w * 64 + r], re = g.pull_ptr[w * 64 + r + 1];
                            for (int64_t k = rs; k < re; k += 64) {
                                const int64_t kk = k + lane;
                                bool h = false;
                                int32_t u = 0;
                                if (kk < re) {
                                    u = g.pull_col[kk];
                                    h = (ld_coherent(&bcur[u >> 6]) >> (u & 63)) & 1ull;
                                }
                                const uint64_t hm = __ballot(h);
                                if (hm) {
                                    const int32_t first = __shfl(u, __ffsll((unsigned long long)hm) - 1, 64);
                                    if (lane == r) par = g.row_order[first];
                                    break;
                                }
                            }
                        }
                    }
                    bool won = false;
                    if (par >= 0) won = atomicMin(&it.key[p], lkey | (uint32_t)par) == ~0ull;
                    const uint64_t fm = __ballot(won);
                    if (fm) {
                        if (lane == 0) {
                            const unsigned long long old =
                                atomicOr(reinterpret_cast<unsigned long long *>(&bnext[w]), fm);
                            atomicOr(reinterpret_cast<unsigned long long *>(&it.visited[w]), fm);
                            my_w += old == 0 ? 1 : 0;
                        }
                        if (won) {
                            my_f += 1;
                            my_e += (unsigned long long)(g.push_ptr[p + 1] - g.push_ptr[p]);
                        }
                    }
                }
            }
            const unsigned long long f = block_sum(S, 0, my_f), me = block_sum(S, 1, my_e), mw = block_sum(S, 2, my_w);
            if (!team_barrier(L, B, ++tag, f, me, mw)) return false;
            F_prev = Fr;
            Fr = uniform64(L.tot[0]);
            mf = uniform64(L.tot[1]);
            nzw = uniform64(L.tot[2]);
            // the lists are of the frontier before
            lists = false;
            old_dirty = true;
            uint64_t *t = bold;
            bold = bcur;
            bcur = bnext;
            bnext = t;
            reached += Fr;
            redges += mf;
            ++Lv;
            prev_choice = ALBBA_CHOICE_PULL;
        }
    }
    // results in vertex order from the keys; the keys go back to all ones
    for (int64_t v = team_tid(); v < g.n; v += gthreads) {
        const int32_t p = g.pos_of[v];
        const unsigned long long k = ld_coherent(&it.key[p]);
        const bool hit = k != ~0ull;
        it.level[v] = hit ? (int32_t)(k >> 32) : -1;
        it.parent[v] = hit ? (int32_t)(uint32_t)k : -1;
        if (hit) st_coherent(&it.key[p], ~0ull);
    }
    if (!team_barrier(L, B, ++tag)) return false;
    if (leader) {
        long long *r = reinterpret_cast<long long *>(it.ctl);
        st_coherent(&r[ALBD_RES_LEVELS], (long long)Lv);
        st_coherent(&r[ALBD_RES_REACHED], (long long)reached);
        st_coherent(&r[ALBD_RES_EDGES], (long long)redges);
        st_coherent(&r[ALBD_RES_PUSHES], pushes);
        st_coherent(&r[ALBD_RES_PULLS], pulls);
        st_coherent(&r[ALBD_RES_T1], (long long)wall_clock64());
    }
    return true;
}

// The descriptor of an instance through the constant address space: nothing
// writes it during the launch, so that its uniform fields come as scalar loads
// into scalar registers (as ordinary memory, which the kernel's stores might
// change, each pointer took a pair of vector registers, and the push loop
// spilled).
__device__ __forceinline__ albd_batch_item load_item(const albd_batch_item *items, int32_t i)
{
    typedef const __attribute__((address_space(4))) uint32_t *ConstWords;
    constexpr int kWords = (int)(sizeof(albd_batch_item) / 4);
    static_assert(sizeof(albd_batch_item) % 4 == 0, "copied by word");
    union {
        albd_batch_item it;
        uint32_t w[kWords];
    } u;
    const ConstWords src = (ConstWords)(uintptr_t)&items[__builtin_amdgcn_readfirstlane(i)];
#pragma unroll
    for (int k = 0; k < kWords; ++k) u.w[k] = src[k];
    return u.it;
}

__global__ __launch_bounds__(kBB, 4) void k_bfs_batch(albd_batch_args a)
{
    __shared__ BLds S;
    if (a.params) mlp_to_lds<kBB>(S.params, a.params);
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(a.wg_team[blockIdx.x]);
    const int rank = (int)blockIdx.x - __builtin_amdgcn_readfirstlane(a.team_first[t]);
    const int T = __builtin_amdgcn_readfirstlane(a.team_size[t]);
    for (int j = a.team_ptr[t]; j < a.team_ptr[t + 1]; ++j) {
        const albd_batch_item it = load_item(a.items, a.team_items[j]);
        if (!run_instance(S, it, rank, T, a.params != nullptr, a.spin_limit)) {
            if (threadIdx.x == 0)
                st_coherent(reinterpret_cast<long long *>(it.ctl) + ALBD_RES_ERROR, 1ll);
            break;
        }
    }
}

// The device tables of albba_batch_run_noalloc (instance descriptors, team
// tables) live here instead of in memory allocated per run.  Each device
// holds its own copy at its own address; host code must use that address
// (from hipGetSymbolAddress), never the array's name, which in host code is
// only a stand-in.  Every run on a device shares the array: runs that
// overlap on one device race.
static __device__ __align__(256) unsigned char scratch[ALBD_BATCH_SCRATCH_BYTES];
static_assert(ALBBA_BATCH_NOALLOC_MAX * sizeof(albd_batch_item) + 256 +
                      sizeof(int32_t) * (4096 + 3 * ALBBA_BATCH_NOALLOC_MAX + 1 + ALBBA_BATCH_NOALLOC_MAX) <=
                  ALBD_BATCH_SCRATCH_BYTES,
              "the scratch holds the tables of the largest no-alloc batch (up to 4096 workgroups)");

constexpr int kMaxDevices = 64;
static void *g_scratch_ptr[kMaxDevices]; // device address of `scratch`, per device

} // namespace

extern "C" {

int albd_batch_scratch_init(int device)
{
    if (device < 0 || device >= kMaxDevices)
        return albd_set_error_msg(ALBBA_ENODEV, "batch scratch: device index beyond the table");
    if (__atomic_load_n(&g_scratch_ptr[device], __ATOMIC_ACQUIRE)) return 0;
    void *p = nullptr;
    HIPCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return albd_set_error_msg(ALBBA_EHIP, "batch scratch: no device address");
    __atomic_store_n(&g_scratch_ptr[device], p, __ATOMIC_RELEASE);
    return 0;
}

int albd_batch_scratch(albd_ctx *c, void **ptr, size_t *bytes)
{
    const int device = albd_ctx_device(c);
    void *p = device >= 0 && device < kMaxDevices ? __atomic_load_n(&g_scratch_ptr[device], __ATOMIC_ACQUIRE)
                                                  : nullptr;
    if (!p) return albd_set_error_msg(ALBBA_EHIP, "batch scratch: not set up on this device");
    *ptr = p;
    *bytes = ALBD_BATCH_SCRATCH_BYTES;
    return 0;
}

int albd_batch_capacity(albd_ctx *c, int *workgroups)
{
    int per_cu = 0;
    HIPCHK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_bfs_batch, kBB, 0));
    *workgroups = per_cu * albd_num_cus(c);
    return 0;
}

int albd_batch_launch(albd_ctx *c, const albd_batch_args *a, int32_t workgroups)
{
    // at most albd_batch_capacity workgroups, all resident at once; an
    // ordinary launch on the context's stream, which starts once the
    // stream's earlier kernels have finished (a team barrier that waited in
    // vain would give up after spin_limit polls, never hang)
    int cap = 0;
    if (int rc = albd_batch_capacity(c, &cap)) return rc;
    if (workgroups < 1 || workgroups > cap)
        return albd_set_error_msg(ALBBA_EINVAL, "batch launch: more workgroups than can be resident");
    hipLaunchKernelGGL(k_bfs_batch, dim3(workgroups), dim3(kBB), 0, albd_stream(c), *a);
    HIPCHK(hipGetLastError());
    return 0;
}

double albd_clock_ticks_per_ms(albd_ctx *c)
{
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, albd_ctx_device(c)) != hipSuccess ||
        khz <= 0)
        return 100000.0; // the 100 MHz constant clock of CDNA
    return (double)khz;
}

} // extern "C"
