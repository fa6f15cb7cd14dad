// The whole BFS of a small graph in one workgroup: every level, both
// directions, the policy's choices and the results, in one launch.
//
// What bounds a small graph's BFS in the level loop is its launches: an RMAT
// s10 search is 22 kernels of 2-6 us, 6-10 us apart, for 0.13 MB of columns.
// Here the state lives in one compute unit's LDS (parents and levels, both
// frontiers as bitmap and queue, row pointers, vertex ids), a level costs a
// few workgroup barriers, and only columns are read from memory: the search
// takes 25 us where the loop took 146.  Past ALBD_ONE_NPOS vertices the state
// would not fit the LDS; at ALBD_ONE_NNZ entries one compute unit's reads come
// near the launches saved (8 000 vertices of mean degree 24, three pulls that
// scan every row: 163 against 191 us; RMAT s13 of 15: 56 against 155; a grid
// of 90 x 90: 441 against 1 558).
//
// Exactness: key = level << 13 | parent id, all ones while unvisited; a push
// edge does an LDS atomicMin, so that a vertex keeps its BFS level and, in
// it, the smallest parent id; the old value names the one discoverer.  A pull
// row is looked at by one lane or one wave, and lists its neighbours by
// ascending id, so that the first one in the frontier is the parent.
//
// The choices, and the runs of levels that the level loop leaves to the
// small-frontier kernel (which report no features), follow bfs_run's rules.
#include "dev_common.h"
#include "select_dev.h"
#include "../../../include/albba.h"

namespace {

constexpr int kOB = 1024, kOWaves = kOB / 64;
constexpr int kNP = ALBD_ONE_NPOS;
constexpr int kIdBits = 13;
static_assert(kNP <= 1 << kIdBits, "a key holds a level and an id");
constexpr uint32_t kFree = ~0u;
// a pulled row's entries beyond this many are left to a whole wave
constexpr int kLaneRow = 64;
constexpr int kLaneStep = 4; // entries a lane has in flight
constexpr int kLongRows = ALBD_ONE_NNZ / kLaneRow;

struct OneLds {
    uint32_t key[kNP];
    int32_t ptr[kNP + 1];
    uint16_t id[kNP];
    uint16_t q[2][kNP];       // the frontier's vertices that have edges
    int32_t pf[kOB];          // degree prefix of up to kOB queue entries
    uint16_t long_rows[kLongRows];
    unsigned long long bm[2][kNP / 64];
    uint32_t wsum[kOWaves];
    // counts of a level, by its parity: found, their edges, nonzero frontier
    // words, queued; pull: entries, words, entries of empty frontier words,
    // long rows
    uint32_t cnt[2][8];
    int choice;
    float params[ALBBA_MLP_NPARAM];
    float xs[ALBBA_MLP_IN], h1[ALBBA_MLP_H1], h2[ALBBA_MLP_H2], ys[ALBBA_MLP_OUT];
};
enum { C_FOUND, C_EDGES, C_NZW, C_QUEUED, C_SCAN, C_WORDS, C_COLB, C_LONG };

struct Found {
    uint32_t n = 0, edges = 0, nzw = 0;
};

// vertices found by the lanes of one wave (call with the wave's lanes
// together): into the next queue and bitmap, counted
__device__ __forceinline__ void found_wave(OneLds &S, bool won, int32_t v, int par, Found &f)
{
    const uint64_t m = __ballot(won);
    if (!m) return;
    uint32_t d = 0;
    if (won) {
        d = (uint32_t)(S.ptr[v + 1] - S.ptr[v]);
        f.n += 1;
        f.edges += d;
        f.nzw += atomicOr(&S.bm[par ^ 1][v >> 6], 1ull << (v & 63)) == 0 ? 1 : 0;
    }
    const uint64_t mq = __ballot(d > 0);
    if (!mq) return;
    const int lane = lane_id(), lead = __ffsll((unsigned long long)mq) - 1;
    uint32_t at = 0;
    if (lane == lead) at = atomicAdd(&S.cnt[par][C_QUEUED], (uint32_t)__popcll(mq));
    at = __shfl(at, lead, 64);
    if (d > 0) S.q[par ^ 1][at + __popcll(mq & lanemask_lt(lane))] = (uint16_t)v;
}

// edges of the queue S.q[par][0 .. nq), kOB vertices at a time, one edge a
// thread
__device__ __forceinline__ void push_level(OneLds &S, const albd_graph &g, int nq, uint32_t newlvl, int par, Found &f)
{
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    for (int base = 0; base < nq; base += kOB) {
        const int i = base + tid;
        int32_t d = 0;
        if (i < nq) {
            const int u = S.q[par][i];
            d = S.ptr[u + 1] - S.ptr[u];
        }
        uint32_t wt;
        uint32_t ex = wave_exclusive_scan<uint32_t>((uint32_t)d, &wt);
        if (lane == 0) S.wsum[wid] = wt;
        __syncthreads();
        uint32_t E = 0;
        for (int k = 0; k < kOWaves; ++k) {
            if (k < wid) ex += S.wsum[k];
            E += S.wsum[k];
        }
        S.pf[tid] = (int32_t)ex;
        __syncthreads();
        const int rows = nq - base < kOB ? nq - base : kOB;
        constexpr int kPer = 4; // edges in flight
        for (uint32_t e0 = 0; e0 < E; e0 += kOB * kPer) {
            int32_t v[kPer];
            uint32_t key[kPer];
#pragma unroll
            for (int k = 0; k < kPer; ++k) {
                const uint32_t e = e0 + (uint32_t)(k * kOB + tid);
                v[k] = -1;
                key[k] = 0;
                if (e < E) {
                    // the last row that starts at or before e
                    int lo = 0, hi = rows;
                    while (hi - lo > 1) {
                        const int mid = (lo + hi) >> 1;
                        if ((uint32_t)S.pf[mid] <= e) lo = mid;
                        else hi = mid;
                    }
                    const int u = S.q[par][base + lo];
                    v[k] = g.push_col[(int64_t)S.ptr[u] + (int64_t)(e - (uint32_t)S.pf[lo])];
                    key[k] = newlvl | S.id[u];
                }
            }
#pragma unroll
            for (int k = 0; k < kPer; ++k) {
                bool won = false;
                if (v[k] >= 0 && S.key[v[k]] > key[k]) won = atomicMin(&S.key[v[k]], key[k]) == kFree;
                found_wave(S, won, v[k], par, f);
            }
        }
        __syncthreads(); // pf and wsum are free again
    }
}

// pull columns [k, k + 4), k a multiple of 4: one load, but at the array's end
__device__ __forceinline__ void load_four(const albd_graph &g, int64_t k, int32_t *u)
{
    if (k + 4 <= g.nnz) {
        const int4 x = *reinterpret_cast<const int4 *>(g.pull_col + k);
        u[0] = x.x;
        u[1] = x.y;
        u[2] = x.z;
        u[3] = x.w;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i] = k + i < g.nnz ? g.pull_col[k + i] : 0;
    }
}

__device__ __forceinline__ void pull_level(OneLds &S, const albd_graph &g, uint32_t newlvl, int par, Found &f)
{
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    uint32_t scan = 0, words = 0, colb = 0; // words: the wave's
    // a lane per row, up to kLaneRow entries of it, kLaneStep at a time
    for (int b = 0; b < (int)g.npos; b += kOB) {
        const int p = b + tid;
        bool won = false, more = false;
        int64_t at = 0, end = 0;
        if (p < (int)g.npos && S.key[p] == kFree) {
            at = g.pull_ptr[p];
            end = g.pull_ptr[p + 1];
        }
        const bool open = end > at;
        words += __ballot(open) != 0 ? 1 : 0;
        const int64_t stop = end - at > kLaneRow ? at + kLaneRow : end;
        more = end > stop;
        // (a wave's load of 64 rows takes the address unit a cycle a row: four
        // entries of a row at once, from the array's 16-byte blocks)
        for (int64_t q = at & ~3ll; q < stop && !won; q += kLaneStep) {
            int32_t u[kLaneStep];
#pragma unroll
            for (int k = 0; k < kLaneStep; k += 4) load_four(g, q + k, u + k);
#pragma unroll
            for (int k = 0; k < kLaneStep; ++k) {
                if (won || q + k < at || q + k >= stop) continue;
                const unsigned long long w = S.bm[par][u[k] >> 6];
                scan += 1;
                colb += w == 0 ? 1 : 0;
                if ((w >> (u[k] & 63)) & 1ull) {
                    won = true;
                    S.key[p] = newlvl | S.id[u[k]];
                }
            }
        }
        if (more && !won) S.long_rows[atomicAdd(&S.cnt[par][C_LONG], 1u)] = (uint16_t)p;
        found_wave(S, won, p, par, f);
    }
    __syncthreads();
    // a wave per long row
    const int nl = (int)S.cnt[par][C_LONG];
    for (int i = wid; i < nl; i += kOWaves) {
        const int p = S.long_rows[i];
        const int64_t end = g.pull_ptr[p + 1];
        bool won = false;
        for (int64_t at = g.pull_ptr[p] + kLaneRow; at < end && !won; at += 64) {
            const int64_t k = at + lane;
            bool hit = false;
            int32_t u = 0;
            if (k < end) {
                u = g.pull_col[k];
                const unsigned long long w = S.bm[par][u >> 6];
                hit = (w >> (u & 63)) & 1ull;
                scan += 1;
                colb += w == 0 ? 1 : 0;
            }
            const uint64_t hm = __ballot(hit);
            if (hm) {
                const int first = __shfl(u, __ffsll((unsigned long long)hm) - 1, 64);
                if (lane == 0) S.key[p] = newlvl | S.id[first];
                won = true;
            }
        }
        found_wave(S, won && lane == 0, p, par, f);
    }
    const uint32_t s = wave_sum(scan), c = wave_sum(colb);
    if (lane == 0) {
        atomicAdd(&S.cnt[par][C_SCAN], s);
        atomicAdd(&S.cnt[par][C_WORDS], words);
        atomicAdd(&S.cnt[par][C_COLB], c);
    }
}

__global__ __launch_bounds__(kOB) void k_bfs_one(albd_graph g, albd_state st, albd_one_args a, albd_one_level *log,
                                                 albd_counters *mail, unsigned int seq)
{
    __shared__ OneLds S;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int npos = (int)g.npos;
    if (a.params) mlp_to_lds<kOB>(S.params, a.params);
    for (int p = tid; p < npos; p += kOB) {
        S.key[p] = kFree;
        S.ptr[p] = (int32_t)g.push_ptr[p];
        S.id[p] = (uint16_t)g.row_order[p];
    }
    if (tid == 0) S.ptr[npos] = (int32_t)g.push_ptr[npos];
    for (int w = tid; w < 2 * (kNP / 64); w += kOB) (&S.bm[0][0])[w] = 0;
    if (tid < 16) (&S.cnt[0][0])[tid] = 0;
    const int32_t rp = g.pos_of[a.root];
    __syncthreads();
    const int32_t rdeg = S.ptr[rp + 1] - S.ptr[rp];
    if (tid == 0) {
        S.key[rp] = (uint32_t)a.root;
        S.bm[0][rp >> 6] = 1ull << (rp & 63);
        S.q[0][0] = (uint16_t)rp;
    }
    int64_t F = 1, mf = rdeg, nzw = 1, reached = 1, redges = rdeg, F_sel = 0, frontier_prev = 0;
    int nq = rdeg > 0 ? 1 : 0, prev_choice = ALBBA_CHOICE_PUSH, choice = ALBBA_CHOICE_PUSH;
    int small_streak = 0, slow_streak = 0, run = 0, level = 0; // run: levels of the current run so far
    int64_t run_F = 0;
    while (F > 0) {
        const int par = level & 1;
        __syncthreads(); // the root, or the last level's counts and bitmap
        if (tid < 8) S.cnt[par ^ 1][tid] = 0;
        bool small = run > 0;
        if (!small) {
            if (wid == 0) {
                level_features(S.xs, g.n, g.nnz, g.nwords, (unsigned long long)F, (unsigned long long)mf,
                               (unsigned long long)nzw, (unsigned long long)reached, (unsigned long long)redges,
                               level, prev_choice, (unsigned long long)F_sel);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                if (lane < ALBBA_MLP_IN) log[level].features[lane] = S.xs[lane];
                const int c = a.params ? mlp_argmin_wave(S.params, S.xs, S.h1, S.h2, S.ys, a.valid_mask) : -1;
                if (lane == 0) S.choice = c;
            }
            if (a.params) __syncthreads();
            choice = a.params ? S.choice : -1;
            if (choice < 0) choice = heuristic_choice((unsigned long long)F, g.n);
            const bool size_ok = a.edge_cap > 0 && mf <= a.edge_cap && F <= a.vertex_cap;
            slow_streak = size_ok && F <= 2 * frontier_prev ? slow_streak + 1 : 0;
            const bool slow = a.params && slow_streak > a.slow_levels;
            if (slow) choice = ALBBA_CHOICE_PUSH;
            const bool small_ok = choice == ALBBA_CHOICE_PUSH && size_ok;
            small = slow || (small_ok && small_streak >= 2);
            small_streak = small_ok && !small ? small_streak + 1 : 0;
            run_F = F;
        }
        const uint32_t newlvl = (uint32_t)(level + 1) << kIdBits;
        Found f;
        if (choice == ALBBA_CHOICE_PUSH) push_level(S, g, nq, newlvl, par, f);
        else pull_level(S, g, newlvl, par, f);
        const uint32_t fn = wave_sum(f.n), fe = wave_sum(f.edges), fw = wave_sum(f.nzw);
        if (lane == 0 && fn) {
            atomicAdd(&S.cnt[par][C_FOUND], fn);
            atomicAdd(&S.cnt[par][C_EDGES], fe);
            atomicAdd(&S.cnt[par][C_NZW], fw);
        }
        __syncthreads();
        const uint32_t *c = S.cnt[par];
        const bool push = choice == ALBBA_CHOICE_PUSH;
        if (tid == 0) {
            albd_one_level &l = log[level];
            l.frontier = (int32_t)F;
            l.choice = choice;
            l.entries = push ? (int32_t)mf : (int32_t)c[C_SCAN];
            l.words = push ? (int32_t)c[C_QUEUED] : (int32_t)c[C_WORDS];
            l.col_bypassed = choice == ALBBA_CHOICE_PULL_CB ? (int32_t)c[C_COLB] : 0;
            l.run = small ? run + 1 : 0;
        }
        for (int w = tid; w < (int)g.nwords; w += kOB) S.bm[par][w] = 0;
        const int64_t nF = c[C_FOUND], nmf = c[C_EDGES];
        nzw = c[C_NZW];
        nq = (int)c[C_QUEUED];
        if (small) {
            ++run;
            if (nF == 0 || nmf > a.edge_cap || nF > a.vertex_cap || run >= ALBD_PERSIST_LEVELS) {
                run = 0;
                frontier_prev = nF;
                F_sel = run_F;
            }
        } else {
            frontier_prev = F;
            F_sel = F;
        }
        prev_choice = choice;
        F = nF;
        mf = nmf;
        reached += nF;
        redges += nmf;
        ++level;
    }
    for (int v = tid; v < g.n; v += kOB) {
        const uint32_t k = S.key[g.pos_of[v]];
        st.level[v] = k == kFree ? -1 : (int32_t)(k >> kIdBits);
        st.parent[v] = k == kFree ? -1 : (int32_t)(k & ((1u << kIdBits) - 1));
    }
    if (tid == 0) {
        // the counters that the host reads, and the post: this wave wrote the
        // log, which the release puts in front of the sequence number
        albd_counters *dst[2] = {st.ctr, mail};
        for (albd_counters *d : dst) {
            d->frontier = 0;
            d->reached = (unsigned long long)reached;
            d->reached_edges = (unsigned long long)redges;
            d->persist_levels = level;
        }
        __hip_atomic_store(&mail->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

} // namespace

extern "C" int albd_bfs_one(albd_ctx *c, const albd_graph *g, const albd_state *st, const albd_one_args *a,
                            const albd_one_level **log, unsigned int *seq)
{
    if (!albd_one_fits(g) || a->root < 0 || a->root >= g->n)
        return albd_set_error_msg(ALBBA_EINVAL, "one-workgroup BFS: graph beyond its LDS");
    albd_one_level *dev = nullptr;
    if (int rc = albd_one_log(c, log, &dev)) return rc;
    albd_counters *mail = albd_mail_next(c, seq);
    hipLaunchKernelGGL(k_bfs_one, dim3(1), dim3(kOB), 0, albd_stream(c), *g, *st, *a, dev, mail, *seq);
    HIPCHK(hipGetLastError());
    return 0;
}

extern "C" int albd_one_fits(const albd_graph *g)
{
    return g->npos <= ALBD_ONE_NPOS && g->n <= g->npos && g->nnz <= ALBD_ONE_NNZ;
}
