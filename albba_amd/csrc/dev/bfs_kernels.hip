// BFS kernels for the SELL-C-sigma layout on CDNA4 (gfx950, wave64).
//
// Index space: every bitmap, queue and per-position array is indexed by the
// layout POSITION p (row p of the SELL matrix is vertex row_order[p]); only
// level[] and parent[] are indexed by vertex id.  One wave owns one 64-bit
// word of positions: w covers positions 64w .. 64w+63, i.e. 64/C slices when
// C <= 64 and half a slice when C == 128, so visited/next words of a pull are
// written without atomics.
//
// Pull (bfs/src/bfs_par_kernels.c:128-198, OR-AND SpMV with visited-slice
// bypass): every unvisited lane walks its row's columns in order and stops at
// the first neighbour in the frontier.  Rows list neighbours by ascending
// vertex id, so that first hit is the min-id parent.  The wave leaves a word
// as soon as every lane is resolved or out of columns.
//
// Push (the SpMSpV slot of bfs/src/bfs_par_kernels.c:566-656, done here as a
// true frontier-driven expansion): edges of the frontier queue are split into
// 64-edge chunks via a degree prefix sum; each edge into a vertex unvisited
// at the start of the level does atomicMin(pmin[v], id(u)); the edge that
// finds pmin[v] still all ones sets v in the next bitmap; a word pass then
// writes level/parent and builds the next queue.
#include "dev_common.h"
// one own edge a thread (512 threads of two: 4 096 x 4 096 grid, a root of 7 120
// levels, 5.6 us a level against 5.4; 256 of two or four 6.5)
#define PUSH_LIST_BLOCK 1024
#include "push_lists.h"
#include "select_dev.h"
#include "../../../include/albba.h"

#include <climits>

namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / 64;

// A kernel queued before its level's direction is known runs only when the
// select kernel chose it: spec < 0 runs always; otherwise the learned (1) or
// the heuristic (0) choice must be `choice`, and the frontier nonempty and at
// most fmax.  The select kernel wrote those counters before this kernel
// started, and nothing in between changes them, so every thread of every
// block decides alike.
struct Spec {
    int32_t spec, choice;
    unsigned long long fmax;
};

__device__ __forceinline__ bool spec_go(const albd_counters *ctr, const Spec &sp)
{
    if (sp.spec < 0) return true;
    const unsigned long long f = ctr->frontier;
    const int c = sp.spec ? ctr->sel_choice : ctr->heur_choice;
    return __builtin_amdgcn_readfirstlane(f != 0 && f <= sp.fmax && c == sp.choice ? 1 : 0) != 0;
}

constexpr Spec kNoSpec{-1, 0, 0ull};

struct PullArgs {
    albd_graph g;
    albd_state st;
    int32_t level;
    const int32_t *items;               // LIST variants: word list
    const unsigned long long *nitems;   // LIST variants: its length (device)
    int32_t sum_words32;                // CB: LDS summary size in 32-bit words
    int32_t per_block;                  // consecutive items per block
    // queued before the level's direction is known: -1 no; else run only if
    // the select kernel's choice (1: the learned one, 0: the heuristic's) is
    // spec_choice and the frontier is not empty
    int32_t spec;
    int32_t spec_choice;
};

__device__ __forceinline__ void slot_add(albd_slot *slots, unsigned long long cnt,
                                         unsigned long long edges, unsigned long long words,
                                         unsigned long long scanned,
                                         unsigned long long words_scanned = 0,
                                         unsigned long long bypassed = 0,
                                         unsigned long long col_bypassed = 0)
{
    albd_slot *s = &slots[(blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6)) % ALBD_NSLOT];
    if (cnt) atomicAdd(&s->next_count, cnt);
    if (edges) atomicAdd(&s->next_edges, edges);
    if (words) atomicAdd(&s->next_words, words);
    if (scanned) atomicAdd(&s->scanned, scanned);
    if (words_scanned) atomicAdd(&s->words, words_scanned);
    if (col_bypassed) atomicAdd(&s->col_bypassed, col_bypassed);
    if (bypassed) atomicAdd(&s->bypassed, bypassed);
}

// ---------------------------------------------------------------------------
// pull

// The column-bypass pull stages a frontier summary of up to 32 KB in LDS per
// block; its blocks are 1024 threads so that two of them (32 waves) share a
// CU, where 256-thread blocks would be held to 16 waves by the LDS.
constexpr int kCBBlock = 1024;

template <int VAR> constexpr int pull_block() { return VAR == ALBD_PULL_LIST_CB ? kCBBlock : kBlock; }

// The pull of one level (NT threads a block).
template <int C, int VAR, int NT>
__device__ __forceinline__ void pull_body(const PullArgs &a, uint32_t *lds_sum)
{
    const albd_graph &g = a.g;
    const int lane = lane_id();

    if constexpr (VAR == ALBD_PULL_LIST_CB) {
        const uint32_t *src = reinterpret_cast<const uint32_t *>(a.st.summary);
        for (int i = threadIdx.x; i < a.sum_words32; i += NT) lds_sum[i] = src[i];
        __syncthreads();
    }
    const int64_t nitems = (VAR == ALBD_PULL_ALL) ? (int64_t)g.nwords : (int64_t)(*a.nitems);
    // Word cost is heavy-tailed (the first slice of every sigma window holds
    // its hubs), so work is balanced twice over without global atomics: the
    // hardware dispatcher hands out blocks of per_block consecutive words,
    // and the block's waves take words one at a time through an LDS counter.
    // Blocks are dispatched round-robin over the 8 XCDs (blockIdx % 8); the
    // block -> range map is XCD-major, so each XCD sweeps its own contiguous
    // stretch of words and the level/parent writes of a sigma window merge in
    // one L2.  gridDim is a multiple of 8 and was sized from an upper bound of
    // the item count, so the share of a block is taken from the real count.
    __shared__ int next_item;
    if (threadIdx.x == 0) next_item = 0;
    __syncthreads();
    const int64_t vb = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    int64_t per = (nitems + gridDim.x - 1) / gridDim.x;
    if (per < 1) per = 1;
    const int64_t b0 = vb * per;
    const int64_t b1 = b0 + per < nitems ? b0 + per : nitems;
    const int padm = g.pad - 1;
    constexpr int SUB = C < 64 ? C : 64;
    const uint64_t gmask = SUB == 64 ? ~0ull : (((1ull << SUB) - 1) << ((lane / SUB) * SUB));

    const bool sym = g.pull_col == g.push_col;
    unsigned long long cnt = 0, nzw = 0, scanned = 0, edges = 0, wscan = 0, wbyp = 0;
    // column bypass: this lane's column entries whose frontier word the
    // summary shows empty (their gathers are skipped)
    unsigned int cbs = 0;
    // One word ahead: while a word's columns are scanned, the next word is
    // claimed, its list entry read, and then its row lengths, visited word
    // and slice pointer loaded, so that a word starts with its first column
    // loads rather than two dependent round trips.  A wave holds one word
    // ahead only, which bounds what it can keep from the block's other waves.
    auto claim = [&]() -> int64_t {
        int k = 0;
        if (lane == 0) k = atomicAdd(&next_item, 1);
        return b0 + __shfl(k, 0, 64);
    };
    auto word_of = [&](int64_t it) -> int32_t {
        if (it >= b1) return -1;
        return (VAR == ALBD_PULL_ALL) ? (int32_t)it : a.items[it];
    };
    struct Head {
        int len, len_o;
        uint64_t vis;
        int64_t cp;
    };
    // row lengths stream like the columns: non-temporal, so that the
    // frontier and visited bitmaps keep their L2 lines
    auto load_head = [&](int32_t w) -> Head {
        Head h{0, 0, ~0ull, 0};
        if (w < 0) return h;
        const int64_t p = (int64_t)w * 64 + lane;
        if constexpr (C <= 64) {
            h.len = __builtin_nontemporal_load(&g.row_len[p]);
            h.cp = g.slice_ptr[p / C];
        } else {
            const int64_t s = w >> 1;
            h.len = __builtin_nontemporal_load(&g.row_len[p]);
            h.len_o = __builtin_nontemporal_load(&g.row_len[s * 128 + (((w & 1) ^ 1) << 6) + lane]);
            h.cp = g.slice_ptr[s];
        }
        h.vis = a.st.visited[w];
        return h;
    };
    int32_t w = word_of(claim());
    Head h = load_head(w);
    while (w >= 0) {
        const int32_t w1 = word_of(claim());
        Head h1{0, 0, ~0ull, 0};
        bool ahead = false; // h1 loaded (wave-uniform)
        {
            const int64_t p = (int64_t)w * 64 + lane;
            // lane row lengths replace per-column active-lane counts: rows of
            // a slice are sorted by length, so column j holds the lanes whose
            // row is longer than j and its size is a ballot away
            int l;
            if constexpr (C <= 64)
                l = (int)(p % C);
            else
                l = ((w & 1) << 6) + lane;
            const int len = h.len, len_o = h.len_o;
            const uint64_t vis = h.vis;
            int64_t cp = h.cp;
            uint64_t unres = __ballot(len > 0) & ~vis;
            if (unres == 0) {
                ++wbyp; // slice bypass: every lane with a row is visited
            } else {
                ++wscan;
                const uint64_t start = unres;
                int parent_pos = -1;
                int j = 0, step = 1;
                // columns are loaded 1, 2, then 4 at a time: most lanes of a
                // dense level hit in the first column, the survivors tend to
                // run long
                for (;;) {
                    const bool mine = (unres >> lane) & 1ull;
                    const uint64_t live = __ballot(mine && j < len);
                    // few live lanes left: their rows go to the row phase below
                    if (__popcll(live) <= g.sparse_lanes) break;
                    int cidx[4];
                    bool av[4], hit[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        av[u] = false;
                        cidx[u] = 0;
                        if (u < step) {
                            const int col = j + u;
                            int act;
                            if constexpr (C <= 64)
                                act = __popcll(__ballot(col < len) & gmask);
                            else
                                act = __popcll(__ballot(col < len)) + __popcll(__ballot(col < len_o));
                            av[u] = mine && col < len;
                            // streaming: non-temporal, so that the frontier
                            // and visited bitmaps stay in L2
                            if (av[u]) cidx[u] = __builtin_nontemporal_load(&g.colidx[cp + l]);
                            cp += (act + padm) & ~padm;
                        }
                    }
                    // the next word's head travels with this word's first
                    // columns
                    if (!ahead) {
                        h1 = load_head(w1);
                        ahead = true;
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        bool hh = false;
                        if (av[u]) {
                            const int c = cidx[u];
                            const int wd = c >> 6;
                            bool maybe = true;
                            if constexpr (VAR == ALBD_PULL_LIST_CB) {
                                maybe = (lds_sum[wd >> 5] >> (wd & 31)) & 1u;
                                cbs += maybe ? 0u : 1u;
                            }
                            if (maybe) hh = (a.st.front[wd] >> (c & 63)) & 1ull;
                        }
                        hit[u] = hh;
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (u < step) {
                            const bool hh = hit[u] && ((unres >> lane) & 1ull);
                            if (hh) parent_pos = cidx[u];
                            unres &= ~__ballot(hh);
                            scanned += __popcll(__ballot(av[u]));
                        }
                    }
                    j += step;
                    if (unres == 0) break;
                    step = step < 4 ? 2 * step : 4;
                }
                if (!ahead) {
                    h1 = load_head(w1);
                    ahead = true;
                }
                // Row phase: the r <= sparse_lanes remaining rows (columns j..
                // onward) are scanned from the row-major copy side by side,
                // each by a group of G = 64/2^ceil(log2 r) lanes reading G
                // consecutive entries per step; the first hit in row order is
                // the min id.
                const uint64_t rem = __ballot(((unres >> lane) & 1ull) && j < len);
                const int r = __popcll(rem);
                if (r) {
                    int G = 64;
                    while (G * r > 64) G >>= 1;
                    const int gid = lane / G, gl = lane % G;
                    const uint64_t gmask_r = (G == 64) ? ~0ull : (((1ull << G) - 1) << (gid * G));
                    int L = -1; // the gid-th remaining lane
                    {
                        uint64_t t = rem;
                        for (int k = 0; k < gid && t; ++k) t &= t - 1;
                        if (gid < r) L = __ffsll((unsigned long long)t) - 1;
                    }
                    const int rl = __shfl(len, L < 0 ? 0 : L, 64);
                    const int64_t rs = L >= 0 ? g.pull_ptr[(int64_t)w * 64 + L] : 0;
                    int got = -1;
                    for (int k = j;; k += G) {
                        const bool live_g = L >= 0 && got < 0 && k < rl;
                        if (__ballot(live_g) == 0) break;
                        const int e = k + gl;
                        bool hh = false;
                        int c = 0;
                        if (live_g && e < rl) {
                            c = g.pull_col[rs + e];
                            const int wd = c >> 6;
                            bool maybe = true;
                            if constexpr (VAR == ALBD_PULL_LIST_CB) {
                                maybe = (lds_sum[wd >> 5] >> (wd & 31)) & 1u;
                                cbs += maybe ? 0u : 1u;
                            }
                            if (maybe) hh = (a.st.front[wd] >> (c & 63)) & 1ull;
                        }
                        scanned += __popcll(__ballot(live_g && e < rl));
                        const uint64_t hm = __ballot(hh) & gmask_r;
                        const int src = hm ? __ffsll((unsigned long long)hm) - 1 : lane;
                        const int first = __shfl(c, src, 64);
                        if (hm && got < 0) got = first;
                    }
                    for (int q = 0; q < r; ++q) {
                        const int Lq = __shfl(L, q * G, 64);
                        const int gq = __shfl(got, q * G, 64);
                        if (gq >= 0) {
                            unres &= ~(1ull << Lq);
                            if (lane == Lq) parent_pos = gq;
                        }
                    }
                }
                const uint64_t found = start & ~unres;
                if (found) {
                    if (lane == 0) {
                        a.st.next[w] = found;
                        a.st.visited[w] = vis | found;
                    }
                    if ((found >> lane) & 1ull) {
                        // position order: the lanes of a word write one run
                        a.st.lp[p] = pack_lp(a.level + 1, g.row_order[parent_pos]);
                        // out-degree: the row's length when the matrix is
                        // symmetric (the pull rows are the push rows)
                        edges += sym ? (unsigned long long)len
                                     : (unsigned long long)(g.push_ptr[p + 1] - g.push_ptr[p]);
                    }
                    cnt += __popcll(found);
                    nzw += 1;
                }
            }
        }
        if (!ahead) h1 = load_head(w1);
        w = w1;
        h = h1;
    }
    edges = wave_sum(edges);
    unsigned long long cb_total = 0;
    if constexpr (VAR == ALBD_PULL_LIST_CB) cb_total = wave_sum((unsigned long long)cbs);
    if (lane == 0) slot_add(a.st.slots, cnt, edges, nzw, scanned, wscan, wbyp, cb_total);
}

template <int C, int VAR>
__global__ __launch_bounds__(pull_block<VAR>()) void k_pull(PullArgs a)
{
    extern __shared__ uint32_t lds_sum[];
    if (!spec_go(a.st.ctr, Spec{a.spec, a.spec_choice, ~0ull})) return;
    pull_body<C, VAR, pull_block<VAR>()>(a, lds_sum);
}


// ---------------------------------------------------------------------------
// word passes

// One reservation per block in a global list: every thread calls it with its
// wave's count (lane 0's value counts); returns the wave's first slot.  Same
// address device atomics serialise, so the word passes take one per block
// step rather than one per wave.
template <int NW = kWavesPerBlock, class T = unsigned int>
__device__ __forceinline__ unsigned long long block_reserve(unsigned long long *counter, T wave_count, T *s_cnt,
                                                           unsigned long long *s_base)
{
    const int wid = threadIdx.x >> 6;
    if (lane_id() == 0) s_cnt[wid] = wave_count;
    __syncthreads();
    if (threadIdx.x == 0) {
        T tot = 0;
        for (int i = 0; i < NW; ++i) tot += s_cnt[i];
        *s_base = tot ? atomicAdd(counter, (unsigned long long)tot) : 0ull;
    }
    __syncthreads();
    unsigned long long off = *s_base;
    for (int i = 0; i < wid; ++i) off += s_cnt[i];
    __syncthreads(); // s_cnt is reused by the next call
    return off;
}

__global__ __launch_bounds__(kBlock) void k_haslen(const int32_t *row_len, uint64_t *haslen,
                                                   int32_t nwords)
{
    const int64_t gt = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int64_t w = gt >> 6;
    const bool pred = (w < nwords) && row_len[gt] > 0;
    const uint64_t m = __ballot(pred);
    if (lane_id() == 0 && w < nwords) haslen[w] = m;
}

// The state of a BFS from vertex ro in one launch: the bitmaps
// and the slot and counter blocks zeroed, except what the root sets -- its
// visited and frontier bits, its level/parent entry, the queue holding it
// (when it has out-edges), and slot 0 seeded as the frontier of "level -1",
// which the first select kernel sums.  lp holds stale values outside the
// visited set (the vertex-order pass masks them), and pmin is all ones at
// rest (the push finalize restores every entry it consumed).
// each row's vertex id as an offset inside its window (two bytes where
// row_order takes four: the vertex-order pass streams these)
__global__ __launch_bounds__(kBlock) void k_row_off(albd_graph g, uint16_t *row_off)
{
    const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (p < g.n) row_off[p] = (uint16_t)(g.row_order[p] - (int32_t)((p / g.win) * g.win));
}

__global__ __launch_bounds__(kBlock) void k_bfs_reset(albd_graph g, albd_state st, int32_t ro)
{
    const int32_t rp = g.pos_of[ro];
    const int64_t deg = g.push_ptr[rp + 1] - g.push_ptr[rp];
    const int32_t rw = rp >> 6;
    const uint64_t bit = 1ull << (rp & 63);
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < g.nwords;
         i += (int64_t)gridDim.x * kBlock) {
        const uint64_t v = i == rw ? bit : 0ull;
        st.visited[i] = v;
        st.front[i] = v;
        st.next[i] = 0;
    }
    static_assert(offsetof(albd_slot, next_count) == 0 && offsetof(albd_slot, next_edges) == 8 &&
                      offsetof(albd_slot, next_words) == 16,
                  "slot 0 seeded by word");
    unsigned long long *slots = reinterpret_cast<unsigned long long *>(st.slots);
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
         i < (int64_t)(ALBD_NSLOT * sizeof(albd_slot) / 8); i += (int64_t)gridDim.x * kBlock)
        slots[i] = i == 0 || i == 2 ? 1ull : (i == 1 ? (unsigned long long)deg : 0ull);
    if (blockIdx.x == 0) {
        constexpr int kQ = (int)(offsetof(albd_counters, queue_len) / 8);
        unsigned long long *c = reinterpret_cast<unsigned long long *>(st.ctr);
        for (int i = threadIdx.x; i < (int)(sizeof(albd_counters) / 8); i += kBlock)
            c[i] = i == kQ && deg > 0 ? 1ull | (unsigned long long)deg << 32 : 0ull;
        if (threadIdx.x == 0) {
            st.lp[rp] = pack_lp(0, ro);
            if (deg > 0) {
                st.queue[0] = rp;
                st.prefix[0] = 0;
            }
        }
    }
}

// End of a level: the frontier it produced, the running totals, the
// selector features (level_features) and the policy's choice for the next
// level.  One block.
constexpr int kSelectBlock = 256;

__device__ __forceinline__ void select_body(const albd_graph &g, const albd_state &st, const albd_select_args &sel,
                                            albd_counters *mail, unsigned int seq)
{
    // the counter block up to the mailbox sequence word, as 64-bit words
    constexpr int kCtrWords = (int)(offsetof(albd_counters, seq) / 8);
    static_assert(kCtrWords <= 64, "one wave moves the counter block");
    __shared__ float xs[ALBBA_MLP_IN], h1[ALBBA_MLP_H1], h2[ALBBA_MLP_H2], ys[ALBBA_MLP_OUT];
    __shared__ float s_params[ALBBA_MLP_NPARAM];
    __shared__ unsigned long long s_red[7][kSelectBlock / 64];
    __shared__ union {
        albd_counters c;
        unsigned long long w[sizeof(albd_counters) / 8];
    } s_ctr;
    const int lane = lane_id(), wid = threadIdx.x >> 6, tid = threadIdx.x;
    unsigned long long *ctr_words = reinterpret_cast<unsigned long long *>(st.ctr);
    // Every load first (the counter block, the weights, the slots), so that
    // they travel together; then the block sums the slots, and wave 0 alone
    // computes the features, runs the MLP and writes the counter block back
    // (one lane per word: thread 0 alone would chain one load per word).
    constexpr int kPer = ALBD_NSLOT / kSelectBlock;
    static_assert(ALBD_NSLOT % kSelectBlock == 0, "slots split evenly over the block");
    static_assert(sizeof(albd_slot) == 64, "slot = 4 x 16 counter bytes");
    // a used unvisited-word list (slot (level - 1) % 3, built by the
    // previous level's preparation) becomes the current list
    const bool list_used = !sel.first && (sel.prev_choice == ALBBA_CHOICE_PULL_SB ||
                                          sel.prev_choice == ALBBA_CHOICE_PULL_CB);
    unsigned long long cw = 0, used_len = 0;
    if (tid < kCtrWords) cw = ctr_words[tid];
    if (tid == 0 && list_used) used_len = st.ctr->list_cnt[(sel.level + 2) % 3];
    // the slot that the level after this one fills starts from zero
    if (tid == 0) st.ctr->list_cnt[(sel.level + 1) % 3] = 0;
    float pr[mlp_per_thread<kSelectBlock>()];
    if (sel.params) mlp_load<kSelectBlock>(pr, sel.params);
    ulonglong2 v[kPer][4];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const ulonglong2 *p = reinterpret_cast<const ulonglong2 *>(&st.slots[tid + k * kSelectBlock]);
        v[k][0] = p[0];
        v[k][1] = p[1];
        v[k][2] = p[2];
        v[k][3] = p[3];
    }
    // read once, by this thread only: the next level starts from zero
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        ulonglong2 *p = reinterpret_cast<ulonglong2 *>(&st.slots[tid + k * kSelectBlock]);
        p[0] = p[1] = p[2] = p[3] = make_ulonglong2(0ull, 0ull);
    }
    if (tid < kCtrWords) s_ctr.w[tid] = cw;
    if (sel.params) mlp_store<kSelectBlock>(s_params, pr);
    unsigned long long F = 0, mf = 0, nzw = 0, scn = 0, wds = 0, byp = 0, cbp = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        F += v[k][0].x;   // next_count
        mf += v[k][0].y;  // next_edges
        nzw += v[k][1].x; // next_words
        scn += v[k][1].y; // scanned
        wds += v[k][2].x; // words
        byp += v[k][2].y; // bypassed
        cbp += v[k][3].x; // col_bypassed
    }
    F = wave_sum(F);
    mf = wave_sum(mf);
    nzw = wave_sum(nzw);
    scn = wave_sum(scn);
    wds = wave_sum(wds);
    byp = wave_sum(byp);
    cbp = wave_sum(cbp);
    if (lane == 0) {
        s_red[0][wid] = F;
        s_red[1][wid] = mf;
        s_red[2][wid] = nzw;
        s_red[3][wid] = scn;
        s_red[4][wid] = wds;
        s_red[5][wid] = byp;
        s_red[6][wid] = cbp;
    }
    __syncthreads();
    if (wid != 0) return;
    albd_counters &c = s_ctr.c;
    // the totals in every lane of wave 0
    F = mf = nzw = scn = wds = byp = cbp = 0;
    for (int i = 0; i < kSelectBlock / 64; ++i) {
        F += s_red[0][i];
        mf += s_red[1][i];
        nzw += s_red[2][i];
        scn += s_red[3][i];
        wds += s_red[4][i];
        byp += s_red[5][i];
        cbp += s_red[6][i];
    }
    const unsigned long long reached = c.reached + F;
    const unsigned long long redges = c.reached_edges + mf;
    level_features(xs, g.n, g.nnz, g.nwords, F, mf, nzw, reached, redges, sel.level, sel.prev_choice,
                   c.frontier);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int choice = sel.params ? mlp_argmin_wave(s_params, xs, h1, h2, ys, sel.valid_mask) : -1;
    if (lane == 0) {
        c.frontier = F;
        c.frontier_edges = mf;
        c.frontier_words = nzw;
        c.scanned = scn;
        c.words = wds;
        c.bypassed = byp;
        c.col_bypassed = cbp;
        c.reached = reached;
        c.reached_edges = redges;
        const int heur = heuristic_choice(F, g.n);
        c.heur_choice = heur;
        c.sel_choice = sel.forced >= 0 ? sel.forced : (choice >= 0 ? choice : heur);
        for (int i = 0; i < ALBBA_MLP_IN; ++i) c.features[i] = xs[i];
        // hand the level's lists over to the next level: a pushed level's
        // queue becomes the queue (after a pull the queue is rebuilt from
        // the bitmap, from zero); a used unvisited-word list becomes the list
        if (!sel.first) c.queue_len = sel.prev_choice == ALBBA_CHOICE_PUSH ? c.qnext_len : 0ull;
        c.qnext_len = 0;
        if (list_used) c.active_len = used_len;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (lane < kCtrWords) {
        const unsigned long long w = s_ctr.w[lane];
        ctr_words[lane] = w;
        if (mail) reinterpret_cast<unsigned long long *>(mail)[lane] = w;
    }
    if (mail) {
        // the whole block to host memory, then the sequence number with a
        // system-scope release: the host sees the data once it sees seq
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) __hip_atomic_store(&mail->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

__global__ __launch_bounds__(kSelectBlock) void k_select(albd_graph g, albd_state st, albd_select_args sel,
                                                         albd_counters *mail, unsigned int seq)
{
    select_body(g, st, sel, mail, seq);
}

// Zero st.next (the select kernel has moved the counters and zeroed the
// slots).  ALBD_LB_SLOTS: zero the slots too (trial runs of one level);
// ALBD_LB_SMALL: the small-frontier kernel follows; zero its grid state, its
// levels' counters and the error flag here instead of in launches of their own.

__global__ __launch_bounds__(kBlock) void k_level_begin(albd_state st, int32_t nwords, int flags)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < nwords;
         i += (int64_t)gridDim.x * kBlock)
        st.next[i] = 0;
    if (flags & ALBD_LB_SLOTS) {
        unsigned long long *slots = reinterpret_cast<unsigned long long *>(st.slots);
        for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
             i < (int64_t)(ALBD_NSLOT * sizeof(albd_slot) / 8); i += (int64_t)gridDim.x * kBlock)
            slots[i] = 0;
    }
    if (flags & ALBD_LB_SMALL) {
        const int64_t i0 = (int64_t)blockIdx.x * kBlock + threadIdx.x, step = (int64_t)gridDim.x * kBlock;
        unsigned long long *p = reinterpret_cast<unsigned long long *>(st.persist);
        static_assert(sizeof(albd_persist) % 8 == 0, "cleared by word");
        for (int64_t i = i0; i < (int64_t)(sizeof(albd_persist) / 8); i += step) p[i] = 0;
        for (int64_t i = i0; i < 4 * ALBD_PERSIST_LEVELS; i += step) st.level_log[i] = 0;
        if (i0 == 0) {
            st.ctr->persist_error = 0;
            // the levels run inside that kernel skip the select kernels
            // that clear the list-count slots
            for (int k = 0; k < 3; ++k) st.ctr->list_cnt[k] = 0;
        }
    }
}

// Where the list preparation of level L finds its counts: the input list's
// length in active_len (in_slot < 0: the select kernel of level L has
// already handed it over) or in list_cnt[in_slot] (the select kernel runs in
// the same launch); the output count in list_cnt[out_slot = L % 3].
struct ListSlots {
    int32_t in_slot, out_slot;
};

// unvisited-word list: from every word (FROM_LIST = false) or from the
// previous list (visited only grows, so an old list is a superset).  Blocks
// bid of nb.
template <bool FROM_LIST>
__device__ __forceinline__ void active_body(const albd_graph &g, const albd_state &st, ListSlots ls, int bid,
                                            int nb, unsigned int *s_cnt, unsigned long long *s_base)
{
    constexpr int kGroups = 4; // 64-item groups per wave per step
    const int lane = lane_id(), wid = threadIdx.x >> 6;
    const int64_t n_in =
        FROM_LIST ? (int64_t)(ls.in_slot < 0 ? st.ctr->active_len : st.ctr->list_cnt[ls.in_slot]) : (int64_t)g.nwords;
    unsigned long long *out_cnt = &st.ctr->list_cnt[ls.out_slot];
    const int64_t step = (int64_t)kBlock * kGroups;
    for (int64_t base = (int64_t)bid * step; base < n_in; base += (int64_t)nb * step) {
        int32_t w[kGroups];
        uint64_t m[kGroups];
        unsigned int cnt = 0;
#pragma unroll
        for (int k = 0; k < kGroups; ++k) {
            const int64_t i = base + (int64_t)(wid * kGroups + k) * 64 + lane;
            bool keep = false;
            w[k] = -1;
            if (i < n_in) {
                w[k] = FROM_LIST ? st.active[i] : (int32_t)i;
                keep = (g.haslen[w[k]] & ~st.visited[w[k]]) != 0;
            }
            m[k] = __ballot(keep);
            cnt += (unsigned int)__popcll(m[k]);
        }
        unsigned long long off = block_reserve(out_cnt, cnt, s_cnt, s_base);
#pragma unroll
        for (int k = 0; k < kGroups; ++k) {
            if ((m[k] >> lane) & 1ull) st.active_next[off + __popcll(m[k] & lanemask_lt(lane))] = w[k];
            off += (unsigned long long)__popcll(m[k]);
        }
    }
}

__device__ __forceinline__ void summary_body(const albd_graph &g, const albd_state &st, int bid, int nb)
{
    const int lane = lane_id();
    const int64_t ngroups = ((int64_t)g.nwords + 63) >> 6;
    const int64_t gw = ((int64_t)bid * kBlock + threadIdx.x) >> 6;
    const int64_t nw = ((int64_t)nb * kBlock) >> 6;
    for (int64_t grp = gw; grp < ngroups; grp += nw) {
        const int64_t w = grp * 64 + lane;
        const bool nz = (w < g.nwords) && st.front[w] != 0;
        const uint64_t m = __ballot(nz);
        if (lane == 0) st.summary[grp] = m;
    }
}

template <bool FROM_LIST>
__global__ __launch_bounds__(kBlock) void k_active(albd_graph g, albd_state st, ListSlots ls)
{
    __shared__ unsigned int s_cnt[kWavesPerBlock];
    __shared__ unsigned long long s_base;
    active_body<FROM_LIST>(g, st, ls, blockIdx.x, gridDim.x, s_cnt, &s_base);
}

__global__ __launch_bounds__(kBlock) void k_summary(albd_graph g, albd_state st)
{
    summary_body(g, st, blockIdx.x, gridDim.x);
}

// The next level's preparation: zero st.next, compact the unvisited-word
// list, build the frontier summary.  The three parts touch disjoint data.
// Blocks bid of nb.
template <bool FROM_LIST, bool SUMMARY>
__device__ __forceinline__ void prep_body(const albd_graph &g, const albd_state &st, ListSlots ls, int bid, int nb)
{
    __shared__ unsigned int s_cnt[kWavesPerBlock];
    __shared__ unsigned long long s_base;
    for (int64_t i = (int64_t)bid * kBlock + threadIdx.x; i < g.nwords; i += (int64_t)nb * kBlock)
        st.next[i] = 0;
    active_body<FROM_LIST>(g, st, ls, bid, nb, s_cnt, &s_base);
    if constexpr (SUMMARY) summary_body(g, st, bid, nb);
}

template <bool FROM_LIST, bool SUMMARY>
__global__ __launch_bounds__(kBlock) void k_prep(albd_graph g, albd_state st, ListSlots ls)
{
    prep_body<FROM_LIST, SUMMARY>(g, st, ls, blockIdx.x, gridDim.x);
}

// The select kernel of level L (block 0) and level L's preparation (the
// other blocks) in one launch, so that neither waits for the other.  They
// share no data: the preparation reads the input list's length from its
// slot rather than from active_len, writes its count into a slot the select
// kernel does not touch, and zeroes st.next, which the select kernel does
// not read; the counters the select kernel sums are in st.slots.
template <bool FROM_LIST, bool SUMMARY>
__global__ __launch_bounds__(kBlock) void k_select_prep(albd_graph g, albd_state st, albd_select_args sel,
                                                        albd_counters *mail, unsigned int seq, ListSlots ls)
{
    static_assert(kSelectBlock == kBlock, "one block shape for both parts");
    if (blockIdx.x == 0) select_body(g, st, sel, mail, seq);
    else prep_body<FROM_LIST, SUMMARY>(g, st, ls, blockIdx.x - 1, gridDim.x - 1);
}

// Words -> queue of positions with out-degree > 0, and the queue's degree
// prefix.  FINALIZE (after a push): the words are st.next; merge them into
// visited, write level/parent from pmin and count the new frontier; the queue
// only while the level's frontier edges (the select kernel's count) are at most
// build_max: a larger push likely leads to a pull, which needs none, and a push
// after it lists the bitmap.  Otherwise the words are st.front.
//
// A block reserves its entries and their edges by one atomic on a packed count
// (edges in the high half), so that the queue's order and the prefix's agree
// whichever block comes first: the push that follows needs no scan of its queue
// (one launch of about 9 us a level, three past 8 192 vertices).
//
// 1024-thread blocks: the reservation is one same-address atomic per block, and
// those serialise (256-thread blocks made the reservations the larger part of a
// big push level's finalize).  A wave takes wpw words, one after the other: 64
// where the words fill the chip, fewer on smaller graphs (RMAT s16, 1 024 words,
// 64 a wave: one block, 21 us).
constexpr int kQBlock = 1024;
constexpr int kQWaves = kQBlock / 64;

template <bool FINALIZE>
__global__ __launch_bounds__(kQBlock) void k_words_to_queue(albd_graph g, albd_state st, int32_t level, Spec sp,
                                                            long long build_max, int wpw)
{
    __shared__ unsigned long long s_cnt[kQWaves];
    __shared__ unsigned long long s_base;
    if (!spec_go(st.ctr, sp)) return;
    const bool build = !FINALIZE || (long long)st.ctr->frontier_edges <= build_max;
    const int lane = lane_id(), wid = threadIdx.x >> 6;
    const uint64_t *words = FINALIZE ? st.next : st.front;
    int32_t *q = FINALIZE ? st.queue_next : st.queue;
    unsigned long long *qlen = FINALIZE ? &st.ctr->qnext_len : &st.ctr->queue_len;
    const int64_t ngroups = ((int64_t)g.nwords + wpw - 1) / wpw;
    unsigned long long cnt = 0, nzw = 0, edges = 0;
    // block-uniform steps of one group of wpw words per wave
    for (int64_t gb = (int64_t)blockIdx.x * kQWaves; gb < ngroups; gb += (int64_t)gridDim.x * kQWaves) {
        const int64_t w0 = (gb + wid) * wpw, w = w0 + lane;
        const uint64_t word = (lane < wpw && w < g.nwords) ? words[w] : 0ull;
        if (FINALIZE && word) {
            st.visited[w] |= word; // only this lane touches word w here
            cnt += __popcll(word);
            nzw += 1;
        }
        const uint64_t nzmask = __ballot(word != 0);
        uint64_t keepw = 0;    // lane k holds the keep mask of word w0 + k
        uint32_t kept_edges = 0; // and the edges of those it keeps
        uint64_t mm = nzmask;
        while (mm) {
            const int k = __ffsll((unsigned long long)mm) - 1;
            mm &= mm - 1;
            const uint64_t bits = __shfl(word, k, 64);
            const int64_t pp = (w0 + k) * 64 + lane;
            uint32_t d = 0;
            if ((bits >> lane) & 1ull) {
                d = (uint32_t)(g.push_ptr[pp + 1] - g.push_ptr[pp]);
                if (FINALIZE) {
                    st.lp[pp] = pack_lp(level + 1, (int32_t)st.pmin[pp]);
                    st.pmin[pp] = 0xFFFFFFFFu;
                    edges += d;
                }
            }
            if (!build) continue; // kernel-uniform
            const uint64_t km = __ballot(d > 0);
            const uint32_t ke = wave_sum(d);
            if (lane == k) {
                keepw = km;
                kept_edges = ke;
            }
        }
        if (!build) continue;
        unsigned long long total;
        const unsigned long long excl = wave_exclusive_scan<unsigned long long>(
            (unsigned long long)kept_edges << 32 | (unsigned long long)__popcll(keepw), &total);
        const unsigned long long base = block_reserve<kQWaves>(qlen, total, s_cnt, &s_base);
        uint64_t km = __ballot(keepw != 0);
        while (km) {
            const int k = __ffsll((unsigned long long)km) - 1;
            km &= km - 1;
            const uint64_t kw = __shfl(keepw, k, 64);
            const unsigned long long off = base + __shfl(excl, k, 64);
            const int64_t pp = (w0 + k) * 64 + lane;
            const bool mine = (kw >> lane) & 1ull;
            uint32_t tot;
            const uint32_t ex = wave_exclusive_scan<uint32_t>(
                mine ? (uint32_t)(g.push_ptr[pp + 1] - g.push_ptr[pp]) : 0u, &tot);
            if (mine) {
                const uint32_t at = (uint32_t)off + (uint32_t)__popcll(kw & lanemask_lt(lane));
                q[at] = (int32_t)pp;
                st.prefix[at] = (int64_t)(off >> 32) + ex;
            }
        }
    }
    if (FINALIZE) {
        cnt = wave_sum(cnt);
        nzw = wave_sum(nzw);
        edges = wave_sum(edges);
        if (lane == 0) slot_add(st.slots, cnt, edges, nzw, 0);
    }
}

// level and parent from position order to vertex order, once per BFS.
// Positions [k*win, (k+1)*win) hold the vertices of the same id range (the
// sigma windows), so a block takes one window: it streams the window's row
// offsets (row_off), lp and visited words in position order, scatters level and
// parent into LDS by vertex, and writes both out in vertex order.  Every
// global access is a coalesced stream.  LDS: 8 bytes per window row.
constexpr int kMaxWin = 8192;

// 512-thread blocks: a window's LDS arrays (32 KB at 4096 rows) allow four
// blocks per CU, which then hold the CU's 32 wave slots
constexpr int kVoBlock = 512;

__global__ __launch_bounds__(kVoBlock) void k_to_vertex_order_win(albd_graph g, albd_state st, int if_done)
{
    // queued before the host knew the BFS had ended: run only if the last
    // select kernel found the frontier empty
    if (if_done && st.ctr->frontier != 0) return;
    extern __shared__ int32_t s_win[];
    int32_t *s_level = s_win, *s_parent = s_win + g.win;
    constexpr int kV = 4; // positions in flight per thread
    const int64_t nwin = ((int64_t)g.n + g.win - 1) / g.win;
    for (int64_t w = blockIdx.x; w < nwin; w += gridDim.x) {
        const int64_t lo = w * g.win;
        const int32_t len = (int32_t)((int64_t)g.n - lo < g.win ? (int64_t)g.n - lo : g.win);
        // unreached vertices keep -1; only reached positions load their
        // offset and lp (a window's empty rows, its last positions, are
        // never reached unless one is the root: 43 % of the positions of an
        // RMAT s22 graph, whose lines are then not read)
        for (int32_t i = threadIdx.x; i < len; i += kVoBlock) {
            s_level[i] = -1;
            s_parent[i] = -1;
        }
        __syncthreads();
        for (int32_t i0 = threadIdx.x; i0 < len; i0 += kVoBlock * kV) {
            bool reached[kV];
#pragma unroll
            for (int k = 0; k < kV; ++k) {
                const int32_t i = i0 + k * kVoBlock;
                const int64_t p = lo + (i < len ? i : 0);
                reached[k] = i < len && ((st.visited[p >> 6] >> (p & 63)) & 1ull);
            }
            int32_t o[kV];
            unsigned long long x[kV];
#pragma unroll
            for (int k = 0; k < kV; ++k) {
                const int64_t p = lo + i0 + k * kVoBlock;
                o[k] = reached[k] ? (int32_t)g.row_off[p] : 0;
                x[k] = reached[k] ? st.lp[p] : 0ull;
            }
#pragma unroll
            for (int k = 0; k < kV; ++k) {
                if (reached[k] && o[k] < len) {
                    s_level[o[k]] = (int32_t)(x[k] >> 32);
                    s_parent[o[k]] = (int32_t)(uint32_t)x[k];
                }
            }
        }
        __syncthreads();
        for (int32_t i = threadIdx.x; i < len; i += kVoBlock) {
            st.level[lo + i] = s_level[i];
            st.parent[lo + i] = s_parent[i];
        }
        __syncthreads(); // the LDS arrays are reused by the next window
    }
}

// The same for windows longer than the LDS arrays: a block takes 4096
// consecutive vertex ids and gathers lp through pos_of.
constexpr int kVertexChunk = 4096;

__global__ __launch_bounds__(kBlock) void k_to_vertex_order(albd_graph g, albd_state st, int if_done)
{
    if (if_done && st.ctr->frontier != 0) return;
    constexpr int kV = 4; // vertices in flight per thread
    for (int64_t c0 = (int64_t)blockIdx.x * kVertexChunk; c0 < g.n; c0 += (int64_t)gridDim.x * kVertexChunk) {
        for (int64_t v0 = c0 + threadIdx.x; v0 < c0 + kVertexChunk && v0 < g.n; v0 += kBlock * kV) {
            int32_t p[kV];
#pragma unroll
            for (int k = 0; k < kV; ++k) {
                const int64_t v = v0 + k * kBlock;
                p[k] = (v < g.n && v < c0 + kVertexChunk) ? g.pos_of[v] : 0;
            }
            uint64_t vis[kV];
            unsigned long long x[kV];
#pragma unroll
            for (int k = 0; k < kV; ++k) {
                vis[k] = st.visited[p[k] >> 6];
                x[k] = st.lp[p[k]];
            }
#pragma unroll
            for (int k = 0; k < kV; ++k) {
                const int64_t v = v0 + k * kBlock;
                if (v >= g.n || v >= c0 + kVertexChunk) break;
                const bool reached = (vis[k] >> (p[k] & 63)) & 1ull;
                st.level[v] = reached ? (int32_t)(x[k] >> 32) : -1;
                st.parent[v] = reached ? (int32_t)(uint32_t)x[k] : -1;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// push: degree prefix over the queue

// the frontier queue's entries (their edges are in the high half)
__device__ __forceinline__ int64_t queue_count(const albd_counters *ctr)
{
    return (int64_t)(ctr->queue_len & 0xffffffffull);
}

__device__ __forceinline__ int64_t out_degree(const albd_graph &g, int32_t u)
{
    return g.push_ptr[u + 1] - g.push_ptr[u];
}

// exclusive scan of one value per thread across a 256-thread block
__device__ __forceinline__ int64_t block_exclusive_scan(int64_t v, int64_t *total,
                                                        int64_t *lds /* >= 5 */)
{
    const int lane = lane_id(), wid = threadIdx.x >> 6;
    int64_t wt;
    int64_t ex = wave_exclusive_scan<int64_t>(v, &wt);
    if (lane == 0) lds[wid] = wt;
    __syncthreads();
    int64_t off = 0, tot = 0;
    for (int i = 0; i < kWavesPerBlock; ++i) {
        if (i < wid) off += lds[i];
        tot += lds[i];
    }
    __syncthreads();
    *total = tot;
    return ex + off;
}

__global__ __launch_bounds__(kBlock) void k_scan_small(albd_graph g, albd_state st, Spec sp)
{
    __shared__ int64_t lds[8];
    if (!spec_go(st.ctr, sp)) return;
    const int64_t qlen = queue_count(st.ctr);
    int64_t carry = 0;
    for (int64_t base = 0; base < qlen; base += kBlock) {
        const int64_t i = base + threadIdx.x;
        const int64_t d = (i < qlen) ? out_degree(g, st.queue[i]) : 0;
        int64_t tot;
        const int64_t ex = block_exclusive_scan(d, &tot, lds);
        if (i < qlen) st.prefix[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) st.ctr->queue_len = (unsigned long long)carry << 32 | (unsigned long long)qlen;
}

__global__ __launch_bounds__(kBlock) void k_scan_p1(albd_graph g, albd_state st)
{
    __shared__ int64_t lds[8];
    const int64_t qlen = queue_count(st.ctr);
    const int64_t cs = (qlen + gridDim.x - 1) / gridDim.x;
    const int64_t lo = cs * blockIdx.x, hi = lo + cs < qlen ? lo + cs : qlen;
    int64_t sum = 0;
    for (int64_t i = lo + threadIdx.x; i < hi; i += kBlock) {
        const int64_t d = out_degree(g, st.queue[i]);
        st.prefix[i] = d;
        sum += d;
    }
    int64_t tot;
    (void)block_exclusive_scan(sum, &tot, lds);
    if (threadIdx.x == 0) st.block_sums[blockIdx.x] = tot;
}

__global__ __launch_bounds__(kBlock) void k_scan_p2(albd_state st, int32_t nblocks)
{
    __shared__ int64_t lds[8];
    const int64_t qlen = queue_count(st.ctr);
    int64_t carry = 0;
    for (int base = 0; base < nblocks; base += kBlock) {
        const int i = base + threadIdx.x;
        const int64_t v = i < nblocks ? st.block_sums[i] : 0;
        int64_t tot;
        const int64_t ex = block_exclusive_scan(v, &tot, lds);
        if (i < nblocks) st.block_sums[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) {
        st.block_sums[nblocks] = carry;
        st.ctr->queue_len = (unsigned long long)carry << 32 | (unsigned long long)qlen;
    }
}

__global__ __launch_bounds__(kBlock) void k_scan_p3(albd_state st)
{
    __shared__ int64_t lds[8];
    const int64_t qlen = queue_count(st.ctr);
    const int64_t cs = (qlen + gridDim.x - 1) / gridDim.x;
    const int64_t lo = cs * blockIdx.x, hi = lo + cs < qlen ? lo + cs : qlen;
    int64_t carry = st.block_sums[blockIdx.x];
    for (int64_t base = lo; base < hi; base += kBlock) {
        const int64_t i = base + threadIdx.x;
        const int64_t d = i < hi ? st.prefix[i] : 0;
        int64_t tot;
        const int64_t ex = block_exclusive_scan(d, &tot, lds);
        if (i < hi) st.prefix[i] = carry + ex;
        carry += tot;
    }
}

// ---------------------------------------------------------------------------
// push: expansion of the frontier's edges

// The queue entry of edge e0: the largest v with prefix[v] <= e0 (wave-uniform,
// 64 probes per round).
__device__ __forceinline__ int64_t entry_of_edge(const int64_t *prefix, int64_t qlen, int64_t e0)
{
    const int lane = lane_id();
    int64_t v = 0;
    for (int64_t hi = qlen; hi - v > 1;) { // prefix[v] <= e0 < prefix[hi]
        const int64_t step = (hi - v + 63) / 64, at = v + lane * step;
        const int c = __popcll(__ballot(at < hi && prefix[at] <= e0)); // lane 0's holds
        v += (c - 1) * step;
        if (v + step < hi) hi = v + step;
    }
    return v;
}

// Expansion over 64-edge chunks: each edge into an unvisited vertex lowers
// the vertex's pmin to its source's id.
//
// What bounds it is the device-scope atomics, which go past the L2 at about
// 30 G/s, so an edge asks first whether it would lower the entry: ids only
// decrease during a level and entries are all ones at rest, so a stale copy
// costs an atomic and never a wrong answer, and of the k edges into one target
// about ln k lower it.  RMAT s22, 11.9 M edges: 435 -> 211 us; s24, 79 M edges:
// 2 533 -> 1 228 us, of which the columns and visited gathers alone are 303.
// (Four edges per lane in flight: 229 and 1 206 us, and 14 instead of 9 us on
// small levels.  Claims as bits and parents from the targets' rows: 237 and
// 990 us plus 190 and 670 us for the rows, with one bitmap; more with one per
// XCD, since the atomics are what costs.)
__global__ __launch_bounds__(kBlock) void k_push_expand(albd_graph g, albd_state st, Spec sp)
{
    if (!spec_go(st.ctr, sp)) return;
    const int lane = lane_id();
    const int64_t qlen = queue_count(st.ctr), E = (int64_t)(st.ctr->queue_len >> 32);
    if (blockIdx.x == 0 && threadIdx.x == 0) st.ctr->push_edges = (unsigned long long)E;
    if (qlen == 0) return;
    const int64_t gw = ((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
    const int64_t nw = ((int64_t)gridDim.x * kBlock) >> 6;
    const int64_t nchunks = (E + 63) >> 6;
    const int64_t per = (nchunks + nw - 1) / nw;
    const int64_t c_lo = gw * per, c_hi = c_lo + per < nchunks ? c_lo + per : nchunks;
    if (c_lo >= c_hi) return;
    int64_t e0 = c_lo << 6;
    int64_t v0 = entry_of_edge(st.prefix, qlen, e0);
    for (int64_t ch = c_lo; ch < c_hi; ++ch) {
        e0 = ch << 6;
        const int64_t e = e0 + lane;
        // v0 holds edge e0 and queue entries have degree >= 1, so the chunk's
        // edges belong to vertices v0 .. v0+63
        const int64_t Pk = (v0 + 1 + lane < qlen) ? st.prefix[v0 + 1 + lane] : LLONG_MAX;
        const int64_t P0 = st.prefix[v0];
        int t = 0;
#pragma unroll
        for (int step = 32; step > 0; step >>= 1) {
            const int64_t probe = __shfl(Pk, t + step - 1, 64);
            if (probe <= e) t += step;
        }
        const int64_t prevP = __shfl(Pk, t > 0 ? t - 1 : 0, 64);
        const int64_t ui = v0 + t;
        if (e < E) {
            const int64_t start = t == 0 ? P0 : prevP;
            const int32_t u = st.queue[ui];
            const uint32_t ou = (uint32_t)g.row_order[u];
            const int32_t v = g.push_col[g.push_ptr[u] + (e - start)];
            if (!((st.visited[v >> 6] >> (v & 63)) & 1ull)) {
                // pmin is all ones at rest: the first edge into v this level
                // sees that value back and is the one that sets v's bit
                if (st.pmin[v] > ou && atomicMin(&st.pmin[v], ou) == 0xFFFFFFFFu)
                    atomicOr(reinterpret_cast<unsigned long long *>(&st.next[v >> 6]),
                             1ull << (v & 63));
            }
        }
        // the next chunk starts at edge e0 + 64; its vertex is v0 plus the
        // number of prefix entries v0+1 .. v0+64 at or below that edge (the
        // lanes hold exactly those 64 entries, so this count may reach 64)
        v0 += __popcll(__ballot(Pk <= e0 + 64));
    }
}

// ---------------------------------------------------------------------------
// small-frontier push levels in one persistent launch
//
// High-diameter graphs spend thousands of levels with a few thousand
// frontier vertices; a launch sequence and a host round trip per level would
// dominate, and one workgroup alone is bound by its CU's gather rate.  A
// grid of G co-resident workgroups runs the push levels back to back with
// one grid barrier per level, until the next frontier has more than edge_cap
// out-edges or more than vertex_cap vertices.
//
// Exactness without a second barrier per level: every position p has a
// 64-bit key, all ones outside this kernel.  An edge u -> v at level L does
// atomicMin(key[v], L << 32 | id(u)).  The old value tells the discoverer
// (all ones: first at this level), and the key keeps the smallest (level,
// parent id) pair, i.e. the min-id parent at v's BFS level: keys of earlier
// levels are smaller and never change.  Two filters save atomics: the
// visited bitmap as it was when the kernel started, and the key itself when
// it already holds an earlier level (keys only decrease, so a stale copy
// costs an atomic, never a wrong answer).  Neither is written during the
// launch: the vertices it finds get their level/parent words, visited bits
// and keys back to all ones when it ends.
//
// What bounds a level is its chain of dependent memory round trips, so
// everything that is not the atomic or the barrier is off that chain:
//   - a workgroup keeps the vertices it finds as its own part of the next
//     frontier, as a list of their edges in LDS (no queue in memory between
//     levels); vertices with more than kListDeg out-edges, and those beyond
//     the list's kListEdges, go to a queue in memory that the workgroups
//     share evenly at the next level;
//   - the edges' columns, filters, degrees and vertex ids -- data that no
//     level changes, but for the keys, which are only a filter -- are loaded
//     while the workgroup waits at the barrier;
//   - the barrier itself carries the level's counts: every workgroup stores
//     its three counts, tagged with the level, into slots of its own, and
//     three waves of every workgroup poll everybody's slots and sum them.
// The slots alternate between two sets: a set is written again only two
// levels later, when every workgroup has passed the barrier after reading it.
// Cross-workgroup data (slots, shared queue, keys, found list) moves through
// device-coherent loads, stores and atomics; a wave that wrote to the shared
// queue waits for its stores before the barrier.
//
// A workgroup whose list grew past twice its part of the level's edges keeps
// half a part of what it finds next and shares the rest.  Without that a
// search stays with the workgroup that holds its root until the list is full:
// one workgroup carried the first 4 096 levels of a 4 096 x 4 096 grid alone
// and the kernel took 8.2 us per level instead of 5.5.
//
// Measured on grids of 0.6, 4.2 and 16.8 M vertices, one root each: 4.2, 4.4
// and 5.4 us per level, where a queue in memory between the levels, with its
// reservations and a counting barrier, took 11.8, 12.3 and 13.6.  (32 roots of
// the largest: 5.4 from the ones with most levels, 7 410, to 6.4 from those with
// fewest, 4 536, whose levels are wider.)  Of the 4 us about 1.3
// are the atomic and the appends, 2.0 the loads behind the barrier (two
// dependent misses) and 0.7 what the barrier waits beyond them.  Keeping all
// workgroups on one XCD changed nothing at 0.6 M vertices (4.1 us) and cost at
// 16.8 M (8.3 us with 32 workgroups): the misses go to memory either way.

struct SmallArgs {
    albd_graph g;
    albd_state st;
    int32_t level0;
    int32_t max_levels;
    int64_t edge_cap;
    int64_t vertex_cap;
    uint32_t spin_limit;
};

__global__ __launch_bounds__(kListBlock) void k_push_small(SmallArgs a)
{
    const albd_graph &g = a.g;
    const albd_state &st = a.st;
    __shared__ PushLds S;
    albd_persist *P = st.persist;
    // every vertex this launch finds goes to the prefix array's memory
    const PushMem M{st.visited, st.pkey, reinterpret_cast<int32_t *>(st.prefix), &P->reserve};
    int32_t *found = M.found;
    const int64_t found_cap = 2 * (g.npos + 1);
    int32_t *qa = st.queue, *qb = st.queue_next;
    const int tid = threadIdx.x, lane = lane_id(), wid = tid >> 6;
    const unsigned int G = gridDim.x, w = blockIdx.x;
    const TeamSlots B{&P->slot[0][0][0], &P->error, ALBD_PERSIST_BLOCKS, (int32_t)G, (int32_t)w, a.spin_limit};
    // the waves that poll the slots: the last ones, which hold the fewest edges
    const int poll = wid - (kListWaves - 3);
    list_reset(S);
    __syncthreads();
    if (tid == 0) reserve_found(S, M, 0);
    int64_t ns = queue_count(st.ctr); // the shared queue's length
    int64_t F = 0;                           // found by this workgroup before the level
    PushEdge e[kListPer];
#pragma unroll
    for (int i = 0; i < kListPer; ++i) e[i].act = false;
    int cap = kListEdges; // edges the list takes at this level
    bool ok = true;
    __syncthreads();
    int k = 0;
    uint32_t lvl = 0;
    for (;; ++k) {
        lvl = (uint32_t)(a.level0 + k + 1);
        const int par = k & 1;
        unsigned long long *spill_ctr = reinterpret_cast<unsigned long long *>(&st.level_log[4 * k + 2]);
        if (tid == 0) S.cnt[par ^ 1] = S.edges[par ^ 1] = S.spill[par ^ 1] = 0;
        bool won[kListPer], spilled = false;
        uint32_t f[kListPer];
        // the workgroup's own edges, loaded while it waited, then its share
        // of the queue in memory
        relax_edges<kListPer, false>(S, g, M, e, lvl, par, cap, spill_ctr, qb, won, f, spilled);
        if (ns > 0) {
            __syncthreads(); // the reservation made since the last level
            store_found<kListPer>(S, found, e, won, f, F);
            push_shared(S, g, M, qa, ns, (int)w, (int)G, lvl, par, cap, spill_ctr, qb, F, spilled);
        }
        // the shared queue's entries are in place before the arrival
        if (spilled) __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (poll == 0) {
            if (lane < 3)
                S.arrive[lane] = lane == 0 ? (S.cnt[par] & 0xffffffffull) : (lane == 1 ? S.edges[par] : S.spill[par]);
            team_arrive(S, B, (unsigned int)(k + 1));
        }
        // off the chain: the found list, and everything about the next
        // level's own edges but the atomic
        if (ns == 0) store_found<kListPer>(S, found, e, won, f, F);
        const unsigned long long mine = uniform64(S.cnt[par]);
        F += (int64_t)(mine & 0xffffffffull);
        load_list(S, g, M, (int)((mine >> 32) < (unsigned long long)cap ? (mine >> 32) : (unsigned long long)cap), e);
        if (poll >= 0) team_poll(S, B, poll, (unsigned int)(k + 1));
        __syncthreads();
        ok = S.ok != 0;
        if (!ok) break;
        const int64_t na = (int64_t)uniform64(S.tot[0]), edges = (int64_t)uniform64(S.tot[1]);
        ns = (int64_t)uniform64(S.tot[2]);
        if (w == 0 && tid == 0) {
            st.level_log[4 * k] = na;
            st.level_log[4 * k + 1] = edges;
        }
        if (na == 0 || edges > a.edge_cap || na > a.vertex_cap || k + 1 >= a.max_levels) break;
        // an intermediate level: the select kernel sees only the last one,
        // so these counts go straight into the running totals
        if (w == 0 && tid == 0) {
            st.ctr->reached += (unsigned long long)na;
            st.ctr->reached_edges += (unsigned long long)edges;
        }
        if (tid == 0) reserve_found(S, M, F);
        cap = list_cap((int64_t)(mine >> 32), edges, (int)G);
        int32_t *t = qa;
        qa = qb;
        qb = t;
    }
    if (ok) {
        const unsigned long long na = S.tot[0], edges = S.tot[1];
        end_found(S, M, F, found_cap);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        // (the counts of this arrival are not used)
        if (poll == 0) team_arrive(S, B, (unsigned int)(k + 2));
        if (poll >= 0) team_poll(S, B, poll, (unsigned int)(k + 2));
        __syncthreads();
        ok = S.ok != 0;
        if (ok) {
            // level, parent and visited of every vertex found, and its key
            // back to all ones; the last level's also into the next frontier
            // and its queue
            int64_t total = (int64_t)ld_coherent(&P->reserve);
            if (total > found_cap) total = found_cap;
            unsigned long long my_words = 0;
            for (int64_t b = ((int64_t)w * kListWaves + wid) * 64; b < total;
                 b += (int64_t)G * kListBlock) { // uniform in the wave
                const int64_t i = b + lane;
                const int32_t v = i < total ? ld_coherent(&found[i]) : -1;
                bool queued = false;
                if (v >= 0) {
                    const unsigned long long key = ld_coherent(&st.pkey[v]);
                    st.lp[v] = key; // the same (level, parent) packing
                    const uint64_t bit = 1ull << (v & 63);
                    atomicOr(reinterpret_cast<unsigned long long *>(&st.visited[v >> 6]), bit);
                    st.pkey[v] = ~0ull;
                    if ((uint32_t)(key >> 32) == lvl) {
                        my_words +=
                            atomicOr(reinterpret_cast<unsigned long long *>(&st.next[v >> 6]), bit) == 0 ? 1 : 0;
                        queued = g.push_ptr[v + 1] > g.push_ptr[v];
                    }
                }
                const uint64_t mq = __ballot(queued);
                if (mq) {
                    unsigned long long q = 0;
                    if (lane == 0) q = atomicAdd(&st.ctr->qnext_len, (unsigned long long)__popcll(mq));
                    q = __shfl(q, 0, 64);
                    if (queued) st.queue_next[q + __popcll(mq & lanemask_lt(lane))] = v;
                }
            }
            my_words = wave_sum(my_words);
            if (lane == 0 && my_words) atomicAdd(&st.slots[1 + (w % (ALBD_NSLOT - 1))].next_words, my_words);
            if (w == 0 && tid == 0) {
                st.slots[0].next_count = na;
                st.slots[0].next_edges = edges;
                st.ctr->persist_levels = k + 1;
            }
        }
    }
    if (!ok && tid == 0) st.ctr->persist_error = 1;
}

int grid_persistent(albd_ctx *c, int blocks_per_cu)
{
    int g = albd_num_cus(c) * blocks_per_cu;
    return g < 8 ? 8 : g;
}

// words per wave of k_words_to_queue, and its blocks of kQWaves such waves
int words_per_wave(const albd_graph *g)
{
    return g->nwords >= 1 << 17 ? 64 : (g->nwords >= 1 << 14 ? 16 : 4);
}

int grid_for_queue(albd_ctx *c, const albd_graph *g)
{
    const int64_t per_block = (int64_t)kQWaves * words_per_wave(g);
    int64_t blocks = ((int64_t)g->nwords + per_block - 1) / per_block;
    int64_t cap = (int64_t)albd_num_cus(c) * 2;
    if (blocks > cap) blocks = cap;
    return blocks < 1 ? 1 : (int)blocks;
}

int grid_for_groups(albd_ctx *c, int64_t groups)
{
    int64_t blocks = (groups + kWavesPerBlock - 1) / kWavesPerBlock;
    int64_t cap = (int64_t)albd_num_cus(c) * 8;
    if (blocks > cap) blocks = cap;
    return blocks < 1 ? 1 : (int)blocks;
}

template <int C>
int launch_pull_c(albd_ctx *c, PullArgs a, int variant, size_t lds, int64_t items)
{
    hipStream_t s = albd_stream(c);
    // blocks of per_block words; the grid is a multiple of 8 (one share per XCD)
    int64_t blocks;
    if (variant == ALBD_PULL_LIST_CB) {
        // the LDS summary is staged once per block: fewer, longer blocks
        int per_cu = (int)(160 * 1024 / (lds + 1024));
        per_cu = per_cu > 2 ? 2 : (per_cu < 1 ? 1 : per_cu);
        const int64_t resident = (int64_t)albd_num_cus(c) * per_cu;
        a.per_block = (int32_t)((items + resident - 1) / resident);
        if (a.per_block < 16) a.per_block = 16;
    } else {
        a.per_block = 16;
    }
    blocks = (items + a.per_block - 1) / a.per_block;
    blocks = (blocks + 7) / 8 * 8;
    if (blocks < 8) blocks = 8;
    if (variant == ALBD_PULL_ALL)
        hipLaunchKernelGGL((k_pull<C, ALBD_PULL_ALL>), dim3((unsigned)blocks), dim3(kBlock), 0, s, a);
    else if (variant == ALBD_PULL_LIST)
        hipLaunchKernelGGL((k_pull<C, ALBD_PULL_LIST>), dim3((unsigned)blocks), dim3(kBlock), 0, s, a);
    else
        hipLaunchKernelGGL((k_pull<C, ALBD_PULL_LIST_CB>), dim3((unsigned)blocks), dim3(kCBBlock), lds, s, a);
    HIPCHK(hipGetLastError());
    return 0;
}

} // namespace

extern "C" {

int albd_build_row_off(albd_ctx *c, const albd_graph *g, uint16_t *row_off)
{
    if (g->n <= 0) return 0;
    if (g->win < 1 || g->win > 65536) return albd_set_error_msg(ALBBA_EINVAL, "row offsets: window too long");
    hipLaunchKernelGGL(k_row_off, dim3((unsigned)(((int64_t)g->n + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                       albd_stream(c), *g, row_off);
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_build_haslen(albd_ctx *c, const albd_graph *g, uint64_t *haslen)
{
    const int64_t threads = (int64_t)g->nwords * 64;
    hipLaunchKernelGGL(k_haslen, dim3((unsigned)((threads + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                       albd_stream(c), g->row_len, haslen, g->nwords);
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_bfs_init(albd_ctx *c, const albd_graph *g, const albd_state *st, int32_t root)
{
    hipStream_t s = albd_stream(c);
    int64_t blocks = ((int64_t)g->nwords + kBlock - 1) / kBlock;
    int64_t cap = (int64_t)albd_num_cus(c) * 16;
    hipLaunchKernelGGL(k_bfs_reset, dim3((unsigned)(blocks < 1 ? 1 : (blocks > cap ? cap : blocks))), dim3(kBlock),
                       0, s, *g, *st, root);
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_to_vertex_order(albd_ctx *c, const albd_graph *g, const albd_state *st, int if_done)
{
    if (g->win >= 1 && g->win <= kMaxWin && g->row_off) {
        int64_t blocks = ((int64_t)g->n + g->win - 1) / g->win;
        int64_t cap = (int64_t)albd_num_cus(c) * 16;
        hipLaunchKernelGGL(k_to_vertex_order_win,
                           dim3((unsigned)(blocks < 1 ? 1 : (blocks > cap ? cap : blocks))), dim3(kVoBlock),
                           sizeof(int32_t) * 2 * (size_t)g->win, albd_stream(c), *g, *st, if_done);
        HIPCHK(hipGetLastError());
        return 0;
    }
    int64_t blocks = ((int64_t)g->n + kVertexChunk - 1) / kVertexChunk;
    int64_t cap = (int64_t)albd_num_cus(c) * 32;
    hipLaunchKernelGGL(k_to_vertex_order, dim3((unsigned)(blocks < 1 ? 1 : (blocks > cap ? cap : blocks))),
                       dim3(kBlock), 0, albd_stream(c), *g, *st, if_done);
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_level_begin(albd_ctx *c, const albd_graph *g, const albd_state *st, int flags)
{
    int64_t blocks = ((int64_t)g->nwords + kBlock - 1) / kBlock;
    int64_t cap = (int64_t)albd_num_cus(c) * 8;
    hipLaunchKernelGGL(k_level_begin, dim3((unsigned)(blocks < 1 ? 1 : (blocks > cap ? cap : blocks))),
                       dim3(kBlock), 0, albd_stream(c), *st, g->nwords, flags);
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_build_active(albd_ctx *c, const albd_graph *g, albd_state *st, int from_list,
                      int64_t prev_len, int32_t level)
{
    hipStream_t s = albd_stream(c);
    const int64_t n_in = from_list ? prev_len : g->nwords;
    const int grid = grid_for_groups(c, (n_in + 63) / 64);
    const ListSlots ls{-1, level % 3};
    if (from_list)
        hipLaunchKernelGGL(k_active<true>, dim3(grid), dim3(kBlock), 0, s, *g, *st, ls);
    else
        hipLaunchKernelGGL(k_active<false>, dim3(grid), dim3(kBlock), 0, s, *g, *st, ls);
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_cb_supported(const albd_graph *g)
{
    // summary bitmap (one bit per frontier word) must fit the LDS budget
    const int64_t bytes = (((int64_t)g->nwords + 63) / 64) * 8;
    return bytes <= 64 * 1024;
}

int albd_prep(albd_ctx *c, const albd_graph *g, const albd_state *st, int from_list, int summary, int32_t level)
{
    const int grid = grid_for_groups(c, ((int64_t)g->nwords + 63) / 64);
    hipStream_t s = albd_stream(c);
    const ListSlots ls{-1, level % 3};
    if (from_list) {
        if (summary) hipLaunchKernelGGL((k_prep<true, true>), dim3(grid), dim3(kBlock), 0, s, *g, *st, ls);
        else hipLaunchKernelGGL((k_prep<true, false>), dim3(grid), dim3(kBlock), 0, s, *g, *st, ls);
    } else {
        if (summary) hipLaunchKernelGGL((k_prep<false, true>), dim3(grid), dim3(kBlock), 0, s, *g, *st, ls);
        else hipLaunchKernelGGL((k_prep<false, false>), dim3(grid), dim3(kBlock), 0, s, *g, *st, ls);
    }
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_select_prep_post(albd_ctx *c, const albd_graph *g, const albd_state *st, const albd_select_args *sel,
                          unsigned int *seq, int from_list, int summary)
{
    albd_counters *mail = albd_mail_next(c, seq);
    // one select block in front of the preparation's grid
    const int grid = 1 + grid_for_groups(c, ((int64_t)g->nwords + 63) / 64);
    hipStream_t s = albd_stream(c);
    const bool list_used = !sel->first && (sel->prev_choice == ALBBA_CHOICE_PULL_SB ||
                                           sel->prev_choice == ALBBA_CHOICE_PULL_CB);
    const ListSlots ls{list_used ? (sel->level + 2) % 3 : -1, sel->level % 3};
    const unsigned int q = *seq;
    if (from_list) {
        if (summary)
            hipLaunchKernelGGL((k_select_prep<true, true>), dim3(grid), dim3(kBlock), 0, s, *g, *st, *sel, mail, q, ls);
        else
            hipLaunchKernelGGL((k_select_prep<true, false>), dim3(grid), dim3(kBlock), 0, s, *g, *st, *sel, mail, q, ls);
    } else {
        if (summary)
            hipLaunchKernelGGL((k_select_prep<false, true>), dim3(grid), dim3(kBlock), 0, s, *g, *st, *sel, mail, q, ls);
        else
            hipLaunchKernelGGL((k_select_prep<false, false>), dim3(grid), dim3(kBlock), 0, s, *g, *st, *sel, mail, q, ls);
    }
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_build_summary(albd_ctx *c, const albd_graph *g, const albd_state *st)
{
    const int grid = grid_for_groups(c, ((int64_t)g->nwords + 63) / 64);
    hipLaunchKernelGGL(k_summary, dim3(grid), dim3(kBlock), 0, albd_stream(c), *g, *st);
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_pull(albd_ctx *c, const albd_graph *g, const albd_state *st, int variant, int32_t level,
              int64_t items_bound)
{
    return albd_pull_spec(c, g, st, variant, level, items_bound, -1);
}

int albd_pull_spec(albd_ctx *c, const albd_graph *g, const albd_state *st, int variant, int32_t level,
                   int64_t items_bound, int spec)
{
    PullArgs a;
    a.g = *g;
    a.st = *st;
    a.level = level;
    a.spec = spec;
    a.spec_choice = variant == ALBD_PULL_ALL ? ALBBA_CHOICE_PULL
                                             : (variant == ALBD_PULL_LIST ? ALBBA_CHOICE_PULL_SB : ALBBA_CHOICE_PULL_CB);
    // the list level `level`'s preparation built, and its count
    a.items = st->active_next;
    a.nitems = &st->ctr->list_cnt[level % 3];
    a.per_block = 16;
    const int64_t sum_words64 = ((int64_t)g->nwords + 63) / 64;
    a.sum_words32 = (int32_t)(sum_words64 * 2);
    size_t lds = 0;
    if (variant == ALBD_PULL_LIST_CB) {
        if (!albd_cb_supported(g)) return albd_set_error_msg(ALBBA_EINVAL, "column bypass: graph too large for the LDS summary");
        lds = (size_t)a.sum_words32 * 4;
    }
    // items: every word, or an upper bound of the list length the device holds
    int64_t items = g->nwords;
    if (variant != ALBD_PULL_ALL && items_bound > 0 && items_bound < items) items = items_bound;
    switch (g->C) {
    case 16: return launch_pull_c<16>(c, a, variant, lds, items);
    case 32: return launch_pull_c<32>(c, a, variant, lds, items);
    case 64: return launch_pull_c<64>(c, a, variant, lds, items);
    case 128: return launch_pull_c<128>(c, a, variant, lds, items);
    default: return albd_set_error_msg(ALBBA_EINVAL, "pull: unsupported slice height");
    }
}

int albd_front_to_queue(albd_ctx *c, const albd_graph *g, const albd_state *st)
{
    hipLaunchKernelGGL(k_words_to_queue<false>, dim3(grid_for_queue(c, g)), dim3(kQBlock), 0, albd_stream(c), *g, *st,
                       0, kNoSpec, LLONG_MAX, words_per_wave(g));
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_push_scan(albd_ctx *c, const albd_graph *g, const albd_state *st, int64_t qlen)
{
    hipStream_t s = albd_stream(c);
    if (qlen <= ALBD_SPEC_PUSH_MAX) {
        hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(kBlock), 0, s, *g, *st, kNoSpec);
        HIPCHK(hipGetLastError());
        return 0;
    }
    hipLaunchKernelGGL(k_scan_p1, dim3(ALBD_SCAN_BLOCKS), dim3(kBlock), 0, s, *g, *st);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_scan_p2, dim3(1), dim3(kBlock), 0, s, *st, (int32_t)ALBD_SCAN_BLOCKS);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_scan_p3, dim3(ALBD_SCAN_BLOCKS), dim3(kBlock), 0, s, *st);
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_push_expand(albd_ctx *c, const albd_graph *g, const albd_state *st)
{
    hipLaunchKernelGGL(k_push_expand, dim3(grid_persistent(c, 8)), dim3(kBlock), 0, albd_stream(c), *g, *st,
                       kNoSpec);
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_push_small(albd_ctx *c, const albd_graph *g, const albd_state *st, int32_t level0,
                    int64_t edge_cap, int64_t vertex_cap, int32_t max_levels, int32_t blocks,
                    uint32_t spin_limit)
{
    if (max_levels > ALBD_PERSIST_LEVELS) max_levels = ALBD_PERSIST_LEVELS;
    if (max_levels < 1) max_levels = 1;
    // Every workgroup of the grid barrier must be resident at once: the grid
    // is at most what the occupancy allows on every CU together, and the
    // launch is an ordinary one on the context's stream, whose earlier
    // kernels have finished before it starts (stream order).  A workgroup
    // that could not become resident would only make the barrier give up
    // after spin_limit polls (ctr->persist_error), never hang.
    int per_cu = 0;
    HIPCHK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_push_small, kListBlock, 0));
    int64_t cap = (int64_t)per_cu * albd_num_cus(c);
    if (cap < 1) return albd_set_error_msg(ALBBA_EHIP, "small-frontier kernel cannot be resident");
    if (cap > ALBD_PERSIST_BLOCKS) cap = ALBD_PERSIST_BLOCKS;
    // the found list (2 (npos + 1) entries) holds every vertex and the up to
    // two unfilled reservations of every workgroup (one workgroup's are in order,
    // so that its vertices alone fit)
    if (cap > g->npos / (2 * kFound)) cap = g->npos / (2 * kFound);
    if (cap < 1) cap = 1;
    // More workgroups shorten each one's part of a level but lengthen the
    // barrier: measured us per level with 16, 32 and 64 workgroups on grids of
    // 0.6, 2.3, 4.2, 7.3 and 16.8 M vertices: 4.1, 4.4, 4.9; 4.8, 4.5, 4.8; 4.8,
    // 4.5, 4.8; 6.9, 5.5, 5.1; 8.5, 6.5, 5.4 (96 workgroups: 5.2-5.6).
    if (blocks <= 0) blocks = g->n < (1 << 20) ? 16 : (g->n < 5 << 20 ? 32 : 64);
    if (blocks > cap) blocks = (int32_t)cap;
    // the grid state, the levels' counters and the error flag were zeroed by
    // the level-begin kernel (ALBD_LB_SMALL)
    SmallArgs a{*g, *st, level0, max_levels, edge_cap, vertex_cap, spin_limit};
    hipLaunchKernelGGL(k_push_small, dim3(blocks), dim3(kListBlock), 0, albd_stream(c), a);
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_select_post(albd_ctx *c, const albd_graph *g, const albd_state *st,
                     const albd_select_args *sel, unsigned int *seq)
{
    albd_counters *mail = albd_mail_next(c, seq);
    hipLaunchKernelGGL(k_select, dim3(1), dim3(kSelectBlock), 0, albd_stream(c), *g, *st, *sel, mail,
                       *seq);
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_select_read(albd_ctx *c, const albd_graph *g, const albd_state *st,
                     const albd_select_args *sel)
{
    unsigned int seq;
    if (int rc = albd_select_post(c, g, st, sel, &seq)) return rc;
    return albd_mail_wait(c, st, seq);
}

int albd_push_finalize(albd_ctx *c, const albd_graph *g, const albd_state *st, int32_t level, int64_t build_max)
{
    hipLaunchKernelGGL(k_words_to_queue<true>, dim3(grid_for_queue(c, g)), dim3(kQBlock), 0, albd_stream(c), *g, *st,
                       level, kNoSpec, (long long)build_max, words_per_wave(g));
    HIPCHK(hipGetLastError());
    return 0;
}

int albd_push_spec(albd_ctx *c, const albd_graph *g, const albd_state *st, int32_t level, int spec,
                   int64_t build_max, int scan)
{
    // with a scan, the frontier bound is the one below which albd_push_scan
    // takes the one-block scan
    const Spec sp{spec, ALBBA_CHOICE_PUSH, scan ? (unsigned long long)ALBD_SPEC_PUSH_MAX : ~0ull};
    hipStream_t s = albd_stream(c);
    if (scan) {
        hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(kBlock), 0, s, *g, *st, sp);
        HIPCHK(hipGetLastError());
    }
    hipLaunchKernelGGL(k_push_expand, dim3(grid_persistent(c, 8)), dim3(kBlock), 0, s, *g, *st, sp);
    HIPCHK(hipGetLastError());
    hipLaunchKernelGGL(k_words_to_queue<true>, dim3(grid_for_queue(c, g)), dim3(kQBlock), 0, s, *g, *st, level, sp,
                       (long long)build_max, words_per_wave(g));
    HIPCHK(hipGetLastError());
    return 0;
}

} // extern "C"
