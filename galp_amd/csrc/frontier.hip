// frontier.hip -- iterations over the rows that can still change.
//
// No reference counterpart: the reference's propagators walk every edge in
// every iteration (lfht.cuh:115-167, dpp.cuh:104-138).  The update is a
// function of the row's neighbour labels, so a vertex none of whose
// neighbours changed in iteration t-1 gets in iteration t the label it got
// in t-1.  Once labels settle almost no row has a changed neighbour (RMAT-20:
// rows holding 23 % of the edges in iteration 6, 3 % from iteration 7;
// LFR-1M: 52, 24, 12 and 8 % in iterations 7 to 10), and the class kernels
// then walk lists of the others only.  The labels and the change counts are
// those of the full pass.
//
// The two label buffers hold iterations t-1 and t-2, so "changed" is a
// comparison of them.  Before an iteration:
//   k_front_count  sums the degrees of the vertices that changed;
//   k_front_mark   if that is a small share of the edges, copies the changed
//                  labels into the other buffer (a vertex left out of the
//                  iteration then holds its label in both) and marks every
//                  neighbour of a changed vertex.  The graph must be
//                  symmetric: v's row holds u exactly when u's holds v, which
//                  the upload checks (k_check_symmetric);
//   k_front_lists  appends the marked vertices to their class's list and sums
//                  the lists' edges.
// The choice is made on the device (front_lists_on), so the loop needs no
// readback and can be captured: the class kernels take their list or their
// whole class.
// Out of core the lists save the copies, not only the gathers: the host reads
// the control words and queues either the batches or the class kernels on the
// lists, whose rows, like those of k_front_mark, are then read from the pinned
// array over the link (ooc.hip).

#include <algorithm>
#include <new>
#include <string>

#include "device_common.hpp"
#include "internal.hpp"

namespace galp {

// A vertex count above which marking cannot pay: half of the vertices
// changed.  Tested first, so that the early iterations cost three empty
// launches.
__device__ __forceinline__ bool front_many_changed(const long long *updated, int64_t n) {
    return 2 * (int64_t)*updated > n;
}

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long x) {
#pragma unroll
    for (int s = kWave / 2; s > 0; s >>= 1) x += __shfl_xor(x, s);
    return x;
}

// ---------------------------------------------------------------------------
// Symmetry of a CSR whose rows strictly ascend (by id, or by iperm[id] for
// rows in the internal numbering).  Order the vertices by
// (degree, id): every edge to a lower vertex is looked up in that vertex's
// (shorter) row by binary search.  Rows hold no vertex twice, so the matches
// are one to one, and the graph is symmetric when every downward edge has a
// match and there are as many upward edges as downward ones.  res[0]: a
// downward edge without a match; res[1] (64-bit, at res + 2): downward minus
// upward edges.  A block takes kSymTile consecutive edges and finds their
// rows by binary search in the offsets.
constexpr int kSymTile = 2048;
template <typename E>
__global__ void __launch_bounds__(256)
k_check_symmetric(const E *__restrict__ off, const int32_t *__restrict__ nbr, const int32_t *__restrict__ iperm,
                  int64_t n, int64_t m, int32_t *__restrict__ res) {
    __shared__ int64_t srow[2];
    __shared__ long long sbal[256 / kWave];
    long long balance = 0;
    bool miss = false;
    // the last row r with off[r] <= e, r in [lo, hi)
    auto row_of = [&](int64_t e, int64_t lo, int64_t hi) {
        while (hi - lo > 1) {
            const int64_t mid = (lo + hi) >> 1;
            if ((int64_t)off[mid] <= e) lo = mid;
            else hi = mid;
        }
        return lo;
    };
    for (int64_t e0 = (int64_t)blockIdx.x * kSymTile; e0 < m; e0 += (int64_t)gridDim.x * kSymTile) {
        const int64_t e1 = min(e0 + kSymTile, m);
        __syncthreads();
        if (threadIdx.x < 2) srow[threadIdx.x] = row_of(threadIdx.x ? e1 - 1 : e0, 0, n);
        __syncthreads();
        const int64_t r0 = srow[0], r1 = srow[1];
        for (int64_t e = e0 + threadIdx.x; e < e1; e += 256) {
            const int64_t v = row_of(e, r0, r1 + 1);
            const int64_t u = nbr[e];
            if (u == v) continue;
            const int64_t dv = (int64_t)off[v + 1] - (int64_t)off[v];
            const int64_t b = (int64_t)off[u], du = (int64_t)off[u + 1] - b;
            if (du > dv || (du == dv && u > v)) {
                --balance;
                continue;
            }
            ++balance;
            const int32_t key = iperm ? iperm[v] : (int32_t)v;
            int64_t lo = b, hi = b + du;   // first position of u's row holding an id >= v
            while (lo < hi) {
                const int64_t mid = (lo + hi) >> 1;
                const int32_t x = nbr[mid];
                if ((iperm ? iperm[x] : x) < key) lo = mid + 1;
                else hi = mid;
            }
            miss |= lo == b + du || (int64_t)nbr[lo] != v;
        }
    }
    if (miss) res[0] = 1;   // every writer writes the same word
    balance = (long long)wave_sum_u64((unsigned long long)balance);
    if (lane_id() == 0) sbal[threadIdx.x / kWave] = balance;
    __syncthreads();
    if (threadIdx.x == 0) {
        long long t = 0;
        for (int w = 0; w < 256 / kWave; ++w) t += sbal[w];
        if (t) atomicAdd((unsigned long long *)(res + 2), (unsigned long long)t);
    }
}

// ---------------------------------------------------------------------------
// Degrees of the vertices that changed in the last iteration, summed into
// ctl[kFrontPush]: a stream over both label buffers, one block per CU (the
// blocks' atomics on the one word then cost 4 us).
constexpr int kFrontThreads = 1024;
template <typename E>
__global__ void __launch_bounds__(kFrontThreads)
k_front_count(const E *__restrict__ off, const int32_t *__restrict__ cur, const int32_t *__restrict__ old,
              int64_t n, const long long *__restrict__ updated, int64_t *__restrict__ ctl,
              const int32_t *__restrict__ stop) {
    __shared__ unsigned long long ssum[kFrontThreads / kWave];
    if (*stop || front_many_changed(updated, n)) return;
    const int64_t nthreads = (int64_t)gridDim.x * kFrontThreads;
    unsigned long long push = 0;
    for (int64_t v0 = (int64_t)blockIdx.x * kFrontThreads + threadIdx.x; v0 < n; v0 += 4 * nthreads) {
        int32_t a[4], b[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int64_t v = v0 + k * nthreads < n ? v0 + k * nthreads : v0;
            a[k] = cur[v];
            b[k] = old[v];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int64_t v = v0 + k * nthreads;
            if (v < n && a[k] != b[k]) push += (unsigned long long)((int64_t)off[v + 1] - (int64_t)off[v]);
        }
    }
    push = wave_sum_u64(push);
    if (lane_id() == 0) ssum[threadIdx.x / kWave] = push;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long t = 0;
        for (int w = 0; w < kFrontThreads / kWave; ++w) t += ssum[w];
        if (t) atomicAdd((unsigned long long *)(ctl + kFrontPush), t);
    }
}

// Marks the neighbours of every changed vertex.  A wave takes 64 vertices;
// the rows of those that changed are walked as one flat range of edges (an
// exclusive scan of their degrees in LDS, searched per edge), so that short
// rows fill the lanes.  Hub rows are left out and walked tile by tile by all
// waves; their labels are copied by k_front_lists, after every tile has
// compared them.
constexpr int kMarkThreads = 256;
template <typename E>
__global__ void __launch_bounds__(kMarkThreads)
k_front_mark(const E *__restrict__ off, const int32_t *__restrict__ nbr, const int32_t *__restrict__ cur,
             int32_t *__restrict__ old, int64_t n, int64_t max_push, const int32_t *__restrict__ tile_hub,
             const int32_t *__restrict__ hub_tile0, const int32_t *__restrict__ hub_vid, int64_t ntiles,
             const long long *__restrict__ updated, uint8_t *__restrict__ mark, int32_t *__restrict__ hub_sel,
             int64_t nhubs, const int64_t *__restrict__ ctl, const int32_t *__restrict__ stop) {
    constexpr int NW = kMarkThreads / kWave;
    __shared__ int32_t sstart[NW][kWave];
    __shared__ int64_t sbase[NW][kWave];
    if (*stop || front_many_changed(updated, n) || ctl[kFrontPush] > max_push) return;
    const int lane = lane_id(), w = (int)(threadIdx.x / kWave);
    const int64_t wave = (int64_t)blockIdx.x * NW + w, nwaves = (int64_t)gridDim.x * NW;
    for (int64_t h = (int64_t)blockIdx.x * kMarkThreads + threadIdx.x; h < nhubs;
         h += (int64_t)gridDim.x * kMarkThreads)
        hub_sel[h] = 0;   // set by k_front_lists
    for (int64_t v0 = wave * kWave; v0 < n; v0 += nwaves * kWave) {
        const int64_t v = v0 + lane;
        bool ch = false;
        int32_t a = 0;
        if (v < n) {
            a = cur[v];
            ch = a != old[v];
        }
        if (!__ballot(ch)) continue;
        int32_t len = 0;
        int64_t b = 0;
        if (ch) {
            b = (int64_t)off[v];
            const int64_t d = (int64_t)off[v + 1] - b;
            if (d <= bucket_hi(B_B4K)) {
                len = (int32_t)d;
                old[v] = a;
            }
        }
        int st = len;   // exclusive scan of the row lengths
#pragma unroll
        for (int s = 1; s < kWave; s <<= 1) {
            const int y = __shfl_up(st, s);
            if (lane >= s) st += y;
        }
        const int total = __shfl(st, kWave - 1);
        sstart[w][lane] = st - len;
        sbase[w][lane] = b;
        __builtin_amdgcn_wave_barrier();
        for (int i = lane; i < total; i += kWave) {
            int r = 0;   // last lane with start <= i
#pragma unroll
            for (int s = kWave / 2; s > 0; s >>= 1)
                if (sstart[w][r + s] <= i) r += s;
            mark[nbr[sbase[w][r] + (i - sstart[w][r])]] = 1;
        }
        __builtin_amdgcn_wave_barrier();   // rewritten by the next 64 vertices
    }
    for (int64_t t = wave; t < ntiles; t += nwaves) {
        const int h = tile_hub[t];
        const int64_t v = hub_vid[h];
        if (cur[v] == old[v]) continue;
        const int64_t e0 = (int64_t)off[v] + (t - (int64_t)hub_tile0[h]) * (int64_t)kHubTile;
        const int64_t e1 = min(e0 + kHubTile, (int64_t)off[v + 1]);
        for (int64_t e = e0 + lane; e < e1; e += kWave) mark[nbr[e]] = 1;
    }
}

// Appends the marked vertices to their classes' lists (list b starts at
// lists + v0[b]) and clears the marks; a marked hub sets its flag and appends
// its tiles to the tile list.  Appends are aggregated per block and 4096
// vertices, as in k_batch_lists.  The edges of each list are summed beside
// its length: every class kernel adds them up and takes the lists when they
// hold few enough edges (front_lists_on).  No block waits for the others: a
// last-block decision needs a device-wide fence in every block, which wrote
// back the L2s: 80 us on RMAT-22 against 30.
struct FrontSpans {
    int64_t v0[NUM_BUCKETS];   // where each class's list starts
};
constexpr int kFrontItems = 4;   // marks per thread and chunk, one 32-bit load
template <typename E>
__global__ void __launch_bounds__(kFrontThreads)
k_front_lists(FrontSpans fs, const E *__restrict__ off, const int32_t *__restrict__ cur, int32_t *__restrict__ old,
              int64_t n, int64_t max_push, const int32_t *__restrict__ hub_vid, int64_t nhubs,
              const int32_t *__restrict__ hub_tile0, const int32_t *__restrict__ hub_ntiles,
              const long long *__restrict__ updated, uint32_t *__restrict__ mark, int32_t *__restrict__ lists,
              int32_t *__restrict__ hub_sel, int32_t *__restrict__ tiles, int64_t *__restrict__ ctl,
              const int32_t *__restrict__ stop) {
    constexpr int64_t kChunk = (int64_t)kFrontThreads * kFrontItems;
    __shared__ uint32_t scnt[NUM_BUCKETS];   // hubs: their tiles
    __shared__ int64_t sbase[NUM_BUCKETS];
    __shared__ unsigned long long sedges[NUM_BUCKETS];
    if (*stop || front_many_changed(updated, n) || ctl[kFrontPush] > max_push) return;
    if (threadIdx.x < NUM_BUCKETS) sedges[threadIdx.x] = 0ull;
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl[kFrontReady] = 1;
    // the hubs' labels, which k_front_mark left to this kernel
    for (int64_t h = (int64_t)blockIdx.x * kFrontThreads + threadIdx.x; h < nhubs;
         h += (int64_t)gridDim.x * kFrontThreads) {
        const int64_t v = hub_vid[h];
        const int32_t a = cur[v];
        if (old[v] != a) old[v] = a;
    }
    const unsigned long long lt = (1ull << lane_id()) - 1ull;
    for (int64_t c0 = (int64_t)blockIdx.x * kChunk; c0 < n; c0 += (int64_t)gridDim.x * kChunk) {
        const int64_t vb = c0 + (int64_t)threadIdx.x * kFrontItems;
        const uint32_t word = vb < n ? mark[vb / kFrontItems] : 0u;   // the array is padded to whole words
        if (!__syncthreads_or(word != 0u)) continue;
        if (threadIdx.x < NUM_BUCKETS) scnt[threadIdx.x] = 0u;
        __syncthreads();
        int cls[kFrontItems];
        uint32_t rank[kFrontItems];
        int32_t hub[kFrontItems];
#pragma unroll
        for (int r = 0; r < kFrontItems; ++r) {
            bool keep = (word >> (8 * r)) & 0xffu;
            int b = -1;
            uint32_t d = 0;
            hub[r] = -1;
            rank[r] = 0u;
            if (keep) {
                const int64_t dd = (int64_t)off[vb + r + 1] - (int64_t)off[vb + r];
                b = bucket_of_deg(dd);
                d = (uint32_t)dd;
                if (b == B_HUB) {
                    int64_t lo = 0, hi = nhubs;   // hub_vid ascends
                    while (hi - lo > 1) {
                        const int64_t mid = (lo + hi) >> 1;
                        if ((int64_t)hub_vid[mid] <= vb + r) lo = mid;
                        else hi = mid;
                    }
                    hub[r] = (int32_t)lo;
                    hub_sel[lo] = 1;
                    rank[r] = atomicAdd(&scnt[B_HUB], (uint32_t)hub_ntiles[lo]);
                    atomicAdd(&sedges[B_HUB], (unsigned long long)dd);
                    keep = false;
                }
            }
            cls[r] = b;
            unsigned long long ball;
            while ((ball = __ballot(keep)) != 0ull) {
                const int leader = __ffsll((long long)ball) - 1;
                const int bl = __builtin_amdgcn_readlane(b, leader);
                const bool mine = keep && b == bl;
                const unsigned long long mm = __ballot(mine);
                const uint32_t es = wave_sum_u32(mine ? d : 0u);   // at most 64 rows of 4096
                uint32_t at = 0u;
                if (lane_id() == leader) {
                    at = atomicAdd(&scnt[bl], (uint32_t)__popcll(mm));
                    atomicAdd(&sedges[bl], (unsigned long long)es);
                }
                at = (uint32_t)__shfl((int)at, leader);
                if (mine) rank[r] = at + (uint32_t)__popcll(mm & lt);
                keep = keep && !mine;
            }
        }
        if (word) mark[vb / kFrontItems] = 0u;
        __syncthreads();
        if (threadIdx.x < NUM_BUCKETS && scnt[threadIdx.x])
            sbase[threadIdx.x] = (int64_t)atomicAdd((unsigned long long *)(ctl + threadIdx.x),
                                                    (unsigned long long)scnt[threadIdx.x]);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kFrontItems; ++r) {
            if (cls[r] < 0) continue;
            const int64_t at = sbase[cls[r]] + rank[r];
            if (hub[r] >= 0) {
                const int32_t t0 = hub_tile0[hub[r]], nt = hub_ntiles[hub[r]];
                for (int32_t t = 0; t < nt; ++t) tiles[at + t] = t0 + t;
            } else {
                lists[fs.v0[cls[r]] + at] = (int32_t)(vb + r);
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < NUM_BUCKETS && sedges[threadIdx.x])
        atomicAdd((unsigned long long *)(ctl + kFrontEdges + threadIdx.x), sedges[threadIdx.x]);
}

// Per-kernel profiling: each class's algorithmic bytes of this iteration, as
// class_bytes counts them, for the rows the class kernel will walk.
struct FrontBytes {
    int64_t nv[NUM_BUCKETS], edges[NUM_BUCKETS];
};
__global__ void k_front_bytes(FrontBytes fb, int esz, FrontList front, int64_t *__restrict__ bytes) {
    const int b = (int)threadIdx.x;
    if (b >= NUM_BUCKETS) return;
    const bool lists = front_lists_on(front);
    const int64_t *ctl = front.ctl;
    const int64_t nv = lists ? ctl[b] : fb.nv[b], edges = lists ? ctl[kFrontEdges + b] : fb.edges[b];
    bytes[b] = b == B_HUB ? 8 * edges : nv ? esz * (nv + 1) + 8 * edges + 8 * nv : 0;
}

// ---------------------------------------------------------------------------
// Host side.

void front_free(galp_graph *g) {
    FrontState *F = g->front;
    if (!F) return;
    if (F->d_mem) (void)hipFree(F->d_mem);
    if (F->d_bytes) (void)hipFree(F->d_bytes);
    delete F;
    g->front = nullptr;
}

// Whether a CSR on the device (rows strictly ascending) is symmetric.
int dev_check_symmetric(galp_graph *g, const void *off, bool off64, const int32_t *nbr, const int32_t *iperm,
                        bool *symmetric) {
    *symmetric = true;
    if (!g->m) return GALP_OK;
    int32_t *res = (int32_t *)g->d_counter;   // free until the first init; 16 bytes of it
    int rc = dev_fill_u32(g, (uint32_t *)res, 4, 0u);
    if (rc != GALP_OK) return rc;
    const int grid = (int)std::min<int64_t>((g->m + kSymTile - 1) / kSymTile,
                                            (int64_t)g->ctx->prop.multiProcessorCount * 8);
    if (off64) k_check_symmetric<int64_t><<<grid, 256, 0, g->stream>>>((const int64_t *)off, nbr, iperm, g->n, g->m, res);
    else k_check_symmetric<int32_t><<<grid, 256, 0, g->stream>>>((const int32_t *)off, nbr, iperm, g->n, g->m, res);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(g->h_pinned, res, 16, hipMemcpyDeviceToHost, g->stream) != hipSuccess ||
        hipStreamSynchronize(g->stream) != hipSuccess)
        return fail(g->ctx, GALP_EHIP, "symmetry check failed");
    *symmetric = g->h_pinned[0] == 0 && g->h_pinned[2] == 0 && g->h_pinned[3] == 0;
    return GALP_OK;
}

// The lists' memory: n marks, n list entries and, for per-kernel profiling, the
// classes' bytes per iteration.  Optional: a graph whose memory
// budget has no room for it, or that leaves less than 64 bytes a vertex free
// on the card (what learned dispatch or a batch may still ask for), runs
// every iteration over all rows.
int front_setup(galp_graph *g) {
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) != hipSuccess || (int64_t)(fr / 64) < g->n + kFrontCtl) return GALP_OK;
    FrontState *F = new (std::nothrow) FrontState();
    if (!F) return fail(g->ctx, GALP_ENOMEM, "host allocation failed");
    g->front = F;
    // one allocation: the control words, one mark per vertex, the class lists,
    // the hubs' flags and tiles, cleared (the lane-group pipeline reads entry 0
    // of a list even when it is empty)
    const int64_t words = (g->n + kFrontItems - 1) / kFrontItems;
    const int64_t total = 2 * kFrontCtl + words + g->n + g->nhubs + g->nhub_tiles;
    const std::string err = g->ctx->err;
    const int64_t before = g->device_bytes;
    if (dev_alloc(g, &F->d_mem, total) != GALP_OK ||
        (g->opts.profile && dev_alloc(g, &F->d_bytes, (int64_t)kMaxIters * NUM_BUCKETS) != GALP_OK)) {
        front_free(g);
        g->device_bytes = before;
        g->ctx->err = err;   // doing without is no failure
        return GALP_OK;
    }
    F->d_ctl = (int64_t *)F->d_mem;
    F->d_mark = F->d_mem + 2 * kFrontCtl;
    F->d_lists = (int32_t *)(F->d_mark + words);
    F->d_hub_sel = F->d_lists + g->n;
    F->d_tiles = F->d_hub_sel + g->nhubs;
    return dev_fill_u32(g, F->d_mem, total, 0u);
}

bool front_now(const galp_graph *g) {
    if (!g->front || (g->learn && g->learn->log_cap)) return false;
    // after the first iteration from labels[i] = i nearly every label is new
    return g->iter >= (g->identity ? 2 : 1);
}

template <typename E>
static void front_launch(galp_graph *g, FrontState *F) {
    const int32_t *cur = g->d_lab[g->cur];
    int32_t *old = g->d_lab[g->cur ^ 1];
    const E *off = (const E *)g->d_off;
    const long long *updated = g->d_iter_counts + (g->iter - 1) % kMaxIters;
    const int cus = g->ctx->prop.multiProcessorCount;
    const int64_t max_push = g->m / (g->ooc ? kFrontPushDivOoc : kFrontPushDiv);
    const int32_t *nbr = g->ooc ? g->ooc->h_nbr : g->d_nbr;   // pinned host memory is mapped
    FrontSpans fs{};
    for (int b = 0; b < NUM_BUCKETS; ++b) fs.v0[b] = g->bucket[b].v0;
    const int grid_c = (int)std::min<int64_t>((g->n + kFrontThreads - 1) / kFrontThreads, cus);
    k_front_count<E><<<grid_c, kFrontThreads, 0, g->stream>>>(off, cur, old, g->n, updated, F->d_ctl, g->d_stop);
    const int grid_m = (int)std::min<int64_t>((g->n + kMarkThreads - 1) / kMarkThreads, (int64_t)cus * 8);
    k_front_mark<E><<<grid_m, kMarkThreads, 0, g->stream>>>(off, nbr, cur, old, g->n, max_push, g->d_tile_hub,
                                                           g->d_hub_tile0, g->d_hub_vid, g->nhub_tiles, updated,
                                                           (uint8_t *)F->d_mark, F->d_hub_sel, g->nhubs, F->d_ctl,
                                                           g->d_stop);
    const int64_t chunk = (int64_t)kFrontThreads * kFrontItems;
    const int grid_l = (int)std::min<int64_t>((g->n + chunk - 1) / chunk, cus);
    k_front_lists<E><<<grid_l, kFrontThreads, 0, g->stream>>>(
        fs, off, cur, old, g->n, max_push, g->d_hub_vid, g->nhubs, g->d_hub_tile0, g->d_hub_ntiles, updated, F->d_mark,
        F->d_lists, F->d_hub_sel, F->d_tiles, F->d_ctl, g->d_stop);
}

int launch_front(galp_graph *g) {
    FrontState *F = g->front;
    PendingLaunch pl;
    prof_begin(g, "front", 0.0, &pl);
    if (g->off64) front_launch<int64_t>(g, F);
    else front_launch<int32_t>(g, F);
    prof_end(g, &pl);
    if (g->prof.on && F->d_bytes) {
        FrontBytes fb{};
        for (int b = 0; b < NUM_BUCKETS; ++b) {
            fb.nv[b] = g->bucket[b].nv;
            fb.edges[b] = g->bucket[b].edges;
        }
        k_front_bytes<<<1, kWave, 0, g->stream>>>(fb, g->off64 ? 8 : 4, front_hubs(g),
                                                  F->d_bytes + (int64_t)(g->iter % kMaxIters) * NUM_BUCKETS);
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? GALP_OK : fail(g->ctx, GALP_EHIP, std::string("frontier launch: ") + hipGetErrorString(e));
}

}  // namespace galp
