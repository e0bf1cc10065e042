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
#include <atomic>
#include <chrono>
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
// Symmetry of a CSR, in any numbering, by Freivalds' method (1977): with A
// its adjacency matrix (an entry counts a row's occurrences of a vertex) and x,
// y random vectors, x'Ay - y'Ax = x'(A - A')y is 0 if A is symmetric, and else
// hardly ever.  In 64-bit wrapping arithmetic, where A - A' has an entry of +-1
// (rows hold no vertex twice): c = (A - A')y is then uniform in that row, and
// x'c = 0 for a share of 2^(t - 64) of x, t the trailing zeros of c; summed
// over t, less than 2^-58.  x and y are splitmix64 of the vertex id under two
// seeds drawn for each upload.  sum (64-bit) receives the difference.
// A stream over the neighbour ids, eight consecutive edges a thread, whose row
// is found by binary search and followed from there; bound by the ids'
// hashing.  Looking up each edge's reverse by binary search instead costs a
// line or two per edge: RMAT-22 (128 M edges) 6.9 ms, more than the lists save
// in a run of ten iterations, against 0.36 ms.
// ROWS (out of core, where the ids come over the link and nothing else has read
// them): sets *bad when a row's ids (input numbering: iperm, may be null) do not
// strictly ascend, and records each row's last neighbour.
constexpr int kSymThreads = 256;
constexpr int kSymEdges = 8;                                  // per thread and round
constexpr int kSymTile = 4 * kSymThreads * kSymEdges;
__host__ __device__ inline unsigned long long splitmix64(unsigned long long z) {
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}
template <typename E, bool ROWS>
__global__ void __launch_bounds__(kSymThreads)
k_check_symmetric(const E *__restrict__ off, const int32_t *__restrict__ nbr, int64_t n, int64_t m,
                  unsigned long long seed_x, unsigned long long seed_y, unsigned long long *__restrict__ sum,
                  const int32_t *__restrict__ iperm, int32_t *__restrict__ last, int32_t *__restrict__ bad) {
    __shared__ int64_t srow[2];
    __shared__ unsigned long long ssum[kSymThreads / kWave];
    using U = unsigned long long;
    auto at = [](U seed, int64_t v) { return splitmix64(seed + (U)v * 0x9e3779b97f4a7c15ull); };
    // the last row r with off[r] <= e, r in [lo, hi)
    auto row_of = [&](int64_t e, int64_t lo, int64_t hi) {
        while (hi - lo > 1) {
            const int64_t mid = (lo + hi) >> 1;
            if ((int64_t)off[mid] <= e) lo = mid;
            else hi = mid;
        }
        return lo;
    };
    U acc = 0;
    bool out_of_order = false;
    for (int64_t e0 = (int64_t)blockIdx.x * kSymTile; e0 < m; e0 += (int64_t)gridDim.x * kSymTile) {
        const int64_t e1 = min(e0 + kSymTile, m);
        __syncthreads();
        if (threadIdx.x < 2) srow[threadIdx.x] = row_of(threadIdx.x ? e1 - 1 : e0, 0, n);
        __syncthreads();
        const int64_t r0 = srow[0], r1 = srow[1];
        for (int64_t e = e0 + kSymEdges * (int64_t)threadIdx.x; e < e1; e += kSymEdges * kSymThreads) {
            int32_t u[kSymEdges];
            const int k = (int)min((int64_t)kSymEdges, e1 - e);
            if (k == kSymEdges) {   // tiles start at multiples of eight edges
                const int4 a = *(const int4 *)(nbr + e), b = *(const int4 *)(nbr + e + 4);
                u[0] = a.x, u[1] = a.y, u[2] = a.z, u[3] = a.w;
                u[4] = b.x, u[5] = b.y, u[6] = b.z, u[7] = b.w;
            } else {
#pragma unroll
                for (int j = 0; j < kSymEdges; ++j) u[j] = j < k ? nbr[e + j] : 0;
            }
            int64_t v = row_of(e, r0, r1 + 1), end = (int64_t)off[v + 1];
            int32_t before = -1;   // the row's id before e; ids are not negative
            if constexpr (ROWS) {
                // the lane below holds the edge before this lane's (lanes past
                // e1 are the upper ones)
                const int32_t tail = __shfl_up(u[kSymEdges - 1], 1);
                if (e > (int64_t)off[v]) {
                    before = lane_id() ? tail : nbr[e - 1];
                    if (iperm) before = iperm[before];
                }
            }
            U sx = 0, sy = 0;   // over the row's edges so far
#pragma unroll
            for (int j = 0; j < kSymEdges; ++j) {
                if (j < k) {
                    if (e + j >= end) {
                        acc += at(seed_x, v) * sy - at(seed_y, v) * sx;
                        sx = sy = 0;
                        before = -1;
                        do end = (int64_t)off[++v + 1];
                        while (e + j >= end);
                    }
                    sx += at(seed_x, u[j]);
                    sy += at(seed_y, u[j]);
                    if constexpr (ROWS) {
                        const int32_t id = iperm ? iperm[u[j]] : u[j];
                        out_of_order |= id <= before;
                        before = id;
                        if (e + j + 1 == end) last[v] = u[j];
                    }
                }
            }
            acc += at(seed_x, v) * sy - at(seed_y, v) * sx;
        }
    }
    if (ROWS && out_of_order) *bad = 1;   // every writer writes the same word
    acc = wave_sum_u64(acc);
    if (lane_id() == 0) ssum[threadIdx.x / kWave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        U t = 0;
        for (int w = 0; w < kSymThreads / kWave; ++w) t += ssum[w];
        atomicAdd(sum, t);
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

template <typename E, bool ROWS>
static void check_launch(galp_graph *g, const int32_t *nbr, unsigned long long *res, int32_t *last) {
    static std::atomic<unsigned long long> calls{0};
    const unsigned long long now = (unsigned long long)std::chrono::steady_clock::now().time_since_epoch().count();
    const unsigned long long sx = splitmix64(now ^ splitmix64((unsigned long long)(uintptr_t)g + ++calls));
    const unsigned long long sy = splitmix64(sx + 0x9e3779b97f4a7c15ull);
    const int grid = (int)std::min<int64_t>((g->m + kSymTile - 1) / kSymTile,
                                            (int64_t)g->ctx->prop.multiProcessorCount * 8);
    k_check_symmetric<E, ROWS><<<grid, kSymThreads, 0, g->stream>>>(
        (const E *)g->d_off, nbr, g->n, g->m, sx, sy, res, g->d_iperm, last, (int32_t *)(res + 1));
}

// Whether the graph is symmetric, its neighbour ids being in nbr (device memory
// or mapped host memory), if rows hold no vertex twice.  last (may be null):
// receives each row's last neighbour (rows without any are left), and *ascend
// whether every row's ids strictly ascend.
int dev_check_symmetric(galp_graph *g, const int32_t *nbr, bool *symmetric, int32_t *last, bool *ascend) {
    *symmetric = true;
    if (last) *ascend = true;
    if (!g->m) return GALP_OK;
    unsigned long long *res = g->d_counter;   // free until the first init: the sum, then the flag
    int rc = dev_fill_u32(g, (uint32_t *)res, 4, 0u);
    if (rc != GALP_OK) return rc;
    if (last && g->off64) check_launch<int64_t, true>(g, nbr, res, last);
    else if (last) check_launch<int32_t, true>(g, nbr, res, last);
    else if (g->off64) check_launch<int64_t, false>(g, nbr, res, nullptr);
    else check_launch<int32_t, false>(g, nbr, res, nullptr);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(g->h_pinned, res, 16, hipMemcpyDeviceToHost, g->stream) != hipSuccess ||
        hipStreamSynchronize(g->stream) != hipSuccess)
        return fail(g->ctx, GALP_EHIP, "symmetry check failed");
    *symmetric = g->h_pinned[0] == 0 && g->h_pinned[1] == 0;
    if (last) *ascend = g->h_pinned[2] == 0;
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
