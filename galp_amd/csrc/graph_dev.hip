// graph_dev.hip -- device-side graph preparation and label bookkeeping.
//
// Replaces InCoreLP::transfer_data (label_propagation/src/common/
// incore.cuh:59-73), initialize_labels (src/dpp/kernel.cuh:15-22) and the
// final label copy of LFHTBase::run (src/lfht/lfht.cuh:103).  The renumbering
// kernel is new: rows are rewritten in degree-descending order so every
// degree class is one contiguous id range and the most-gathered labels (the
// hubs') share cache lines.  Each row keeps its neighbour order, which keeps
// the tie rule's last positions, so labels mapped back through the inverse
// permutation equal the labels of the original numbering.

#include <algorithm>

#include "device_common.hpp"
#include "internal.hpp"

namespace galp {

// labels[i] = i in both buffers; the first block clears the control words, with
// them the iteration count and the error word.
__global__ void k_init_labels(int32_t *a, int32_t *b, int64_t n, unsigned long long *counter, int32_t *stop,
                              int64_t *front) {
    if (blockIdx.x == 0) {
        if (threadIdx.x < kCountShards)
            for (int k = 0; k < 3; ++k) counter[threadIdx.x * kCountStride + k] = 0ull;
        if (front && threadIdx.x < kFrontCtl) front[threadIdx.x] = 0;
        if (threadIdx.x < kCtlWords) stop[threadIdx.x] = 0;
    }
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        a[i] = (int32_t)i;
        b[i] = (int32_t)i;
    }
}

__global__ void k_fill_u32(uint32_t *p, int64_t n, uint32_t val) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = val;
}

// Clears the stop flag and what an unfinished iteration may have left; one
// thread per shard of the change counter.
__global__ void __launch_bounds__(kCountShards)
k_clear_stop(unsigned long long *counter, int32_t *stop, int64_t *front) {
    for (int k = 0; k < 3; ++k) counter[threadIdx.x * kCountStride + k] = 0ull;
    if (front && threadIdx.x < kFrontCtl) front[threadIdx.x] = 0;
    if (threadIdx.x == 0) *stop = 0;
}

// One wave per internal row k: copy row iperm[k] of the original CSR,
// mapping every neighbour through perm, in the original order.
template <typename E>
__global__ void k_permute_rows(const int64_t *__restrict__ off_old, const int32_t *__restrict__ nbr_old,
                               const int32_t *__restrict__ iperm, const int32_t *__restrict__ perm,
                               const E *__restrict__ off_new, int32_t *__restrict__ nbr_new, int64_t n,
                               int32_t *__restrict__ bad) {
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) / kWave;
    const int lane = lane_id();
    for (int64_t k = wave; k < n; k += nwaves) {
        const int64_t v = iperm[k];
        const int64_t b = off_old[v], d = off_old[v + 1] - b;
        const int64_t nb = (int64_t)off_new[k];
        bool out_of_order = false;
        for (int64_t j = lane; j < d; j += kWave) {
            const int32_t u = nbr_old[b + j];
            out_of_order |= j > 0 && nbr_old[b + j - 1] >= u;
            nbr_new[nb + j] = perm[u];
        }
        if (out_of_order) *bad = 1;   // every writer writes the same word
    }
}

// The same check on rows kept in their input numbering, one wave per row.
template <typename E>
__global__ void __launch_bounds__(256)
k_check_rows(const E *__restrict__ off, const int32_t *__restrict__ nbr, int64_t n, int32_t *__restrict__ bad) {
    const int64_t wave = ((int64_t)blockIdx.x * 256 + threadIdx.x) / kWave;
    const int64_t nwaves = (int64_t)gridDim.x * (256 / kWave);
    for (int64_t v = wave; v < n; v += nwaves) {
        const int64_t b = (int64_t)off[v], d = (int64_t)off[v + 1] - b;
        bool out_of_order = false;
        for (int64_t j = lane_id() + 1; j < d; j += kWave) out_of_order |= nbr[b + j - 1] >= nbr[b + j];
        if (out_of_order) *bad = 1;
    }
}

// The first iteration from labels[i] = i when no row holds a neighbour twice:
// every label of a row counts once, so argmax (count, last position) is the
// label at the row's last position, which is its last neighbour's id -- one
// load per vertex in place of the class kernels' pass over all edges.
// `last` (out of core) holds the last neighbours; else they are read from
// the rows.  dist (may be null) receives the distinct-label counts of the
// rows above degree 64, which are their degrees.  Bound by the one line per
// row it touches: RMAT-22 (4.2 M rows) 29 us against 2.05 ms for the
// class kernels.
constexpr int kFirstUnroll = 4;   // rows in flight per thread
template <typename E>
__global__ void __launch_bounds__(256)
k_first_iteration(const E *__restrict__ off, const int32_t *__restrict__ nbr, const int32_t *__restrict__ last,
                  int32_t *__restrict__ next, int32_t *__restrict__ dist, int64_t n,
                  unsigned long long *__restrict__ counter, IterEnd end) {
    __shared__ uint32_t scratch[256 / kWave];
    if (*end.stop) return;
    const int64_t nthreads = (int64_t)gridDim.x * 256;
    uint32_t changed = 0;
    for (int64_t v0 = (int64_t)blockIdx.x * 256 + threadIdx.x; v0 < n; v0 += kFirstUnroll * nthreads) {
        int64_t b[kFirstUnroll], e[kFirstUnroll];
        int32_t w[kFirstUnroll];
#pragma unroll
        for (int k = 0; k < kFirstUnroll; ++k) {
            const int64_t v = v0 + k * nthreads;
            const int64_t vc = v < n ? v : 0;
            b[k] = (int64_t)off[vc];
            e[k] = v < n ? (int64_t)off[vc + 1] : b[k];   // empty past the end
        }
#pragma unroll
        for (int k = 0; k < kFirstUnroll; ++k) {
            const int64_t v = v0 + k * nthreads;
            w[k] = e[k] > b[k] ? (last ? last[v] : nbr[e[k] - 1]) : -1;
        }
#pragma unroll
        for (int k = 0; k < kFirstUnroll; ++k) {
            const int64_t v = v0 + k * nthreads;
            if (e[k] > b[k]) {
                next[v] = w[k];
                changed += (int64_t)w[k] != v;
                if (dist && e[k] - b[k] > bucket_hi(B_G64)) dist[v] = (int32_t)(e[k] - b[k]);
            }
        }
    }
    block_count_end<4>(changed, counter, scratch, end);
}

// out[v] = iperm[labels[perm[v]]]: internal labels back to original ids.
__global__ void k_map_labels(const int32_t *__restrict__ lab, const int32_t *__restrict__ perm,
                             const int32_t *__restrict__ iperm, int32_t *__restrict__ out, int64_t n) {
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
         v += (int64_t)gridDim.x * blockDim.x)
        out[v] = iperm[lab[perm[v]]];
}

// The same for the buffer a run of *done iterations from lab0 ended in, so the
// read-out is queued without waiting for the count.
__global__ void k_map_labels_done(const int32_t *__restrict__ lab0, const int32_t *__restrict__ lab1,
                                  const int32_t *__restrict__ done, const int32_t *__restrict__ perm,
                                  const int32_t *__restrict__ iperm, int32_t *__restrict__ out, int64_t n) {
    const int32_t *lab = (*done & 1) ? lab1 : lab0;
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
         v += (int64_t)gridDim.x * blockDim.x)
        out[v] = iperm[lab[perm[v]]];
}

// lab[perm[v]] = perm[in[v]]: original labels into the internal numbering.
__global__ void k_unmap_labels(const int32_t *__restrict__ in, const int32_t *__restrict__ perm,
                               int32_t *__restrict__ lab, int64_t n) {
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
         v += (int64_t)gridDim.x * blockDim.x)
        lab[perm[v]] = perm[in[v]];
}

static int grid1d(int64_t n, int threads) {
    int64_t b = (n + threads - 1) / threads;
    if (b > 65536) b = 65536;
    return (int)(b < 1 ? 1 : b);
}

int dev_init_labels(galp_graph *g) {
    k_init_labels<<<grid1d(g->n, 256), 256, 0, g->stream>>>(g->d_lab[0], g->d_lab[1], g->n, g->d_counter, g->d_stop,
                                                            front_ctl(g));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(g->ctx, GALP_EHIP, std::string("init kernels: ") + hipGetErrorString(e));
    return GALP_OK;
}

int dev_clear_stop(galp_graph *g) {
    k_clear_stop<<<1, kCountShards, 0, g->stream>>>(g->d_counter, g->d_stop, front_ctl(g));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(g->ctx, GALP_EHIP, std::string("reset kernel: ") + hipGetErrorString(e));
    return GALP_OK;
}

int dev_fill_u32(galp_graph *g, uint32_t *p, int64_t n, uint32_t val) {
    if (n) k_fill_u32<<<grid1d(n, 256), 256, 0, g->stream>>>(p, n, val);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(g->ctx, GALP_EHIP, std::string("fill kernel: ") + hipGetErrorString(e));
    return GALP_OK;
}

int dev_permute_rows(galp_graph *g, const int64_t *d_off_old, const int32_t *d_nbr_old,
                     int32_t *d_nbr_new, int32_t *bad) {
    if (!g->n) return GALP_OK;
    const int64_t blocks = std::min<int64_t>((g->n + 3) / 4, 65536);
    if (g->off64)
        k_permute_rows<int64_t><<<(int)blocks, 256, 0, g->stream>>>(
            d_off_old, d_nbr_old, g->d_iperm, g->d_perm, (const int64_t *)g->d_off, d_nbr_new, g->n, bad);
    else
        k_permute_rows<int32_t><<<(int)blocks, 256, 0, g->stream>>>(
            d_off_old, d_nbr_old, g->d_iperm, g->d_perm, (const int32_t *)g->d_off, d_nbr_new, g->n, bad);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(g->ctx, GALP_EHIP, std::string("permute kernel: ") + hipGetErrorString(e));
    return GALP_OK;
}

int dev_check_rows(galp_graph *g, int32_t *bad) {
    if (!g->n) return GALP_OK;
    const int blocks = (int)std::min<int64_t>((g->n + 3) / 4, 65536);
    if (g->off64) k_check_rows<int64_t><<<blocks, 256, 0, g->stream>>>((const int64_t *)g->d_off, g->d_nbr, g->n, bad);
    else k_check_rows<int32_t><<<blocks, 256, 0, g->stream>>>((const int32_t *)g->d_off, g->d_nbr, g->n, bad);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(g->ctx, GALP_EHIP, std::string("row check kernel: ") + hipGetErrorString(e));
    return GALP_OK;
}

int launch_first_iteration(galp_graph *g) {
    if (!g->n) return GALP_OK;
    const int32_t *last = g->ooc ? g->ooc->d_last : nullptr;
    int32_t *next = g->d_lab[g->cur ^ 1], *dist = distinct_out(g);
    const int64_t per_block = 256 * kFirstUnroll;
    const int grid = (int)std::min<int64_t>((g->n + per_block - 1) / per_block,
                                            (int64_t)g->ctx->prop.multiProcessorCount * 8);
    PendingLaunch pl;
    g->ended = may_end(g);
    const IterEnd end = iter_end_args(g, g->ended);
    prof_begin(g, "first", (double)g->n * (8.0 + 2.0 * (g->off64 ? 8 : 4)), &pl);   // offsets, last id, next label
    if (g->off64)
        k_first_iteration<int64_t><<<grid, 256, 0, g->stream>>>((const int64_t *)g->d_off, g->d_nbr, last, next, dist,
                                                                g->n, g->d_counter, end);
    else
        k_first_iteration<int32_t><<<grid, 256, 0, g->stream>>>((const int32_t *)g->d_off, g->d_nbr, last, next, dist,
                                                                g->n, g->d_counter, end);
    prof_end(g, &pl);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(g->ctx, GALP_EHIP, std::string("first iteration: ") + hipGetErrorString(e));
    return GALP_OK;
}

int dev_map_labels(galp_graph *g, const int32_t *lab, int32_t *out) {
    if (g->n) k_map_labels<<<grid1d(g->n, 256), 256, 0, g->stream>>>(lab, g->d_perm, g->d_iperm, out, g->n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(g->ctx, GALP_EHIP, std::string("map kernel: ") + hipGetErrorString(e));
    return GALP_OK;
}

int dev_map_labels_done(galp_graph *g, int cur0, int32_t *out) {
    if (g->n)
        k_map_labels_done<<<grid1d(g->n, 256), 256, 0, g->stream>>>(g->d_lab[cur0], g->d_lab[cur0 ^ 1], g->d_iters_done,
                                                                   g->d_perm, g->d_iperm, out, g->n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(g->ctx, GALP_EHIP, std::string("map kernel: ") + hipGetErrorString(e));
    return GALP_OK;
}

int dev_unmap_labels(galp_graph *g, const int32_t *in, int32_t *lab) {
    if (g->n) k_unmap_labels<<<grid1d(g->n, 256), 256, 0, g->stream>>>(in, g->d_perm, lab, g->n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(g->ctx, GALP_EHIP, std::string("unmap kernel: ") + hipGetErrorString(e));
    return GALP_OK;
}

}  // namespace galp
