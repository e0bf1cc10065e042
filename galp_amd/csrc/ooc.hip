// ooc.hip -- out-of-core policies: the neighbour array stays in pinned host
// memory and streams to the GPU in vertex-aligned batches every iteration.
//
// Replaces the reference's out-of-core propagators:
//   OutOfCore::compute_batch_boundaries  label_propagation/src/common/outofcore.cuh:38-60
//   OutOfCore::transfer_batch / transfer_next_batch   outofcore.cuh:63-97
//   SyncLP::iterate                     src/common/sync.cuh:43-59   (policy 1)
//   AsyncLP::iterate, swap_buffers      src/common/async.cuh:66-107 (policy 2)
// Design: offsets and both label arrays live in HBM; only the neighbour ids
// move.  A batch is [bv0, bv1) with fewer than 2^b edges (one vertex of
// degree >= 2^b gets a batch of its own: the reference's cut loop would not
// advance there).  For each batch the GPU copies the slice into one of two
// device buffers, rebases the batch's offsets into a per-buffer offset array
// (off[v] - off[bv0]), and runs the method's kernels on the batch's share of
// each degree class and of the hub lists.  Every batch reads labels(t-1)
// and writes labels(t), so the labels equal the in-core ones for any 2^b.
//   policy 1: copy and kernels in order on the graph's stream;
//   policy 2: copies on a second stream, double-buffered: the copy of batch
//             b+1 overlaps the kernels of batch b; events order each buffer's
//             reuse after the kernels that read it.
// What bounds a streamed iteration is the link: all edges once, 50-57 GB/s.
// Once few rows can still change (frontier.hip) the iteration reads those rows
// over the link from where they lie, and nothing else.  RMAT-20 (31 M edges,
// 10 iterations, batches of 2^22 edges): 27.3 ms streaming every iteration,
// 12.1 with the lists, of which three streamed iterations take 7.5.
// A run copies its own batches: a buffer's batch is used again only within the
// run that copied it (with at most two batches, from its second iteration on).

#include <algorithm>
#include <cstring>
#include <vector>

#include "device_common.hpp"
#include "internal.hpp"
#include "parallel.hpp"

namespace galp {

template <typename E>
__global__ void __launch_bounds__(256)
k_rebase(const E *__restrict__ off, E *__restrict__ offb, int64_t v0, int64_t v1) {
    const E base = off[v0];
    for (int64_t v = v0 + (int64_t)blockIdx.x * 256 + threadIdx.x; v <= v1; v += (int64_t)gridDim.x * 256)
        offb[v] = off[v] - base;
}

// The cut rule of outofcore.cuh:38-60 with the degree >= B case cut off
// into a batch of its own (restated by the oracle's oracle_batch_boundaries).
static std::vector<int64_t> batch_boundaries(const std::vector<int64_t> &off, int64_t B) {
    const int64_t n = (int64_t)off.size() - 1, m = off[(size_t)n];
    std::vector<int64_t> bbs{0};
    int64_t batch_offset = B, last = 0;
    while (batch_offset < m) {
        const int64_t left = std::lower_bound(off.begin(), off.end(), batch_offset) - off.begin();
        int64_t cut = left - 1;
        if (cut <= last) cut = last + 1;
        if (cut >= n) break;
        bbs.push_back(cut);
        last = cut;
        batch_offset = off[(size_t)cut] + B;
    }
    bbs.push_back(n);
    return bbs;
}

void ooc_free(galp_graph *g) {
    OocState *O = g->ooc;
    if (!O) return;
    if (O->copy_stream) (void)hipStreamSynchronize(O->copy_stream);   // copies of a call that failed
    for (int k = 0; k < 2; ++k) {
        if (O->d_buf[k]) (void)hipFree(O->d_buf[k]);
        if (O->d_offb[k]) (void)hipFree(O->d_offb[k]);
        if (O->ev_copied[k]) (void)hipEventDestroy(O->ev_copied[k]);
        if (O->ev_free[k]) (void)hipEventDestroy(O->ev_free[k]);
    }
    if (O->copy_stream) (void)hipStreamDestroy(O->copy_stream);
    if (O->d_last) (void)hipFree(O->d_last);
    if (O->h_ctl) (void)hipHostFree(O->h_ctl);
    if (O->h_nbr) (void)hipHostFree(O->h_nbr);
    delete O;
    g->ooc = nullptr;
}

int ooc_setup(galp_graph *g, const galp_csr_view *c, const std::vector<int64_t> &offi,
              const std::vector<int32_t> &perm, const std::vector<int32_t> &iperm,
              const std::vector<int32_t> &vlist, const std::vector<int32_t> &hub_vertices,
              const std::vector<int32_t> &hub_tile0, const std::vector<int64_t> &hub_item0, bool *symmetric) {
    OocState *O = new (std::nothrow) OocState();
    if (!O) return fail(g->ctx, GALP_ENOMEM, "host allocation failed");
    g->ooc = O;
    const int64_t n = g->n, m = g->m;
    // the neighbour array, in the internal numbering, in pinned host memory
    if (hipHostMalloc((void **)&O->h_nbr, 4 * (size_t)std::max<int64_t>(m, 1), hipHostMallocDefault) != hipSuccess) {
        O->h_nbr = nullptr;
        return fail(g->ctx, GALP_ENOMEM, "pinned host buffer for the neighbour array");
    }
    const int32_t *src = c->neighbors;
    if (g->reorder) {
        const bool o64 = c->offsets_are_64 != 0;
        parallel_for(0, n, [&](int64_t k) {
            const int64_t v = iperm[(size_t)k];
            const int64_t b = o64 ? ((const int64_t *)c->offsets)[v] : ((const int32_t *)c->offsets)[v];
            const int64_t d = offi[(size_t)k + 1] - offi[(size_t)k];
            int32_t *dst = O->h_nbr + offi[(size_t)k];
            for (int64_t j = 0; j < d; ++j) dst[j] = perm[(size_t)src[b + j]];
        });
    } else {
        const int64_t chunk = 1 << 22;
        parallel_for(0, (m + chunk - 1) / chunk, [&](int64_t k) {
            const int64_t lo = k * chunk, hi = std::min(m, lo + chunk);
            std::memcpy(O->h_nbr + lo, src + lo, 4 * (size_t)(hi - lo));
        });
    }
    // batches and their share of every class and of the hub lists
    const int64_t B = (int64_t)1 << g->opts.buffer_pow;
    O->bbs = batch_boundaries(offi, B);
    const int64_t nb = (int64_t)O->bbs.size() - 1;
    int64_t maxe = 0;
    O->views.resize((size_t)std::max<int64_t>(nb, 0));
    O->e0.resize((size_t)std::max<int64_t>(nb, 0));
    O->e1.resize((size_t)std::max<int64_t>(nb, 0));
    auto cut_list = [&](int64_t lo, int64_t hi, int64_t s0, int64_t cnt, int64_t &k0, int64_t &k1) {
        if (g->reorder) {   // class = ids [s0, s0 + cnt)
            k0 = std::min(std::max(lo, s0), s0 + cnt);
            k1 = std::min(std::max(hi, s0), s0 + cnt);
        } else {            // class = vlist[s0, s0 + cnt), sorted by id
            auto b = vlist.begin() + s0, e = vlist.begin() + s0 + cnt;
            k0 = s0 + (std::lower_bound(b, e, (int32_t)lo) - b);
            k1 = s0 + (std::lower_bound(b, e, (int32_t)std::min<int64_t>(hi, INT32_MAX)) - b);
        }
    };
    for (int64_t b = 0; b < nb; ++b) {
        const int64_t lo = O->bbs[(size_t)b], hi = O->bbs[(size_t)b + 1];
        O->e0[(size_t)b] = offi[(size_t)lo];
        O->e1[(size_t)b] = offi[(size_t)hi];
        maxe = std::max(maxe, O->e1[(size_t)b] - O->e0[(size_t)b]);
        IterView &w = O->views[(size_t)b];
        for (int cl = 0; cl < NUM_BUCKETS; ++cl) {
            const BucketRange &r = g->bucket[cl];
            int64_t k0, k1;
            cut_list(lo, hi, r.v0, r.nv, k0, k1);
            w.cls[cl].v0 = k0;
            w.cls[cl].nv = k1 - k0;
            w.cls[cl].edges = 0;   // read by per-kernel profiling only
            if (g->opts.profile && g->reorder) w.cls[cl].edges = offi[(size_t)k1] - offi[(size_t)k0];
            else if (g->opts.profile)
                for (int64_t k = k0; k < k1; ++k)
                    w.cls[cl].edges += offi[(size_t)vlist[(size_t)k] + 1] - offi[(size_t)vlist[(size_t)k]];
        }
        // hubs: ascending ids in both numberings
        w.h0 = std::lower_bound(hub_vertices.begin(), hub_vertices.end(), (int32_t)lo) - hub_vertices.begin();
        w.h1 = std::lower_bound(hub_vertices.begin(), hub_vertices.end(), (int32_t)std::min<int64_t>(hi, INT32_MAX)) -
               hub_vertices.begin();
        const int64_t nh = (int64_t)hub_vertices.size();
        w.t0 = w.h0 < nh ? hub_tile0[(size_t)w.h0] : g->nhub_tiles;
        w.t1 = w.h1 < nh ? hub_tile0[(size_t)w.h1] : g->nhub_tiles;
        w.i0 = hub_item0[(size_t)w.h0];
        w.i1 = hub_item0[(size_t)w.h1];
    }
    if (hipHostMalloc((void **)&O->h_ctl, 8 * (kFrontCtl + 1), hipHostMallocDefault) != hipSuccess) {
        O->h_ctl = nullptr;
        return fail(g->ctx, GALP_ENOMEM, "out-of-core control words");
    }
    O->bufcap = std::max<int64_t>(maxe, 1);
    const size_t esz = g->off64 ? 8 : 4;
    for (int k = 0; k < 2; ++k) {
        if (hipMalloc((void **)&O->d_buf[k], 4 * (size_t)O->bufcap) != hipSuccess ||
            hipMalloc(&O->d_offb[k], esz * (size_t)(n + 1)) != hipSuccess)
            return fail(g->ctx, GALP_ENOMEM, "out-of-core batch buffers");
        g->device_bytes += (int64_t)(4 * (size_t)O->bufcap + esz * (size_t)(n + 1));
        if (hipEventCreateWithFlags(&O->ev_copied[k], hipEventDisableTiming) != hipSuccess ||
            hipEventCreateWithFlags(&O->ev_free[k], hipEventDisableTiming) != hipSuccess)
            return fail(g->ctx, GALP_EHIP, "out-of-core events");
    }
    if (g->opts.policy == GALP_POLICY_OOC_ASYNC &&
        hipStreamCreateWithFlags(&O->copy_stream, hipStreamNonBlocking) != hipSuccess)
        return fail(g->ctx, GALP_EHIP, "out-of-core copy stream");
    // Each row's last neighbour, with which the first iteration needs no batch
    // where every row's ids ascend; that, and whether the graph is symmetric, is
    // found in the same pass over the link (RMAT-20: 2.3 ms of an upload of 88;
    // in the host's loop above the check and the records cost 10).  Kept only
    // where the memory budget has room: without it the first iteration streams
    // like the others.
    const std::string err = g->ctx->err;
    const int64_t bytes = g->device_bytes;
    if (dev_alloc(g, &O->d_last, n) != GALP_OK) {
        g->ctx->err = err;   // doing without is no failure
        return GALP_OK;
    }
    const int rc = dev_check_symmetric(g, O->h_nbr, symmetric, O->d_last, &g->rows_ascend);
    if (rc != GALP_OK) return rc;
    if (!g->rows_ascend) {
        (void)hipFree(O->d_last);
        O->d_last = nullptr;
        g->device_bytes = bytes;
    }
    return GALP_OK;
}

int ooc_finish_copies(galp_graph *g) {
    OocState *O = g->ooc;
    if (!O || !O->copy_stream) return GALP_OK;
    for (int k = 0; k < 2; ++k)
        if (hipStreamWaitEvent(g->stream, O->ev_copied[k], 0) != hipSuccess)
            return fail(g->ctx, GALP_EHIP, "out-of-core copy event");
    return GALP_OK;
}

void ooc_forget_batches(galp_graph *g) {
    if (g->ooc) g->ooc->resident[0] = g->ooc->resident[1] = -1;
}

// Policy 2: queues the copy of batch b into its buffer on the copy stream,
// after the kernels that read the buffer, unless the buffer holds it.
static int ooc_copy_async(galp_graph *g, int64_t b) {
    OocState *O = g->ooc;
    const int k = (int)(b & 1);
    if (O->resident[k] == b) return GALP_OK;
    if (O->used[k] && hipStreamWaitEvent(O->copy_stream, O->ev_free[k], 0) != hipSuccess)
        return fail(g->ctx, GALP_EHIP, "out-of-core wait");
    const int64_t e0 = O->e0[(size_t)b], ne = O->e1[(size_t)b] - e0;
    O->resident[k] = -1;
    PendingLaunch pl;
    prof_begin(g, "h2d", 4.0 * (double)ne, &pl, O->copy_stream);
    if (ne && hipMemcpyAsync(O->d_buf[k], O->h_nbr + e0, 4 * (size_t)ne, hipMemcpyHostToDevice, O->copy_stream) !=
                  hipSuccess)
        return fail(g->ctx, GALP_EHIP, "out-of-core batch copy");
    prof_end(g, &pl, O->copy_stream);
    if (hipEventRecord(O->ev_copied[k], O->copy_stream) != hipSuccess)
        return fail(g->ctx, GALP_EHIP, "out-of-core copy event");
    O->resident[k] = b;
    return GALP_OK;
}

template <typename E>
static int ooc_round(galp_graph *g) {
    OocState *O = g->ooc;
    const int64_t nb = (int64_t)O->views.size();
    const bool async = g->opts.policy == GALP_POLICY_OOC_ASYNC;
    for (int64_t b = 0; b < nb; ++b) {
        const int k = async ? (int)(b & 1) : 0;
        const int64_t e0 = O->e0[(size_t)b], ne = O->e1[(size_t)b] - e0;
        const int64_t lo = O->bbs[(size_t)b], hi = O->bbs[(size_t)b + 1];
        if (async) {
            const int rc = ooc_copy_async(g, b);
            if (rc != GALP_OK) return rc;
            if (hipStreamWaitEvent(g->stream, O->ev_copied[k], 0) != hipSuccess)
                return fail(g->ctx, GALP_EHIP, "out-of-core copy event");
        } else {
            PendingLaunch pl;
            prof_begin(g, "h2d", 4.0 * (double)ne, &pl);
            if (ne && hipMemcpyAsync(O->d_buf[k], O->h_nbr + e0, 4 * (size_t)ne, hipMemcpyHostToDevice, g->stream) !=
                          hipSuccess)
                return fail(g->ctx, GALP_EHIP, "out-of-core batch copy");
            prof_end(g, &pl);
        }
        const int64_t nv = hi - lo + 1;
        const int grid = (int)std::max<int64_t>(1, std::min<int64_t>((nv + 255) / 256, 1024));
        k_rebase<E><<<grid, 256, 0, g->stream>>>((const E *)g->d_off, (E *)O->d_offb[k], lo, hi);
        IterView w = O->views[(size_t)b];
        w.off = O->d_offb[k];
        w.nbr = O->d_buf[k];
        if (g->opts.method == GALP_METHOD_HASH && g->opts.dispatch == GALP_DISPATCH_LEARNED) {
            const int rcf = launch_learned_front_batch(g, w, lo, hi);   // this batch's lists and candidates
            if (rcf != GALP_OK) return rcf;
        }
        const int rc = g->opts.method == GALP_METHOD_HASH ? launch_hash_iteration(g, w)
                                                            : launch_sort_iteration(g, w);
        if (rc != GALP_OK) return rc;
        if (async) {
            if (hipEventRecord(O->ev_free[k], g->stream) != hipSuccess)
                return fail(g->ctx, GALP_EHIP, "out-of-core event");
            O->used[k] = true;
        }
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(g->ctx, GALP_EHIP, std::string("out-of-core launch: ") + hipGetErrorString(e));
    return GALP_OK;
}

// Learned dispatch set-up: every batch is copied (synchronously, before any
// iteration) and its big vertices' features computed from its rows.
int ooc_features(galp_graph *g) {
    OocState *O = g->ooc;
    const int64_t nb = (int64_t)O->views.size();
    // buffer 0 is written on the graph's stream here: a batch loaded ahead into it comes first
    if (const int rc = ooc_finish_copies(g); rc != GALP_OK) return rc;
    O->resident[0] = -1;
    for (int64_t b = 0; b < nb; ++b) {
        const int64_t e0 = O->e0[(size_t)b], ne = O->e1[(size_t)b] - e0;
        const int64_t lo = O->bbs[(size_t)b], hi = O->bbs[(size_t)b + 1];
        if (ne && hipMemcpyAsync(O->d_buf[0], O->h_nbr + e0, 4 * (size_t)ne, hipMemcpyHostToDevice, g->stream) !=
                      hipSuccess)
            return fail(g->ctx, GALP_EHIP, "out-of-core batch copy");
        const int grid = (int)std::max<int64_t>(1, std::min<int64_t>((hi - lo + 256) / 256, 1024));
        if (g->off64)
            k_rebase<int64_t><<<grid, 256, 0, g->stream>>>((const int64_t *)g->d_off, (int64_t *)O->d_offb[0], lo, hi);
        else
            k_rebase<int32_t><<<grid, 256, 0, g->stream>>>((const int32_t *)g->d_off, (int32_t *)O->d_offb[0], lo, hi);
        const int rc = learn_features_view(g, O->d_offb[0], O->d_buf[0], lo, hi);
        if (rc != GALP_OK) return rc;
        // the next copy reuses the buffer
        if (hipStreamSynchronize(g->stream) != hipSuccess) return fail(g->ctx, GALP_EHIP, "feature pass failed");
    }
    return GALP_OK;
}

// An iteration over the rows that can still change (frontier.hip) reads them
// from the pinned array where they lie, instead of streaming every batch.
// Which it is, the host has to know before it queues the copies: one wait per
// iteration, after the list kernels.
int launch_ooc_iteration(galp_graph *g) {
    OocState *O = g->ooc;
    if (!O) return fail(g->ctx, GALP_ESTATE, "internal: out-of-core state missing");
    O->on_lists = false;
    if (front_now(g)) {
        const int rc = launch_front(g);
        if (rc != GALP_OK) return rc;
        // the first two batches load while the lists are built and read back;
        // if the lists are walked they stay for the run's next streamed iteration
        if (g->opts.policy == GALP_POLICY_OOC_ASYNC)
            for (int64_t b = 0; b < 2 && b < (int64_t)O->views.size(); ++b) {
                const int rcc = ooc_copy_async(g, b);
                if (rcc != GALP_OK) return rcc;
            }
        int64_t *ctl = O->h_ctl;
        if (hipMemcpyAsync(ctl, g->front->d_ctl, 8 * kFrontCtl, hipMemcpyDeviceToHost, g->stream) != hipSuccess ||
            hipMemcpyAsync(ctl + kFrontCtl, g->d_stop, 4, hipMemcpyDeviceToHost, g->stream) != hipSuccess ||
            hipStreamSynchronize(g->stream) != hipSuccess)
            return fail(g->ctx, GALP_EHIP, "out-of-core list readback");
        if ((int32_t)ctl[kFrontCtl] != 0) return GALP_OK;   // the run has stopped
        int64_t edges = 0;
        for (int b = 0; b < NUM_BUCKETS; ++b) edges += ctl[kFrontEdges + b];
        if (ctl[kFrontReady] && edges <= front_list(g, 0).max_edges) {   // as front_lists_on
            O->on_lists = true;
            if (learned_now(g))
                if (const int rcl = learn_route_nothing(g); rcl != GALP_OK) return rcl;
            IterView w = full_view(g);
            w.nbr = O->h_nbr;   // mapped
            return g->opts.method == GALP_METHOD_HASH ? launch_hash_iteration(g, w) : launch_sort_iteration(g, w);
        }
    }
    return g->off64 ? ooc_round<int64_t>(g) : ooc_round<int32_t>(g);
}

}  // namespace galp
