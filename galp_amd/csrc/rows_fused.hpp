// rows_fused.hpp -- one launch for all row classes of a small or mid-sized
// graph, shared by both methods.
//
// A class kernel of a graph of a few million edges runs for 5 to 20 us, most
// of it the launch, the first dependent loads and the last blocks, and an
// iteration makes ten such launches one after another.  The fused kernel
// gives every class a contiguous range of blocks, in proportion to its work
// and the largest rows first, and each block runs its class's code.  Its
// register and LDS need is the largest class's (four 256-thread blocks per
// CU), which costs the lane groups of a large graph more than the launches
// do, so large graphs keep one kernel per class (kFusedMaxEdges).
#pragma once

#include <algorithm>

#include "device_common.hpp"
#include "internal.hpp"

namespace galp {

constexpr int kRowsThreads = 256;
constexpr int kRowsWaves = kRowsThreads / kWave;
constexpr int kRowsPerCu = 4;   // 32 KB of tables and a little more each

// One class's rows: a vertex list or (null) the ids v0, v0 + 1, ..., nv of
// them or *nv_dev; then list B (learned dispatch's high-distinct rows; may be
// null).  front_list / front_len: the rows that can still change.  cost: work
// of an average row.
struct RowsClass {
    const int32_t *vlist;
    int64_t v0, nv;
    const int64_t *nv_dev;
    const int32_t *vlistB;
    const int64_t *nvB_dev;
    const int32_t *front_list;
    const int64_t *front_len;
    float cost;
    int32_t per_block;   // rows a block takes at a time
};

template <int NC>
struct RowsArgs {
    RowsClass c[NC];     // class b, lane groups first
    FrontList front;     // ctl and max_edges
};

// This block's class (-1: none), its rows (or, once front_lists_on, those
// that can still change) and its place among the class's blocks.
struct RowsWork {
    int cls;
    RowsClass r;
    int64_t bi, nb;
};

// Shares the grid out by the work of the rows there are now, which lists
// built on the device change from iteration to iteration, so every block
// computes the same partition: at least one block for a class with rows, no
// more than one round of its rows, the largest class first.
template <int NC>
__device__ __forceinline__ RowsWork rows_work(const RowsArgs<NC> &a) {
    const bool lists = front_lists_on(a.front);
    int64_t nv[NC];
    float total = 0.f;
#pragma unroll
    for (int b = 0; b < NC; ++b) {
        const RowsClass &c = a.c[b];
        nv[b] = lists ? *c.front_len : c.nv_dev ? *c.nv_dev + (c.nvB_dev ? *c.nvB_dev : 0) : c.nv;
        total += (float)nv[b] * c.cost;
    }
    const float scale = (float)((int)gridDim.x - NC) / fmaxf(total, 1.f);
    RowsWork w;
    w.cls = -1;
    w.bi = 0;
    w.nb = 1;
    int64_t at = 0;
#pragma unroll
    for (int b = NC - 1; b >= 0; --b) {
        const RowsClass &c = a.c[b];
        int64_t nb = 0;
        if (nv[b]) {
            nb = 1 + (int64_t)fmaxf((float)nv[b] * c.cost * scale, 0.f);
            const int64_t most = (nv[b] + c.per_block - 1) / c.per_block;
            nb = nb < most ? nb : most;
        }
        if ((int64_t)blockIdx.x >= at && (int64_t)blockIdx.x < at + nb) {
            w.cls = b;
            w.bi = (int64_t)blockIdx.x - at;
            w.nb = nb;
        }
        at += nb;
    }
    w.cls = __builtin_amdgcn_readfirstlane(w.cls);
    if (w.cls < 0) return w;
    w.r = a.c[w.cls];
    if (lists) {
        w.r.vlist = w.r.front_list;
        w.r.v0 = 0;
        w.r.nv = *w.r.front_len;
        w.r.vlistB = nullptr;
    } else if (w.r.nv_dev) {
        w.r.nv = *w.r.nv_dev;
    }
    return w;
}

// The average row costs of a view's classes and the grid: what is resident,
// at most one round of every class's rows.  An edge costs about the same in
// every class (8 to 11 ps at 8 M edges; rows with tables a quarter more than
// lane groups), a row about one more edge.
template <int NC>
int rows_plan(const galp_graph *g, const IterView &w, RowsArgs<NC> &a, int first_table) {
    int64_t most = 0;
    for (int b = 0; b < NC; ++b) {
        const BucketRange &r = w.cls[b];
        a.c[b].cost = r.nv ? (b >= first_table ? 1.25f : 1.f) * (float)r.edges / (float)r.nv + 1.f : 1.f;
        most += (r.nv + a.c[b].per_block - 1) / a.c[b].per_block;
    }
    if (!most) return 0;
    const int64_t grid = (int64_t)g->ctx->prop.multiProcessorCount * kRowsPerCu;
    return (int)std::min(grid, most + NC);
}

}  // namespace galp
