// group_kernel.hpp -- the degree <= 64 driver shared by both LP methods.
#pragma once

#include <type_traits>

#include "device_common.hpp"
#include "internal.hpp"

namespace galp {

// Degree <= G: one aligned group of G lanes per vertex; lane p holds the
// label of the p-th neighbour (-1 past the degree).  Resolve::best<G>(L)
// returns the group's max of (count << 8 | last), the same in every lane of
// the group, `last` being a lane index (a CSR position in the row), so the
// winner is the label of lane `last`.
// One wave holds 64/G vertices per round; rounds are software-pipelined:
// while round t is resolved, the labels of round t+1 and the neighbour ids
// of round t+2 are loading, the offsets of round t+3 and, from a vertex list,
// the ids of round t+4 (an id loaded with the offsets that need it is the
// youngest load in flight, and waiting for it drains all the others).  This
// block is number bi of the nb that share the class.
template <int G, class Resolve, bool VLIST, typename E>
__device__ __forceinline__ uint32_t group_rounds_lanes(const E *__restrict__ off, const int32_t *__restrict__ nbr,
                                                 const int32_t *__restrict__ prev, int32_t *__restrict__ next,
                                                 const int32_t *__restrict__ vlist, int64_t v0, int64_t nv,
                                                 int64_t bi, int64_t nb) {
    const int p = lane_id() & (G - 1);
    constexpr int64_t per_block = 256 / G;
    const int64_t stride = nb * per_block;
    // Raw offsets stay in the pipeline registers until the next stage uses
    // them (any arithmetic on a just-loaded value would wait for it), and
    // every load is issued by every lane from a clamped address, so no load
    // sits under a branch (see pipelined()).
    struct St {
        int64_t v;
        E ob, oe;     // off[v], off[v+1], raw
        bool ok;      // i < nv
    };
    auto ident = [&](int64_t i) -> int32_t { return VLIST ? vlist[v0 + (i < nv ? i : 0)] : 0; };
    auto state = [&](int64_t i, int32_t id) {   // id: ident(i)
        St s;
        s.ok = i < nv;
        if constexpr (VLIST) s.v = (int64_t)id;
        else s.v = v0 + (s.ok ? i : 0);
        s.ob = off[s.v];
        s.oe = off[s.v + 1];
        return s;
    };
    auto has = [&](const St &s) { return s.ok && (int64_t)p < (int64_t)(s.oe - s.ob); };
    auto ldn = [&](const St &s) -> int32_t {
        return __builtin_nontemporal_load(&nbr[has(s) ? (int64_t)s.ob + p : 0]);
    };
    auto gat = [&](int32_t u, const St &s) -> int32_t { return prev[has(s) ? (uint32_t)u : 0u]; };
    uint32_t changed = 0;
    // the winner lane (best's low byte) holds the new label and writes it
    auto resolve = [&](const St &s, int32_t Lraw, int32_t old) {
        const int32_t L = has(s) ? Lraw : -1;
        const uint32_t best = Resolve::template best<G>(L);
        if (p == (int)(best & 0xffu) && s.ok && s.oe != s.ob) {
            next[s.v] = L;
            changed += (L != old);
        }
    };
    int64_t base = bi * per_block;                    // uniform round index
    int64_t i = base + threadIdx.x / G;               // this lane's vertex index
    // Four state slots rotate through the stages; the loop is unrolled by
    // the rotation period so no register holding an in-flight load is ever
    // copied (a copy would wait for it).
    const int32_t ia = ident(i), ib = ident(i + stride), ic = ident(i + 2 * stride);
    int32_t id = ident(i + 3 * stride);
    St sa = state(i, ia), sb = state(i + stride, ib), sc = state(i + 2 * stride, ic), sd;
    int32_t u = ldn(sa);
    int32_t LA = gat(u, sa), oA = prev[sa.v], LB, oB;
    u = ldn(sb);
#define GALP_GROUP_STAGE(S0, S1, S2, S3, LC, OC, LN, ON) \
    LN = gat(u, S1);                                     \
    ON = prev[S1.v];                                     \
    u = ldn(S2);                                         \
    S3 = state(i + 3 * stride, id);                      \
    id = ident(i + 4 * stride);                          \
    resolve(S0, LC, OC);                                 \
    i += stride;                                         \
    base += stride;                                      \
    if (base >= nv) break;
    while (base < nv) {
        GALP_GROUP_STAGE(sa, sb, sc, sd, LA, oA, LB, oB)
        GALP_GROUP_STAGE(sb, sc, sd, sa, LB, oB, LA, oA)
        GALP_GROUP_STAGE(sc, sd, sa, sb, LA, oA, LB, oB)
        GALP_GROUP_STAGE(sd, sa, sb, sc, LB, oB, LA, oA)
    }
#undef GALP_GROUP_STAGE
    return changed;
}

// Degree 33..64, a wave per row: the same pipeline with the row's offsets, old
// label and list id loaded through the scalar cache into scalar registers,
// since they are the same in all lanes.  A round issues three vector memory
// instructions (ids, gather, label) for six, and holds 25 vector registers for
// 52, which the fused kernel's mix of classes gains from: LFR-1M learned 2127
// -> 2058 us.  (The 512-graph batch, bound by the resolver's issue, is
// unchanged, and two rows a wave, for G = 32, lost as much again to selects.)
template <class Resolve, bool VLIST, typename E>
__device__ __forceinline__ uint32_t wave_rounds(const E *__restrict__ off, const int32_t *__restrict__ nbr,
                                                const int32_t *__restrict__ prev, int32_t *__restrict__ next,
                                                const int32_t *__restrict__ vlist, int64_t v0, int64_t nv,
                                                int64_t bi, int64_t nb) {
    constexpr int NW = 256 / kWave;
    const int lane = lane_id();
    const int64_t stride = nb * NW;
    int64_t i = bi * NW + __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);   // uniform
    struct St {
        int64_t v;
        E ob, oe;      // off[v], off[v + 1]
        int32_t old;   // prev[v]
        int32_t len;   // set by ldn; 0 past the end
    };
    auto ident = [&](int64_t i) -> int32_t { return VLIST ? vlist[v0 + (i < nv ? i : 0)] : 0; };
    auto state = [&](int64_t i, int32_t id) {
        St t;
        t.v = VLIST ? (int64_t)id : v0 + (i < nv ? i : 0);
        t.ob = off[t.v];
        t.oe = off[t.v + 1];
        t.old = prev[t.v];
        t.len = 0;
        return t;
    };
    auto ldn = [&](St &t, int64_t i) -> int32_t {
        t.len = i < nv ? (int32_t)(t.oe - t.ob) : 0;
        using U = typename std::conditional<sizeof(E) == 4, uint32_t, uint64_t>::type;
        return __builtin_nontemporal_load(&nbr[lane < t.len ? (U)t.ob + (U)lane : (U)0]);
    };
    auto gat = [&](int32_t u, const St &t) -> int32_t { return prev[lane < t.len ? (uint32_t)u : 0u]; };
    uint32_t changed = 0;
    // the winner lane (best's low byte) holds the new label and writes it
    auto resolve = [&](const St &t, int32_t Lraw) {
        const int32_t L = lane < t.len ? Lraw : -1;
        const uint32_t best = Resolve::template best<kWave>(L);
        if (lane == (int)(best & 0xffu) && t.len > 0) {
            next[t.v] = L;
            changed += (L != t.old);
        }
    };
    const int32_t ia = ident(i), ib = ident(i + stride), ic = ident(i + 2 * stride);
    int32_t id = ident(i + 3 * stride);
    St sa = state(i, ia), sb = state(i + stride, ib), sc = state(i + 2 * stride, ic), sd;
    int32_t u = ldn(sa, i);
    int32_t LA = gat(u, sa), LB;
    u = ldn(sb, i + stride);
#define GALP_GROUP_STAGE(S0, S1, S2, S3, LC, LN) \
    LN = gat(u, S1);                             \
    u = ldn(S2, i + 2 * stride);                 \
    S3 = state(i + 3 * stride, id);              \
    id = ident(i + 4 * stride);                  \
    resolve(S0, LC);                             \
    i += stride;                                 \
    if (i >= nv) break;
    while (i < nv) {
        GALP_GROUP_STAGE(sa, sb, sc, sd, LA, LB)
        GALP_GROUP_STAGE(sb, sc, sd, sa, LB, LA)
        GALP_GROUP_STAGE(sc, sd, sa, sb, LA, LB)
        GALP_GROUP_STAGE(sd, sa, sb, sc, LB, LA)
    }
#undef GALP_GROUP_STAGE
    return changed;
}

template <int G, class Resolve, bool VLIST, typename E>
__device__ __forceinline__ uint32_t group_rounds(const E *__restrict__ off, const int32_t *__restrict__ nbr,
                                                 const int32_t *__restrict__ prev, int32_t *__restrict__ next,
                                                 const int32_t *__restrict__ vlist, int64_t v0, int64_t nv,
                                                 int64_t bi, int64_t nb) {
    if constexpr (G == kWave) return wave_rounds<Resolve, VLIST, E>(off, nbr, prev, next, vlist, v0, nv, bi, nb);
    else return group_rounds_lanes<G, Resolve, VLIST, E>(off, nbr, prev, next, vlist, v0, nv, bi, nb);
}

// Alt: the resolver of iterations where most rows are high-distinct (the
// learned dispatcher's count of such big vertices, *hd_count, exceeds half of
// hd_total); chosen once per launch, so each choice is its own pipeline.
// nv_dev, when given, holds the list's length (written on the device by an
// earlier kernel; nv is then only its capacity).  front: the rows that can
// still change (frontier.hip), walked instead when front_lists_on.
template <int G, class Resolve, class Alt, bool VLIST, typename E>
__global__ void __launch_bounds__(256)
k_group(const E *__restrict__ off, const int32_t *__restrict__ nbr,
        const int32_t *__restrict__ prev, int32_t *__restrict__ next,
        const int32_t *__restrict__ vlist, int64_t v0, int64_t nv, const int64_t *__restrict__ nv_dev,
        unsigned long long *__restrict__ counter, const int32_t *__restrict__ stop,
        const int64_t *__restrict__ hd_count, int64_t hd_total, FrontList front) {
    __shared__ uint32_t scratch[256 / kWave];
    if (*stop) return;
    if (front_lists_on(front)) {   // uniform
        nv = *front.len;
        if ((int64_t)blockIdx.x * (256 / G) >= nv) return;
        const uint32_t ch = group_rounds<G, Resolve, true, E>(off, nbr, prev, next, front.list, 0, nv,
                                                                   (int64_t)blockIdx.x, (int64_t)gridDim.x);
        block_count_add<4>(ch, counter, scratch);
        return;
    }
    if (nv_dev) nv = *nv_dev;
    const bool alt = hd_count && 2 * (*hd_count) > hd_total;   // uniform
    const int64_t bi = blockIdx.x, nb = gridDim.x;
    const uint32_t changed = alt ? group_rounds<G, Alt, VLIST, E>(off, nbr, prev, next, vlist, v0, nv, bi, nb)
                                 : group_rounds<G, Resolve, VLIST, E>(off, nbr, prev, next, vlist, v0, nv, bi, nb);
    block_count_add<4>(changed, counter, scratch);
}

}  // namespace galp
