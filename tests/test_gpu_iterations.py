"""Iterations that do not run the class kernels over every row: the closed
form of the first iteration (rows without repeated neighbours) and the later
iterations over the rows with a changed neighbour (symmetric graphs of at
least 2^23 edges).  Every iteration is compared with the oracle; labels and
counts are whole numbers, so they are equal or wrong."""
import numpy as np
import pytest

import oracle
from galp_amd import _abi

pytestmark = pytest.mark.gpu


def csr(rows):
    off = np.zeros(len(rows) + 1, np.int64)
    off[1:] = np.cumsum([len(r) for r in rows])
    return off, np.array([u for r in rows for u in r], np.int32)


def mixed_rows(seed, order):
    """Rows of every class (up to a hub), empty rows and self-loops; `order`:
    ascending, one row descending, or one repeated neighbour."""
    rng = np.random.default_rng(seed)
    n = 9001
    sizes = [0, 1, 4, 5, 64, 65, 129, 513, 1025, 2049, 4096, 4097, 6500]
    rows = [np.sort(rng.choice(n, size=sizes[v % len(sizes)] if v < 40 else int(rng.integers(0, 9)),
                               replace=False)).tolist() for v in range(n)]
    rows[50] = [50]
    rows[51] = [7, 51, 90]
    if order == "descending":
        rows[60] = [9, 8, 3]
    elif order == "repeated":
        rows[60] = [3, 8, 8, 9]
    return csr(rows)


def check_steps(g, off, nbr, steps):
    prev = np.arange(len(off) - 1, dtype=np.int32)
    for it in range(steps):
        ref, cnt = oracle.lp_iterate(off, nbr, prev)
        st = g.step()
        assert st["updated"] == cnt, it + 1
        assert np.array_equal(g.labels(), ref), it + 1
        prev = ref


@pytest.mark.parametrize("order", ["ascending", "descending", "repeated"])
@pytest.mark.parametrize("opts", [dict(), dict(reorder=0), dict(method=_abi.METHOD_SORT), dict(offsets64=1),
                                  dict(policy=_abi.POLICY_OOC_ASYNC, buffer_pow=12),
                                  dict(policy=_abi.POLICY_OOC_SYNC, buffer_pow=12, reorder=0)],
                         ids=["hash", "noreorder", "sort", "off64", "ooc", "ooc-noreorder"])
def test_first_iteration(ctx, order, opts):
    off, nbr = mixed_rows(1, order)
    print(f"[first] {order} {opts}", flush=True)
    with _abi.Graph(ctx, off, nbr, **opts) as g:
        g.init()
        check_steps(g, off, nbr, 2)
        # labels set by the caller are not labels[i] = i: the general path
        lab = np.random.default_rng(3).integers(0, len(off) - 1, size=len(off) - 1).astype(np.int32)
        g.set_labels(lab)
        ref, cnt = oracle.lp_iterate(off, nbr, lab)
        assert g.step()["updated"] == cnt
        assert np.array_equal(g.labels(), ref)


@pytest.mark.parametrize("reorder", [1, 0])
def test_repeats_found_out_of_core(ctx, reorder):
    """A repeated neighbour at any place of the pass over the ids: inside a
    thread's eight edges, between two threads, waves, rounds and tiles, first
    and last in its row.  Its label counts twice, so the closed form is wrong."""
    n, d = 20000, 9001
    rest = [[(3 * v + 1) % n] if v % 3 else [] for v in range(n - 2)]
    for p in [1, 7, 8, 9, 511, 512, 513, 2047, 2048, 2049, 8191, 8192, 8193, d - 1, 0]:
        row = np.arange(5, 5 + 2 * d, 2)
        if p:
            row[p] = row[p - 1]
        off, nbr = csr([row.tolist(), [1, 2, 3]] + rest)   # p = 0: nothing repeated
        with _abi.Graph(ctx, off, nbr, policy=_abi.POLICY_OOC_ASYNC, buffer_pow=14, reorder=reorder) as g:
            g.init()
            check_steps(g, off, nbr, 2)


def test_first_iteration_logs_distinct_counts(ctx):
    """The distinct-label counts logged for the first iteration are the degrees."""
    off, nbr = mixed_rows(2, "ascending")
    big = np.diff(off) > 64
    with _abi.Graph(ctx, off, nbr) as g:
        g.log_enable(4 * int(big.sum()))
        g.init()
        g.step()
        x, y = g.log_read()
    assert len(y) == big.sum() and np.all(x[:, 3] == -1.0)
    got = np.sort(np.rint(np.exp2(y.astype(np.float64)) - 1).astype(np.int64))
    assert np.array_equal(got, np.sort(np.diff(off)[big]))


@pytest.mark.parametrize("distinct", [1, 2, 3, 17, 63, 5000])
def test_lane_group_rows(ctx, distinct):
    """Rows of 1..64 edges over labels of `distinct` values, the lowest and
    the highest vertex id among them: every mix of settled and diverse rows."""
    rng = np.random.default_rng(distinct)
    n = 6007
    rows = [rng.integers(0, n, size=v % 65).tolist() for v in range(n)]
    off, nbr = csr(rows)
    values = np.unique(np.concatenate([[0, n - 1], rng.integers(0, n, size=distinct)]))[:max(distinct, 1)]
    lab = values[rng.integers(0, len(values), size=n)].astype(np.int32)
    lab[:n // 2:3] = values[0]   # some rows mostly one label
    for opts in (dict(), dict(reorder=0), dict(method=_abi.METHOD_SORT)):
        print(f"[groups] distinct={distinct} {opts}", flush=True)
        with _abi.Graph(ctx, off, nbr, **opts) as g:
            g.set_labels(lab)
            ref, cnt = oracle.lp_iterate(off, nbr, lab)
            assert g.step()["updated"] == cnt
            assert np.array_equal(g.labels(), ref)


@pytest.fixture(scope="module")
def settling():
    """A symmetric graph of at least 2^23 edges that settles within a dozen
    iterations, with rows of every class: communities of 400 vertices, and
    vertices of degree 1..9000 joined to whole communities' members, in two
    copies that share no edge."""
    rng = np.random.default_rng(5)
    n, comm = 190000, 400
    u = np.repeat(np.arange(n), 12)
    v = u // comm * comm + rng.integers(0, comm, size=len(u))
    keep = u % comm >= 8   # eight vertices of each community draw nothing: short rows
    u, v = u[keep], v[keep]
    v = np.where(v % comm < 8, v + 8, v)
    pairs = [np.stack([u, v], 1), rng.integers(0, n, size=(20000, 2))]
    for k, d in enumerate([66, 130, 260, 520, 1030, 2050, 4096, 4097, 9000, 6000]):
        others = rng.choice(n, size=d, replace=False)
        pairs.append(np.stack([np.full(d, 7 + 397 * k), others], 1))
    e = np.concatenate(pairs)
    e = e[e[:, 0] != e[:, 1]]
    key = np.unique(np.concatenate([e[:, 0] * n + e[:, 1], e[:, 1] * n + e[:, 0]]))
    off = np.searchsorted(key // n, np.arange(n + 1)).astype(np.int64)
    nbr = (key % n).astype(np.int32)
    off = np.concatenate([off, off[1:] + off[-1], [2 * off[-1]]])   # and one vertex without edges
    nbr = np.concatenate([nbr, nbr + np.int32(n)])
    assert len(nbr) >= 1 << 23
    refs, prev = [], np.arange(2 * n + 1, dtype=np.int32)
    for _ in range(12):
        prev, cnt = oracle.lp_iterate(off, nbr, prev)
        refs.append((prev, cnt))
    return off, nbr, refs


VARIANTS = [dict(), dict(reorder=0), dict(method=_abi.METHOD_SORT), dict(method=_abi.METHOD_SORT, reorder=0),
            dict(offsets64=1), dict(profile=1)]


@pytest.mark.parametrize("opts", VARIANTS, ids=["hash", "hash-noreorder", "sort", "sort-noreorder", "off64", "profile"])
def test_changed_rows_only(ctx, settling, opts):
    off, nbr, refs = settling
    print(f"[lists] {opts} m={len(nbr)}", flush=True)
    with _abi.Graph(ctx, off, nbr, **opts) as g:
        g.init()
        for it, (ref, cnt) in enumerate(refs):
            st = g.step()
            assert st["updated"] == cnt, it + 1
            assert np.array_equal(g.labels(), ref), it + 1
        if opts.get("profile"):   # the class kernels' bytes show that the lists were walked
            prof = {k["name"]: k for k in g.profile()}
            assert prof["front"]["launches"] >= 9
            full = sum(g.info()["bucket_edges"]) * 8.0 * (len(refs) - 1)
            assert 0 < sum(k["alg_bytes"] for nm, k in prof.items() if nm != "first") < 0.8 * full
        # any other state: the lists start over
        lab = refs[-1][0].copy()
        lab[::9773] = np.arange(len(lab))[::9773]
        g.set_labels(lab)
        for it in range(3):
            lab, cnt = oracle.lp_iterate(off, nbr, lab)
            assert g.step()["updated"] == cnt, it
            assert np.array_equal(g.labels(), lab), it


@pytest.mark.parametrize("method", [_abi.METHOD_HASH, _abi.METHOD_SORT])
def test_lists_need_no_budget(ctx, settling, method):
    """A budget without room for all of the lists' memory, the last of which
    holds a profiled graph's byte counts, runs every iteration over all rows."""
    off, nbr, refs = settling
    opts = dict(method=method, reorder=0, profile=1)   # renumbering peaks higher than the lists
    with _abi.Graph(ctx, off, nbr, **opts) as g:
        total = g.info()["device_bytes"]
    with _abi.Graph(ctx, off, nbr, mem_budget=total, **opts) as g:
        g.run(4, want_labels=False)
        assert "front" in {k["name"] for k in g.profile()}
    with _abi.Graph(ctx, off, nbr, mem_budget=total - 1, **opts) as g:
        assert g.info()["device_bytes"] < total
        g.init()
        for it, (ref, cnt) in enumerate(refs[:8]):
            assert g.step()["updated"] == cnt, it + 1
            assert np.array_equal(g.labels(), ref), it + 1
        assert "front" not in {k["name"] for k in g.profile()}


@pytest.mark.parametrize("capture", [0, 1])
def test_changed_rows_only_device_loop(ctx, settling, capture):
    off, nbr, refs = settling
    stop = next((i for i, (_, c) in enumerate(refs) if c <= (len(off) - 1) * 1e-5), len(refs) - 1)
    with _abi.Graph(ctx, off, nbr, graph_capture=capture) as g, _abi.Graph(ctx, off, nbr) as other:
        for rep in range(3):
            labels, res = g.run(len(refs))
            assert res["iterations"] == stop + 1, rep
            assert np.array_equal(labels, refs[stop][0]), rep
            other.run(3)   # eager work between the replays


def test_one_way_edges_take_every_row(ctx, settling):
    """Without the reverse of one edge the lists would miss a row."""
    off, nbr, _ = settling
    e = int(off[100])
    off2 = off.copy()
    off2[101:] -= 1
    nbr2 = np.delete(nbr, e)
    with _abi.Graph(ctx, off2, nbr2, profile=1) as g:
        g.init()
        check_steps(g, off2, nbr2, 8)
        assert "front" not in {k["name"] for k in g.profile()}


@pytest.mark.parametrize("edit", ["none", "one-way", "swap", "triangle", "last-row"])
@pytest.mark.parametrize("opts", [dict(), dict(reorder=0), dict(offsets64=1),
                                  dict(policy=_abi.POLICY_OOC_ASYNC, buffer_pow=20, mem_budget=1 << 30)],
                         ids=["hash", "noreorder", "off64", "ooc-budget"])
def test_symmetry_check(ctx, settling, opts, edit):
    """Lists are used on symmetric graphs, out of core also under a memory
    budget, and on no other: one edge without its reverse, two edges whose
    ends are exchanged (all degrees as before), a directed triangle, an edge
    of the last rows."""
    off, nbr, _ = settling
    rows = np.repeat(np.arange(len(off) - 1), np.diff(off))
    key = rows * np.int64(len(off)) + nbr

    if edit == "one-way":
        key = np.delete(key, 12345)
    elif edit == "last-row":
        key = np.delete(key, len(key) - 1)
    elif edit == "swap":   # a -> b, c -> d become a -> d, c -> b
        e, f = 1000, 5000000
        (a, b), (c, d) = (rows[e], nbr[e]), (rows[f], nbr[f])
        assert len({a, b, c, d}) == 4
        key[[e, f]] = a * len(off) + d, c * len(off) + b
    elif edit == "triangle":
        tri = np.array([100, 150000, 300000])
        key = np.concatenate([key, tri * np.int64(len(off)) + np.roll(tri, 1)])
    key.sort()
    assert np.all(key[1:] > key[:-1])
    off2 = np.searchsorted(key // len(off), np.arange(len(off))).astype(np.int64)
    with _abi.Graph(ctx, off2, (key % len(off)).astype(np.int32), profile=1, **opts) as g:
        g.run(3, want_labels=False)
        assert ("front" in {k["name"] for k in g.profile()}) == (edit == "none")


@pytest.mark.parametrize("net", ["all-cand", "rand"])
def test_changed_rows_only_learned(ctx, settling, net):
    off, nbr, refs = settling
    params = np.zeros(_abi.mlp_num_params(8), np.float32) if net == "all-cand" else _abi.mlp_init(8, 3)
    with _abi.Graph(ctx, off, nbr, dispatch=_abi.DISPATCH_LEARNED) as g:
        g.set_mlp(8, params, 6.0)
        g.init()
        for it, (ref, cnt) in enumerate(refs):
            assert g.step()["updated"] == cnt, it + 1
            assert np.array_equal(g.labels(), ref), it + 1


@pytest.mark.parametrize("opts", [dict(), dict(reorder=0), dict(policy=_abi.POLICY_OOC_ASYNC, buffer_pow=20)],
                         ids=["hash", "noreorder", "ooc"])
def test_dispatch_counters_over_lists(ctx, settling, opts):
    """The dispatch counters after an iteration are its own: every big row
    where the network routed it, nothing after the closed form or the lists."""
    off, nbr, refs = settling
    deg = np.diff(off)
    routed = int(((deg > 64) & (deg <= (1024 if "policy" in opts else 1 << 30))).sum())   # one tile out of core
    with _abi.Graph(ctx, off, nbr, dispatch=_abi.DISPATCH_LEARNED, **opts) as g:
        g.set_mlp(8, np.zeros(_abi.mlp_num_params(8), np.float32), 6.0)   # predicts 0 labels: every big row
        for _ in range(2):
            g.init()
            for it, (ref, cnt) in enumerate(refs):
                st = g.step()
                assert st["updated"] == cnt
                ds = g.dispatch_stats()
                assert st["overflowed"] == ds[_abi.DS_OVERFLOW], it + 1
                if it in (1, 2):   # too many changes for the lists
                    assert ds[_abi.DS_CAND_VERTS] == routed, it + 1
                elif it == 0 or it == len(refs) - 1:
                    assert not ds.any(), it + 1
            assert np.array_equal(g.labels(), refs[-1][0])


@pytest.mark.parametrize("mask", [None, 0b1111111], ids=["every", "to-7"])
def test_counts_of_rows_left_out(ctx, mask):
    """Distinct-label counts, the network's input: samples logged after
    iterations on the lists hold each row's count of the iteration before,
    also for rows that were left out of it."""
    off, nbr = _abi.gen_lfr(400000, avg_deg=24.0, max_deg=1500, mu=0.3, seed=9)
    assert len(nbr) >= 1 << 23
    big = np.nonzero(np.diff(off) > 64)[0]
    labs = [np.arange(len(off) - 1, dtype=np.int32)]
    for _ in range(9):
        labs.append(oracle.lp_iterate(off, nbr, labs[-1])[0])

    def counts(lab):
        return np.array([len(np.unique(lab[nbr[off[v]:off[v + 1]]])) for v in big])

    with _abi.Graph(ctx, off, nbr, dispatch=_abi.DISPATCH_LEARNED) as g:
        g.set_mlp(8, _abi.mlp_init(8, 3), 6.0)
        if mask is not None:   # the last two by the classes alone, which need and keep no counts
            g.set_learned_iterations(mask | (0b11 << 8))
        g.init()
        for it in range(8):
            g.step()
        assert np.array_equal(g.labels(), labs[8])
        g.log_enable(len(big))
        g.step()
        x, y = g.log_read()
        assert np.array_equal(g.labels(), labs[9])
    before, now = (np.rint(np.exp2(z.astype(np.float64)) - 1).astype(np.int64) for z in (x[:, 3], y))
    want = np.stack([np.diff(off)[big], counts(labs[7]), counts(labs[8])], 1)
    got = np.stack([np.rint(np.exp2(x[:, 0].astype(np.float64)) - 1).astype(np.int64), before, now], 1)
    assert len(got) == len(big)
    assert np.array_equal(got[np.lexsort(got.T)], want[np.lexsort(want.T)])


@pytest.mark.parametrize("method", [_abi.METHOD_HASH, _abi.METHOD_SORT])
def test_changed_rows_only_batch(ctx, settling, method):
    """The two copies as two graphs of a batch: each stops by its own rule."""
    off, nbr, refs = settling
    n = (len(off) - 2) // 2
    final, per, counts = oracle.lp_run(off[:n + 1], nbr[:off[n]], niter=12)
    with _abi.Graph(ctx, off, nbr, method=method, reorder=0) as g:
        g.set_batch([0, n, 2 * n + 1])
        labels, _ = g.run(12)
        iters = g.batch_iterations()
    assert iters[0] == len(counts)
    assert np.array_equal(labels[:n], final) and np.array_equal(labels[n:2 * n] - n, final)


@pytest.mark.parametrize("opts", [dict(policy=_abi.POLICY_OOC_ASYNC, buffer_pow=20),
                                  dict(policy=_abi.POLICY_OOC_SYNC, buffer_pow=21, reorder=0),
                                  dict(policy=_abi.POLICY_OOC_ASYNC, buffer_pow=24),
                                  dict(policy=_abi.POLICY_OOC_ASYNC, buffer_pow=20, method=_abi.METHOD_SORT),
                                  dict(policy=_abi.POLICY_OOC_ASYNC, buffer_pow=20, dispatch=_abi.DISPATCH_LEARNED)],
                         ids=["async", "sync-noreorder", "one-batch", "sort", "learned"])
def test_changed_rows_only_out_of_core(ctx, settling, opts):
    """Streamed iterations, then lists read from host memory, and from new
    labels streamed again (the prefetched batches are still in place)."""
    off, nbr, refs = settling
    print(f"[lists] {opts}", flush=True)
    with _abi.Graph(ctx, off, nbr, **opts) as g:
        if "dispatch" in opts:
            g.set_mlp(8, _abi.mlp_init(8, 4), 6.0)
        for _ in range(2):
            g.init()
            for it, (ref, cnt) in enumerate(refs):
                st = g.step()
                assert st["updated"] == cnt, it + 1
                assert np.array_equal(g.labels(), ref), it + 1
        stop = next((i for i, (_, c) in enumerate(refs) if c <= (len(off) - 1) * 1e-5), len(refs) - 1)
        labels, res = g.run(len(refs) + 3 if stop < len(refs) - 1 else len(refs))
        assert res["iterations"] == stop + 1 and np.array_equal(labels, refs[stop][0])


ROW_KERNELS = ("g4", "g8", "g16", "g32", "g64", "w128", "w256", "w512", "b1k", "b2k", "b4k", "hub_tile", "hub_sort")


@pytest.mark.parametrize("opts", [dict(policy=_abi.POLICY_OOC_ASYNC, buffer_pow=20),
                                  dict(policy=_abi.POLICY_OOC_SYNC, buffer_pow=21, reorder=0),
                                  dict(policy=_abi.POLICY_OOC_ASYNC, buffer_pow=24),
                                  dict(policy=_abi.POLICY_OOC_ASYNC, buffer_pow=20, method=_abi.METHOD_SORT)],
                         ids=["async", "sync-noreorder", "one-batch", "sort"])
def test_profiled_bytes_out_of_core(ctx, settling, opts):
    """The row kernels of an iteration that streams every batch count each
    edge once (id and label), each row's labels and offsets, and one offset
    more per kernel; those of an iteration on the lists only what they walk."""
    off, nbr, refs = settling
    rows, m = int((np.diff(off) > 0).sum()), len(nbr)
    with _abi.Graph(ctx, off, nbr, profile=1, **opts) as g:
        g.init()
        read = []
        for it, (ref, cnt) in enumerate(refs):
            g.profile_reset()
            assert g.step()["updated"] == cnt, it + 1
            prof = [k for k in g.profile() if k["name"] in ROW_KERNELS]
            read.append(sum(k["alg_bytes"] for k in prof))
            launches = sum(k["launches"] for k in prof)
            if it in (1, 2):   # streamed: the second without the lists, the third after looking at them
                hubs = g.info()["bucket_vertices"][11]
                assert read[it] == 8 * m + 12 * (rows - hubs) + 4 * (launches - hub_launches(prof)), it + 1
    assert 0 < read[-1] < 0.4 * read[2]


@pytest.mark.parametrize("pow2", [20, 24], ids=["nine-batches", "one-batch"])
def test_out_of_core_copies(ctx, settling, pow2):
    """Every run copies its batches itself: what an earlier run left in the
    buffers, or copied ahead and did not use, is not counted on.  The copies
    are complete when the call returns (else they would not be counted)."""
    off, nbr, refs = settling
    m = len(nbr)

    def copied(g):
        b = sum(k["alg_bytes"] for k in g.profile() if k["name"] == "h2d")
        g.profile_reset()
        return b

    with _abi.Graph(ctx, off, nbr, policy=_abi.POLICY_OOC_ASYNC, buffer_pow=pow2, profile=1) as g:
        per_run = []
        for _ in range(3):
            g.run(len(refs), want_labels=False)
            per_run.append(copied(g))
        print(f"[ooc] copied per run {per_run}, m={m}", flush=True)
        assert per_run[0] == per_run[1] == per_run[2]
        assert per_run[0] == 4 * m if pow2 == 24 else per_run[0] >= 8 * m
        for _ in range(2):
            g.set_labels(refs[-1][0])
            ref, cnt = oracle.lp_iterate(off, nbr, refs[-1][0])
            assert g.step()["updated"] == cnt and copied(g) == 4 * m
            assert np.array_equal(g.labels(), ref)
        for _ in range(2):
            g.init()
            for it in range(2):   # the first iteration's closed form needs no batch
                assert g.step()["updated"] == refs[it][1] and copied(g) == 4 * m * it


def hub_launches(prof):
    return sum(k["launches"] for k in prof if k["name"].startswith("hub_"))


@pytest.mark.parametrize("reorder", [1, 0])
@pytest.mark.parametrize("sizes", ["tiny", "edge"])
def test_batch_counts_per_graph(ctx, sizes, reorder):
    """Batches whose graphs end anywhere in a block's run of vertices: more
    than 64 graphs in one run, graphs of one vertex, and graphs that end at,
    before and behind a run's end (4096 vertices), the last one ragged."""
    rng = np.random.default_rng(12)
    ns = [int(x) for x in rng.integers(1, 90, 400)] if sizes == "tiny" else [4096, 4095, 1, 2, 8193, 1, 3]
    rows, parts, vbase = [], [], [0]
    for n in ns:
        a, b = rng.integers(0, n, 3 * n), rng.integers(0, n, 3 * n)
        nb = [set() for _ in range(n)]
        for x, y in zip(a.tolist(), b.tolist()):
            if x != y:
                nb[x].add(y)
                nb[y].add(x)
        own = [sorted(s) for s in nb]
        parts.append(csr(own))
        rows += [[u + vbase[-1] for u in r] for r in own]
        vbase.append(vbase[-1] + n)
    off, nbr = csr(rows)
    print(f"[batch] {sizes} reorder={reorder} graphs={len(ns)} n={len(rows)}", flush=True)
    with _abi.Graph(ctx, off, nbr, reorder=reorder) as g:
        g.set_batch(vbase)
        for _ in range(2):
            labels, _ = g.run(10)
            iters = g.batch_iterations()
            for k, (o, u) in enumerate(parts):
                final, _, counts = oracle.lp_run(o, u, niter=10)
                assert np.array_equal(labels[vbase[k]:vbase[k + 1]] - vbase[k], final), k
                assert iters[k] == len(counts), k
