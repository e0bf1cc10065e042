"""Iterations that do not run the class kernels over every row: the closed
form of the first iteration (rows without repeated neighbours).  Every
iteration is compared with the oracle; labels and counts are whole numbers,
so they are equal or wrong."""
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
