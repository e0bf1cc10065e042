"""The memory budget (mem_budget) a graph needs: what it holds on the device
at the upload's peak, byte by byte.  Bookkeeping that is spread over cache
lines counts as the words it stands for."""
import numpy as np
import pytest

import oracle
from galp_amd import _abi

pytestmark = pytest.mark.gpu

ITER_COUNTS = 8 * 4096   # a change count per iteration


def least_budget(off, nbr, reorder):
    n, m = len(off) - 1, len(nbr)
    rows = int((np.diff(off) > 0).sum())
    fixed = 4 * m + 8 * n + 4 * (n + 1) + 8 + 3 * 4 + ITER_COUNTS   # CSR, labels, counter, control words
    if not reorder:
        return fixed + 4 * rows                              # the class lists
    return fixed + 12 * n + 8 * (n + 1) + 4 * m              # renumbering, read-out, and the original CSR


@pytest.mark.parametrize("reorder", [0, 1])
@pytest.mark.parametrize("method", [_abi.METHOD_HASH, _abi.METHOD_SORT])
def test_least_budget(ctx, method, reorder):
    off, nbr = _abi.gen_planted_partition(1000, 50, 8, 2, 1)   # small: the fixed part decides; no hubs
    final, _, _ = oracle.lp_run(off, nbr, niter=10)
    need = least_budget(off, nbr, reorder)
    with _abi.Graph(ctx, off, nbr, method=method, reorder=reorder, mem_budget=need) as g:
        labels, _ = g.run(10)
        assert np.array_equal(labels, final)
    with pytest.raises(_abi.GalpError) as e:
        _abi.Graph(ctx, off, nbr, method=method, reorder=reorder, mem_budget=need - 1)
    assert e.value.code == -2
