"""Captured launch sequences with two streams: each half of a chunk has launches of
its own, and a sequence is replayed for every batch of the same shape, whichever
half its largest solve is in.  The same solves in two orders, replayed in turn
with eager work between, equal the eager results bitwise."""
import numpy as np
import pytest

from lsms_amd import capi
from lsms_amd import configs as CF
from tests.test_gpu_batch import pick

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [capi.PREC_FP64, capi.PREC_MIXED_FP32, capi.PREC_MIXED_F16])
@pytest.mark.parametrize("shared", [False, True])
def test_halves_in_either_order(precision, shared):
    s = CF.config_c4()
    ctx = capi.Context(0)
    ctx.load_system(s)
    ctx.set_schedule(capi.SCHED_TWO_STREAMS)
    small, big = pick(s, 2)
    assert s.nrmat_ns(small) < s.nrmat_ns(big)
    # shared: two solves of one zone and energy, so the structure constants are
    # formed once and the blocks come from them
    up = ([small, small, big, big], [3, 3, 17, 17] if shared else [3, 8, 17, 25])
    orders = [up, (up[0][::-1], up[1][::-1])]

    def solve(order, graph):
        ctx.set_graph(graph)
        tau, info = ctx.tau00_batched(*order, [s.prel(i) for i in order[1]], 16,
                                      precision=precision)
        assert np.all(info == 0)
        return tau

    eager = [solve(o, False) for o in orders]
    for rep in range(3):
        for o, ref in zip(orders, eager):
            assert [np.array_equal(x, y) for x, y in zip(solve(o, True), ref)] == [True] * 4, rep
            solve((up[0][1:3], up[1][1:3]), False)
    ctx.close()
