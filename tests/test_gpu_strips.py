"""Large split-FP16 batches.  Those of one size take their panels as strips
(k_lu_strip_h, from 4864 strips a launch), whose products are those of the
step-by-step panels; uneven ones do not.  Either way a solve's result must not
depend on how many others are in its batch: 256 solves (24 tile rows and columns
beyond the first group's block) against the same solves eight at a time, bitwise
and with the same sweeps, under each schedule and replayed from a graph.  A solve
that did not refine would be redone in FP64 and agree all the same, so iters > 0;
tau00 is held to the 1e-10 bar of the mixed path."""
import numpy as np
import pytest

from lsms_amd import capi
from lsms_amd import configs as CF
from tests.test_gpu_batch import lapack_tau00, pick, rel

pytestmark = pytest.mark.gpu
COPIES = 32


@pytest.fixture(scope="module")
def c4():
    s = CF.config_c4()
    ctx = capi.Context(0)
    ctx.load_system(s)
    yield s, ctx
    ctx.close()


@pytest.mark.parametrize("group", [4, 8])
@pytest.mark.parametrize("uneven", [True, False])
def test_large_batch_equals_small_ones(c4, uneven, group):
    s, ctx = c4
    atoms = pick(s, 8) if uneven else [pick(s, 2)[1]] * 8
    iies = [1, 5, 9, 13, 17, 21, 25, 29]
    prels = [s.prel(i) for i in iies]
    ctx.set_split_group(group)

    def solve(copies):
        tau, info = ctx.tau00_batched(atoms * copies, iies * copies, prels * copies, 16,
                                      precision=capi.PREC_MIXED_F16)
        iters, _ = ctx.last_stats(8 * copies)
        assert np.all(info == 0) and np.all(iters > 0)
        return tau, iters

    tau8, iters8 = solve(1)
    runs = []
    for flags in (0, capi.SCHED_RIGHT_ALIGN, capi.SCHED_RIGHT_ALIGN | capi.SCHED_XCD_SWIZZLE,
                  capi.SCHED_RIGHT_ALIGN | capi.SCHED_TWO_STREAMS):
        ctx.set_schedule(flags)
        runs.append(solve(COPIES))
    ctx.set_graph(True)
    for rep in range(2):
        runs.append(solve(COPIES))
        ctx.set_graph(False)
        solve(1)
        ctx.set_graph(True)
    ctx.set_graph(False)
    ctx.set_schedule(0)
    ctx.set_split_group(8)
    for tau, iters in runs:
        assert np.array_equal(tau, np.tile(tau8, (COPIES, 1, 1))) is True
        assert np.array_equal(iters, np.tile(iters8, COPIES)) is True
    for b in (0, 7):
        assert rel(tau8[b], lapack_tau00(s, atoms[b], iies[b])) < 1e-10
