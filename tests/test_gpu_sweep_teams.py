"""Refinement sweeps with a tile row by one wave and by a pair of waves.

The split is chosen by the largest solve of a launch and changes which wave
computes a row, never the arithmetic: a small solve alone (pairs) and the same
solve beside the largest one (single waves) must agree bitwise, and both are
held to the 1e-10 bar of the mixed path against LAPACK."""
import numpy as np
import pytest

from lsms_amd import capi
from lsms_amd import configs as CF
from tests.test_gpu_batch import lapack_tau00, pick, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [capi.PREC_MIXED_FP32, capi.PREC_MIXED_F16])
@pytest.mark.parametrize("nsites", [1, 4, 5, 20, 43, 44, 45, 48, 49])
def test_alone_and_beside_a_large_solve(precision, nsites):
    s = CF.config_c4()
    small, big = pick(s, 2)
    a, n = s.atoms[small], nsites
    a.LIZPos = np.asfortranarray(a.LIZPos[:, :n])
    a.LIZlmax, a.LIZStoreIdx = a.LIZlmax[:n].copy(), a.LIZStoreIdx[:n].copy()
    a.numLIZ, a.nrmat = n, int(np.sum((a.LIZlmax + 1) ** 2))
    ctx = capi.Context(0)
    ctx.load_system(s)
    ie = 11
    one, info = ctx.tau00_batched([small], [ie], [s.prel(ie)], 16, precision=precision)
    two, info2 = ctx.tau00_batched([small, big], [ie] * 2, [s.prel(ie)] * 2, 16, precision=precision)
    assert np.all(info == 0) and np.all(info2 == 0)
    assert s.nrmat_ns(big) > 12 * 64
    assert np.array_equal(one[0], two[0])
    assert rel(one[0], lapack_tau00(s, small, ie)) < 1e-10


@pytest.mark.parametrize("precision", [capi.PREC_MIXED_FP32, capi.PREC_MIXED_F16])
def test_both_sides_of_the_line(precision):
    """14 to 16 tiles (the line is at 15, where the pairs' y just fit LDS): each
    size alone, beside others on the pairs' side and beside the largest zone."""
    s = CF.config_c4()
    sizes = [56, 57, 60, 61, 64]
    big = pick(s, 2)[1]
    small = [a for a in range(len(s.atoms)) if s.atoms[a].numLIZ >= 64 and a != big][:len(sizes)]
    for i, n in zip(small, sizes):
        a = s.atoms[i]
        a.LIZPos = np.asfortranarray(a.LIZPos[:, :n])
        a.LIZlmax, a.LIZStoreIdx = a.LIZlmax[:n].copy(), a.LIZStoreIdx[:n].copy()
        a.numLIZ, a.nrmat = n, int(np.sum((a.LIZlmax + 1) ** 2))
    assert [-(-s.nrmat_ns(i) // 64) for i in small] == [14, 15, 15, 16, 16]
    assert s.nrmat_ns(big) > 16 * 64
    ctx = capi.Context(0)
    ctx.load_system(s)
    ie = 11

    def solve(atoms):
        tau, info = ctx.tau00_batched(atoms, [ie] * len(atoms), [s.prel(ie)] * len(atoms), 16,
                                      precision=precision)
        assert np.all(info == 0) and np.all(ctx.last_stats(len(atoms))[0] > 0)
        return tau

    for i, beside in zip(small, solve(small + [big])):
        alone = solve([i])[0]
        assert np.array_equal(alone, beside), s.atoms[i].numLIZ
        assert np.array_equal(alone, solve([small[0], i])[1])
        assert rel(alone, lapack_tau00(s, i, ie)) < 1e-10
