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
