"""Refinement sweeps with 32 right-hand sides: up to 15 tiles a half sweep is one
launch (left-looking, sums over a whole tile row in registers), above that a
launch per tile column (right-looking, the residual rounded after every step).

The two round differently, so a solve's form must be chosen by its own size: the
same solve alone and beside a larger one agrees bitwise, with the same number of
sweeps, at 1 tile, 14, and on both sides of the line.  A solve that did not
refine would be redone in FP64 and still meet LAPACK, so the sweeps have to be
counted (iters > 0); tau00 is held to the 1e-10 bar of the mixed path."""
import numpy as np
import pytest

from lsms_amd import capi
from lsms_amd import configs as CF
from tests.test_gpu_batch import lapack_tau00, rel

pytestmark = pytest.mark.gpu
MODES = [capi.PREC_MIXED_FP32, capi.PREC_MIXED_F16]


def canted(sizes, rcut):
    """Spin-canted system whose atom i has a zone of its first sizes[i] sites."""
    e, w = CF.contour_semicircle(-0.5, 0.7, 5)
    s = CF.make_system("columns", "bcc", 5.42, (2, 2, 2), rcut, 3, e, w, nspecies=2, seed=17,
                       local_atoms=list(range(len(sizes))), n_spin_cant=2, n_spin_pola=2)
    for a, n in zip(s.atoms, sizes):
        assert a.numLIZ >= n
        a.LIZPos = np.asfortranarray(a.LIZPos[:, :n])
        a.LIZlmax, a.LIZStoreIdx = a.LIZlmax[:n].copy(), a.LIZStoreIdx[:n].copy()
        a.numLIZ, a.nrmat = n, int(np.sum((a.LIZlmax + 1) ** 2))
    return s


@pytest.mark.parametrize("precision", MODES)
def test_alone_and_beside_larger_solves(precision):
    sizes = [2, 28, 30, 31, 32, 65]  # tiles: 1, 14, 15, 16, 16, 33
    s = canted(sizes, 12.0)
    assert [(s.nrmat_ns(a) + 63) // 64 for a in range(len(sizes))] == [1, 14, 15, 16, 16, 33]
    ctx = capi.Context(0)
    ctx.load_system(s)
    ie = 2

    def solve(atoms):
        tau, info = ctx.tau00_batched(atoms, [ie] * len(atoms), [s.prel(ie)] * len(atoms), 32,
                                      precision=precision)
        iters, _ = ctx.last_stats(len(atoms))
        assert np.all(info == 0) and np.all(iters > 0)
        return tau, iters

    alone = [solve([a]) for a in range(len(sizes))]
    for atoms in ([0, 1, 2], [3, 4, 5], [5, 2, 0, 3, 1, 4], [4, 1]):
        tau, iters = solve(atoms)
        for a, t, it in zip(atoms, tau, iters):
            assert np.array_equal(alone[a][0][0], t), (atoms, a)
            assert alone[a][1][0] == it
    for a in range(len(sizes)):
        assert rel(alone[a][0][0], lapack_tau00(s, a, ie)) < 1e-10
    ctx.close()


@pytest.mark.parametrize("precision", MODES)
def test_relativistic_solves_refine(precision):
    s = CF.config_rel()
    ctx = capi.Context(0)
    ctx.load_system(s)
    ctx.upload_tmats_rel(s.tmatStore, s.blkSizeTmatStore, len(s.energies), s.energies)
    _, info = ctx.tau00_batched([0, 1, 0, 1], [0, 1, 2, 3], [s.prel(i) for i in range(4)], 32,
                                precision=precision)
    iters, _ = ctx.last_stats(4)
    ctx.close()
    assert np.all(info == 0) and np.all(iters > 0)
