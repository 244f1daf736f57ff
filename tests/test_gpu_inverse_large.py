"""Explicit inverse of matrices whose tile rows span more than 2^31 bytes (728
sites at lmax 3, Ns = 11648, by quarter tiles) and more than 2^32 (1028 sites, Ns
= 16448, by whole tiles): every operand offset of the products has to hold there.

M (tau x) = T x for a random x, with M assembled by build_kkr and T taken from
the store.  The explicit inverse of a matrix near 1 has a residual of a small
multiple of n eps (4e-12 here), so 1e-10 leaves room for its condition; a product
that loses or mistakes rows is off by orders of magnitude more."""
import numpy as np
import pytest

from lsms_amd import capi
from lsms_amd import configs as CF
from oracle import oracle as O
from tests.test_gpu_batch import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsites", [728, 1028])
def test_tau_full_inverts_a_large_zone(nsites):
    e, w = CF.contour_semicircle(-0.5, 0.7, 5)
    s = CF.make_system("large", "bcc", 5.42, (1, 1, 1), 27.5, 3, e, w, nspecies=2, seed=5,
                       local_atoms=[0])
    a = s.atoms[0]
    assert a.numLIZ >= nsites
    a.LIZPos = np.asfortranarray(a.LIZPos[:, :nsites])
    a.LIZlmax, a.LIZStoreIdx = a.LIZlmax[:nsites].copy(), a.LIZStoreIdx[:nsites].copy()
    a.numLIZ, a.nrmat = nsites, 16 * nsites
    ctx = capi.Context(0)
    ctx.load_system(s)
    ie, n = 2, 16 * nsites
    rng = np.random.default_rng(nsites)
    x = rng.normal(size=n) + 1j * rng.normal(size=n)
    tau, info = ctx.tau_full(0, ie, s.prel(ie), n)
    assert info == 0
    y = tau @ x
    del tau
    t = [O.t0(3, i, s.tmatStore, s.blkSizeTmatStore, ie) for i in range(2)]
    tx = np.concatenate([t[i] @ v for i, v in zip(a.LIZStoreIdx, x.reshape(nsites, 16))])
    assert rel(ctx.build_kkr(0, ie, s.prel(ie), n) @ y, tx) < 1e-10
    ctx.close()
