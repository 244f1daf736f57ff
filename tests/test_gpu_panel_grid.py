"""Groups of elimination steps and the two splits of their panels and trailing
updates (a 64x64 tile per workgroup, or a quarter of one where the launch would
leave compute units idle).

The split changes which workgroup computes an entry, never its arithmetic: a
solve's result must not depend on how many others are in its launch, so copies
of one solve in batches on both sides of the line are compared bitwise.  Sizes
with every remainder of a group of four steps are checked against LAPACK; LU of
matrices near 1 has a backward error of a small multiple of n eps, so the
forward error is held to 8 n eps cond(M)."""
import numpy as np
import pytest

from lsms_amd import capi
from lsms_amd import configs as CF
from tests.test_gpu_batch import lapack_tau00, pick, rel
from tests.test_gpu_tile_lu import EPS, matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [capi.PREC_FP64, capi.PREC_MIXED_FP32])
def test_split_is_bitwise_the_same(precision):
    s = CF.config_c4()
    ctx = capi.Context(0)
    ctx.load_system(s)
    for a, ie in zip(pick(s, 3), (2, 17, 30)):
        one, info = ctx.tau00_batched([a], [ie], [s.prel(ie)], 16, precision=precision)
        assert np.all(info == 0)
        assert rel(one[0], lapack_tau00(s, a, ie)) < 1e-10
        for nb in (7, 33, 120):
            tau, info = ctx.tau00_batched([a] * nb, [ie] * nb, [s.prel(ie)] * nb, 16,
                                          precision=precision)
            assert np.all(info == 0)
            assert np.array_equal(tau, np.broadcast_to(one, tau.shape)), (a, nb)


@pytest.mark.parametrize("n", [128, 192, 256, 257, 320, 384, 449, 576, 641])
def test_group_remainders(n):
    rng = np.random.default_rng(n)
    m = matrix("near1", n, 16, rng)
    t0 = rng.normal(size=(16, 16)) + 1j * rng.normal(size=(16, 16))
    rhs = np.zeros((n, 16), dtype=complex)
    rhs[:16] = t0
    ref = np.linalg.solve(m, rhs)
    tau, info = capi.Context(0).solve_tau00_matrix(m, t0)
    assert info == 0
    assert np.linalg.norm(tau - ref[:16]) <= 8 * n * EPS * np.linalg.cond(m) * np.linalg.norm(ref)


@pytest.mark.parametrize("precision", [capi.PREC_FP64, capi.PREC_MIXED_FP32])
@pytest.mark.parametrize("right_align", [0, 1])
def test_cross_updates_of_uneven_batch(precision, right_align):
    """Solves of different tile counts in one launch sequence: a solve whose group
    ends early leaves the later cross updates out.  A wrong FP32 update shows as a
    refinement that does not converge and falls back to FP64 (iters = -1)."""
    s = CF.config_c4()
    ctx = capi.Context(0)
    ctx.load_system(s)
    ctx.set_schedule(right_align)
    atoms, ie = pick(s, 6), 9
    tau, info = ctx.tau00_batched(atoms, [ie] * 6, [s.prel(ie)] * 6, 16, precision=precision)
    assert np.all(info == 0)
    iters, _ = ctx.last_stats(6)
    assert np.all(iters == 0 if precision == capi.PREC_FP64 else iters > 0)
    for a, t in zip(atoms, tau):
        assert rel(t, lapack_tau00(s, a, ie)) < 1e-10
