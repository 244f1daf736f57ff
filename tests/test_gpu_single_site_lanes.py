"""Both splits of the radial integration: a quad of lanes per integration in
small batches, one thread per integration in batches that fill the chip.

The two take the same steps with the same tableau, so they differ by rounding
only: 450 intervals at a few eps each, with the growth of the irregular
solution inwards well under a factor of 100 per eps; held to 1e-11 relative to
the largest value of a column."""
import numpy as np
import pytest

from lsms_amd import capi
from lsms_amd import configs as CF

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrel", [0, 10])
def test_large_batch_equals_small_ones(nrel):
    ctx = capi.Context(0)
    rr, vr, jm, jw, rs, e, pr = CF.single_site_batch(nspecies=2, ne=8)
    rep = 70  # 4 potentials x 560 energies x 4 l, both directions: 17920 integrations
    big = ctx.single_site_nonrel(nrel, 3, vr, rr, jm, jw, rs, np.tile(e, rep), np.tile(pr, rep))
    one = ctx.single_site_nonrel(nrel, 3, vr, rr, jm, jw, rs, e, pr)
    assert big[4] == 0 and one[4] == 0
    for q in (0, 2, 3):  # matom, zlr, jlr
        x = np.asarray(big[q]).reshape((rep, len(e)) + np.asarray(one[q]).shape[1:])
        ref = np.asarray(one[q])
        scale = np.abs(ref) if q == 0 else np.abs(ref).max(axis=-1, keepdims=True)
        for k in (0, 1, rep - 1):
            assert np.all(np.abs(x[k] - ref) <= 1e-11 * scale), q
    # first and last repetition sit in different waves: bitwise the same
    assert np.array_equal(np.asarray(big[0])[:8], np.asarray(big[0])[-8:])
