"""Interstitial cell integrals with s channels alone (lmax = 0), which have no
recursion: against the sum over the same Gauss points with scipy's spherical
Bessel functions, Z = m j_0(pr) - i p h_0(pr), J = i p h_0(pr) / m, h_0 = j_0 +
i y_0, sigma_00 without the muffin-tin sphere.  A sum of positive weights, so the
1e-12 bar of the other channels holds."""
import numpy as np
import pytest
import scipy.special as sp

from lsms_amd import capi
from lsms_amd import configs as CF
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def test_s_channel_alone():
    rs, cell = 2.3, CF.sphere_cell(0, 2.0, 2.9, ngauss=8)
    _, _, gr, gw, wy = cell
    cg = O.cgaunt(3)[0].ravel()[0]
    rng = np.random.default_rng(0)
    energies = np.array([0.01 + 0.001j, 0.45 + 0.03j, -0.2 + 0.4j, 9.0 + 0.5j])
    n, p = len(energies), np.array([complex(CF.prel_of(e)) for e in energies])
    m = rng.normal(size=n) + 1j * rng.normal(size=n)
    tau = rng.normal(size=(n, 1, 1)) + 1j * rng.normal(size=(n, 1, 1))
    ctx = capi.Context(0)
    ctx.set_tables(3)
    dos, pzz, pzj = ctx.green_interstitial(0, p, m, m, tau, [cell], np.zeros(n, int), [rs])
    ctx.close()
    r, w, sigma = np.asarray(gr).ravel(), np.asarray(gw).ravel(), np.asarray(wy)[0].ravel()
    sigma = sigma - np.sqrt(4 * np.pi) * (r < rs)
    for b in range(n):
        j = sp.spherical_jn(0, p[b] * r)
        h = j + 1j * sp.spherical_yn(0, p[b] * r)
        z = m[b] * j - 1j * p[b] * h
        zz, zj = np.sum(w * cg * sigma * z * z), np.sum(w * cg * sigma * z * 1j * p[b] * h / m[b])
        assert abs(pzz[b, 0, 0] - zz) <= 1e-12 * abs(zz), b
        assert abs(pzj[b] - zj) <= 1e-12 * abs(zj), b
        d = -2.0 * (zz * tau[b, 0, 0] - zj) / np.pi
        assert abs(dos[b] - d) <= 1e-12 * (abs(zz * tau[b, 0, 0]) + abs(zj)), b
