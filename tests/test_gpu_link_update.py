"""The exponential of the link update over the sizes of its argument: tiny,
around the line where scaling and squaring starts (the sum of the entries'
magnitudes at 1), and large.  Against scipy's matrix exponential in numpy; each
squaring doubles an error of 1e-16, so that 1e-13 holds up to some ten of them."""
import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [0.0, 1e-9, 0.02, 0.08, 0.12, 0.2, 1.0, 10.0])
def test_link_update_exponential(size):
    from scipy.linalg import expm
    import bqcd_hip
    L = (4, 4, 2, 2)
    lat = ol.Lattice(L)
    u = lat.gauge_exp_random(17, 0.5)
    p = lat.momenta_gauss(18)
    g = bqcd_hip.Lattice(L)
    g.load_gauge(u)
    g.hmc_u(p, size)
    got = g.save_gauge()
    g.close()
    lam = np.zeros((8, 3, 3), complex)
    lam[0][0, 1] = lam[0][1, 0] = lam[3][0, 2] = lam[3][2, 0] = lam[5][1, 2] = lam[5][2, 1] = 1
    lam[1][0, 1], lam[4][0, 2], lam[6][1, 2] = -1j, -1j, -1j
    lam[1][1, 0], lam[4][2, 0], lam[6][2, 1] = 1j, 1j, 1j
    lam[2] = np.diag([1, -1, 0])
    lam[7] = np.diag([1, 1, -2]) / np.sqrt(3)
    m = (u[..., 0] + 1j * u[..., 1]).reshape(-1, 3, 3)  # [column, row]
    e = np.stack([expm(1j * size * np.einsum("j,jab", q, lam)) for q in p.reshape(-1, 8)])
    want = np.einsum("nab,ncb->nca", e, m)
    new = (got[..., 0] + 1j * got[..., 1]).reshape(-1, 3, 3)
    assert np.max(np.abs(new - want)) < 1e-13
