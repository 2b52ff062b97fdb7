"""Beyn's contour on the device at the sizes where its kernels change form: the SVD's column
copy in LDS up to 88 KB (88 x 64) and in global memory above, fewer and more column pairs
than waves, an odd number of columns, quadrature points that do not fill a launch of 16, and
energies in chunks.  Against the converged decimation and the oracle at 1e-8, the bound of
the other tests of this path."""

import numpy as np
import pytest

from oracle import obc as O
from oracle import spectral as SP
from quatrex_amd import _lib
from quatrex_amd import solve as S
from quatrex_amd.boundary_conditions import Spectral
from quatrex_amd.nevp import Beyn
from tests.test_gpu_spectral import _rel, _t
from tests.test_spectral_oracle import contour_radii, low_rank_lead

pytestmark = pytest.mark.gpu

TOL = 1e-8


@pytest.mark.parametrize("b,r,m0,nq,E,chunk", [(5, 1, 3, 50, 4, 0), (33, 6, 15, 72, 5, 2), (40, 8, 33, 57, 3, 0),
                                               (88, 16, 64, 64, 2, 0), (89, 16, 64, 64, 2, 1)])
def test_contour_forms(device, b, r, m0, nq, E, chunk):
    print(f"contour b={b} r={r} m0={m0} nq={nq} E={E} chunk={chunk}", flush=True)
    a = low_rank_lead(b, r, np.linspace(-0.6, 0.7, E), 1e-6, seed=b)
    r_i, r_o = contour_radii(*a)
    kw = dict(max_decay=1.5 * np.log(r_o))
    ctx = S.default_context(device)
    ctx.set_option(_lib.RGF_OPT_MAX_CHUNK, chunk)
    try:
        sp = Spectral(Beyn(r_o=r_o, r_i=r_i, m_0=m0, num_quad_points=nq), **kw)
        x = sp(*(_t(v, device) for v in a), contact="left").cpu().numpy()
    finally:
        ctx.set_option(_lib.RGF_OPT_MAX_CHUNK, 0)
    assert _rel(x, O.sancho_rubio(*a, 400, 1e-13)[0]) <= TOL
    xo, mask, _, _ = SP.spectral_x_ii(*a, r_o=r_o, r_i=r_i, m_0=m0, num_quad_points=nq, **kw)
    assert _rel(x, xo) <= TOL
    np.testing.assert_array_equal(sp.n_reflected.cpu().numpy(), mask.sum(axis=1))
