"""The surface Green's function leaves its inputs as they are (its first iteration reads
them in place), also where the energies go in chunks and as the number of energies a
context has seen grows and shrinks; against the oracle at 1e-10, the bound of the other tests."""

import numpy as np
import pytest

from oracle import obc as O
from quatrex_amd import _lib
from quatrex_amd import solve as S
from quatrex_amd.boundary_conditions import SanchoRubio
from tests.test_gpu_obc import _rel, _t
from tests.test_obc_oracle import _lead

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b", [33, 65])
def test_inputs_stay_and_energy_counts_change(device, b):
    ctx = S.default_context(device)
    for E, chunk in ((2, 0), (7, 0), (7, 3), (1, 0), (4, 2)):
        a = _lead(b, E, 1e-2, seed=b + E)
        ref, it, _ = O.sancho_rubio(*a, 100, 1e-8)
        dev = [_t(x, device) for x in a]
        ctx.set_option(_lib.RGF_OPT_MAX_CHUNK, chunk)
        try:
            sr = SanchoRubio(100, 1e-8)
            x = sr(*dev, "c").cpu().numpy()
        finally:
            ctx.set_option(_lib.RGF_OPT_MAX_CHUNK, 0)
        assert sr.iterations == it
        assert _rel(x, ref) <= 1e-10
        for d, h in zip(dev, a):
            np.testing.assert_array_equal(d.cpu().numpy(), h)
