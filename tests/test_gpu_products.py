"""GPU parity of the FP64 products at the sizes where their tiles end.

The product kernel stages k in steps of 8 and computes tiles of 64 x 64,
64 x 32 or 32 x 32 by four waves, chosen from the sizes and the energy count;
block sizes one below, at and one above those edges, unequal neighbours (so that m, n and K
differ), and energy counts that leave most CUs idle or fill them.  Checked
through the selected solve (products of every operand order, two-term products of equal and
opposite sign, transposed addends, copies and conjugate transposes) against the dense
oracle at 1e-10 per block, the bound of the other parity tests.
"""

import numpy as np
import pytest

from oracle.dense import dense_solve
from quatrex_amd import solve as S
from quatrex_amd.layout import Geometry
from tests.helpers import block_rel_errors, edge_case

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _run(g, A, SL, SG, obc, device):
    import torch

    t = lambda x: torch.as_tensor(np.ascontiguousarray(x), device=device)  # noqa: E731
    E = A[0].shape[0]
    out = [S.packed_empty(g, E, device) for _ in range(3)]
    ob = [[None if x is None else t(x) for x in row] for row in obc] if obc is not None else None
    S.selected_solve(g, tuple(map(t, A)), tuple(map(t, SL)), tuple(map(t, SG)), g_lesser=out[1], g_greater=out[2],
                     g_retarded=out[0], obc=ob)
    S.default_context(device).status()
    return [tuple(x.cpu().numpy() for x in o) for o in out]


def _dense(g, A, SL, SG, obc):
    full = lambda s: g.to_dense(*s, -_lower(g, s[1]))  # noqa: E731
    a, sl, sg = g.to_dense(*A), full(SL), full(SG)
    bo = g.block_offsets
    for k, m, sign in ((0, a, -1), (1, sl, 1), (2, sg, 1)):
        for i, x in enumerate(obc[k] if obc is not None else ()):
            if x is not None:
                m[:, bo[i]:bo[i + 1], bo[i]:bo[i + 1]] += sign * x
    return dense_solve(a, sl, sg)


def _lower(g, upper):
    low = np.empty_like(upper)
    for i in range(g.n_blocks - 1):
        g.lower(low, i)[...] = g.upper(upper, i).conj().swapaxes(-1, -2)
    return low


def _check(g, got, want):
    for x, ref in zip(got, want):
        assert block_rel_errors(g.to_dense(*x), ref, g.block_sizes) <= TOL


@pytest.mark.parametrize("bs,E", [
    ((33, 32, 31), 2), ((63, 64, 65), 2), ((64, 64, 64), 300), ((65, 17, 96), 40), ((127, 33, 129), 3),
    ((96, 95, 97), 64), ((128, 128), 200), ((192, 40, 130), 2), ((48, 1, 47, 8), 5), ((256, 255), 4),
])
def test_products_at_tile_edges_vs_dense(device, bs, E):
    print(f"products bs={bs} E={E}", flush=True)
    g, A, SL, SG, obc = edge_case(bs, seed=sum(bs), E=min(E, 4))
    rep = lambda x: np.ascontiguousarray(np.resize(x, (E, *x.shape[1:])))  # noqa: E731
    A4, SL4, SG4 = A, SL, SG
    big = [tuple(map(rep, m)) for m in (A, SL, SG)]
    bobc = [[None if x is None else rep(x) for x in row] for row in obc]
    got = _run(g, *big, bobc, device)
    want = _dense(g, A4, SL4, SG4, obc)
    n = A4[0].shape[0]
    _check(g, [tuple(p[:n] for p in x) for x in got], want)
    for x in got:  # the same energies further on in the batch
        for p in x:
            np.testing.assert_array_equal(p, np.resize(p[:n], p.shape))


def test_infinities_stay_in_their_energy(device):
    """An energy whose matrix holds Inf and NaN leaves the others untouched, also at
    sizes whose last k-tile and last tile are partial."""
    g, A, SL, SG, obc = edge_case((37, 45, 41), seed=5, E=3)
    want = _run(g, A, SL, SG, obc, device)
    bad = tuple(np.array(x) for x in A)
    bad[0][1, :7] = np.inf
    bad[1][1, 3:9] = np.nan
    got = _run(g, bad, SL, SG, obc, device)
    for x, ref in zip(got, want):
        for p, r in zip(x, ref):
            np.testing.assert_array_equal(p[[0, 2]], r[[0, 2]])
            assert not np.isfinite(p[1]).all()
